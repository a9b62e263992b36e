"""Which calls the row GEMMs, the routing kernels and the prompt attention kernels
take.  The rules are about sizes, types and addresses, so they are checked here
on stand-ins, without a GPU: whatever the row GEMMs take, for instance, is read by
kernels that know only x's sizes and the number of weight rows."""
import ctypes
import re
from collections import defaultdict
from pathlib import Path
from types import SimpleNamespace

import pytest
import torch

from agentfield_amd import ops


def mat(*shape, dtype=torch.bfloat16, device="cuda:0", contiguous=True,
        addr=1 << 20):
    return SimpleNamespace(
        shape=torch.Size(shape), dtype=dtype, device=torch.device(device),
        is_cuda=device.startswith("cuda"), is_contiguous=lambda: contiguous,
        data_ptr=lambda: addr, dim=lambda: len(shape))


@pytest.mark.parametrize("M", [1, 16, 17, 128])
@pytest.mark.parametrize("N,K", [(64, 64), (4096, 512), (128256, 4096)])
def test_taken(M, N, K):
    assert ops._rows_ok(mat(M, K), mat(N, K))


@pytest.mark.parametrize("x,w", [
    (mat(4, 512), mat(128, 448)),            # rows longer than the weights'
    (mat(4, 448), mat(128, 512)),            # and shorter
    (mat(512), mat(128, 512)),
    (mat(2, 4, 512), mat(128, 512)),
    (mat(4, 512), mat(2, 128, 512)),
    (mat(0, 512), mat(128, 512)),
    (mat(129, 512), mat(128, 512)),
    (mat(4, 0), mat(128, 0)),
    (mat(4, 512), mat(0, 512)),
    (mat(4, 512), mat(96, 512)),
    (mat(4, 480), mat(128, 480)),
    (mat(4, 512), mat(128, 512, device="cpu")),
    (mat(4, 512, device="cpu"), mat(128, 512)),
    (mat(4, 512), mat(128, 512, device="cuda:1")),
    (mat(4, 512, dtype=torch.float32), mat(128, 512, dtype=torch.float32)),
    (mat(4, 512), mat(128, 512, dtype=torch.float16)),
    (mat(4, 512, contiguous=False), mat(128, 512)),
    (mat(4, 512), mat(128, 512, contiguous=False)),
    (mat(4, 512, addr=8), mat(128, 512)),
    (mat(4, 512), mat(128, 512, addr=2)),
], ids=lambda t: f"{'x'.join(map(str, t.shape))}")
def test_left_to_the_library(x, w):
    assert not ops._rows_ok(x, w)


def test_few_row_path_needs_plain_bf16_weights():
    """The few-row path of the dense decoder serves bf16 models, and of these the
    layers whose weights the row GEMMs read; everything else keeps the general
    path, prompts included."""
    from agentfield_amd.models import CONFIGS
    from agentfield_amd.models.llama import LlamaForCausalLM

    def model(dtype):
        return LlamaForCausalLM(CONFIGS["tiny"], dtype=dtype).init_random(
            0).fold_norm_weights()
    assert not model(torch.float32)._can_fuse_rows(4)
    assert not model(torch.float16)._can_fuse_rows(4)
    m = model(torch.bfloat16)
    assert m._can_fuse_rows(1) and m._can_fuse_rows(128)
    assert not m._can_fuse_rows(129) and not m._can_fuse_rows(0)
    layer = m.layers[1]
    for part, name in (("attn", "qkv"), ("attn", "o"), ("mlp", "gate_up"),
                       ("mlp", "down")):
        assert layer.rows_weights(m.cfg) is not None
        p = getattr(getattr(layer, part), name)
        flat = p.data.clone()
        p.data = flat.t().contiguous().t()          # strided
        assert layer.rows_weights(m.cfg) is None
        p.data = torch.cat([flat.flatten()[:1], flat.flatten()])[1:].view_as(
            flat)                                   # off the 16-byte grid
        assert layer.rows_weights(m.cfg) is None
        p.data = flat[:-64]                         # of another size
        assert layer.rows_weights(m.cfg) is None
        p.data = flat
    p.data = flat.float()
    assert layer.rows_weights(m.cfg) is None
    p.data = flat
    torch.nn.utils.parametrize.register_parametrization(
        layer.mlp, "down", torch.nn.Identity())
    with torch.no_grad():
        assert torch.equal(layer.rows_weights(m.cfg)[3], flat)


def test_watched_products():
    """Autograd, forward mode, transforms and tracers see a product; grad mode
    alone, with nothing that requires a gradient, does not keep it from the
    kernels."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    x, w = torch.randn(4, 8), torch.randn(6, 8)
    p = torch.nn.Parameter(w)
    seen = []
    assert not ops.watched(x, w)
    assert ops.watched(x, p) and ops.watched(x.clone().requires_grad_(), w)
    assert not ops.watched(x, p, grad=False)
    with torch.no_grad():
        assert not ops.watched(x, p)
    with torch.inference_mode():
        assert not ops.watched(x, p)

    def look(a):
        seen.append(ops.watched(a, w))
        return a * 2
    torch.func.vmap(look)(torch.stack([x, x]))
    torch.func.grad(lambda a: look(a).sum())(x)
    torch.func.jvp(look, (x,), (x,))
    with forward_ad.dual_level(), torch.no_grad():
        look(forward_ad.make_dual(x, x))
    with FakeTensorMode() as m:
        look(m.from_tensor(x))
    torch.fx.experimental.proxy_tensor.make_fx(look)(x)

    class Sub(torch.Tensor):
        pass
    look(x.as_subclass(Sub))
    assert seen == [True] * 7
    assert not ops.watched(x, w)


@pytest.mark.parametrize("ok,x,router,k", [
    (True, mat(1, 520), mat(4, 520), 2),
    (True, mat(700, 4096), mat(64, 4096), 8),
    (False, mat(4, 520), mat(4, 512), 2),           # other row lengths
    (False, mat(4, 512), mat(4, 520), 2),
    (False, mat(4, 516), mat(4, 516), 2),
    (False, mat(4, 520), mat(4, 520, contiguous=False), 2),
    (False, mat(4, 520), mat(4, 520, addr=8), 2),
    (False, mat(4, 520), mat(4, 520, device="cpu"), 2),
    (False, mat(4, 520), mat(4, 520, device="cuda:1"), 2),
    (False, mat(4, 520), mat(4, 520, dtype=torch.float32), 2),
    (False, mat(4, 520, contiguous=False), mat(4, 520), 2),
    (False, mat(4, 520, device="cpu"), mat(4, 520), 2),
    (False, mat(0, 520), mat(4, 520), 2),
    (False, mat(4, 520), mat(65, 520), 2),
    (False, mat(4, 520), mat(16, 520), 9),
    (False, mat(4, 520), mat(4, 520), 5),            # more choices than experts
    (False, mat(4, 520), mat(4, 520), 0),
])
def test_rows_that_the_routing_kernels_take(monkeypatch, ok, x, router, k):
    from agentfield_amd.models.llama import MoEMLP
    monkeypatch.setattr(ops, "watched", lambda *t, **kw: False)
    layer = SimpleNamespace(router=router, gate_up=None, down=None, top_k=k)
    assert MoEMLP._can_sort(layer, x) == ok


@pytest.mark.parametrize("ok,gate_up,down", [
    (True, mat(4, 128, 64), mat(4, 64, 64)),
    (True, mat(4, 384, 64), mat(4, 64, 192)),
    (False, mat(5, 128, 64), mat(5, 64, 64)),         # experts without a router row
    (False, mat(3, 128, 64), mat(3, 64, 64)),
    (False, mat(4, 128, 64), mat(3, 64, 64)),
    (False, mat(4, 192, 64), mat(4, 64, 96)),         # lengths in 64s only
    (False, mat(4, 128, 128), mat(4, 128, 64)),       # other rows than x's
    (False, mat(4, 128, 64), mat(4, 64, 128)),
    (False, mat(4, 128, 64), mat(4, 128, 64)),
    (False, mat(128, 64), mat(64, 64)),
    (False, mat(4, 128, 64, contiguous=False), mat(4, 64, 64)),
    (False, mat(4, 128, 64), mat(4, 64, 64, addr=8)),
    (False, mat(4, 128, 64), mat(4, 64, 64, dtype=torch.float32)),
    (False, mat(4, 128, 64), mat(4, 64, 64, device="cuda:1")),
])
def test_experts_that_the_sorted_products_take(ok, gate_up, down):
    assert ops.moe_gemm_ok(mat(5, 64), mat(4, 64), gate_up, down) == ok


@pytest.mark.parametrize("n,E,H,I,pays", [
    (2, 8, 4096, 14336, False), (4, 4, 4096, 14336, False),
    (6, 8, 4096, 14336, True), (8, 4, 4096, 14336, True),
    (2, 8, 4096, 8192, True), (2, 8, 6144, 16384, False), (4, 8, 6144, 16384, True),
    (64, 2, 8192, 28672, False), (65, 2, 8192, 28672, True), (2, 4, 256, 512, True)])
def test_when_one_launch_per_projection_pays(n, E, H, I, pays):
    assert ops.moe_gemm_pays(n, E, H, I) == pays


@pytest.mark.parametrize("lens,want", [
    ([8000], (32, 250, 0, 1)),                     # one long prompt
    ([700, 3, 8, 500, 9], (32, 39, 2, 4)),         # both kinds of items
    ([60] * 4, (1 << 30, 0, 32, 1)),               # few 128-column blocks
    ([5] * 16, (1 << 30, 0, 16, 2)),               # drafts: keys split
    ([5], (1 << 30, 0, 1, 8)),
    ([300, 0, 400], (32, 23, 0, 1)),
    ([], (1 << 30, 0, 0, 1)),
])
def test_prefill_split_reaches_every_kernel(lens, want):
    """The rule by which prompt attention is cut (8 K/V heads, four query heads
    each, pages for 8192 tokens): a change of it shows which kernels a step
    still reaches."""
    assert ops.prefill_split(lens, 4, 8, 8192) == want


@pytest.mark.parametrize("K", [64, 128, 832, 4096, 14336, 65536])
@pytest.mark.parametrize("N", [64, 192, 4096, 6144, 24576, 128256])
def test_rows_splits_leave_no_split_empty(N, K):
    for M in (1, 16, 17, 32, 33, 64, 65, 128):
        n, pieces = ops.rows_splits(M, N, K), K // 64
        assert 1 <= n <= min(16, pieces)
        assert (n - 1) * -(-pieces // n) < pieces


@pytest.mark.parametrize("x,w,ok", [
    (mat(256, 128), mat(256, 128), True),
    (mat(10077, 4096), mat(28672, 4096), True),
    (mat(257, 192), mat(320, 192), True),
    (mat(300, 8192), mat(57344, 8192), True),
    (mat(255, 128), mat(256, 128), False),        # tiles are 256 rows at most
    (mat(256, 128), mat(192, 128), False),
    (mat(256, 128), mat(288, 128), False),
    (mat(256, 64), mat(256, 64), False),          # two pieces of K are on their way
    (mat(256, 160), mat(256, 160), False),
    (mat(256, 128), mat(256, 192), False),
    (mat(256, 1 << 18), mat(1 << 14, 1 << 18), False),   # offsets of 32 bits
    (mat(4, 64, 128), mat(256, 128), False),
    (mat(256, 128, dtype=torch.float16), mat(256, 128, dtype=torch.float16), False),
    (mat(256, 128, contiguous=False), mat(256, 128), False),
    (mat(256, 128), mat(256, 128, addr=8), False),
    (mat(256, 128), mat(256, 128, device="cuda:1"), False),
    (mat(256, 128, device="cpu"), mat(256, 128, device="cpu"), False),
])
def test_wide_gemm_operands(x, w, ok):
    assert ops._wide_ok(x, w) == ok


@pytest.mark.parametrize("M,N,K,glu,pays", [
    (4096, 28672, 4096, True, True), (384, 14848, 4096, True, True),
    (384, 14336, 4096, True, False),              # 168 tiles: few blocks at work
    (4096, 4096, 4096, False, False),             # one whole round
    (4097, 4096, 4096, False, True),              # a second one begun
    (6144, 4096, 4096, False, True), (6145, 4096, 4096, False, False),
    (6145, 4096, 14336, False, True), (7680, 4096, 14336, False, False),
    (2048, 4096, 4096, False, False),
])
def test_wide_gemm_pays(M, N, K, glu, pays):
    assert ops._wide_pays(M, N, K, glu) == pays


@pytest.mark.parametrize("M,N,K,glu,pays", [
    (5120, 4096, 14336, False, False),            # 64 begun, even shares of K
    (5121, 4096, 14336, False, True), (5632, 5120, 13824, False, True),
    (2500, 8192, 28672, False, False), (2700, 8192, 28672, False, True),
    (4500, 8192, 28672, False, False), (6300, 8192, 28672, False, False),
    (2030, 12288, 4096, False, False), (1500, 12288, 4096, False, True),
    (10077, 12288, 4096, False, False), (9900, 10240, 8192, False, False),
    (4000, 10240, 8192, False, True), (6500, 8192, 8192, False, False),
    (6500, 8192, 3584, False, True), (6900, 8192, 3584, False, False),
    (1100, 28672, 4096, False, False), (2048, 28672, 4096, False, False),
    (1024, 22016, 4096, False, False), (5000, 14336, 4096, False, False),
    (257, 16384, 2048, True, False), (384, 16384, 3072, True, False),
    (385, 16384, 3072, True, True), (257, 20480, 2048, True, True),
    (384, 16384, 1024, True, True), (257, 22016, 4096, True, True),
    (448, 22016, 4096, True, True), (449, 22016, 4096, True, False),
    (512, 24576, 8192, True, False), (513, 22016, 4096, True, True),
    (512, 22016, 2048, True, True), (512, 20480, 4096, True, True),
    (2560, 22016, 4096, False, False), (2300, 22016, 4096, False, True),
])
def test_wide_gemm_leaves_what_the_library_does_better(M, N, K, glu, pays):
    assert ops._wide_pays(M, N, K, glu) == pays


@pytest.mark.parametrize("M,N,K,pays", [
    (10284, 4096, 4096, True), (11000, 4096, 4096, True),    # 219, 229 blocks come out even
    (7634, 8256, 2048, True), (1500, 6144, 4096, True),      # none; below one round
    (7634, 8192, 2048, False), (7634, 2048, 2048, False),    # 240 do
    (10284, 6144, 4096, False), (9000, 10240, 2048, False),  # 246, 240
    (1500, 4096, 4096, False), (2000, 4096, 4096, False),    # up to 128 tiles
    (2400, 8192, 8192, False), (11157, 12288, 4096, False),  # a long K; many rounds
    (255, 6144, 4096, False),
])
def test_wide_gemm_where_the_library_cannot_divide(M, N, K, pays):
    assert ops._wide_pays(M, N, K, False) == pays


@pytest.mark.parametrize("M,N,K,pays", [
    (1280, 2048, 10240, True), (1281, 2048, 10240, False), (2068, 2048, 10240, False),
    (2048, 2048, 16384, True)])
def test_wide_gemm_split_of_few_columns(M, N, K, pays):
    assert ops._wide_split_pays(M, N, K) == pays


@pytest.mark.parametrize("M,N,K,pays", [
    (128, 4096, 14336, False), (257, 4096, 14336, True), (2048, 4096, 14336, True),
    (2049, 4096, 14336, False),                   # 144 tiles
    (512, 8192, 28672, True), (513, 8192, 28672, False),
    (300, 2048, 8192, False), (300, 8192, 14336, False), (300, 4096, 14368, False),
    (300, 4096, 4096, False),
    (300, 4096, 8384, False),                     # 131 pieces: no shares
    (256, 4096, 11008, False), (257, 4096, 11008, True),      # 128 and 192 blocks
])
def test_wide_gemm_split_pays(M, N, K, pays):
    assert ops._wide_split_pays(M, N, K) == pays


@pytest.mark.parametrize("x_rows,n,E,N,K,glu,pays", [
    (800, 1600, 8, 28672, 4096, True, True), (799, 1599, 8, 28672, 4096, True, False),
    (2000, 2000, 8, 4096, 14336, False, True),
    (1999, 1999, 8, 4096, 14336, False, False),
    (800, 1600, 8, 128, 4096, True, False), (800, 2000, 8, 4096, 64, False, False),
    (1 << 19, 1 << 20, 8, 28672, 4096, True, False),      # 4 GB of rows
])
def test_wide_experts_pay(x_rows, n, E, N, K, glu, pays):
    assert ops.wide_experts_pay(x_rows, n, E, N, K, glu) == pays


@pytest.mark.parametrize("M,N,pays", [
    (32, 16384, True), (33, 12288, True), (33, 12352, False), (128, 24512, False),
    (128, 24576, True)])
def test_rows_pay(M, N, pays):
    assert ops.rows_pay(M, N) == pays


class Operand(SimpleNamespace):
    """A stand-in that torch would multiply."""

    def t(self):
        return self

    def __matmul__(self, other):
        return "torch"


@pytest.mark.parametrize("index,cast,own", [
    (0, False, True), (1, False, False), (0, True, False)])
@pytest.mark.parametrize("M,N,K,glu", [
    (4353, 4096, 4096, False), (300, 4096, 14336, False),
    (4096, 28672, 4096, True)])
def test_wide_products_that_stay_with_torch(monkeypatch, index, cast, own, M, N, K,
                                            glu):
    """Operands on another device than the current one, whose stream a launch would
    take, stay with torch, which goes to theirs; so do products under autocast, which
    may want another type than the operands'."""
    from agentfield_amd.ops import seqmix
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda kind: cast)
    monkeypatch.setattr(ops, "watched", lambda *t, **kw: False)
    monkeypatch.setattr(ops, "silu_and_mul", lambda y: y)
    for name in ("launch_wide", "launch_wide_split"):
        monkeypatch.setattr(ops, name, lambda *a, **kw: "own")
    x, w = (Operand(**vars(mat(n, K, device=f"cuda:{index}"))) for n in (M, N))
    want = "own" if own else "torch"
    assert ops.linear(x, w, silu_fuse=glu) == want
    if not glu and K == 4096:
        assert seqmix.matmul(x, w) == want


def test_wide_split_without_room_for_its_parts(monkeypatch):
    """Where the shares' sums find no memory the product is torch's, which needs none."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(ops, "watched", lambda *t, **kw: False)

    def full(*a, **kw):
        raise torch.OutOfMemoryError("full")
    monkeypatch.setattr(ops, "launch_wide_split", full)
    x, w = (Operand(**vars(mat(n, 14336))) for n in (300, 4096))
    assert ops.linear(x, w) == "torch"


@pytest.mark.parametrize("B,Hk,G,nsplit,window,shares", [
    (24, 8, 4, 2, 0, True), (48, 8, 4, 2, 0, True), (49, 8, 4, 2, 0, False),
    (32, 8, 8, 2, 0, True), (33, 8, 8, 2, 0, False), (64, 1, 4, 4, 0, True),
    (65, 1, 4, 2, 0, False), (1, 8, 4, 4, 0, False), (2, 8, 4, 1, 0, False),
    (9, 8, 4, 5, 0, False), (24, 8, 4, 2, 4096, False)])
def test_decode_steps_that_may_be_cut_in_shares(B, Hk, G, nsplit, window, shares):
    """Room for all blocks at once, a lane per sequence, two to four parts, no window; the
    scratch has room for one piece more of each sequence there, and only there."""
    assert ops.decode_shares(B, Hk, G, nsplit, window) == shares
    po, pml = ops.decode_scratch(B, Hk, nsplit, G, "cpu", shares=shares)
    assert po.shape == (B, Hk, nsplit + shares, G, 128)
    assert pml.shape == (B, Hk, nsplit + shares, G, 2)
    assert ops.decode_cut(torch.ones(B, dtype=torch.int32), Hk, G, nsplit, window) is None


ROOT = Path(__file__).resolve().parent.parent


def prototypes(text, mark):
    """{name: kinds of its arguments} of the C entry points that are declared or defined
    behind mark."""
    kinds = {"int": "i", "long": "l", "i64": "l", "int64_t": "l", "float": "f", "u32": "u", "uint32_t": "u",
             "unsigned long long": "q", "uint64_t": "q"}
    out = {}
    for name, args in re.findall(mark + r"int (af_\w+)\(([^)]*)\)", text):
        args = [a.replace("const", " ").strip() for a in args.split(",")]
        out[name] = "".join(
            "" if a in ("", "void") else "p" if "*" in a
            else kinds[" ".join(a.split()[:-1]) or a] for a in args)
    return out


def defined():
    text = "".join(f.read_text() for f in (ROOT / "agentfield_amd" / "csrc").glob("*.hip"))
    return prototypes(text, "AF_EXPORT ")


@pytest.mark.parametrize("path", sorted((ROOT / "tools").glob("*.cpp")), ids=lambda p: p.name)
def test_tools_call_the_kernels_as_they_are(path):
    """A declaration of other arguments links all the same, and passes sizes for streams."""
    want, got = defined(), prototypes(path.read_text(), r"(?m)^")
    assert got and {n: want[n] for n in got} == got


def test_bindings_call_the_kernels_as_they_are():
    """The loader's argument types against the entry points' own."""
    from agentfield_amd.ops import _lib
    fake = defaultdict(SimpleNamespace)

    class Library:
        def __getattr__(self, name):
            return fake[name]
    _lib._declare(Library())
    kinds = {ctypes.c_void_p: "p", ctypes.c_int: "i", ctypes.c_int64: "l",
             ctypes.c_float: "f", ctypes.c_uint32: "u"}
    want = defined()
    got = {n: "".join(kinds.get(t, "?") for t in f.argtypes) for n, f in fake.items()
           if hasattr(f, "argtypes")}
    assert len(got) > 30
    for name, args in got.items():
        if "?" not in args:
            assert args == want[name], name
