"""cSwiGLU's w13 projection and gate as one kernel (fused.swiglu_linear, ffn.hip) against the
reference's two steps (primitives.py:92-105): h = x w13^T as a bf16 Linear (fp32
accumulation, rounded to bf16), then the gate with the eager bf16 rounding points."""
import contextlib

import pytest
import torch
import torch.nn.functional as F
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from mosaic_amd import fused
from mosaic_amd.model import cSwiGLU

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def reference(x, w13, noise):
    """fp32-accumulated projection rounded to bf16, then the gate in eager bf16 ops."""
    h = (x.float() @ w13.float().t()).to(torch.bfloat16)
    x1, x3 = h.chunk(2, dim=-1)
    if noise is not None:
        x1 = x1 + noise.to(torch.bfloat16)          # [S, B, H] + [B, H], rounded to bf16
    return F.silu(x1) * x3


def check(got, ref, name):
    g, r = got.float().cpu(), ref.float().cpu()
    assert torch.isfinite(g).all(), f"{name}: non-finite"
    rel = ((g - r).norm() / r.norm().clamp_min(1e-30)).item()
    err = (g - r).abs().max().item()
    bound = 2e-2 * max(1.0, r.abs().max().item())
    print(f"  {name}: rel_l2 {rel:.2e} max_abs {err:.2e} (bound {bound:.2e})", flush=True)
    assert rel <= 1e-2 and err <= bound, f"{name}: rel_l2 {rel:.3e} max_abs {err:.3e}"


@pytest.mark.parametrize("S,B,dim,hidden,noise", [
    (128, 4, 256, 256, True),
    (256, 1, 128, 384, False),
    (64, 24, 768, 3072, True),      # stage-1 widths of the era5 preset, 24 members
    (64, 12, 1024, 4096, True),     # stage-2 widths
    (32, 8, 1280, 5120, False),     # bottleneck widths
])
def test_swiglu_linear_matches_reference(S, B, dim, hidden, noise):
    print(f"swiglu_linear S={S} B={B} dim={dim} hidden={hidden} noise={noise}", flush=True)
    g = torch.Generator().manual_seed(S + dim + hidden)
    x = torch.randn(S, B, dim, generator=g).to(torch.bfloat16)
    w13 = (torch.randn(2 * hidden, dim, generator=g) * dim ** -0.5).to(torch.bfloat16)
    nz = torch.randn(B, hidden, generator=g).to(torch.bfloat16) if noise else None
    xd, wd = x.to(DEV), w13.to(DEV)
    nd = nz.to(DEV) if nz is not None else None
    with torch.no_grad():
        got = fused.swiglu_linear(xd, fused.permute_w13(wd), nd)
        two_step = fused.swiglu((xd @ wd.t()), nd)      # library GEMM, then the gate kernel
    torch.cuda.synchronize()
    assert got.shape == (S, B, hidden) and got.dtype == torch.bfloat16
    check(got, reference(x, w13, nz), "vs fp32-accumulate reference")
    check(got, two_step, "vs library GEMM + gate kernel")


def test_swiglu_linear_strided_rows():
    """x as a row-strided view (a slice of a wider activation)."""
    g = torch.Generator().manual_seed(7)
    xw = torch.randn(512, 384, generator=g).to(torch.bfloat16)
    x = xw[:, :256]                                     # row stride 384
    w13 = (torch.randn(512, 256, generator=g) * 256 ** -0.5).to(torch.bfloat16)
    with torch.no_grad():
        got = fused.swiglu_linear(x.to(DEV), fused.permute_w13(w13.to(DEV)))
    check(got, reference(x, w13, None), "strided x")


def test_swiglu_linear_wide_hidden():
    """A tile of out that spans more than 4 GB: byte offsets past 32 bits, every row and noise row."""
    hidden, dim = (1 << 23) + (1 << 16), 128
    g = torch.Generator(DEV).manual_seed(8)
    x = torch.randn(128, 2, dim, generator=g, device=DEV).to(torch.bfloat16)
    w13 = torch.empty(2 * hidden, dim, dtype=torch.bfloat16, device=DEV).normal_(0, dim ** -0.5, generator=g)
    nz = torch.empty(2, hidden, dtype=torch.bfloat16, device=DEV).normal_(generator=g)
    got = fused.swiglu_linear(x, fused.permute_w13(w13), nz)
    cols = torch.cat([torch.arange(c, c + 256) for c in (0, hidden // 2, hidden - 256)]).to(DEV)
    ref = reference(x, torch.cat([w13[cols], w13[hidden + cols]]), nz[:, cols])
    check(got[..., cols], ref, "wide hidden")


def test_cswiglu_module_fused_equals_unfused():
    """cSwiGLU.forward through the fused kernel and through w13 + gate kernel + w2."""
    torch.manual_seed(0)
    m = cSwiGLU(768, 3072, 64).to(DEV)
    x = torch.randn(64, 24, 768, device=DEV).to(torch.bfloat16)
    z = torch.randn(24, 64, device=DEV)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        m.fused_linear_gate = True
        a = m(x, z)
        m.fused_linear_gate = False
        b = m(x, z)
    check(a, b, "module fused vs unfused")
    # a changed weight is seen by the next region
    with torch.no_grad():
        m.w13.weight.mul_(0.5)
        m.fused_linear_gate = True
        with torch.autocast("cuda", dtype=torch.bfloat16):
            c = m(x, z)
            m.fused_linear_gate = False
            d = m(x, z)
    check(c, d, "after a weight update")


@pytest.mark.parametrize("fused_gate", [True, False])
def test_cswiglu_refuses_grad(fused_gate):
    """With grad mode on and weights that require grad, both paths raise rather than return an
    output cut off from the graph."""
    m = cSwiGLU(256, 256, 0).to(DEV).to(torch.bfloat16)
    m.fused_linear_gate = fused_gate
    x = torch.randn(256, 1, 256, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no backward"):
        m(x)


@pytest.mark.parametrize("S,B,dim,hidden,noise", [
    (256, 1, 128, 128, True),       # one tile, the shortest reduction
    (257, 1, 256, 128, True),       # a last row tile that starts one row after the first
    (1000, 3, 384, 256, True),      # ragged rows, members that do not divide a tile
    (19, 56, 256, 384, True),       # the most noise rows staged in LDS
    (18, 57, 256, 384, True),       # one more: noise from global memory
    (4100, 1, 1280, 640, False),    # 85 tiles in a partial last round over the XCDs, no noise
    (2048, 2, 128, 1280, True),     # several tiles per workgroup with two iterations each
])
def test_swiglu_linear_w13_shapes(S, B, dim, hidden, noise):
    """The kernel on w13 as stored, at the edges of its tiles, noise paths and tile rounds, on a
    poisoned allocation: every row written, against the fp32-accumulate reference."""
    print(f"swiglu_linear_w13 S={S} B={B} dim={dim} hidden={hidden} noise={noise}", flush=True)
    g = torch.Generator().manual_seed(S + B + dim)
    x = torch.randn(S, B, dim, generator=g).to(torch.bfloat16)
    w13 = (torch.randn(2 * hidden, dim, generator=g) * dim ** -0.5).to(torch.bfloat16)
    nz = torch.randn(B, hidden, generator=g).to(torch.bfloat16) if noise else None
    xd, wd, nd = x.to(DEV), w13.to(DEV), nz.to(DEV) if noise else None
    torch.cuda.empty_cache()
    poison = torch.full((S, B, hidden), float("nan"), dtype=torch.bfloat16, device=DEV)
    memory = poison.data_ptr()
    del poison                                   # the next output's memory
    got = fused.swiglu_linear_w13(xd, wd, nd)
    assert got.data_ptr() == memory
    ref = reference(x, w13, nz)
    check(got, ref, "vs fp32-accumulate reference")
    # only sums in another order and the silu's last fp32 bits differ: bf16 roundings rarely flip
    assert (got.cpu() == ref).float().mean().item() >= 0.999


def test_swiglu_linear_w13_non_finite_rows_stay_in_their_rows():
    x = torch.randn(600, 1, 256, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    w13 = (torch.randn(512, 256, generator=torch.Generator().manual_seed(4)) / 16).to(torch.bfloat16)
    clean = fused.swiglu_linear_w13(x.to(DEV), w13.to(DEV)).cpu()
    x[5, 0, 7], x[599, 0, 0] = float("inf"), float("nan")
    got = fused.swiglu_linear_w13(x.to(DEV), w13.to(DEV)).cpu()
    keep = torch.ones(600, dtype=torch.bool)
    keep[[5, 599]] = False
    assert torch.equal(got[keep], clean[keep]) and got[599].isnan().all()
    want = fused.swiglu((x[5:6].to(DEV) @ w13.to(DEV).t())).cpu()
    assert torch.equal(got[5].isnan(), want[0].isnan()) and torch.equal(got[5].isinf(), want[0].isinf())


class _SeenFunctions(TorchFunctionMode):
    def __init__(self, seen):
        super().__init__()
        self.seen = seen

    def __torch_function__(self, func, types, args=(), kwargs=None):
        if func is F.linear and args[1].shape[0] == 2048:
            self.seen.append(1)
        return func(*args, **(kwargs or {}))


class _SeenOperators(TorchDispatchMode):
    def __init__(self, seen):
        super().__init__()
        self.seen = seen

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if func in (torch.ops.aten.mm.default, torch.ops.aten.addmm.default) and args[-1].shape[-1] == 2048:
            self.seen.append(1)
        return func(*args, **(kwargs or {}))


class _Casts(TorchDispatchMode):
    """Counts the casts of a 2048-row weight to bf16."""
    n = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.n += func is torch.ops.aten._to_copy.default and args[0].shape[0] == 2048 and args[0].dtype == torch.float32
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("change", ["none", "default_device", "hook", "global_hook", "bias", "replaced", "fp32_noise",
                                    "odd_rows", "view", "forward", "class_forward", "linear", "compiled",
                                    "function_mode", "dispatch_mode"])
def test_cswiglu_routes(change, monkeypatch):
    """The module takes the one kernel only where nothing observes or replaces w13 and the shape
    fits, and its result is the two-step one on every route."""
    torch.manual_seed(1)
    m = cSwiGLU(256, 1024, 64).to(DEV)
    x = torch.randn(1030, 2, 256, device=DEV).to(torch.bfloat16)
    z = torch.randn(2, 64, device=DEV)
    calls, seen = [], []
    real = fused.swiglu_linear_w13
    monkeypatch.setattr(fused, "swiglu_linear_w13", lambda *a: calls.append(1) or real(*a))
    handle, mode = None, contextlib.nullcontext()
    if change == "forward":
        own = m.w13.forward
        m.w13.forward = lambda t: seen.append(1) or own(t)
    elif change == "class_forward":
        base = torch.nn.Linear.forward
        monkeypatch.setattr(torch.nn.Linear, "forward", lambda lin, t: (lin is m.w13 and seen.append(1)) or base(lin, t))
    elif change == "linear":
        base = F.linear
        monkeypatch.setattr(F, "linear", lambda t, w, b=None: (w is m.w13.weight and seen.append(1)) or base(t, w, b))
    elif change == "compiled":
        m.w13._compiled_call_impl = lambda t: seen.append(1) or F.linear(t, m.w13.weight)
    elif change == "function_mode":
        mode = _SeenFunctions(seen)
    elif change == "dispatch_mode":
        mode = _SeenOperators(seen)
    elif change == "default_device":
        mode = torch.device(DEV)
    if change == "hook":
        m.w13.register_forward_hook(lambda *a: seen.append(1))
    elif change == "global_hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda mod, *a: seen.append(1) if mod is m.w13 else None)
    elif change == "bias":
        lin = torch.nn.Linear(256, 2048).to(DEV)
        lin.weight = m.w13.weight
        m.w13 = lin
    elif change == "replaced":
        m.w13 = torch.nn.Sequential(m.w13)
    elif change == "fp32_noise":
        m.noise_bias = torch.nn.Identity()
        z = torch.randn(2, 1024, device=DEV)
    elif change == "odd_rows":
        x = x[:100]
    elif change == "view":
        x = torch.randn(1030, 2, 512, device=DEV).to(torch.bfloat16)[..., 128:384]
    try:
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16), mode:
            got = m(x, z)
            n, m.fused_linear_gate = len(calls), False
            want = m(x, z)
    finally:
        if handle is not None:
            handle.remove()
    assert n == (1 if change in ("none", "default_device") else 0) and len(calls) == n
    watched = ("hook", "global_hook", "forward", "class_forward", "linear", "compiled", "function_mode", "dispatch_mode")
    assert len(seen) == (2 if change in watched else 0)
    check(got, want, change)


@pytest.mark.parametrize("cache,frozen", [(True, False), (False, False), (True, True)])
def test_cswiglu_weight_cast_is_autocasts(cache, frozen, monkeypatch):
    """Inside one autocast region w13 is cast as often as its Linear would: once where autocast
    caches the cast, at every call with its cache off or a weight that needs no gradient."""
    m = cSwiGLU(256, 1024, 0).to(DEV).requires_grad_(not frozen)
    x = torch.randn(2048, 1, 256, device=DEV).to(torch.bfloat16)
    weights = []
    real = fused.swiglu_linear_w13
    monkeypatch.setattr(fused, "swiglu_linear_w13", lambda x, w, n: weights.append(w) or real(x, w, n))
    linear_casts = _Casts()
    with torch.no_grad():
        with torch.autocast("cuda", dtype=torch.bfloat16, cache_enabled=cache):
            m(x), m(x)
        with torch.autocast("cuda", dtype=torch.bfloat16, cache_enabled=cache), linear_casts:
            m.w13(x), m.w13(x)
    assert len(weights) == 2 and all(w.dtype == torch.bfloat16 for w in weights)
    assert len({w.data_ptr() for w in weights}) == linear_casts.n == (1 if cache and not frozen else 2)


def test_swiglu_linear_gate_every_argument():
    """silu of every bf16 value (negative zero aside: a sum of products has none), subnormal, infinite
    and NaN ones among them, each as one product 1 * value: the bits of the gate kernel (expf and a
    division), and where the float64 silu is a normal value, its bf16 rounding."""
    hidden, dim = 65536, 128
    values = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    values[values == 0] = 0.0
    x = torch.zeros(256, 1, dim, dtype=torch.bfloat16)
    x[..., 0] = 1.0
    w13 = torch.zeros(2 * hidden, dim, dtype=torch.bfloat16)
    w13[:hidden, 0] = values
    w13[hidden:, 0] = 1.0
    got = fused.swiglu_linear_w13(x.to(DEV), w13.to(DEV))[[0, 255], 0].cpu()
    h = torch.cat([values, torch.ones_like(values)]).to(DEV).expand(2, 1, -1).contiguous()
    want = fused.swiglu(h)[:, 0].cpu()
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])
    a = values.double()
    exact = a / (1 + torch.exp(-a))
    normal = exact.isfinite() & (exact.abs() >= 2.0 ** -126) & (a > -88.7)   # below, expf overflows: -0
    assert normal.sum() > 64000 // 2 and torch.equal(got[:, normal], exact[normal].to(torch.bfloat16).expand(2, -1))
