"""Cases of the framework's main paths, timed and compared through its public entry points.

Each case is one call (or one training step, or one model forward) as a program makes it:

* ``op``: ``mosaic_attn_func``, the three-branch block-sparse attention forward;
* ``rope_op``: ``mosaic_attn_func_rope``, the same op with RoPE fused, as the model calls it;
* ``train``: ``mosaic_sparse_attn`` forward and backward through autograd;
* ``interp``: ``knn_attention``, the grid interpolation's gather-attention, as the module calls it;
* ``ffn``: ``cSwiGLU`` and ``block``: ``MosaicBlock``, single layers under bf16 autocast;
* ``unet``: one forecast step of the era5 preset.

Sizes are those of the bench workloads and the shipped model: HEALPix nside 16 / 32 / 64
sequences (3072, 12288, 49152 tokens), 20/5, 16/4 and 12/3 heads, 1 to 24 ensemble members, the
op's 64-token blocks and the model's 1024 / 128-token blocks.  ``draw`` spreads over the same
ranges (any number of blocks and members between, other head groupings, the op's other modes).

``exact`` evaluates the same formulas in float64.  Top-k selection is discontinuous, so there
the selection scores of the ``op`` kinds keep the path's bf16 values (pooled means, scores and
head means rounded to bf16); everything else is unrounded.
"""

from __future__ import annotations

import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

import mosaic_amd as M
from mosaic_amd import fused
from mosaic_amd.healpix import get_healpix_grid, rope_tables
from mosaic_amd.interp import get_neighbors, knn_attention, knn_tiles, rad_to_xyz, spatial_order
from mosaic_amd.model import MosaicBlock, Transformer, cSwiGLU, era5_config, model_flops

DEV = "cuda"
BF16 = torch.bfloat16


def _op(name, kind, seq, batch, hq, hk, bl, bs, top, mode="full"):
    return dict(name=name, kind=kind, seq=seq, batch=batch, hq=hq, hk=hk, bl=bl, bs=bs, top=top, mode=mode)


def listed():
    return [
        # the bottleneck's attention at one member: the smallest call, where launches and host work count
        _op("op_nside16_b1", "op", 3072, 1, 20, 5, 64, 64, 4),
        # a mid-size single-member call: too few query tiles to fill the chip evenly
        _op("op_nside32_b1", "op", 12288, 1, 12, 3, 64, 64, 16),
        # the headline workload of the benchmark
        _op("op_nside64_b1", "op", 49152, 1, 12, 3, 64, 64, 16),
        # the ensemble: 24 members at stage 2
        _op("op_nside32_b24", "op", 12288, 24, 16, 4, 64, 64, 16),
        # the shipped model's stage-1 attention for one member, RoPE included
        _op("rope_model_nside64_b1", "rope_op", 49152, 1, 12, 3, 1024, 128, 24),
        # training the selected branch at stage 1 (blocks of 64) and at stage 2 with the model's blocks
        _op("train_nside64_b1", "train", 49152, 1, 12, 3, 64, 64, 16),
        _op("train_nside32_b1", "train", 12288, 1, 16, 4, 128, 128, 12),
        # the model's two grid interpolations: 24 members in, one member out
        dict(name="interp_to_hp_b24", kind="interp", nlon=240, nlat=121, nside=64, to_hp=True, batch=24, heads=12, k=24),
        dict(name="interp_to_ll_b1", kind="interp", nlon=240, nlat=121, nside=64, to_hp=False, batch=1, heads=12, k=24),
        # the widest feed-forward layer of the ensemble forecast
        dict(name="ffn_nside64_b24", kind="ffn", seq=49152, batch=24, dim=768, hidden=3072),
        # a whole stage-2 transformer block at a few members
        dict(name="block_nside32_b3", kind="block", nside=32, batch=3, dim=1024, heads=16, bl=1024, bs=128, top=12),
        # one forecast step of a single member
        dict(name="unet_b1", kind="unet", members=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_heads(rng):
    group = rng.choice((4, 4, 4, 2, 1))
    hk = rng.randint(2, 5)
    return hk * group, hk


def draw(rng):
    kind = rng.choice(("op", "op", "op", "rope_op", "rope_op", "train", "train", "interp", "ffn", "block"))
    if kind in ("op", "rope_op", "train"):
        hq, hk = _draw_heads(rng)
        bl, bs = rng.choice(((64, 64), (64, 64), (1024, 128), (256, 64)))
        if kind == "train":
            bl = bs
        unit = max(bl, bs)
        seq = unit * max(1, round(_log_int(rng, 3072, 49152) / unit))
        top = min(rng.randint(4, 24 if bs == 128 else 16), seq // bs)
        # at most the listed ensemble call's tokens x query heads, and its work (a training step's is several times a call's)
        work = seq * hq * (bl + top * bs) * (5 if kind == "train" else 1)
        most = min(24.0, 24 * 12288 * 16 / (seq * hq), 24 * 12288 * 16 * 1088 / work)
        batch = _log_int(rng, 1, max(1.0, most))
        mode = rng.choice(("full", "full", "full", "no_compression", "no_selection", "local")) if kind != "train" else "full"
        c = _op("", kind, seq, batch, hq, hk, bl, bs, 0 if mode == "no_selection" else top, mode)
        del c["name"]
        return c
    if kind == "interp":
        nlat = rng.choice((61, 91, 121))
        return dict(kind="interp", nlon=2 * (nlat - 1), nlat=nlat, nside=rng.choice((32, 64)), to_hp=rng.random() < 0.5,
                    batch=_log_int(rng, 1, 24), heads=rng.choice((4, 8, 12)), k=rng.randint(8, 24))
    dim, heads, nside, top = rng.choice(((768, 12, 64, 24), (1024, 16, 32, 12), (1280, 20, 16, 4)))
    if kind == "ffn":
        seq = rng.choice((12 * nside * nside, _log_int(rng, 192, 49152)))
        return dict(kind="ffn", seq=seq, batch=_log_int(rng, 1, min(24.0, 24 * 49152 * 768 / (seq * dim))), dim=dim, hidden=4 * dim)
    return dict(kind="block", nside=nside, batch=_log_int(rng, 1, 8), dim=dim, heads=heads, bl=1024, bs=128, top=top)


# ------------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 + 7919 * int(seed))


def _randn(gen, *shape, dtype=BF16, scale=1.0):
    x = torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32)
    return (x * scale if scale != 1.0 else x).to(dtype)


@functools.lru_cache(maxsize=4)
def _rope(seq):
    """RoPE tables of ``seq`` positions: the HEALPix pixel centres where seq is 12 nside^2, else the
    first pixels of the next finer grid."""
    nside = 1
    while 12 * nside * nside < seq:
        nside *= 2
    return tuple(t.to(DEV) for t in rope_tables(get_healpix_grid(nside)[:seq], 64))


def _rotate(x, cos, sin):
    c, s = cos[None, :, None].to(x.dtype), sin[None, :, None].to(x.dtype)
    out = torch.empty_like(x)
    out[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    out[..., 1::2] = x[..., 1::2] * c + x[..., 0::2] * s
    return out


def _qkv(case, gen):
    B, N = case["batch"], case["seq"]
    return [_randn(gen, B, N, h, 64) for h in (case["hq"], case["hk"], case["hk"])]


def _selection(case, gen):
    """Blocks as the model selects them: half around the query block, half anywhere, each once."""
    B, nb, Hk, K = case["batch"], case["seq"] // case["bs"], case["hk"], case["top"]
    near = (torch.arange(nb, device=DEV)[:, None] - torch.arange(nb, device=DEV)[None, :]).abs() * 2 < K
    score = torch.rand(B, nb, Hk, nb, generator=gen, device=DEV) + near[None, :, None, :].float()
    return score.topk(K, dim=-1).indices.contiguous()


@functools.lru_cache(maxsize=8)
def _grids(nlon, nlat, nside, to_hp, k):
    """The neighbour lists, target order and target tiles of a grid pair: a program builds them once."""
    lon, lat = torch.linspace(0, 360 - 360 / nlon, nlon), torch.linspace(-90, 90, nlat)
    ll = torch.deg2rad(torch.stack(torch.meshgrid(lon, lat, indexing="ij"), -1).reshape(-1, 2))
    hp = torch.deg2rad(get_healpix_grid(nside))
    src, dst = (ll, hp) if to_hp else (hp, ll)
    nb = torch.from_numpy(np.ascontiguousarray(get_neighbors(src.numpy(), dst.numpy(), k=k))).long()
    rel = torch.nn.functional.normalize(rad_to_xyz(dst).unsqueeze(1) - rad_to_xyz(src)[nb], dim=-1)
    order = spatial_order(dst)
    tiles = {n: (t.to(DEV) if torch.is_tensor(t) else t) for n, t in knn_tiles(nb, order).items()}
    return len(src), nb.to(DEV), rel.to(DEV), order.to(DEV, torch.int32), tiles


def _init(module, gen):
    """N(0, 1 / fan_in) weights: activations keep their scale through the layer."""
    with torch.no_grad():
        for p in module.parameters():
            if p.dim() == 2:
                p.copy_(_randn(gen, *p.shape, dtype=torch.float32, scale=p.shape[1] ** -0.5))
    return module.eval()


def _block_config(case):
    return SimpleNamespace(dim=case["dim"], num_heads=case["heads"], block_attn_size=case["bl"],
                           sparse_block_size=case["bs"], sparse_block_count=case["top"], gqa_ratio=4,
                           qkv_compress_ratio=1, rope=True, rope_theta=10000, mlp_ratio=4.0, noise_dim=32,
                           rmsnorm_elementwise_affine=False)


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("op", "rope_op"):
        q, k, v = _qkv(case, gen)
        if kind == "op":
            cos, sin = _rope(case["seq"])
            q, k = (_rotate(t.float(), cos, sin).to(BF16) for t in (q, k))
        else:
            s["cos"], s["sin"] = _rope(case["seq"])
        logits = _randn(gen, 3, case["batch"], case["seq"], case["hq"], 1, dtype=torch.float32)
        # sigmoid gates as in the benchmark; the model's are a softmax over the branches
        w = (torch.sigmoid(logits) if kind == "op" else torch.softmax(logits, dim=0)).to(BF16)
        s.update(q=q, k=k, v=v, w=w)
    elif kind == "train":
        q, k, v = (t.requires_grad_() for t in _qkv(case, gen))
        s.update(q=q, k=k, v=v, idx=_selection(case, gen), go=_randn(gen, case["batch"], case["seq"], case["hq"], 64))
    elif kind == "interp":
        n_src, nb, rel, order, tiles = _grids(case["nlon"], case["nlat"], case["nside"], case["to_hp"], case["k"])
        H = case["heads"]
        kv = _randn(gen, n_src, case["batch"], 2 * H * 64)   # the kv projection's output
        s.update(k=kv[..., :H * 64].unflatten(-1, (H, 64)), v=kv[..., H * 64:].unflatten(-1, (H, 64)), nb=nb, rel=rel,
                 order=order, tiles=tiles, wq=_randn(gen, H * 64, 3))
    elif kind == "ffn":
        s["m"] = _init(cSwiGLU(case["dim"], case["hidden"], 32).to(DEV), gen)
        s["x"] = _randn(gen, case["seq"], case["batch"], case["dim"])
        s["z"] = _randn(gen, case["batch"], 32, dtype=torch.float32)
    elif kind == "block":
        m = MosaicBlock(_block_config(case), block_attn_only=False)
        grid = get_healpix_grid(case["nside"])
        for r in (m.attention.q_rope, m.attention.k_rope):
            r.initialize_rope(grid)
        s["m"] = _init(m.to(DEV), gen)
        s["x"] = _randn(gen, 12 * case["nside"] ** 2, case["batch"], case["dim"])
        s["z"] = _randn(gen, case["batch"], 32, dtype=torch.float32)
    else:
        torch.manual_seed(int(seed))
        m = Transformer(era5_config(), seed=int(seed))
        lon, lat = torch.linspace(0, 358.5, 240), torch.linspace(-90, 90, 121)
        m.initialize_interpolation(lon, lat)
        m = m.to(DEV)
        m.initialize_static_vars(_randn(gen, 240, 121, 3, dtype=torch.float32), lon.to(DEV), lat.to(DEV))
        s["m"] = m.eval()
        s["x"] = _randn(gen, 1, 1, 2, 240, 121, 82, dtype=torch.float32)
        s["dyt"] = torch.rand(1, 1, 2, generator=gen, device=DEV)
    return s


# ------------------------------------------------------------------------------------ one pass

def _flags(case):
    return dict(block_attn_only=case["mode"] == "local", no_compression=case["mode"] == "no_compression")


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "op":
        return M.mosaic_attn_func(s["q"], s["k"], s["v"], s["w"], case["bl"], case["bs"], case["top"], **_flags(case))
    if kind == "rope_op":
        return M.mosaic_attn_func_rope(s["q"], s["k"], s["v"], s["w"], s["cos"], s["sin"], case["bl"], case["bs"],
                                       case["top"], **_flags(case))
    if kind == "train":
        s["q"].grad = s["k"].grad = s["v"].grad = None
        out = M.mosaic_sparse_attn(s["q"], s["k"], s["v"], s["idx"], case["bs"])
        out.backward(s["go"])
        return out.detach(), s["q"].grad, s["k"].grad, s["v"].grad
    if kind == "interp":
        return knn_attention(s["k"], s["v"], s["nb"], s["rel"], s["wq"], 0.125, s["order"], tiles=s["tiles"])
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
        if kind == "unet":
            s["m"].noise_generator.generator = None      # every step draws the same member noise
            return s["m"](s["x"], s["dyt"], case["members"])
        return s["m"](s["x"], s["z"])


# ------------------------------------------------------------------------------------ work

def _attn_flops(B, N, Hq, bl, bs, K, mode):
    nb = N // bs
    f = 0 if mode == "selected" else N * bl
    if mode in ("full", "no_compression", "selected"):
        f += N * K * bs
    if mode in ("full", "no_selection"):
        f += nb * nb
    f *= 4 * B * Hq * 64
    return f + (2 * B * Hq * 64 * nb * nb if mode in ("full", "no_compression") else 0)


def work(case):
    kind = case["kind"]
    if kind in ("op", "rope_op", "train"):
        B, N, Hq, Hk, K = (case[n] for n in ("batch", "seq", "hq", "hk", "top"))
        qo, kv = 2 * B * N * Hq * 64, 2 * B * N * Hk * 64
        if kind == "train":
            # q, k, v, grad of out and the indices in; out and three gradients out; the forward's
            # two products and the backward's five (S and dP once)
            f = B * Hq * N * K * case["bs"] * 64 * 2 * 7
            return dict(bytes=4 * qo + 4 * kv + 8 * B * (N // case["bs"]) * Hk * K, flops=f)
        gates = 0 if case["mode"] == "local" else 2 * 3 * B * N * Hq
        return dict(bytes=2 * qo + 2 * kv + gates + (256 * N if kind == "rope_op" else 0),
                    flops=_attn_flops(B, N, Hq, case["bl"], case["bs"], K, case["mode"]))
    if kind == "interp":
        hp, ll = 12 * case["nside"] ** 2, case["nlon"] * case["nlat"]
        n_from, n_to = (ll, hp) if case["to_hp"] else (hp, ll)
        row = 2 * case["batch"] * case["heads"] * 64
        return dict(bytes=2 * n_from * row + n_to * row + n_to * case["k"] * 16,
                    flops=4 * n_to * case["batch"] * case["heads"] * 64 * case["k"])
    if kind == "ffn":
        rows, D, H = case["seq"] * case["batch"], case["dim"], case["hidden"]
        return dict(bytes=2 * 2 * rows * D + 4 * 3 * D * H, flops=2 * rows * 3 * D * H)
    if kind == "block":
        N, B, D, Hq = 12 * case["nside"] ** 2, case["batch"], case["dim"], case["heads"]
        Hk = Hq // 4
        params = D * 64 * (2 * Hq + 2 * Hk) + D * 3 * Hq + 3 * D * 4 * D
        return dict(bytes=2 * 2 * N * B * D + 4 * params,
                    flops=2 * N * B * params + _attn_flops(B, N, Hq, case["bl"], case["bs"], case["top"], "full"))
    n_ll = 240 * 121
    return dict(bytes=4 * 214184448 + 4 * n_ll * (2 + case["members"]) * 82,
                flops=model_flops(era5_config(), case["members"], n_ll)["total"])


def tolerance(case):
    """Four times what the path measures against its own formulas in float64 (bf16 operands and
    probabilities, fp32 sums).  A block swapped in an exact tie of bf16 scores moves single rows
    by up to their own size, hence the wide largest difference where blocks are selected."""
    rel = {"op": 1.1e-2, "rope_op": 1.1e-2, "train": 1.3e-2, "interp": 1.7e-2, "ffn": 2.1e-2, "block": 2e-2,
           "unet": 3e-2}[case["kind"]]
    return dict(rel=rel, max=0.99 if case["kind"] in ("op", "rope_op", "block", "unet") else 0.4)


# ------------------------------------------------------------------------------------ float64

def _pool(x, bs):
    B, N, H, d = x.shape
    return x.view(B, N // bs, bs, H, d).mean(2)


def _softmax_pv(q, k, v):
    """softmax(q k^T / 8) v over the last two dimensions, batched, in float64."""
    p = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) * 0.125, dim=-1)
    return torch.matmul(p, v)


def _local64(q, k, v, bl):
    B, N, Hq, _ = q.shape
    Hk, out = k.shape[2], torch.empty_like(q)
    G = Hq // Hk
    for b in range(B):
        for c in range(Hk):
            kk, vv = (t[b, :, c].reshape(N // bl, bl, 64) for t in (k, v))
            for j in range(c * G, (c + 1) * G):
                out[b, :, j] = _softmax_pv(q[b, :, j].reshape(N // bl, bl, 64), kk, vv).reshape(N, 64)
    return out


def _selected64(q, k, v, idx, bs, lse=None):
    B, N, Hq, _ = q.shape
    Hk, nb, out = k.shape[2], N // bs, torch.empty_like(q)
    G = Hq // Hk
    for b in range(B):
        for c in range(Hk):
            kk, vv = (t[b, :, c].reshape(nb, bs, 64)[idx[b, :, c]].reshape(nb, -1, 64) for t in (k, v))
            for j in range(c * G, (c + 1) * G):
                out[b, :, j] = _softmax_pv(q[b, :, j].reshape(nb, bs, 64), kk, vv).reshape(N, 64)
    return out


def _select64(qc, kc, K, rounded):
    """Top-K blocks [B, nb, Hk, K]: the mean over heads g Hk + h of the scores of row h, ties to the
    lower block; with ``rounded`` the pooled values, the scores and their means are bf16."""
    r = (lambda x: x.to(BF16).double()) if rounded else (lambda x: x)
    B, nb, Hq, _ = qc.shape
    Hk = kc.shape[2]
    G = Hq // Hk
    qc, kc = r(qc), r(kc)
    rows = []
    for h in range(Hk):
        total = 0
        for g in range(G):
            j = g * Hk + h
            total = total + r(torch.matmul(qc[:, :, j], kc[:, :, j // G].transpose(-1, -2).contiguous()))
        rows.append(torch.sort(r(total / G), dim=-1, descending=True, stable=True).indices[..., :K])
    return torch.stack(rows, 2)


def _attention64(q, k, v, w, bl, bs, K, mode, rounded):
    """The op in float64 ([B, N, H, 64]; w [3, B, N, Hq, 1])."""
    o = _local64(q, k, v, bl)
    if mode == "local":
        return o
    o = o * w[0]
    qc, kc = _pool(q, bs), _pool(k, bs)
    if mode in ("full", "no_selection"):
        vc, G = _pool(v, bs), q.shape[2] // k.shape[2]
        oc = torch.stack([_softmax_pv(qc[:, :, j], kc[:, :, j // G], vc[:, :, j // G]) for j in range(q.shape[2])], 2)
        o += oc.repeat_interleave(bs, 1) * w[1]
    if mode in ("full", "no_compression"):
        o += _selected64(q, k, v, _select64(qc, kc, K, rounded), bs) * w[2]
    if mode == "no_compression":
        o /= w[0] + w[2] + 1e-8
    if mode == "no_selection":
        o /= w[0] + w[1] + 1e-8
    return o


def _train64(q, k, v, idx, go, bs):
    """Output and gradients of the selected branch, head by head."""
    B, N, Hq, _ = q.shape
    Hk, nb = k.shape[2], N // bs
    G = Hq // Hk
    out, gq, gk, gv = torch.empty_like(q), torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for c in range(Hk):
            sel = idx[b, :, c]
            kk, vv = (t[b, :, c].reshape(nb, bs, 64)[sel].reshape(nb, -1, 64) for t in (k, v))
            for j in range(c * G, (c + 1) * G):
                qq, dd = (t[b, :, j].reshape(nb, bs, 64) for t in (q, go))
                p = torch.softmax(torch.matmul(qq, kk.transpose(-1, -2).contiguous()) * 0.125, dim=-1)
                o = torch.matmul(p, vv)
                ds = torch.matmul(dd, vv.transpose(-1, -2).contiguous())
                ds = (ds - (o * dd).sum(-1, keepdim=True)) * p * 0.125
                out[b, :, j], gq[b, :, j] = o.reshape(N, 64), torch.matmul(ds, kk).reshape(N, 64)
                for dst, m, x in ((gk, ds, qq), (gv, p, dd)):
                    part = torch.matmul(m.transpose(-1, -2).contiguous(), x).reshape(-1, bs, 64)
                    acc = torch.zeros(nb, bs, 64, dtype=torch.float64, device=q.device)
                    dst[b, :, c] += acc.index_add_(0, sel.reshape(-1), part).reshape(N, 64)
    return out, gq, gk, gv


def _interp64(k, v, nb, rel, wq, scale):
    """[S_to, B, H, 64] in float64, targets in chunks."""
    H = k.shape[2]
    out = torch.empty(nb.shape[0], *k.shape[1:], dtype=torch.float64, device=k.device)
    q = (rel.double() @ wq.double().t()).unflatten(-1, (H, 64))          # [S_to, K, H, 64]
    step = max(1, 300_000_000 // (nb.shape[1] * k.shape[1] * H * 64))
    for a in range(0, nb.shape[0], step):
        n = nb[a:a + step]
        score = (q[a:a + step].unsqueeze(2) * k[n].double()).sum(-1) * scale    # [t, K, B, H]
        out[a:a + step] = (torch.softmax(score, dim=1).unsqueeze(-1) * v[n].double()).sum(1)
    return out


def _lin(m, x):
    return x @ m.weight.double().t()


def _norm64(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + fused.DEFAULT_EPS)


def _ffn64(m, x, z):
    """cSwiGLU on [S, B, dim], rows in chunks."""
    noise = _lin(m.noise_bias, z.double()) if z is not None else 0.0
    out = torch.empty(*x.shape, dtype=torch.float64, device=x.device)
    step = max(1, 200_000_000 // (x.shape[1] * m.w2.in_features))
    for a in range(0, x.shape[0], step):
        x1, x3 = _lin(m.w13, x[a:a + step].double()).chunk(2, -1)
        out[a:a + step] = _lin(m.w2, torch.nn.functional.silu(x1 + noise) * x3)
    return out


def _layer64(m, x):
    """MosaicAttention on [S, B, dim]."""
    def heads(lin, H):
        return _lin(lin, x).unflatten(-1, (H, 64)).transpose(0, 1).contiguous()
    q, k, v = heads(m.to_q, m.q_heads), heads(m.to_k, m.kv_heads), heads(m.to_v, m.kv_heads)
    q, k = _rotate(q, m.q_rope.cos_freqs, m.q_rope.sin_freqs), _rotate(k, m.k_rope.cos_freqs, m.k_rope.sin_freqs)
    w = torch.softmax(_lin(m.to_strategy_combine_mlp, x).unflatten(-1, (m.q_heads, 3)), -1).permute(3, 1, 0, 2).unsqueeze(-1)
    o = _attention64(q, k, v, w, m.block_attn_size, m.sparse_block_size, m.sparse_block_count, "full", False)
    return _lin(m.to_o, o.transpose(0, 1).flatten(2))


def _block64(m, x, z):
    x = x + _layer64(m.attention, _norm64(x))
    return x + _ffn64(m.ffn, _norm64(x), z)


def _cross64(m, x):
    kv = _lin(m.to_kv, _norm64(x))
    k, v = (t.unflatten(-1, (m.num_heads, 64)) for t in kv.chunk(2, -1))
    return _lin(m.to_o, _interp64(k, v, m.neighbors, m.rel_pos, m.to_q.weight, m.scale).flatten(2))


def _unet64(m, x, dyt, members, seed):
    b, n, t, lon, lat, c = x.shape
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    z = _lin(m.noise_generator.to_noise, torch.randn(members, 32, generator=gen, device=DEV).double())
    xs = x.double().permute(3, 4, 0, 1, 2, 5).reshape(lon * lat, 1, t * c).expand(-1, members, -1)
    day, year = (2 * math.pi * dyt.double().reshape(-1)).tolist()
    time = torch.tensor([math.sin(day), math.cos(day), math.sin(year), math.cos(year)], dtype=torch.float64, device=DEV)
    h = torch.cat([xs, m.static_vars.double().expand(-1, members, -1), time.expand(lon * lat, members, 4)], -1)
    h = _norm64(_lin(m.preprocess[3], torch.nn.functional.silu(_norm64(_lin(m.preprocess[0], h)))))
    h = _cross64(m.interp_to_hp, h)
    skips = []
    for stage, down in zip(m.encoder_stages, m.downsample_layers):
        for blk in stage.blocks:
            h = _block64(blk, h, z)
        skips.append(h)
        h = h.unflatten(0, (-1, down.factor)).transpose(1, 2).flatten(2)
        h = _norm64(_lin(down.proj_x, h) + _lin(down.proj_pos, down.rel_pos.double()).unsqueeze(1))
    for blk in m.bottleneck.blocks:
        h = _block64(blk, h, z)
    for stage, up, skip in zip(m.decoder_stages, m.upsample_layers, reversed(skips)):
        h = _lin(up.proj_x, h) + _lin(up.proj_pos, up.rel_pos.double()).unsqueeze(1)
        h = h.unflatten(-1, (up.factor, -1)).permute(0, 2, 1, 3).flatten(0, 1)
        h = _norm64(h + skip)
        for blk in stage.blocks:
            h = _block64(blk, h, z)
    h = _norm64(_cross64(m.interp_to_ll, _norm64(h)))
    h = _lin(m.postprocess[3], torch.nn.functional.silu(_lin(m.postprocess[1], h)))
    return h.view(lon, lat, 1, members, -1).permute(2, 3, 0, 1, 4)


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("op", "rope_op"):
        q, k, v, w = (s[n].double() for n in ("q", "k", "v", "w"))
        if kind == "rope_op":
            q, k = (_rotate(t, s["cos"], s["sin"]) for t in (q, k))
            # the path's rotated q and k are bf16, and the selection follows them
            q, k = q.to(BF16).double(), k.to(BF16).double()
        return _attention64(q, k, v, w, case["bl"], case["bs"], case["top"], case["mode"], True)
    if kind == "train":
        q, k, v, go = (s[n].detach().double() for n in ("q", "k", "v", "go"))
        return _train64(q, k, v, s["idx"], go, case["bs"])
    if kind == "interp":
        return _interp64(s["k"], s["v"], s["nb"], s["rel"], s["wq"], 0.125)
    if kind == "unet":
        return _unet64(s["m"], s["x"], s["dyt"], case["members"], seed)
    if kind == "ffn":
        return _ffn64(s["m"], s["x"], s["z"])
    return _block64(s["m"], s["x"].double(), s["z"].double())
