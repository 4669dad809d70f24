// pool.hip -- mean pooling of q, k, v over runs of sparse_block_size tokens (gfx950).
//
// Replaces reduce(x, 'b (nb bs) h d -> b nb h d', 'mean') (primitives.py:65-66,76): fp32
// sum over the block's tokens in token order, divided by the block size, rounded to bf16.
// The workgroups of (pooled block t, batch b), one or a few that share its columns, read the
// block's q, k and v rows once (HBM-bound).  TPC adjacent threads share one 16-byte column chunk
// of a row: each streams it down its own contiguous run of the block's tokens, summing in token
// order, and the partial sums are added pairwise through DPP.  More threads per chunk shorten
// the serial walk and put more loads in flight where the grid alone leaves the chip idle
// (pool_shape).
// Outputs: [B, nb, H, 64] for the pooled tensors and, for k and v, the MFMA-operand-ordered
// layouts read by the compressed-attention kernel (kfrag_index / vfrag_index; zero for the
// padding blocks nb .. nb_pad-1).
// Optionally, for the keys (tensor 1), the largest squared norm of each 8-dim chunk over the
// block's tokens: the sum of a head's 8 values bounds |k|^2 for every key of the block, which
// the attention kernel uses to bound its logits.
// Optionally, q and k (tensors 0 and 1) are first rotated by the 2-D RoPE of the tokens'
// positions (primitives.py:125-135: x * cos + rotate_half(x) * sin in fp32, back to bf16):
// pair m = (2m, 2m+1) of a head becomes (x0 c_m - x1 s_m, x1 c_m + x0 s_m), each product and
// the sum rounded as the reference rounds them.  The rotated rows are written out (the
// attention reads them) and pooled, so the rotation costs no extra read of q and k.
#include <algorithm>

#include "bsa_common.h"

namespace mosaic {
namespace {

// a[which] for which in 0..2 through selects, so a per-thread choice of tensor does not index
// the kernel's parameter block at run time (which would read it from memory)
template <typename T>
__device__ __forceinline__ T sel3(const T (&a)[3], int which) {
    return which == 0 ? a[0] : (which == 1 ? a[1] : a[2]);
}

// x of lane l ^ 1 (quad_perm [1, 0, 3, 2]), of lane l ^ 2 (quad_perm [2, 3, 0, 1]) and of the
// mirror lane in the group of eight (row_half_mirror)
template <int STEP>
__device__ __forceinline__ float other_lane(float x) {
    constexpr int kCtrl = STEP == 1 ? 0xb1 : STEP == 2 ? 0x4e : 0x141;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, false));
}
// Sum (maximum) over the TPC lanes of a chunk, the same value in all of them: at each step the
// lanes of a half all hold that half's value, so the mirror lane is as good as l ^ 4.
// Addition is commutative, so both halves round alike.
template <int TPC>
__device__ __forceinline__ float chunk_add(float x) {
    if constexpr (TPC > 1) x += other_lane<1>(x);
    if constexpr (TPC > 2) x += other_lane<2>(x);
    if constexpr (TPC > 4) x += other_lane<4>(x);
    return x;
}
template <int TPC>
__device__ __forceinline__ float chunk_max(float x) {
    if constexpr (TPC > 1) x = fmaxf(x, other_lane<1>(x));
    if constexpr (TPC > 2) x = fmaxf(x, other_lane<2>(x));
    if constexpr (TPC > 4) x = fmaxf(x, other_lane<4>(x));
    return x;
}

// ROPE: 0 no rotation; 1 rotation with the block's table rows staged in LDS; 2 rotation with
// the table rows read from global memory (blocks too large for the LDS staging).  Separate
// instantiations keep the LDS reads ds_read instructions (a runtime choice between the two
// address spaces compiled to generic loads).
template <int ROPE>
constexpr int kPoolMaxThreads = ROPE == 2 ? 512 : 1024;  // the global-table variant needs more registers

template <int ROPE, int TPC>
__global__ __launch_bounds__(kPoolMaxThreads<ROPE>) void pool_kernel(PoolParams p) {
    const int t = blockIdx.x, b = blockIdx.y;
    // RoPE tables of the block's tokens, read once per workgroup: [token][8 float4] of cos,
    // then of sin (every head of a token uses the same row)
    extern __shared__ float4 rope_rows[];
    if (ROPE == 1 && t < p.nb) {
        const float4* c4 = reinterpret_cast<const float4*>(p.rope_cos) + (int64_t)t * p.bs * 8;
        const float4* s4 = reinterpret_cast<const float4*>(p.rope_sin) + (int64_t)t * p.bs * 8;
        for (int i = threadIdx.x; i < 16 * p.bs; i += blockDim.x)
            rope_rows[i] = i < 8 * p.bs ? c4[i] : s4[i - 8 * p.bs];
        __syncthreads();
    }
    const int c0 = p.heads[0] * 8, c1 = p.heads[1] * 8, c2 = p.heads[2] * 8;
    const int ctot = c0 + c1 + c2;
    // whole waves (blockDim.x is a multiple of 64): the threads of a chunk are adjacent lanes of
    // one iteration
    for (int item = threadIdx.x + blockIdx.z * blockDim.x; item < TPC * ctot; item += blockDim.x * gridDim.z) {
        const int col = item / TPC, part = item % TPC;
        const int which = col < c0 ? 0 : (col < c0 + c1 ? 1 : 2);
        const int cc = col - (which == 0 ? 0 : (which == 1 ? c0 : c0 + c1));
        const int hd = cc >> 3, ch = cc & 7;
        // this thread's tensor, selected once (no runtime indexing of the parameter block)
        const int heads = sel3(p.heads, which);
        bf16_t* frag = which == 1 ? p.kfrag : (which == 2 ? p.vfrag : nullptr);
        // operand-ordered output of this thread's 8 dims of block t (zero past nb)
        auto store_frag = [&](const float (&x)[8]) {
            const int UT = p.nb_pad >> 5, ut = t >> 5, w = t & 31;
            if (which == 1) {
                uint4 u;
                u.x = pack_bf16x2(x[0], x[1]); u.y = pack_bf16x2(x[2], x[3]);
                u.z = pack_bf16x2(x[4], x[5]); u.w = pack_bf16x2(x[6], x[7]);
                *reinterpret_cast<uint4*>(frag + kfrag_index(b, hd, heads, UT, ut, ch >> 1, 32 * (ch & 1) + w)) = u;
            } else {
                const int s2 = w >> 4, rem = w & 15, slot = 4 * (rem >> 3) + (rem & 3), hh = (rem & 7) >> 2;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int d = 8 * ch + e;
                    frag[vfrag_index(b, hd, heads, UT, ut, d >> 5, s2, 32 * hh + (d & 31)) + slot] =
                        (bf16_t)(pack_bf16x2(x[e], 0.f) & 0xffffu);
                }
            }
        };
        if (t >= p.nb) {  // padding blocks of the operand-ordered outputs
            if (frag && part == 0) {
                const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                store_frag(zero);
            }
            continue;
        }
        // tokens n0 .. n1-1 of the block: this thread's run
        const int n0 = part * p.bs / TPC, n1 = (part + 1) * p.bs / TPC;
        const int64_t sn = sel3(p.sn, which);
        const int64_t tok0 = (int64_t)t * p.bs + n0;
        const bf16_t* src = sel3(p.x, which) + b * sel3(p.sb, which) + tok0 * sn + (int64_t)hd * sel3(p.sh, which) + ch * 8;
        // RoPE of this thread's 4 pairs (frequencies 4 ch .. 4 ch + 3): table rows of token n0 + i
        const bool rope = ROPE != 0 && which < 2;
        bf16_t* rot = which == 0 ? p.rot[0] : (which == 1 ? p.rot[1] : nullptr);
        bf16_t* rdst = rope && rot != nullptr
                           ? rot + (((int64_t)b * p.nb * p.bs + tok0) * heads + hd) * kHeadDim + ch * 8
                           : nullptr;
        const int64_t rstride = (int64_t)heads * kHeadDim;
        const float4* ctab = ROPE == 1 ? rope_rows + n0 * 8 + ch
                                       : reinterpret_cast<const float4*>(p.rope_cos + tok0 * 32 + 4 * ch);
        const float4* stab = ROPE == 1 ? rope_rows + 8 * p.bs + n0 * 8 + ch
                                       : reinterpret_cast<const float4*>(p.rope_sin + tok0 * 32 + 4 * ch);
        auto rotate = [&](uint4 v, int i) __attribute__((always_inline)) -> uint4 {
            const float4 c = ctab[8 * i], s = stab[8 * i];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
            const float cf[4] = {c.x, c.y, c.z, c.w}, sf[4] = {s.x, s.y, s.z, s.w};
            uint32_t o[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = rope_pair(w[k], cf[k], sf[k]);
            return make_uint4(o[0], o[1], o[2], o[3]);
        };
        float acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = 0.f;
        float sqmax = 0.f;  // largest squared norm of this 8-dim chunk over the block's tokens
        auto add_token = [&](uint4 v) __attribute__((always_inline)) {
            const float x[8] = {bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y),
                                bf_lo(v.z), bf_hi(v.z), bf_lo(v.w), bf_hi(v.w)};
            float sq = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                acc[e] += x[e];
                sq = fmaf(x[e], x[e], sq);
            }
            sqmax = fmaxf(sqmax, sq);
        };
        const int count = n1 - n0;
        int i = 0;
        for (; i + 8 <= count; i += 8) {  // eight tokens' loads in flight, summed in token order
            uint4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = ld16(src + (int64_t)u * sn);
            src += 8 * sn;
            if (rope) {
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = rotate(v[u], i + u);
                if (rdst) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) *reinterpret_cast<uint4*>(rdst + (int64_t)u * rstride) = v[u];
                    rdst += 8 * rstride;
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) add_token(v[u]);
        }
        for (; i < count; ++i) {
            uint4 v = ld16(src);
            src += sn;
            if (rope) {
                v = rotate(v, i);
                if (rdst) {
                    *reinterpret_cast<uint4*>(rdst) = v;
                    rdst += rstride;
                }
            }
            add_token(v);
        }
        // the block's sum and maximum in every thread of the chunk (an empty run adds 0)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = chunk_add<TPC>(acc[e]);
        sqmax = chunk_max<TPC>(sqmax);
        if (which == 1 && p.kbnd != nullptr && part == 0)
            p.kbnd[(((int64_t)b * p.nb + t) * heads + hd) * 8 + ch] = sqmax;
        const float denom = (float)p.bs;
        float mean[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) mean[e] = acc[e] / denom;
        bf16_t* out = sel3(p.out_bnhd, which);
        if (out && part == 0) {
            uint4 w;
            w.x = pack_bf16x2(mean[0], mean[1]);
            w.y = pack_bf16x2(mean[2], mean[3]);
            w.z = pack_bf16x2(mean[4], mean[5]);
            w.w = pack_bf16x2(mean[6], mean[7]);
            *reinterpret_cast<uint4*>(out + (((int64_t)b * p.nb + t) * heads + hd) * kHeadDim + ch * 8) = w;
        }
        if (frag && part == TPC - 1) store_frag(mean);  // every part holds the mean
    }
}

// Threads per column chunk and per workgroup (0: one workgroup for all columns of a block).
// One thread per chunk (two with RoPE, whose rotation doubles the arithmetic) is the fastest
// while the blocks alone keep the chip busy; below that the pass is one serial walk of the
// block per thread, so the walk is split, to runs of eight tokens (one round of loads) at the
// shortest, until about one wave per SIMD is in flight (three with RoPE), and a block's columns
// go to workgroups of their own.  Pass alone, 1 thread -> the split: Nside 16, 20/5 heads 6.7 ->
// 4.9 us (180 -> 1440 waves), Nside 32, 12/3 heads 7.5 -> 5.8 us, 16/4 heads with 128-token
// blocks 13.4 -> 8.4 us, that shape's keys alone 11.7 -> 4.1 us; with RoPE the whole op there
// 118 -> 109 us.  With RoPE and 768 waves or more, only to runs of 32 tokens: 24,576 tokens in
// 64-token blocks, 12/3 heads (864 waves), whole op 86.9 us at two threads, 87.4 at four.  At Nside 64 splitting only adds the sums' exchange (18.6 -> 19.3 us at four
// threads).  The largest passes (24 members) stream from HBM and gain from two threads and
// smaller workgroups again: 176 -> 167 us (8 members: 48.4 -> 51.3 us, so not there).
struct PoolShape { int tpc, wg; };
PoolShape pool_shape(const PoolParams& p, int chunks) {
    const int64_t waves = (int64_t)chunks * p.nb * p.B / 64;  // at one thread per chunk
    if (waves >= 8192) return {2, 256};
    const bool rope = p.rope_cos != nullptr;
    int tpc = rope ? 2 : 1;
    const int first = tpc;
    const int run = rope && waves >= 768 ? 64 : 16;
    while (tpc < 8 && waves * tpc < (rope ? 3072 : 768) && p.bs >= run * tpc) tpc *= 2;
    return {tpc, tpc > first ? (rope ? 256 : 128) : 0};
}

template <int ROPE>
const void* pool_fn(int tpc) {
    switch (tpc) {
        case 1: return (const void*)pool_kernel<ROPE, 1>;
        case 2: return (const void*)pool_kernel<ROPE, 2>;
        case 4: return (const void*)pool_kernel<ROPE, 4>;
        default: return (const void*)pool_kernel<ROPE, 8>;
    }
}

}  // namespace

hipError_t launch_pool(const PoolParams& p, hipStream_t s) {
    PoolParams q = p;
    // stage the RoPE rows in LDS when the block's rows fit the default dynamic limit (256 tokens, 64 KB)
    q.rope_lds = p.rope_cos != nullptr && p.bs <= 256;
    void* args[] = {&q};
    const int tgrid = (p.kfrag || p.vfrag) ? p.nb_pad : p.nb;
    const size_t lds = q.rope_lds ? (size_t)p.bs * 256 : 0;
    const int chunks = 8 * (p.heads[0] + p.heads[1] + p.heads[2]);
    const PoolShape shape = pool_shape(p, chunks);
    const void* fn = p.rope_cos == nullptr ? pool_fn<0>(shape.tpc) : q.rope_lds ? pool_fn<1>(shape.tpc) : pool_fn<2>(shape.tpc);
    // tpc threads per 16-byte column chunk of the q, k, v rows, in whole waves
    const int items = shape.tpc * chunks;
    const int cap = p.rope_cos == nullptr ? kPoolMaxThreads<0> : q.rope_lds ? kPoolMaxThreads<1> : kPoolMaxThreads<2>;
    const int threads = std::min((items + 63) / 64 * 64, shape.wg > 0 ? shape.wg : cap);
    const int z = shape.wg > 0 ? (items + threads - 1) / threads : 1;
    return hipLaunchKernel(fn, dim3(tgrid, p.B, z), dim3(threads), args, lds, s);
}

}  // namespace mosaic
