// pool.hip -- mean pooling of q, k, v over runs of sparse_block_size tokens (gfx950).
//
// Replaces reduce(x, 'b (nb bs) h d -> b nb h d', 'mean') (primitives.py:65-66,76): fp32
// sum over the block's tokens, divided by the block size, rounded to bf16.
// The workgroups of (pooled block t, batch b), one or a few that share its columns, read the
// block's q, k and v rows once (HBM-bound).  TPC adjacent threads share one 16-byte column chunk
// of a row and each streams it down its own part of the block's tokens.  More threads per chunk
// shorten the serial walk and put more loads in flight where the grid alone leaves the chip idle
// (pool_shape).
// The order of the sum is a function of the block size alone, so a member's pooled means, and the
// blocks selected from them, are the same alone and in an ensemble, with RoPE and without: the
// block's groups of eight tokens fall into 2, 4 or 8 contiguous runs (run_bits), each group is summed
// in token order and each run in the order of its groups, and the run sums are added as a binary
// tree, by the thread that holds several runs and then through DPP.
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

// x of lane l ^ STEP, STEP 1, 2 or 4: quad_perm [1, 0, 3, 2] and [2, 3, 0, 1]; row_shl:4 into the
// banks of four lanes with bit 2 clear and row_shr:4 into the others
template <int STEP>
__device__ __forceinline__ float other_lane(float x) {
    const int v = __float_as_int(x);
    if constexpr (STEP == 4)
        return __int_as_float(__builtin_amdgcn_update_dpp(__builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false), v, 0x114,
                                                          0xf, 0xa, false));
    else
        return __int_as_float(__builtin_amdgcn_update_dpp(0, v, STEP == 1 ? 0xb1 : 0x4e, 0xf, 0xf, false));
}
// Half of x summed over lanes l and l ^ STEP: the lane with that bit clear gets the sums of the
// first N values, the other one of the last N.
template <int STEP, int N>
__device__ __forceinline__ void halve(const float (&x)[2 * N], float (&sum)[N], bool upper) {
#pragma unroll
    for (int e = 0; e < N; ++e) {
        const float keep = upper ? x[N + e] : x[e], give = upper ? x[e] : x[N + e];
        sum[e] = keep + other_lane<STEP>(give);
    }
}
template <int N>
__device__ __forceinline__ void copy(float (&to)[N], const float (&x)[N]) {
#pragma unroll
    for (int e = 0; e < N; ++e) to[e] = x[e];
}
template <int TPC>
__device__ __forceinline__ float chunk_max(float x) {  // over the TPC lanes of a chunk
    x = fmaxf(x, other_lane<1>(x));
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

// 2^run_bits runs of a block: as many as threads can share a chunk
__host__ __device__ __forceinline__ int run_bits(int bs) { return bs >= 64 ? 3 : bs >= 32 ? 2 : 1; }

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
        // The means that this thread ends up with, dimensions e0 .. e0 + M - 1 of the chunk, to the
        // operand-ordered output of block t (zero past nb)
        constexpr int M = 8 / TPC;
        const int e0 = 4 * (part & 1) + (TPC > 2 ? 2 * ((part >> 1) & 1) : 0) + (TPC > 4 ? part >> 2 : 0);
        auto store = [&](bf16_t* dst, const float (&x)[M]) __attribute__((always_inline)) {
            if constexpr (M == 4) *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]));
            else if constexpr (M == 2) *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2(x[0], x[1]);
            else *dst = (bf16_t)(pack_bf16x2(x[0], 0.f) & 0xffffu);
        };
        auto store_frag = [&](const float (&x)[M]) __attribute__((always_inline)) {
            const int UT = p.nb_pad >> 5, ut = t >> 5, w = t & 31;
            if (which == 1) {
                store(frag + kfrag_index(b, hd, heads, UT, ut, ch >> 1, 32 * (ch & 1) + w) + e0, x);
            } else {
                const int s2 = w >> 4, rem = w & 15, slot = 4 * (rem >> 3) + (rem & 3), hh = (rem & 7) >> 2;
#pragma unroll
                for (int e = 0; e < M; ++e) {
                    const int d = 8 * ch + e0 + e;
                    frag[vfrag_index(b, hd, heads, UT, ut, d >> 5, s2, 32 * hh + (d & 31)) + slot] =
                        (bf16_t)(pack_bf16x2(x[e], 0.f) & 0xffffu);
                }
            }
        };
        if (t >= p.nb) {  // padding blocks of the operand-ordered outputs
            const float zero[M] = {};
            if (frag) store_frag(zero);
            continue;
        }
        // this thread's runs of per_run groups of eight tokens (the block's last ones shorter or empty)
        const int bits = run_bits(p.bs), per_thread = TPC == 8 ? 1 : (1 << bits) / TPC;
        const int per_run = (((p.bs + 7) >> 3) + (1 << bits) - 1) >> bits;
        const int n0 = min(8 * part * per_thread * per_run, p.bs);
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
        float sqmax = 0.f;  // largest squared norm of this 8-dim chunk over the block's tokens
        auto add_token = [&](float (&sum)[8], uint4 v, bool first) __attribute__((always_inline)) {
            const float x[8] = {bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y),
                                bf_lo(v.z), bf_hi(v.z), bf_lo(v.w), bf_hi(v.w)};
            float sq = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sum[e] = first ? x[e] : sum[e] + x[e];
                sq = fmaf(x[e], x[e], sq);
            }
            sqmax = fmaxf(sqmax, sq);
        };
        const int count = p.bs - n0;
        int i = 0;
        auto add_group = [&](float (&sum)[8]) __attribute__((always_inline)) {  // the next eight tokens, or what is left
            if (i + 8 <= count) {  // all loads in flight
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
                for (int u = 0; u < 8; ++u) add_token(sum, v[u], u == 0);
                i += 8;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[e] = 0.f;
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
                    add_token(sum, v, false);
                }
            }
        };
        auto add = [](float (&sum)[8], const float (&x)[8]) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] = x[e] + sum[e];
        };
        // acc: the run's sum, then with the waiting sums of one and two runs that of the largest
        // subtree ending with it
        float acc[8], sum1[8], sum2[8];
        for (int j = 0; j < per_thread; ++j) {
            for (int g = 0; g < per_run; ++g) {
                float sum[8];
                add_group(sum);
                if (g > 0) add(acc, sum);
                else copy(acc, sum);
            }
            if constexpr (TPC < 8) {  // up to 8 / TPC runs
                if (j & 1) {
                    add(acc, sum1);
                    if constexpr (TPC < 4)
                        if (j & 2) add(acc, sum2);
                }
                if (j + 1 == per_thread) break;
                if (j & 1) copy(sum2, acc);
                else copy(sum1, acc);
            }
        }
        // The block's sums, each thread of the chunk left with its M of the 8 (an empty run adds 0),
        // and in every thread the maximum
        float mean[M];
        {
            float s4[4];
            halve<1>(acc, s4, part & 1);
            if constexpr (TPC == 2) {
                copy(mean, s4);
            } else {
                float s2[2];
                halve<2>(s4, s2, part & 2);
                if constexpr (TPC == 4) copy(mean, s2);
                else halve<4>(s2, mean, part & 4);
            }
        }
        sqmax = chunk_max<TPC>(sqmax);
        if (which == 1 && p.kbnd != nullptr && part == 0)
            p.kbnd[(((int64_t)b * p.nb + t) * heads + hd) * 8 + ch] = sqmax;
        const float denom = (float)p.bs;
#pragma unroll
        for (int e = 0; e < M; ++e) mean[e] = (mean[e] + 0.f) / denom;  // a sum of negative zeros is 0
        bf16_t* out = sel3(p.out_bnhd, which);
        if (out) store(out + (((int64_t)b * p.nb + t) * heads + hd) * kHeadDim + ch * 8 + e0, mean);
        if (frag) store_frag(mean);
    }
}

// Threads per column chunk (at most the block's runs) and per workgroup, by the waves that one
// thread per chunk would make.  All choices give the same bits.  Pass alone, us.
//
// Without RoPE, few waves leave most of the chip waiting on one serial walk of the block per thread,
// so the walk is split until about one wave per SIMD is in flight: 20/5 heads, 3072 tokens (180 waves) 5.3 at
// two threads, 4.5 at eight; 12/3 heads, 12,288 tokens (432 waves) 6.0 at two, 6.1 at eight; with 16/4 heads
// and 128-token blocks the keys alone 6.9 and 3.8.  Between, from the MALL, more threads shorten
// the contiguous part of a row that a wave reads: 16/4 heads, three members (1728 waves) 18.9 at two threads, 20.7 at
// eight; six members (3456) 34.5 at two and four, 37.4 at eight.  The largest passes stream from HBM and
// gain from loads in flight again: 24 members (13,824) 167 at two, 160 at eight in workgroups of 256.
//
// With RoPE every workgroup of a block stages the block's table rows, so its columns go to few
// workgroups: 12/3 heads, 128-token blocks, 49,152 tokens (864 waves) 26.2 at four threads and 512 per workgroup,
// 27.0 at 256, 36.0 at 128; 24 members of that (20,736) 641 at four threads, 607 at eight, both at 512.  Runs of
// eight tokens do not pay there: 64-token blocks, 49,152 tokens (1728 waves) 24.4 at two threads in one
// workgroup, 28.3 at eight in workgroups of 512.
constexpr int kOneWorkgroup = 1024;  // all columns of a block in one, passing over them if there are more
struct PoolShape { int tpc, wg; };
PoolShape pool_shape(const PoolParams& p, int chunks) {
    const int64_t waves = (int64_t)chunks * p.nb * p.B / 64;
    const int runs = 1 << run_bits(p.bs);
    if (p.rope_cos != nullptr) {
        if (waves < 768 || !p.rope_lds) return {runs, 256};
        if (p.bs < 128) return {2, kOneWorkgroup};
        return {waves < 4096 ? 4 : 8, 512};
    }
    if (waves < 768) {
        int tpc = 2;
        while (tpc < runs && waves * tpc < 768) tpc *= 2;
        return {tpc, 128};
    }
    if (waves < 2048) return {2, 64};
    if (waves < 6144) return {std::min(runs, 4), 128};
    return {runs, 256};
}

template <int ROPE>
const void* pool_fn(int tpc) {
    return tpc == 2 ? (const void*)pool_kernel<ROPE, 2> : tpc == 4 ? (const void*)pool_kernel<ROPE, 4> : (const void*)pool_kernel<ROPE, 8>;
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
    const PoolShape shape = pool_shape(q, chunks);
    const void* fn = p.rope_cos == nullptr ? pool_fn<0>(shape.tpc) : q.rope_lds ? pool_fn<1>(shape.tpc) : pool_fn<2>(shape.tpc);
    // tpc threads per 16-byte column chunk of the q, k, v rows, in whole waves
    const int items = shape.tpc * chunks;
    const int threads = std::min((items + 63) / 64 * 64, shape.wg);
    const int z = shape.wg == kOneWorkgroup ? 1 : std::min((items + threads - 1) / threads, 65535);
    return hipLaunchKernel(fn, dim3(tgrid, p.B, z), dim3(threads), args, lds, s);
}

}  // namespace mosaic
