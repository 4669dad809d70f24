// interp.hip -- k-nearest-neighbour cross-attention between two grids (gfx950).
//
// Replaces the gather-attention of CrossAttentionInterpolate.forward (primitives.py:265-283):
//   q[s, j]    = to_q(rel_pos[s, j])            (Linear 3 -> H*64, bf16 out)
//   score      = sum_d bf16(q[s, j, h, d] * k[n(s, j), b, h, d])  -> bf16, * scale -> bf16
//   w          = softmax_j(score) in fp32, then bf16        (softmax over the K neighbours)
//   out[s,b,h] = sum_j bf16(w[j] * v[n(s, j), b, h, :])      -> bf16
// with the reference's rounding points (bf16 elementwise products, fp32 sums rounded once).
// The reference materialises q [S_to, K, H*64] and the gathered k, v [S_to, K, B, H*64];
// here q is formed in registers from the three rel_pos numbers and the head's 64x3 slice of
// to_q, and the k / v rows are read straight from [S_from, B, H, 64] (neighbouring targets
// share most of their neighbours, so rows are reused from L2).
//
// Two forms of the two weighted sums: products rounded to bf16 before they are added (the
// reference's eager elementwise ops) and exact products summed in fp32 (its compiled path).
//
// The bf16-product form is VALU-bound: every (target, member, head) takes 2 K 64 rounded
// products.  Each product is one v_dot2_f32_bf16 of the packed k / v pair against (x, 0) or
// (0, x) (exact: a bf16 x bf16 product fits fp32), then half a v_cvt_pk_bf16_f32 and half a
// v_dot2_f32_bf16 that adds the rounded pair; no k / v element is unpacked to fp32.
//
// Per-target kernel: one wave per (target s, head h) pair, looping over the batch members b with
// the next member's k / v loaded as soon as the current member is done with them.  Lane l = 8
// jg + dc holds the 8-dim chunk dc of neighbours jg + 8 i (its "slots"): every k / v read is a
// 16-byte load and each 128-byte row is read by 8 adjacent lanes.  Scores are summed over the 8
// chunk lanes with DPP, the softmax max / sum over the 8 neighbour groups with DPP row_ror:8,
// v_permlane16_swap and v_permlane32_swap.  The output of the bf16-product form: the 8 partial
// sums per lane are reduce-scattered over the groups by the same three exchanges, leaving one
// dimension per lane; of the fp32 form: v and the weights go through LDS (weighted_sum).
// The fp32 form also has an LDS-staged kernel, for tiles of targets (below).
// Workgroups are remapped so that each XCD takes one contiguous range of targets, in
// the caller's target order when one is given: with targets sorted along a space-filling
// curve, the waves in flight on an XCD share most of their neighbours' rows in its L2.
#include "bsa_common.h"

#include <type_traits>

namespace mosaic {
namespace {

constexpr int kInterpWaves = 4;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    // every lane's source lane exists for the patterns used here, so the old value and the
    // bound control never matter; with an undefined old value the compiler folds the move
    // into the add (with old = 0 it kept a separate move and a zeroing move for
    // row_half_mirror)
    return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ float dpp_max(float x) {
    return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false)));
}

// x summed over the 8 chunk lanes of its neighbour group (lanes l ^ 1, l ^ 2, l ^ 4)
__device__ __forceinline__ float chunk_sum(float x) {
    x = dpp_add<0xb1>(x);      // quad_perm [1,0,3,2]
    x = dpp_add<0x4e>(x);      // quad_perm [2,3,0,1]
    return dpp_add<0x141>(x);  // row_half_mirror
}

// the same sum in the order of the fp32-product form: lane 7 - l of the group, then l ^ 2, l ^ 1
__device__ __forceinline__ float dot_chunk_sum(float x) {
    x = dpp_add<0x141>(x);
    x = dpp_add<0x4e>(x);
    return dpp_add<0xb1>(x);
}

// v_permlane16_swap(a, b): rows 1 and 3 of a trade places with rows 0 and 2 of b.  The
// returned pair, summed, is a[l] + a[l ^ 16] in even rows and b[l] + b[l ^ 16] in odd rows.
__device__ __forceinline__ float swap16_add(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// v_permlane32_swap(a, b): lanes 32-63 of a trade places with lanes 0-31 of b.  The pair,
// summed, is a[l] + a[l ^ 32] in lanes 0-31 and b[l] + b[l ^ 32] in lanes 32-63.
__device__ __forceinline__ float swap32_add(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// x summed / maximised over the 8 neighbour groups (lanes l ^ 8, l ^ 16, l ^ 32)
__device__ __forceinline__ float group_sum(float x) {
    x = dpp_add<0x128>(x);  // row_ror:8 within a 16-lane row: lane l ^ 8
    return xor32_add(swap16_add(x, x));
}
__device__ __forceinline__ float group_max(float x) {
    x = dpp_max<0x128>(x);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Exact bf16 products without unpacking: with a = (x, 0) or (0, x) (x bf16 in the low or
// high half), v_dot2_f32_bf16 of a and a packed bf16 pair b is x times the matching half of b,
// plus 0 (a bf16 x bf16 product is exact in fp32).  A dot product's result needs three wait
// states before another VALU instruction reads it, and the compiler does not track that
// through inline assembly, so the blocks below put their eight products first, every
// rounding (v_cvt_pk_bf16_f32 of a pair) reads products at least three instructions old, and
// each block ends with s_nop 2 before its sums are read.  The additions are dot products
// too, chained through the accumulator operand of the same instruction, which needs no wait.
//
// A neighbour's score partial over this lane's 8 dimensions: the eight products q[i] . k
// (q[i] = (x, 0) or (0, x) against the packed pairs of k), rounded to bf16 in pairs and added
// in fp32 by dot products with ones = (1, 1), in dimension order from 0.
__device__ __forceinline__ float score_partial(const uint32_t (&q)[8], const uint4& k, uint32_t ones) {
    float part, t0, t1, t2, t3, t4, t5, t6, t7;
    uint32_t c0, c1, c2, c3;
    asm("v_dot2_f32_bf16 %5, %13, %21, 0\n\t"
        "v_dot2_f32_bf16 %6, %14, %21, 0\n\t"
        "v_dot2_f32_bf16 %7, %15, %22, 0\n\t"
        "v_dot2_f32_bf16 %8, %16, %22, 0\n\t"
        "v_dot2_f32_bf16 %9, %17, %23, 0\n\t"
        "v_dot2_f32_bf16 %10, %18, %23, 0\n\t"
        "v_dot2_f32_bf16 %11, %19, %24, 0\n\t"
        "v_dot2_f32_bf16 %12, %20, %24, 0\n\t"
        "v_cvt_pk_bf16_f32 %1, %5, %6\n\t"
        "v_cvt_pk_bf16_f32 %2, %7, %8\n\t"
        "v_cvt_pk_bf16_f32 %3, %9, %10\n\t"
        "v_cvt_pk_bf16_f32 %4, %11, %12\n\t"
        "v_dot2_f32_bf16 %0, %1, %25, 0\n\t"
        "v_dot2_f32_bf16 %0, %2, %25, %0\n\t"
        "v_dot2_f32_bf16 %0, %3, %25, %0\n\t"
        "v_dot2_f32_bf16 %0, %4, %25, %0\n\t"
        "s_nop 2"
        : "=v"(part), "=v"(c0), "=v"(c1), "=v"(c2), "=v"(c3),
          "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(t4), "=&v"(t5), "=&v"(t6), "=&v"(t7)
        : "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]), "v"(q[4]), "v"(q[5]), "v"(q[6]), "v"(q[7]),
          "v"(k.x), "v"(k.y), "v"(k.z), "v"(k.w), "s"(ones));
    return part;
}

// Two neighbours' (weights a and b) contributions to four output dimensions 2m .. 2m + 3:
// acc[e] (+)= bf16(wa v_a[d]) + bf16(wb v_b[d]) for d = 2m + e, the products formed as above
// from (w, 0) / (0, w) and the packed pairs va0 = v_a[2m, 2m+1], va1 = v_a[2m+2, 2m+3] (vb0,
// vb1 of b), each pair rounded by one v_cvt_pk_bf16_f32 and added by a dot product with
// (1, 1) -- starting from 0 when FIRST.  Ends with the three wait states the sums need.
template <bool FIRST>
__device__ __forceinline__ void out_pair(uint32_t wa_lo, uint32_t wb_lo, uint32_t wa_hi, uint32_t wb_hi,
                                         uint32_t va0, uint32_t vb0, uint32_t va1, uint32_t vb1, uint32_t ones,
                                         float* acc) {
    float t0, t1, t2, t3, t4, t5, t6, t7;
    uint32_t c0, c1, c2, c3;
#define MOSAIC_OUT_PAIR_PRODUCTS                          \
    "v_dot2_f32_bf16 %8, %16, %20, 0\n\t"                \
    "v_dot2_f32_bf16 %9, %17, %21, 0\n\t"                \
    "v_dot2_f32_bf16 %10, %18, %20, 0\n\t"               \
    "v_dot2_f32_bf16 %11, %19, %21, 0\n\t"               \
    "v_dot2_f32_bf16 %12, %16, %22, 0\n\t"               \
    "v_dot2_f32_bf16 %13, %17, %23, 0\n\t"               \
    "v_dot2_f32_bf16 %14, %18, %22, 0\n\t"               \
    "v_dot2_f32_bf16 %15, %19, %23, 0\n\t"               \
    "v_cvt_pk_bf16_f32 %4, %8, %9\n\t"                   \
    "v_cvt_pk_bf16_f32 %5, %10, %11\n\t"                 \
    "v_cvt_pk_bf16_f32 %6, %12, %13\n\t"                 \
    "v_cvt_pk_bf16_f32 %7, %14, %15\n\t"
#define MOSAIC_OUT_PAIR_OPERANDS                                                                      \
    "=v"(c0), "=v"(c1), "=v"(c2), "=v"(c3),                                                           \
        "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(t4), "=&v"(t5), "=&v"(t6), "=&v"(t7)      \
        : "v"(wa_lo), "v"(wb_lo), "v"(wa_hi), "v"(wb_hi), "v"(va0), "v"(vb0), "v"(va1), "v"(vb1), "s"(ones)
    if constexpr (FIRST) {
        asm(MOSAIC_OUT_PAIR_PRODUCTS
            "v_dot2_f32_bf16 %0, %4, %24, 0\n\t"
            "v_dot2_f32_bf16 %1, %5, %24, 0\n\t"
            "v_dot2_f32_bf16 %2, %6, %24, 0\n\t"
            "v_dot2_f32_bf16 %3, %7, %24, 0\n\t"
            "s_nop 2"
            : "=v"(acc[0]), "=v"(acc[1]), "=v"(acc[2]), "=v"(acc[3]), MOSAIC_OUT_PAIR_OPERANDS);
    } else {
        asm(MOSAIC_OUT_PAIR_PRODUCTS
            "v_dot2_f32_bf16 %0, %4, %24, %0\n\t"
            "v_dot2_f32_bf16 %1, %5, %24, %1\n\t"
            "v_dot2_f32_bf16 %2, %6, %24, %2\n\t"
            "v_dot2_f32_bf16 %3, %7, %24, %3\n\t"
            "s_nop 2"
            : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), MOSAIC_OUT_PAIR_OPERANDS);
    }
#undef MOSAIC_OUT_PAIR_PRODUCTS
#undef MOSAIC_OUT_PAIR_OPERANDS
}

// One neighbour (weight w, as (w, 0) and (0, w)) against all eight output dimensions of the
// lane: acc[d] (+)= bf16(w v[d]), the pair (2m, 2m + 1) rounded by one v_cvt_pk_bf16_f32 and
// its halves added by dot products with pick_lo = (1, 0) and pick_hi = (0, 1) (scalar
// registers: as a constant operand the compiler would encode (1, 0) as the inline constant
// 1.0, which the dot product reads as (0, 1)) -- starting from 0 when FIRST.
template <bool FIRST>
__device__ __forceinline__ void out_single(uint32_t w_lo, uint32_t w_hi, const uint4& v, uint32_t pick_lo,
                                           uint32_t pick_hi, float* acc) {
    float t0, t1, t2, t3, t4, t5, t6, t7;
    uint32_t c0, c1, c2, c3;
#define MOSAIC_OUT_SINGLE_PRODUCTS                        \
    "v_dot2_f32_bf16 %12, %20, %22, 0\n\t"               \
    "v_dot2_f32_bf16 %13, %21, %22, 0\n\t"               \
    "v_dot2_f32_bf16 %14, %20, %23, 0\n\t"               \
    "v_dot2_f32_bf16 %15, %21, %23, 0\n\t"               \
    "v_dot2_f32_bf16 %16, %20, %24, 0\n\t"               \
    "v_dot2_f32_bf16 %17, %21, %24, 0\n\t"               \
    "v_dot2_f32_bf16 %18, %20, %25, 0\n\t"               \
    "v_dot2_f32_bf16 %19, %21, %25, 0\n\t"               \
    "v_cvt_pk_bf16_f32 %8, %12, %13\n\t"                 \
    "v_cvt_pk_bf16_f32 %9, %14, %15\n\t"                 \
    "v_cvt_pk_bf16_f32 %10, %16, %17\n\t"                \
    "v_cvt_pk_bf16_f32 %11, %18, %19\n\t"
#define MOSAIC_OUT_SINGLE_OPERANDS                                                                    \
    "=v"(c0), "=v"(c1), "=v"(c2), "=v"(c3),                                                           \
        "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(t4), "=&v"(t5), "=&v"(t6), "=&v"(t7)      \
        : "v"(w_lo), "v"(w_hi), "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w), "s"(pick_lo), "s"(pick_hi)
    if constexpr (FIRST) {
        asm(MOSAIC_OUT_SINGLE_PRODUCTS
            "v_dot2_f32_bf16 %0, %8, %26, 0\n\t"
            "v_dot2_f32_bf16 %1, %8, %27, 0\n\t"
            "v_dot2_f32_bf16 %2, %9, %26, 0\n\t"
            "v_dot2_f32_bf16 %3, %9, %27, 0\n\t"
            "v_dot2_f32_bf16 %4, %10, %26, 0\n\t"
            "v_dot2_f32_bf16 %5, %10, %27, 0\n\t"
            "v_dot2_f32_bf16 %6, %11, %26, 0\n\t"
            "v_dot2_f32_bf16 %7, %11, %27, 0\n\t"
            "s_nop 2"
            : "=v"(acc[0]), "=v"(acc[1]), "=v"(acc[2]), "=v"(acc[3]), "=v"(acc[4]), "=v"(acc[5]), "=v"(acc[6]),
              "=v"(acc[7]), MOSAIC_OUT_SINGLE_OPERANDS);
    } else {
        asm(MOSAIC_OUT_SINGLE_PRODUCTS
            "v_dot2_f32_bf16 %0, %8, %26, %0\n\t"
            "v_dot2_f32_bf16 %1, %8, %27, %1\n\t"
            "v_dot2_f32_bf16 %2, %9, %26, %2\n\t"
            "v_dot2_f32_bf16 %3, %9, %27, %3\n\t"
            "v_dot2_f32_bf16 %4, %10, %26, %4\n\t"
            "v_dot2_f32_bf16 %5, %10, %27, %5\n\t"
            "v_dot2_f32_bf16 %6, %11, %26, %6\n\t"
            "v_dot2_f32_bf16 %7, %11, %27, %7\n\t"
            "s_nop 2"
            : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4]), "+v"(acc[5]), "+v"(acc[6]),
              "+v"(acc[7]), MOSAIC_OUT_SINGLE_OPERANDS);
    }
#undef MOSAIC_OUT_SINGLE_PRODUCTS
#undef MOSAIC_OUT_SINGLE_OPERANDS
}

// fp32 products (the reference under torch.compile: its fused reductions of (q * k).sum and
// (w * v).sum multiply and add in fp32 and round only the sums).  A neighbour's score partial
// over this lane's 8 dimensions: four dot products of packed (q, q) pairs against k's pairs,
// chained through the accumulator, in dimension order from 0.
__device__ __forceinline__ bf16x2_t as_bf2(uint32_t w) { return __builtin_bit_cast(bf16x2_t, w); }
__device__ __forceinline__ float score_dot(const uint32_t (&q)[4], const uint4& k) {
    float a = __builtin_amdgcn_fdot2_f32_bf16(as_bf2(q[0]), as_bf2(k.x), 0.f, false);
    a = __builtin_amdgcn_fdot2_f32_bf16(as_bf2(q[1]), as_bf2(k.y), a, false);
    a = __builtin_amdgcn_fdot2_f32_bf16(as_bf2(q[2]), as_bf2(k.z), a, false);
    return __builtin_amdgcn_fdot2_f32_bf16(as_bf2(q[3]), as_bf2(k.w), a, false);
}
// The score of a slot in base-2 units, sc = bf16(bf16(part) * scale) * log2 e.  A power-of-two
// scale leaves bf16(part) * scale a bf16 value (a product too small to be normal is below
// 2^-126 in magnitude, and so is the difference its rounding would make), so that case takes
// one multiply by scale * log2 e.
template <bool POW2>
__device__ __forceinline__ float scaled_score(float part, const InterpParams& p) {
    return POW2 ? round_bf16(part) * p.scale_log2e : round_bf16(round_bf16(part) * p.scale) * kLog2e;
}

// Softmax weights of the lane's slots over the K neighbours, from the slots' base-2 scores and
// the lane's own maximum m: exp2(sc - max) / sum (0 for an absent neighbour: score -inf, the
// maximum finite).
template <int NSLOT>
__device__ __forceinline__ void softmax_weights(const float (&sc)[NSLOT], float m, float (&w)[NSLOT]) {
    m = group_max(m);
    float l = 0.f;
#pragma unroll
    for (int i = 0; i < NSLOT; ++i) {
        w[i] = __builtin_amdgcn_exp2f(sc[i] - m);
        l += w[i];
    }
    const float inv = __builtin_amdgcn_rcpf(group_sum(l));
#pragma unroll
    for (int i = 0; i < NSLOT; ++i) w[i] *= inv;
}

// The order of the neighbours in the fp32-product output sum: position pos of 8 NSLOT holds
// neighbour knn_order(pos).  Slots 2m and 2m + 1 alternate, so the weights of a neighbour group
// (jg) form one packed pair; an odd last slot follows in its own order.
template <int NSLOT>
__device__ __forceinline__ constexpr int knn_order(int pos) {
    return pos < 16 * (NSLOT / 2) ? 16 * (pos / 16) + 8 * (pos & 1) + (pos % 16) / 2 : pos;
}
// This lane's weights (slots w[i], neighbours jg + 8 i) into a target's weight table at lds:
// bf16, in the order of knn_order.
template <int NSLOT>
__device__ __forceinline__ void put_weights(const float (&w)[NSLOT], char* lds, int jg) {
#pragma unroll
    for (int i = 0; i + 1 < NSLOT; i += 2) *reinterpret_cast<uint32_t*>(lds + 16 * i + 4 * jg) = pack_bf16x2(w[i], w[i + 1]);
    if constexpr (NSLOT & 1)
        *reinterpret_cast<uint16_t*>(lds + 16 * (NSLOT - 1) + 2 * jg) = (uint16_t)(pack_bf16x2(w[NSLOT - 1], 0.f) & 0xffffu);
}
// Four neighbours' values of dimension d = lane: a transposing read, in which lane l addresses
// dimensions 16 (l / 16) + 4 (l % 4) .. + 3 of the row of position (l / 4) % 4.
typedef short v4i16_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 read_v4(uint32_t lds, int offset = 0) {
    auto* const a = (__attribute__((address_space(3))) char*)(uintptr_t)lds + offset;
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)a));
}
// Output dimension d = lane of one target, fp32 products: v_mfma_f32_4x4x4_16b_bf16 multiplies,
// in each block of four lanes, four neighbours' values of the lanes' dimensions (vv) with rows
// of weights; every lane holds the same weights (ww), so every row of the result is the output.
// One instruction takes four neighbours, in position order, accumulating in fp32.
template <int NSLOT>
__device__ __forceinline__ float weighted_sum(const uint4 (&ww)[NSLOT], const uint2 (&vv)[2 * NSLOT]) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NSLOT; ++i) {
        a = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(v4i16_t, make_uint2(ww[i].x, ww[i].y)),
                                                   __builtin_bit_cast(v4i16_t, vv[2 * i]), a, 0, 0, 0);
        a = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(v4i16_t, make_uint2(ww[i].z, ww[i].w)),
                                                   __builtin_bit_cast(v4i16_t, vv[2 * i + 1]), a, 0, 0, 0);
    }
    return a[0];
}

// The to_q rows of a lane's eight dimensions (three bf16 weights each: 48 bytes, 16-byte
// aligned) as packed (w0, w1) and (w2, 0), and eight query values bf16(rel . w) from a
// neighbour's rel = (r0, r1), (r2, 0), as packed pairs: fp32 sums of the exact products.
struct QueryRows { uint32_t w01[8], w2[8]; };
__device__ __forceinline__ QueryRows query_rows(const bf16_t* wr) {
    uint32_t u[12];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const uint4 x = ld16(wr + 8 * c);
        u[4 * c] = x.x; u[4 * c + 1] = x.y; u[4 * c + 2] = x.z; u[4 * c + 3] = x.w;
    }
    QueryRows r;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const uint32_t* t = u + 3 * (e / 2);  // w0 w1 | w2 w0' | w1' w2'
        r.w01[e] = t[0];
        r.w2[e] = t[1] & 0xffffu;
        r.w01[e + 1] = (t[1] >> 16) | (t[2] << 16);
        r.w2[e + 1] = t[2] >> 16;
    }
    return r;
}
__device__ __forceinline__ void query_pairs(const QueryRows& w, uint32_t r01, uint32_t r2, uint32_t (&q)[4]) {
    float a0, a1, a2, a3, a4, a5, a6, a7;
    // the eight first products from a literal 0 addend, the second ones through the
    // accumulator (no wait between them), then the three wait states before the conversions
    asm("v_dot2_f32_bf16 %0, %8, %10, 0\n\t"
        "v_dot2_f32_bf16 %1, %8, %11, 0\n\t"
        "v_dot2_f32_bf16 %2, %8, %12, 0\n\t"
        "v_dot2_f32_bf16 %3, %8, %13, 0\n\t"
        "v_dot2_f32_bf16 %4, %8, %14, 0\n\t"
        "v_dot2_f32_bf16 %5, %8, %15, 0\n\t"
        "v_dot2_f32_bf16 %6, %8, %16, 0\n\t"
        "v_dot2_f32_bf16 %7, %8, %17, 0\n\t"
        "v_dot2_f32_bf16 %0, %9, %18, %0\n\t"
        "v_dot2_f32_bf16 %1, %9, %19, %1\n\t"
        "v_dot2_f32_bf16 %2, %9, %20, %2\n\t"
        "v_dot2_f32_bf16 %3, %9, %21, %3\n\t"
        "v_dot2_f32_bf16 %4, %9, %22, %4\n\t"
        "v_dot2_f32_bf16 %5, %9, %23, %5\n\t"
        "v_dot2_f32_bf16 %6, %9, %24, %6\n\t"
        "v_dot2_f32_bf16 %7, %9, %25, %7\n\t"
        "s_nop 2"
        : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3), "=&v"(a4), "=&v"(a5), "=&v"(a6), "=&v"(a7)
        : "v"(r01), "v"(r2), "v"(w.w01[0]), "v"(w.w01[1]), "v"(w.w01[2]), "v"(w.w01[3]), "v"(w.w01[4]), "v"(w.w01[5]),
          "v"(w.w01[6]), "v"(w.w01[7]), "v"(w.w2[0]), "v"(w.w2[1]), "v"(w.w2[2]), "v"(w.w2[3]), "v"(w.w2[4]),
          "v"(w.w2[5]), "v"(w.w2[6]), "v"(w.w2[7]));
    q[0] = pack_bf16x2(a0, a1); q[1] = pack_bf16x2(a2, a3); q[2] = pack_bf16x2(a4, a5); q[3] = pack_bf16x2(a6, a7);
}

__device__ __forceinline__ void unpack8(const uint4& w, float (&f)[8]) {
    const uint32_t a[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) { f[2 * e] = bf_lo(a[e]); f[2 * e + 1] = bf_hi(a[e]); }
}

// The 16-byte chunk at byte offset off from a member's base (wave-uniform).  With 32-bit
// offsets the load is a raw buffer load: base in the resource (scalar registers), the offset
// as its per-lane offset, so the member loop spends no vector instruction on addresses.
template <bool OFF32, typename Off>
__device__ __forceinline__ uint4 ld_member(const bf16_t* base, Off off) {
    if constexpr (OFF32) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), (short)0, -1, 0x00020000);
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
        return make_uint4(v[0], v[1], v[2], v[3]);
    } else {
        return ld16(reinterpret_cast<const char*>(base) + off);
    }
}

// Waves per SIMD each instantiation is compiled for (the register budget): 6 at three slots
// with 32-bit offsets (the model's K = 24), what fits without spilling elsewhere.
constexpr int knn_waves(int nslot, bool off32) { return nslot <= 1 ? 8 : nslot == 2 ? 7 : nslot == 3 ? (off32 ? 6 : 5) : 4; }

// RP: products rounded to bf16 (the reference's eager elementwise ops); else fp32 products
template <int NSLOT, bool OFF32, bool POW2, bool RP>
__global__ __launch_bounds__(kInterpWaves * 64) __attribute__((amdgpu_waves_per_eu(knn_waves(NSLOT, OFF32)))) void knn_attn_kernel(InterpParams p) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t pair = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * kInterpWaves + wave;
    if (pair >= (int64_t)p.S_to * p.H) return;  // wave-uniform; the kernel has no barrier
    const int pos = (int)(pair / p.H), h = (int)(pair - (int64_t)pos * p.H);
    // targets outside [0, S_to) in the order are clamped (memory safety)
    const int s = p.target_order ? min(max(p.target_order[pos], 0), p.S_to - 1) : pos;
    const int K = p.K, dc = lane & 7, jg = lane >> 3;

    // to_q rows h*64 + 8 dc .. + 7 (three bf16 weights each: 48 bytes, 16-byte aligned)
    const bf16_t* const wr = p.w_q + ((int64_t)h * 64 + 8 * dc) * 3;
    float wq[RP ? 24 : 1];
    QueryRows wp;
    if constexpr (RP) {
        float t[8];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            unpack8(ld16(wr + 8 * c), t);
#pragma unroll
            for (int e = 0; e < 8; ++e) wq[8 * c + e] = t[e];
        }
    } else {
        wp = query_rows(wr);
    }
    // per slot: the neighbour's row offsets and this lane's 8 query values,
    // q[j][d] = bf16(rel[j] . W[h*64 + d]) (fp32 sum of the three bf16 products: the
    // Linear's bf16 inputs)
    // byte offsets of this lane's k / v chunks within a member (32 bits when they fit)
    using Off = typename std::conditional<OFF32, uint32_t, int64_t>::type;
    Off koff[NSLOT], voff[NSLOT];
    // RP: q[j][d] as a bf16 in the half of a word that k's dim d occupies; else the packed
    // pairs (q[j][2m], q[j][2m + 1])
    uint32_t qp[NSLOT][RP ? 8 : 4];
#pragma unroll
    for (int i = 0; i < NSLOT; ++i) {
        const int64_t sj = (int64_t)s * K + min(jg + 8 * i, K - 1);
        // indices outside [0, S_from) are clamped (memory safety; the reference would raise)
        const int64_t n = min(max(p.neighbors[sj], 0), p.S_from - 1);
        koff[i] = (Off)(2 * (n * p.k_sn + (int64_t)h * p.k_sh + 8 * dc));
        voff[i] = (Off)(2 * (n * p.v_sn + (int64_t)h * p.v_sh + 8 * dc));
        if constexpr (RP) {
            const float r0 = round_bf16(p.rel_pos[3 * sj]), r1 = round_bf16(p.rel_pos[3 * sj + 1]),
                        r2 = round_bf16(p.rel_pos[3 * sj + 2]);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t bits = __float_as_uint(round_bf16(fmaf(r2, wq[3 * e + 2], fmaf(r1, wq[3 * e + 1], r0 * wq[3 * e]))));
                qp[i][e] = (e & 1) ? bits : bits >> 16;
            }
        } else {
            query_pairs(wp, pack_bf16x2(p.rel_pos[3 * sj], p.rel_pos[3 * sj + 1]), pack_bf16x2(p.rel_pos[3 * sj + 2], 0.f), qp[i]);
        }
    }
    // the output dimension this lane ends up holding: RP, after the reduce-scatter; else its own
    const int dout = RP ? 8 * dc + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1) + ((lane >> 3) & 1) : lane;
    // fp32 products: this wave's rows of v (row j at byte 128 j) and its weights, in LDS
    constexpr int kRows = 8 * NSLOT * 128, kWaveLds = kRows + 16 * NSLOT;
    __shared__ __attribute__((aligned(16))) char v_lds[RP ? 16 : kInterpWaves * kWaveLds];
    char* const vl = v_lds + (RP ? 0 : wave * kWaveLds);
    uint32_t vaddr[2 * NSLOT];
#pragma unroll
    for (int g = 0; g < 2 * NSLOT; ++g)
        vaddr[g] = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)vl +
                   128 * knn_order<NSLOT>(4 * g + ((lane >> 2) & 3)) + 32 * (lane >> 4) + 8 * (lane & 3);
    bf16_t* out = p.out + ((int64_t)s * p.B * p.H + h) * 64 + dout;

    // k / v chunks of the current member; the next member's k is loaded as soon as the scores
    // are done with k, its v once the output is done with v
    uint4 kw[NSLOT], vw[NSLOT];
#pragma unroll
    for (int i = 0; i < NSLOT; ++i) { kw[i] = ld_member<OFF32>(p.k, koff[i]); vw[i] = ld_member<OFF32>(p.v, voff[i]); }
    const uint32_t ones = 0x3f803f80u, pick_lo = 0x3f80u, pick_hi = 0x3f800000u;  // bf16 pairs (1, 1), (1, 0), (0, 1)
    for (int b = 0; b < p.B; ++b) {
        const bool more = b + 1 < p.B;
        // the fp32-product form loads the next member unconditionally (the last member again
        // after the last): a conditional load made the compiler copy every k / v register at
        // the loop's end
        const int64_t bn = more ? b + 1 : b;
        // scores of this lane's slots (every lane of a neighbour group holds its score)
        float sc[NSLOT], m;
#pragma unroll
        for (int i = 0; i < NSLOT; ++i) {
            float part;
            if constexpr (RP) part = chunk_sum(score_partial(qp[i], kw[i], ones));
            else part = dot_chunk_sum(score_dot(qp[i], kw[i]));
            // the score in base-2 units, sc = bf16(bf16(part) * scale) * log2 e.  A power-of-two
            // scale leaves bf16(part) * scale a bf16 value (a product too small to be normal is
            // below 2^-126 in magnitude, and so is the difference its rounding would make), so
            // that case takes one multiply by scale * log2 e.
            const float t = POW2 ? round_bf16(part) * p.scale_log2e : round_bf16(round_bf16(part) * p.scale) * kLog2e;
            // only the last slot can hold absent neighbours (j >= K): NSLOT = ceil(K / 8)
            sc[i] = i < NSLOT - 1 || jg + 8 * i < K ? t : -INFINITY;
            m = i == 0 ? sc[0] : fmaxf(m, sc[i]);
        }
        if (!RP || more) {
#pragma unroll
            for (int i = 0; i < NSLOT; ++i) kw[i] = ld_member<OFF32>(p.k + bn * p.k_sb, koff[i]);
        }
        m = group_max(m);
        float ex[NSLOT], l = 0.f;
#pragma unroll
        for (int i = 0; i < NSLOT; ++i) {
            ex[i] = __builtin_amdgcn_exp2f(sc[i] - m);  // 0 for an absent neighbour (score -inf; m is finite)
            l += ex[i];
        }
        const float inv = __builtin_amdgcn_rcpf(group_sum(l));
        // out[d] = sum over slots of bf16(w * v[d]); two slots at a time share one rounding
        // instruction and one dot-product add.  An absent neighbour (j >= K) has weight 0; its
        // row (a duplicate of a present one) then adds bf16(0 * v) = 0.  The weights are bf16, so
        // each product is one dot product of (w, 0) or (0, w) with a packed pair of v.
        float acc[8];
        if constexpr (!RP) {
            // fp32 products: v and the weights through LDS, lane = dimension
            float wt[NSLOT];
#pragma unroll
            for (int i = 0; i < NSLOT; ++i) {
                wt[i] = ex[i] * inv;
                *reinterpret_cast<uint4*>(vl + 1024 * i + 16 * lane) = vw[i];
            }
            put_weights(wt, vl + kRows, jg);
            asm volatile("" ::: "memory");
        } else {
#pragma unroll
        for (int i = 0; i < NSLOT; i += 2) {
            // the weight as (w, 0) and (0, w): one conversion each
            const float xa = ex[i] * inv;
            const uint32_t wa_lo = pack_bf16x2(xa, 0.f), wa_hi = pack_bf16x2(0.f, xa);
            if (i + 1 < NSLOT) {
                const float xb = ex[i + 1] * inv;
                const uint32_t wb_lo = pack_bf16x2(xb, 0.f), wb_hi = pack_bf16x2(0.f, xb);
                const uint4 &va = vw[i], &vb = vw[i + 1];
                if (i == 0) {
                    out_pair<true>(wa_lo, wb_lo, wa_hi, wb_hi, va.x, vb.x, va.y, vb.y, ones, acc);
                    out_pair<true>(wa_lo, wb_lo, wa_hi, wb_hi, va.z, vb.z, va.w, vb.w, ones, acc + 4);
                } else {
                    out_pair<false>(wa_lo, wb_lo, wa_hi, wb_hi, va.x, vb.x, va.y, vb.y, ones, acc);
                    out_pair<false>(wa_lo, wb_lo, wa_hi, wb_hi, va.z, vb.z, va.w, vb.w, ones, acc + 4);
                }
            } else if (i == 0) {
                out_single<true>(wa_lo, wa_hi, vw[i], pick_lo, pick_hi, acc);
            } else {
                out_single<false>(wa_lo, wa_hi, vw[i], pick_lo, pick_hi, acc);
            }
        }
        }
        if (!RP || more) {
#pragma unroll
            for (int i = 0; i < NSLOT; ++i) vw[i] = ld_member<OFF32>(p.v + bn * p.v_sb, voff[i]);
        }
        float o;
        if constexpr (!RP) {
            uint4 ww[NSLOT];
            uint2 vv[2 * NSLOT];
#pragma unroll
            for (int i = 0; i < NSLOT; ++i) ww[i] = *reinterpret_cast<const uint4*>(vl + kRows + 16 * i);
#pragma unroll
            for (int g = 0; g < 2 * NSLOT; ++g) vv[g] = read_v4(vaddr[g]);
            o = weighted_sum<NSLOT>(ww, vv);
            asm volatile("" ::: "memory");
        } else {
        // reduce-scatter over the 8 neighbour groups: halves (dims e / e + 4), row pairs
        // (e / e + 2), then lanes l ^ 8 (e / e + 1)
        float r4[4], r2[2];
#pragma unroll
        for (int e = 0; e < 4; ++e) r4[e] = swap32_add(acc[e], acc[e + 4]);
#pragma unroll
        for (int e = 0; e < 2; ++e) r2[e] = swap16_add(r4[e], r4[e + 2]);
        const bool odd8 = lane & 8;
        const float keep = odd8 ? r2[1] : r2[0], give = odd8 ? r2[0] : r2[1];
        o = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0x128, 0xf, 0xf, false));
        }
        out[(int64_t)b * p.H * 64] = (bf16_t)(pack_bf16x2(o, 0.f) & 0xffffu);
    }
}

// LDS-staged form (fp32 products): one workgroup per (tile of up to 16 targets, group of hg
// heads), passing over the group's heads and their members.  The tile's distinct source rows
// of k and v (the host-built tables) go into LDS once per pass with direct-to-LDS loads (lane l
// of an instruction lands at byte 16 l of a 1 KB run of 8 rows), double-buffered; waves 0 and 1
// stage k, 2 and 3 v.  The arithmetic per (target, member, head) is the fp32-product form of
// the kernel above in the same order, so both give the same bits.
//
// The bound is vector-instruction issue and LDS reads together (57 % each at 24 members, and
// bank conflicts 22 % of the LDS cycles), so the work per (target, member, head) is cut where it was the same in many lanes.
// Each wave takes a quarter of the tile's targets (up to 4) together:
//   scores   lane 8 jg + dc, as above, holds chunk dc of neighbours jg + 8 i of every target;
//            the sums over the 8 chunk lanes leave target dc % 4's scores in lane (jg, dc), so
//   softmax  one instruction sequence serves the wave's targets;
//   output   lane = dimension: the weights go through LDS (the same in every lane), v comes
//            through transposing LDS reads, four neighbours at once, and the matrix pipe sums
//            over the neighbours (weighted_sum): no sum over lanes is left.
// 24 members, lat-lon 121 x 240 -> HEALPix nside 64, 12 heads, K 24: 3324 -> 2503 us; one
// member back: 268 -> 125 us.  Eight targets per wave and two waves (fewer instructions, but
// two waves per SIMD): 2590 and 202 us.  Member groups as separate workgroups (for the L2's
// sake) only repeat the prologue (4 us per workgroup): 2705 us at 8 members, 2990 at 4.
//
// LDS: per group of 8 rows, four 1 KB runs [k buffer 0][k buffer 1][v buffer 0][v buffer 1],
// so a row's k and v in either buffer sit at fixed distances from its k in buffer 0 (the
// reads take them as immediate offsets; the pass is instantiated for either buffer); 16-byte
// chunk c of v's row r sits at position c ^ (r & 6), which spreads the four rows of a
// transposing read over the banks.  One barrier per pass: after it the next pass's rows have
// landed (every wave waited for its own loads) and no wave still reads the buffer that the
// next pass's loads overwrite.
__device__ __forceinline__ uint32_t lds_addr(const void* ptr) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)ptr;
}
__device__ __forceinline__ uint4 read_k(uint32_t lds) {
    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    const v4u v = *(const __attribute__((address_space(3))) v4u*)(uintptr_t)lds;
    return make_uint4(v[0], v[1], v[2], v[3]);
}
// address = base (uniform) + voff (per lane); LDS destination M0 + 16 l.  Inline assembly: the
// compiler's own direct-to-LDS builtin makes it wait for these loads before every LDS read of
// the other buffer.  M0 is declared clobbered; the compiler sets it again before its own uses.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Three slots' score partials (K 17..24, the model's 24) as one block: the three dot-product
// chains interleaved, each from a literal 0 addend (the builtin form moves 0 into each
// accumulator first), accumulating through their own addend (no wait between them); then the
// three wait states a dot product's result needs before another VALU instruction reads it.
__device__ __forceinline__ void score_dot3(const uint32_t (&q)[3][4], const uint4 (&k)[3], float (&a)[3]) {
    asm("v_dot2_f32_bf16 %0, %3, %15, 0\n\t"
        "v_dot2_f32_bf16 %1, %7, %19, 0\n\t"
        "v_dot2_f32_bf16 %2, %11, %23, 0\n\t"
        "v_dot2_f32_bf16 %0, %4, %16, %0\n\t"
        "v_dot2_f32_bf16 %1, %8, %20, %1\n\t"
        "v_dot2_f32_bf16 %2, %12, %24, %2\n\t"
        "v_dot2_f32_bf16 %0, %5, %17, %0\n\t"
        "v_dot2_f32_bf16 %1, %9, %21, %1\n\t"
        "v_dot2_f32_bf16 %2, %13, %25, %2\n\t"
        "v_dot2_f32_bf16 %0, %6, %18, %0\n\t"
        "v_dot2_f32_bf16 %1, %10, %22, %1\n\t"
        "v_dot2_f32_bf16 %2, %14, %26, %2\n\t"
        "s_nop 2"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2])
        : "v"(q[0][0]), "v"(q[0][1]), "v"(q[0][2]), "v"(q[0][3]), "v"(q[1][0]), "v"(q[1][1]), "v"(q[1][2]),
          "v"(q[1][3]), "v"(q[2][0]), "v"(q[2][1]), "v"(q[2][2]), "v"(q[2][3]), "v"(k[0].x), "v"(k[0].y),
          "v"(k[0].z), "v"(k[0].w), "v"(k[1].x), "v"(k[1].y), "v"(k[1].z), "v"(k[1].w), "v"(k[2].x), "v"(k[2].y),
          "v"(k[2].z), "v"(k[2].w));
}

constexpr int kTileWaves = 4;
constexpr int kWaveTargets = kKnnTileTargets / kTileWaves;  // 4

// The sums over the 8 chunk lanes of one slot's partials of 4 targets: lane dc of each
// neighbour group gets target dc % 4's, in the tree of dot_chunk_sum: the half-row mirror, then
// lanes l ^ 2 (even or odd pairs of targets kept) and l ^ 1 (one target kept).
__device__ __forceinline__ float targets_chunk_sum(const float (&x)[kWaveTargets], int lane) {
    float y[kWaveTargets];
#pragma unroll
    for (int e = 0; e < kWaveTargets; ++e) y[e] = dpp_add<0x141>(x[e]);
    const bool b1 = lane & 2, b0 = lane & 1;
    float z[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float keep = b1 ? y[e + 2] : y[e], give = b1 ? y[e] : y[e + 2];
        z[e] = keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(give), 0x4e, 0xf, 0xf, true));
    }
    const float keep = b0 ? z[1] : z[0], give = b0 ? z[0] : z[1];
    return keep + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(give), 0xb1, 0xf, 0xf, true));
}

template <int N>
using I = std::integral_constant<int, N>;

template <int NSLOT, bool POW2>
__global__ __launch_bounds__(kTileWaves * 64) __attribute__((amdgpu_waves_per_eu(NSLOT == 4 ? 2 : 3)))
void knn_tile_kernel(InterpParams p, KnnTiles tl, int hg) {
    constexpr int KP = 8 * NSLOT, WT = kWaveTargets, HW = kTileWaves / 2;
    constexpr int kLoads = kKnnTileRows / 8 / HW;  // staging instructions per wave at most
    extern __shared__ __attribute__((aligned(16))) uint4 kv_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int groups = (p.H + hg - 1) / hg;
    const int pair = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = __builtin_amdgcn_readfirstlane(pair / groups);
    const int h0 = __builtin_amdgcn_readfirstlane((pair - tile * groups) * hg), h1 = min(h0 + hg, p.H);
    const int K = p.K, dc = lane & 7, jg = lane >> 3;
    const int rows = tl.rows;
    // the tables are clamped into range (memory safety; a malformed table gives wrong rows)
    const int t0 = __builtin_amdgcn_readfirstlane(min(max(tl.start[tile], 0), p.S_to));
    const int t1 = __builtin_amdgcn_readfirstlane(min(max(tl.start[tile + 1], t0), min(t0 + kKnnTileTargets, p.S_to)));
    const int nsrc = __builtin_amdgcn_readfirstlane(min(max(tl.nsrc[tile], 1), rows));
    const int ng = (nsrc + 7) >> 3;  // 8-row groups per tensor
    // this wave's targets
    const int first = t0 + (t1 - t0) * wave / kTileWaves, nt = t0 + (t1 - t0) * (wave + 1) / kTileWaves - first;

    const uint32_t lds0 = lds_addr(kv_lds);
    char* const mem = reinterpret_cast<char*>(kv_lds);
    // after the staging buffers, per wave: rel (bf16: 8 bytes per target and neighbour), the
    // weight tables and the neighbours' rows (LDS offsets)
    char* const rel_lds = mem + 512 * rows + wave * (WT * KP * 12);
    char* const w_lds = rel_lds + WT * KP * 8;
    char* const row_lds = w_lds + WT * KP * 2;

    // the first half of the waves stage k, the second v: instruction r of a wave stages 8-row
    // group g0 + HW r of its tensor
    const bool isv = wave >= HW;
    const int g0 = wave & (HW - 1);
    const bf16_t* const src = isv ? p.v : p.k;
    const int64_t s_n = isv ? p.v_sn : p.k_sn, s_b = isv ? p.v_sb : p.k_sb, s_h = isv ? p.v_sh : p.k_sh;
    uint32_t soff[kLoads];
#pragma unroll
    for (int r = 0; r < kLoads; ++r) {
        // the whole table row, so that these loads do not wait for nsrc
        const int row = min(8 * (g0 + HW * r) + jg, rows - 1);
        const int n = min(max(tl.src[(int64_t)tile * rows + row], 0), p.S_from - 1);
        soff[r] = (uint32_t)(2 * (n * s_n + 8 * (isv ? dc ^ (jg & 6) : dc)));
    }
    auto stage = [&](int h, int b, int buf) __attribute__((always_inline)) {
        const bf16_t* base = src + (int64_t)b * s_b + (int64_t)h * s_h;
        const uint32_t dst = lds0 + 4096u * g0 + (uint32_t)(2 * isv + buf) * 1024u;
#pragma unroll
        for (int r = 0; r < kLoads; ++r) {
            if (g0 + HW * r >= ng) break;  // uniform
            dma16(base, soff[r], __builtin_amdgcn_readfirstlane(dst + 4096u * HW * r));
        }
    };
    stage(h0, 0, 0);

    // this wave's targets: rel and row offsets into LDS, target indices
    for (int x = lane; x < WT * KP; x += 64) {
        const int pos = min(first + x / KP, p.S_to - 1), j = min(x % KP, K - 1);
        const int s = p.target_order ? min(max(p.target_order[pos], 0), p.S_to - 1) : pos;
        const int sl = min(max(tl.slot[(int64_t)pos * K + j], 0), rows - 1);
        const float* r = p.rel_pos + 3 * ((int64_t)s * K + j);
        reinterpret_cast<uint2*>(rel_lds)[x] = make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], 0.f));
        reinterpret_cast<uint16_t*>(row_lds)[x] = (uint16_t)(4096 * (sl >> 3) + 128 * (sl & 7));
    }
    int tgt[WT];
#pragma unroll
    for (int r = 0; r < WT; ++r) {
        const int pos = min(first + r, p.S_to - 1);
        tgt[r] = __builtin_amdgcn_readfirstlane(p.target_order ? min(max(p.target_order[pos], 0), p.S_to - 1) : pos);
    }
    wait_vmem();
    __syncthreads();
    // LDS addresses in buffer 0: k chunk dc of neighbours jg + 8 i; v, as read_v4 takes them
    uint32_t kaddr[WT][NSLOT], vaddr[WT][2 * NSLOT];
#pragma unroll
    for (int r = 0; r < WT; ++r) {
        const uint16_t* row = reinterpret_cast<const uint16_t*>(row_lds) + r * KP;
#pragma unroll
        for (int i = 0; i < NSLOT; ++i) kaddr[r][i] = lds0 + row[jg + 8 * i] + 16 * dc;
#pragma unroll
        for (int g = 0; g < 2 * NSLOT; ++g) {
            const uint32_t o = row[knn_order<NSLOT>(4 * g + ((lane >> 2) & 3))];
            vaddr[r][g] = lds0 + o + ((((uint32_t)lane >> 4) ^ ((o >> 8) & 3)) << 5) + 8 * (lane & 3);
        }
    }

    // opaque from here: kept as sums of two registers each otherwise
#pragma unroll
    for (int r = 0; r < WT; ++r) {
#pragma unroll
        for (uint32_t& a : kaddr[r]) asm volatile("" : "+v"(a));
#pragma unroll
        for (uint32_t& a : vaddr[r]) asm volatile("" : "+v"(a));
    }

    uint32_t qp[WT][NSLOT][4];
    // pass (h, b) from buffer BUF (the next pass staged into the other one meanwhile)
    auto pass = [&](int h, int b, auto BUF) __attribute__((always_inline)) {
        constexpr int buf = decltype(BUF)::value;
        const bool last = b + 1 == p.B;
        if (!last || h + 1 < h1) stage(last ? h + 1 : h, last ? 0 : b + 1, buf ^ 1);
        // targets [R0, R1) at a time, the next target's rows read before this one's products
        float part[NSLOT][WT];
        auto scores = [&](auto R0, auto R1) __attribute__((always_inline)) {
            constexpr int r0 = decltype(R0)::value, r1 = decltype(R1)::value;
            uint4 kw[2][NSLOT];
            auto fetch = [&](int r) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NSLOT; ++i) kw[r & 1][i] = read_k(kaddr[r][i] + 1024 * buf);
            };
            fetch(r0);
#pragma unroll
            for (int r = r0; r < r1; ++r) {
                if (r + 1 < r1) fetch(r + 1);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (NSLOT == 3) {
                    float a[3];
                    score_dot3(qp[r], kw[r & 1], a);
#pragma unroll
                    for (int i = 0; i < 3; ++i) part[i][r] = a[i];
                } else {
#pragma unroll
                    for (int i = 0; i < NSLOT; ++i) part[i][r] = score_dot(qp[r][i], kw[r & 1][i]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
#pragma unroll
        for (int i = 0; i < NSLOT; ++i)
#pragma unroll
            for (int r = 2; r < WT; ++r) part[i][r] = 0.f;
        scores(I<0>{}, I<2>{});
        if (nt > 2) scores(I<2>{}, I<3>{});
        if (nt > 3) scores(I<3>{}, I<4>{});
        // the first target's values are on their way during the softmax
        uint2 vv[2][2 * NSLOT];
        auto fetch_v = [&](int r) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 2 * NSLOT; ++g) vv[r & 1][g] = read_v4(vaddr[r][g], 2048 + 1024 * buf);
        };
        fetch_v(0);
        __builtin_amdgcn_sched_barrier(0);
        float sc[NSLOT], wt[NSLOT], m;
#pragma unroll
        for (int i = 0; i < NSLOT; ++i) {
            const float t = scaled_score<POW2>(targets_chunk_sum(part[i], lane), p);
            sc[i] = i < NSLOT - 1 || jg + 8 * i < K ? t : -INFINITY;
            m = i == 0 ? sc[0] : fmaxf(m, sc[i]);
        }
        softmax_weights(sc, m, wt);
        put_weights(wt, w_lds + (dc & (WT - 1)) * (KP * 2), jg);
        asm volatile("" ::: "memory");
        // outputs likewise
        auto outputs = [&](auto R0, auto R1) __attribute__((always_inline)) {
            constexpr int r0 = decltype(R0)::value, r1 = decltype(R1)::value;
            uint4 ww[2][NSLOT];
            auto fetch = [&](int r) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NSLOT; ++i) ww[r & 1][i] = *reinterpret_cast<const uint4*>(w_lds + r * (KP * 2) + 16 * i);
                if (r > 0) fetch_v(r);
            };
            fetch(r0);
#pragma unroll
            for (int r = r0; r < r1; ++r) {
                if (r + 1 < r1) fetch(r + 1);
                __builtin_amdgcn_sched_barrier(0);
                const float o = weighted_sum<NSLOT>(ww[r & 1], vv[r & 1]);
                bf16_t* orow = p.out + (((int64_t)tgt[r] * p.B + b) * p.H + h) * 64;  // uniform
                // targets past the wave's last: a store of no lane's
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(orow, (short)0, r < nt ? 128 : 0, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b16((bf16_t)(pack_bf16x2(o, 0.f) & 0xffffu), rs, 2 * lane, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        outputs(I<0>{}, I<2>{});
        if (nt > 2) outputs(I<2>{}, I<3>{});
        if (nt > 3) outputs(I<3>{}, I<4>{});
        // the staging loads are older than the outputs' stores, of which there are two at least
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        __syncthreads();
    };

    int buf = 0;
    for (int h = h0; h < h1; ++h) {
        const QueryRows wr = query_rows(p.w_q + ((int64_t)h * 64 + 8 * dc) * 3);
#pragma unroll
        for (int r = 0; r < WT; ++r)
#pragma unroll
            for (int i = 0; i < NSLOT; ++i) {
                const uint2 rel = reinterpret_cast<const uint2*>(rel_lds)[r * KP + jg + 8 * i];
                query_pairs(wr, rel.x, rel.y, qp[r][i]);
            }
        for (int b = 0; b < p.B; ++b, buf ^= 1) {
            if (buf) pass(h, b, std::integral_constant<int, 1>{});
            else pass(h, b, std::integral_constant<int, 0>{});
        }
    }
}

template <int NSLOT, bool RP>
const void* pick(bool off32, bool pow2) {
    return off32 ? (pow2 ? (const void*)&knn_attn_kernel<NSLOT, true, true, RP> : (const void*)&knn_attn_kernel<NSLOT, true, false, RP>)
                 : (pow2 ? (const void*)&knn_attn_kernel<NSLOT, false, true, RP> : (const void*)&knn_attn_kernel<NSLOT, false, false, RP>);
}

bool knn_off32(const InterpParams& p) {
    // 32-bit chunk offsets when every chunk of a member lies within 4 GiB of its start
    const int64_t kmax = (int64_t)(p.S_from - 1) * p.k_sn + (int64_t)(p.H - 1) * p.k_sh + 64;
    const int64_t vmax = (int64_t)(p.S_from - 1) * p.v_sn + (int64_t)(p.H - 1) * p.v_sh + 64;
    return p.k_sn >= 0 && p.k_sh >= 0 && p.v_sn >= 0 && p.v_sh >= 0 && 2 * kmax <= 0xffffffffLL &&
           2 * vmax <= 0xffffffffLL;
}

template <int NSLOT>
hipError_t launch_slots(const InterpParams& p, unsigned wgs, hipStream_t s) {
    void* args[] = {const_cast<InterpParams*>(&p)};
    const bool off32 = knn_off32(p);
    const void* fn = p.round_products ? pick<NSLOT, true>(off32, p.scale_pow2) : pick<NSLOT, false>(off32, p.scale_pow2);
    return hipLaunchKernel(fn, dim3(wgs), dim3(kInterpWaves * 64), args, 0, s);
}

}  // namespace

hipError_t launch_knn_attn(const InterpParams& p, hipStream_t s) {
    const int64_t pairs = (int64_t)p.S_to * p.H;
    const int64_t wgs = (pairs + kInterpWaves - 1) / kInterpWaves;
    if (wgs <= 0) return hipSuccess;
    if (wgs > 0x7fffffff) return hipErrorInvalidValue;
    switch ((p.K + 7) / 8) {
        case 1: return launch_slots<1>(p, (unsigned)wgs, s);
        case 2: return launch_slots<2>(p, (unsigned)wgs, s);
        case 3: return launch_slots<3>(p, (unsigned)wgs, s);
        case 4: return launch_slots<4>(p, (unsigned)wgs, s);
        default: return hipErrorInvalidValue;
    }
}

// The LDS-staged form: fp32 products with 32-bit chunk offsets only (the caller falls back to
// launch_knn_attn otherwise).
bool knn_tiled_supported(const InterpParams& p) { return !p.round_products && knn_off32(p); }

// Heads per workgroup of the tiled kernel, for a chip with room for slots workgroups at a time.  A
// workgroup's time is its passes (heads times members) and a prologue, the tables' chained loads,
// worth one and a half; the choice is the least product of that with the rounds of workgroups
// (whole ones up to two, above that with a quarter for the uneven end) among groups of at most 48
// passes, above which the prologue no longer counts.  Over 120 shapes (205 to 3878 tiles, 64 to
// 128 rows, 8 to 32 neighbours, 4 to 20 heads, 1 to 24 members) it is within 7 % of the fastest
// group, 0.6 % on average.  us at one head, at the fastest group, at the choice: 3878 tiles, 12 heads,
// one member 332, 194 (12 heads), 194; 24 members 2571, 2469 (3), 2488 (2); 837 tiles of 128 rows,
// 4 heads, one member 43, 32 (4), 32; 205 tiles of 128 rows, 12 heads, one member 31.7, 24.5 (6), 24.5.
static int heads_per_workgroup(int64_t tiles, int H, int B, int slots) {
    int best = 1;
    double least = 0.;
    for (int h = 1; h <= H && (h == 1 || (int64_t)h * B <= 48); ++h) {
        const int groups = (H + h - 1) / h, hg = (H + groups - 1) / groups;  // groups as equal as they get
        const double rounds = (double)(tiles * groups) / slots, whole = ceil(rounds);
        const double cost = (whole <= 2. ? whole : rounds + 0.25) * (1.5 + (double)hg * B);
        if (h == 1 || cost < least) {
            least = cost;
            best = hg;
        }
    }
    return best;
}

hipError_t launch_knn_attn_tiled(const InterpParams& p, const KnnTiles& t, hipStream_t s) {
    if (!knn_tiled_supported(p) || t.rows <= 0 || t.rows % 8 || t.rows > kKnnTileRows) return hipErrorInvalidValue;
    // per row: k and v, two buffers each; then the waves' tables (12 bytes per target and
    // neighbour)
    const size_t lds = 512u * (size_t)t.rows + (size_t)kKnnTileTargets * 8u * ((p.K + 7) / 8) * 12u;
    // three workgroups per CU; two from 25 neighbours on (compiled for two waves per SIMD) and where
    // the LDS holds no third
    const int per_cu = (int)min((size_t)(p.K > 24 ? 2 : 3), (size_t)163840 / lds);
    int hg = heads_per_workgroup(t.n, p.H, p.B, 256 * per_cu);
    const int64_t wgs = (int64_t)t.n * ((p.H + hg - 1) / hg);
    if (wgs <= 0) return hipSuccess;
    if (wgs > 0x7fffffff) return hipErrorInvalidValue;
    void* args[] = {const_cast<InterpParams*>(&p), const_cast<KnnTiles*>(&t), &hg};
    const void* fn = nullptr;
    switch ((p.K + 7) / 8) {
        case 1: fn = p.scale_pow2 ? (const void*)&knn_tile_kernel<1, true> : (const void*)&knn_tile_kernel<1, false>; break;
        case 2: fn = p.scale_pow2 ? (const void*)&knn_tile_kernel<2, true> : (const void*)&knn_tile_kernel<2, false>; break;
        case 3: fn = p.scale_pow2 ? (const void*)&knn_tile_kernel<3, true> : (const void*)&knn_tile_kernel<3, false>; break;
        case 4: fn = p.scale_pow2 ? (const void*)&knn_tile_kernel<4, true> : (const void*)&knn_tile_kernel<4, false>; break;
        default: return hipErrorInvalidValue;
    }
    return hipLaunchKernel(fn, dim3((unsigned)wgs), dim3(kTileWaves * 64), args, lds, s);
}

}  // namespace mosaic
