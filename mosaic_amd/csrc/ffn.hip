// ffn.hip -- cSwiGLU's first projection with the gate in its epilogue (gfx950).
//
// Replaces, for cSwiGLU.forward (primitives.py:92-105), h = w13(x) (a bf16 Linear: fp32
// accumulation, rounded to bf16) followed by the gate with the rounding points of the
// reference's eager bf16 ops (the same ones swiglu_kernel in fused.hip applies):
//   a = bf16(x1 + noise[member]),  s = bf16(a / (1 + exp(-a))),  g = bf16(s * x3)
// for x1, x3 = h.chunk(2): h (two hidden-wide halves per row) is never written or read back.
//
// Tile: 256 rows x 128 hidden indices (their x1 and their x3 rows of w13: 256 weight rows), K in
// iterations of 64, eight waves (2 x 4), one workgroup per CU.  Wave (wm, wn) owns rows 128 ah +
// 64 wm .. + 63 (ah = 0, 1) and hidden indices 32 wn .. + 31, x1 and x3 alike, so both values of a
// pair meet in one lane.  The products are computed transposed (weights as the A operand): a
// lane then holds one row and four consecutive hidden indices per accumulator, so noise is one
// 8-byte read and the output four packed values.
//
// What bounds it: the board's power limit in the main loop (its marginal rate, from two dims: 2340
// TFLOP/s on all-zero operands, 93% of the 2.5 PFLOP/s matrix peak, 1630-1660 on random ones), then the
// vector work of the gate between two tiles: 1200 TFLOP/s over the whole kernel at dim 768, 1300 at
// 1024, 1490 at 3072.  The choices that follow:
//  - v_mfma_f32_16x16x32_bf16 instead of 32x32x16: it reads and writes the fp32 accumulators
//    half as often per product, and under the power limit the same loop runs 1505 -> 1659 TFLOP/s;
//  - ping-pong: the four waves of one row half run half a phase behind the others, so on every
//    SIMD one wave issues LDS reads and loads while the other one feeds the matrix cores;
//  - persistent workgroups: the loads of a tile's first iterations are issued during the tile
//    before it, so no tile starts on an empty pipeline, and the epilogue runs over them;
//  - hardware exp2 and reciprocal in the gate, arranged so that silu rounds to the same bf16 value
//    as with expf and a division for every bf16 argument (gate).
// Measured (24 members, 1,179,648 rows): 768 -> 2 x 3072 in 9.40 ms, against 13.76 ms for the
// library GEMM and the gate kernel (GEMM alone 9.55 ms) and 15.0 ms for a 32x32x16 kernel with
// one barrier per 32-wide step; 1024 -> 2 x 4096 on 294,912 rows 3.86 against 5.27 ms; one member
// (49,152 rows) 389 against 602 us.
#include "bsa_common.h"
#include "mosaic_bsa.h"

namespace mosaic {
namespace {

constexpr int kM = 256;              // rows per tile
constexpr int kHid = 128;            // hidden indices per tile
constexpr int kK = 64;               // reduction step of an iteration
constexpr int kHalf = 128 * kK;      // elements of an operand half in LDS: 128 rows of 128 bytes
constexpr int kStage = 32 * 32;      // elements of a wave's output staging (a 32 x 32 piece)
constexpr int kNoiseRows = 56;       // noise rows staged in LDS (the 160 KB would leave 64)
constexpr int kStores = 8;           // global stores of a wave per tile
constexpr int kWorkgroups = 256;     // one per CU
// Row tiles per group: the group's x rows stay in an XCD's L2 (4 MB) while the weights pass by, and a
// longer group reads the weights less often.  Random operands, 294,912 rows, at 2, 4, 8 and 16 row
// tiles: 1024 -> 2 x 4096 3878, 3801, 3804, 4052 us; 3072 -> 2 x 3072 7645, 7487, 7499, 7602; 1,179,648 rows,
// 768 -> 2 x 3072 9419, 9244, 9249, 9331; 73,728 rows, 1280 -> 2 x 5120 1455, 1437, 1431, 1443.
constexpr int kGroupRows = 8;

struct SwigluLinearParams {
    const bf16_t* x;        // [rows, D], row stride x_sr (elements)
    const bf16_t* w;        // weight rows; tile nt's x1 rows start at row nt * w_tile, 16 rows per wave
    const bf16_t* noise;    // [noise_rows, hidden] contiguous, or null
    bf16_t* out;            // [rows, hidden] contiguous
    int64_t x_sr, rows;
    int64_t w_x3;           // rows from an x1 row to its x3 row
    int w_tile, w_wave1, w_wave2;   // weight row of wave w in a tile: (w / 2) * w_wave2 + (w % 2) * w_wave1
    int D, hidden, noise_rows, n_tiles, row_tiles, tiles;
    uint32_t noise_magic;   // ceil(2^32 / noise_rows): x / noise_rows as a high product
};

__device__ __forceinline__ uint32_t lds_addr(const void* ptr) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)ptr;
}
// Direct-to-LDS load issued as inline assembly: address = base (uniform) + voff (per lane), LDS
// destination M0 + 16 l.  The compiler does not see a load, so it inserts no wait for the loads
// in flight before the LDS reads of other buffers; the kernel counts and waits for them itself.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }
__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// bf16(silu(a)) * b in fp32, for a bf16 value a: a / (1 + exp(-a)) as (a / 4) / (1/4 + exp(-a) / 4).
// For every one of the 65,536 arguments the bf16 value is that of expf and a correctly rounded
// division, which take about 20 vector instructions against these 4: the rounding of a log2 e grows to
// 55 fp32 spacings of the result at a = -88 (3 for |a| < 4), a bf16 spacing is 65,536 of them, and
// no argument's result is that near to where the rounding changes.  The quarters keep the
// reciprocal out of the subnormal range, which the hardware flushes (a from -88.5 to -87.5).  The
// addend is one spacing above 1/4: with 1/4 itself one argument, 5.9375, rounds the other way.
// 768 -> 2 x 3072 on 1,179,648 rows: 9.40 ms; a rcp(1 + exp2(a * -log2 e)), which is wrong for
// these four arguments, 9.28 ms.
__device__ __forceinline__ float gate(float a, float b) {
    const float e = __builtin_amdgcn_exp2f(fmaf(a, -1.44269504088896f, -2.0f));
    return round_bf16(a * 0.25f * __builtin_amdgcn_rcpf(e + 0.25000003f)) * b;
}

// Where a row's noise comes from: none, its slice of the tile's columns staged in LDS (up to
// kNoiseRows rows: the ensemble members), or global memory
enum NoiseMode { kNoNoise = 0, kNoiseLds = 1, kNoiseGlobal = 2 };

template <int NOISE>
__global__ __attribute__((amdgpu_flat_work_group_size(512, 512), amdgpu_waves_per_eu(2, 2)))
void swiglu_linear_kernel(SwigluLinearParams p) {
    // operand halves: x at (2 buffer + half), weights at 4 + (2 buffer + half) (half: the 128-row
    // half ah of x; x1 or x3 of the weights); then the waves' staging, then the noise slice
    __shared__ __attribute__((aligned(1024))) bf16_t S[8 * kHalf + 8 * kStage + (NOISE == kNoiseLds ? kNoiseRows * kHid : 0)];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = w >> 2, wn = w & 3;
    // Each XCD owns a contiguous range of tiles, taken round robin by its workgroups: the ones it
    // runs at one time then share x and weight tiles in its L2.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nslot = gridDim.x >> 3;
    const int per = p.tiles >> 3, rem = p.tiles & 7;
    const int tbeg = xcd * per + min(xcd, rem), tend = tbeg + per + (xcd < rem ? 1 : 0);
    int tile = tbeg + slot;
    if (tile >= tend) return;  // the whole workgroup, before any barrier
    // tiles in groups of kGroupRows row tiles, the row tile varying fastest inside a group
    int rt, nt;
    auto tile_of = [&](int t, int& row_tile, int& col_tile) __attribute__((always_inline)) {
        const int per_group = kGroupRows * p.n_tiles;
        const int grp = t / per_group, within = t - grp * per_group;
        const int rows_here = min(kGroupRows, p.row_tiles - grp * kGroupRows);
        col_tile = within / rows_here;
        row_tile = grp * kGroupRows + (within - col_tile * rows_here);
    };
    // the last row tile of a ragged row count starts early and repeats rows of the one before
    auto first_row = [&](int row_tile) __attribute__((always_inline)) -> int64_t {
        return min((int64_t)row_tile * kM, p.rows - kM);
    };

    // Loads: a half is 128 rows of 128 bytes, two 1 KB runs of 8 rows per wave (rows 16 w + 8 i ..);
    // lane l lands at row l / 8, chunk position l % 8, and fetches chunk position ^ ((row / 2) % 8):
    // 16 lanes of an operand read (16 consecutive rows, one chunk) then cover all banks once.
    uint32_t xo[2], wo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = (lane & 7) ^ (4 * i + (lane >> 4));
        xo[i] = 2u * (uint32_t)((8 * i + (lane >> 3)) * p.x_sr + 8 * c);
        wo[i] = 2u * (uint32_t)((8 * i + (lane >> 3)) * p.D + 8 * c);
    }
    const uint32_t lds0 = lds_addr(S) + 16 * w * 128;
    const int w_row = (w >> 1) * p.w_wave2 + (w & 1) * p.w_wave1;
    const char *xa[2], *wb[2];  // the load cursor: two halves of x and of the weights
    int ltile = tile, lk = 0, lrt, lnt;
    auto load_tile = [&]() __attribute__((always_inline)) {
        tile_of(ltile, lrt, lnt);
        xa[0] = reinterpret_cast<const char*>(p.x + (first_row(lrt) + 16 * w) * p.x_sr);
        xa[1] = xa[0] + 256 * p.x_sr;
        wb[0] = reinterpret_cast<const char*>(p.w + ((int64_t)lnt * p.w_tile + w_row) * p.D);
        wb[1] = wb[0] + 2 * p.w_x3 * p.D;
    };
    auto load_x = [&](int buf, int h) __attribute__((always_inline)) {
        dma16(xa[h], xo[0], lds0 + (2 * buf + h) * kHalf * 2);
        dma16(xa[h], xo[1], lds0 + (2 * buf + h) * kHalf * 2 + 1024);
    };
    auto load_w = [&](int buf, int h) __attribute__((always_inline)) {
        dma16(wb[h], wo[0], lds0 + (4 + 2 * buf + h) * kHalf * 2);
        dma16(wb[h], wo[1], lds0 + (4 + 2 * buf + h) * kHalf * 2 + 1024);
    };
    // next iteration; past a tile's last one the next tile's first (past the last tile: that tile
    // again, loaded and never used, so no wait depends on the position)
    const int T = p.D / kK;
    auto advance = [&]() __attribute__((always_inline)) {
        xa[0] += 2 * kK; xa[1] += 2 * kK; wb[0] += 2 * kK; wb[1] += 2 * kK;
        if (++lk == T) {
            lk = 0;
            if (ltile + nslot < tend) ltile += nslot;
            load_tile();
        }
    };

    // operand reads: row l % 16 of a 16-row block, chunk 4 ds + l / 16 of its 64 k (ds = 0, 1)
    const int r16 = lane & 15, q4 = lane >> 4;
    int rd[2];
#pragma unroll
    for (int ds = 0; ds < 2; ++ds) rd[ds] = r16 * kK + 8 * ((4 * ds + q4) ^ ((r16 >> 1) & 7));
    bf16x8 a[4][2], b0[2][2], b1[2][2];  // x: 16-row blocks; weights: 16-index blocks
    auto read_x = [&](int buf, int h) __attribute__((always_inline)) {
        const bf16_t* A = S + (2 * buf + h) * kHalf + 64 * wm * kK;
#pragma unroll
        for (int ds = 0; ds < 2; ++ds)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) a[mt][ds] = as_bf16x8(*reinterpret_cast<const uint4*>(A + 16 * mt * kK + rd[ds]));
    };
    auto read_w = [&](bf16x8 (&b)[2][2], int buf, int h) __attribute__((always_inline)) {
        const bf16_t* B = S + (4 + 2 * buf + h) * kHalf + 32 * wn * kK;
#pragma unroll
        for (int ds = 0; ds < 2; ++ds)
#pragma unroll
            for (int nn = 0; nn < 2; ++nn) b[nn][ds] = as_bf16x8(*reinterpret_cast<const uint4*>(B + 16 * nn * kK + rd[ds]));
    };
    f32x4 acc[2][4][2][2];  // [row half][16-row block][16-index block][x1, x3]
    auto products = [&](int ah, const bf16x8 (&b)[2][2], int h) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ds = 0; ds < 2; ++ds)
#pragma unroll
            for (int nn = 0; nn < 2; ++nn)
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) acc[ah][mt][nn][h] = mfma16(b[nn][ds], a[mt][ds], acc[ah][mt][nn][h]);
        __builtin_amdgcn_sched_barrier(0);
    };
    // End of a memory phase: this wave's reads are in registers and its loads of the half that the
    // next phase reads have landed; after the barrier every wave's have.  Halves are loaded in the
    // order x1 weights, x rows 0-127, x3 weights, x rows 128-255, two loads each, about seven phases
    // before they are read, and five halves (ten loads) are newer than the one waited for.  In the
    // five phases after an epilogue its stores are among the newer operations too (the counter
    // retires in order); any further operation in between only makes the wait stricter.
    auto end_memory = [&](bool after_stores) __attribute__((always_inline)) {
        if (after_stores) wait_vmem<10 + kStores>();
        else wait_vmem<10>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        barrier();
    };
    // The tile's noise: row n of the members at 256 n bytes, 16-byte chunk c at position c ^ (n % 16)
    const bf16_t* noise_lds = S + 8 * kHalf + 8 * kStage;
    auto load_noise = [&]() __attribute__((always_inline)) {
        if constexpr (NOISE == kNoiseLds) {
#pragma unroll
            for (int i = 0; i < (kNoiseRows + 31) / 32; ++i) {
                const int n0 = 4 * (8 * i + w), n = n0 + q4;
                if (n0 < p.noise_rows)  // uniform; noise_rows <= kNoiseRows
                    dma16(p.noise + (int64_t)nt * kHid,
                          2u * (uint32_t)(min(n, p.noise_rows - 1) * p.hidden + 8 * (r16 ^ (n & 15))),
                          lds_addr(noise_lds) + 256 * n0);
            }
        }
    };

    load_tile();
    rt = lrt;
    nt = lnt;
    load_x(0, 0); load_w(0, 0); load_w(0, 1); load_x(0, 1); advance();
    load_w(1, 0); load_x(1, 0); load_w(1, 1);
    wait_vmem<6>();  // iteration 0 is in LDS
    barrier();
    if (wm == 1) barrier();  // the second row group runs half a phase behind
    bool stored = false;     // stores of the tile before may be in flight
    for (;;) {
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i >> 4][(i >> 2) & 3][(i >> 1) & 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
        read_w(b0, 0, 0);
        // Two iterations per round (buffers 0 and 1; T is even).  A phase is a memory part (the
        // operands of this phase's products, the loads of a half two iterations ahead into the
        // space read last) and 16 products of 64 rows x 32 indices x 64 k.  Over the four phases
        // of an iteration the products go (rows 0, x1), (rows 0, x3), (rows 1, x3), (rows 1, x1).
        for (int t = 0; t < T; t += 2) {
            const bool f = stored && t == 0;
            read_x(0, 0); load_x(1, 1); advance(); end_memory(f); products(0, b0, 0); barrier();
            // every wave is past the epilogue before: its noise slice may be replaced
            if (t == 0) load_noise();
            read_w(b1, 0, 1); load_w(0, 0); end_memory(f); products(0, b1, 1); barrier();
            read_x(0, 1); load_x(0, 0); end_memory(f); products(1, b1, 1); barrier();
            read_w(b1, 1, 0); load_w(0, 1); end_memory(f); products(1, b0, 0); barrier();
            read_x(1, 0); load_x(0, 1); advance(); end_memory(f); products(0, b1, 0); barrier();
            read_w(b0, 1, 1); load_w(1, 0); end_memory(false); products(0, b0, 1); barrier();
            read_x(1, 1); load_x(1, 0); end_memory(false); products(1, b0, 1); barrier();
            read_w(b0, 0, 0); load_w(1, 1); end_memory(false); products(1, b1, 0); barrier();
        }
        wait_vmem<6>();  // the next tile's first iteration (and this tile's noise) are in LDS
        barrier();

        // Epilogue: lane l holds row 16 mt + l % 16 of a 64-row block and hidden indices
        // 16 nn + 4 (l / 16) .. + 3.  Each 32 x 32 piece goes through the wave's staging (64-byte
        // rows, 16-byte chunk c at c ^ ((row / 4) % 4)) and leaves as whole 64-byte rows.
        const int64_t row0 = first_row(rt);
        uint32_t base = 0;
        if constexpr (NOISE != kNoNoise) base = (uint32_t)(row0 % p.noise_rows);
        char* ob = reinterpret_cast<char*>(p.out + row0 * p.hidden + nt * kHid + 32 * wn);
        bf16_t* stg = S + 8 * kHalf + kStage * w;
#pragma unroll
        for (int ah = 0; ah < 2; ++ah)
#pragma unroll
            for (int m2 = 0; m2 < 2; ++m2) {
                const int piece = 128 * ah + 64 * wm + 32 * m2;  // first row in the tile
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    uint2 nz[2];
                    if constexpr (NOISE != kNoNoise) {
                        const uint32_t x = base + piece + 16 * m + r16;
                        if constexpr (NOISE == kNoiseLds) {
                            // x mod noise_rows (one row: the high product is x - 1, hence the clamp)
                            const uint32_t n = min(x - p.noise_rows * __umulhi(x, p.noise_magic), (uint32_t)p.noise_rows - 1u);
#pragma unroll
                            for (int nn = 0; nn < 2; ++nn)
                                nz[nn] = ld8(noise_lds + n * kHid + 8 * ((4 * wn + 2 * nn + (q4 >> 1)) ^ (n & 15)) + 4 * (q4 & 1));
                        } else {
                            const int64_t n = x % (uint32_t)p.noise_rows;
#pragma unroll
                            for (int nn = 0; nn < 2; ++nn)
                                nz[nn] = ld8(p.noise + n * p.hidden + nt * kHid + 32 * wn + 16 * nn + 4 * q4);
                        }
                    }
#pragma unroll
                    for (int nn = 0; nn < 2; ++nn) {
                        const float nv[4] = {bf_lo(nz[nn].x), bf_hi(nz[nn].x), bf_lo(nz[nn].y), bf_hi(nz[nn].y)};
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float x1 = round_bf16(acc[ah][2 * m2 + m][nn][0][e]);
                            if constexpr (NOISE != kNoNoise) x1 = round_bf16(x1 + nv[e]);
                            v[e] = gate(x1, round_bf16(acc[ah][2 * m2 + m][nn][1][e]));
                        }
                        const int row = 16 * m + r16, c = 2 * nn + (q4 >> 1);
                        *reinterpret_cast<uint2*>(stg + row * 32 + 8 * (c ^ ((row >> 2) & 3)) + 4 * (q4 & 1)) =
                            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                    }
                }
                // only this wave touches its staging, and its LDS operations complete in order
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int row = 16 * i + (lane >> 2), c = lane & 3;
                    *reinterpret_cast<uint4*>(ob + 2 * ((int64_t)(piece + row) * p.hidden + 8 * c)) =
                        *reinterpret_cast<const uint4*>(stg + row * 32 + 8 * (c ^ ((row >> 2) & 3)));
                }
                __builtin_amdgcn_wave_barrier();
            }
        tile += nslot;
        if (tile >= tend) break;
        rt = lrt;  // the load cursor is in this tile's second iteration
        nt = lnt;
        stored = true;
    }
    if (wm == 0) barrier();  // the second group's last barrier
    wait_vmem<0>();          // no load may land in LDS after the workgroup has ended
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// permuted: the weight's 64-row groups hold 32 x1 rows, then the same 32 x3 rows
int swiglu_linear(const void* x, int64_t rows, int32_t dim, int64_t x_row_stride, const void* weight, bool permuted,
                  int32_t hidden, const void* noise, int32_t noise_rows, void* out, void* stream) {
    if (rows <= 0 || dim <= 0 || hidden <= 0) return MOSAIC_ERR_SHAPE;
    if (!x || !weight || !out) return MOSAIC_ERR_NULL_POINTER;
    if (noise && noise_rows <= 0) return MOSAIC_ERR_SHAPE;
    if (rows < kM || (permuted && rows % kM) || dim % (2 * kK) || hidden % kHid) return MOSAIC_ERR_UNSUPPORTED;
    if (x_row_stride < dim || x_row_stride % 8) return MOSAIC_ERR_ALIGNMENT;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(out) || (noise && !aligned16(noise)))
        return MOSAIC_ERR_ALIGNMENT;
    // byte offsets within a wave's 16 rows of x or w13 are 32-bit
    if (x_row_stride >= ((int64_t)1 << 26) || dim >= (1 << 26)) return MOSAIC_ERR_UNSUPPORTED;
    const int64_t row_tiles = (rows + kM - 1) / kM, n_tiles = hidden / kHid;
    if (row_tiles > 0x7fffffff / n_tiles / 8) return MOSAIC_ERR_SHAPE;
    SwigluLinearParams p{};
    p.x = static_cast<const bf16_t*>(x);
    p.w = static_cast<const bf16_t*>(weight);
    p.noise = static_cast<const bf16_t*>(noise);
    p.out = static_cast<bf16_t*>(out);
    p.x_sr = x_row_stride;
    p.rows = rows;
    p.w_x3 = permuted ? 32 : hidden;
    p.w_tile = permuted ? 2 * kHid : kHid;
    p.w_wave1 = 16;
    p.w_wave2 = permuted ? 64 : 32;
    p.D = dim;
    p.hidden = hidden;
    p.noise_rows = noise ? noise_rows : 1;
    p.noise_magic = p.noise_rows > 1 ? (uint32_t)((((uint64_t)1 << 32) + p.noise_rows - 1) / p.noise_rows) : 0xffffffffu;
    p.n_tiles = (int)n_tiles;
    p.row_tiles = (int)row_tiles;
    p.tiles = (int)(row_tiles * n_tiles);
    const void* fn = !noise ? (const void*)&swiglu_linear_kernel<kNoNoise>
                   : noise_rows <= kNoiseRows && hidden < (1 << 25)  // byte offsets of the staged rows are 32-bit
                       ? (const void*)&swiglu_linear_kernel<kNoiseLds>
                       : (const void*)&swiglu_linear_kernel<kNoiseGlobal>;
    const int grid = p.tiles >= kWorkgroups ? kWorkgroups : (p.tiles + 7) / 8 * 8;
    void* args[] = {&p};
    const hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(512), args, 0, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? MOSAIC_OK : MOSAIC_ERR_LAUNCH;
}

}  // namespace
}  // namespace mosaic

using namespace mosaic;

extern "C" {

int mosaic_swiglu_linear_fwd(const void* x, int64_t rows, int32_t dim, int64_t x_row_stride, const void* weight,
                             int32_t hidden, const void* noise, int32_t noise_rows, void* out, void* stream) {
    return swiglu_linear(x, rows, dim, x_row_stride, weight, true, hidden, noise, noise_rows, out, stream);
}

int mosaic_swiglu_linear_w13_fwd(const void* x, int64_t rows, int32_t dim, int64_t x_row_stride, const void* w13,
                                 int32_t hidden, const void* noise, int32_t noise_rows, void* out, void* stream) {
    return swiglu_linear(x, rows, dim, x_row_stride, w13, false, hidden, noise, noise_rows, out, stream);
}

}  // extern "C"
