// p8x_gemv_mx.hip -- single-call GEMV on the matrix cores: 2..8 multiplied columns of 8-bit-per-128 activations (x16:
// two planes per column), or 1..8 columns of block_q8_1, any class.
//
// A tile's integer products for all columns are a small matrix product that v_mfma_i32_32x32x32_i8 computes exactly:
// the looked-up codewords are the B operand (n = row = lane & 31), the activations the A operand (m = column). One MFMA
// takes 32 columns of K: for 32-block i of a half, lane (row j, half hs) looks up its chunks 8 i .. 8 i + 7 and one
// v_permlane32_swap per pair (8 i + e, 8 i + 4 + e) turns the two halves' words into per-half operands (lanes 0..31
// chunks 8 i .. + 3, lanes 32..63 chunks 8 i + 4 .. + 7), so each MFMA is one block_q8_1 block of one half, and the four
// of a half add up to its 128-column sum. Multi-stage classes add their stages Horner-wise (the stage shifts fall on
// the four accumulator registers that hold columns). Output lane (row j, group g) holds columns 4 g .. 4 g + 3.
//
// The work is split as the row-group GEMV splits it: a workgroup takes whole 32-row groups over its K-chunk, builds
// the coset table, quantizes (or copies) its chunk of the activations into LDS, its waves split the chunk into block
// ranges, and the partial rows meet in LDS in wave order. The products, the x16 planes' sum, the clamp delta and the row
// permutation happen in one launch. Bound by latency (launch, table, one to three tiles per wave), not by the weights:
// 14336 x 4096, class 3, four columns 15.7 -> 10.4 us a call against the dot kernel; 2560 x 9728, ffn_down mix, seven
// columns 33.0 -> 14.5; x16 4096 x 14336 mix 19.4 -> 12.4 (prep, GEMV and plane sum were three launches); block_q8_1 4096 x
// 4096 9.5 -> 7.6. Error against 64 bits 0.6 to 0.9 of the dot kernel's (one fused step fewer per product, the waves' sums
// in 64 bits).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "p8x_gemv.h"

namespace p8x {

struct MxJob {
    const uint32_t *M; const uint16_t *Sg; const uint32_t *D; const uint32_t *a2;
    const uint16_t *prmd;
    const int *cp; const uint16_t *cc; const float *cv;
    const void *q; const float *d;    // prepared activations (q8: int8 [ncv][K] + f32 [ncv][nsl]; block_q8_1 [ncv][K / 32]), or null
    const float *ic;
    const float *x; unsigned ldx;     // original activations (quantized here when q is null; clamp delta), may be null with q
    float *y; unsigned ldy;
    float *wpart; unsigned *wcnt; unsigned long long *wslot;
    int rows, K, nb, ng, nsl;
    int ncols, planes;                // output columns; planes 2: x16, column n is multiplied columns 2 n and 2 n + 1
    int nks, kchunk, gc;
    uint32_t dbytes, sbytes;
};

// LDS: coset table | activation records | scales | partial rows. A record is one (block, column): its 256 int8 in order,
// at a stride of 272 bytes, so that the 16-byte operand reads of the eight columns fall on different banks.
constexpr int kMxRecs = 240, kMxRecStride = 272, kMxBlocks = 64;
__host__ __device__ constexpr int mxs_waves() { return 16; }
template <int ACT>
struct MxsSmem {
    static constexpr int kSub = ACT == P8X_ACT_Q8_128 ? 2 : 8;   // scales per block and column
    uint32_t tab[kTabWords];                            // LDS address 0
    uint8_t rec[kMxRecs * kMxRecStride];
    float xd[kMxBlocks * kSub * 8];                     // [block][half and 32-block][column]
    float red[mxs_waves()][8][32];                      // [wave][column][row]
};

template <int ACT, int C, int NC>
__device__ __forceinline__ void mxs_tile(const MxsSmem<ACT> &sm, const QuadSlice<C> &p, uint32_t bankbytes, const uint8_t *arec, const float *xd,
                                         int g, float (&ya)[2][NC]) {
    constexpr int NST = nstage_of(C), SH1 = sh1_of(C), SH2 = sh2_of(C);
    const uint32_t H = p.coset_bits();
    const float sc = half_to_float(p.s);
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    // codewords of stage S, 32-block i, as the operands of both halves; then one MFMA per half
    auto products = [&](auto stage, int i, i32x16_t (&acc)[2]) {
        constexpr int S = decltype(stage)::value;
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = lds_word(sm.tab, p.template addr<S>(8 * i + e, coset_bytes(H, bankbytes, 2 * i + (e >> 2))));
        i32x4 b0, b1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const auto sw = __builtin_amdgcn_permlane32_swap(w[e], w[e + 4], false, false);
            b0[e] = (int)sw[0];
            b1[e] = (int)sw[1];
        }
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const i32x4 *>(arec + 32 * i), b0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(*reinterpret_cast<const i32x4 *>(arec + 128 + 32 * i), b1, acc[1], 0, 0, 0);
        __asm__ volatile("" ::: "memory");   // one 32-block at a time: bounds the live registers
    };
    auto shift = [&](i32x16_t (&acc)[2], int n) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[h][c] = (int)((uint32_t)acc[h][c] << n);
    };
    auto scale = [&](const i32x16_t (&acc)[2], int sub0, int substep) {   // y_h += ((float)isum d) S, the last two steps rounded once
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float *dp = xd + (sub0 + h * substep) * 8 + 4 * g;
#pragma unroll
            for (int c = 0; c < NC; ++c) ya[h][c] = __builtin_fmaf((float)acc[h][c] * dp[c], sc, ya[h][c]);
        }
    };
    constexpr auto s0 = std::integral_constant<int, 0>{};
    constexpr auto s1 = std::integral_constant<int, (NST > 1 ? 1 : 0)>{};
    constexpr auto s2 = std::integral_constant<int, (NST > 2 ? 2 : 0)>{};
    if constexpr (ACT == P8X_ACT_Q8_128) {
        i32x16_t acc[2] = {i32x16_t{}, i32x16_t{}};
#pragma unroll
        for (int i = 0; i < 4; ++i) products(s0, i, acc);
        if constexpr (NST > 1) {
            shift(acc, SH1 - SH2);
#pragma unroll
            for (int i = 0; i < 4; ++i) products(s1, i, acc);
        }
        if constexpr (NST > 2) {
            shift(acc, SH2);
#pragma unroll
            for (int i = 0; i < 4; ++i) products(s2, i, acc);
        }
        static_assert(NST > 1 || SH1 == 0, "the last stage is not shifted");
        scale(acc, 0, 1);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            i32x16_t acc[2] = {i32x16_t{}, i32x16_t{}};
            products(s0, i, acc);
            if constexpr (NST > 1) { shift(acc, SH1 - SH2); products(s1, i, acc); }
            if constexpr (NST > 2) { shift(acc, SH2); products(s2, i, acc); }
            scale(acc, i, 4);
        }
    }
}

// Spilled registers at 128: all classes 12 and 15 (q8, x16) and 2 to 12 (block_q8_1), classes 2-4 and 6 with NC 4 of q8 4,
// class 3 with NC 2 of block_q8_1 7; the other instantiations none.
// NC: columns a lane group holds (1, 2 or 4; 4 for more than two multiplied columns, the second group columns 4 .. 7)
template <int ACT, int CM, int NC>
__global__ __launch_bounds__(64 * mxs_waves()) __attribute__((amdgpu_waves_per_eu(mxs_waves() / 4, mxs_waves() / 4)))
void k_gemv_mx(MxJob J) {
    constexpr int WAVES = mxs_waves(), NT = 64 * WAVES, NQ = CM == kCmC3 || CM == kCmC234 ? 2 : CM == kCmC2346 ? 4 : 6, SUB = MxsSmem<ACT>::kSub;
    __shared__ MxsSmem<ACT> sm;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, hs = lane >> 5;
    const uint32_t bankbytes = (uint32_t)(j << 2) * 0x01010101u;
    const int ncv = J.ncols * J.planes;
    // workgroup b: K-chunk b % nks of row groups b / nks, + gstep, ...; its waves form gc teams of wpg
    const int ks = (int)blockIdx.x % J.nks, gfirst = (int)blockIdx.x / J.nks, gstep = (int)gridDim.x / J.nks;
    const int c0 = ks * J.kchunk, nbk = min(J.kchunk, J.nb - c0);
    const int wpg = WAVES / J.gc, team = w / wpg, wk = w % wpg;
    const int per = nbk / wpg, rem = nbk % wpg;
    const int b0 = c0 + wk * per + min(wk, rem), b1 = team < J.gc ? b0 + per + (wk < rem ? 1 : 0) : b0;
    // the first activations, the table and the wave's first tile, in the order they are needed
    const int items = J.ncols * nbk;
    BlockLane in{};
    if (!J.q && w < items) {   // the wave's one block to quantize (kMxInline)
        const int n = w / nbk, b = c0 + w % nbk;
        in.load(J.x + (size_t)n * J.ldx + 256 * b, J.ic + 256 * b, lane);
    }
    CosetTableFill<NT> fill;
    fill.load(J.a2, tid);
    using Raw = std::conditional_t<CM == kCmC3, QuadSlice<3>, AnyQuads<NQ>>;
    Raw nxt;
    uint32_t cn = 3;
    const __amdgpu_buffer_rsrc_t rd = buffer_rsrc(J.D, J.dbytes), rs = buffer_rsrc(J.Sg, J.sbytes);
    auto issue = [&](int g, int b) {   // past the tensor: its last tile, loaded and never used
        const int gi = min(g, J.ng - 1), bi = min(b, J.nb - 1);
        const uint32_t mt = as_const(J.M)[(size_t)gi * J.nb + bi];
        const uint32_t toff = (mt & 0x1FFFFFFFu) * 4u, soff = ((uint32_t)gi * (uint32_t)J.nb + (uint32_t)bi) * 64u;
        if constexpr (CM == kCmC3) {
            nxt.load(rd, toff, QuadSlice<3>::quad_offset(hs, j), 0u, rs, soff, 2u * j);
        } else {
            cn = mt >> 29;
            nxt.load(rd, toff, nw_run(cn), hs, j, rs, soff, 2u * j);
        }
    };
    int g = gfirst + min(team, J.gc - 1) * gstep;
    __asm__ volatile("" ::: "memory");
    issue(g, b0);
    __asm__ volatile("" ::: "memory");
    fill.store(sm.tab, tid);
    if (J.q) {   // prepared activations: 16-byte pieces of the records, then the scales
        if constexpr (ACT == P8X_ACT_Q8_128) {
            for (int i = tid; i < ncv * nbk * 16; i += NT) {
                const int r = i >> 4, bl = r / ncv, n = r % ncv;
                *reinterpret_cast<u32x4_t *>(sm.rec + r * kMxRecStride + 16 * (i & 15)) =
                    as_global(reinterpret_cast<const u32x4_t *>((const int8_t *)J.q + (size_t)n * J.K + 256 * (c0 + bl)))[i & 15];
            }
            for (int i = tid; i < ncv * nbk * 2; i += NT) {
                const int n = i / (2 * nbk), k = i % (2 * nbk);
                sm.xd[k * 8 + n] = as_global(J.d)[(size_t)n * J.nsl + 2 * c0 + k];
            }
        } else {
            for (int i = tid; i < ncv * nbk * 64; i += NT) {
                const int r = i >> 6, bl = r / ncv, n = r % ncv, wi = i & 63;
                const uint8_t *blk = (const uint8_t *)J.q + ((size_t)n * (J.K / 32) + 8 * (c0 + bl) + (wi >> 3)) * 36;
                *reinterpret_cast<uint32_t *>(sm.rec + r * kMxRecStride + 4 * wi) = as_global(reinterpret_cast<const uint32_t *>(blk + 4))[wi & 7];
                if ((wi & 7) == 0) sm.xd[(8 * bl + (wi >> 3)) * 8 + n] = half_to_float(*as_global(reinterpret_cast<const uint16_t *>(blk)));
            }
        }
    } else if (w < items) {   // one wave per (column, block)
        const int n = w / nbk, bl = w % nbk;
        uint8_t *r0 = sm.rec + (bl * ncv + n * J.planes) * kMxRecStride + 4 * lane;
        if constexpr (ACT == P8X_ACT_Q8_1) {
            uint32_t packed;
            float dd, s;
            quantize_loaded_q8_1(in, lane, packed, dd, s);
            *reinterpret_cast<uint32_t *>(r0) = packed;
            if ((lane & 7) == 0) sm.xd[(8 * bl + (lane >> 3)) * 8 + n] = half_to_float(float_to_half(dd));   // as the block stores it
        } else if (J.planes == 2) {
            uint32_t hi, lo;
            float dd;
            quantize_loaded_x16(in, lane, hi, lo, dd);
            *reinterpret_cast<uint32_t *>(r0) = hi;
            *reinterpret_cast<uint32_t *>(r0 + kMxRecStride) = lo;
            if (j == 0) {
                sm.xd[(2 * bl + hs) * 8 + 2 * n] = 128.f * dd;
                sm.xd[(2 * bl + hs) * 8 + 2 * n + 1] = dd;
            }
        } else {
            uint32_t packed;
            float dd;
            int qs;
            quantize_loaded_q8_128(in, lane, packed, dd, qs);
            *reinterpret_cast<uint32_t *>(r0) = packed;
            if (j == 0) sm.xd[(2 * bl + hs) * 8 + n] = dd;
        }
    }
    __syncthreads();
    // operand row of this lane: its column's record (rows of A past the columns repeat them; their products are not used)
    const uint8_t *arow = sm.rec + min(lane & 7, ncv - 1) * kMxRecStride + 16 * hs;
    for (int g0 = gfirst; g0 < J.ng; g0 += gstep * J.gc, g += gstep * J.gc) {
        const bool active = team < J.gc && g < J.ng;
        float ya[2][NC];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int c = 0; c < NC; ++c) ya[h][c] = 0.f;
        if (active)
            for (int b = b0; b < b1; ++b) {
                Raw cur = nxt;
                const uint32_t c = cn;
                const bool last = b + 1 == b1;
                issue(last ? g + gstep * J.gc : g, last ? b0 : b + 1);
                __asm__ volatile("" ::: "memory");
                pin(cur.w);
                const uint8_t *ar = arow + (b - c0) * ncv * kMxRecStride;
                const float *xd = sm.xd + (b - c0) * SUB * 8;
                auto tile = [&](const auto &p) { mxs_tile<ACT>(sm, p, bankbytes, ar, xd, hs, ya); };
                if constexpr (CM == kCmC3) {
                    tile(cur);
                } else {
                    switch (c) {
                        case 1: if constexpr ((CM >> 1) & 1) tile(cur.template as<1>()); break;
                        case 2: if constexpr ((CM >> 2) & 1) tile(cur.template as<2>()); break;
                        case 3: if constexpr ((CM >> 3) & 1) tile(cur.template as<3>()); break;
                        case 4: if constexpr ((CM >> 4) & 1) tile(cur.template as<4>()); break;
                        case 5: if constexpr ((CM >> 5) & 1) tile(cur.template as<5>()); break;
                        case 6: if constexpr ((CM >> 6) & 1) tile(cur.template as<6>()); break;
                        case 7: if constexpr ((CM >> 7) & 1) tile(cur.template as<7>()); break;
                        default: break;   // class 0: zero weights
                    }
                }
            }
#pragma unroll
        for (int c = 0; c < NC; ++c) sm.red[w][4 * hs + c][j] = ya[0][c] + ya[1][c];
        __syncthreads();
        // (row, output column) pairs of the team's row group: wave k of the team takes columns 2 k, 2 k + 1 first; in
        // a K split that counts arrivals the team's first wave takes them all
        const bool pairs = J.nks == 2 && J.ncols == 1, counted = J.nks > 1 && !pairs;
        // the waves' partial rows, summed in 64 bits and rounded once: a wave often has one tile, so in 32 bits this sum
        // of up to 16 terms (32 for x16, both planes) was most of a call's rounding
        auto rowsum = [&](int col) {
            double v = 0.0;
            for (int k0 = 0; k0 < wpg; k0 += 4) {   // four reads in flight, added in wave order
                float pv[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) pv[k] = sm.red[team * wpg + min(k0 + k, wpg - 1)][col][j];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k0 + k < wpg) v += (double)pv[k];
            }
            return v;
        };
        auto finish = [&](int n, float v) {   // clamp delta on the original activations, original row
            const int ro = as_global(J.prmd)[32 * g + j], r = ro & 0x7FFF;
            if ((ro & 0x8000) && J.x) {
                const gptr<const float> xr = as_global(J.x) + (size_t)n * J.ldx;
                for (int e = as_global(J.cp)[r]; e < as_global(J.cp)[r + 1]; ++e) v += as_global(J.cv)[e] * xr[as_global(J.cc)[e]];
            }
            as_global_rw(J.y)[(size_t)n * J.ldy + r] = v;
        };
        if (active && (!counted || wk == 0)) {
            const gptr<float> wpart = as_global_rw(J.wpart);
            for (int n = hs + (counted ? 0 : 2 * wk); n < J.ncols; n += counted ? 2 : 2 * wpg) {
                const float v = (float)(J.planes == 2 ? rowsum(2 * n) + rowsum(2 * n + 1) : rowsum(n));
                if (counted) {
                    __hip_atomic_store(&wpart[((size_t)ks * J.ncols + n) * J.rows + 32 * g + j], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else if (pairs) {   // the row's two K-halves meet in its slot; chunk 0 + chunk 1 either way
                    int oi;
                    float other;
                    if (pair_meet(as_global_rw(J.wslot) + 32 * g + j, ks, v, oi, other)) finish(n, ks == 0 ? v + other : other + v);
                } else {
                    finish(n, v);
                }
            }
            if (counted && arrive_after_stores(J.wcnt + g, lane) == (unsigned)(J.nks - 1)) {   // the last chunk sums them in order
                for (int n = hs; n < J.ncols; n += 2) {
                    float v = 0.f;
                    for (int k0 = 0; k0 < J.nks; k0 += 4) {
                        float pv[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            pv[k] = __hip_atomic_load(&wpart[((size_t)min(k0 + k, J.nks - 1) * J.ncols + n) * J.rows + 32 * g + j], __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (k0 + k < J.nks) v += pv[k];
                    }
                    finish(n, v);
                }
                if (lane == 0) __hip_atomic_store(as_global_rw(J.wcnt) + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();   // red is written again in the next round
    }
}

// K-chunks: a chunk's records fit LDS; two when the row groups fill at most half the CUs and K is long
int mx_plan(const p8x_tensor *t, int ncv, int *kc) {
    const int kmax = std::min(kMxBlocks, kMxRecs / ncv);
    int nks = (t->nb + kmax - 1) / kmax;
    if (nks == 1 && 2 * t->ng <= num_cus() && t->nb >= 32) nks = 2;
    *kc = (t->nb + nks - 1) / nks;
    return (t->nb + *kc - 1) / *kc;
}

size_t mx_part_floats(const p8x_tensor *t, int ncols, int planes) {
    int kc;
    const int nks = mx_plan(t, ncols * planes, &kc);
    return nks == 1 || (nks == 2 && ncols == 1) ? 0 : (size_t)nks * ncols * t->rows;
}

template <int ACT, int CM>
static void launch_mx_nc(const MxJob &J, int grid, hipStream_t st) {
    const int ncv = J.ncols * J.planes;
    if (ACT == P8X_ACT_Q8_1 && ncv == 1) hipLaunchKernelGGL((k_gemv_mx<ACT, CM, ACT == P8X_ACT_Q8_1 ? 1 : 2>), dim3(grid), dim3(64 * mxs_waves()), 0, st, J);
    else if (ncv == 2) hipLaunchKernelGGL((k_gemv_mx<ACT, CM, 2>), dim3(grid), dim3(64 * mxs_waves()), 0, st, J);
    else hipLaunchKernelGGL((k_gemv_mx<ACT, CM, 4>), dim3(grid), dim3(64 * mxs_waves()), 0, st, J);
}

template <int ACT>
static void launch_mx_cm(int cm, const MxJob &J, int grid, hipStream_t st) {
    if (cm == kCmC3) launch_mx_nc<ACT, kCmC3>(J, grid, st);
    else if (cm == kCmC234) launch_mx_nc<ACT, kCmC234>(J, grid, st);
    else if (cm == kCmC6 || cm == kCmC2346) launch_mx_nc<ACT, kCmC2346>(J, grid, st);
    else launch_mx_nc<ACT, kCmAll>(J, grid, st);
}

constexpr int kMxInline = mxs_waves();   // blocks a workgroup quantizes itself

int launch_gemv_mx(const p8x_tensor *t, int act, const void *q, const float *d, int ncols, int planes, const float *x, size_t ldx, float *y, size_t ldy,
                   hipStream_t st) {
    MxJob J{};
    J.nks = mx_plan(t, ncols * planes, &J.kchunk);
    const size_t need = mx_part_floats(t, ncols, planes);
    // Quantized by every workgroup where each wave has at most one block of it, else once by a launch of its own: a
    // second block per wave costs as much as the launch, a third and fourth more (4096 x 4096, four columns: 9.0 us with
    // the launch, 12.2 us without; x16, one column: 7.8 us without).
    if (!q && ncols * J.kchunk > kMxInline) {
        int rc;
        if (act == P8X_ACT_Q8_1) {
            rc = launch_act_q8_1(t, x, ncols, ldx, t->wq81, st);
            q = t->wq81;
        } else {
            rc = planes == 2 ? launch_act_x16(t, x, ncols, ldx, t->wq, t->wd, nullptr, t->wq + t->K, t->wd + t->nsl, nullptr, 2 * t->K, st)
                             : launch_act_q8_128(t, x, ncols, ldx, t->wq, t->wd, nullptr, st);
            q = t->wq;
            d = t->wd;
        }
        if (rc) return rc;
    }
    if (need > t->wpart_floats) return set_error(P8X_ERR_UNSUPPORTED, "gemv: partial workspace too small");
    J.M = t->M; J.Sg = t->Sg; J.D = t->D; J.a2 = t->a2; J.prmd = t->prmd;
    J.cp = t->cp; J.cc = t->cc; J.cv = t->cv;
    J.q = q; J.d = d; J.ic = t->ic; J.x = x; J.ldx = (unsigned)ldx; J.y = y; J.ldy = (unsigned)ldy;
    J.wpart = t->wpart; J.wcnt = t->wcnt; J.wslot = t->wslot;
    J.rows = t->rows; J.K = t->K; J.nb = t->nb; J.ng = t->ng; J.nsl = t->nsl; J.ncols = ncols; J.planes = planes;
    J.dbytes = (uint32_t)(t->kbytes - offset_D(t->nt));
    J.sbytes = (uint32_t)t->nb * (uint32_t)t->rows * 2u;
    const int per = (t->ng * J.nks + num_cus() - 1) / num_cus();   // row groups per workgroup (one workgroup per CU)
    J.gc = std::min(per, 4);
    const int grid = (t->ng + per - 1) / per * J.nks;
    const int cm = class_set(t->class_tiles);
    if (act == P8X_ACT_Q8_1) launch_mx_cm<P8X_ACT_Q8_1>(cm, J, grid, st);
    else launch_mx_cm<P8X_ACT_Q8_128>(cm, J, grid, st);
    return hip_check(hipGetLastError(), "k_gemv_mx launch");
}

}  // namespace p8x
