// p8x_mm_rg.hip -- prompt GEMM of few tokens (1 .. 64): Y [N][rows] = X [N][K] W^T in one pass over the weights.
//
// The products are those of p8x_gemm.hip (x' = FWHT(x ic) / 16 in fp16, weights v S rounded once to fp16, fp32 sums on
// v_mfma_f32_32x32x16_f16); the work is split as the row-group GEMV splits it. A workgroup takes whole 32-row groups,
// its waves contiguous ranges of K, and their partial tiles meet in LDS in wave order, so y is written here, in
// original rows with the clamp delta: no output planes, no finishing launch. A tile's decoded B operand feeds all the
// call's token tiles (one or two). The x' operands come straight from memory in operand order (k_mm_rg_act): a wave's
// 16-byte loads of one MFMA operand are 1 KB contiguous, and the whole x' of such a call stays in the L2s.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "p8x_act.h"
#include "p8x_internal.h"
#include "p8x_lane.h"
#include "p8x_mm.h"

namespace p8x {

// x' in operand order: [block b][step s][token tile][lane][8 halves]; lane (token m = lane & 31, half kh = lane >> 5)
// of step s holds columns 256 b + 128 kh + 8 s .. + 7 of its token. One wave per (block, token); tokens past N in the
// last tile stay unwritten (their products reach only output rows that are never stored).
constexpr int kMmRgActWaves = 4;
template <typename XT>
__global__ __launch_bounds__(64 * kMmRgActWaves) void k_mm_rg_act(const XT *__restrict__ x, size_t ldx, const float *__restrict__ ic, int nb, int tiles,
                                                                  _Float16 *__restrict__ xf) {
    const int lane = threadIdx.x & 63, b = kMmRgActWaves * (int)blockIdx.x + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.y;
    if (b >= nb) return;
    half2v lo, hi;
    rotate_f16(x + (size_t)n * ldx + 256 * b, ic + 256 * b, lane, lo, hi);
    const int kh = lane >> 5, s = (lane & 31) >> 1;
    uint2 out;
    out.x = __builtin_bit_cast(uint32_t, lo);
    out.y = __builtin_bit_cast(uint32_t, hi);
    *reinterpret_cast<uint2 *>(xf + ((((size_t)b * 16 + s) * tiles + (n >> 5)) * 64 + 32 * kh + (n & 31)) * 8 + 4 * (lane & 1)) = out;
}

struct MmRgJob {
    const uint32_t *M; const uint16_t *Sg; const uint32_t *D;
    const _Float16 *xf;
    const uint32_t *a2;
    const uint16_t *prmd;
    const int *cp; const uint16_t *cc; const float *cv;
    const void *x; size_t ldx; int x_bf16;   // original activations (clamp delta)
    float *y; size_t ldy;
    int N, rows, nb, ng, gc;                 // gc: row groups a workgroup streams together (teams of waves)
    uint32_t dbytes, sbytes;
};

// class 3 with one token tile: 16 waves at 128 VGPRs; two tiles or any class: 8 waves at 256 (any class with two tiles
// spills 44 of them, the others none)
__host__ __device__ constexpr int mm_rg_waves(int cm, int tt) { return cm == kMmCmC3 && tt == 1 ? 16 : 8; }

// A wave's x' operands are loaded a segment of steps ahead: SEG steps x T token tiles = 8 operands, 32 registers.
__host__ __device__ constexpr int mm_rg_seg(int tt) { return 8 / tt; }

// table words of step s (two chunks), and the step's operand from them
template <int CM, int C>
struct MmRgWords {
    uint32_t w[2][CM == kMmCmC3 ? 2 : nstage_of(C)];
    __device__ __forceinline__ void load(const uint32_t *tab, const QuadSlice<C> &p, uint32_t H, uint32_t bankbytes, int s) {
        const uint32_t hq = coset_bytes(H, bankbytes, s >> 1);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t a = p.template addr<0>(2 * s + u, hq);
            if constexpr (CM == kMmCmC3) {   // fp16 table entry: the chunk's four weights
                const uint2 e = *reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(tab) + a);
                w[u][0] = e.x;
                w[u][1] = e.y;
            } else {
                w[u][0] = lds_word(tab, a);
                if constexpr (nstage_of(C) > 1) w[u][1] = lds_word(tab, p.template addr<1>(2 * s + u, hq));
                if constexpr (nstage_of(C) > 2) w[u][2] = lds_word(tab, p.template addr<2>(2 * s + u, hq));
            }
        }
    }
    __device__ __forceinline__ half8v operand(half2v s2) const {
        half2v v[4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if constexpr (CM == kMmCmC3) {
                v[2 * u] = __builtin_bit_cast(half2v, w[u][0]) * s2;
                v[2 * u + 1] = __builtin_bit_cast(half2v, w[u][1]) * s2;
            } else {
                uint32_t x[3] = {w[u][0], 0u, 0u};
                if constexpr (nstage_of(C) > 1) x[1] = w[u][1];
                if constexpr (nstage_of(C) > 2) x[2] = w[u][2];
                weights_chunk<C>(x, s2, v[2 * u], v[2 * u + 1]);
            }
        }
        half8v B;
#pragma unroll
        for (int k = 0; k < 4; ++k) { B[2 * k] = v[k].x; B[2 * k + 1] = v[k].y; }
        return B;
    }
};

template <int CM, int T>
__global__ __launch_bounds__(64 * mm_rg_waves(CM, T)) __attribute__((amdgpu_waves_per_eu(mm_rg_waves(CM, T) / 4, mm_rg_waves(CM, T) / 4)))
void k_mm_rg(MmRgJob J) {
    constexpr int WAVES = mm_rg_waves(CM, T), NT = 64 * WAVES, NQ = CM == kMmCmC3 ? 2 : 6;
    __shared__ uint32_t tab[kTabWords];          // LDS address 0
    __shared__ float red[WAVES][16 * T][64];     // each wave's partial tiles
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kh = lane >> 5;
    const uint32_t bankbytes = (uint32_t)((CM == kMmCmC3 ? (j & 15) << 1 : j) << 2) * 0x01010101u;
    const int gstep = gridDim.x, wpg = WAVES / J.gc, team = w / wpg, wk = w % wpg;
    const int per = J.nb / wpg, rem = J.nb % wpg;
    const int b0 = wk * per + min(wk, rem), b1 = team < J.gc ? b0 + per + (wk < rem ? 1 : 0) : b0;   // the wave's K range
    const __amdgpu_buffer_rsrc_t rd = buffer_rsrc(J.D, J.dbytes), rs = buffer_rsrc(J.Sg, J.sbytes);
    using Raw = std::conditional_t<CM == kMmCmC3, QuadSlice<3>, AnyQuads<NQ>>;
    // tile (g, b): its class and payload loads; indices past the tensor are clamped (loaded, never used)
    auto issue_raw = [&](Raw &r, uint32_t &c, int g, int b) {
        const int gi = min(g, J.ng - 1), bi = min(b, J.nb - 1);
        const uint32_t mt = as_const(J.M)[(size_t)gi * J.nb + bi];
        const uint32_t toff = (mt & 0x1FFFFFFFu) * 4u, soff = ((uint32_t)gi * (uint32_t)J.nb + (uint32_t)bi) * 64u;
        c = mt >> 29;
        if constexpr (CM == kMmCmC3) {   // class-0 tiles read zero words and a zero scale: zero weights
            const bool on = c == 3u;
            r.load(buffer_rsrc(J.D, on ? J.dbytes : 0u), toff, QuadSlice<3>::quad_offset(kh, j), 0u, buffer_rsrc(J.Sg, on ? J.sbytes : 0u), soff, 2u * j);
        } else {
            r.load(rd, toff, nw_run(c), kh, j, rs, soff, 2u * j);
        }
    };
    constexpr int SEG = mm_rg_seg(T);
    auto issue_a = [&](half8v (&A)[SEG][T], int b, int q) {
        const int bi = min(b, J.nb - 1);
        const gptr<const half8v> p = as_global(reinterpret_cast<const half8v *>(J.xf)) + ((size_t)bi * 16 + SEG * q) * T * 64 + lane;
#pragma unroll
        for (int s = 0; s < SEG; ++s)
#pragma unroll
            for (int t = 0; t < T; ++t) A[s][t] = p[(s * T + t) * 64];
        __asm__ volatile("" ::: "memory");   // issued here, ahead of the products they overlap
    };
    Raw nxt;
    uint32_t cn;
    half8v A0[SEG][T], A1[SEG][T];
    int g = (int)blockIdx.x + min(team, J.gc - 1) * gstep;
    // the first tile's loads and the table's go out together
    issue_raw(nxt, cn, g, b0);
    constexpr int TPT = kTabWords / 4 / NT;
    uint4 *t4 = reinterpret_cast<uint4 *>(tab);
    if constexpr (CM == kMmCmC3) {   // 16 copies of the fp16 entries (the tensor's tables carry them after the words)
        const uint2 *e16 = reinterpret_cast<const uint2 *>(J.a2 + 512);
        uint2 v[TPT];
#pragma unroll
        for (int k = 0; k < TPT; ++k) v[k] = e16[(tid + k * NT) >> 3];
        issue_a(A0, b0, 0);
#pragma unroll
        for (int k = 0; k < TPT; ++k) t4[tid + k * NT] = make_uint4(v[k].x, v[k].y, v[k].x, v[k].y);
    } else {                         // 32 copies of the words, bytes offset by 128
        uint32_t v[TPT];
#pragma unroll
        for (int k = 0; k < TPT; ++k) {
            const int i = tid + k * NT;
            v[k] = J.a2[((i >> 3) & 1) * 256 + (i >> 4)] ^ 0x80808080u;
        }
        issue_a(A0, b0, 0);
#pragma unroll
        for (int k = 0; k < TPT; ++k) t4[tid + k * NT] = make_uint4(v[k], v[k], v[k], v[k]);
    }
    __syncthreads();
    for (int g0 = blockIdx.x; g0 < J.ng; g0 += gstep * J.gc, g += gstep * J.gc) {
        const bool active = team < J.gc && g < J.ng;
        const int ro = active ? as_global(J.prmd)[32 * g + j] : 0;
        float16v acc[T];
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t] = float16v{};
        if (active) {
            for (int b = b0; b < b1; ++b) {
                const Raw cur = nxt;
                const uint32_t c = cn;
                // the tile after this one: the wave's next block, or its first block of the next round's row group
                const bool last = b + 1 == b1;
                const int gn = last ? g + gstep * J.gc : g, bn = last ? b0 : b + 1;
                issue_a(A1, b, 1);
                issue_raw(nxt, cn, gn, bn);
                __asm__ volatile("" ::: "memory");
                const half2v s2 = {__builtin_bit_cast(_Float16, (uint16_t)cur.s), __builtin_bit_cast(_Float16, (uint16_t)cur.s)};
                auto tile = [&](auto cls, const auto &p) {
                    constexpr int C = decltype(cls)::value;
                    const uint32_t H = p.coset_bits();
                    MmRgWords<CM, C> W[2];   // the next step's table words are read before this step's products
                    W[0].load(tab, p, H, bankbytes, 0);
#pragma unroll
                    for (int st = 0; st < 16; ++st) {
                        const int q = st / SEG, i = st % SEG;
                        if (st < 15) W[(st + 1) & 1].load(tab, p, H, bankbytes, st + 1);
                        const half8v B = W[st & 1].operand(s2);
#pragma unroll
                        for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16((q & 1) ? A1[i][t] : A0[i][t], B, acc[t], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);   // one step's table words ahead, no more: bounds the live registers
                        if (i == SEG - 1) {   // the segment's registers take the one two ahead (the next tile's first two at the end)
                            if (q & 1) {
                                if (q + 2 < 2 * T) issue_a(A1, b, q + 2);
                            } else {
                                if (q + 2 < 2 * T) issue_a(A0, b, q + 2);
                                else issue_a(A0, bn, 0);
                            }
                        }
                    }
                };
                if constexpr (CM == kMmCmC3) {
                    tile(std::integral_constant<int, 3>{}, cur);
                } else {
                    switch (c) {
                        case 1: tile(std::integral_constant<int, 1>{}, cur.template as<1>()); break;
                        case 2: tile(std::integral_constant<int, 2>{}, cur.template as<2>()); break;
                        case 3: tile(std::integral_constant<int, 3>{}, cur.template as<3>()); break;
                        case 4: tile(std::integral_constant<int, 4>{}, cur.template as<4>()); break;
                        case 5: tile(std::integral_constant<int, 5>{}, cur.template as<5>()); break;
                        case 6: tile(std::integral_constant<int, 6>{}, cur.template as<6>()); break;
                        case 7: tile(std::integral_constant<int, 7>{}, cur.template as<7>()); break;
                        default: issue_a(A0, bn, 0); break;   // class 0: zero weights
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 16; ++q) red[w][16 * t + q][lane] = acc[t][q];
        __syncthreads();
        // the team's waves share its 16 T output registers: element (t, q) of lane (j, kh) is token 32 t + 8 (q >> 2) +
        // 4 kh + (q & 3) of sorted row 32 g + j
        if (active)
            for (int i = wk; i < 16 * T; i += wpg) {
                float v = 0.f;
                for (int k0 = 0; k0 < wpg; k0 += 4) {   // four reads in flight, added in wave order
                    float pv[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) pv[k] = red[team * wpg + min(k0 + k, wpg - 1)][i][lane];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k0 + k < wpg) v += pv[k];
                }
                const int q = i & 15, tok = 32 * (i >> 4) + 8 * (q >> 2) + 4 * kh + (q & 3), r = ro & 0x7FFF;
                if (tok >= J.N) continue;
                if (ro & 0x8000)
                    for (int e = as_global(J.cp)[r]; e < as_global(J.cp)[r + 1]; ++e) {
                        const size_t xi = (size_t)tok * J.ldx + as_global(J.cc)[e];
                        const float xv = J.x_bf16 ? bf16_to_float(as_global((const uint16_t *)J.x)[xi]) : as_global((const float *)J.x)[xi];
                        v += as_global(J.cv)[e] * xv;
                    }
                as_global_rw(J.y)[(size_t)tok * J.ldy + r] = v;
            }
        __syncthreads();   // red is written again in the next round
    }
}

// Up to 64 tokens: the 128-token tile of k_mm does 2 to 14 times their products and needs planes and a finishing
// launch of one workgroup per token. Measured, 9728 x 2560 class 3, 19 tokens: k_mm 33.5 us a call (k_mm 15, finish 17),
// this path 13.3 us; what is left is latency (two launches, the table build, two to three tiles per wave).
int mm_rg_tiles(const p8x_tensor *t, int N) {
    if (N > kMmRgMaxTokens) return 0;
    const int tiles = (N + 31) / 32;
    // x' of the padded tiles fits the no-allocation scratch for every K below ~786,000; longer rows keep k_mm's plan
    return mm_rg_x_bytes(t, tiles) <= (size_t)P8X_NOALLOC_SCRATCH_BYTES ? tiles : 0;
}

size_t mm_rg_x_bytes(const p8x_tensor *t, int tiles) { return (size_t)32 * tiles * t->K * sizeof(_Float16); }

template <int CM, int T>
static int launch_mm_rg_t(const MmRgJob &J_, hipStream_t st) {
    MmRgJob J = J_;
    const int per = (J.ng + num_cus() - 1) / num_cus();   // row groups per workgroup (one workgroup per CU)
    J.gc = std::min(per, 4);
    hipLaunchKernelGGL((k_mm_rg<CM, T>), dim3((J.ng + per - 1) / per), dim3(64 * mm_rg_waves(CM, T)), 0, st, J);
    return hip_check(hipGetLastError(), "k_mm_rg launch");
}

int launch_mm_rg(const p8x_tensor *t, int tiles, const void *x, int x_dtype, int N, size_t ldx, float *y, size_t ldy, void *xf, hipStream_t st) {
    int rc;
    const dim3 agrid((t->nb + kMmRgActWaves - 1) / kMmRgActWaves, N);
    if (x_dtype == P8X_F32) hipLaunchKernelGGL(k_mm_rg_act<float>, agrid, dim3(64 * kMmRgActWaves), 0, st, (const float *)x, ldx, t->ic, t->nb, tiles, (_Float16 *)xf);
    else hipLaunchKernelGGL(k_mm_rg_act<uint16_t>, agrid, dim3(64 * kMmRgActWaves), 0, st, (const uint16_t *)x, ldx, t->ic, t->nb, tiles, (_Float16 *)xf);
    if ((rc = hip_check(hipGetLastError(), "k_mm_rg_act launch"))) return rc;
    MmRgJob J{};
    J.M = t->M; J.Sg = t->Sg; J.D = t->D; J.xf = (const _Float16 *)xf; J.a2 = t->a2; J.prmd = t->prmd;
    J.cp = t->cp; J.cc = t->cc; J.cv = t->cv; J.x = x; J.ldx = ldx; J.x_bf16 = x_dtype == P8X_BF16; J.y = y; J.ldy = ldy;
    J.N = N; J.rows = t->rows; J.nb = t->nb; J.ng = t->ng;
    J.dbytes = (uint32_t)(t->kbytes - offset_D(t->nt));
    J.sbytes = (uint32_t)t->nb * (uint32_t)t->rows * 2u;
    const bool c3 = mm_only_c3(t);
    if (tiles == 1) return c3 ? launch_mm_rg_t<kMmCmC3, 1>(J, st) : launch_mm_rg_t<kMmCmAll, 1>(J, st);
    return c3 ? launch_mm_rg_t<kMmCmC3, 2>(J, st) : launch_mm_rg_t<kMmCmAll, 2>(J, st);
}

}  // namespace p8x
