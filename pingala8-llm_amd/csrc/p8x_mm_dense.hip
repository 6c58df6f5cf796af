// p8x_mm_dense.hip -- prompt GEMM of many tokens in two launches: the weights decoded once into fp16 MFMA operands
// (k_mm_decode), then a dense kernel on them (k_mm_dense).
//
// k_mm decodes a weight tile again for every 128 or 256 tokens, and its decode (5 to 9 VALU instructions per MFMA and
// the table reads) holds the matrix cores at about a third of their rate, less for mixed classes. Past a few hundred
// tokens it is cheaper to write the operands v S once (2 bytes per weight, in memory that calls share: p8x_operands.h)
// and to read them back per token tile; a tensor with more than kMmOperandBytes goes through in bands of row tiles. The
// operands and the order in which they are summed are k_mm's, so both give the same bits for the same K split.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "p8x_internal.h"
#include "p8x_lane.h"
#include "p8x_mm.h"

namespace p8x {

// Decoded operands: [row group g of the band][block b][step s][lane][8 halves]: lane (row j = lane & 31, half kh = lane >> 5) of
// step s holds the eight weights of sorted row 32 g + j at columns 256 b + 128 kh + 8 s .., what v_mfma_f32_32x32x16_f16
// takes as its second operand. 16 KB per tile (kMmTileHalves); a wave stores and loads a step as 1 KB of consecutive bytes.
constexpr int kMmDecWaves = 8;
struct MmDecJob {
    const uint32_t *M; const uint16_t *Sg; const uint32_t *D; const uint32_t *a2;
    _Float16 *bw;
    int nt;
    uint32_t dbytes, sbytes;
};

template <int C>
__device__ __forceinline__ void mm_decode_tile(const uint32_t *tab, const QuadSlice<C> &p, uint32_t bankbytes, gptr<half8v> out) {
    const uint32_t H = p.coset_bits();
    const half2v s2 = {__builtin_bit_cast(_Float16, (uint16_t)p.s), __builtin_bit_cast(_Float16, (uint16_t)p.s)};
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const uint32_t hq = coset_bytes(H, bankbytes, s >> 1);
        half2v v[4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t a = p.template addr<0>(2 * s + u, hq);
            uint32_t w[3] = {lds_word(tab, a), 0u, 0u};
            if constexpr (nstage_of(C) > 1) w[1] = lds_word(tab, p.template addr<1>(2 * s + u, hq));
            if constexpr (nstage_of(C) > 2) w[2] = lds_word(tab, p.template addr<2>(2 * s + u, hq));
            weights_chunk<C>(w, s2, v[2 * u], v[2 * u + 1]);
        }
        half8v B;
#pragma unroll
        for (int i = 0; i < 4; ++i) { B[2 * i] = v[i].x; B[2 * i + 1] = v[i].y; }
        __builtin_nontemporal_store(B, out + s * 64);
    }
}

// One tile per wave and step, the next tile's payload in flight. Two workgroups per CU (64 KB table each); bound by
// its stores (16 KB per 2.1 KB tile read), which are non-temporal: 28 to 34 us for 117 MB (36 to 38 as plain stores).
__global__ __launch_bounds__(64 * kMmDecWaves) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_mm_decode(MmDecJob J) {
    constexpr int NT = 64 * kMmDecWaves, NQ = 6;
    __shared__ uint32_t tab[kTabWords];   // LDS address 0
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kh = lane >> 5;
    const uint32_t bankbytes = (uint32_t)(j << 2) * 0x01010101u;
    const int nw = (int)gridDim.x * kMmDecWaves;
    int t = (int)blockIdx.x * kMmDecWaves + w;
    const __amdgpu_buffer_rsrc_t rd = buffer_rsrc(J.D, J.dbytes), rs = buffer_rsrc(J.Sg, J.sbytes);
    AnyQuads<NQ> nxt;
    uint32_t cn = 0;
    auto issue = [&](int tt) {   // past the last tile the last one is loaded again, never used
        const int ti = min(tt, J.nt - 1);
        const uint32_t mt = as_const(J.M)[ti];
        cn = mt >> 29;
        nxt.load(rd, (mt & 0x1FFFFFFFu) * 4u, nw_run(cn), kh, j, rs, (uint32_t)ti * 64u, 2u * j);
    };
    issue(t);
    constexpr int TPT = kTabWords / 4 / NT;
    uint4 *t4 = reinterpret_cast<uint4 *>(tab);
    // 32 copies of the table words, bytes offset by 128
    uint32_t v[TPT];
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
        const int i = tid + k * NT;
        v[k] = J.a2[((i >> 3) & 1) * 256 + (i >> 4)] ^ 0x80808080u;
    }
#pragma unroll
    for (int k = 0; k < TPT; ++k) t4[tid + k * NT] = make_uint4(v[k], v[k], v[k], v[k]);
    __syncthreads();
    for (; t < J.nt; t += nw) {
        const AnyQuads<NQ> cur = nxt;
        const uint32_t c = cn;
        issue(t + nw);
        const gptr<half8v> out = as_global_rw(reinterpret_cast<half8v *>(J.bw + (size_t)t * kMmTileHalves)) + lane;
        switch (c) {
            case 1: mm_decode_tile(tab, cur.template as<1>(), bankbytes, out); break;
            case 2: mm_decode_tile(tab, cur.template as<2>(), bankbytes, out); break;
            case 3: mm_decode_tile(tab, cur.template as<3>(), bankbytes, out); break;
            case 4: mm_decode_tile(tab, cur.template as<4>(), bankbytes, out); break;
            case 5: mm_decode_tile(tab, cur.template as<5>(), bankbytes, out); break;
            case 6: mm_decode_tile(tab, cur.template as<6>(), bankbytes, out); break;
            case 7: mm_decode_tile(tab, cur.template as<7>(), bankbytes, out); break;
            default: break;   // no class-0 tiles here (mm_plan)
        }
    }
}

// 256 rows x 32 NTI tokens per workgroup of four waves, one per SIMD, as k_mm: x' half-blocks through registers into
// two LDS buffers, written while the other half is multiplied. A wave's weight operands come from memory in operand
// order, eight steps ahead in a ring of registers: step s's registers are loaded with step s of the next half-block
// right after its products. NTI 4 .. 6: at 7 and 8 the accumulators and the ring spill (measured 30 to 70% slower).
// Measured 165 us for 4096 x 14336 x 1500 tokens (NTI 6, 1.07 PFLOP/s); 190 us with NTI 4 on 192 of the CUs.
template <int NTI>
__global__ __launch_bounds__(64 * mm_waves()) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_mm_dense(MmJob J) {
    constexpr int NWAVES = mm_waves(), NTJ = mm_ntj(), TOK = mm_tok(NTI), IPW = XStage<NWAVES, TOK>::IPW, PPS = (IPW + 3) / 4;
    __shared__ __attribute__((aligned(16))) _Float16 xs[2][TOK * 128];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kh = lane >> 5;
    // Tile order: K split, then bands of 8 row tiles, then token tile, then row tile; each XCD takes one contiguous
    // run of it, so that the workgroups on one L2 share a few row tiles' operands and a few token tiles' x'.
    const int total = J.tiles_m * J.tiles_n * J.nsplit, per = (total + kXcds - 1) / kXcds;
    const int lin = ((int)blockIdx.x % kXcds) * per + (int)blockIdx.x / kXcds;
    if ((int)blockIdx.x / kXcds >= per || lin >= total) return;
    const int ks = lin / (J.tiles_m * J.tiles_n), l2 = lin % (J.tiles_m * J.tiles_n);
    const int band = l2 / (8 * J.tiles_n), l3 = l2 % (8 * J.tiles_n), bm = min(8, J.tiles_m - 8 * band);
    const int tn = l3 / bm, tm = 8 * band + l3 % bm;
    const int tok0 = tn * TOK, b0 = ks * J.kper, b1 = min(J.nb, b0 + J.kper);
    int g[NTJ];
    gptr<const half8v> bp[NTJ];
#pragma unroll
    for (int tj = 0; tj < NTJ; ++tj) {
        g[tj] = J.g0 + (tm * mm_rows()) / 32 + NTJ * w + tj;   // row groups past the tensor repeat the last (never stored)
        bp[tj] = as_global(reinterpret_cast<const half8v *>(J.bw + ((size_t)(min(g[tj], J.ng - 1) - J.g0) * J.nb + b0) * kMmTileHalves)) + lane;
    }
    float16v acc[NTI][NTJ];
#pragma unroll
    for (int ti = 0; ti < NTI; ++ti)
#pragma unroll
        for (int tj = 0; tj < NTJ; ++tj) acc[ti][tj] = float16v{};
    XStage<NWAVES, TOK> xq;
    half8v B[8][NTJ];
    mm_fetch<NWAVES, TOK>(J, xq, tok0, b0, 0, w, lane);
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int tj = 0; tj < NTJ; ++tj) B[s][tj] = bp[tj][s * 64];
    mm_put<NWAVES, TOK>(xq, xs[0], w, lane);
    __syncthreads();
    const int nh = 2 * (b1 - b0);
    for (int h2 = 0; h2 < nh; h2 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int hn = min(h2 + u + 1, nh - 1);   // the next half-block (the last one again at the end, never used)
            const _Float16 *xb = xs[u];
            _Float16 *xn = xs[u ^ 1];
            mm_fetch<NWAVES, TOK>(J, xq, tok0, b0 + (hn >> 1), hn & 1, w, lane);
            auto read_a = [&](int s8, half8v (&A)[NTI]) {
#pragma unroll
                for (int ti = 0; ti < NTI; ++ti)
                    A[ti] = *reinterpret_cast<const half8v *>(xb + (32 * ti + j) * 128 + 8 * ((8 * kh + s8) ^ (j & 15)));
            };
            half8v A[NTI];
            read_a(0, A);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s8 = 0; s8 < 8; ++s8) {
                half8v An[NTI];
                if (s8 < 7) read_a(s8 + 1, An);
#pragma unroll
                for (int tj = 0; tj < NTJ; ++tj)
#pragma unroll
                    for (int ti = 0; ti < NTI; ++ti) acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[ti], B[s8][tj], acc[ti][tj], 0, 0, 0);
#pragma unroll
                for (int tj = 0; tj < NTJ; ++tj) B[s8][tj] = bp[tj][(8 * hn + s8) * 64];
                if (s8 >= 4) {
#pragma unroll
                    for (int i = 0; i < PPS; ++i)
                        if ((s8 - 4) * PPS + i < IPW)
                            *reinterpret_cast<u32x4 *>(xn + 4 * (IPW * w + (s8 - 4) * PPS + i) * 128 + 8 * lane) = xq.v[(s8 - 4) * PPS + i];
                }
                // one x' read behind each of the first MFMAs of the step, the x' writes behind the later ones
#pragma unroll
                for (int i = 0; i < NTI * NTJ; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (i < NTI && s8 < 7) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (i >= NTI && i - NTI < PPS && s8 >= 4) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                    if (i >= NTI * NTJ - NTJ) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (s8 < 7) {
#pragma unroll
                    for (int ti = 0; ti < NTI; ++ti) A[ti] = An[ti];
                }
            }
            __syncthreads();
        }
    }
    // element (ti, tj, q) of lane (j, kh): token 32 ti + 8 (q >> 2) + 4 kh + (q & 3), sorted row 32 g[tj] + j
    float *dst = J.direct ? J.y : J.ws + (size_t)ks * J.N * J.rows;
    const size_t ld = J.direct ? (size_t)J.ldy : (size_t)J.rows;
#pragma unroll
    for (int tj = 0; tj < NTJ; ++tj) {
        if (g[tj] >= J.ng) continue;
        const gptr<float> o = as_global_rw(dst) + 32 * g[tj] + j;
#pragma unroll
        for (int ti = 0; ti < NTI; ++ti)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int tok = tok0 + 32 * ti + 8 * (q >> 2) + 4 * kh + (q & 3);
                if (tok < J.N) o[(size_t)tok * ld] = acc[ti][tj][q];
            }
    }
}

int mm_dense_band(const p8x_tensor *t) {
    const int tiles = (t->rows + mm_rows() - 1) / mm_rows();
    const size_t per = (size_t)(mm_rows() / 32) * t->nb * kMmTileHalves * sizeof(_Float16);
    const int most = std::max(1, (int)(kMmOperandBytes / per)), bands = (tiles + most - 1) / most;
    return (tiles + bands - 1) / bands;
}

size_t mm_dense_w_bytes(const p8x_tensor *t) {
    return (size_t)std::min(mm_dense_band(t) * (mm_rows() / 32), t->ng) * t->nb * kMmTileHalves * sizeof(_Float16);
}

// operands of row groups g0 .. g0 + gn - 1
int launch_mm_decode(const p8x_tensor *t, int g0, int gn, void *bw, hipStream_t st) {
    const size_t t0 = (size_t)g0 * t->nb;
    const int nt = gn * t->nb;
    MmDecJob J{t->M + t0, t->Sg + 32 * t0, t->D, t->a2, (_Float16 *)bw, nt, (uint32_t)(t->kbytes - offset_D(t->nt)), (uint32_t)nt * 64u};
    const int grid = std::min((nt + kMmDecWaves - 1) / kMmDecWaves, 2 * num_cus());
    hipLaunchKernelGGL(k_mm_decode, dim3(grid), dim3(64 * kMmDecWaves), 0, st, J);
    return hip_check(hipGetLastError(), "k_mm_decode launch");
}

int launch_mm_dense(int nti, const MmJob &J, hipStream_t st) {
    const dim3 grid((J.tiles_m * J.tiles_n * J.nsplit + kXcds - 1) / kXcds * kXcds), block(64 * mm_waves());
    switch (nti) {
        case 4: hipLaunchKernelGGL((k_mm_dense<4>), grid, block, 0, st, J); break;
        case 5: hipLaunchKernelGGL((k_mm_dense<5>), grid, block, 0, st, J); break;
        case 6: hipLaunchKernelGGL((k_mm_dense<6>), grid, block, 0, st, J); break;
        default: return set_error(P8X_ERR_ARG, "k_mm_dense: %d token tiles", nti);
    }
    return hip_check(hipGetLastError(), "k_mm_dense launch");
}

}  // namespace p8x
