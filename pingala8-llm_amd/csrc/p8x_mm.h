// p8x_mm.h -- fp16 weight decode shared by the prompt GEMM kernels (p8x_gemm.hip, p8x_mm_rg.hip): table words to
// fp16 MFMA operands v S (v exact, one rounding for the product).
#pragma once
#include <hip/hip_runtime.h>

#include "p8x_act.h"
#include "p8x_internal.h"
#include "p8x_lane.h"

namespace p8x {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

// x' = FWHT(x ic) / 16 of one 256-block rounded to fp16: lane holds 4 consecutive elements (x 16-byte aligned);
// butterflies h = 1, 2 in the lane, 4 .. 128 across lanes (DPP row moves for distances 1-8, lane swaps for 16 and 32).
template <typename XT>
__device__ __forceinline__ void rotate_f16(const XT *__restrict__ x, const float *__restrict__ ic, int lane, half2v &lo, half2v &hi) {
    BlockLane in;
    in.c = as_global(reinterpret_cast<const f32x4 *>(ic))[lane];
    if constexpr (sizeof(XT) == 4) {
        in.x = as_global(reinterpret_cast<const f32x4 *>(x))[lane];
    } else {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 raw = as_global(reinterpret_cast<const u32x2 *>(x))[lane];
        in.x = f32x4{bf16_to_float((uint16_t)raw.x), bf16_to_float((uint16_t)(raw.x >> 16)), bf16_to_float((uint16_t)raw.y),
                     bf16_to_float((uint16_t)(raw.y >> 16))};
    }
    float v[4];
    rotate_block_lane(in, lane, v);
    lo.x = (_Float16)v[0]; lo.y = (_Float16)v[1];
    hi.x = (_Float16)v[2]; hi.y = (_Float16)v[3];
}

// offset-binary int8x4 (v + 128 per byte) -> two fp16 pairs holding 1152 + v exactly
__device__ __forceinline__ half2v ob_lo(uint32_t w) { return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)); }
__device__ __forceinline__ half2v ob_hi(uint32_t w) { return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)); }

// LDS words of chunk t, all stages (table bytes are A[f] + h c offset by 128)
template <int C, int NWMAX>
__device__ __forceinline__ void lookup_chunk(const AnySlice<NWMAX> &ls, const uint32_t *tab, int t, uint32_t hq, uint32_t (&w)[3]) {
    constexpr int NST = nstage_of(C);
    w[0] = lds_word(tab, ls.template addr<C, 0>(t, hq));
    if constexpr (NST > 1) w[1] = lds_word(tab, ls.template addr<C, 1>(t, hq));
    if constexpr (NST > 2) w[2] = lds_word(tab, ls.template addr<C, 2>(t, hq));
}

// table words of one chunk -> 4 fp16 weights v S (v exact in fp16, |v| <= 1596; one rounding for the product)
template <int C>
__device__ __forceinline__ void weights_chunk(const uint32_t (&w)[3], half2v s2, half2v &lo, half2v &hi) {
    constexpr int NST = nstage_of(C), SH1 = sh1_of(C), SH2 = sh2_of(C);
    const half2v bias = {(_Float16)-1152.f, (_Float16)-1152.f};
    half2v vl = ob_lo(w[0]) + bias, vh = ob_hi(w[0]) + bias;
    if constexpr (NST > 1) {
        const half2v m1 = {(_Float16)(float)(1 << SH1), (_Float16)(float)(1 << SH1)};
        const half2v m2 = {(_Float16)(float)(1 << SH2), (_Float16)(float)(1 << SH2)};
        half2v al = (ob_lo(w[1]) + bias) * m2, ah = (ob_hi(w[1]) + bias) * m2;
        if constexpr (NST > 2) { al += ob_lo(w[2]) + bias; ah += ob_hi(w[2]) + bias; }
        vl = vl * m1 + al;   // integers below 2048: exact in fp16
        vh = vh * m1 + ah;
    }
    lo = vl * s2;
    hi = vh * s2;
}

// classes decoded by an instantiation: the tensor's class set (class 0 decodes as zeros in all of them)
constexpr int kMmCmC3 = 1 << 3, kMmCmAll = 0xFE;
constexpr int kMmMain = 3;   // the class with a branch-free path in every instantiation (the 2-bit bulk)
__host__ __device__ constexpr int mm_nwmax(int cm) { return cm == kMmCmC3 ? 8 : 24; }

// ------------------------------------------------------------------------------------------------ tiled kernels
struct MmJob {
    const uint32_t *M; const uint16_t *S; const uint32_t *D;
    const _Float16 *xr;     // x' [N][K]
    float *y; unsigned ldy; // direct output (original rows = sorted rows, one K range)
    float *ws;              // sorted-row planes [nsplit][N][rows] otherwise
    const uint32_t *a2;     // [2][256] coset table words (A[f] + h c), h-major, then the same as fp16: entry 2 f + h,
                            // 4 halves
    int N, rows, K, nb, ng;
    const _Float16 *bw;     // k_mm_dense: the decoded weights (k_mm_decode) of the launch's row groups, g0 the first
    int g0;
    int tiles_m, tiles_n, nsplit, kper, direct;
#ifdef P8X_TIMELINE
    unsigned long long *tl;
#endif
};

// workgroup tile of k_mm and k_mm_dense: four waves, one per SIMD, each 64 weight rows x all of the tile's tokens
__host__ __device__ constexpr int mm_waves() { return 4; }
__host__ __device__ constexpr int mm_ntj() { return 2; }
__host__ __device__ constexpr int mm_rows() { return 32 * mm_ntj() * mm_waves(); }
__host__ __device__ constexpr int mm_tok(int nti) { return 32 * nti; }

// x' half-block tile in LDS: half sh of block b holds, per token, columns 128 kh + 64 sh + 8 c8 + (0..7) as
// chunk c = 8 kh + c8 at position c ^ (t & 15) of the token's 256-byte row, so the 16-byte operand reads of
// 16 consecutive tokens cover all 64 banks once. TOK tokens: TOK x 128 halves per buffer.

// Stage half sh of block b in two parts: mm_fetch loads it into registers, mm_put writes it to LDS. With IPW =
// TOK / (4 NWAVES) rows of four tokens per wave, row i of wave w holds token rows 4 (IPW w + i) + (0..3); lane l
// carries token row + (l >> 4), position l & 15 and writes it at the row's LDS base + 16 l bytes. (Direct-to-LDS loads
// would save the registers, but while one may be in flight the compiler waits for every LDS read to finish
// before using any, which serializes the operand reads of consecutive MFMA steps.)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <int NWAVES, int TOK>
struct XStage {
    static constexpr int IPW = TOK / (4 * NWAVES);
    u32x4 v[IPW];   // a native vector type: kept in registers (HIP's uint4 struct made the array a stack object)
};

template <int NWAVES, int TOK>
__device__ __forceinline__ void mm_fetch(const MmJob &J, XStage<NWAVES, TOK> &xs, int tok0, int b, int sh, int w, int lane) {
    constexpr int IPW = XStage<NWAVES, TOK>::IPW;
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
        const int row = 4 * (IPW * w + i), t = row + (lane >> 4);
        const int ts = min(tok0 + t, J.N - 1);   // rows past N repeat the last token (never written out)
        const int c = (lane & 15) ^ (t & 15);
        xs.v[i] = *reinterpret_cast<const u32x4 *>(J.xr + (size_t)ts * J.K + 256 * b + 128 * (c >> 3) + 64 * sh + 8 * (c & 7));
    }
    __asm__ volatile("" ::: "memory");   // issued here, ahead of the products they overlap
}

// rows I0 .. I1 - 1 of the wave's share
template <int NWAVES, int TOK, int I0 = 0, int I1 = XStage<NWAVES, TOK>::IPW>
__device__ __forceinline__ void mm_put(const XStage<NWAVES, TOK> &xs, _Float16 *xb, int w, int lane) {
    constexpr int IPW = XStage<NWAVES, TOK>::IPW;
#pragma unroll
    for (int i = I0; i < I1; ++i) *reinterpret_cast<u32x4 *>(xb + 4 * (IPW * w + i) * 128 + 8 * lane) = xs.v[i];
}

// the row-group GEMM (p8x_mm_rg.hip): up to kMmRgMaxTokens tokens in one pass over the weights
constexpr int kMmRgMaxTokens = 64;
bool mm_only_c3(const p8x_tensor *t);
int mm_rg_tiles(const p8x_tensor *t, int N);                  // 32-token tiles of the call, 0: not served
size_t mm_rg_x_bytes(const p8x_tensor *t, int tiles);         // its x' workspace
// the decoded-weights GEMM (p8x_mm_dense.hip): weight operands decoded once per call, then a dense kernel of
// 256 rows x 32 nti tokens per workgroup, nti 4 .. 6
constexpr int kMmTileHalves = 16 * 64 * 8;             // decoded operands of a weight tile
constexpr size_t kMmOperandBytes = (size_t)192 << 20;  // at most this much of them at a time: 17408 x 5120 in one band
int mm_dense_band(const p8x_tensor *t);                // row tiles of a band
size_t mm_dense_w_bytes(const p8x_tensor *t);          // its operands
int launch_mm_decode(const p8x_tensor *t, int g0, int gn, void *bw, hipStream_t st);
int launch_mm_dense(int nti, const MmJob &J, hipStream_t st);
int launch_mm_rg(const p8x_tensor *t, int tiles, const void *x, int x_dtype, int N, size_t ldx, float *y, size_t ldy, void *xf, hipStream_t st);

}  // namespace p8x
