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

// the row-group GEMM (p8x_mm_rg.hip): up to kMmRgMaxTokens tokens in one pass over the weights
constexpr int kMmRgMaxTokens = 64;
bool mm_only_c3(const p8x_tensor *t);
int mm_rg_tiles(const p8x_tensor *t, int N);                  // 32-token tiles of the call, 0: not served
size_t mm_rg_x_bytes(const p8x_tensor *t, int tiles);         // its x' workspace
int launch_mm_rg(const p8x_tensor *t, int tiles, const void *x, int x_dtype, int N, size_t ldx, float *y, size_t ldy, void *xf, hipStream_t st);

}  // namespace p8x
