// fp32 values as pieces of 16 bits (fp32 products on the matrix instructions of 16-bit operands).
#pragma once
#include "common.hpp"

namespace sd3 {
namespace {

// x * 2^16 = h + m + l, each a bf16 value: h the first 8 significant bits, rounded to nearest, m the next 8 of what is left, l the rest, at most 8 bits. Without a
// remainder for every |x| < 2^112, subnormal numbers included: the last bit of the smallest, 2^-149, becomes the last bit of the smallest bf16 value, which the matrix instructions take as
// it is (with no scale, values below 2^-110 would lose bits; the scale costs 4 %). Beyond, as for infinities and NaNs, h is infinite or a NaN. |m| <= 2^-8 |x| and
// |l| <= 2^-17 |x|. Step by step for all values, as each step waits for the one before. N values, two to a register.
constexpr float PIECES_SCALE = 0x1p16f;
constexpr int NOT_VECTOR = 0x94;  // what may cross: scalar operations, memory and LDS
template <int N>
__device__ __forceinline__ void bf16_high(const float (&x)[N], uint32_t (&piece)[N / 2]) {
#pragma unroll
    for (int p = 0; p < N / 2; p++) piece[p] = pack_bf16x2(x[2 * p], x[2 * p + 1]);
}
template <int N, bool FENCES = true>
__device__ __forceinline__ void bf16_rest(float (&x)[N], const uint32_t (&piece)[N / 2]) {
    float t[N];
#pragma unroll
    for (int k = 0; k < N; k++) t[k] = __uint_as_float(k & 1 ? piece[k / 2] & 0xffff0000u : piece[k / 2] << 16);
    if constexpr (FENCES) __builtin_amdgcn_sched_barrier(NOT_VECTOR);
#pragma unroll
    for (int k = 0; k < N; k++) x[k] -= t[k];
    if constexpr (FENCES) __builtin_amdgcn_sched_barrier(NOT_VECTOR);
}
template <int N>
__device__ __forceinline__ void bf16_pieces(float (&x)[N], uint32_t (&h)[N / 2], uint32_t (&m)[N / 2], uint32_t (&l)[N / 2]) {
#pragma unroll
    for (int k = 0; k < N; k++) x[k] *= PIECES_SCALE;
    bf16_high<N>(x, h);
    __builtin_amdgcn_sched_barrier(NOT_VECTOR);
    bf16_rest<N>(x, h);
    bf16_high<N>(x, m);
    __builtin_amdgcn_sched_barrier(NOT_VECTOR);
    bf16_rest<N>(x, m);
    bf16_high<N>(x, l);
}

// Where `chunk`, 8 k values, of a row of a plane lies; MULT: how far rows 16 apart, written by neighbouring lanes, are moved apart
template <int MULT>
__device__ __forceinline__ unsigned piece_slot(unsigned row, unsigned chunk) {
    return row * 64 + ((chunk ^ (0u - (row >> 2)) ^ ((row >> 1) & 1) ^ ((row >> 4) * MULT)) & 3) * 16;
}
template <int KEEP>  // all but the last KEEP LDS operations of this wavefront are done, and behind the barrier those of the others too
__device__ __forceinline__ void barrier_behind_lds() {
    __builtin_amdgcn_s_waitcnt(15 | (KEEP << 8) | (7 << 4) | (3 << 14));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ bool finite(float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; }

}  // namespace
}  // namespace sd3
