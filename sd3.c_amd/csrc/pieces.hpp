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

// A matrix in pieces in memory, as what produces an operand writes it for the kernel that multiplies it: three planes (h, m, l), each in blocks of 16 rows x 32 k values
// of 1024 bytes that are the GEMM's LDS rows as they are (piece_slot; chunk c of 8 values: k = 4c .. 4c + 3 and 16 + 4c ..): a direct load of a wavefront is a block,
// whole cache lines; the blocks of 16 rows follow each other along k. (As rows of 192
// bytes per K tile, whose lines neighbouring K tiles share, 10656 x 768 x 3072 took 227 us, with the planes of a block side by side, 3 KB that few memory channels
// hold, 233, so 215; few workgroups of 256x128 tiles 1.42, 1.63 and 1.41 us a K tile.) K is a multiple of 32; a
// last block of fewer rows has room for 16. What the pieces cannot hold (|x| from 2^112 on, infinities, NaNs) has a NaN for h and its own bits for m and l: products
// with it are NaNs, and it can be had back.
constexpr unsigned PIECES_NAN = 0x7fc0;
__host__ __device__ inline size_t pieces_bytes(size_t rows, size_t K) { return (rows + 15) / 16 * 16 * K * 6; }
struct PieceMatrix {
    bf16_t* p;
    long long plane;  // values
    int K;
    __device__ __forceinline__ PieceMatrix(void* q, long long M, int K_) : p(reinterpret_cast<bf16_t*>(q)), plane((M + 15) / 16 * 16 * K_), K(K_) {}
};
__device__ __forceinline__ long long piece_index(long long row, unsigned k, int K) {
    return ((row >> 4) * (K / 32) + k / 32) * 512 + piece_slot<0>((unsigned)row & 15, k % 16 / 4) / 2 + k / 16 % 2 * 4 + k % 4;
}
// The pieces of N values as they are written
template <int N>
__device__ __forceinline__ void pieces_for_memory(const float (&v)[N], uint32_t (&piece)[3][(N + 1) / 2]) {
    constexpr int P = N == 1 ? 2 : N;
    float x[P];
#pragma unroll
    for (int i = 0; i < P; i++) x[i] = i < N ? v[i] : 0.f;
    bf16_pieces<P>(x, piece[0], piece[1], piece[2]);
    // what is left of a value that has no pieces is a NaN (infinity less infinity)
    float rest = x[0];
#pragma unroll
    for (int i = 1; i < P; i++) rest += x[i];
    if (__builtin_expect(rest != rest, 0)) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const unsigned sh = i & 1 ? 16 : 0;
            if ((piece[0][i / 2] >> sh & 0x7f80u) == 0x7f80u) {
                const uint32_t bits = __float_as_uint(v[i]), others = ~(0xffffu << sh);
                piece[0][i / 2] = (piece[0][i / 2] & others) | PIECES_NAN << sh;
                piece[1][i / 2] = (piece[1][i / 2] & others) | (bits >> 16) << sh;
                piece[2][i / 2] = (piece[2][i / 2] & others) | (bits & 0xffffu) << sh;
            }
        }
    }
}
// N = 1, 2 or 4 consecutive values of a row from k on, k a multiple of N
template <int N>
__device__ __forceinline__ void put_pieces(const PieceMatrix& to, long long row, unsigned k, const float (&v)[N]) {
    uint32_t piece[3][(N + 1) / 2];
    pieces_for_memory<N>(v, piece);
    bf16_t* at = to.p + piece_index(row, k, to.K);
#pragma unroll
    for (int p = 0; p < 3; p++) __builtin_memcpy(__builtin_assume_aligned(at + p * to.plane, N * 2), piece[p], N * 2);
}
__device__ __forceinline__ float of_pieces(const PieceMatrix& of, long long row, unsigned k) {
    const bf16_t* at = of.p + piece_index(row, k, of.K);
    const uint32_t h = at[0], m = at[of.plane], l = at[2 * of.plane];
    if ((h & 0x7f80u) == 0x7f80u) return __uint_as_float(m << 16 | l);
    return ((__uint_as_float(h << 16) + __uint_as_float(m << 16)) + __uint_as_float(l << 16)) * (1.0f / PIECES_SCALE);
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
