// Shared declarations of the HIP library: status/error plumbing, bf16 helpers, kernel launchers.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

#include "../../include/sd3_hip.h"
#include "device.hpp"
#include "offsets.hpp"
#include "passengers.hpp"

namespace sd3 {

// ---- error plumbing (thread-local message, never exit) ----
int fail(int status, const char* fmt, ...);
void set_error(const char* msg);

#define SD3_HIP_TRY(expr)                                                                                       \
    do {                                                                                                        \
        hipError_t e_ = (expr);                                                                                 \
        if (e_ != hipSuccess) return ::sd3::fail(SD3_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)
#define SD3_TRY(expr)               \
    do {                            \
        int s_ = (expr);            \
        if (s_ != SD3_OK) return s_; \
    } while (0)
#define SD3_REQUIRE(cond, ...)                                           \
    do {                                                                 \
        if (!(cond)) return ::sd3::fail(SD3_ERR_INVALID_ARG, __VA_ARGS__); \
    } while (0)

inline int launch_status(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(SD3_ERR_HIP, "launch of %s failed: %s", what, hipGetErrorString(e));
    return SD3_OK;
}

// ---- bf16 as raw 16-bit storage ----
typedef uint16_t bf16_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_t;
// fp32 -> bf16, round to nearest even (the gfx950 v_cvt_pk_bf16_f32 instruction)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
    const __bf16 r = (__bf16)f;
    return __builtin_bit_cast(bf16_t, r);
}
__device__ __forceinline__ float bf16_to_f32(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    const f32x2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// tanh-GELU in 8 full-rate operations: 0.5 x (1 + tanh(u)) = x * sigmoid(2u) = x / (1 + 2^(-2u log2 e)),
// u = sqrt(2/pi) (x + 0.044715 x^3). Saturates cleanly: the exponential overflows to +inf -> 0, or underflows to 0 -> x.
__device__ __forceinline__ float gelu_tanh_f(float x) {
    const float k1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;  // -2 sqrt(2/pi) log2(e)
    const float k3 = k1 * 0.044715f;
    const float x2 = x * x;
    const float e = __builtin_amdgcn_exp2f(x * (k3 * x2 + k1));
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}
// The same to fp32 precision: the quotient x / d and the sum d = 1 + 2^t with their remainders. 11 full-rate operations and two others instead of tanhf's, whose time stood behind every tile of
// the fp32 MLP (10656 x 3072 x 768 286 -> 277 us).
__device__ __forceinline__ float gelu_tanh_precise(float x) {
    const float k1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
    const float e = __builtin_amdgcn_exp2f(x * fmaf(k1 * 0.044715f, x * x, k1)), d = 1.0f + e, r = __builtin_amdgcn_rcpf(d), q = x * r;
    const float rest = fmaf(-q, e - (d - 1.0f), fmaf(-q, d, x));
    return __builtin_amdgcn_div_fixupf(fmaf(rest, r, q), d, x);  // (infinities)
}
__device__ __forceinline__ float silu_precise(float x) { return x / (1.0f + expf(-x)); }

// the value of another lane of the same row of 16 lanes, chosen by a DPP control word (no trip through the LDS crossbar)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// RMSNorm's factor of a head of 64 * NV values (modules.cpp:192-198), of which each of 16 consecutive lanes has the squares of NV groups of four. For the fp32 path's two forms of it, in the
// projection's epilogue and in a kernel of its own: explicit multiply-adds and one order of the sums, so that they have the same bits.
__device__ __forceinline__ float head_squares(const float (&v)[4]) { return fmaf(v[0], v[0], v[1] * v[1]) + fmaf(v[2], v[2], v[3] * v[3]); }
template <int NV>
__device__ __forceinline__ float head_factor(float ss, float eps) {
    ss += dpp_move<0xB1>(ss);   // quad_perm [1,0,3,2]
    ss += dpp_move<0x4E>(ss);   // quad_perm [2,3,0,1]
    ss += dpp_move<0x141>(ss);  // row_half_mirror
    ss += dpp_move<0x140>(ss);  // row_mirror
    return 1.0f / sqrtf(fmaf(ss, 1.0f / (64 * NV), eps));
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// ---- direct global -> LDS loads and the tile order of the GEMM kernels ----
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;

// s_waitcnt vmcnt(n) with the other counters left unconstrained (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[15:14])
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup -> output tile. The hardware hands consecutive workgroup ids to the 8 XCDs in turn, and each XCD has its own L2, so
// the workgroups that land on one XCD should share as few A row panels and W column panels as possible. When the tile grid
// divides that way, the XCDs take a 4 x 2 arrangement of rectangular blocks of it (for 32 x 24 tiles: 8 x 12 each, 8 + 12 panels
// through that L2 instead of 4 + 24 with contiguous runs of tile rows), walked in bands of 4 tile rows so that the 32 tiles an XCD
// works on at a time form a 4 x 8 patch. Otherwise every XCD gets a contiguous run of tiles, walked in bands of 2 tile rows
// (measured over 1, 2, 3, 4, 8, 16 on the 24-block forward).
__device__ __forceinline__ void tile_of_workgroup(int wg, int tiles_m, int tiles_n, int& tile_m, int& tile_n) {
    constexpr int XCDS = 8, XR = 4, XC = 2, BAND = 4, GROUP_M = 2;
    const int total = tiles_m * tiles_n;
    const int xcd = wg % XCDS, local = wg / XCDS;
    if (tiles_m % (XR * BAND) == 0 && tiles_n % XC == 0) {
        const int bm = tiles_m / XR, bc = tiles_n / XC;  // the XCD's block: bm x bc tiles, exactly total / 8
        const int band = local / (BAND * bc), r = local % (BAND * bc);
        tile_m = (xcd / XC) * bm + band * BAND + r % BAND;
        tile_n = (xcd % XC) * bc + r / BAND;
        return;
    }
    const int per = (total + XCDS - 1) / XCDS, tall = (total % XCDS) ? (total % XCDS) : XCDS;  // `tall` XCDs get `per` tiles, the rest per-1
    const int t = (xcd < tall) ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
    const int in_group = GROUP_M * tiles_n, group = t / in_group, first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    tile_m = first_m + (t % in_group) % gsize;
    tile_n = (t % in_group) / gsize;
}

// ---- reading ahead ----
// Memory that launches to come are about to stream (weights); as much of it as fits a launch's idle workgroup slots is read once, in order,
// so that it lies in the last-level cache (256 MB, shared by the XCDs) when they ask for it.
constexpr int MAX_AHEAD = 7;
struct Ahead {
    const char* p[MAX_AHEAD];
    uint32_t bytes[MAX_AHEAD];
    // keeps the first `budget` bytes and says how many there are
    size_t trim(size_t budget) {
        size_t taken = 0;
        for (int i = 0; i < MAX_AHEAD; i++) {
            if (bytes[i] > budget - taken) bytes[i] = (uint32_t)(budget - taken);
            taken += bytes[i];
        }
        return taken;
    }
};
// One load per 128-byte line of every run, the value dropped: workgroup `wg` of `wgs`, NT threads each.
// Attention leaves HBM idle and the layers behind it wait for their weights (a launch of 333 / 1178 / 2356 / 4250 rows of mlp-1 and mlp-2
// takes 51 / 74 / 108 / 173 us with weights from HBM, 36 / 60 / 94 / 156 from the last-level cache), so the workgroup slots that its
// last round leaves free stream the block's remaining weights: forwards of 256px 2967 -> 2947 us, 512px 4631 -> 4548, its guided pair 6519 ->
// 6442, 1024px 12610 -> 12505. (The same in the LayerNorm launches, 16 MB each: 256px 0.9 % slower, 1024px 0.5 % faster.)
template <int NT>
__device__ __forceinline__ void read_ahead(const Ahead& a, unsigned wg, unsigned wgs) {
    constexpr uint32_t LINE = 128, UNROLL = 4;
    const uint32_t stride = wgs * NT;
#pragma unroll
    for (int s = 0; s < MAX_AHEAD; s++) {
        const uint32_t lines = a.bytes[s] / LINE;  // (runs are whole lines, or their last few bytes are left out)
        for (uint32_t l = wg * NT + threadIdx.x; l < lines; l += stride * UNROLL) {
            uint32_t v[UNROLL];
#pragma unroll
            for (uint32_t i = 0; i < UNROLL; i++) v[i] = *reinterpret_cast<const uint32_t*>(a.p[s] + (size_t)min(l + i * stride, lines - 1) * LINE);
#pragma unroll
            for (uint32_t i = 0; i < UNROLL; i++) asm volatile("" ::"v"(v[i]));
        }
    }
}

// ---- modulation projections of the bf16 path ----
// out (B, N) = y (B, K) @ W + bias, W bf16 as panels of 64 columns (N/64, K, 64). A panel is K * 128 bytes that one workgroup streams from
// end to end; the launches' own kernel is in small_linear.hip, and a GEMM launch that leaves compute units idle takes panels of the NEXT
// block along (AdaCarry), in workgroups behind those of its tiles.
struct AdaJob {
    const bf16_t* W;
    const float* bias;
    float* out;
    int N, ld;  // columns (whole panels) and the row stride of out
};
constexpr int ADA_CARRY_JOBS = 3, ADA_CARRY_ROWS = 4;  // what a GEMM launch takes along at most: the two streams of a block and the output layer; batch elements
constexpr int ADA_SLICES = 32;
struct AdaWork {
    AdaJob job[ADA_CARRY_JOBS];
    const float* y;
    int B, K;
    int first, count;  // panels of this launch, counted over the jobs
};
constexpr int ada_lds_bytes(int rows, int K) { return (rows * K + ADA_SLICES * rows * 64) * 4; }
// y transposed into LDS, xs[k][m]
template <int NT, int M>
__device__ __forceinline__ void ada_stage_rows(const float* __restrict__ y, int B, int K, float* xs) {
#pragma unroll
    for (int m = 0; m < M; m++)
        for (int k = threadIdx.x; k < K; k += NT) xs[k * M + m] = m < B ? y[(long long)m * K + k] : 0.f;
    __syncthreads();
}
// One panel. A thread has 4 columns and one (NT = 512) or two of the 32 slices of K, 16 rows of weights in flight; the order of the sums does
// not depend on NT or M (explicit multiply-adds), so that a row has the same bits in either kernel and in any batch.
// ONCE: nobody reads these weights again in a forward, so they are not to push the blocks' activations and the weights that attention reads
// ahead out of the last-level cache (non-temporal loads; forwards of 256px, 512px, its pair 0.6, 0.7, 0.6 % less). The launches that do nothing else
// read them with plain loads: a block that is called over and over finds them in the cache (106.3 -> 104 us).
template <int NT, int M, bool ONCE>
__device__ __forceinline__ void ada_panel(const bf16_t* __restrict__ W, const float* __restrict__ bias, float* __restrict__ out, int ld, int B, int K,
                                          const float* xs, float* red) {
    const int cg = threadIdx.x % 16, kper = K / ADA_SLICES;
    for (int sl = threadIdx.x / 16; sl < ADA_SLICES; sl += NT / 16) {
        const bf16_t* p = W + ((long long)sl * kper) * 64 + cg * 4;
        const float* xk = xs + sl * kper * M;
        float acc[M][4];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[m][j] = 0.f;
        auto add = [&](int k, const uint2 v) {
            const float w[4] = {__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float xv = xk[k * M + m];
#pragma unroll
                for (int j = 0; j < 4; j++) acc[m][j] = fmaf(xv, w[j], acc[m][j]);
            }
        };
        auto row = [](const bf16_t* q) {
            const unsigned long long* p8 = reinterpret_cast<const unsigned long long*>(q);
            return __builtin_bit_cast(uint2, ONCE ? __builtin_nontemporal_load(p8) : *p8);
        };
        constexpr int U = 16;  // rows of weights in flight (and as many again while they are used)
        uint2 v[U], n[U];
        const int whole = kper / U * U;
        if (whole) {
#pragma unroll
            for (int i = 0; i < U; i++) v[i] = row(p + i * 64);
            for (int k = 0; k < whole; k += U) {
                const bf16_t* q = p + min(k + U, kper - U) * 64;  // in the end the last U rows: brings those of the remainder near
#pragma unroll
                for (int i = 0; i < U; i++) n[i] = row(q + i * 64);
#pragma unroll
                for (int i = 0; i < U; i++) add(k + i, v[i]);
#pragma unroll
                for (int i = 0; i < U; i++) v[i] = n[i];
            }
        }
        // The rest requested together as well, rows beyond the end as the last one once more. Row by row, each behind its own load, a panel of 768, 2432
        // and 192 rows (24, 76 and 6 per slice) took its workgroup 6.4, 13.1 and 3.5 us instead of 4.0, 9.0 and 2.5 (512 threads, one row of y), and
        // forwards of 512px at width 768 2785 instead of 2319, of 256px at width 2432 (eight blocks) 2031 instead of 1570.
        int rest = kper - whole;
        asm volatile("" : "+s"(rest));  // (or sixteen comparisons are kept, through spilled scalar registers, from one panel to the next)
        if (rest) {
            const bf16_t* q = p + whole * 64;
#pragma unroll
            for (int i = 0; i < U; i++) v[i] = row(q + min(i, rest - 1) * 64);
#pragma unroll
            for (int i = 0; i < U; i++)
                if (i < rest) add(whole + i, v[i]);
        }
#pragma unroll
        for (int m = 0; m < M; m++) *reinterpret_cast<float4*>(red + (sl * M + m) * 64 + cg * 4) = make_float4(acc[m][0], acc[m][1], acc[m][2], acc[m][3]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < M * 64; e += NT) {
        const int m = e / 64, c = e % 64;
        if (m < B) {
            float s = 0.f;
#pragma unroll
            for (int sl = 0; sl < ADA_SLICES; sl++) s += red[(sl * M + m) * 64 + c];
            out[(long long)m * ld + c] = s + bias[c];
        }
    }
    __syncthreads();
}
// Workgroup `wg` of `wgs` that a GEMM launch has added to its own
template <int NT, int M>
__device__ __forceinline__ void ada_carried_rows(const AdaWork& a, int wg, int wgs, char* smem) {
    float* xs = reinterpret_cast<float*>(smem);
    ada_stage_rows<NT, M>(a.y, a.B, a.K, xs);
    for (int i = wg; i < a.count; i += wgs) {
        int t = a.first + i, j = 0;
        while (j + 1 < ADA_CARRY_JOBS && t >= a.job[j].N / 64) t -= a.job[j++].N / 64;
        const AdaJob& q = a.job[j];
        ada_panel<NT, M, true>(q.W + (long long)t * 64 * a.K, q.bias + t * 64, q.out + t * 64, q.ld, a.B, a.K, xs, xs + M * a.K);
    }
}
template <int NT>
__device__ __forceinline__ void ada_carried(const AdaWork& a, int wg, int wgs, char* smem) {
    if (a.B == 1) ada_carried_rows<NT, 1>(a, wg, wgs, smem);
    else if (a.B == 2) ada_carried_rows<NT, 2>(a, wg, wgs, smem);
    else ada_carried_rows<NT, ADA_CARRY_ROWS>(a, wg, wgs, smem);
}
// What is left of a block's panels; a GEMM launch takes `first` onwards as many as it has room for and moves `first` on.
struct AdaCarry {
    AdaWork work{};
    int total = 0;
    bool last = false;  // the block's last launch
    Ahead ahead{};      // what the launch may read ahead once it has taken its panels
    int left() const { return total - work.first; }
};
int ada_panels(const float* y, int B, int K, const AdaJob* jobs, int n, hipStream_t st);
int pack_ada_panels(const float* W, bf16_t* out, int K, int N, hipStream_t st);

// ---- epilogues of the GEMM kernels ----
enum Epilogue : int {
    EPI_BIAS = 0,         // out = acc + bias
    EPI_BIAS_GELU = 1,    // out = gelu_tanh(acc + bias)
    EPI_BIAS_SILU = 2,    // out = silu(acc + bias)
    EPI_GATE_RESID = 3,   // out = resid + gate[m / rows_per_batch][n] * (acc + bias)   (out may alias resid)
    EPI_BIAS_ROWADD = 4,  // out = acc + bias + table[m % rows_per_batch][n]
    EPI_QKV_NORM = 5,     // packed q|k|v projection (N = 3C): acc + bias, then per-head RMSNorm (64 columns, eps 1e-6) of the q and k thirds
                          // with weights `gate` (q) and `resid` (k), each 64 floats; C is given in gate_ld. fp32: A in pieces
};

struct GemmEpilogueArgs {
    const float* bias = nullptr;   // (N) or null
    const float* gate = nullptr;   // (B, gate_ld) for EPI_GATE_RESID
    int gate_ld = 0;
    const float* resid = nullptr;  // (M, ldc) fp32 for EPI_GATE_RESID
    const float* table = nullptr;  // (rows_per_batch, N) for EPI_BIAS_ROWADD
    int rows_per_batch = 1;
    const float* a_scale = nullptr;  // fp8 GEMM: factor per row of A (M) and per output column (N); null = 1
    const float* w_scale = nullptr;
};

// fp32 GEMM: out(M,N) = A(M,K; lda) @ W(K, ldw)[:, n0:n0+N] (+ epilogue); out fp32 with row stride ldc.
int gemm_f32(const float* A, int lda, const float* W, int ldw, int n0, float* out, int ldc, int M, int N, int K, int epi, const GemmEpilogueArgs& ea,
             hipStream_t st);
// Up to three independent fp32 GEMMs with the same epilogue kind: one launch where all rows are made of whole 16-byte chunks.
struct GemmF32Problem {
    const float* A;
    const float* W;
    float* out;
    int lda, ldw, n0, ldc, M, N, K;
    GemmEpilogueArgs ea;
    bool a_pieces = false;    // A: a matrix of pieces (pieces.hpp), in all problems of the launch and where gemm_f32_takes_a_pieces
    bool out_pieces = false;  // EPI_BIAS_GELU, A in pieces: the output as a matrix of pieces of ldc columns
};
bool gemm_f32_takes_a_pieces(const float* W, int ldw, int n0, int N, int K);
int gemm_f32_grouped(const GemmF32Problem* probs, int n, int epi, hipStream_t st);
extern int g_gemm_f32_tile, g_gemm_f32_no_pieces;
// bf16 GEMM: A bf16 (M,K) row-major; Wp = packed weight, bf16, K-contiguous (see GemmBf16Problem::w_tiled); out bf16 (out_is_f32 = 0) or fp32.
int gemm_bf16(const bf16_t* A, const bf16_t* Wp, bool w_tiled, void* out, int out_is_f32, int ldc, int M, int N, int K, int epi, const GemmEpilogueArgs& ea,
              hipStream_t st);
// Up to three independent bf16 GEMMs (same epilogue kind and output type) in one launch.
struct GemmBf16Problem {
    const bf16_t* A;
    const bf16_t* Wp;
    void* out;
    int ldc, M, N, K;
    GemmEpilogueArgs ea;
    // Wp as K tiles (K/64, N, 64): the workgroups of a launch walk along K side by side, and what they ask for at a time is then one run of
    // memory (128 N bytes) instead of 128 bytes out of every row. With cold weights, 333 / 1178 / 2356 rows: mlp-2 30.1 -> 27.4, 44.6 -> 42.8,
    // 60.8 -> 57.8 us; mlp-1 of 333 rows 20.0 -> 18.8; nothing with warm ones.
    bool w_tiled = false;
    const GemmBf16Problem* then = nullptr;  // EPI_GATE_RESID: a second layer of the same M, N, K and out whose residual is this one's result
};
extern std::atomic<long long> g_gemm_bf16_launches;  // kernels launched by the bf16 GEMM so far (for per-launch profile figures)
int gemm_bf16_grouped(const GemmBf16Problem* probs, int n, int out_is_f32, int epi, hipStream_t st, AdaCarry* carry = nullptr);
// The same with OCP fp8 (e4m3) operands: A (M,K) and Wp (N,K) are bytes, K % 128 == 0, and the accumulators are multiplied by
// ea.a_scale[m] * ea.w_scale[n] before the epilogue (epilogues: bias, bias+GELU, gate+residual, q|k|v with qk-norm).
int gemm_fp8_grouped(const GemmBf16Problem* probs, int n, int out_is_f32, int epi, hipStream_t st);
// fp8 quantisation. Rows of a bf16 matrix: aq[m][k] = fp8(A[m][k] / s[m]), s[m] = max_k |A[m][k]| / 448 (one common s with per_tensor).
int quantize_rows_fp8(const bf16_t* A, uint8_t* aq, float* scale, int M, int K, int per_tensor, hipStream_t st);
// A (K,N) fp32 weight -> (N,K) fp8 with one factor per output column n (one common factor with per_tensor)
int quantize_weight_fp8(const float* W, uint8_t* wq, float* scale, int K, int N, int per_tensor, hipStream_t st);
// (K,N) fp32 row-major -> (N,K) bf16 row-major, or (tiled, K % 64 == 0) as K tiles (K/64, N, 64)
int pack_weight_bf16(const float* W, bf16_t* out, int K, int N, bool tiled, hipStream_t st);
int cast_f32_to_bf16(const float* in, bf16_t* out, long long n, hipStream_t st);
// (K,N) fp32 -> (N,K) fp32
int transpose_f32(const float* W, float* out, int K, int N, hipStream_t st);
int patch_embed_direct(const float* latent, float* out, const float* kernel, const float* bias, int B, int H, int W, int Cin, int C, int p, int pos_max,
                       int base_height, hipStream_t st);

// LayerNorm without affine over the last axis + optional modulation: out = LN(x)*(1+scale[b])+shift[b]; a second modulated
// output (shift2/scale2/out2) may be produced from the same normalised row. scale/shift rows have stride mod_ld.
// out_bf16 selects bf16 (1) or fp32 (0) outputs.
// LayerNorm (no affine) + optional modulation of one tensor (B, T, C) into one or two outputs; two such jobs with the same C
// and eps (the two streams of a block) can share a launch
struct LayerNormJob {
    const float* x;
    void* out;
    void* out2;
    const float* shift;
    const float* scale;
    const float* shift2;
    const float* scale2;
    int mod_ld, B, T;
};
enum LayerNormOut : int { LN_F32 = 0, LN_BF16 = 1, LN_PIECES = 2 };  // fp32, bf16, a matrix of bf16 pieces (pieces.hpp)
int layernorm_modulate_pair(const LayerNormJob* jobs, int n, float eps, int C, int out, hipStream_t st);
int layernorm_modulate(const float* x, void* out, void* out2, const float* shift, const float* scale, const float* shift2, const float* scale2,
                       int mod_ld, float eps, int B, int T, int C, int out_bf16, hipStream_t st);
int layernorm_full(const float* x, float* y, float* mean, float* rstd, const float* w, const float* bias, float eps, long long rows, int C,
                   hipStream_t st);
// RMSNorm over groups of `hs` consecutive values inside rows of stride `ld` (in place allowed): x[r*ld + g*hs + i], g < groups
int rmsnorm_rows(const float* x, float* y, const float* w, float* rms, float eps, long long rows, int groups, int hs, int ld_in, int ld_out,
                 hipStream_t st);
// In-place per-head RMSNorm of the q and k thirds of packed q|k|v rows (3 * heads * hs values, row stride ld), several buffers per launch
struct QkNormJob {
    float* qkv;
    const float *wq, *wk;
    long long rows;
};
int qk_norm_rows(const QkNormJob* jobs, int n, float eps, int heads, int hs, int ld, hipStream_t st);
// Whether these go by whole chunks (head_squares, head_factor); else the sums have another order
bool qk_norm_by_chunks(const QkNormJob* jobs, int n, int hs, int ld);
int unary_op(const float* in, float* out, long long n, int act, hipStream_t st);
int add_op(const float* a, const float* b, float* out, long long n, hipStream_t st);
int add_silu_op(const float* a, const float* b, float* out, long long n, hipStream_t st);
int modulate_op(const float* in, float* out, const float* shift, const float* scale, int B, int T, int C, hipStream_t st);  // scale null -> gate with `shift` as gate
int gate_op(const float* in, float* out, const float* gate, int B, int T, int C, hipStream_t st);
int copy_rows(const float* in, long long in_batch_stride, float* out, long long out_batch_stride, int B, long long n_per_batch, hipStream_t st);
int timestep_embedding(const float* t, float* out, int B, int dim, hipStream_t st);
int pos_embed_table(float* out, int C, int height, int width, int base_size, hipStream_t st);
int pos_embed_crop(const float* table, float* out, int max_size, int h, int w, int C, hipStream_t st);
// cropped table written directly (what PatchEmbedding needs): out (h*w, C)
int pos_embed_cropped(float* out, int C, int max_size, int base_size, int h, int w, hipStream_t st);
int conv2d_direct(const float* in, float* out, const float* kernel, const float* bias, int B, int kh, int kw, int Cin, int Cout, int ih, int iw, int oh,
                  int ow, int stride, int pad, hipStream_t st);
// latent (B,Cin,H,W) -> patch rows (B*h*w, Cin*p*p), k index = (ic*p + r)*p + s; fp32 or bf16 output
int im2col_patches(const float* latent, void* out, int out_bf16, int B, int Cin, int H, int W, int p, hipStream_t st);
// tokens (B, h*w, p*p*Cin) -> pixels (B,Cin,H,W)
int unpatchify(const float* tokens, float* out, int B, int Cin, int H, int W, int p, hipStream_t st);
int unpatchify_cfg_euler(const float* tokens, const float* latent, float* out, int n_samples, int Cin, int H, int W, int p, float guidance, float dsigma,
                         hipStream_t st);

// Small-M linear (M <= 8): out(M, N) = act(x(M,K) @ W[:, n0:n0+N] + b[n0:n0+N]); W fp32 (K, ldw), N-contiguous.
struct SmallLinearJob {
    const float* W;
    const float* bias;
    float* out;
    int N;    // columns of this job
    int ldw;  // row stride of W
    int n0;   // first column
    const float* x = nullptr;  // this job's own left operand (M, K) instead of the launch's, or null
    int K = 0;                 // its depth (with x)
};
constexpr int SMALL_LINEAR_JOBS_PER_LAUNCH = 52;
int small_linear_batched(const float* x, int M, int K, const SmallLinearJob* jobs_host, int n_jobs, int act /* -1 none */,
                         hipStream_t st);

// Attention. Two token segments (segment 0 first in the joint sequence); each has its own q/k/v/out pointers and row strides.
struct AttnSegments {
    const void* q[2];
    const void* k[2];
    const void* v[2];
    void* out[2];
    int ld_qkv[2];  // row stride (elements) of q/k/v
    int ld_out[2];
    int T[2];       // keys/values per batch element in each segment (T[1] may be 0)
    int Tq[2];      // queries per batch element in each segment (equal to T for self-attention)
    const float* rms_q[2];  // bf16 kernel only: fused per-head RMSNorm weights (null = no norm)
    const float* rms_k[2];
    bool out_pieces = false;  // fp32 kernel, heads of 64 or 128: the outputs as matrices of bf16 pieces (pieces.hpp) of ld_out columns
};
int attention_f32(const AttnSegments& s, int B, int NH, int HS, hipStream_t st);
extern int g_attention_f32_no_pieces;
int attention_bf16(const AttnSegments& s, int B, int NH, int HS, hipStream_t st);
// Up to three attention problems in one launch. kv_splits[i] > 1 (or null: all 1) splits the keys of set i into that many runs, one
// work item each, whose partial results go through split_ws[i] (attention_bf16_split_workspace_floats floats) and are merged by a
// second, small kernel. attention_bf16_context_splits: the number of splits that pays for the Tc context queries of a joint
// attention next to Tx latent ones, or 0 when the plain one-set launch is the better choice.
// ahead (or null): what the launch's idle workgroup slots read ahead.
int attention_bf16_multi(const AttnSegments* sets, const int* kv_splits, float* const* split_ws, int n, int B, int NH, int HS, hipStream_t st,
                         const Ahead* ahead = nullptr, AdaCarry* carry = nullptr);
int attention_bf16_context_splits(int Tc, int Tx, int NH, bool dual);
size_t attention_bf16_split_workspace_floats(int B, int NH, int Tc, int splits);

}  // namespace sd3
