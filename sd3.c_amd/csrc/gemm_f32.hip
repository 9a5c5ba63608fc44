// fp32 GEMM on the gfx950 matrix cores, for the fp32 parity path and the fp32 operators:
//   out(M,N) = A(M,K) @ W(K,N)[:, n0:n0+N] + epilogue
// replacing linear / partial_linear of the reference (modules.cpp:475-511, naive triple loops).
//
// gemm_f32_pieces_kernel (operands as three bf16 pieces each, on the bf16 matrix instruction) takes depths from 512 on;
// gemm_f32_tile_kernel (v_mfma_f32_16x16x4_f32) everything else whose operand rows are made of whole 16-byte chunks; both up to three problems
// per launch. gemm_f32_kernel (v_mfma_f32_32x32x2_f32, 128x128x16 tiles, element-wise loads) takes operands of any other stride or alignment.
#include <type_traits>

#include "common.hpp"
#include "pieces.hpp"
#include "tiles_f32.hpp"

namespace sd3 {

namespace {
constexpr int BM = 128, BN = 128, BK = 16;  // tile of the any-stride kernel
constexpr int A_PITCH = BM + 4;  // As[k][m]: 4*(BM+4) = 528 = 16 mod 64 -> the four k-quads of a wave hit disjoint banks on store
constexpr int B_PITCH = BN + 4;

struct EpiDev {
    const float* bias;
    const float* gate;
    const float* resid;
    const float* table;
    int gate_ld;
    int rows_per_batch;
};

template <int EPI>
__device__ __forceinline__ float apply_epilogue(float acc, int m, int n, int n_glob, const EpiDev& e, long long out_idx) {
    float v = acc;
    if (e.bias) v += e.bias[n_glob];
    if (EPI == EPI_BIAS_GELU) v = gelu_tanh_precise(v);
    else if (EPI == EPI_BIAS_SILU) v = silu_precise(v);
    else if (EPI == EPI_GATE_RESID) {
        v *= e.gate[(long long)(m / e.rows_per_batch) * e.gate_ld + n];
        v += e.resid[out_idx];
    } else if (EPI == EPI_BIAS_ROWADD) {
        v += e.table[(long long)(m % e.rows_per_batch) * /*table row stride = N, passed in gate_ld*/ e.gate_ld + n];
    }
    return v;
}

template <int EPI>
__global__ void __launch_bounds__(256) gemm_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw, int n0,
                                                       float* __restrict__ out, int ldc, int M, int N, int K, EpiDev epi) {
    __shared__ float As[BK * A_PITCH];
    __shared__ float Bs[BK * B_PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m_blk = blockIdx.y * BM, n_blk = blockIdx.x * BN;

    // global -> register staging: A tile 128x16 (2 float4 per thread along k), W tile 16x128 (2 float4 per thread along n)
    const int a_row = tid >> 2, a_kq = (tid & 3) * 4;  // rows a_row and a_row+64
    const int b_k = tid >> 5, b_n = (tid & 31) * 4;    // k rows b_k and b_k+8
    float4 ra[2], rb[2];

    auto load_tiles = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int m = m_blk + a_row + i * 64;
            const int k = k0 + a_kq;
            float t[4];
#pragma unroll
            for (int j = 0; j < 4; j++) t[j] = (m < M && k + j < K) ? A[(long long)m * lda + k + j] : 0.f;
            ra[i] = make_float4(t[0], t[1], t[2], t[3]);
            const int kk = k0 + b_k + i * 8;
            const int n = n_blk + b_n;
#pragma unroll
            for (int j = 0; j < 4; j++) t[j] = (kk < K && n + j < N) ? W[(long long)kk * ldw + n0 + n + j] : 0.f;
            rb[i] = make_float4(t[0], t[1], t[2], t[3]);
        }
    };
    auto store_tiles = [&]() {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int m = a_row + i * 64;
            As[(a_kq + 0) * A_PITCH + m] = ra[i].x;
            As[(a_kq + 1) * A_PITCH + m] = ra[i].y;
            As[(a_kq + 2) * A_PITCH + m] = ra[i].z;
            As[(a_kq + 3) * A_PITCH + m] = ra[i].w;
            *reinterpret_cast<float4*>(&Bs[(b_k + i * 8) * B_PITCH + b_n]) = rb[i];
        }
    };

    f32x16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const int l32 = lane & 31, lk = lane >> 5;
    load_tiles(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
        store_tiles();
        __syncthreads();
        if (k0 + BK < K) load_tiles(k0 + BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 2) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++) a[i] = As[(kk + lk) * A_PITCH + wm * 64 + i * 32 + l32];
#pragma unroll
            for (int j = 0; j < 2; j++) b[j] = Bs[(kk + lk) * B_PITCH + wn * 64 + j * 32 + l32];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    // C layout of the 32x32 MFMA: lane holds column (lane % 32); register r is row 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int n = n_blk + wn * 64 + j * 32 + l32;
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m_blk + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
                if (m < M) {
                    const long long idx = (long long)m * ldc + n;
                    out[idx] = apply_epilogue<EPI>(acc[i][j][r], m, n, n0 + n, epi, idx);
                }
            }
        }
}

// ---- the tile kernel ----
// fp32 matrix instructions are slow (64 FLOP per cycle and SIMD: a 64x64 wavefront tile works 2048 cycles on 16 k values), so the
// matrix unit is the bound as soon as every SIMD has a tile; LDS and global traffic are not. What costs is SIMDs without work: the
// layers of a 512 x 512 image are 96 tiles of 128x128 on 256 compute units. Hence a range of tile shapes down to 32x32, chosen per
// launch by the number of rounds (pick_f32_tile), and one launch for the layers of the same kind of both token streams.
//
// Both operands go global -> LDS by direct loads. A tile rows are 128 bytes (32 k values), 16-byte chunks XOR-swizzled by the row as
// in the bf16 kernel's 16x16 layout: lane l reads chunk 4h + l/16 of row l%16, i.e. k values 16h + 4(l/16) .. +3 of one half h of the
// tile, and matrix instruction s of the half contracts k = 16h + 4g + s, g = 0..3 (the same order of k whatever the tile shape:
// a row's result depends on neither the shape nor the grouping). W stays N-contiguous as the reference stores it: lane l reads the NJ
// consecutive columns NJ*(l%16) .. of its k row, one for each of its NJ column blocks, so column block j holds columns NJ*c + j and
// a lane ends with NJ consecutive columns of a row: the epilogue stores straight from the accumulators, 16 lanes covering 16*NJ columns.
struct TileProb {
    const float* A;  // (A in pieces: a matrix of them, pieces.hpp)
    const float* W;
    float* out;
    int lda, ldw, ldc, M, N, K, n0;
    bool out_pieces;  // EPI_BIAS_GELU: a matrix of pieces of ldc columns
    EpiDev epi;
};
constexpr int MAX_PROBS = 3;
struct TileProbSet {
    TileProb p[MAX_PROBS];
    int end[MAX_PROBS];  // running totals of tiles
};
constexpr int TK = 32;  // k values per tile = 128-byte rows of A in LDS
__device__ __align__(16) float zero_chunk[4];  // source of the k values beyond K (A and W)

// NJ consecutive floats, loaded and stored as one: `lds` there (aligned as the layout has it), `mem` at any float of global memory, where
// wide accesses need no more than the alignment of their elements
template <int NJ>
struct Cols;
template <>
struct Cols<4> { typedef f32x4_t lds; typedef f32x4_t mem __attribute__((aligned(4))); };
template <>
struct Cols<2> { typedef f32x2_t lds; typedef f32x2_t mem __attribute__((aligned(4))); };
template <>
struct Cols<1> { typedef float lds; typedef float mem; };
template <typename T, int NJ>
__device__ __forceinline__ void load_as(const float* p, float (&v)[NJ]) {
    const T t = *reinterpret_cast<const T*>(p);
    __builtin_memcpy(v, &t, sizeof(v));
}
template <int NJ>
__device__ __forceinline__ void load_cols(const float* p, float (&v)[NJ]) {
    load_as<typename Cols<NJ>::mem>(p, v);
}
template <int NJ>
__device__ __forceinline__ void store_cols(float* p, const float (&v)[NJ]) {
    typename Cols<NJ>::lds t;
    __builtin_memcpy(&t, v, sizeof(t));
    *reinterpret_cast<typename Cols<NJ>::mem*>(p) = t;
}

// Epilogue and stores of TI x NJ blocks of 16x16. C layout of a block: lane = column l%16 (of block j: column NJ*(l%16) + j), register r = row 4*(l/16) + r;
// m0: the lane's first row, n: its first column. Everything that is to be read is requested before the first store and waited for together: row by row, each behind the other's store,
// 16 rows were 16 trips to memory. With the gate, 10656 x 768 x 768: tiles of 128x128 93 -> 84 us, of
// 64x64 132 -> 116; 333 x 1536 x 1536 25.7 -> 23.5.
// LEAN: row by row all the same, for the 256x128 tiles of the kernel that splits A itself, whose K loop spills registers beside anything else (K = 6144 370 -> 486 us). PIECES: the output may be one of pieces (A comes in them).
template <int TI, int NJ, int EPI, bool PIECES, bool LEAN = false>
__device__ __forceinline__ void store_tile(const TileProb& pr, const f32x4_t (&acc)[TI][NJ], int m0, int n) {
    asm volatile("" : "+v"(m0), "+v"(n));  // (or addresses are formed in front of the K loop and held through it)
    const int m_wave = __builtin_amdgcn_readfirstlane(m0) & ~15;  // the wavefront's first row
    if (n >= pr.N || m_wave >= pr.M) return;  // (N is a multiple of 4, so a lane's columns are all inside or all outside)
    const EpiDev& e = pr.epi;
    float bias[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) bias[j] = e.bias ? e.bias[pr.n0 + n + j] : 0.f;
    auto arrived = [](float (&v)[NJ]) {  // (named, so that it is waited for here)
#pragma unroll
        for (int j = 0; j < NJ; j++) asm volatile("" : "+v"(v[j]));
    };
    if constexpr (EPI == EPI_BIAS_GELU && PIECES) {
        if (pr.out_pieces) {
            // Rows m0 + 16 i + r, m0 = 4(l/16) mod 16: the places of a block's rows in 32-bit offsets, the blocks in a scalar address (a 64-bit address for every
            // store and plane costs more than the split)
            const PieceMatrix to(pr.out, pr.M, pr.ldc);
            const unsigned at[2] = {(unsigned)piece_index(m0 & 15, n, to.K) * 2, (unsigned)(piece_index((m0 & 15) + 2, n, to.K) - 64) * 2};
            arrived(bias);
#pragma unroll
            for (int i = 0; i < TI; i++) {
                char* const block = reinterpret_cast<char*>(to.p) + (long long)(m_wave / 16 + i) * to.K * 32;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float v[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; j++) v[j] = gelu_tanh_precise(acc[i][j][r] + bias[j]);
                    uint32_t piece[3][(NJ + 1) / 2];
                    pieces_for_memory<NJ>(v, piece);
                    if (m0 + i * 16 + r < pr.M)
#pragma unroll
                        for (int p = 0; p < 3; p++) __builtin_memcpy(__builtin_assume_aligned(block + p * to.plane * 2 + at[r / 2] + r * 64, NJ * 2), piece[p], NJ * 2);
                }
            }
            return;
        }
    }
    const int rpb = e.rows_per_batch;
    if constexpr (EPI == EPI_QKV_NORM) {
        // q and k: a wavefront's 64 columns are one head, four a lane. (16 x 666 tokens, width 768: 368 us and 49 in a kernel of its own -> 370)
        static_assert(NJ == 4, "a head per wavefront");
        const int third = __builtin_amdgcn_readfirstlane(n / e.gate_ld);
        float w[NJ] = {};
        if (third < 2) load_cols<NJ>((third ? e.resid : e.gate) + n % 64, w);
        arrived(bias);
        arrived(w);
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + i * 16 + r;
                float v[NJ];
#pragma unroll
                for (int j = 0; j < NJ; j++) v[j] = acc[i][j][r] + bias[j];
                if (third < 2) {
                    const float inv = head_factor<1>(head_squares(v), 1e-6f);
#pragma unroll
                    for (int j = 0; j < NJ; j++) v[j] = (v[j] * inv) * w[j];
                }
                if (m < pr.M) store_cols<NJ>(pr.out + (long long)m * pr.ldc + n, v);
            }
        return;
    }
    // Rows of at most two batch elements, as all but those of very few rows: a gate for each
    const int b_first = EPI == EPI_GATE_RESID ? m_wave / rpb : 0, b_last = EPI == EPI_GATE_RESID ? min(m_wave + TI * 16 - 1, pr.M - 1) / rpb : 0;
    if (!LEAN && b_last - b_first <= 1) {
        constexpr bool READS = EPI == EPI_GATE_RESID || EPI == EPI_BIAS_ROWADD;
        // (tiles with few registers to spare ask for half of their blocks' rows, and behind these for the others', before the first stores)
        constexpr int PARTS = READS && TI * NJ >= 16 ? 2 : 1, PI = TI / PARTS;
        float g[2][NJ], t[READS ? TI : 1][4][NJ];
        if (EPI == EPI_GATE_RESID) {
            load_cols<NJ>(e.gate + (long long)b_first * e.gate_ld + n, g[0]);
            load_cols<NJ>(e.gate + (long long)b_last * e.gate_ld + n, g[1]);
        }
        auto request = [&](int part) {
            if constexpr (READS) {
#pragma unroll
                for (int i = part * PI; i < (part + 1) * PI; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int m = min(m0 + i * 16 + r, pr.M - 1);
                        load_cols<NJ>(EPI == EPI_GATE_RESID ? e.resid + (long long)m * pr.ldc + n : e.table + (long long)(m % rpb) * e.gate_ld + n, t[i][r]);
                    }
            }
        };
        auto wait = [&](int part) {
            if constexpr (READS) {
#pragma unroll
                for (int i = part * PI; i < (part + 1) * PI; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) arrived(t[i][r]);
            }
        };
        auto value = [&](int i, int r, float (&v)[NJ]) {
            const bool second = EPI == EPI_GATE_RESID && m0 + i * 16 + r >= b_last * rpb;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                v[j] = acc[i][j][r] + bias[j];
                if (EPI == EPI_BIAS_GELU) v[j] = gelu_tanh_precise(v[j]);
                else if (EPI == EPI_BIAS_SILU) v[j] = silu_precise(v[j]);
                else if (EPI == EPI_GATE_RESID) v[j] = fmaf(v[j], second ? g[1][j] : g[0][j], t[READS ? i : 0][r][j]);
                else if (EPI == EPI_BIAS_ROWADD) v[j] += t[READS ? i : 0][r][j];
            }
        };
        request(0);
        arrived(bias);
        if (EPI == EPI_GATE_RESID) {
            arrived(g[0]);
            arrived(g[1]);
        }
        wait(0);
#pragma unroll
        for (int part = 0; part < PARTS; part++) {
            float out[PARTS > 1 ? PI : 1][4][NJ];
            if (PARTS > 1) {  // (the sums and what they were added to give way to the results, and these to the next requests)
#pragma unroll
                for (int i = 0; i < PI; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) value(part * PI + i, r, out[PARTS > 1 ? i : 0][r]);
                if (part + 1 < PARTS) {
                    request(part + 1);
                    wait(part + 1);
                }
            }
#pragma unroll
            for (int i = 0; i < PI; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + (part * PI + i) * 16 + r;
                    float v[NJ];
                    if (PARTS == 1) value(i, r, v);
                    if (m < pr.M) store_cols<NJ>(pr.out + (long long)m * pr.ldc + n, PARTS > 1 ? out[PARTS > 1 ? i : 0][r] : v);
                }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = m0 + i * 16 + r;
            if (m >= pr.M) continue;
            const long long idx = (long long)m * pr.ldc + n;
            float v[NJ], g[NJ], t[NJ];
            if (EPI == EPI_GATE_RESID) {
                load_cols<NJ>(e.gate + (long long)(m / rpb) * e.gate_ld + n, g);
                load_cols<NJ>(e.resid + idx, t);
            } else if (EPI == EPI_BIAS_ROWADD) {
                load_cols<NJ>(e.table + (long long)(m % rpb) * e.gate_ld + n, t);
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                v[j] = acc[i][j][r] + bias[j];
                if (EPI == EPI_BIAS_GELU) v[j] = gelu_tanh_precise(v[j]);
                else if (EPI == EPI_BIAS_SILU) v[j] = silu_precise(v[j]);
                else if (EPI == EPI_GATE_RESID) v[j] = fmaf(v[j], g[j], t[j]);
                else if (EPI == EPI_BIAS_ROWADD) v[j] += t[j];
            }
            store_cols<NJ>(pr.out + idx, v);
        }
}

// WHOLE_K: K is made of whole tiles in every problem
template <int TM, int TN, int WM, int WN, int STAGES, int EPI, bool WHOLE_K>
__global__ void __launch_bounds__(WM* WN * 64, 2) gemm_f32_tile_kernel(const TileProbSet set) {
    constexpr int NT = WM * WN * 64, TI = TM / WM / 16, NJ = TN / WN / 16;
    constexpr int A_BYTES = TM * 128, STAGE_BYTES = A_BYTES + TK * TN * 4;
    constexpr int LA = TM * 8 / NT, LB = TN * 8 / NT, CPR = TN / 4;  // 16-byte chunks per thread and tile; chunks per W row
    static_assert(TM * 8 % NT == 0 && TN * 8 % NT == 0 && TI >= 1 && (NJ == 1 || NJ == 2 || NJ == 4), "tile shape");
    // W rows whose k differs by 4 are read together; with fewer than 64 columns per wavefront their chunks are moved apart
    constexpr int WX = NJ == 4 ? 0 : NJ == 2 ? 8 : 4, WXM = NJ == 2 ? 1 : 3;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int w = blockIdx.x;
    const int which = (w >= set.end[0]) + (w >= set.end[1]);
    const TileProb& pr = set.p[which];
    const int M = pr.M, N = pr.N, K = pr.K;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tile_m, tile_n;
    tile_of_workgroup(w - (which ? set.end[which - 1] : 0), (M + TM - 1) / TM, (N + TN - 1) / TN, tile_m, tile_n);
    const int m_blk = tile_m * TM, n_blk = tile_n * TN;

    const float* ga[LA];
    const float* gb[LB];
    int ka[LA], kb[LB];            // k of the chunk within its tile
    unsigned a_off[LA], b_off[LB];  // WHOLE_K: bytes of the chunk behind the tile's first one
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int q = i * NT + tid, row = q >> 3;
        ka[i] = ((q & 7) ^ (row & 6)) * 4;
        ga[i] = pr.A + (long long)min(m_blk + row, M - 1) * pr.lda + ka[i];  // rows beyond M re-read the last one and are never stored
        a_off[i] = ((unsigned)min(row, M - 1 - m_blk) * pr.lda + ka[i]) * 4;
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int q = i * NT + tid;
        kb[i] = q / CPR;
        const int c = (q % CPR) ^ ((((kb[i] >> 2) & WXM) * WX) & (CPR - 1));
        gb[i] = pr.W + (long long)kb[i] * pr.ldw + pr.n0 + min(n_blk + c * 4, N - 4);
        b_off[i] = ((unsigned)kb[i] * pr.ldw + min(n_blk + c * 4, N - 4)) * 4;
    }
    const char* a_tile = reinterpret_cast<const char*>(pr.A + (long long)m_blk * pr.lda);
    const char* b_tile = reinterpret_cast<const char*>(pr.W + pr.n0);
    const long long b_step = (long long)TK * pr.ldw;
    const int nkt = (K + TK - 1) / TK;
    const float* zeros = zero_chunk;
    asm volatile("" : "+s"(zeros));  // (kept in registers: the compiler would fetch the address anew inside the loop)
    // requests the next tile (the pointers advance with every call); past the last one zeros, into a stage that nobody reads again.
    // No branches, so that the requests can be spread over the matrix instructions.
    // WHOLE_K: one scalar address per operand that moves on and a 32-bit offset per thread that does not, which the load takes as they are: a
    // 64-bit address per load costs the vector unit two or three operations between the matrix instructions and the load more cycles to issue. Past
    // the end the last tile once more. 1178 x 1536 x 6144 (128x64 tiles) 207 -> 180 us, 1178 x 4608 x 1536 150 -> 135, 10656 x 3072 x 768 375 -> 352,
    // 4096 x 6144 x 1536 557 -> 520 (149 of 157 TFLOP/s).
    auto issue_tile = [&](int kt, int stage) {
        const int left = K - kt * TK;
        char* sa = smem + stage * STAGE_BYTES + wave * 1024;
        char* sb = sa + A_BYTES;
        if constexpr (WHOLE_K) {
#pragma unroll
            for (int i = 0; i < LA; i++) {
                asm volatile("" : "+v"(a_off[i]));  // (or the compiler widens the offset outside the loop and adds it to the address inside)
                __builtin_amdgcn_global_load_lds((glb_ptr_t)(a_tile + a_off[i]), (lds_ptr_t)(sa + i * NT * 16), 16, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < LB; i++) {
                asm volatile("" : "+v"(b_off[i]));
                __builtin_amdgcn_global_load_lds((glb_ptr_t)(b_tile + b_off[i]), (lds_ptr_t)(sb + i * NT * 16), 16, 0, 0);
            }
            const bool more = left > TK;
            a_tile += more ? TK * 4 : 0;
            b_tile += more ? b_step * 4 : 0;
            return;
        }
#pragma unroll
        for (int i = 0; i < LA; i++) {
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(ka[i] < left ? ga[i] : zeros), (lds_ptr_t)(sa + i * NT * 16), 16, 0, 0);
            ga[i] += TK;
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(kb[i] < left ? gb[i] : zeros), (lds_ptr_t)(sb + i * NT * 16), 16, 0, 0);
            gb[i] += b_step;
        }
    };

    f32x4_t acc[TI][NJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.f;

    static_assert(STAGES >= 2 && (STAGES - 1) * (LA + LB) < 64, "the loads in flight must fit the 6-bit counter");
    f32x4_t a[2][TI];
    float b[2][4][NJ];
    // The operands of one half (16 k values) of a tile. They are fetched while the matrix unit works on the half before, across the
    // barrier between tiles too: fetched when they are needed, their latency cost a quarter of the time of a lone workgroup.
    auto fetch = [&](int stage, int h) {
        const char* sa = smem + stage * STAGE_BYTES + (wm * (TM / WM) + lr) * 128;
        const float* sb = reinterpret_cast<const float*>(smem + stage * STAGE_BYTES + A_BYTES);
        const int col = (wn * (TN / WN) + NJ * lr) ^ ((((4 * h + lg) & WXM) * WX * 4) & (TN - 1));
#pragma unroll
        for (int i = 0; i < TI; i++) a[h][i] = *reinterpret_cast<const f32x4_t*>(sa + i * 16 * 128 + (((4 * h + lg) ^ (lr & 6)) * 16));
#pragma unroll
        for (int s = 0; s < 4; s++) load_as<typename Cols<NJ>::lds>(sb + (16 * h + 4 * lg + s) * TN + col, b[h][s]);
    };
    auto multiply = [&](int h) {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][i][s], b[h][s][j], acc[i][j], 0, 0, 0);
    };
    // Schedule of a half: an LDS read behind each of the first matrix instructions, then one direct load behind every second. Issued in
    // one go the four wavefronts queue up for the LDS and the address unit while the matrix units stand still (4096 x 6144 x 1536: 618 -> 559 us).
    auto spread = [&](auto loads_tag) {
        constexpr int NM = TI * NJ * 4, R = TI + 4, LOADS = decltype(loads_tag)::value ? LA + LB : 0;
        constexpr int PER_READ = NM / 2 >= R * 2 ? 2 : 1;                    // matrix instructions in front of a read
        constexpr int USED = R * PER_READ < NM ? R * PER_READ : NM;
        constexpr int PER_LOAD = (NM - USED) / (LA + LB) > 0 ? (NM - USED) / (LA + LB) : 1;
#pragma unroll
        for (int x = 0; x < R; x++) {
            __builtin_amdgcn_sched_group_barrier(0x008, PER_READ, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
#pragma unroll
        for (int x = 0; x < LOADS; x++) {
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, PER_LOAD, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < STAGES; s++) issue_tile(s, s);
    wait_vmcnt<(STAGES - 1) * (LA + LB)>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(0, 0);
    for (int kt = 0, stage = 0; kt < nkt; kt++) {
        fetch(stage, 1);
        multiply(0);
        spread(std::false_type{});
        // this thread's loads of tile kt+1 have landed and its LDS reads of tile kt are done; behind the barrier that holds for everyone
        constexpr int INFLIGHT = (STAGES - 2) * (LA + LB);
        __builtin_amdgcn_s_waitcnt((INFLIGHT & 15) | (7 << 4) | ((INFLIGHT >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int freed = stage;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        fetch(stage, 0);
        issue_tile(kt + STAGES, freed);
        multiply(1);
        spread(std::true_type{});
    }
    wait_vmcnt<0>();  // no direct load may still be on its way into this workgroup's LDS when it ends
    store_tile<TI, NJ, EPI, false>(pr, acc, m_blk + wm * (TM / WM) + 4 * lg, n_blk + wn * (TN / WN) + NJ * lr);
}

template <int TM, int TN, int WM, int WN, int STAGES, int EPI, bool WHOLE_K>
int launch_tile_k(TileProbSet& set, int n, hipStream_t st) {
    auto kern = gemm_f32_tile_kernel<TM, TN, WM, WN, STAGES, EPI, WHOLE_K>;
    constexpr int smem = STAGES * (TM * 128 + TK * TN * 4);
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(kern), smem));
    int total = 0;
    for (int i = 0; i < MAX_PROBS; i++) {
        if (i < n) total += ((set.p[i].M + TM - 1) / TM) * ((set.p[i].N + TN - 1) / TN);
        set.end[i] = total;
    }
    hipLaunchKernelGGL(kern, dim3(total), dim3(WM * WN * 64), smem, st, set);
    return launch_status("gemm_f32");
}

// whether the launch takes the kernel of whole K tiles (whose offsets within a tile are 32 bits)
bool whole_k_tiles(const TileProbSet& set, int n) {
    for (int i = 0; i < n; i++)
        if (set.p[i].K % TK || set.p[i].lda > (1 << 22) || set.p[i].ldw > (1 << 22)) return false;
    return true;
}
template <int TM, int TN, int WM, int WN, int STAGES, int EPI>
int launch_tile(TileProbSet& set, int n, hipStream_t st) {
    return whole_k_tiles(set, n) ? launch_tile_k<TM, TN, WM, WN, STAGES, EPI, true>(set, n, st) : launch_tile_k<TM, TN, WM, WN, STAGES, EPI, false>(set, n, st);
}

template <int EPI>
int launch_shape(int shape, TileProbSet& set, int n, hipStream_t st) {
    switch (shape) {
        // (rings no deeper than that two or three workgroups fit a compute unit: they hide each other's waits better than a deeper ring)
        case 0: return launch_tile<128, 128, 2, 2, 2, EPI>(set, n, st);
        case 1: return launch_tile<128, 64, 4, 1, 3, EPI>(set, n, st);
        // (64 columns per wavefront: W in 16-byte LDS reads; as 2x2 wavefronts of 32x32 2202 x 4608 x 1536 took 260 us instead of 255)
        case 2: return launch_tile<64, 64, 4, 1, 3, EPI>(set, n, st);
        case 3: return launch_tile<32, 64, 2, 2, 4, EPI>(set, n, st);
        default: return launch_tile<32, 32, 2, 2, 5, EPI>(set, n, st);
    }
}

// ---- the pieces kernel ----
// The bf16 matrix instruction does sixteen times the operations of the fp32 one per cycle. An fp32 value is the sum of three bf16 values, h + m + l, without a
// remainder (bf16_pieces), and a product of two values that of nine products of pieces, which are exact. Six of them are formed: what m*l, l*m and l*l would add is at
// most 2^-24 + 2^-34 of the product, half a unit in its last place. No value is lost beside a larger one of its row, column or product. (Two f16 pieces per value and
// three products took 0.65 of this time, 1178 x 6144 x 1536 69 us, but hold 22 of the 24 bits, and only of values within 2^-7 of the largest that the scale is
// made for: rows of one channel 2^20 times the others, which W leaves out, came out with an error of 9e-4.)
// The products of a K tile (32 k values) are summed by themselves, and that sum is then added to the fp32 sum of the tiles before: one rounding per K tile that counts,
// where the fp32 instruction has eight. Relative error against 64 bits, normal operands, with this kernel (with the tile kernel): K = 512 9.0e-8 (4.1e-7), 1536
// 1.4e-7 (7.0e-7), 6144 2.7e-7 (1.41e-6); one in 16 values of A not zero 1536 1.4e-7 (1.8e-7); all values 1 + 2^-11 1.6e-7 (1.6e-7). All six products added to one sum:
// 0.85 of the tile kernel's error for normal operands but 1.9 times it for one in 16, 8192 x 3072 x 768 177 us instead of 189; the five small products in a second
// sum: 0.34 of it, but 256x128 tiles have no registers for that, 219 us.
// Sums that are not finite (infinities, NaNs, values from 2^112 and sums from 2^96 on) are formed anew by the fp32 instruction, 16 rows at a time from memory: 1178 x 1536 x
// 1536 43 us, 104 with one such row, 250 with one in 16 or all (tile kernel 50 to 55).
//
// Six products per K tile of 32 are 96 matrix instructions of 17 cycles for a wavefront of 64x64. Splitting the operands takes 12 vector operations per pair of values:
// wavefronts of their own do it. They fetch both operands from memory, K tiles ahead, and write the pieces to LDS, while the others read fragments and
// multiply. One barrier per GROUP K tiles, two buffers. (x - h as one v_dot2c_f32_bf16 instead of two operations: it takes turns with the matrix instructions,
// 168 -> 188 us for 8192 x 3072 x 768 with one sum and no scale.) Matrix instructions of 16 cycles leave the vector unit little room: 256x128 tiles take 4460 cycles per K tile, the matrix
// instructions 3260; 128x128 2290 (1630), 128x64 1290 (820), 64x64 740 (410), 32x64 545 (205), 32x32 370 (100; the tile kernel's 440).
// us, tile kernel -> this one, rows x columns x depth: 8192 x 3072 x 768 312 -> 189 (205 TFLOP/s), 10656 x 768 x 1536 181 -> 121, 1178 x 6144 x 1536 182 -> 116,
// 1178 x 4608 x 1536 139 -> 107, 1178 x 1536 x 6144 187 -> 142, 1178 x 1536 x 1536 52 -> 40, 333 x 1536 x 1536 24.6 -> 22.2, 64 x 1536 x 6144 39 -> 41, 64 x 1536 x 1536 11.9 -> 12.6.
//
// An LDS row is the 32 k values of one plane of pieces (64 bytes); its four chunks of 8 lie where neither the reads (16 lanes at a time: rows 0-3 and 12-15 with
// 4-11 of the next chunk) nor the writes (8 consecutive lanes) meet in a bank (piece_slot). Chunk c holds k = 4c .. 4c + 3 and 16 + 4c .. 16 + 4c + 3, so that the four lanes of a row
// of A read 64 contiguous bytes at a time (3 % at 256x128). Columns of W are assigned to lanes as in the tile kernel.

// A wavefront that fetches operands and writes their pieces: per thread and K tile CA runs of H k values of rows of A and CW ones of columns of W, by PT threads
template <int TM, int TN, int NJ, int CA, int CW, int H, int PT, int SETS, int GROUP, int W_AT = TM * 192, int STAGE_BYTES = (TM + TN) * 192>
__device__ __forceinline__ void produce_pieces(const TileProb& pr, int m_blk, int n_blk, int nkt, unsigned tid, char* smem) {
    constexpr int A_PLANE = TM * 64, B_PLANE = TN * 64, WMULT = NJ == 2 ? 2 : 1, RUNS = TK / H;
    static_assert((H == 8 || H == 4) && (CA == 0 || CA * PT == TM * RUNS) && (CW == 0 || CW * PT == TN * RUNS) && CW <= 2, "shares of a K tile");
    unsigned a_off[CA + 1], w_off[H], a_dst[CA + 1], w_dst[CW + 1];
#pragma unroll
    for (int i = 0; i < CA; i++) {
        const unsigned q = i * PT + tid, row = q / RUNS, k = q % RUNS * 4;
        a_off[i] = (min(row, (unsigned)(pr.M - 1 - m_blk)) * pr.lda + k) * 4;  // rows beyond M re-read the last one and are never stored
        a_dst[i] = piece_slot<0>(row, k / 4 % 4) + k / 16 * 8;
    }
    if constexpr (CW > 0) {
        const unsigned c = tid % (TN / CW) * CW, k0 = tid / (TN / CW) * 4;
#pragma unroll
        for (int k = 0; k < H; k++) w_off[k] = ((k0 + k % 4 + k / 4 * 16) * pr.ldw + min(n_blk + c, (unsigned)(pr.N - CW))) * 4;
#pragma unroll
        for (int x = 0; x < CW; x++) {
            const unsigned cc = c + x, in = cc % (16 * NJ);
            w_dst[x] = W_AT + piece_slot<WMULT>(cc / (16 * NJ) * (16 * NJ) + in % NJ * 16 + in / NJ, k0 / 4 % 4) + k0 / 16 * 8;
        }
    }
    const char* a_tile = reinterpret_cast<const char*>(pr.A + (long long)m_blk * pr.lda);
    const char* w_tile = reinterpret_cast<const char*>(pr.W + pr.n0);
    const long long w_step = (long long)pr.ldw * 4 * TK;
    f32x4_t ra[SETS][CA + 1][H / 4];  // K tiles on their way from memory
    float rw[SETS][H][CW + 1];
    auto load_a = [&](int set, int i) {
        asm volatile("" : "+v"(a_off[i]));
#pragma unroll
        for (int x = 0; x < H / 4; x++) ra[set][i][x] = *reinterpret_cast<const f32x4_t*>(a_tile + a_off[i] + 64 * x);
    };
    auto load_w = [&](int set) {
        if constexpr (CW > 0) {
#pragma unroll
            for (int k = 0; k < H; k++) {
                asm volatile("" : "+v"(w_off[k]));
                float t[CW];
                load_as<typename Cols<CW>::lds>(reinterpret_cast<const float*>(w_tile + w_off[k]), t);
#pragma unroll
                for (int c = 0; c < CW; c++) rw[set][k][c] = t[c];
            }
        }
    };
    auto advance = [&](int kt) {  // the addresses, to K tile kt (past the last one: that one again)
        const bool more = kt < nkt;
        if (CA) a_tile += more ? TK * 4 : 0;
        if (CW) w_tile += more ? w_step : 0;
    };
    // the pieces of set `set` into `stage`, and the requests of the K tile SETS behind it, which is where the addresses are
    auto stage_tile = [&](int set, char* stage) {
        float x[H];
        auto put = [&](char* at, int plane) {
            uint32_t piece[3][H / 2];
            bf16_pieces<H>(x, piece[0], piece[1], piece[2]);
#pragma unroll
            for (int p = 0; p < 3; p++) __builtin_memcpy(__builtin_assume_aligned(at + p * plane, H * 2), piece[p], H * 2);
        };
#pragma unroll
        for (int i = 0; i < CA; i++) {
#pragma unroll
            for (int k = 0; k < H; k++) x[k] = ra[set][i][k >> 2][k & 3];
            put(stage + a_dst[i], A_PLANE);
            load_a(set, i);
            if (CA + CW > 4) __builtin_amdgcn_sched_barrier(0);  // (or the runs share too many registers)
        }
#pragma unroll
        for (int c = 0; c < CW; c++) {
#pragma unroll
            for (int k = 0; k < H; k++) x[k] = rw[set][k][c];
            put(stage + w_dst[c], B_PLANE);
            if (CA + CW > 4) __builtin_amdgcn_sched_barrier(0);
        }
        load_w(set);
        __builtin_amdgcn_sched_barrier(0);  // (or the products of all sets' values with their scale come first, and wait for all loads in flight)
    };
#pragma unroll
    for (int t = 0; t < SETS; t++) {
#pragma unroll
        for (int i = 0; i < CA; i++) load_a(t, i);
        load_w(t);
        advance(t + 1);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < GROUP; t++) {
        stage_tile(t, smem + t * STAGE_BYTES);
        advance(t + 1 + SETS);
    }
    barrier_behind_lds<0>();
    for (int kt = 0; kt < nkt; kt += SETS) {  // (whole groups of SETS: an end in between would make every round wait for all loads in flight)
#pragma unroll
        for (int t = 0; t < SETS; t++) {
            stage_tile((t + GROUP) % SETS, smem + (t + GROUP) % (2 * GROUP) * STAGE_BYTES);
            advance(kt + t + GROUP + 1 + SETS);
            if (t % GROUP == GROUP - 1) barrier_behind_lds<0>();
        }
    }
    wait_vmcnt<0>();
}

// Where what produces A has written its pieces (TileProb::A) they go from memory to LDS by direct loads, requested by PA wavefronts: a ring of RING K tiles (whole pairs of groups),
// RING - GROUP of them ahead.
template <int TM, int PA, int GROUP, int RING>
__device__ __forceinline__ void request_a_pieces(const TileProb& pr, int m_blk, int nkt, unsigned tid, char* smem) {
    constexpr int A_STAGE = TM * 192, REQUESTS = A_STAGE / 1024, LA = (REQUESTS + PA - 1) / PA;  // direct loads of a K tile: all wavefronts' and one's
    static_assert(RING % (2 * GROUP) == 0 && (RING / GROUP - 1) * GROUP * LA < 64, "whole rounds, and the requests in flight must fit the 6-bit counter");
    const unsigned lane = tid & 63, block_row = (unsigned)pr.K * 32;
    const long long plane_bytes = (pr.M + 15) / 16 * (long long)block_row;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned off[LA], dst[LA];
    long long plane_at[LA];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        // request q: a plane of a block. (Where the requests do not divide evenly, several wavefronts make the last one.)
        const unsigned q = min(i * PA + wave, (unsigned)REQUESTS - 1), block = q / 3, plane = q % 3;
        off[i] = min(block, (unsigned)(pr.M - 1 - m_blk) / 16) * block_row + lane * 16;  // blocks beyond M re-read the last one and are never stored
        plane_at[i] = plane * plane_bytes;
        dst[i] = plane * (TM * 64) + block * 1024;
    }
    const char* tile = reinterpret_cast<const char*>(pr.A) + (m_blk / 16) * (long long)block_row;
    int next = 0;
    unsigned slot = 0;
    auto request = [&]() {  // the next K tile; past the end the last one once more, into a stage that nobody reads again
#pragma unroll
        for (int i = 0; i < LA; i++) {
            asm volatile("" : "+v"(off[i]));
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(tile + plane_at[i] + off[i]), (lds_ptr_t)(smem + dst[i] + slot), 16, 0, 0);
        }
        next++;
        tile += next < nkt ? 1024 : 0;
        slot = slot == (RING - 1) * A_STAGE ? 0 : slot + A_STAGE;
    };
    auto publish = []() {  // all but the groups that are requested ahead of the one to publish
        wait_vmcnt<(RING / GROUP - 2) * GROUP * LA>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int t = 0; t < RING - GROUP; t++) request();
    publish();
    for (int kt = 0; kt < nkt; kt += GROUP) {
#pragma unroll
        for (int t = 0; t < GROUP; t++) request();  // into the stages that the last barrier has freed
        publish();
    }
    wait_vmcnt<0>();  // no direct load may still be on its way into this workgroup's LDS when it ends
}

// LDS writes as assembly: behind direct loads into LDS the compiler has every write that it knows of wait for all of them (publish() waits for these)
__device__ __forceinline__ void write_lds(char* at, const uint32_t (&v)[4]) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    asm volatile("ds_write_b128 %0, %1" ::"v"((uint32_t)(uintptr_t)(lds_ptr_t)at), "v"(u32x4_t{v[0], v[1], v[2], v[3]}) : "memory");
}
__device__ __forceinline__ void write_lds(char* at, const uint32_t (&v)[2]) {
    asm volatile("ds_write_b64 %0, %1" ::"v"((uint32_t)(uintptr_t)(lds_ptr_t)at), "v"((unsigned long long)v[1] << 32 | v[0]) : "memory");
}
// Both by the same PT threads: the requests of A's pieces, and W's split.
template <int TM, int TN, int NJ, int CW, int H, int PT, int SETS, int GROUP, int RING>
__device__ __forceinline__ void produce_with_a_pieces(const TileProb& pr, int m_blk, int n_blk, int nkt, unsigned tid, char* smem) {
    constexpr int A_PLANE = TM * 64, B_PLANE = TN * 64, W_STAGE = 3 * B_PLANE, A_STAGE = 3 * A_PLANE, WMULT = NJ == 2 ? 2 : 1, RUNS = TK / H, PW = PT / 64;
    constexpr int REQUESTS = A_STAGE / 1024, LA = (REQUESTS + PW - 1) / PW;  // direct loads of a K tile: all wavefronts' and one's
    static_assert((H == 8 || H == 4) && CW * PT == TN * RUNS && CW <= 2 && SETS % GROUP == 0 && RING % (2 * GROUP) == 0, "shares of a K tile");
    const unsigned lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned block_row = (unsigned)pr.K * 32;
    const long long plane_bytes = (pr.M + 15) / 16 * (long long)block_row;
    unsigned a_off[LA], a_dst[LA], w_off[H], w_dst[CW];
    long long plane_at[LA];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const unsigned q = min(i * PW + wave, REQUESTS - 1), block = q / 3, plane = q % 3;
        a_off[i] = min(block, (unsigned)(pr.M - 1 - m_blk) / 16) * block_row + lane * 16;
        plane_at[i] = plane * plane_bytes;
        a_dst[i] = 2 * GROUP * W_STAGE + plane * A_PLANE + block * 1024;
    }
    const unsigned c = tid % (TN / CW) * CW, k0 = tid / (TN / CW) * 4;
#pragma unroll
    for (int k = 0; k < H; k++) w_off[k] = ((k0 + k % 4 + k / 4 * 16) * pr.ldw + min(n_blk + c, (unsigned)(pr.N - CW))) * 4;
#pragma unroll
    for (int x = 0; x < CW; x++) {
        const unsigned cc = c + x, in = cc % (16 * NJ);
        w_dst[x] = piece_slot<WMULT>(cc / (16 * NJ) * (16 * NJ) + in % NJ * 16 + in / NJ, k0 / 4 % 4) + k0 / 16 * 8;
    }
    const char* a_tile = reinterpret_cast<const char*>(pr.A) + (m_blk / 16) * (long long)block_row;
    const char* w_tile = reinterpret_cast<const char*>(pr.W + pr.n0);
    const long long w_step = (long long)pr.ldw * 4 * TK;
    float rw[SETS][H][CW];
    int w_next = 0, a_next = 0;  // the K tiles that the addresses are at
    unsigned a_slot = 0;         // and where in the ring
    // requests of the next K tile; past the end the last one once more, into a stage that nobody reads again
    auto request_a = [&]() {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            asm volatile("" : "+v"(a_off[i]));
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a_tile + plane_at[i] + a_off[i]), (lds_ptr_t)(smem + a_dst[i] + a_slot), 16, 0, 0);
        }
        a_next++;
        a_tile += a_next < nkt ? 1024 : 0;
        a_slot = a_slot == (RING - 1) * A_STAGE ? 0 : a_slot + A_STAGE;
    };
    auto request_w = [&](int set) {
#pragma unroll
        for (int k = 0; k < H; k++) {
            asm volatile("" : "+v"(w_off[k]));
            float t[CW];
            load_as<typename Cols<CW>::lds>(reinterpret_cast<const float*>(w_tile + w_off[k]), t);
#pragma unroll
            for (int x = 0; x < CW; x++) rw[set][k][x] = t[x];
        }
        w_next++;
        w_tile += w_next < nkt ? w_step : 0;
    };
    auto stage_w = [&](int set, char* stage) {
#pragma unroll
        for (int x = 0; x < CW; x++) {
            float v[H];
#pragma unroll
            for (int k = 0; k < H; k++) v[k] = rw[set][k][x];
            uint32_t piece[3][H / 2];
            bf16_pieces<H>(v, piece[0], piece[1], piece[2]);
#pragma unroll
            for (int p = 0; p < 3; p++) write_lds(stage + w_dst[x] + p * B_PLANE, piece[p]);
        }
        request_w(set);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Everything but the newest NEWER requests of this wavefront has landed, its LDS writes are done; behind the barrier that holds for the others too
    auto publish = [](auto newer) {
        constexpr int NEWER = decltype(newer)::value < 63 ? decltype(newer)::value : 63;
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt((NEWER & 15) | (7 << 4) | ((NEWER >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto fence = []() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int AHEAD = RING / GROUP - 2;  // groups of K tiles between the one that a round requests and the one it publishes
#pragma unroll
    for (int t = 0; t < RING - GROUP; t++) request_a();
    fence();
#pragma unroll
    for (int t = 0; t < SETS; t++) {
        request_w(t);
        fence();
    }
#pragma unroll
    for (int t = 0; t < GROUP; t++) stage_w(t, smem + t * W_STAGE);
    publish(std::integral_constant<int, AHEAD * GROUP * LA + (SETS + GROUP) * H>());
    for (int kt = 0; kt < nkt; kt += SETS) {
#pragma unroll
        for (int t = 0; t < SETS; t++) {
            if (t % GROUP == 0) {
#pragma unroll
                for (int i = 0; i < GROUP; i++) request_a();  // into the stages that the last barrier has freed
                fence();
            }
            stage_w((t + GROUP) % SETS, smem + (t + GROUP) % (2 * GROUP) * W_STAGE);
            // (newer than the A tiles to publish: the W tiles of the round that requested them and all that the rounds behind it requested; in the first rounds more)
            if (t % GROUP == GROUP - 1) publish(std::integral_constant<int, GROUP * H + AHEAD * GROUP * (LA + H)>());
        }
    }
    wait_vmcnt<0>();  // no direct load may still be on its way into this workgroup's LDS when it ends
}

// WM x WN wavefronts multiply; PA fetch and split A and PB W (PB = 0: PA both). GROUP: K tiles per barrier. SETS: K tiles on their way from memory. WAVES: wavefronts
// per SIMD that the registers are to allow. RING: A comes in pieces, in a ring of so many K tiles, which PA request; 0: it does not. The depth
// is made of whole groups of four K tiles.
template <int TM, int TN, int WM, int WN, int PA, int PB, int HA, int HB, int GROUP, int SETS, int WAVES, int RING, int EPI>
__global__ void __launch_bounds__((WM * WN + PA + PB) * 64, WAVES) gemm_f32_pieces_kernel(const TileProbSet set) {
    constexpr int TI = TM / WM / 16, NJ = TN / WN / 16, CONSUMERS = WM * WN;
    // A stage holds A and W; with RING the W stages come first and A's ring behind them
    constexpr int A_PLANE = TM * 64, B_PLANE = TN * 64, W_STAGE = 3 * (RING ? B_PLANE : A_PLANE + B_PLANE), A_STAGE = RING ? 3 * A_PLANE : W_STAGE;
    constexpr int A_AT = RING ? 2 * GROUP * W_STAGE : 0, W_AT = RING ? 0 : 3 * A_PLANE;
    static_assert(TI >= 1 && (NJ == 1 || NJ == 2 || NJ == 4), "tile shape");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int w = blockIdx.x;
    const int which = (w >= set.end[0]) + (w >= set.end[1]);
    const TileProb& pr = set.p[which];
    const int M = pr.M, N = pr.N;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tile_m, tile_n;
    tile_of_workgroup(w - (which ? set.end[which - 1] : 0), (M + TM - 1) / TM, (N + TN - 1) / TN, tile_m, tile_n);
    const int m_blk = tile_m * TM, n_blk = tile_n * TN;
    const int nkt = pr.K / TK;
    if (wave >= CONSUMERS) {
        const unsigned tid = threadIdx.x - CONSUMERS * 64;
        constexpr int CA = RING ? 0 : TM * (TK / HA) / (PA * 64), CB = TN * (TK / HB) / ((PB ? PB : PA) * 64);
        if constexpr (RING > 0) {
            if constexpr (PA == 0) produce_with_a_pieces<TM, TN, NJ, CB, HB, PB * 64, SETS, GROUP, RING>(pr, m_blk, n_blk, nkt, tid, smem);
            else if (wave < CONSUMERS + PA) request_a_pieces<TM, PA, GROUP, RING>(pr, m_blk, nkt, tid, smem + A_AT);
            else produce_pieces<TM, TN, NJ, 0, CB, HB, PB * 64, SETS, GROUP, W_AT, W_STAGE>(pr, m_blk, n_blk, nkt, tid - PA * 64, smem);
        } else if constexpr (PB == 0) {
            produce_pieces<TM, TN, NJ, CA, CB, HA, PA * 64, SETS, GROUP>(pr, m_blk, n_blk, nkt, tid, smem);
        } else {
            if (wave < CONSUMERS + PA) produce_pieces<TM, TN, NJ, CA, 0, HA, PA * 64, SETS, GROUP>(pr, m_blk, n_blk, nkt, tid, smem);
            else produce_pieces<TM, TN, NJ, 0, CB, HB, PB * 64, SETS, GROUP>(pr, m_blk, n_blk, nkt, tid - PA * 64, smem);
        }
        return;
    }

    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4, wm = wave / WN, wn = wave % WN;
    f32x4_t acc[TI][NJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    constexpr int WMULT = NJ == 2 ? 2 : 1;
    const unsigned a_src = A_AT + piece_slot<0>(wm * (TM / WM) + lr, lg), b_src = W_AT + piece_slot<WMULT>(wn * (TN / WN) + lr, lg);
    auto read_a = [&](bf16x8_t (&f)[TI], const char* stage, int plane) {
#pragma unroll
        for (int i = 0; i < TI; i++) f[i] = *reinterpret_cast<const bf16x8_t*>(stage + plane * A_PLANE + a_src + i * 1024);
    };
    auto read_b = [&](const char* stage, int plane, int j) {
        const unsigned key = ((((wn * (TN / WN) >> 4) + j) ^ ((wn * (TN / WN)) >> 4)) * WMULT & 3) * 16;  // (columns 16 apart have other chunks: piece_slot())
        return *reinterpret_cast<const bf16x8_t*>(stage + plane * B_PLANE + (b_src ^ key) + j * 1024);
    };
    auto multiply = [&](const bf16x8_t (&x)[TI], const bf16x8_t& y, f32x4_t (&to)[TI]) {
#pragma unroll
        for (int i = 0; i < TI; i++) to[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i], y, to[i], 0, 0, 0);
    };
    // an LDS read behind each of the first matrix instructions: issued in one go the matrix unit stands still meanwhile; ADDS vector operations behind each
    auto spread = [](auto reads, auto products, auto adds) {
        constexpr int R = decltype(reads)::value, NM = decltype(products)::value, ADDS = decltype(adds)::value;
#pragma unroll
        for (int x = 0; x < NM; x++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (x < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (ADDS) __builtin_amdgcn_sched_group_barrier(0x002, ADDS, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    typedef std::integral_constant<int, 0> None;
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 4> Four;
    typedef std::integral_constant<int, TI> Rows;
    // Column block by column block: its products over the 32 k values of the tile in the order l*h, m*h, m*m, h*m, h*l, h*h, whatever the tile shape (a row's result depends on
    // neither the shape nor the grouping), in sums of their own (u), which are added to acc beside the first products of the block after. A register is
    // loaded for the next block or K tile behind its last use; behind the barrier nothing of the current stage is read any more.
    bf16x8_t ah[TI], am[TI], al[TI], bh[2], bm, bl;
    f32x4_t u[2][TI];
    barrier_behind_lds<0>();
    bh[0] = read_b(smem, 0, 0);
    read_a(al, smem, 2);
    read_a(am, smem, 1);
    bm = read_b(smem, 1, 0);
    read_a(ah, smem, 0);
    bl = read_b(smem, 2, 0);
#pragma unroll
    for (int i = 0; i < TI; i++) u[1][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    unsigned ring = 0;  // where in A's ring this round's K tiles begin
    for (int kt = 0; kt < nkt; kt += 2 * GROUP) {
        const unsigned ring_next = RING > 2 * GROUP ? (ring + 2 * GROUP * A_STAGE) % (RING * A_STAGE) : 0;
#pragma unroll
        for (int t = 0; t < 2 * GROUP; t++) {
            const char *cur = smem + t * W_STAGE, *next = smem + (t + 1) % (2 * GROUP) * W_STAGE;
            const char* const next_a = smem + (t + 1 < 2 * GROUP ? ring + (t + 1) * A_STAGE : ring_next);
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int p = (t * NJ + j) & 1;
                const bool last = j == NJ - 1;
                const char* const stage = last ? next : cur;
                const int column = last ? 0 : j + 1;
                if (last && t % GROUP == GROUP - 1) barrier_behind_lds<0>();
                bh[p ^ 1] = read_b(stage, 0, column);
#pragma unroll
                for (int i = 0; i < TI; i++) u[p][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                multiply(al, bh[p], u[p]);
#pragma unroll
                for (int i = 0; i < TI; i++) acc[i][(j + NJ - 1) % NJ] += u[p ^ 1][i];
                spread(One{}, Rows{}, Four{});
                if (last) read_a(al, next_a, 2);
                multiply(am, bh[p], u[p]);
                multiply(am, bm, u[p]);
                if (last) spread(Rows{}, std::integral_constant<int, 2 * TI>{}, None{});
                else spread(None{}, std::integral_constant<int, 2 * TI>{}, None{});
                if (last) read_a(am, next_a, 1);
                multiply(ah, bm, u[p]);
                if (last) spread(Rows{}, Rows{}, None{});
                else spread(None{}, Rows{}, None{});
                bm = read_b(stage, 1, column);
                multiply(ah, bl, u[p]);
                spread(One{}, Rows{}, None{});
                bl = read_b(stage, 2, column);
                multiply(ah, bh[p], u[p]);
                spread(One{}, Rows{}, None{});
                if (last) read_a(ah, next_a, 0);
            }
        }
        ring = ring_next;
    }
#pragma unroll
    for (int i = 0; i < TI; i++) acc[i][NJ - 1] += u[1][i];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] *= 1.0f / (PIECES_SCALE * PIECES_SCALE);
    // A sum that is not finite (values or sums too large for the pieces, infinities, NaNs) is formed anew from the operands themselves
    const int m0 = m_blk + wm * (TM / WM), n0 = n_blk + wn * (TN / WN);
    auto infinite = [&](const f32x4_t& v, int i) {  // (rows beyond M may be anything)
        bool bad = false;
#pragma unroll
        for (int r = 0; r < 4; r++) bad |= (!RING || m0 + i * 16 + 4 * lg + r < M) && (__float_as_uint(v[r]) & 0x7f800000u) == 0x7f800000u;
        return bad;
    };
    bool bad = false;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) bad |= infinite(acc[i][j], i);
    if (__builtin_amdgcn_ballot_w64(bad)) {
#pragma unroll
        for (int i = 0; i < TI; i++) {
            bad = false;
#pragma unroll
            for (int j = 0; j < NJ; j++) bad |= infinite(acc[i][j], i);
            if (!__builtin_amdgcn_ballot_w64(bad)) continue;
            const int row = min(m0 + i * 16 + lr, M - 1);
            const float* pa = pr.A + (long long)row * pr.lda + lg;
            const float* pw = pr.W + (long long)lg * pr.ldw + pr.n0 + min(n0 + NJ * lr, N - NJ);
            f32x4_t sum[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) sum[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k < pr.K; k += 16, pa += 16, pw += 16 * (long long)pr.ldw)
#pragma unroll
                for (int step = 0; step < 16; step += 4) {
                    float w[NJ];
                    load_cols<NJ>(pw + step * (long long)pr.ldw, w);
#pragma unroll
                    for (int j = 0; j < NJ; j++) sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(RING ? of_pieces(PieceMatrix(const_cast<float*>(pr.A), M, pr.K), row, k + step + lg) : pa[step], w[j], sum[j], 0, 0, 0);
                }
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (!finite(acc[i][j][r])) acc[i][j][r] = sum[j][r];
        }
    }
    store_tile<TI, NJ, EPI, (RING > 0), RING == 0 && TI * NJ >= 16>(pr, acc, m0 + 4 * lg, n0 + NJ * lr);
}

template <int TM, int TN, int WM, int WN, int PA, int PB, int HA, int HB, int GROUP, int SETS, int WAVES, int RING, int EPI>
int launch_pieces(TileProbSet& set, int n, hipStream_t st) {
    auto kern = gemm_f32_pieces_kernel<TM, TN, WM, WN, PA, PB, HA, HB, GROUP, SETS, WAVES, RING, EPI>;
    constexpr int smem = (RING ? RING * TM + 2 * GROUP * TN : 2 * GROUP * (TM + TN)) * 3 * 64;
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(kern), smem));
    int total = 0;
    for (int i = 0; i < MAX_PROBS; i++) {
        if (i < n) total += ((set.p[i].M + TM - 1) / TM) * ((set.p[i].N + TN - 1) / TN);
        set.end[i] = total;
    }
    hipLaunchKernelGGL(kern, dim3(total), dim3((WM * WN + PA + PB) * 64), smem, st, set);
    return launch_status("gemm_f32");
}
template <int EPI>
int launch_pieces_shape(int shape, TileProbSet& set, int n, hipStream_t st) {
    switch (shape) {
        case 0: return launch_pieces<128, 128, 2, 4, 4, 4, 8, 8, 1, 2, 4, 0, EPI>(set, n, st);
        case 1: return launch_pieces<128, 64, 4, 2, 4, 4, 8, 4, 2, 4, 4, 0, EPI>(set, n, st);
        // (columns of W by runs of four: a thread's eight loads, one per k value, were what it spent most time on. 128x64 at 512 rows, K = 1536 31 -> 29 us,
        // 64x64 22.3 -> 20.7, 32x64 17.7 -> 15.4)
        case 2: return launch_pieces<64, 64, 2, 2, 4, 8, 8, 4, 2, 4, 4, 0, EPI>(set, n, st);
        case 3: return launch_pieces<32, 64, 2, 2, 4, 8, 4, 4, 2, 4, 4, 0, EPI>(set, n, st);
        case 4: return launch_pieces<32, 32, 2, 2, 4, 4, 4, 4, 2, 4, 3, 0, EPI>(set, n, st);
        default: return launch_pieces<256, 128, 4, 2, 4, 0, 8, 8, 1, 2, 3, 0, EPI>(set, n, st);
    }
}

// A in pieces. What the launch of a layer costs then: two thirds (128x64, 256x128) or half of the splitting is gone, A moves half as many bytes more. us, A split here | A in pieces, cold
// weights: 1178 x 4608 x 1536 117 | 90, 1178 x 6144 x 1536 with the GELU and its output in pieces 126 | 110, 1178 x 1536 x 1536 44.5 | 39, 1178 x 1536 x 6144 153 | 144, 3226 x 4608 x
// 1536 240 | 205, 10656 x 768 x 3072 248 | 219, 10656 x 3072 x 768 286 | 246, 18848 x 2304 x 768 369 | 326; below some 600 rows nothing (333 x 1536 x 1536 24.4 | 25.4, 333 x 1536 x 6144
// 77 | 84). With operands of zeros, so without the power limit, 256x128 tiles gain up to a quarter (1178 x 6144 x 1536 103 | 81).
// Wavefronts of their own request A: behind the requests of the same wavefront the split of W started a third of a K tile late (128x128 1178 x 1536 x 1536 65 -> 59 us). 256x128 tiles
// have no registers for a fourth wavefront per SIMD and keep both in one (produce_with_a_pieces). 128x64 as waves of 32x64 instead of 32x32: a quarter of the LDS reads less, 1178 x 1536 x
// 6144 149 -> 139; 64x64 as waves of 16x64, two workgroups to a unit, 57 -> 45.
template <int EPI>
int launch_a_pieces_shape(int shape, TileProbSet& set, int n, hipStream_t st) {
    switch (shape) {
        case 0: return launch_pieces<128, 128, 4, 2, 4, 4, 8, 8, 1, 2, 4, 4, EPI>(set, n, st);
        case 1: return launch_pieces<128, 64, 4, 1, 4, 4, 8, 4, 2, 4, 3, 4, EPI>(set, n, st);
        case 2: return launch_pieces<64, 64, 4, 1, 2, 4, 8, 4, 1, 4, 5, 4, EPI>(set, n, st);
        case 3: return launch_pieces<32, 64, 2, 2, 4, 8, 4, 4, 2, 4, 4, 4, EPI>(set, n, st);
        case 4: return launch_pieces<32, 32, 2, 2, 2, 4, 4, 4, 2, 4, 4, 8, EPI>(set, n, st);
        default: return launch_pieces<256, 128, 4, 2, 0, 4, 8, 8, 1, 2, 3, 2, EPI>(set, n, st);
    }
}

// ... with the norms of q and k: the shapes whose wavefronts have 64 columns. (Of 66 500 sizes from the line on at which A comes in pieces, the table has another one ahead for 16, of 335 to 440
// rows of 2304 to 3072 columns: by it up to 14 % in the projection; blocks there take 0.95 to 1.00 of their time with a launch for the norms.)
int launch_qkv_norm_shape(int shape, TileProbSet& set, int n, hipStream_t st) {
    switch (shape) {
        case 0: return launch_pieces<128, 128, 4, 2, 4, 4, 8, 8, 1, 2, 4, 4, EPI_QKV_NORM>(set, n, st);
        case 1: return launch_pieces<128, 64, 4, 1, 4, 4, 8, 4, 2, 4, 3, 4, EPI_QKV_NORM>(set, n, st);
        case 5: return launch_pieces<256, 128, 4, 2, 0, 4, 8, 8, 1, 2, 3, 2, EPI_QKV_NORM>(set, n, st);
        default: return launch_pieces<64, 64, 4, 1, 2, 4, 8, 4, 1, 4, 5, 4, EPI_QKV_NORM>(set, n, st);
    }
}

struct Layers {
    F32Layer l[MAX_PROBS];
    Layers(const TileProbSet& set, int n) {
        for (int i = 0; i < n; i++) l[i] = F32Layer{set.p[i].M, set.p[i].N, set.p[i].K};
    }
};

// What the tile kernel asks for: operands whose rows are made of aligned 16-byte chunks (its direct loads into LDS) and outputs in whole
// groups of four columns. The output side may lie at any float with any stride (1024 x 4608 x 1536 into an output that is 4 bytes off: 314 us
// with the element-wise kernel, 130 with this one, as much as aligned).
bool whole_chunks(const GemmF32Problem& q) {
    auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    return al(q.A) && al(q.W) && q.lda % 4 == 0 && q.ldw % 4 == 0 && q.n0 % 4 == 0 && q.K % 4 == 0 && q.N % 4 == 0;
}
}  // namespace

// (the widths as in whole_chunks and whole_k_tiles, the depth as in f32_by_pieces)
bool gemm_f32_takes_a_pieces(const float* W, int ldw, int n0, int N, int K) {
    const F32Layer layer{1, N, K};
    return (reinterpret_cast<uintptr_t>(W) & 15) == 0 && ldw % 4 == 0 && ldw <= (1 << 22) && n0 % 4 == 0 && N % 4 == 0 && K <= (1 << 22) && f32_by_pieces(&layer, 1) &&
           !g_gemm_f32_no_pieces;
}

int gemm_f32_grouped(const GemmF32Problem* probs, int n, int epi, hipStream_t st) {
    if (n < 1 || n > MAX_PROBS) return fail(SD3_ERR_INVALID_ARG, "gemm_f32: 1 to %d problems (got %d)", MAX_PROBS, n);
    TileProbSet set{};
    int m = 0;
    const bool a_pieces = probs[0].a_pieces;
    for (int i = 0; i < n; i++) {
        const GemmF32Problem& q = probs[i];
        if (q.M <= 0 || q.N <= 0) continue;
        if (q.K <= 0) return fail(SD3_ERR_INVALID_ARG, "gemm_f32: K must be positive");
        if (q.a_pieces != a_pieces || (a_pieces && !gemm_f32_takes_a_pieces(q.W, q.ldw, q.n0, q.N, q.K)) || (q.out_pieces && (epi != EPI_BIAS_GELU || !a_pieces)))
            return fail(SD3_ERR_INVALID_ARG, "gemm_f32: operands or outputs in pieces that this launch does not take");
        if (epi == EPI_QKV_NORM && (!a_pieces || q.n0 || q.N % 192))
            return fail(SD3_ERR_INVALID_ARG, "gemm_f32: the norms of q and k are for A in pieces and heads of 64");
        EpiDev e{q.ea.bias, q.ea.gate, q.ea.resid, q.ea.table, q.ea.gate_ld, q.ea.rows_per_batch > 0 ? q.ea.rows_per_batch : 1};
        if (epi == EPI_BIAS_ROWADD) e.gate_ld = q.N;
        if (epi == EPI_QKV_NORM) e.gate_ld = q.N / 3;
        if (!whole_chunks(q)) {
            dim3 grid((q.N + BN - 1) / BN, (q.M + BM - 1) / BM), block(256);
#define SD3_GEMM_F32_LAUNCH(E) \
    case E: hipLaunchKernelGGL((gemm_f32_kernel<E>), grid, block, 0, st, q.A, q.lda, q.W, q.ldw, q.n0, q.out, q.ldc, q.M, q.N, q.K, e); break
            switch (epi) {
                SD3_GEMM_F32_LAUNCH(EPI_BIAS);
                SD3_GEMM_F32_LAUNCH(EPI_BIAS_GELU);
                SD3_GEMM_F32_LAUNCH(EPI_BIAS_SILU);
                SD3_GEMM_F32_LAUNCH(EPI_GATE_RESID);
                SD3_GEMM_F32_LAUNCH(EPI_BIAS_ROWADD);
                default: return fail(SD3_ERR_INVALID_ARG, "gemm_f32: unknown epilogue %d", epi);
            }
#undef SD3_GEMM_F32_LAUNCH
            SD3_TRY(launch_status("gemm_f32"));
            continue;
        }
        set.p[m++] = TileProb{q.A, q.W, q.out, q.lda, q.ldw, q.ldc, q.M, q.N, q.K, q.n0, q.out_pieces, e};
    }
    if (m == 0) return SD3_OK;
    const int cus = compute_units();
    if (cus <= 0) return SD3_ERR_HIP;
    const Layers layers(set, m);
    if (a_pieces) {
        const int shape = g_gemm_f32_tile >= 0 ? g_gemm_f32_tile : pick_f32_piece_tile(layers.l, m, cus, f32_a_piece_tiles);
        switch (epi) {
            case EPI_BIAS: return launch_a_pieces_shape<EPI_BIAS>(shape, set, m, st);
            case EPI_BIAS_GELU: return launch_a_pieces_shape<EPI_BIAS_GELU>(shape, set, m, st);
            case EPI_GATE_RESID: return launch_a_pieces_shape<EPI_GATE_RESID>(shape, set, m, st);
            case EPI_QKV_NORM: return launch_qkv_norm_shape(shape, set, m, st);
            default: return fail(SD3_ERR_INVALID_ARG, "gemm_f32: no epilogue %d with A in pieces", epi);
        }
    }
    if (whole_k_tiles(set, m) && f32_by_pieces(layers.l, m) && !g_gemm_f32_no_pieces) {
        const int shape = g_gemm_f32_tile >= 0 ? g_gemm_f32_tile : pick_f32_piece_tile(layers.l, m, cus);
        switch (epi) {
            case EPI_BIAS: return launch_pieces_shape<EPI_BIAS>(shape, set, m, st);
            case EPI_BIAS_GELU: return launch_pieces_shape<EPI_BIAS_GELU>(shape, set, m, st);
            case EPI_BIAS_SILU: return launch_pieces_shape<EPI_BIAS_SILU>(shape, set, m, st);
            case EPI_GATE_RESID: return launch_pieces_shape<EPI_GATE_RESID>(shape, set, m, st);
            case EPI_BIAS_ROWADD: return launch_pieces_shape<EPI_BIAS_ROWADD>(shape, set, m, st);
            default: return fail(SD3_ERR_INVALID_ARG, "gemm_f32: unknown epilogue %d", epi);
        }
    }
    const int shape = g_gemm_f32_tile >= 0 ? g_gemm_f32_tile % F32_TILES : pick_f32_tile(layers.l, m, cus, whole_k_tiles(set, m));
    switch (epi) {
        case EPI_BIAS: return launch_shape<EPI_BIAS>(shape, set, m, st);
        case EPI_BIAS_GELU: return launch_shape<EPI_BIAS_GELU>(shape, set, m, st);
        case EPI_BIAS_SILU: return launch_shape<EPI_BIAS_SILU>(shape, set, m, st);
        case EPI_GATE_RESID: return launch_shape<EPI_GATE_RESID>(shape, set, m, st);
        case EPI_BIAS_ROWADD: return launch_shape<EPI_BIAS_ROWADD>(shape, set, m, st);
        default: return fail(SD3_ERR_INVALID_ARG, "gemm_f32: unknown epilogue %d", epi);
    }
}

int gemm_f32(const float* A, int lda, const float* W, int ldw, int n0, float* out, int ldc, int M, int N, int K, int epi, const GemmEpilogueArgs& ea,
             hipStream_t st) {
    const GemmF32Problem q{A, W, out, lda, ldw, n0, ldc, M, N, K, ea};
    return gemm_f32_grouped(&q, 1, epi, st);
}

int g_gemm_f32_tile = -1;  // -1: chosen from the sizes; 0..5: that entry of f32_tiles or f32_piece_tiles (sd3_tune)
int g_gemm_f32_no_pieces = 0;  // 1: the kernels of the fp32 instruction at every depth (sd3_tune)

}  // namespace sd3
