// bf16 GEMM on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16), fp32 accumulation:
//   out(M,N) = A(M,K) @ Wp^T + epilogue,  A bf16 row-major, Wp bf16 (N,K) row-major or as K tiles (K/64, N, 64) (the reference's (K,N)
//   fp32 weight transposed and rounded once by pack_weight_bf16), so that both operands are K-contiguous.
// It replaces linear / partial_linear of the reference (modules.cpp:475-511) for the QKV, out-projection and MLP
// layers. Epilogues: bias | bias+GELU-tanh | bias+SiLU | gate*(.)+residual (fp32, in place) | bias + row table.
//
// Data path: global -> LDS with direct loads (global_load_lds_dwordx4: no registers, no VALU), a ring of STAGES
// LDS buffers with one workgroup barrier per 64-deep K tile; LDS rows are 128 bytes with the 16-byte chunk index
// XOR-swizzled by a key of the row, which makes both the linear LDS fill and the 16-byte MFMA operand reads conflict-free.
// Two kernels: gemm_bf16_kernel (256x256 tiles by persistent workgroups; also the fp8 form) for launches that fill the device with
// them, gemm_bf16_ring_kernel (64x64 to 256x128 tiles; 192x256 ones are the first kernel's) for the others; tile_shapes says where the line is.
#include "common.hpp"

#include <type_traits>

namespace sd3 {
namespace {

constexpr int BK = 64;  // bf16 elements per K tile = 128 bytes per LDS row

typedef f32x4_t f32x4_any_t __attribute__((aligned(4)));  // four floats at any float
struct EpiDev {
    const float* a_scale;  // fp8 operands: one factor per row of A (null: 1)
    const float* w_scale;  // fp8 operands: one factor per output column (null: 1)
    const float* bias;
    const float* gate;
    const float* resid;
    const float* table;
    int gate_ld;
    int rows_per_batch;
};

// XOR key of an LDS row: rows r..r+7 get 8 different keys (no conflicts on 8-lane / 32-bank groups) and rows r, r+8 get
// keys that differ in bit 0 (no conflicts on 16-lane / 64-bank groups either).
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }
// The key for tiles whose fragments are read in the 16x16x32 layout (lane l: row l % 16, chunk 4 * step + l / 16). A 16-byte LDS
// read is served in four phases of 16 lanes (lanes 0-3, 12-15, 20-23, 24-27; 4-7, 8-11, 16-19, 28-31; the same + 32), so a phase
// holds rows 0-3 and 12-15 with one chunk index and rows 4-11 with the next: even and odd rows lie in different halves of the 64
// banks, and row & 6 gives the four even (odd) rows of either group the keys 0, 2, 4, 6 -- with the chunk indices one apart, all
// eight 16-byte slots of a half. (With swz() that pattern hits every slot twice: the bank-conflict counter read 47 % of the LDS
// cycles; the 32x32 layout, lane l: row l % 32, is conflict-free with swz() and would not be with this key.)
__device__ __forceinline__ int swz16(int row) { return row & 6; }

// RMSNorm of one head of one token (modules.cpp:192-198) held by 16 consecutive lanes, four columns each
__device__ __forceinline__ void qk_norm4(float (&v)[4], const float4 w4) {
    // explicit fused multiply-adds: left to the compiler, each unrolled copy of this code may pick a different product to fuse, and a row's
    // result would depend on where in the tile it sits
    float ss = fmaf(v[3], v[3], fmaf(v[2], v[2], fmaf(v[1], v[1], v[0] * v[0])));
    // butterfly over the 16 lanes with data-parallel-primitive moves (no trip through the LDS crossbar): lanes ^1 and ^2 by quad permutes;
    // after those every quad holds one value, so mirroring the half row (i <-> 7-i) and then the row (i <-> 15-i) pairs the same
    // partial sums as lanes ^4 and ^8 would
    ss += dpp_move<0xB1>(ss);   // quad_perm [1,0,3,2]
    ss += dpp_move<0x4E>(ss);   // quad_perm [2,3,0,1]
    ss += dpp_move<0x141>(ss);  // row_half_mirror
    ss += dpp_move<0x140>(ss);  // row_mirror
    // (the hardware's reciprocal square root, 1 ulp: a divide and a square root here cost 0.2 ms per forward of the 1024x1024 pair, and
    // the result is rounded to bf16 anyway)
    const float inv = __builtin_amdgcn_rsqf(1e-6f + ss * (1.0f / 64.0f));
    v[0] = (v[0] * inv) * w4.x; v[1] = (v[1] * inv) * w4.y; v[2] = (v[2] * inv) * w4.z; v[3] = (v[3] * inv) * w4.w;
}

// LDS bytes of a configuration: the tile ring, or the epilogue staging slabs if those are larger
template <int BM, int BN, int WM, int WN, int STAGES>
constexpr int smem_bytes() {
    constexpr int ring = STAGES * (BM + BN) * 128, epi = WM * WN * 32 * (BN / WN + 4) * 4;
    return ring > epi ? ring : epi;
}

// One launch covers up to three independent problems of the same kind (latent-stream, dual-branch and context-stream
// layer): work items [0, end[0]) belong to problem 0, [end[0], end[1]) to problem 1, [end[1], end[2]) to problem 2.
struct Prob {
    const bf16_t* A;
    const bf16_t* Wp;
    void* out;
    int ldc, M, N, K;
    bool tiled;  // layout of Wp (GemmBf16Problem::w_tiled)
    EpiDev epi;
    bool then;   // ring kernel, EPI_GATE_RESID: the same tile of ProbSet::second follows in the same workgroup
    bool whole;  // rows are made of aligned groups of four columns, in the output and in what the epilogue reads (whole_rows)
};
constexpr int MAX_PROBS = 3;
struct ProbSet {
    Prob p[MAX_PROBS];
    // What a workgroup asks for first stands together: kernel arguments are a read from memory, and with `tiles_wgs` in another line of them than the
    // ends it waits for two such reads in front of its tile. Blocks of 256 + 77 tokens, width 768, 1536: 67.9, 104.0 us so, 67.2, 103.2 together.
    int end[MAX_PROBS];  // running totals of tiles
    int tiles_wgs;       // workgroups from here on work on `ada`
    Prob second;         // (see Prob::then)
    AdaWork ada;
    Ahead ahead;
    float us;            // (host) about how long the launch takes
    bool ada_last;       // (host) no launch behind this one can take any
};
// the layers of a block, whose launches take modulation projections along and read ahead
constexpr bool carries(int epi, bool out_f32) { return epi == EPI_GATE_RESID ? out_f32 : (epi == EPI_BIAS_GELU || epi == EPI_QKV_NORM) && !out_f32; }
// ... among the ring kernels not those of two workgroups per compute unit (four wavefronts per SIMD, MW), which are launched only where the tiles are more
// than the units, so that none is idle
constexpr bool ring_carries(int epi, bool out_f32, bool whole_rows, int mw) { return carries(epi, out_f32) && whole_rows && mw == 2; }

// One output tile: K loop + epilogue. `wg` is the tile's position in the XCD-aware order of its problem.
typedef __attribute__((__vector_size__(8 * sizeof(int)))) int i32x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4_t;

// FP8: the operands are OCP e4m3 bytes (A (M,K) and Wp (N,K), both K-contiguous); a 128-byte LDS row then holds 128 k values and
// the matrix instruction is v_mfma_f32_32x32x64_f8f6f4; the accumulators are multiplied by a_scale[m] * w_scale[n] in the epilogue.
// WIDE: operand rows so long that offsets inside a tile do not fit 32 bits (offsets_fit).
template <int BM, int BN, int WM, int WN, int STAGES, int EPI, bool OUT_F32, bool FP8, bool WIDE>
__device__ __forceinline__ void gemm_tile(const Prob& pr, const int wg, char* smem) {
    constexpr int ESZ = FP8 ? 1 : 2;                  // bytes per operand element
    const char* __restrict__ A = reinterpret_cast<const char*>(pr.A);
    const char* __restrict__ Wp = reinterpret_cast<const char*>(pr.Wp);
    void* __restrict__ out_ = pr.out;
    const int ldc = pr.ldc, M = pr.M, N = pr.N, K = pr.K;
    const EpiDev epi = pr.epi;
    constexpr int NT = WM * WN * 64;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;      // 32x32 MFMA blocks per wavefront
    constexpr int A_BYTES = BM * 128, STAGE_BYTES = (BM + BN) * 128;
    constexpr int LA = BM * 8 / NT, LB = BN * 8 / NT;        // 16-byte chunks per thread per tile
    static_assert(BM * 8 % NT == 0 && BN * 8 % NT == 0, "tile rows must divide evenly over the threads");
    static_assert(BM % (WM * 16) == 0 && BN % (WN * 16) == 0 && (!FP8 || (BM % (WM * 32) == 0 && BN % (WN * 32) == 0)), "wavefront tiles are made of 16x16 (bf16) or 32x32 (fp8) blocks");

    constexpr bool M16 = !FP8;  // bf16: 16x16x32 matrix instructions (see below); fp8: 32x32x64
    auto key = [](int row) { return M16 ? swz16(row) : swz(row); };
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS destinations of the direct loads are then scalar
    const int wm = wave / WN, wn = wave % WN;
    int tile_m, tile_n;
    tile_of_workgroup(wg, (M + BM - 1) / BM, (N + BN - 1) / BN, tile_m, tile_n);
    const int m_blk = tile_m * BM, n_blk = tile_n * BN;

    // ---- loader: chunk q = i*NT + tid lands at LDS byte q*16 of its tile, i.e. row q/8, physical chunk q%8 ----
    // Direct loads take one scalar address per operand, which moves on with the K tiles, and a 32-bit offset per thread, which does not: a 64-bit
    // address per load costs the vector unit an addition between the matrix instructions. 8192 + 308 rows, 256x256 tiles, warm: q|k|v 140 -> 132 us,
    // mlp-1 175 -> 168; the smaller tiles of the ring kernel gain 0 to 1 %; forwards 1.8 % (guided 512px pair), 256px 0, and nothing that lasts for the pair of
    // 1024px and for 2048px, which the power limit holds.
    typedef typename std::conditional<WIDE, long long, unsigned>::type offset_t;
    offset_t a_off[LA], b_off[LB];
    const long long row_bytes = (long long)K * ESZ;
    // bytes from one row of Wp to the next, and from one K tile to the next
    const long long w_row = !FP8 && pr.tiled ? 128 : row_bytes, w_tile = !FP8 && pr.tiled ? 128LL * N : 128;
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int q = i * NT + tid, row = q >> 3, lc = (q & 7) ^ key(row);
        const int m = min(row, M - 1 - m_blk);  // rows beyond M re-read the last row; their results are never stored
        a_off[i] = (offset_t)m * (offset_t)row_bytes + lc * 16;
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int q = i * NT + tid, row = q >> 3, lc = (q & 7) ^ key(row);
        const int n = min(row, N - 1 - n_blk);
        b_off[i] = (offset_t)n * (offset_t)w_row + lc * 16;
    }
    const char *a_base = A + (long long)m_blk * row_bytes, *b_base = Wp + (long long)n_blk * w_row;
    auto issue_tile = [&](int kt, int stage) {
        char* sa = smem + stage * STAGE_BYTES + wave * 1024;
        char* sb = sa + A_BYTES;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            if (!WIDE) asm volatile("" : "+v"(a_off[i]));  // (or the compiler widens the offset outside the loop and adds it to the address inside)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a_base + kt * 128LL + a_off[i]), (lds_ptr_t)(sa + i * NT * 16), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            if (!WIDE) asm volatile("" : "+v"(b_off[i]));
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(b_base + kt * w_tile + b_off[i]), (lds_ptr_t)(sb + i * NT * 16), 16, 0, 0);
        }
    };

    // bf16 uses v_mfma_f32_16x16x32_bf16: on this device the clock under matrix load is set by the power limit, and measured on
    // random operands the 16x16x32 form sustains 15-24 % more than 32x32x16 at the same nominal rate (half as many accumulator
    // updates per product). Both forms give bit-identical results.
    constexpr int MI = BM / WM / 16, NJ = BN / WN / 16;      // 16x16 blocks per wavefront
    f32x16_t acc[M16 ? 1 : TM][M16 ? 1 : TN];
    f32x4_t acc16[M16 ? MI : 1][M16 ? NJ : 1];
#pragma unroll
    for (int i = 0; i < (M16 ? 1 : TM); i++)
#pragma unroll
        for (int j = 0; j < (M16 ? 1 : TN); j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
#pragma unroll
    for (int i = 0; i < (M16 ? MI : 1); i++)
#pragma unroll
        for (int j = 0; j < (M16 ? NJ : 1); j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc16[i][j][r] = 0.f;

    static_assert(STAGES >= 2 && (STAGES - 1) * (LA + LB) < 64, "ring depth: at least two stages, and the loads in flight must fit the 6-bit counter");
    const int nkt = (int)(row_bytes / 128);
    const int l32 = lane & 31, lk = lane >> 5;   // position in a 32x32 block
    const int lr = lane & 15, lg = lane >> 4;    // position in a 16x16 block

    // ---- epilogue set-up ----
    constexpr int WNC = BN / WN;        // columns per wavefront
    constexpr int EP = WNC + 4;         // fp32 pitch of the staging slab
    static_assert(WM * WN * 32 * EP * 4 <= smem_bytes<BM, BN, WM, WN, STAGES>(), "epilogue staging must fit in the LDS allocation");
    constexpr int CPR = WNC / 4;        // float4 chunks per row
    static_assert(WNC % 4 == 0 && CPR <= 64, "a row of the wavefront's slab is made of float4 chunks");
    // rows covered by one pass of the wavefront: the largest power of two with RPI * CPR <= 64 (when CPR does not divide 64, as with
    // 48-column slabs, the lanes beyond RPI * CPR sit the epilogue out)
    constexpr int RPI = CPR > 32 ? 1 : CPR > 16 ? 2 : CPR > 8 ? 4 : CPR > 4 ? 8 : CPR > 2 ? 16 : 32;
    // rows per slab: 32 (measured faster than 16 on the 64-column slabs of the 256x256 tile), 16 for 48-column slabs
    constexpr int SR = (M16 && WNC % 64 != 0) ? 16 : 32;
    constexpr int NSLAB = BM / WM / SR;
    constexpr int NP = SR / RPI;        // rows of a slab per lane
    float* slab = reinterpret_cast<float*>(smem) + wave * 32 * EP;
    float* outf = reinterpret_cast<float*>(out_);
    bf16_t* outh = reinterpret_cast<bf16_t*>(out_);
    const bool lane_on = lane < RPI * CPR;
    const int e_row = lane_on ? lane / CPR : 0, e_col = lane_on ? (lane % CPR) * 4 : 0;
    const int n0 = n_blk + wn * WNC + e_col;
    const bool vec_ok = ((N & 3) == 0) && ((ldc & 3) == 0);
    const bool table_vec = EPI == EPI_BIAS_ROWADD && ((epi.gate_ld & 3) == 0) && ((reinterpret_cast<uintptr_t>(epi.table) & 15) == 0);
    const int nvalid = lane_on ? min(4, N - n0) : 0;  // <= 0 for lanes beyond the last column (and for lanes that sit out)
    // batch index of a row without a division per row: the tile starts in batch b0 and crosses a boundary every rpb rows
    const int rpb = epi.rows_per_batch, b0 = m_blk / rpb;
    // gated layers: the residual rows of the NEXT slab are requested before the current slab goes through LDS, so that
    // their latency is not paid once per slab with nothing else to do
    constexpr bool PREFETCH_RESID = (EPI == EPI_GATE_RESID);
    float4 rnext[PREFETCH_RESID ? NP : 1];
    auto request_resid = [&](int i) {
        if (PREFETCH_RESID && vec_ok)
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const int m = m_blk + wm * (BM / WM) + i * SR + p * RPI + e_row;
                if (m < M && nvalid > 0) rnext[p] = *reinterpret_cast<const float4*>(epi.resid + (long long)m * ldc + n0);
            }
    };
    if constexpr (M16) {
        // v_mfma_f32_16x16x32_bf16 operands: lane l holds row (column) l%16 of its block and the 8 consecutive k values 8*(l/16).. of
        // the 32-deep step: one 16-byte chunk of the row's 128-byte LDS line, chunk (4*step + l/16) ^ swz16(row)
        const int sw = swz16(lr);  // (block offsets are multiples of 16 rows, which the key does not see)
        const int a_off = (wm * (BM / WM) + lr) * 128, b_off = A_BYTES + (wn * (BN / WN) + lr) * 128;
        // A fragments: one buffer (the fragment of the next step replaces a[i] as soon as row block i is done), except for the last
        // TAIL row blocks, which have two so that no fragment read is left to issue behind the last matrix instructions of a step
        // (it would be waited for at once); B fragments: two buffers
        // (one such row block for the large tiles: more of them cost registers, which the gated fp32 epilogue then spills)
        constexpr int TAIL = MI >= 6 ? 1 : MI / 2, HEAD = MI - TAIL;
        // Where the direct loads of the next-but-one tile go among the 32 matrix instructions of a tile's last step: one behind every
        // second instruction, from the seventh on (behind the fragment reads of the first row block). Swept on the 24-block forward,
        // ms per step: first slot 0 / 2 / 3 / 4 / 5 / 6 / 7 / 8 / 16 with one load per instruction: +0.43 / +0.2 / +0.03 / 0 / -0.05 /
        // -0.1 / +0.18 / +0.15 / +0.56; from slot 6 every second / third instruction: -0.14 / -0.1.
        constexpr int LOAD_FIRST = 6, LOAD_EVERY = 2;
        static_assert(HEAD >= TAIL && TAIL >= 1, "every tail fragment is fetched behind a head row block");
        bf16x8_t a[HEAD], at[2][TAIL], b[2][NJ];
        auto a_addr = [&](const char* st, int s, int i) { return reinterpret_cast<const bf16x8_t*>(st + a_off + i * 16 * 128 + (((4 * s + lg) ^ sw) * 16)); };
        auto load_b = [&](const char* st, int s, int buf) {
#pragma unroll
            for (int j = 0; j < NJ; j++) b[buf][j] = *reinterpret_cast<const bf16x8_t*>(st + b_off + j * 16 * 128 + (((4 * s + lg) ^ sw) * 16));
        };

        // Every stage is filled up front and exactly one tile is requested per K tile after that (past the end: the last tile
        // once more, into a buffer nobody reads again), so "tile kt+1 has landed" is always "all but the newest STAGES-2 tiles".
#pragma unroll
        for (int s = 0; s < STAGES; s++) issue_tile(min(s, nkt - 1), s);
        wait_vmcnt<(STAGES - 1) * (LA + LB)>();
        // tile 0 is in LDS. A bare barrier between compiler fences: __syncthreads() would add a wait for ALL loads in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load_b(smem, 0, 0);
#pragma unroll
        for (int i = 0; i < HEAD; i++) a[i] = *a_addr(smem, 0, i);
#pragma unroll
        for (int i = 0; i < TAIL; i++) at[0][i] = *a_addr(smem, 0, HEAD + i);
        __builtin_amdgcn_sched_group_barrier(0x100, MI + NJ, 0);

        constexpr int KS = BK / 32;
        static_assert(KS == 2, "two 32-deep steps per K tile");
        // one 32-deep step on the fragments in a[], at[buf] and b[buf]; with FETCH, the fragments of step ns of stage nst are fetched
        // behind the matrix instructions: the B fragments first, the A fragment of head row block i once that block is done, the tail
        // fragments (into the other buffer) behind the first head blocks
        auto step = [&](int buf, const char* nst, int ns, auto fetch_tag, auto loads_tag) {
            constexpr bool FETCH = decltype(fetch_tag)::value, LOADS = decltype(loads_tag)::value;
            constexpr int NLOADS = LA + LB;
            static_assert(LOAD_FIRST + NLOADS * LOAD_EVERY <= MI * NJ, "the direct loads fit between the matrix instructions of one step");
            if (FETCH) load_b(nst, ns, buf ^ 1);
#pragma unroll
            for (int i = 0; i < MI; i++) {
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    acc16[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(i < HEAD ? a[i] : at[buf][i - HEAD], b[buf][j], acc16[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (FETCH && i == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                       // B fragment j of the next step
                    if (LOADS && i * NJ + j >= LOAD_FIRST && i * NJ + j < LOAD_FIRST + NLOADS * LOAD_EVERY && (i * NJ + j - LOAD_FIRST) % LOAD_EVERY == 0) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one direct load
                }
                if (FETCH && i < HEAD) {
                    a[i] = *a_addr(nst, ns, i);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (i < TAIL) {
                        at[buf ^ 1][i] = *a_addr(nst, ns, HEAD + i);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    }
                }
            }
        };
        // One K tile. The workgroup barrier sits in front of the LAST step of a tile, not behind it: by then every fragment
        // of tile kt is in registers (or on its way: waited for), so its buffer can be handed to the loads of tile kt+STAGES, and the
        // loads' issue and the fragment reads of tile kt+1 are interleaved with the matrix instructions of that last step.
        auto k_tile = [&](const int kt, auto has_next_tag) {
            constexpr bool HAS_NEXT = decltype(has_next_tag)::value;
            const char* st = smem + (kt % STAGES) * STAGE_BYTES;
            step(0, st, 1, std::true_type{}, std::false_type{});
            if (HAS_NEXT) {
                // this thread's loads of tile kt+1 have landed (vmcnt: all but the newest STAGES-2 tiles) and its reads of tile kt are done (lgkmcnt(0))
                constexpr int INFLIGHT = (STAGES - 2) * (LA + LB);
                __builtin_amdgcn_s_waitcnt((INFLIGHT & 15) | (7 << 4) | ((INFLIGHT >> 4) << 14));
                asm volatile("" ::: "memory");  // (the barrier builtin alone does not keep the compiler from moving LDS reads across it)
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                issue_tile(min(kt + STAGES, nkt - 1), kt % STAGES);
                step(1, smem + ((kt + 1) % STAGES) * STAGE_BYTES, 0, std::true_type{}, std::true_type{});
            } else {
                step(1, st, 0, std::false_type{}, std::false_type{});
            }
        };
        for (int kt = 0; kt + 1 < nkt; kt++) k_tile(kt, std::true_type{});
        k_tile(nkt - 1, std::false_type{});
    } else {
        // operand addresses inside a stage: row*128 + (chunk ^ sw)*16 with sw = swz(row) = swz(l32) (block offsets are multiples of 16).
        // k-step ks (64 deep) takes the two chunks 4*ks + 2*lk, +1
        const int sw = swz(l32);
        const int a_off = (wm * (BM / WM) + l32) * 128, b_off = A_BYTES + (wn * (BN / WN) + l32) * 128;
        // operand fragments of k-step ks live in buffer ks&1; those of step ks+1 are fetched from LDS while the matrix cores work on step ks
        i32x8_t a[2][TM], b[2][TN];
        auto read_frag = [&](const char* row, int ks) -> i32x8_t {
            const i32x4_t lo = *reinterpret_cast<const i32x4_t*>(row + (((4 * ks + 2 * lk) ^ sw) * 16));
            const i32x4_t hi = *reinterpret_cast<const i32x4_t*>(row + (((4 * ks + 2 * lk + 1) ^ sw) * 16));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        auto fetch = [&](const char* st, int ks, int buf) {
#pragma unroll
            for (int i = 0; i < TM; i++) a[buf][i] = read_frag(st + a_off + i * 32 * 128, ks);
#pragma unroll
            for (int j = 0; j < TN; j++) b[buf][j] = read_frag(st + b_off + j * 32 * 128, ks);
        };
        constexpr int DSR = 2;  // LDS reads per fragment

        // Every stage is filled up front and exactly one tile is requested per K tile after that (past the end: the last tile
        // once more, into a buffer nobody reads again), so "tile kt+1 has landed" is always "all but the newest STAGES-2 tiles".
#pragma unroll
        for (int s = 0; s < STAGES; s++) issue_tile(min(s, nkt - 1), s);
        wait_vmcnt<(STAGES - 1) * (LA + LB)>();
        // tile 0 is in LDS. A bare barrier between compiler fences: __syncthreads() would add a wait for ALL loads in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(smem, 0, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, DSR * (TM + TN), 0);

        constexpr int KS = 2;  // k-steps per 128-byte K tile
        // One K tile. The workgroup barrier sits in front of the LAST k-step of a tile, not behind it: by then every fragment
        // of tile kt is in registers (or on its way: waited for), so its buffer can be handed to the loads of tile kt+2, and the
        // loads' issue and the first fragment reads of tile kt+1 are interleaved with the matrix instructions of that last
        // step. With the barrier between tiles instead, the matrix pipeline drains at every tile boundary while all
        // wavefronts of the compute unit wait for the barrier, issue their loads and wait for their first LDS reads.
        auto k_tile = [&](const int kt, auto has_next_tag) {
            constexpr bool HAS_NEXT = decltype(has_next_tag)::value;
            const char* st = smem + (kt % STAGES) * STAGE_BYTES;
            auto mfmas = [&](int buf) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[buf][i], b[buf][j], acc[i][j], 0, 0, 0, 0, 0, 0);
            };
            // scheduling pattern of a step: behind each of the first matrix instructions one LDS fragment read of the next step
            // (and, in the last step, one direct global->LDS load of the tile after next), so that their issue and latency are
            // covered by matrix work
#pragma unroll
            for (int ks = 0; ks + 1 < KS; ks++) {
                fetch(st, ks + 1, (ks + 1) & 1);
                mfmas(ks & 1);
#pragma unroll
                for (int x = 0; x < TM + TN; x++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // 1 MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, DSR, 0);  // 1 fragment read
                }
                __builtin_amdgcn_sched_group_barrier(0x008, TM * TN - (TM + TN), 0);
            }
            if (HAS_NEXT) {
                // this thread's loads of tile kt+1 have landed (vmcnt: all but the newest STAGES-2 tiles) and its reads of tile kt are done (lgkmcnt(0))
                constexpr int INFLIGHT = (STAGES - 2) * (LA + LB);
                __builtin_amdgcn_s_waitcnt((INFLIGHT & 15) | (7 << 4) | ((INFLIGHT >> 4) << 14));
                asm volatile("" ::: "memory");  // (the barrier builtin alone does not keep the compiler from moving LDS reads across it)
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                issue_tile(min(kt + STAGES, nkt - 1), kt % STAGES);
                fetch(smem + ((kt + 1) % STAGES) * STAGE_BYTES, 0, 0);
            }
            mfmas((KS - 1) & 1);
            if (HAS_NEXT) {
                constexpr int NLOADS = LA + LB, NM = TM * TN;
                constexpr int LPS = (NLOADS + NM - 1) / NM;   // loads per slot
                static_assert(TM + TN <= NM, "more fragment reads than matrix instructions to hide them behind");
#pragma unroll
                for (int x = 0; x < NM; x++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                              // 1 MFMA
                    if (x < TM + TN) __builtin_amdgcn_sched_group_barrier(0x100, DSR, 0);            // 1 fragment read
                    if (x * LPS < NLOADS) __builtin_amdgcn_sched_group_barrier(0x020, LPS, 0);       // VMEM reads
                }
            }
        };
        for (int kt = 0; kt + 1 < nkt; kt++) k_tile(kt, std::true_type{});
        k_tile(nkt - 1, std::false_type{});
    }

    // ---- epilogue. The MFMA C layouts (32x32: lane = column, register r = row 8*(r/4) + 4*(lane/32) + r%4) would give 2- or
    // 4-byte scattered stores; each wavefront instead transposes one 32-row slab at a time through its private LDS
    // region (the tile ring is free now) and leaves with 16 lanes covering 64 contiguous columns of one row.
    __syncthreads();
    if constexpr (EPI == EPI_GATE_RESID && OUT_F32 && M16 && WNC % 64 == 0) {
        // Gated tiles that lie inside the matrix, with rows of at most two batch elements per wavefront: nothing is read or stored under a condition, so that the waits are counted
        // exactly: a slab's residual rows, requested a slab ahead, are waited for without the stores behind them, and the gates are read once. (Else every row's gate waits for
        // everything in flight, 32 times a tile: the pair of 1024px 22915 -> 22845 us without this form and 23426 -> 22919 with
        // it, 2048px 82564 -> 81467.)
        const int m_wave = m_blk + wm * (BM / WM), first = m_wave / rpb, last = (m_wave + BM / WM - 1) / rpb;
        if (vec_ok && m_blk + BM <= M && n_blk + BN <= N && last - first <= 1) {
            const long long lane_at = (long long)(m_wave + e_row) * ldc + n0;
            auto at4 = [](const float* p) { return *reinterpret_cast<const f32x4_t*>(p); };
            f32x4_t bias = epi.bias ? *reinterpret_cast<const f32x4_any_t*>(epi.bias + n0) : f32x4_any_t{0.f, 0.f, 0.f, 0.f};
            f32x4_t gate_first = at4(epi.gate + (long long)first * epi.gate_ld + n0), gate_last = at4(epi.gate + (long long)last * epi.gate_ld + n0), next[NP];
            auto request = [&](int i) {
#pragma unroll
                for (int p = 0; p < NP; p++) next[p] = at4(epi.resid + lane_at + (long long)(i * SR + p * RPI) * ldc);
            };
            request(0);
            asm volatile("" : "+v"(bias), "+v"(gate_first), "+v"(gate_last));  // (named, so that they are waited for here)
#pragma unroll
            for (int i = 0; i < NSLAB; i++) {
                f32x4_t cur[NP], vals[NP];
#pragma unroll
                for (int p = 0; p < NP; p++) cur[p] = next[p];
                if (i + 1 < NSLAB) request(i + 1);
#pragma unroll
                for (int ii = 0; ii < SR / 16; ii++)
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++) slab[(16 * ii + 4 * lg + r) * EP + j * 16 + lr] = acc16[(SR / 16) * i + ii][j][r];
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int p = 0; p < NP; p++) vals[p] = at4(&slab[(p * RPI + e_row) * EP + e_col]);
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    const bool second = m_wave + i * SR + p * RPI + e_row >= last * rpb;
                    f32x4_t v;
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = fmaf(second ? gate_last[c] : gate_first[c], vals[p][c] + bias[c], cur[p][c]);
                    *reinterpret_cast<f32x4_t*>(outf + lane_at + (long long)(i * SR + p * RPI) * ldc) = v;
                }
                __builtin_amdgcn_wave_barrier();
            }
            return;
        }
    }
    float bias4[4] = {0.f, 0.f, 0.f, 0.f};
    if (epi.bias)
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c < nvalid) bias4[c] = epi.bias[n0 + c];
    float ws4[4] = {1.f, 1.f, 1.f, 1.f};  // fp8: the output column's factor
    if (FP8 && epi.w_scale)
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c < nvalid) ws4[c] = epi.w_scale[n0 + c];
    // 0 = q, 1 = k, 2 = v (uniform over 16 lanes: C is a multiple of 64). The weights are read once: row by row, each read waits for everything in flight (forwards of
    // 1024px 12376 -> 12267 us, its pair 22388 -> 22159, the 512px pair 6128 -> 6065).
    const int third = EPI == EPI_QKV_NORM ? n0 / epi.gate_ld : 2;
    f32x4_t norm_w = {1.f, 1.f, 1.f, 1.f};
    if (EPI == EPI_QKV_NORM && WNC % 64 == 0) {
        if (third < 2 && nvalid > 0) norm_w = *reinterpret_cast<const f32x4_t*>((third == 0 ? epi.gate : epi.resid) + (n0 & 63));
        asm volatile("" : "+v"(norm_w));
#pragma unroll
        for (int c = 0; c < 4; c++) asm volatile("" : "+v"(bias4[c]));
    }
    request_resid(0);
#pragma unroll
    for (int i = 0; i < NSLAB; i++) {
        float4 rcur[PREFETCH_RESID ? NP : 1];
        if (PREFETCH_RESID) {
#pragma unroll
            for (int p = 0; p < NP; p++) rcur[p] = rnext[p];
            if (i + 1 < NSLAB) request_resid(i + 1);
        }
        if constexpr (M16) {
            // C layout of a 16x16 block: lane = column l%16, register r = row 4*(l/16) + r
#pragma unroll
            for (int ii = 0; ii < SR / 16; ii++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) slab[(16 * ii + 4 * lg + r) * EP + j * 16 + lr] = acc16[(SR / 16) * i + ii][j][r];
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) slab[(8 * (r >> 2) + 4 * lk + (r & 3)) * EP + j * 32 + l32] = acc[i][j][r];
        }
        // LDS operations of one wavefront execute in program order, so the reads below see the writes above without a
        // fence (a fence would also make the wavefront wait for its outstanding global stores on every pass)
        __builtin_amdgcn_wave_barrier();
        // all rows of the slab are read into registers of their own before the first store is issued: a store keeps its data
        // registers busy until it has left, so reusing one register set per row would put a full store round trip between rows
        float4 vals[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) vals[p] = *reinterpret_cast<const float4*>(&slab[(p * RPI + e_row) * EP + e_col]);
        float4 res[NP];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int row = p * RPI + e_row;
            const int m = m_blk + wm * (BM / WM) + i * SR + row;
            if (m < M && nvalid > 0) {
                float4 a4 = vals[p];
                if constexpr (FP8) {
                    const float sa = epi.a_scale ? epi.a_scale[m] : 1.0f;
                    a4.x *= sa * ws4[0]; a4.y *= sa * ws4[1]; a4.z *= sa * ws4[2]; a4.w *= sa * ws4[3];
                }
                float v[4] = {a4.x + bias4[0], a4.y + bias4[1], a4.z + bias4[2], a4.w + bias4[3]};
                const long long idx = (long long)m * ldc + n0;
                if (EPI == EPI_BIAS_GELU) {
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = gelu_tanh_f(v[c]);
                } else if (EPI == EPI_BIAS_SILU) {
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = v[c] / (1.0f + __expf(-v[c]));
                } else if (EPI == EPI_GATE_RESID) {
                    int bi = b0;
                    for (int nb = (b0 + 1) * rpb; nb <= m; nb += rpb) bi++;  // at most BM/rpb + 1 steps, 0 or 1 in practice
                    const float* g = epi.gate + (long long)bi * epi.gate_ld + n0;
                    if (vec_ok) {
                        const float4 g4 = *reinterpret_cast<const float4*>(g), r4 = rcur[PREFETCH_RESID ? p : 0];
                        v[0] = fmaf(g4.x, v[0], r4.x); v[1] = fmaf(g4.y, v[1], r4.y); v[2] = fmaf(g4.z, v[2], r4.z); v[3] = fmaf(g4.w, v[3], r4.w);
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; c++)
                            if (c < nvalid) v[c] = fmaf(g[c], v[c], epi.resid[idx + c]);
                    }
                } else if (EPI == EPI_BIAS_ROWADD) {
                    const float* t = epi.table + (long long)(m % rpb) * epi.gate_ld + n0;
                    if (vec_ok && table_vec) {
                        const float4 t4 = *reinterpret_cast<const float4*>(t);
                        v[0] += t4.x; v[1] += t4.y; v[2] += t4.z; v[3] += t4.w;
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; c++)
                            if (c < nvalid) v[c] += t[c];
                    }
                }
                if constexpr (EPI == EPI_QKV_NORM && WNC % 64 == 0) {
                    // 16 consecutive lanes hold 64 consecutive columns of this row = one head of one token (modules.cpp:192-198, fused)
                    if (third < 2) qk_norm4(v, make_float4(norm_w[0], norm_w[1], norm_w[2], norm_w[3]));
                }
                res[p] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
        // ... and all stores of the slab leave back to back
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int m = m_blk + wm * (BM / WM) + i * SR + p * RPI + e_row;
            if (m < M && nvalid > 0) {
                const long long idx = (long long)m * ldc + n0;
                const float v[4] = {res[p].x, res[p].y, res[p].z, res[p].w};
                if (vec_ok) {
                    if (OUT_F32) *reinterpret_cast<float4*>(outf + idx) = make_float4(v[0], v[1], v[2], v[3]);
                    else *reinterpret_cast<uint2*>(outh + idx) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        if (c < nvalid) {
                            if (OUT_F32) outf[idx + c] = v[c];
                            else outh[idx + c] = f32_to_bf16(v[c]);
                        }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Persistent kernel: one workgroup per compute unit walks over the tiles of up to three problems. The stores of a finished
// tile drain while the next tile's K loop is already running, instead of holding the compute unit until they retire.
// Workgroup g takes work items g, g + G, g + 2G ... (G = grid size, a multiple of 8), so it stays on its XCD's run of tiles.
template <int BM, int BN, int WM, int WN, int STAGES, int EPI, bool OUT_F32, bool FP8 = false, bool WIDE = false>
__global__ void __launch_bounds__(WM* WN * 64) gemm_bf16_kernel(const ProbSet args) {
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    if (carries(EPI, OUT_F32) && !FP8 && !WIDE && (int)blockIdx.x >= args.tiles_wgs) {
        ada_carried<WM * WN * 64>(args.ada, blockIdx.x - args.tiles_wgs, gridDim.x - args.tiles_wgs, smem);
        read_ahead<WM * WN * 64>(args.ahead, blockIdx.x - args.tiles_wgs, gridDim.x - args.tiles_wgs);
        return;
    }
    for (int w = blockIdx.x; w < args.end[MAX_PROBS - 1]; w += args.tiles_wgs) {
        const int which = (w >= args.end[0]) + (w >= args.end[1]);
        gemm_tile<BM, BN, WM, WN, STAGES, EPI, OUT_F32, FP8, WIDE>(args.p[which], w - (which ? args.end[which - 1] : 0), smem);
        __syncthreads();  // the staging slabs of this tile's epilogue alias the ring the next tile fills
    }
}

// How many workgroups a launch of `wgs` adds for the modulation projections (args.ada.count panels at most; what it takes is left there): one
// for every compute unit that it leaves idle, each as many panels as it has time for (passenger_panels). At width 1536, with 5.5 us for a panel and
// 5 for the start instead of 6.5 and 6, forwards of 512px and its guided pair are 0.8 % slower. A share per launch (a third of the block's panels)
// instead of as many as there is room: 256px 0, 496x272 +3.3 %.
// In the time that is left they read the weights ahead that the next launches ask for (args.ahead; what is read is left there). At 12, 24, 40, 60,
// 100 KB per us and workgroup: forwards of 256px -0.9, -2.4, -3.0, -3.1, -3.3 %, its pair -6.0 from 40 on, of the 512px pair +0.1, -0.7, -1.25, -1.25,
// -1.0, 496x272 batch 3 -0.1, -0.2, 0, +0.9, +13 (the launch is then longer for it), 512px 0 (16 to 28 idle units).
template <bool CARRIES>
int carried_wgs(ProbSet& args, int wgs, int cus, int smem) {
    constexpr double RATE = 40960;  // bytes per us and workgroup that reads ahead
    const int idle = cus - wgs, want = args.ada.count;
    args.ada.count = 0;
    if (!CARRIES || idle <= 0) {
        args.ahead = Ahead{};
        return 0;
    }
    int panels = 0;  // a workgroup's
    if (want > 0 && smem >= ada_lds_bytes(ADA_CARRY_ROWS, args.ada.K)) {
        panels = passenger_panels(args.us, args.ada.K, want, idle, args.ada_last);
        args.ada.count = want < panels * idle ? want : panels * idle;
    }
    const double us = args.us - (panels ? PASSENGER_START + panels * passenger_panel_us(args.ada.K) : PASSENGER_START / 2);
    const size_t ahead = args.ahead.trim(us > 0 ? (size_t)(us * RATE * idle) : 0);
    const int readers = (int)(ahead / 32768 < (size_t)idle ? ahead / 32768 : idle), takers = panels ? (args.ada.count + panels - 1) / panels : 0;
    return readers > takers ? readers : takers;
}

template <int BM, int BN, int WM, int WN, int STAGES, int EPI, bool OUT_F32, bool FP8 = false, bool WIDE = false>
int launch_cfg(ProbSet& args, int n, hipStream_t st) {
    auto kern = gemm_bf16_kernel<BM, BN, WM, WN, STAGES, EPI, OUT_F32, FP8, WIDE>;
    constexpr int smem = smem_bytes<BM, BN, WM, WN, STAGES>();
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(kern), smem));
    if (EPI == EPI_QKV_NORM && (BN / WN) % 64 != 0) return fail(SD3_ERR_UNSUPPORTED, "gemm_bf16: this tile shape cannot fuse the qk-norm");
    int total = 0;
    for (int i = 0; i < MAX_PROBS; i++) {
        if (i < n) total += ((args.p[i].N + BN - 1) / BN) * ((args.p[i].M + BM - 1) / BM);
        args.end[i] = total;
    }
    // as many workgroups as can be resident at once (LDS allows one 256x256 or two 128x128 workgroups per compute unit), rounded
    // down to a multiple of the 8 XCDs
    const int cus = compute_units();
    if (cus <= 0) return SD3_ERR_HIP;
    constexpr int per_cu = (160 * 1024) / smem > 1 ? 2 : 1;
    const int resident = (cus * per_cu / 8 * 8) > 8 ? (cus * per_cu / 8 * 8) : 8;
    args.tiles_wgs = total < resident ? total : resident;
    const dim3 grid(args.tiles_wgs + carried_wgs<carries(EPI, OUT_F32) && !FP8 && !WIDE>(args, args.tiles_wgs, cus, smem)), block(WM * WN * 64);
    hipLaunchKernelGGL(kern, grid, block, smem, st, args);
    g_gemm_bf16_launches.fetch_add(1, std::memory_order_relaxed);
    return launch_status("gemm_bf16");
}

// whether tiles of `rows` rows (of either operand) address their operands, `esz` bytes a value, by 32-bit offsets
bool addresses(const ProbSet& set, int n, int rows, int esz) {
    for (int i = 0; i < n; i++)
        if (!offsets_fit(rows, (long long)set.p[i].K * esz)) return false;
    return true;
}

// fp8 operands: 256x256 tiles (variant 4) or 128x128 tiles with a ring of two stages (anything else)
template <int EPI, bool OUT_F32>
int launch_epi_fp8(int variant, ProbSet& args, int n, hipStream_t st) {
    if (!addresses(args, n, 128, 1)) return launch_cfg<128, 128, 2, 2, 2, EPI, OUT_F32, true, true>(args, n, st);
    if (variant == 4 && addresses(args, n, 256, 1)) return launch_cfg<256, 256, 2, 4, 2, EPI, OUT_F32, true>(args, n, st);
    return launch_cfg<128, 128, 2, 2, 2, EPI, OUT_F32, true>(args, n, st);
}

// ---- launches that do not fill the device with 256x256 tiles ----
// A layer of a few hundred to a few thousand rows is fewer 256x256 tiles than there are compute units, and what it waits for is its
// weights, which nobody has touched yet: the K loop's pace is set by how many compute units take part and by the bytes each has in
// flight, less by the matrix instructions. So: a range of smaller tiles (64-column wavefronts: one attention head, so that the qk-norm
// stays inside a wavefront), one workgroup per tile, eight wavefronts for all but the smallest (two per SIMD: 128x128 tiles of 8 against 4
// wavefronts, mlp-2 of 2356 rows, 59 against 65 us), a ring of stages as deep as the LDS allows, fragments fetched a whole K tile (or half
// of one) ahead of their matrix instructions, one barrier per K tile. mlp-2 with cold weights, rows 333 / 1178 / 2356 / 4250: 64 -> 31,
// 86 -> 44, 86 -> 60, 99 -> 83 us.
// Lane l of a 16-column block of W holds row l%16 of its LDS block; the loader puts output column NJ*(l%16) + j there (block j), so a lane
// ends with NJ consecutive columns of a row and the epilogue stores straight from the accumulators.
// The order of k is that of the other tiles (bit-identical results).
// waits until all but the newest `ahead` tiles (at most MAX, PER loads of this thread each) have landed
template <int MAX, int PER>
__device__ __forceinline__ void wait_tiles(int ahead) {
    if constexpr (MAX == 0) wait_vmcnt<0>();
    else if (ahead >= MAX) wait_vmcnt<MAX * PER>();
    else wait_tiles<MAX - 1, PER>(ahead);
}
// WHOLE_ROWS: the epilogue stores (and reads back) four columns at a time, as every problem of the launch allows; else element by element
template <int TM, int TN, int WM, int WN, int STAGES, int MW, int EPI, bool OUT_F32, bool WHOLE_ROWS>
__global__ void __launch_bounds__(WM* WN * 64, MW) gemm_bf16_ring_kernel(const ProbSet args) {
    constexpr int NT = WM * WN * 64, TI = TM / WM / 16, WC = TN / WN, NJ = WC / 16;
    constexpr int A_BYTES = TM * 128, STAGE_BYTES = (TM + TN) * 128;
    constexpr int LA = TM * 8 / NT, LB = TN * 8 / NT;
    static_assert(NJ == 4 && TI >= 1 && TM * 8 % NT == 0 && TN * 8 % NT == 0, "tile shape");
    static_assert(STAGES >= 2 && (STAGES - 1) * (LA + LB) < 64, "the loads in flight must fit the 6-bit counter");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    if (ring_carries(EPI, OUT_F32, WHOLE_ROWS, MW) && (int)blockIdx.x >= args.tiles_wgs) {
        ada_carried<NT>(args.ada, blockIdx.x - args.tiles_wgs, gridDim.x - args.tiles_wgs, smem);
        read_ahead<NT>(args.ahead, blockIdx.x - args.tiles_wgs, gridDim.x - args.tiles_wgs);
        return;
    }
    const int w = blockIdx.x;
    const int which = (w >= args.end[0]) + (w >= args.end[1]);
    const Prob& pr = args.p[which];
    const int M = pr.M, N = pr.N, K = pr.K, ldc = pr.ldc;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    int tile_m, tile_n;
    tile_of_workgroup(w - (which ? args.end[which - 1] : 0), (M + TM - 1) / TM, (N + TN - 1) / TN, tile_m, tile_n);
    const int m_blk = tile_m * TM, n_blk = tile_n * TN;

    // Direct loads take one scalar address per operand, which moves on with the K tiles, and a 32-bit offset per thread, which does not
    unsigned a_off[LA], b_off[LB];
    const char *a_base, *b_base;
    long long w_tile;  // bytes from one K tile of the weight to the next
    auto operands = [&](const bf16_t* A, const bf16_t* Wp, bool tiled) {
        const int w_row = tiled ? 128 : 2 * K;
        w_tile = tiled ? 128LL * N : 128;
        a_base = reinterpret_cast<const char*>(A + (long long)m_blk * K);
        b_base = reinterpret_cast<const char*>(Wp) + (long long)n_blk * w_row;
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int q = i * NT + tid, row = q >> 3;
            a_off[i] = (unsigned)min(row, M - 1 - m_blk) * (2 * K) + ((q & 7) ^ swz16(row)) * 16;
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            const int q = i * NT + tid, row = q >> 3;
            const int n = row / WC * WC + NJ * (row % 16) + row % WC / 16;
            b_off[i] = (unsigned)min(n, N - 1 - n_blk) * w_row + ((q & 7) ^ swz16(row)) * 16;
        }
    };
    operands(pr.A, pr.Wp, pr.tiled);
    const int nkt = K / BK;
    auto issue_tile = [&](int kt, int stage) {
        char* sa = smem + stage * STAGE_BYTES + wave * 1024;
        char* sb = sa + A_BYTES;
        const char *a = a_base + kt * 128, *b = b_base + kt * w_tile;
        asm volatile("" : "+s"(a), "+s"(b));  // (or of two tiles that are unrolled together one gets 64-bit addresses per thread again)
#pragma unroll
        for (int i = 0; i < LA; i++) {
            asm volatile("" : "+v"(a_off[i]));  // (or the compiler widens the offset outside the loop and adds it to the address inside)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(a + a_off[i]), (lds_ptr_t)(sa + i * NT * 16), 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            asm volatile("" : "+v"(b_off[i]));
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(b + b_off[i]), (lds_ptr_t)(sb + i * NT * 16), 16, 0, 0);
        }
    };
    f32x4_t acc[TI][NJ];
    // Fragments are fetched ahead of their matrix instructions: a whole K tile ahead where it fits the registers, else one 32-deep half
    constexpr bool WHOLE = TI * NJ < 16 && MW <= 2;
    bf16x8_t a[WHOLE ? 2 : 1][2][TI], b[WHOLE ? 2 : 1][2][NJ];  // [buffer][half]
    auto fetch_half = [&](int stage, int buf, int h) {
        const char* st = smem + stage * STAGE_BYTES;
        const int chunk = ((4 * h + lg) ^ swz16(lr)) * 16;
#pragma unroll
        for (int i = 0; i < TI; i++) a[buf][h][i] = *reinterpret_cast<const bf16x8_t*>(st + (wm * (TM / WM) + i * 16 + lr) * 128 + chunk);
#pragma unroll
        for (int j = 0; j < NJ; j++) b[buf][h][j] = *reinterpret_cast<const bf16x8_t*>(st + A_BYTES + (wn * WC + j * 16 + lr) * 128 + chunk);
    };
    auto multiply_half = [&](int buf, int h) {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[buf][h][i], b[buf][h][j], acc[i][j], 0, 0, 0);
    };
    // schedule: NR LDS reads behind the first matrix instructions, then (with LOADS) one direct load behind each of the next ones
    auto spread = [&](auto nm_tag, auto nr_tag, auto loads_tag) {
        constexpr int NM = decltype(nm_tag)::value, NR = decltype(nr_tag)::value, PER = (NR + NM - 1) / NM, SLOTS = (NR + PER - 1) / PER;
#pragma unroll
        for (int x = 0; x < SLOTS; x++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);
        }
        if (decltype(loads_tag)::value)
#pragma unroll
            for (int x = 0; x < LA + LB; x++) {
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
        __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto fill_ring = [&]() {
#pragma unroll
        for (int s = 0; s < STAGES; s++)
            if (s < nkt) issue_tile(s, s);
    };
    int stage;
    // One K tile: once its fragments are in registers hand its stage back, request the tile STAGES ahead into it, and fetch the next tile's
    // fragments beside the matrix instructions. (Past the end nothing is requested: a deep ring's surplus tiles would be a quarter of the
    // traffic of a launch with 24 K tiles.)
    auto k_tile = [&](int kt, auto buf_tag, auto more_tag) {
        constexpr bool MORE = decltype(more_tag)::value;
        constexpr int BUF = WHOLE ? decltype(buf_tag)::value : 0;
        using std::integral_constant;
        if constexpr (!WHOLE) {
            fetch_half(stage, 0, 1);
            multiply_half(0, 0);
            spread(integral_constant<int, TI * NJ>{}, integral_constant<int, TI + NJ>{}, std::false_type{});
        }
        if (MORE) wait_tiles<STAGES - 2, LA + LB>(STAGES - 2);
        else wait_tiles<STAGES - 2, LA + LB>(nkt - 2 - kt);  // tile kt+1 has landed ...
        __builtin_amdgcn_s_waitcnt(0xc07f);                  // ... and this thread's LDS reads of tile kt are done (lgkmcnt(0))
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int freed = stage;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        fetch_half(stage, WHOLE ? BUF ^ 1 : 0, 0);
        if (WHOLE) fetch_half(stage, BUF ^ 1, 1);
        if (MORE) issue_tile(kt + STAGES, freed);
        if constexpr (WHOLE) {
            multiply_half(BUF, 0);
            multiply_half(BUF, 1);
            spread(integral_constant<int, 2 * TI * NJ>{}, integral_constant<int, 2 * (TI + NJ)>{}, more_tag);
        } else {
            multiply_half(0, 1);
            spread(integral_constant<int, TI * NJ>{}, integral_constant<int, TI + NJ>{}, more_tag);
        }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    auto k_loop = [&]() {
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        wait_tiles<STAGES - 1, LA + LB>(nkt - 1);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch_half(0, 0, 0);
        if (WHOLE) fetch_half(0, 0, 1);
        stage = 0;
        int kt = 0;
        for (; kt + 1 + STAGES < nkt; kt += 2) {
            k_tile(kt, even, std::true_type{});
            k_tile(kt + 1, odd, std::true_type{});
        }
        if (kt + STAGES < nkt) {
            k_tile(kt++, even, std::true_type{});
#pragma unroll 1
            for (; kt < nkt; kt += 2) {
                k_tile(kt, odd, std::false_type{});
                if (kt + 1 < nkt) k_tile(kt + 1, even, std::false_type{});
            }
        } else {
#pragma unroll 1
            for (; kt < nkt; kt += 2) {
                k_tile(kt, even, std::false_type{});
                if (kt + 1 < nkt) k_tile(kt + 1, odd, std::false_type{});
            }
        }
    };
    const int n0 = n_blk + wn * WC + NJ * lr, m_wave = m_blk + wm * (TM / WM);  // the lane's first column, the wavefront's first row
    // What the epilogue of whole rows reads, requested together and waited for once (row by row, each behind the store of the one before, a tile's
    // 4 to 16 rows were as many trips to memory; outputs the same bits: forwards of 256px 2519 -> 2456 us, 512px 4015 -> 3951, its pair 6153 -> 6089, 496x272 6657 -> 6499, 1024px 12650
    // -> 12399, the block of 256 + 77 tokens 103.7 -> 100.1. In front of the K loop they would hide altogether, but spill in it: +1 to +2.4 %). Gates: of the batch elements of the wavefront's first and last row; rows of more than
    // two (`few` is false) read theirs one by one.
    constexpr bool READS = EPI == EPI_GATE_RESID || EPI == EPI_BIAS_ROWADD;
    f32x4_t bias4, norm_w, gate_first, gate_last, rows[READS ? TI : 1][4];
    int third = 0, second_from = 0;
    bool few = true;
    auto request = [&](const Prob& pr) {
        if (!WHOLE_ROWS) return;
        const EpiDev& epi = pr.epi;
        const int n = min(n0, N - 4), rpb = epi.rows_per_batch;
        bias4 = epi.bias ? *reinterpret_cast<const f32x4_any_t*>(epi.bias + n) : f32x4_any_t{0.f, 0.f, 0.f, 0.f};
        if (EPI == EPI_QKV_NORM) {
            third = n / epi.gate_ld;
            norm_w = third < 2 ? *reinterpret_cast<const f32x4_t*>((third == 0 ? epi.gate : epi.resid) + (n & 63)) : f32x4_t{1.f, 1.f, 1.f, 1.f};
        }
        if (EPI == EPI_GATE_RESID) {
            const int first = min(m_wave, M - 1) / rpb, last = min(m_wave + TI * 16, M) - 1 > 0 ? (min(m_wave + TI * 16, M) - 1) / rpb : 0;
            few = last - first <= 1;
            second_from = last * rpb;
            gate_first = *reinterpret_cast<const f32x4_t*>(epi.gate + (long long)first * epi.gate_ld + n);
            gate_last = *reinterpret_cast<const f32x4_t*>(epi.gate + (long long)last * epi.gate_ld + n);
        }
        if constexpr (READS) {
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = min(m_wave + i * 16 + 4 * lg + r, M - 1);
                    rows[i][r] = *reinterpret_cast<const f32x4_t*>(EPI == EPI_GATE_RESID ? epi.resid + (long long)m * ldc + n : epi.table + (long long)(m % rpb) * epi.gate_ld + n);
                }
        }
    };
    auto arrived = [](f32x4_t& v) { asm volatile("" : "+v"(v)); };  // (named, so that it is waited for here)
    auto epilogue = [&](const Prob& pr) {
        if (n0 >= N) return;
        int n = n0, row0 = m_wave + 4 * lg;
        asm volatile("" : "+v"(n), "+v"(row0));  // (or addresses are formed in front of the K loop and held through it)
        const EpiDev& epi = pr.epi;
        const int rpb = epi.rows_per_batch;
        if constexpr (WHOLE_ROWS) {
            arrived(bias4);
            if (EPI == EPI_QKV_NORM) arrived(norm_w);
            if (EPI == EPI_GATE_RESID) {
                arrived(gate_first);
                arrived(gate_last);
            }
            if constexpr (READS) {
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) arrived(rows[i][r]);
            }
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = row0 + i * 16 + r;  // (uniform over the 16 lanes that share a head)
                    float v[4] = {acc[i][0][r] + bias4[0], acc[i][1][r] + bias4[1], acc[i][2][r] + bias4[2], acc[i][3][r] + bias4[3]};
                    if (EPI == EPI_BIAS_GELU) {
#pragma unroll
                        for (int c = 0; c < 4; c++) v[c] = gelu_tanh_f(v[c]);
                    } else if (EPI == EPI_BIAS_SILU) {
#pragma unroll
                        for (int c = 0; c < 4; c++) v[c] = v[c] / (1.0f + __expf(-v[c]));
                    } else if (EPI == EPI_GATE_RESID) {
                        f32x4_t g4;
#pragma unroll
                        for (int c = 0; c < 4; c++) g4[c] = m >= second_from ? gate_last[c] : gate_first[c];
                        if (!few) {
                            g4 = *reinterpret_cast<const f32x4_t*>(epi.gate + (long long)(min(m, M - 1) / rpb) * epi.gate_ld + n);
                            arrived(g4);  // (in here, or the others wait as well)
                        }
                        const f32x4_t r4 = rows[READS ? i : 0][r];
#pragma unroll
                        for (int c = 0; c < 4; c++) v[c] = fmaf(g4[c], v[c], r4[c]);
                    } else if (EPI == EPI_BIAS_ROWADD) {
                        const f32x4_t t4 = rows[READS ? i : 0][r];
                        v[0] += t4[0]; v[1] += t4[1]; v[2] += t4[2]; v[3] += t4[3];
                    } else if (EPI == EPI_QKV_NORM && third < 2) {
                        qk_norm4(v, make_float4(norm_w[0], norm_w[1], norm_w[2], norm_w[3]));
                    }
                    const long long idx = (long long)m * ldc + n;
                    if (m < M) {
                        if (OUT_F32) *reinterpret_cast<float4*>(reinterpret_cast<float*>(pr.out) + idx) = make_float4(v[0], v[1], v[2], v[3]);
                        else *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(pr.out) + idx) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                    }
                }
            return;
        }
        const int valid = N - n0;  // (element by element: columns of this lane's four that exist, if fewer than four)
        auto four = [&](const float* p) { return make_float4(p[0], valid > 1 ? p[1] : 0.f, valid > 2 ? p[2] : 0.f, valid > 3 ? p[3] : 0.f); };
        float bias4[4] = {0.f, 0.f, 0.f, 0.f};
        if (epi.bias)
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (c < valid) bias4[c] = epi.bias[n0 + c];
        const int third_e = EPI == EPI_QKV_NORM ? n0 / epi.gate_ld : 0;
        float4 norm_w = make_float4(1.f, 1.f, 1.f, 1.f);
        if (EPI == EPI_QKV_NORM && third_e < 2) norm_w = *reinterpret_cast<const float4*>((third_e == 0 ? epi.gate : epi.resid) + (n0 & 63));
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m_wave + i * 16 + 4 * lg + r;
                if (m >= M) continue;
                const long long idx = (long long)m * ldc + n0;
                float v[4];
#pragma unroll
                for (int c = 0; c < 4; c++) v[c] = acc[i][c][r] + bias4[c];
                if (EPI == EPI_BIAS_GELU) {
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = gelu_tanh_f(v[c]);
                } else if (EPI == EPI_BIAS_SILU) {
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = v[c] / (1.0f + __expf(-v[c]));
                } else if (EPI == EPI_GATE_RESID) {
                    const float4 g4 = four(epi.gate + (long long)(m / rpb) * epi.gate_ld + n0);
                    const float4 r4 = four(epi.resid + idx);
                    v[0] = fmaf(g4.x, v[0], r4.x); v[1] = fmaf(g4.y, v[1], r4.y); v[2] = fmaf(g4.z, v[2], r4.z); v[3] = fmaf(g4.w, v[3], r4.w);
                } else if (EPI == EPI_BIAS_ROWADD) {
                    const float4 t4 = four(epi.table + (long long)(m % rpb) * epi.gate_ld + n0);
                    v[0] += t4.x; v[1] += t4.y; v[2] += t4.z; v[3] += t4.w;
                } else if (EPI == EPI_QKV_NORM && third_e < 2) {
                    qk_norm4(v, norm_w);
                }
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < valid) {
                        if (OUT_F32) reinterpret_cast<float*>(pr.out)[idx + c] = v[c];
                        else reinterpret_cast<bf16_t*>(pr.out)[idx + c] = f32_to_bf16(v[c]);
                    }
            }
    };

    fill_ring();
    k_loop();
    constexpr bool PAIR = WHOLE_ROWS && EPI == EPI_GATE_RESID && TM * TN <= 64 * 128;  // (see grouped_impl)
    if (PAIR && pr.then) {
        // The second layer of the same rows and columns (the two out-projections of a block with dual attention): its ring is filled behind
        // the last LDS reads of the first and lands while the first one's results are on their way out; a thread reads back what it wrote.
        const Prob& next = args.second;
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this thread's fragment reads are done; behind the barrier everyone's are
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        operands(next.A, next.Wp, next.tiled);
        request(pr);
        fill_ring();
        epilogue(pr);
        k_loop();
        wait_vmcnt<0>();
        request(next);
        epilogue(next);
        return;
    }
    request(pr);
    wait_vmcnt<0>();
    epilogue(pr);
}

template <int TM, int TN, int WM, int WN, int STAGES, int MW, int EPI, bool OUT_F32, bool WHOLE_ROWS = true>
int launch_ring(ProbSet& args, int n, hipStream_t st) {
    auto kern = gemm_bf16_ring_kernel<TM, TN, WM, WN, STAGES, MW, EPI, OUT_F32, WHOLE_ROWS>;
    constexpr int smem = STAGES * (TM + TN) * 128;
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(kern), smem));
    int total = 0;
    for (int i = 0; i < MAX_PROBS; i++) {
        if (i < n) total += ((args.p[i].N + TN - 1) / TN) * ((args.p[i].M + TM - 1) / TM);
        args.end[i] = total;
    }
    const int cus = compute_units();
    if (cus <= 0) return SD3_ERR_HIP;
    args.tiles_wgs = total;
    hipLaunchKernelGGL(kern, dim3(total + carried_wgs<ring_carries(EPI, OUT_F32, WHOLE_ROWS, MW)>(args, total, cus, smem)), dim3(WM * WN * 64), smem, st, args);
    g_gemm_bf16_launches.fetch_add(1, std::memory_order_relaxed);
    return launch_status("gemm_bf16");
}

// The tile shapes of the bf16 GEMM, smallest first, and what an output tile costs its compute unit in microseconds: `fixed` + `per_k` for
// each K tile of 64. Fitted to launches with cold weights at K = 1536 and 6144, 333 to 4250 rows, N = 1536 .. 6144 (a constant for the
// first round, the same for all shapes, left out); what they stand for is the traffic of (tm + tn) * 128 bytes per K tile through one
// compute unit's load path and, from 128x128 on, the matrix instructions. 192x256 tiles (the persistent kernel's, like 256x256) save little
// per tile but are there for what is left of a round: q|k|v of 2 x 1024 + 154 rows, 162 or 234 tiles, 50.2 -> 46.0 us; 128x256 beside 256x128
// for rows that are not multiples of 256: mlp-1 of 1581 + 999 rows, 504 tiles instead of 528 in two rounds of 256, 73 -> 60 us.
// Where 128x64 and 64x128 are the same number of rounds the former is taken: out-projection and mlp-2 of 1024 + 154 rows 16.7 -> 15.8 and 44.4 ->
// 42.4 us; forwards of 24 x 40 patches -3.4 %, two of 256px -1.6 %, 512px +0.3 %. That is what its fixed cost says: 2.25 where the fit gives 2.3 for both.
struct TileShape {
    int tm, tn;
    double fixed, per_k;
};
enum { TILE_64, TILE_128_64, TILE_64_128, TILE_128, TILE_256_128, TILE_128_256, TILE_192_256, TILE_256, TILE_SHAPES };
constexpr TileShape tile_shapes[TILE_SHAPES] = {{64, 64, 1.3, 0.19},    {128, 64, 2.25, 0.285}, {64, 128, 2.3, 0.285},
                                                {128, 128, 7.3, 0.403}, {256, 128, 11.3, 0.59}, {128, 256, 11.5, 0.615},
                                                {192, 256, 6.0, 1.315}, {256, 256, 11.3, 1.28}};

long long tiles_of(const Prob& q, int shape) {
    const TileShape& t = tile_shapes[shape];
    return (long long)((q.M + t.tm - 1) / t.tm) * ((q.N + t.tn - 1) / t.tn);
}
double launch_cost(const ProbSet& set, int n, int shape, int cus) {
    long long tiles = 0, depth = 0;
    for (int i = 0; i < n; i++) {
        const long long c = tiles_of(set.p[i], shape);
        tiles += c;
        depth += c * (set.p[i].K / BK);
    }
    const TileShape& t = tile_shapes[shape];
    const long long rounds = (tiles + cus - 1) / cus;
    // The table is a first round's. A further round costs more the fuller it is, since its tiles share what feeds the compute units. 128x256
    // tiles in two rounds, measured over the table's figure (cold weights, K = 1536 and 6144, N = 1536 .. 6144, 512 .. 12288 rows): 0.89 .. 1.07 with the
    // second round 12 % full, 0.94 .. 1.16 with 48 to 69 %, 1.17 .. 1.23 with 85 to 97 % (504 tiles, mlp-1 of 2580 rows: 64.7 us, the table 52.5).
    // The factor is that of a nearly full round, so that beyond one round the shape is taken where it saves a round (504 tiles instead of 528 of
    // 256x128) and not for a few percent of the model. From three rounds on it measured 0.94 .. 1.14 and is overrated; there another shape was
    // always within 1 % of it (up to 12288 rows). 192x256 tiles: 1.02 .. 1.13 in two rounds at K = 1536 where there are more than 270 (0.94 at 336 of
    // mlp-1), 0.87 .. 0.91 at K = 6144, 0.95 .. 1.05 from three rounds on. Their factor matters only where 256x256 tiles take two rounds as
    // well: with 1, 12255 + 770 rows take them and the forward is 0.8 % slower.
    const double again = rounds == 1 ? 1.0 : shape == TILE_128_256 ? 1.25 : shape == TILE_192_256 ? 1.06 : 1.0;
    return again * (double)rounds * (t.fixed + t.per_k * ((double)depth / tiles));
}
// Rows that are not made of aligned groups of four columns go element by element. Of the ring kernel three shapes are built for them: with
// 256x256 tiles alone 333 x 1541 x 1536 took, gated, 69.7 us instead of 9.5 (1536 columns: 7.7), 4250 rows, plain, 41.9 instead of 28.3,
// and as a run-time branch in every shape the form cost the other rows 0.3 us a launch (the compiler merges parts of the two).
bool all_whole(const ProbSet& set, int n) {
    for (int i = 0; i < n; i++)
        if (!set.p[i].whole) return false;
    return true;
}
bool shape_takes(int shape, bool whole) {
    return whole || shape == TILE_64 || shape == TILE_128 || shape == TILE_256_128 || shape == TILE_192_256 || shape == TILE_256;
}

int cheapest_shape(const ProbSet& set, int n, int cus, double& cost) {
    const bool whole = all_whole(set, n);
    int best = TILE_256;
    cost = launch_cost(set, n, TILE_256, cus);
    for (int s = TILE_256 - 1; s >= 0; s--) {
        if (!shape_takes(s, whole)) continue;
        const double c = launch_cost(set, n, s, cus);
        if (c < cost) {
            best = s;
            cost = c;
        }
    }
    return best;
}

// Rings: as deep as one workgroup per compute unit allows where a launch is a single round; 64x64 tiles and, with more than one round, the
// next two shapes leave room for a second workgroup (mlp-2 of 1178 rows as 64x128 tiles: one round 45 against 49 us, two rounds of
// 2356 rows 90 against 81).
template <int EPI, bool OUT_F32>
int launch_shape(int shape, ProbSet& args, int n, int cus, hipStream_t st) {
    const bool whole = all_whole(args, n);
    if (!shape_takes(shape, whole)) shape = TILE_256;
    // Rows of more than 2^23 values: the next smaller tiles that can address them. (64-bit addresses are built for one shape only, which takes 64 ms for 3 x 68 x
    // (2^22 + 64) where 64x64 tiles take 12, and 90 ms for 1024 x 512 instead of 17.)
    auto fits = [&](int s) { return addresses(args, n, tile_shapes[s].tm > tile_shapes[s].tn ? tile_shapes[s].tm : tile_shapes[s].tn, 2); };
    while (shape > TILE_64 && !fits(shape)) shape--;
    if (!fits(shape)) return launch_cfg<128, 256, 1, 4, 2, EPI, OUT_F32, false, true>(args, n, st);
    long long tiles = 0;
    for (int i = 0; i < n; i++) tiles += tiles_of(args.p[i], shape);
    const bool one_round = tiles <= cus;
    if (!whole) {
        if (shape == TILE_64) return launch_ring<64, 64, 4, 1, 5, 2, EPI, OUT_F32, false>(args, n, st);
        if (shape == TILE_128) return launch_ring<128, 128, 4, 2, 4, 2, EPI, OUT_F32, false>(args, n, st);
        if (shape == TILE_256_128) return launch_ring<256, 128, 4, 2, 3, 2, EPI, OUT_F32, false>(args, n, st);
    }
    switch (shape) {
        case TILE_64: return launch_ring<64, 64, 4, 1, 5, 2, EPI, OUT_F32>(args, n, st);
        case TILE_128_64:
            if (one_round) return launch_ring<128, 64, 8, 1, 6, 2, EPI, OUT_F32>(args, n, st);
            return launch_ring<128, 64, 8, 1, 3, 4, EPI, OUT_F32>(args, n, st);
        case TILE_64_128:
            if (one_round) return launch_ring<64, 128, 4, 2, 6, 2, EPI, OUT_F32>(args, n, st);
            return launch_ring<64, 128, 4, 2, 3, 4, EPI, OUT_F32>(args, n, st);
        case TILE_128: return launch_ring<128, 128, 4, 2, 4, 2, EPI, OUT_F32>(args, n, st);
        case TILE_256_128: return launch_ring<256, 128, 4, 2, 3, 2, EPI, OUT_F32>(args, n, st);
        case TILE_128_256: return launch_ring<128, 256, 2, 4, 3, 2, EPI, OUT_F32>(args, n, st);
        case TILE_192_256: return launch_cfg<192, 256, 2, 4, 2, EPI, OUT_F32>(args, n, st);
        default: return launch_cfg<256, 256, 2, 4, 2, EPI, OUT_F32>(args, n, st);
    }
}

}  // namespace

std::atomic<long long> g_gemm_bf16_launches{0};
int g_gemm_bf16_row_split = 1;  // 0: never split a problem's rows over two launches (sd3_tune)
int g_gemm_bf16_tile = 0;       // 0: chosen from the sizes; else a forced tile shape (sd3_gemm_bf16_force_tile)

// the shape behind a value of sd3_gemm_bf16_force_tile (-1: none): 128 or 256 for those squares, else rows * 1000 + columns
static int forced_shape(int tile) {
    if (tile == 128 || tile == 256) tile *= 1001;
    for (int s = 0; s < TILE_SHAPES; s++)
        if (tile == tile_shapes[s].tm * 1000 + tile_shapes[s].tn) return s;
    return -1;
}
// whether rows are made of aligned groups of four columns, in the output and in what the epilogue reads
static bool whole_rows(const Prob& q, int epi) {
    auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (q.N % 4 || q.ldc % 4 || !al(q.out)) return false;
    if (epi == EPI_GATE_RESID) return al(q.epi.gate) && al(q.epi.resid) && q.epi.gate_ld % 4 == 0;
    if (epi == EPI_BIAS_ROWADD) return al(q.epi.table);
    return true;
}

// fp8 operands: 256x256 (one workgroup per compute unit) or 128x128 tiles (two), by rounds: measured on full rounds, a round of 128x128
// tiles takes 0.62 of one of 256x256 tiles, a launch of its own for problems with few rows about 0.38
static int fp8_launches(ProbSet& args, int m, int out_is_f32, int epi, int cus, hipStream_t st) {
    auto launch = [&](ProbSet& pp, int count, int v) -> int {
#define SD3_GEMM_FP8_LAUNCH(E) return out_is_f32 ? launch_epi_fp8<E, true>(v, pp, count, st) : launch_epi_fp8<E, false>(v, pp, count, st)
        switch (epi) {
            case EPI_BIAS: SD3_GEMM_FP8_LAUNCH(EPI_BIAS);
            case EPI_BIAS_GELU: SD3_GEMM_FP8_LAUNCH(EPI_BIAS_GELU);
            case EPI_GATE_RESID: SD3_GEMM_FP8_LAUNCH(EPI_GATE_RESID);
            case EPI_QKV_NORM: SD3_GEMM_FP8_LAUNCH(EPI_QKV_NORM);
            default: return fail(SD3_ERR_UNSUPPORTED, "gemm_fp8: epilogue %d is not built for fp8 operands", epi);
        }
#undef SD3_GEMM_FP8_LAUNCH
    };
    if (g_gemm_bf16_tile) return launch(args, m, g_gemm_bf16_tile == 256 ? 4 : 0);
    constexpr double ROUND128 = 0.62, SMALL_LAUNCH = 0.38;
    auto tiles = [](const Prob& q, int t) { return ((q.M + t - 1) / t) * ((q.N + t - 1) / t); };
    auto rounds = [](long long t, int slots) { return (double)((t + slots - 1) / slots); };
    ProbSet big{}, small{};
    int nb = 0, ns = 0;
    long long big256 = 0, big128 = 0, small256 = 0, small128 = 0;
    for (int i = 0; i < m; i++) {
        if (args.p[i].M < 1024) {
            small.p[ns++] = args.p[i];
            small256 += tiles(args.p[i], 256);
            small128 += tiles(args.p[i], 128);
        } else {
            big.p[nb++] = args.p[i];
            big256 += tiles(args.p[i], 256);
            big128 += tiles(args.p[i], 128);
        }
    }
    if (nb == 0) return launch(args, m, 0);
    const double together256 = rounds(big256 + small256, cus), together128 = ROUND128 * rounds(big128 + small128, 2 * cus);
    double best = together256 <= together128 ? together256 : together128;
    int plan = together256 <= together128 ? 0 : 1;  // 0/1: one launch with 256/128 tiles; 2/3: the small problems first, alone
    if (ns > 0) {
        const double apart256 = rounds(big256, cus) + SMALL_LAUNCH, apart128 = ROUND128 * rounds(big128, 2 * cus) + SMALL_LAUNCH;
        if (apart256 < best) { best = apart256; plan = 2; }
        if (apart128 < best) { best = apart128; plan = 3; }
    }
    if (plan >= 2) {
        SD3_TRY(launch(small, ns, 0));
        return launch(big, nb, plan == 2 ? 4 : 0);
    }
    return launch(args, m, plan == 0 ? 4 : 0);
}

static int grouped_impl(const GemmBf16Problem* probs, int n, int out_is_f32, int epi, bool fp8, hipStream_t st, AdaCarry* carry) {
    if (n < 1 || n > MAX_PROBS) return fail(SD3_ERR_INVALID_ARG, "gemm_bf16_grouped: 1 to %d problems (got %d)", MAX_PROBS, n);
    ProbSet args{};
    int m = 0;
    const GemmBf16Problem* then = nullptr;
    int chained = 0;
    auto fill = [&](const GemmBf16Problem& q, Prob& d) -> int {
        const int kmult = fp8 ? 128 : BK;  // one LDS row of a K tile is 128 bytes
        if (q.K <= 0 || (q.K % kmult) != 0) return fail(SD3_ERR_UNSUPPORTED, "gemm_%s: K=%d must be a positive multiple of %d", fp8 ? "fp8" : "bf16", q.K, kmult);
        if ((reinterpret_cast<uintptr_t>(q.A) & 15) || (reinterpret_cast<uintptr_t>(q.Wp) & 15))
            return fail(SD3_ERR_INVALID_ARG, "gemm_bf16: operands must be 16-byte aligned");
        d.A = q.A; d.Wp = q.Wp; d.out = q.out; d.ldc = q.ldc; d.M = q.M; d.N = q.N; d.K = q.K; d.tiled = q.w_tiled && !fp8;
        d.epi = EpiDev{fp8 ? q.ea.a_scale : nullptr, fp8 ? q.ea.w_scale : nullptr, q.ea.bias, q.ea.gate, q.ea.resid, q.ea.table, q.ea.gate_ld,
                       q.ea.rows_per_batch > 0 ? q.ea.rows_per_batch : 1};
        if (epi == EPI_BIAS_ROWADD) d.epi.gate_ld = q.N;
        if (epi == EPI_QKV_NORM) {
            if (q.N % 192 || !q.ea.gate || !q.ea.resid || (reinterpret_cast<uintptr_t>(q.ea.gate) & 15) || (reinterpret_cast<uintptr_t>(q.ea.resid) & 15))
                return fail(SD3_ERR_INVALID_ARG, "gemm_bf16: the fused qk-norm needs N = 3C with C a multiple of 64 and two aligned weight vectors");
            d.epi.gate_ld = q.N / 3;
        }
        d.whole = whole_rows(d, epi);
        return SD3_OK;
    };
    for (int i = 0; i < n; i++) {
        const GemmBf16Problem& q = probs[i];
        if (q.M <= 0 || q.N <= 0) continue;  // an empty problem simply contributes no tiles
        if (q.then) {
            if (then || fp8 || epi != EPI_GATE_RESID || q.then->M != q.M || q.then->N != q.N || q.then->K != q.K || q.then->out != q.out || q.then->ldc != q.ldc)
                return fail(SD3_ERR_INVALID_ARG, "gemm_bf16: a following layer needs the gated epilogue and its predecessor's sizes and output");
            then = q.then;
            chained = m;
        }
        SD3_TRY(fill(q, args.p[m++]));
    }
    if (m == 0) return SD3_OK;
    const int cus = compute_units();
    if (cus <= 0) return SD3_ERR_HIP;
    if (fp8) return fp8_launches(args, m, out_is_f32, epi, cus, st);
    auto launch_tiles = [&](ProbSet& pp, int count, int shape) -> int {
#define SD3_GEMM_BF16_LAUNCH(E) return out_is_f32 ? launch_shape<E, true>(shape, pp, count, cus, st) : launch_shape<E, false>(shape, pp, count, cus, st)
        switch (epi) {
            case EPI_BIAS: SD3_GEMM_BF16_LAUNCH(EPI_BIAS);
            case EPI_BIAS_GELU: SD3_GEMM_BF16_LAUNCH(EPI_BIAS_GELU);
            case EPI_BIAS_SILU: SD3_GEMM_BF16_LAUNCH(EPI_BIAS_SILU);
            case EPI_GATE_RESID: SD3_GEMM_BF16_LAUNCH(EPI_GATE_RESID);
            case EPI_BIAS_ROWADD: SD3_GEMM_BF16_LAUNCH(EPI_BIAS_ROWADD);
            case EPI_QKV_NORM: SD3_GEMM_BF16_LAUNCH(EPI_QKV_NORM);
            default: return fail(SD3_ERR_INVALID_ARG, "gemm_bf16: unknown epilogue %d", epi);
        }
#undef SD3_GEMM_BF16_LAUNCH
    };
    auto launch = [&](ProbSet& pp, int count, int shape) -> int {
        if (!carry) return launch_tiles(pp, count, shape);
        constexpr double START = 3.0;  // the constant of a first round that the cost table leaves out
        pp.ada = carry->work;
        pp.ada.count = carry->left();
        pp.ada_last = carry->last;
        pp.ahead = carry->ahead;
        pp.us = (float)(START + launch_cost(pp, count, shape, cus) * (pp.p[0].then ? 2 : 1));
        SD3_TRY(launch_tiles(pp, count, shape));
        carry->work.first += pp.ada.count;
        carry->ahead = Ahead{};  // (of the launches of a layer the first one reads)
        return SD3_OK;
    };
    if (then) {
        // Both layers in one launch where they are one round of small tiles, i.e. a launch's start and end are a good part of it: dual blocks
        // of 256 + 77, 1024 + 154 tokens 106.7 -> 105.3 us, forwards 2972 -> 2951, 4708 -> 4681 us. From 128x128 tiles on the second layer
        // does better in a launch (and tiles) of its own: 2048 + 308, 1581 + 999, 8192 + 308 rows, forwards 0.1, 0.6, 1 % slower together.
        // GAP: what a launch less saves, us. A launch of one tile behind another launch takes 2.7 to 3.5; the chained layer keeps some of that
        // (between its K loops lie a barrier and a filling of the ring). With 5 instead of 2, blocks with 308 to 999 context rows beside 512 to
        // 1344 latent ones were up to 1.1 % faster at widths 768 and 1536 and 0.8 % slower at 2432, the forwards the same.
        constexpr double GAP = 2.0;
        SD3_TRY(fill(*then, args.second));
        const bool whole = all_whole(args, m) && args.second.whole;
        int pair = -1;
        if (g_gemm_bf16_tile) {
            if (whole) pair = forced_shape(g_gemm_bf16_tile);  // (256x192 tiles, 192, have no shape of the table: two launches)
            if (pair > TILE_64_128) pair = -1;
        } else if (whole) {
            ProbSet second{};
            second.p[0] = args.second;
            double best, after;
            cheapest_shape(args, m, cus, best);
            cheapest_shape(second, 1, cus, after);
            best += GAP + after;
            for (int s : {TILE_64, TILE_128_64, TILE_64_128}) {
                long long tiles = 0;
                for (int i = 0; i < m; i++) tiles += tiles_of(args.p[i], s);
                const double c = 2 * (tile_shapes[s].fixed + tile_shapes[s].per_k * (args.second.K / BK));
                if (tiles <= cus && c < best) {
                    best = c;
                    pair = s;
                }
            }
        }
        if (pair >= 0) {
            args.p[chained].then = true;
            return launch(args, m, pair);
        }
        GemmBf16Problem rest[MAX_PROBS];
        for (int i = 0; i < n; i++) {
            rest[i] = probs[i];
            rest[i].then = nullptr;
        }
        SD3_TRY(grouped_impl(rest, n, out_is_f32, epi, false, st, carry));
        return grouped_impl(then, 1, out_is_f32, epi, false, st, carry);
    }
    if (g_gemm_bf16_tile == 192) {
        if (epi == EPI_QKV_NORM) return fail(SD3_ERR_UNSUPPORTED, "gemm_bf16: this tile shape cannot fuse the qk-norm");
#define SD3_GEMM_BF16_192(E) \
    case E: return out_is_f32 ? launch_cfg<256, 192, 2, 4, 2, E, true>(args, m, st) : launch_cfg<256, 192, 2, 4, 2, E, false>(args, m, st)
        switch (epi) {
            SD3_GEMM_BF16_192(EPI_BIAS);
            SD3_GEMM_BF16_192(EPI_BIAS_GELU);
            SD3_GEMM_BF16_192(EPI_BIAS_SILU);
            SD3_GEMM_BF16_192(EPI_GATE_RESID);
            SD3_GEMM_BF16_192(EPI_BIAS_ROWADD);
            default: return fail(SD3_ERR_INVALID_ARG, "gemm_bf16: unknown epilogue %d", epi);
        }
#undef SD3_GEMM_BF16_192
    }
    if (g_gemm_bf16_tile) return launch(args, m, forced_shape(g_gemm_bf16_tile));
    // One launch with the cheapest shape, or two: the many-row problems apart from the few-row ones (a launch of its own costs LAUNCH), or
    // full rounds of 256x256 tiles first and the last rows of the last many-row problem with the few-row problems behind them. The
    // latter only for epilogues that do not look at the row index (a row split would shift the batch boundaries).
    // LAUNCH, us: the 2.7 to 3.5 of a launch behind another and the part of a first round that the table leaves out. (With 3.5 the batch-1
    // forward of 1024 x 1024 pixels takes 12.80 instead of 12.72 ms, the others the same.)
    constexpr double LAUNCH = 5.0;
    double best;
    const int together = cheapest_shape(args, m, cus, best);
    ProbSet big{}, small{};
    int nb = 0, ns = 0;
    for (int i = 0; i < m; i++) {
        if (args.p[i].M < 1024) small.p[ns++] = args.p[i];
        else big.p[nb++] = args.p[i];
    }
    int apart_big = -1, apart_small = -1;
    if (nb > 0 && ns > 0) {
        double cb, cs;
        const int sb = cheapest_shape(big, nb, cus, cb), ss = cheapest_shape(small, ns, cus, cs);
        if (cb + cs + LAUNCH < best) {
            best = cb + cs + LAUNCH;
            apart_big = sb;
            apart_small = ss;
        }
    }
    if (g_gemm_bf16_row_split && nb >= 1 && nb + ns <= MAX_PROBS &&
        (epi == EPI_BIAS || epi == EPI_BIAS_GELU || epi == EPI_BIAS_SILU || epi == EPI_QKV_NORM)) {
        const Prob& q = big.p[nb - 1];
        long long before = 0, all = 0;  // 256x256 tiles of the many-row problems in front of the one that is split, and of all of them
        for (int i = 0; i < nb; i++) {
            if (i + 1 < nb) before += tiles_of(big.p[i], TILE_256);
            all += tiles_of(big.p[i], TILE_256);
        }
        const int tn = (q.N + 255) / 256, tm = (q.M + 255) / 256;
        const long long avail = all / cus * cus - before;
        const int m1 = avail > 0 ? (int)(avail / tn) : 0;  // row tiles of q that fit the full rounds
        if (m1 > 0 && m1 < tm) {
            Prob head = q, tail = q;
            head.M = m1 * 256;
            tail.M = q.M - head.M;
            tail.A = q.A + (long long)head.M * q.K;
            tail.out = (char*)q.out + (long long)head.M * q.ldc * (out_is_f32 ? 4 : 2);
            ProbSet first{}, second{};
            for (int i = 0; i + 1 < nb; i++) first.p[i] = big.p[i];
            first.p[nb - 1] = head;
            second.p[0] = tail;
            for (int i = 0; i < ns; i++) second.p[1 + i] = small.p[i];
            double c2;
            const int s2 = cheapest_shape(second, 1 + ns, cus, c2);
            if (launch_cost(first, nb, TILE_256, cus) + c2 + LAUNCH < best) {
                SD3_TRY(launch(first, nb, TILE_256));
                return launch(second, 1 + ns, s2);
            }
        }
    }
    if (apart_big >= 0) {
        SD3_TRY(launch(small, ns, apart_small));
        return launch(big, nb, apart_big);
    }
    return launch(args, m, together);
}

int gemm_bf16_grouped(const GemmBf16Problem* probs, int n, int out_is_f32, int epi, hipStream_t st, AdaCarry* carry) {
    return grouped_impl(probs, n, out_is_f32, epi, false, st, carry);
}
int gemm_fp8_grouped(const GemmBf16Problem* probs, int n, int out_is_f32, int epi, hipStream_t st) { return grouped_impl(probs, n, out_is_f32, epi, true, st, nullptr); }

int gemm_bf16(const bf16_t* A, const bf16_t* Wp, bool w_tiled, void* out, int out_is_f32, int ldc, int M, int N, int K, int epi, const GemmEpilogueArgs& ea,
              hipStream_t st) {
    GemmBf16Problem q{A, Wp, out, ldc, M, N, K, ea, w_tiled};
    return gemm_bf16_grouped(&q, 1, out_is_f32, epi, st);
}

}  // namespace sd3

extern "C" int sd3_gemm_bf16_force_tile(int tile) {
    if (tile != 0 && tile != 192 && sd3::forced_shape(tile) < 0)
        return sd3::fail(SD3_ERR_INVALID_ARG, "sd3_gemm_bf16_force_tile: tile must be 0, 128, 192, 256, 64064, 64128, 128064, 256128, 128256 or 192256 (got %d)", tile);
    sd3::g_gemm_bf16_tile = tile;
    return SD3_OK;
}
