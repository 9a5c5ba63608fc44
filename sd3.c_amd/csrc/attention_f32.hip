// fp32 multi-head attention on the fp32 matrix cores, for the fp32 parity path and the attention operator.
// Replaces multihead_attention (modules.cpp:766-831) and, through its two-segment addressing, the token
// concatenation / split around it (modules.cpp:1427-1432): keys/values/queries of the joint sequence are read
// straight from the context buffers (first T[0] tokens) and the latent buffers (next T[1] tokens).
//
// Three kernels: attn_f32_split_kernel (fp32 matrix instruction) for head_dim 64 and 128 with 16-byte aligned rows, attn_f32_pieces_kernel (values as three bf16
// pieces each, on the bf16 matrix instruction) for head_dim 64 where there are many queries and heads, attn_f32_kernel for any other head_dim up to 128. Formulation of
// all: everything is kept transposed so that the probabilities never leave registers.
//   S^T (keys x queries) = K . Q^T      -> C-layout: a lane owns ONE query column and 16 keys per 32-key block
//   O^T (d x queries)   += V^T . P^T    -> the lane's own S^T registers are exactly the P^T operand it must supply
// Online softmax statistics are per query = per lane (plus one exchange with lane^32).
#include <type_traits>

#include "common.hpp"
#include "pieces.hpp"

namespace sd3 {
namespace {

constexpr int BQ = 128;   // queries per workgroup (4 wavefronts x 32)

struct SegDev {
    const float* q[2];
    const float* k[2];
    const float* v[2];
    float* out[2];
    int ld_qkv[2];
    int ld_out[2];
    int T[2];   // keys/values per batch element in each segment
    int Tq[2];  // queries per batch element in each segment
    int B;
};
// Four values of an output row, from column `col` on. PIECES: AttnSegments::out_pieces
template <bool PIECES>
__device__ __forceinline__ void put_output(const SegDev& s, int seg, long long row, int col, const f32x4_t& v) {
    if constexpr (PIECES) put_pieces<4>(PieceMatrix(s.out[seg], (long long)s.B * s.Tq[seg], s.ld_out[seg]), row, col, {v[0], v[1], v[2], v[3]});
    else *reinterpret_cast<f32x4_t*>(s.out[seg] + row * s.ld_out[seg] + col) = v;
}

template <int HSP, bool VEC>
__global__ void __launch_bounds__(256) attn_f32_kernel(SegDev s, int HS, float scale) {
    constexpr int KP = HSP + 1;
    constexpr int BKV = (HSP == 128) ? 32 : 64;  // keys per LDS tile (both tiles must fit 64 KiB of static LDS)
    constexpr int NKB = BKV / 32;
    __shared__ float Ks[BKV * KP];
    __shared__ float Vs[BKV * HSP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, lk = lane >> 5;
    const int h = blockIdx.y, b = blockIdx.z;
    const int T0 = s.T[0], T = s.T[0] + s.T[1];
    const int Tq0 = s.Tq[0], TQ = s.Tq[0] + s.Tq[1];

    // ---- this lane's query row (as the B operand of S^T = K.Q^T: element [d = 2*kk + lk][q = l32]) ----
    const int qt = blockIdx.x * BQ + wave * 32 + l32;
    float qreg[HSP / 2];
    {
        const int seg = (qt < Tq0) ? 0 : 1;
        const int tl = seg ? qt - Tq0 : qt;
        const float* qp = s.q[seg] + ((long long)b * s.Tq[seg] + tl) * s.ld_qkv[seg] + (long long)h * HS;
#pragma unroll
        for (int kk = 0; kk < HSP / 2; kk++) {
            const int d = 2 * kk + lk;
            qreg[kk] = (qt < TQ && d < HS) ? qp[d] * scale : 0.f;
        }
    }

    f32x16_t oacc[HSP / 32];
#pragma unroll
    for (int i = 0; i < HSP / 32; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.f;
    float m_run = -1e30f, l_run = 0.f;  // l_run: partial sum over the keys this lane owns

    for (int t0 = 0; t0 < T; t0 += BKV) {
        __syncthreads();  // previous tile fully consumed
        // ---- stage K and V rows t0..t0+BKV-1 of head h (zero beyond T or beyond HS) ----
        if (VEC) {
            constexpr int VPR = HSP / 4;  // float4 per row
            for (int e = tid; e < BKV * VPR; e += 256) {
                const int row = e / VPR, dv = (e % VPR) * 4;
                const int t = t0 + row;
                float4 kv = make_float4(0.f, 0.f, 0.f, 0.f), vv = kv;
                if (t < T && dv < HS) {
                    const int seg = (t < T0) ? 0 : 1;
                    const long long off = ((long long)b * s.T[seg] + (seg ? t - T0 : t)) * s.ld_qkv[seg] + (long long)h * HS + dv;
                    kv = *reinterpret_cast<const float4*>(s.k[seg] + off);
                    vv = *reinterpret_cast<const float4*>(s.v[seg] + off);
                }
                float* kd = &Ks[row * KP + dv];
                kd[0] = kv.x; kd[1] = kv.y; kd[2] = kv.z; kd[3] = kv.w;
                *reinterpret_cast<float4*>(&Vs[row * HSP + dv]) = vv;
            }
        } else {
            for (int e = tid; e < BKV * HSP; e += 256) {
                const int row = e / HSP, d = e % HSP;
                const int t = t0 + row;
                float kv = 0.f, vv = 0.f;
                if (t < T && d < HS) {
                    const int seg = (t < T0) ? 0 : 1;
                    const long long off = ((long long)b * s.T[seg] + (seg ? t - T0 : t)) * s.ld_qkv[seg] + (long long)h * HS + d;
                    kv = s.k[seg][off];
                    vv = s.v[seg][off];
                }
                Ks[row * KP + d] = kv;
                Vs[row * HSP + d] = vv;
            }
        }
        __syncthreads();

        // ---- S^T for the 32-key blocks of the tile ----
        f32x16_t sacc[NKB];
#pragma unroll
        for (int kb = 0; kb < NKB; kb++) {
#pragma unroll
            for (int r = 0; r < 16; r++) sacc[kb][r] = 0.f;
#pragma unroll
            for (int kk = 0; kk < HSP / 2; kk++) {
                const float a = Ks[(kb * 32 + l32) * KP + 2 * kk + lk];
                sacc[kb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, qreg[kk], sacc[kb], 0, 0, 0);
            }
        }
        // lane holds keys  t0 + kb*32 + 8*(r/4) + 4*lk + (r%4)  of query column l32
        float tmax = -1e30f;
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = t0 + kb * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
                if (key >= T) sacc[kb][r] = -1e30f;
                tmax = fmaxf(tmax, sacc[kb][r]);
            }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = expf(m_run - m_new);
        m_run = m_new;
        float psum = 0.f;
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float p = expf(sacc[kb][r] - m_new);
                sacc[kb][r] = p;
                psum += p;
            }
        l_run = l_run * alpha + psum;
#pragma unroll
        for (int i = 0; i < HSP / 32; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;

        // ---- O^T += V^T . P^T : step r of block kb contracts key (8*(r/4) + 4*lk + r%4) of each lane half ----
#pragma unroll
        for (int kb = 0; kb < NKB; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int key = kb * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
#pragma unroll
                for (int i = 0; i < HSP / 32; i++) {
                    const float a = Vs[key * HSP + i * 32 + l32];
                    oacc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, sacc[kb][r], oacc[i], 0, 0, 0);
                }
            }
    }

    // ---- normalise and store: lane owns query qt, rows d = i*32 + 8*(r/4) + 4*lk + r%4 ----
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    if (qt < TQ) {
        const int seg = (qt < Tq0) ? 0 : 1;
        if (s.out[seg]) {
            const int tl = seg ? qt - Tq0 : qt;
            float* op = s.out[seg] + ((long long)b * s.Tq[seg] + tl) * s.ld_out[seg] + (long long)h * HS;
            const float inv = 1.0f / l_tot;
#pragma unroll
            for (int i = 0; i < HSP / 32; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int d = i * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
                    if (d < HS) op[d] = oacc[i][r] * inv;
                }
        }
    }
}

// The largest of the values of the lanes l%16
__device__ __forceinline__ float max_of_groups(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// ---- head_dim 64 and 128 ----
// The matrix unit (v_mfma_f32_16x16x4_f32: 64 FLOP per cycle and SIMD) is the bound, and everything it needs fits the registers of one
// wavefront: 16*QB queries and 16*KB keys at a time. So no LDS tiles and no barriers: the KS wavefronts of a workgroup share its queries
// and split the KEYS (tile t goes to wavefront t % KS); K and V rows come straight from memory (L2: all workgroups of a head run on one
// XCD) into registers, half a tile of matrix work ahead of their use; the KS partial results are merged in a fixed tree at the end.
// This gives every SIMD work also where there are few queries: 1178 tokens and 2 heads are 20 workgroups of 128 queries with the keys in
// one run (290 us), 592 wavefronts this way (28 us). 2 x 24 heads of 64, 1178 tokens (which go by pieces now): 244 -> 148 us, 70 -> 115 TFLOP/s of 155 (the matrix
// instructions alone about 127, the softmax 12, the loads 9).
//
// Contraction order: K and Q are read as float4 along d, so step s of 16-wide chunk c contracts d = 16c + 4g + s over the lane groups
// g = l/16. S^T registers r of a 16x16 block are keys 4g + r of query l%16: as they are, the operand of step r of O^T += V^T P^T, whose
// V rows 4g + r are read as float4 along d: block j of the four takes d = 4(l%16) + j, so a lane ends with 16 consecutive d of its query.
// LONG_ROWS: rows are 2^22 floats or more apart (and less than 2^24): four times the stride does not fit the 24-bit product of the row offsets. An
// instantiation of its own, since the shift behind the product, done in every case, costs the others up to 2 %. 65536 heads of 64, 2 queries, 40 keys:
// 691 us, with attn_f32_kernel 2204.
template <int HS, int QB, int KB, int KS, bool LONG_ROWS, bool PIECES>
__global__ void __launch_bounds__(KS * 64, 2) attn_f32_split_kernel(SegDev s, int NH, int n_q, int total, float scale) {
    constexpr int NC = HS / 16, NU = HS / 64, TKEYS = 16 * KB, QW = 16 * QB;
    constexpr int PITCH = NU * 16 * QB + 2 * QB;  // floats per lane in the merge buffer
    __shared__ float merge[(KS / 2) * 64 * PITCH];
    const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // consecutive workgroup ids go to the 8 XCDs in turn: every XCD gets a contiguous run of (batch, head, query tile)
    const int xcd = blockIdx.x % 8, local = blockIdx.x / 8, per = (total + 7) / 8, tall = (total % 8) ? (total % 8) : 8;
    const int item = xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
    const int bh = item / n_q, h = bh % NH, b = bh / NH, q0 = (item % n_q) * QW;
    const int T0 = s.T[0], T1 = s.T[1], Tq0 = s.Tq[0], TQ = s.Tq[0] + s.Tq[1];

    f32x4_t q[QB][NC];
#pragma unroll
    for (int i = 0; i < QB; i++) {
        const int qt = min(q0 + 16 * i + lr, TQ - 1), seg = qt < Tq0 ? 0 : 1;  // (queries past the end repeat the last one and are not stored)
        const float* p = s.q[seg] + ((long long)b * s.Tq[seg] + (seg ? qt - Tq0 : qt)) * s.ld_qkv[seg] + h * HS + 4 * lg;
#pragma unroll
        for (int c = 0; c < NC; c++) q[i][c] = *reinterpret_cast<const f32x4_t*>(p + 16 * c) * scale;
    }
    f32x4_t o[QB][NU][4];
    float m_run[QB], l_run[QB];  // l_run: over the keys of this lane
#pragma unroll
    for (int i = 0; i < QB; i++) {
        m_run[i] = -1e30f;
        l_run[i] = 0.f;
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int j = 0; j < 4; j++) o[i][u][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // Key tiles are counted segment by segment (the last one of a segment may be partly empty), so that a tile's rows have one scalar
    // base and 32-bit offsets.
    const int nt0 = (T0 + TKEYS - 1) / TKEYS, n_t = nt0 + (s.T[1] + TKEYS - 1) / TKEYS;
    const int ld0 = s.ld_qkv[0], ld1 = s.ld_qkv[1];
    const float* k0 = s.k[0] + (long long)b * T0 * ld0 + h * HS;
    const float* k1 = s.k[1] + (long long)b * s.T[1] * ld1 + h * HS;
    const float* v0 = s.v[0] + (long long)b * T0 * ld0 + h * HS;
    const float* v1 = s.v[1] + (long long)b * s.T[1] * ld1 + h * HS;
    f32x4_t k[KB][NC], v[KB][4][NU];
    auto keys_of = [&](int t, int& seg, int& t0) {  // tile t: its segment, its first key in it
        seg = t < nt0 ? 0 : 1;
        t0 = (seg ? t - nt0 : t) * TKEYS;
        return (seg ? T1 : T0) - t0;  // keys from here to the end of the segment
    };
    // Where a lane's chunks of a tile's rows are: a scalar base and 32-bit row offsets in bytes, which the loads take as they are (as 64-bit addresses,
    // both before the last tile had a form of its own: 24 heads of 64, 1178 tokens, batch 2 160 us instead of 152, 4250 tokens 967 instead of 916; 2 heads
    // of 128, batch 8 138 instead of 127; calls of few keys 1 to 2 % less). The chunks are requested one by one, each right behind the last use of the
    // register it goes to, so that the requests are spread over the matrix work of a whole tile.
    auto row_at = [](int row, int ld) { return LONG_ROWS ? __umul24(row, ld) * 4u : (unsigned)__umul24(row, 4 * ld); };
    struct Rows {
        const char* base;
        unsigned off[4 * KB];  // bytes
    };
    auto k_rows = [&](int t, Rows& w) {
        int seg, t0;
        const int left = keys_of(t, seg, t0), ld = seg ? ld1 : ld0;
        w.base = reinterpret_cast<const char*>((seg ? k1 : k0) + (long long)t0 * ld);
#pragma unroll
        for (int kb = 0; kb < KB; kb++) w.off[kb] = row_at(min(16 * kb + lr, left - 1), ld) + 16 * lg;
    };
    auto v_rows = [&](int t, Rows& w) {
        int seg, t0;
        const int left = keys_of(t, seg, t0), ld = seg ? ld1 : ld0;
        w.base = reinterpret_cast<const char*>((seg ? v1 : v0) + (long long)t0 * ld);
#pragma unroll
        for (int x = 0; x < 4 * KB; x++) w.off[x] = row_at(min(16 * (x / 4) + 4 * lg + x % 4, left - 1), ld) + 16 * lr;
    };
    auto load_k = [&](const Rows& w, int c) {
#pragma unroll
        for (int kb = 0; kb < KB; kb++) k[kb][c] = *reinterpret_cast<const f32x4_t*>(w.base + w.off[kb] + 64 * c);
    };
    auto load_v = [&](const Rows& w, int x) {
#pragma unroll
        for (int u = 0; u < NU; u++) v[x / 4][x % 4][u] = *reinterpret_cast<const f32x4_t*>(w.base + w.off[x] + 256 * u);
    };
    constexpr int VECTOR_ONLY = 0x486;  // what may cross: vector, scalar and transcendental instructions and LDS exchanges

    f32x4_t sc[KB][QB], sn[KB][QB];  // scores of the current and of the next tile
    auto scores = [&](f32x4_t (&x)[KB][QB], const Rows& w) {  // (and requests the K chunks of the tile after)
#pragma unroll
        for (int kb = 0; kb < KB; kb++)
#pragma unroll
            for (int i = 0; i < QB; i++) x[kb][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; c++) {
#pragma unroll
            for (int st = 0; st < 4; st++)
#pragma unroll
                for (int kb = 0; kb < KB; kb++)
#pragma unroll
                    for (int i = 0; i < QB; i++) x[kb][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[kb][c][st], q[i][c][st], x[kb][i], 0, 0, 0);
            load_k(w, c);
            __builtin_amdgcn_sched_barrier(VECTOR_ONLY);
        }
    };
    int t = wave;
    if (t < n_t) {
        Rows w;
        k_rows(t, w);
#pragma unroll
        for (int c = 0; c < NC; c++) load_k(w, c);
        v_rows(t, w);
#pragma unroll
        for (int x = 0; x < 4 * KB; x++) load_v(w, x);
        k_rows(t + KS < n_t ? t + KS : t, w);
        scores(sc, w);
    }
    // One key tile. MORE: this wavefront has another one behind it. Its last tile asks for no rows and computes no scores of a next one, which is most of what
    // calls of few keys do: with them 4250 queries of 64 keys, 24 heads of 64, take 46.2 us instead of 38.5; 4 x 1024 of 154, 12 heads of 128 64.2 (1.1 %
    // more than with 64-bit addresses) instead of 59.1; 2 x 1178 of 1178, 24 heads 150.8 instead of 148.0.
    auto tile = [&](auto more) {
        constexpr bool MORE = decltype(more)::value;
        const int next = t + KS, next2 = t + 2 * KS < n_t ? t + 2 * KS : t;  // (past the end: any tile, never used)
        int seg, t0;
        const int left = keys_of(t, seg, t0);
        if (left < TKEYS) {
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (16 * kb + 4 * lg + r >= left)
#pragma unroll
                        for (int i = 0; i < QB; i++) sc[kb][i][r] = -1e30f;
        }
        // the scores of the next tile on the matrix unit beside the softmax of this one on the vector unit (wavefronts of a SIMD fall
        // into step, so one of them does not fill the other's pauses)
        Rows wk, wv;
        if constexpr (MORE) {
            k_rows(next2, wk);
            v_rows(next, wv);
            scores(sn, wk);
        }
#pragma unroll
        for (int i = 0; i < QB; i++) {
            float mx = sc[0][i][0];
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) mx = fmaxf(mx, sc[kb][i][r]);
            mx = max_of_groups(mx);
            // The reference moves only where a score exceeds it by 2^8: in the first tile and hardly ever again. With the largest score itself, and shuffles through LDS to
            // find it, 2 heads of 128, 1178 tokens took 29.4 us instead of 28.0, 128 queries of 1000 keys, 24 heads of 64 15.6 instead of 15.1.
            const bool moves = mx > m_run[i] + 8.f;
            if (__builtin_amdgcn_ballot_w64(moves)) {
                const float m = moves ? mx : m_run[i], alpha = __builtin_amdgcn_exp2f(m_run[i] - m);
                m_run[i] = m;
                l_run[i] *= alpha;
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++) o[i][u][j] *= alpha;
            }
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = __builtin_amdgcn_exp2f(sc[kb][i][r] - m_run[i]);
                    sc[kb][i][r] = p;
                    l_run[i] += p;
                }
        }
#pragma unroll
        for (int x = 0; x < 4 * KB; x++) {
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int i = 0; i < QB; i++) o[i][u][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x / 4][x % 4][u][j], sc[x / 4][i][x % 4], o[i][u][j], 0, 0, 0);
            if constexpr (MORE) load_v(wv, x);
            __builtin_amdgcn_sched_barrier(VECTOR_ONLY);
        }
        if constexpr (MORE)
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int i = 0; i < QB; i++) sc[kb][i] = sn[kb][i];
    };
    for (; t + KS < n_t; t += KS) tile(std::true_type());
    if (t < n_t) tile(std::false_type());

    // merge: in each step the upper half of the wavefronts hands its state to the lower half
#pragma unroll
    for (int half = KS / 2; half >= 1; half /= 2) {
        float* mine = merge + ((wave < half ? wave : wave - half) * 64 + lane) * PITCH;
        __syncthreads();
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int i = 0; i < QB; i++) {
                mine[2 * i] = m_run[i];
                mine[2 * i + 1] = l_run[i];
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++) mine[2 * QB + ((i * NU + u) * 4 + j) * 4 + r] = o[i][u][j][r];
            }
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int i = 0; i < QB; i++) {
                const float om = mine[2 * i], mx = fmaxf(m_run[i], om);
                const float wa = __builtin_amdgcn_exp2f(m_run[i] - mx), wb = __builtin_amdgcn_exp2f(om - mx);  // (a wavefront that had no tile: its factor is 0)
                m_run[i] = mx;
                l_run[i] = l_run[i] * wa + mine[2 * i + 1] * wb;
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int r = 0; r < 4; r++) o[i][u][j][r] = o[i][u][j][r] * wa + mine[2 * QB + ((i * NU + u) * 4 + j) * 4 + r] * wb;
            }
        }
    }
    if (wave) return;
#pragma unroll
    for (int i = 0; i < QB; i++) {
        const int qt = q0 + 16 * i + lr, seg = qt < Tq0 ? 0 : 1;
        float l = l_run[i] + __shfl_xor(l_run[i], 16, 64);
        l += __shfl_xor(l, 32, 64);
        if (qt >= TQ || !s.out[seg]) continue;
        const float inv = 1.0f / l;
        const long long row = (long long)b * s.Tq[seg] + (seg ? qt - Tq0 : qt);
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                put_output<PIECES>(s, seg, row, h * HS + 16 * lg + 64 * u + 4 * r,
                           f32x4_t{o[i][u][0][r] * inv, o[i][u][1][r] * inv, o[i][u][2][r] * inv, o[i][u][3][r] * inv});
    }
}

template <int HS, int QB, int KB, int KS, bool LONG_ROWS, bool PIECES>
int launch_split_as(const SegDev& s, int B, int NH, float scale, hipStream_t st) {
    const int TQ = s.Tq[0] + s.Tq[1], n_q = (TQ + 16 * QB - 1) / (16 * QB);
    const long long total = (long long)B * NH * n_q;
    if (total > 0x7fffffff) return fail(SD3_ERR_UNSUPPORTED, "attention (fp32): too many work items");
    hipLaunchKernelGGL((attn_f32_split_kernel<HS, QB, KB, KS, LONG_ROWS, PIECES>), dim3((unsigned)total), dim3(KS * 64), 0, st, s, NH, n_q, (int)total, scale);
    return launch_status("attention_f32");
}

template <int HS, int QB, int KB, int KS>
int launch_split(const SegDev& s, int B, int NH, float scale, bool pieces, hipStream_t st) {
    return pieces ? launch_split_as<HS, QB, KB, KS, false, true>(s, B, NH, scale, st) : launch_split_as<HS, QB, KB, KS, false, false>(s, B, NH, scale, st);
}

// ---- head_dim 64 by bf16 pieces ----
// Products as in gemm_f32_pieces_kernel: an fp32 value is the sum of three bf16 values without a remainder (bf16_pieces), six of the nine products of pieces are formed. No
// value is lost beside a larger one of its head, channel or token. Probabilities are split as they are: those below 2^-110 keep the bits down to 2^-133, and an exponential
// below 2^-126 is 0 in any case (times 2^16 first: 2 x 1178 tokens 109 -> 112 us, the same error where a result is made of weights of 2^-118). Scores, probabilities, their
// sums and the outputs are fp32 throughout. Two sums per score, of the products of first pieces and of the others, because the matrix instruction does not round to
// nearest; the products of a key tile are summed by themselves before they join the outputs, one rounding per tile. Relative error against 64 bits, 24 heads of 64 (fp32
// instruction): 32 keys 1.1e-7 (2.3e-7), 77 1.3e-7 (2.7e-7), 1178 1.8e-7 (4.3e-7), 4250 2.4e-7 (6.6e-7); equal weights, 77 keys 7.7e-8 (1.1e-7), constant values 7.0e-8
// (7.9e-8). (Two f16 pieces per value and three products took 68 us for 2 x 1178 tokens, 24 heads, but hold 22 of the 24 bits, and only of values within 2^-7 of the
// largest of the head: with one channel of V 2^16 times the others these came out with an error of 4e-5, beside a key that takes 1 - 2^-20 of the weight 7e-5. One sum per
// score 104 us instead of 108, and up to 1.25 times the fp32 instruction's error where a score is one large product.)
// Results that are not finite (infinities, NaNs, values from 2^112 and sums from 2^96 on) are formed anew on the fp32 instruction (attend_in_f32), 32 queries at a time: 2 x 1178
// tokens, 24 heads, 108 us, with one such query 200, with one such head 260, with 24 of the 48 380. (A score of -2^96 and below counts as minus infinity: its rounding error in
// fp32 is 2^72.)
//
// A wavefront has 32 queries; QG of them share the K and V tiles, which each splits a share of, into LDS. Per tile of 32 keys a wavefront issues 48 matrix instructions
// (1536 cycles) and 370 vector operations (about 1400), and the two hardly overlap however they are interleaved: the vector unit gets few slots beside matrix
// instructions, which is also why these are the ones of 32 cycles and not of 16. So vector operations count: a reference that moves only past a margin, offsets that stay from
// tile to tile.
// The keys are two runs, even and odd tiles, with a reference and sums of their own, merged at the end: half the additions to one sum, and few queries get twice the
// wavefronts. KR = 2: side by side; SEQ = 2: one after the other, with the same bits.
// us, fp32 instruction -> pieces, 24 heads: 2 x 1178 tokens 145 -> 108 (158 TFLOP/s, 950 of products of pieces), 4250 tokens 901 -> 695, 8 x 512 tokens 114 -> 81, 3 x 860
// 121 -> 85, one element of 1178 85 -> 57.
// head_dim 128 has no registers for the pieces of its queries beside a second wavefront: with one per SIMD 12 heads, 1178 tokens 84 -> 83, two of these 159 -> 121, but 3 x 1000
// tokens 173 -> 206, 666 tokens 30 -> 52. It stays on the fp32 instruction.
// What the pieces cannot give (values beyond their range, infinities, NaNs): the lane's query `qt`, all lanes 32 of them, over all keys on the fp32
// matrix instruction; row: where the query's result goes in its segment (-1: not stored). For the rare case, so as plain as can be.
template <bool PIECES>
__device__ void attend_in_f32(const SegDev& s, int b, int h, int qt, float scale, long long row) {
    constexpr int HS = 64;
    const int l32 = threadIdx.x & 31, lk = threadIdx.x >> 5 & 1;
    const int qseg = qt < s.Tq[0] ? 0 : 1;
    const float* q = s.q[qseg] + ((long long)b * s.Tq[qseg] + (qseg ? qt - s.Tq[0] : qt)) * s.ld_qkv[qseg] + h * HS + lk;
    float m = -1e30f, l = 0.f;
    f32x16_t o[HS / 32];
#pragma unroll
    for (int j = 0; j < HS / 32; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = 0.f;
    for (int seg = 0; seg < 2; seg++)
        for (int t0 = 0; t0 < s.T[seg]; t0 += 32) {
            const int last = s.T[seg] - 1;
            const long long ld = s.ld_qkv[seg], first = (long long)b * s.T[seg];
            const float* k = s.k[seg] + (first + min(t0 + l32, last)) * ld + h * HS + lk;
            f32x16_t x;
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = 0.f;
            for (int d = 0; d < HS; d += 2) x = __builtin_amdgcn_mfma_f32_32x32x2f32(k[d], q[d] * scale, x, 0, 0, 0);
            float mx = m;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (t0 + 8 * (r >> 2) + 4 * lk + (r & 3) > last) x[r] = -1e30f;
                mx = fmaxf(mx, x[r]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float alpha = __builtin_amdgcn_exp2f(m - mx);
            m = mx;
            l *= alpha;
#pragma unroll
            for (int j = 0; j < HS / 32; j++) o[j] *= alpha;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float p = __builtin_amdgcn_exp2f(x[r] - mx);
                l += p;
                const float* v = s.v[seg] + (first + min(t0 + 8 * (r >> 2) + 4 * lk + (r & 3), last)) * ld + h * HS + l32;
#pragma unroll
                for (int j = 0; j < HS / 32; j++) o[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[32 * j], p, o[j], 0, 0, 0);
            }
        }
    const float inv = 1.0f / (l + __shfl_xor(l, 32, 64));
    if (row >= 0)
#pragma unroll
        for (int j = 0; j < HS / 32; j++)
#pragma unroll
            for (int r = 0; r < 16; r += 4)
                put_output<PIECES>(s, qseg, row, h * HS + 4 * lk + 32 * j + 2 * r, f32x4_t{o[j][r] * inv, o[j][r + 1] * inv, o[j][r + 2] * inv, o[j][r + 3] * inv});
}

// The split of eight values into pieces (bf16_pieces) in steps, to be spread over matrix instructions
struct Split {
    static constexpr int STEPS = 5;
    float x[8];
    uint32_t piece[3][4];
    __device__ __forceinline__ void step(int n) {
        if (n % 2 == 0) bf16_high<8>(x, piece[n / 2]);
        else bf16_rest<8, false>(x, piece[n / 2]);
    }
};

template <int QG, int KR, int SEQ>
struct PiecesShape {
    static constexpr int HS = 64, QWG = 32 * QG, THREADS = QG * KR * 64;
    static constexpr int K_PLANE = 32 * 64, V_PLANE = HS * 64;  // bytes: 32 k values of 32 keys; 32 keys of HS values
    static constexpr int K_BYTES = HS / 32 * 3 * K_PLANE, V_BYTES = 3 * V_PLANE, RUN_BYTES = K_BYTES + 2 * V_BYTES;
    static constexpr int PITCH = HS / 2 + 4;                    // floats per lane of a run's result
    static constexpr int MERGE_BYTES = KR / 2 * QG * 64 * PITCH * 4, KEPT_BYTES = SEQ > 1 ? QG * 64 * PITCH * 4 : 0;
    static constexpr int LDS = (KR * RUN_BYTES > MERGE_BYTES ? KR * RUN_BYTES : MERGE_BYTES) + KEPT_BYTES;
};

// Where 16 bytes (8 k values) of a 64-byte row lie: neither the reads (32 rows, 16 of them at a time: 0-3, 12-15, 20-27 and the others) nor the writes
// (8 consecutive lanes) meet in a bank
__device__ __forceinline__ unsigned row_slot(unsigned row, unsigned chunk) { return row * 64 + ((chunk ^ (row >> 2)) & 3) * 16; }

template <int QG, int KR, int SEQ, bool PIECES>
__global__ void __launch_bounds__(QG* KR * 64, SEQ * QG * KR / 4) attn_f32_pieces_kernel(SegDev s, int NH, int n_q, int total, float scale) {
    typedef PiecesShape<QG, KR, SEQ> S;
    constexpr int HS = S::HS, NC = HS / 16, ND = HS / 32, PT = QG * 64, CK = 4 * HS / PT, TKEYS = 32, RUNS = KR * SEQ;
    static_assert(SEQ == 1 || (KR == 1 && SEQ == 2), "runs side by side or two one after the other");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, lk = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), run = wave / QG, group = wave % QG;
    const unsigned tid = threadIdx.x - run * PT;  // among the threads of the run
    // consecutive workgroup ids go to the 8 XCDs in turn: every XCD gets a contiguous run of (batch, head, query tile)
    const int xcd = blockIdx.x % 8, local = blockIdx.x / 8, per = (total + 7) / 8, tall = (total % 8) ? (total % 8) : 8;
    const int item = xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
    const int bh = item / n_q, h = bh % NH, b = bh / NH, qt = (item % n_q) * S::QWG + group * 32 + l32;
    const int T0 = s.T[0], T1 = s.T[1], Tq0 = s.Tq[0], TQ = s.Tq[0] + s.Tq[1];

    f32x16_t o[ND];
    float m_run = -1e30f, l_run = 0.f;  // l_run: over the keys of this lane
#pragma unroll
    for (int j = 0; j < ND; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = 0.f;

    const int nt0 = (T0 + TKEYS - 1) / TKEYS, n_t = nt0 + (T1 + TKEYS - 1) / TKEYS, first = (n_t + RUNS - 1) / RUNS;
    const int ld0 = s.ld_qkv[0], ld1 = s.ld_qkv[1];
    const float* k0 = s.k[0] + (long long)b * T0 * ld0 + h * HS;
    const float* k1 = s.k[1] + (long long)b * T1 * ld1 + h * HS;
    const float* v0 = s.v[0] + (long long)b * T0 * ld0 + h * HS;
    const float* v1 = s.v[1] + (long long)b * T1 * ld1 + h * HS;
    auto keys_of = [&](int t, int& seg, int& t0) {  // tile t: its segment, its first key in it
        seg = t < nt0 ? 0 : 1;
        t0 = (seg ? t - nt0 : t) * TKEYS;
        return (seg ? T1 : T0) - t0;  // keys from here to the end of the segment
    };
    char* const k_lds = smem + run * S::RUN_BYTES;
    char* const v_lds = k_lds + S::K_BYTES;

    // This thread's share of a tile: CK runs of 8 values of a K row, and CK squares of 4 keys x 2 values of V: d = 16 * (u / 64) + 2 * (u % 8); keys 4 * quad ..: bits
    // 3, 4, 5 of u are bits 1, 0, 2 of the quad.
    auto quad_of = [](unsigned u) { return (u >> 3 & 1) << 1 | (u >> 4 & 1) | (u >> 5 & 1) << 2; };
    f32x4_t kr[CK][2];
    f32x2_t vr[CK][4];
    // Where they are: a scalar base per tile, and offsets in bytes that stay as they are from one whole tile of a segment to the next
    const char *k_base, *v_base;
    unsigned k_off[CK], v_off[CK][4];
    int k_rows = -1, v_rows = -1;  // segment and rows of the tile that the offsets are for
    auto rows_of = [&](int& t, int& ld, int& rows) {  // (tiles past the end: the last one)
        t = min(t, n_t - 1);
        const int seg = t < nt0 ? 0 : 1;
        t = (seg ? t - nt0 : t) * TKEYS;
        ld = seg ? ld1 : ld0;
        rows = min((seg ? T1 : T0) - t, TKEYS);
        return seg;
    };
    auto find_k = [&](int t) {
        int ld, rows;
        const int seg = rows_of(t, ld, rows), state = seg * 64 + rows;
        k_base = reinterpret_cast<const char*>((seg ? k1 : k0) + (long long)t * ld);
        if (state == k_rows) return;
        k_rows = state;
#pragma unroll
        for (int i = 0; i < CK; i++) {
            const unsigned u = i * PT + tid;
            k_off[i] = __umul24(min((int)(u / 4 % 32), rows - 1), ld) * 4u + (u / 128 * 32 + u % 4 * 4) * 4;
        }
    };
    auto find_v = [&](int t) {
        int ld, rows;
        const int seg = rows_of(t, ld, rows), state = seg * 64 + rows;
        v_base = reinterpret_cast<const char*>((seg ? v1 : v0) + (long long)t * ld);
        if (state == v_rows) return;
        v_rows = state;
#pragma unroll
        for (int i = 0; i < CK; i++) {
            const unsigned u = i * PT + tid;
#pragma unroll
            for (int x = 0; x < 4; x++) v_off[i][x] = __umul24(min((int)quad_of(u) * 4 + x, rows - 1), ld) * 4u + (u / 64 * 16 + u % 8 * 2) * 4;
        }
    };
    auto load_k = [&]() {
#pragma unroll
        for (int i = 0; i < CK; i++) {
            kr[i][0] = *reinterpret_cast<const f32x4_t*>(k_base + k_off[i]);
            kr[i][1] = *reinterpret_cast<const f32x4_t*>(k_base + k_off[i] + 64);
        }
    };
    auto load_v = [&]() {
#pragma unroll
        for (int i = 0; i < CK; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) vr[i][x] = *reinterpret_cast<const f32x2_t*>(v_base + v_off[i][x]);
    };
    // (all requests before the first wait)
    const int first_tile = SEQ > 1 ? 0 : run;
    find_k(first_tile);
    find_v(first_tile);
    load_k();
    load_v();
    // pieces of the lane's query: of step c the 8 values d = 32(c/2) + 8(c%2) + 4(l/32) .. +3 and 16 behind them
    bf16x8_t q[3][NC];
    {
        const int t = min(qt, TQ - 1), seg = t < Tq0 ? 0 : 1;  // (queries past the end repeat the last one and are not stored)
        const float* p = s.q[seg] + ((long long)b * s.Tq[seg] + (seg ? t - Tq0 : t)) * s.ld_qkv[seg] + h * HS + 4 * lk;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(p + c / 2 * 32 + c % 2 * 8), hi = *reinterpret_cast<const f32x4_t*>(p + c / 2 * 32 + c % 2 * 8 + 16);
            float x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) x[k] = (k < 4 ? lo[k & 3] : hi[k & 3]) * scale;
            uint32_t piece[3][4];
            bf16_pieces<8>(x, piece[0], piece[1], piece[2]);
#pragma unroll
            for (int w = 0; w < 3; w++) __builtin_memcpy(&q[w][c], piece[w], 16);
        }
    }
    Split part;
    auto put_k = [&](int i) {
        const unsigned u = i * PT + tid, key = u / 4 % 32, c = u / 128;
        char* at = k_lds + c * 3 * S::K_PLANE + row_slot(key, u % 4);
#pragma unroll
        for (int p = 0; p < 3; p++) __builtin_memcpy(__builtin_assume_aligned(at + p * S::K_PLANE, 16), part.piece[p], 16);
    };
    auto put_v = [&](int i, int buffer) {
        // of 16 keys, 4(l/32) .. +3 of either half are the k values 8(l/32) .. +7 of the matrix instruction, as the scores have them
        const unsigned u = i * PT + tid, d = u / 64 * 16 + u % 8 * 2, quad = quad_of(u), chunk = quad / 4 * 2 + quad % 2, half = quad / 2 % 2;
#pragma unroll
        for (int y = 0; y < 2; y++) {
            char* at = v_lds + buffer * S::V_BYTES + row_slot(d + y, chunk) + half * 8;
#pragma unroll
            for (int p = 0; p < 3; p++) __builtin_memcpy(__builtin_assume_aligned(at + p * S::V_PLANE, 8), &part.piece[p][2 * y], 8);
        }
    };
    // fragments: row l%32, chunk l/32 of one of the two k steps of a 64-byte row
    const unsigned src = row_slot(l32, lk);
    auto k_frag = [&](int c, int p) { return *reinterpret_cast<const bf16x8_t*>(k_lds + (c / 2 * 3 + p) * S::K_PLANE + (src ^ c % 2 * 32)); };
    auto v_frag = [&](int buffer, int n, int p) {  // n: d block n / 2, k step n % 2
        return *reinterpret_cast<const bf16x8_t*>(v_lds + buffer * S::V_BYTES + p * S::V_PLANE + n / 2 * 2048 + (src ^ n % 2 * 32));
    };
    // The products of pieces of a k step in the order l*h, m*m, h*l, m*h, h*m, h*h. `beside(n)`, n = 0 .. COUNT - 1, is what the vector unit does meanwhile, spread
    // over the k steps.
    auto spread = [](int products, int reads) {
#pragma unroll
        for (int x = 0; x < products; x++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (x < reads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mfma = [](const bf16x8_t& a, const bf16x8_t& b, const f32x16_t& c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); };
    auto five = [&](const bf16x8_t (&a)[3], const bf16x8_t& h, const bf16x8_t& m, const bf16x8_t& l, f32x16_t& x) {
        x = mfma(a[2], h, x);
        x = mfma(a[1], m, x);
        x = mfma(a[0], l, x);
        x = mfma(a[1], h, x);
        x = mfma(a[0], m, x);
    };
    f32x16_t sc, sn;
    bf16x8_t p[3][2];
    constexpr float UNIT = 1.f / (PIECES_SCALE * PIECES_SCALE);  // of the scores as they leave the matrix unit
    constexpr int MARGIN = 8;
    auto scores = [&](f32x16_t& x, auto count, auto beside) {
        constexpr int COUNT = decltype(count)::value;
        bf16x8_t frag[2][3];
#pragma unroll
        for (int w = 2; w >= 0; w--) frag[0][w] = k_frag(0, w);
        f32x16_t large;
#pragma unroll
        for (int r = 0; r < 16; r++) x[r] = large[r] = 0.f;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int now = c & 1;
            five(frag[now], q[0][c], q[1][c], q[2][c], x);
            large = mfma(frag[now][0], q[0][c], large);
            if (c + 1 < NC)
#pragma unroll
                for (int w = 2; w >= 0; w--) frag[now ^ 1][w] = k_frag(c + 1, w);
#pragma unroll
            for (int z = c * COUNT / NC; z < (c + 1) * COUNT / NC; z++) beside(z);
            spread(6, c + 1 < NC ? 3 : 0);
        }
        x += large;
    };
    auto outputs = [&](int buffer, auto count, auto beside) {
        constexpr int COUNT = decltype(count)::value;
        bf16x8_t frag[2][3];
#pragma unroll
        for (int w = 2; w >= 0; w--) frag[0][w] = v_frag(buffer, 0, w);
#pragma unroll
        for (int j = 0; j < ND; j++) {
            f32x16_t x;  // of this tile, so that o is rounded once per tile
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = 0.f;
#pragma unroll
            for (int step = 0; step < 2; step++) {
                const int n = 2 * j + step;
                five(frag[step], p[0][step], p[1][step], p[2][step], x);
                if (step == 1) {
                    x = mfma(frag[0][0], p[0][0], x);
                    x = mfma(frag[1][0], p[0][1], x);
                }
                if (step == 0 || j + 1 < ND)
#pragma unroll
                    for (int w = 2; w >= 0; w--) frag[step ^ 1][w] = v_frag(buffer, n + 1, w);
#pragma unroll
                for (int z = n * COUNT / (2 * ND); z < (n + 1) * COUNT / (2 * ND); z++) beside(z);
                spread(step ? 7 : 5, step == 0 || j + 1 < ND ? 3 : 0);
            }
            o[j] += x;
        }
    };
    // The softmax of the current tile in steps, for each half of the lane's keys: their probabilities, the sum and the pieces
    constexpr int SOFTMAX = (3 + Split::STEPS) * 2;
    auto softmax = [&](f32x16_t& x, int n) {
        const int half = n / (3 + Split::STEPS), step = n % (3 + Split::STEPS);
        if (step == 0) {
#pragma unroll
            for (int k = 0; k < 8; k++) part.x[k] = __builtin_fmaf(x[8 * half + k], UNIT, -m_run);
        } else if (step == 1) {
#pragma unroll
            for (int k = 0; k < 8; k++) part.x[k] = __builtin_amdgcn_exp2f(part.x[k]);
        } else if (step == 2) {
            l_run += ((part.x[0] + part.x[1]) + (part.x[2] + part.x[3])) + ((part.x[4] + part.x[5]) + (part.x[6] + part.x[7]));
        } else {
            part.step(step - 3);
            if (step == 2 + Split::STEPS)
#pragma unroll
                for (int w = 0; w < 3; w++) __builtin_memcpy(&p[w][half], part.piece[w], 16);
        }
    };
    // The largest score of a tile, in two steps
    float most_a, most_b, top;
    auto largest = [&](const f32x16_t& x, int n) {
        if (n == 0) {
            most_a = x[0];
            most_b = x[8];
#pragma unroll
            for (int r = 1; r < 8; r++) {
                most_a = fmaxf(most_a, x[r]);
                most_b = fmaxf(most_b, x[8 + r]);
            }
        } else {
            most_a = fmaxf(most_a, most_b);
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(most_a), __float_as_uint(most_a), false, false);
            top = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
        }
    };

    // A run's tiles are run, run + RUNS, ...; one without a tile in the last iteration keeps the barriers' company only. With SEQ = 2 a wavefront has the tiles of the
    // second run behind those of the first.
    const int n_it = SEQ > 1 ? n_t : first;
    auto tile_of = [&](int it) { return SEQ > 1 && it >= first ? it < n_t ? (it - first) * 2 + 1 : n_t : it * RUNS + run; };
    // K and V tiles to LDS and the requests of the next ones, in steps
    constexpr int STEPS = Split::STEPS + 1, STAGING = 2 * STEPS * CK;
    auto stage_k = [&](int i, int n) {
        if (n == 0)
#pragma unroll
            for (int k = 0; k < 8; k++) part.x[k] = kr[i][k >> 2][k & 3] * PIECES_SCALE;
        if (n < Split::STEPS) part.step(n);
        if (n == Split::STEPS - 1) put_k(i);
        if (n == Split::STEPS && i == CK - 1) load_k();
    };
    auto stage_v = [&](int i, int n, int buffer) {
        if (n == 0)
#pragma unroll
            for (int k = 0; k < 8; k++) part.x[k] = vr[i][k & 3][k >> 2] * PIECES_SCALE;
        if (n < Split::STEPS) part.step(n);
        if (n == Split::STEPS - 1) put_v(i, buffer);
        if (n == Split::STEPS && i == CK - 1) load_v();
    };
    typedef std::integral_constant<int, 0> None;
    find_k(tile_of(1));
    find_v(tile_of(1));
#pragma unroll
    for (int n = 0; n < STEPS * CK; n++) stage_k(n / STEPS, n % STEPS);
#pragma unroll
    for (int n = 0; n < STEPS * CK; n++) stage_v(n / STEPS, n % STEPS, 0);
    barrier_behind_lds<0>();
    scores(sc, None(), [](int) {});
    barrier_behind_lds<0>();
    find_k(tile_of(2));
#pragma unroll
    for (int n = 0; n < STEPS * CK; n++) stage_k(n / STEPS, n % STEPS);
    auto mask = [&](f32x16_t& x, int it) {  // keys past the end of the tile's segment
        int seg, t0;
        const int left = keys_of(tile_of(it), seg, t0);
        if (left < TKEYS) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (8 * (r >> 2) + 4 * lk + (r & 3) >= left) x[r] = -__builtin_inff();
        }
    };
    mask(sc, 0);
    largest(sc, 0);
    largest(sc, 1);
    barrier_behind_lds<0>();
    // Tile `it` of the run, whose scores are x and their largest `top`; y: the scores of the next one. Two barriers: the scores of the next tile beside the softmax of this one;
    // the outputs beside the split of the K tile after the next and of the next V tile.
    float* const kept = reinterpret_cast<float*>(smem + S::LDS - S::KEPT_BYTES) + threadIdx.x * S::PITCH;
    auto keep = [&](float* at) {
        at[0] = m_run;
        at[1] = l_run;
#pragma unroll
        for (int j = 0; j < ND; j++)
#pragma unroll
            for (int r = 0; r < 16; r += 4) *reinterpret_cast<f32x4_t*>(at + 4 + j * 16 + r) = f32x4_t{o[j][r], o[j][r + 1], o[j][r + 2], o[j][r + 3]};
    };
    // This wavefront's run and another one; EARLIER: the other one is the earlier of the two (the sums round the same either way round)
    auto merge_with = [&](const float* at, auto earlier) {
        constexpr bool EARLIER = decltype(earlier)::value;
        const float om = at[0], mx = fmaxf(m_run, om);
        const float wa = __builtin_amdgcn_exp2f(m_run - mx), wb = __builtin_amdgcn_exp2f(om - mx);  // (a run that had no tile: its factor is 0)
        auto sum = [&](float mine, float other) { return EARLIER ? __builtin_fmaf(other, wb, mine * wa) : __builtin_fmaf(mine, wa, other * wb); };
        m_run = mx;
        l_run = sum(l_run, at[1]);
#pragma unroll
        for (int j = 0; j < ND; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[j][r] = sum(o[j][r], at[4 + j * 16 + r]);
    };
    auto tile = [&](int it, f32x16_t& x, f32x16_t& y, auto buffer_tag) {
        constexpr int buffer = decltype(buffer_tag)::value;
        const bool mine = tile_of(it) < n_t;
        if (SEQ > 1 && it == first) {  // the second run starts
            keep(kept);
            m_run = -1e30f;
            l_run = 0.f;
#pragma unroll
            for (int j = 0; j < ND; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[j][r] = 0.f;
        }
        if (mine) {
            // The reference moves only where a score exceeds it by 2^MARGIN: in the first tile and hardly ever again (with the largest score as the reference some of
            // 32 queries have a larger one in most tiles)
            const bool moves = top * UNIT > m_run + MARGIN;
            if (__builtin_amdgcn_ballot_w64(moves)) {
                const float m = moves ? top * UNIT : m_run, alpha = __builtin_amdgcn_exp2f(m_run - m);
                m_run = m;
                l_run *= alpha;
#pragma unroll
                for (int j = 0; j < ND; j++) o[j] *= alpha;
            }
            find_k(tile_of(it + 3));
            find_v(tile_of(it + 2));
            scores(y, std::integral_constant<int, SOFTMAX>(), [&](int n) { softmax(x, n); });
            // (named here, or the compiler moves what makes them behind the branches that follow, away from the products that it is to run beside)
            asm volatile("" : "+v"(y), "+v"(l_run));
#pragma unroll
            for (int w = 0; w < 3; w++) asm volatile("" : "+v"(p[w][0]), "+v"(p[w][1]));
        }
        barrier_behind_lds<0>();
        if (mine) {
            mask(y, it + 1);
            outputs(buffer, std::integral_constant<int, STAGING + 2>(), [&](int n) {
                if (n < STEPS * CK) stage_k(n / STEPS, n % STEPS);
                else if (n < STAGING) stage_v(n / STEPS - CK, n % STEPS, buffer ^ 1);
                else largest(y, n - STAGING);
            });
        }
        barrier_behind_lds<0>();
    };
    for (int it = 0; it < n_it; it += 2) {
        tile(it, sc, sn, std::integral_constant<int, 0>());
        if (it + 1 < n_it) tile(it + 1, sn, sc, std::integral_constant<int, 1>());
    }

    // merge: in each step the upper half of the runs hands its state to the lower half
    float* merge = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int half = KR / 2; half >= 1; half /= 2) {
        float* at = merge + (((run < half ? run : run - half) * QG + group) * 64 + lane) * S::PITCH;
        __syncthreads();
        if (run >= half && run < 2 * half) keep(at);
        __syncthreads();
        if (run < half) merge_with(at, std::false_type());
    }
    if (SEQ > 1 && n_t > 1) merge_with(kept, std::true_type());
#pragma unroll
    for (int j = 0; j < ND; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[j][r] = o[j][r] * (1.f / PIECES_SCALE);
    if (run) return;
    const float l = l_run + __shfl_xor(l_run, 32, 64), inv = 1.0f / l;
    bool bad = !finite(l) || l == 0.f;
#pragma unroll
    for (int j = 0; j < ND; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            bad |= !finite(o[j][r]);
            o[j][r] *= inv;
        }
    const int seg = qt < Tq0 ? 0 : 1;
    const bool store = qt < TQ && s.out[seg];
    const long long row = store ? (long long)b * s.Tq[seg] + (seg ? qt - Tq0 : qt) : -1;
    if (__builtin_amdgcn_ballot_w64(bad)) {
        attend_in_f32<PIECES>(s, b, h, min(qt, TQ - 1), scale, row);
        return;
    }
    if (store)
#pragma unroll
        for (int j = 0; j < ND; j++)
#pragma unroll
            for (int r = 0; r < 16; r += 4) put_output<PIECES>(s, seg, row, h * HS + 4 * lk + 32 * j + 2 * r, f32x4_t{o[j][r], o[j][r + 1], o[j][r + 2], o[j][r + 3]});
}

template <int QG, int KR, int SEQ, bool PIECES>
int launch_attn_pieces_as(const SegDev& s, int B, int NH, float scale, hipStream_t st) {
    typedef PiecesShape<QG, KR, SEQ> S;
    auto kern = attn_f32_pieces_kernel<QG, KR, SEQ, PIECES>;
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(kern), S::LDS));
    const int TQ = s.Tq[0] + s.Tq[1], n_q = (TQ + S::QWG - 1) / S::QWG;
    const long long total = (long long)B * NH * n_q;
    if (total > 0x7fffffff) return fail(SD3_ERR_UNSUPPORTED, "attention (fp32): too many work items");
    hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(S::THREADS), S::LDS, st, s, NH, n_q, (int)total, scale);
    return launch_status("attention_f32");
}
template <int QG, int KR, int SEQ>
int launch_attn_pieces(const SegDev& s, int B, int NH, float scale, bool pieces, hipStream_t st) {
    return pieces ? launch_attn_pieces_as<QG, KR, SEQ, true>(s, B, NH, scale, st) : launch_attn_pieces_as<QG, KR, SEQ, false>(s, B, NH, scale, st);
}
}  // namespace

int g_attention_f32_no_pieces = 0;  // 1: fp32 matrix instruction in every call (sd3_tune)

int attention_f32(const AttnSegments& a, int B, int NH, int HS, hipStream_t st) {
    const int T = a.T[0] + a.T[1], TQ = a.Tq[0] + a.Tq[1];
    if (B <= 0 || NH <= 0 || TQ <= 0) return SD3_OK;
    if (T <= 0) return fail(SD3_ERR_INVALID_ARG, "attention: no keys");
    if (HS <= 0 || HS > 128) return fail(SD3_ERR_UNSUPPORTED, "attention (fp32): head_dim %d not in 1..128", HS);
    SegDev s;
    s.B = B;
    bool vec = (HS % 4 == 0), vec_io = true;  // vec_io: queries and outputs too are made of aligned 16-byte chunks
    for (int i = 0; i < 2; i++) {
        s.q[i] = (const float*)a.q[i]; s.k[i] = (const float*)a.k[i]; s.v[i] = (const float*)a.v[i]; s.out[i] = (float*)a.out[i];
        s.ld_qkv[i] = a.ld_qkv[i]; s.ld_out[i] = a.ld_out[i]; s.T[i] = a.T[i]; s.Tq[i] = a.Tq[i];
        if (a.Tq[i] > 0 && !a.q[i]) return fail(SD3_ERR_INVALID_ARG, "attention: null q for segment %d", i);
        if (a.Tq[i] > 0 && ((a.ld_qkv[i] % 4) || (a.ld_out[i] % 4) || (reinterpret_cast<uintptr_t>(a.q[i]) & 15) || (reinterpret_cast<uintptr_t>(a.out[i]) & 15)))
            vec_io = false;
        if (a.T[i] > 0) {
            if (!a.k[i] || !a.v[i]) return fail(SD3_ERR_INVALID_ARG, "attention: null k/v for segment %d", i);
            if ((a.ld_qkv[i] % 4) || (reinterpret_cast<uintptr_t>(a.k[i]) & 15) || (reinterpret_cast<uintptr_t>(a.v[i]) & 15)) vec = false;
        }
    }
    const float scale = (float)(1.0 / sqrtf((float)HS));
    const float scale2 = (float)(1.4426950408889634 / sqrt((double)HS));  // scores in powers of two: the exponentials are one instruction
    if (vec && vec_io && (HS == 64 || HS == 128) && a.ld_qkv[0] < (1 << 24) && a.ld_qkv[1] < (1 << 24)) {
        // By pieces where an element alone is not slower: heads x blocks of 128 queries from 96 on, and these x tiles of 32 keys from 1536. us, fp32 instruction | pieces: one
        // element of 24 heads: 333 tokens (72 blocks) 17.2 | 18.6, 400 (96 blocks, 1248 with tiles) 20.4 | 21.6, 512 23.9 | 23.7, 640 28.3 | 28.2, 700 42 | 34, 1024 58 | 46, 512
        // queries of 77 keys 10.2 | 11.5, 1024 of 333 25.0 | 22.8; 12 heads, 666 tokens (72) 19 | 29, 1000 (96) 40.5 | 39.6. 24 heads, 666 tokens (144) 29.8 | 33.2: one more query and the
        // fp32 kernel takes 42. Batches gain more, 8 x 24 heads, 333 tokens 63 | 56, 16 x 12 heads, 666 tokens 187 | 155, but an element's result stays what it is alone.
        // (Up to 64 queries more than half of a block would be empty.)
        const long long element_blocks = (long long)NH * ((TQ + 127) / 128);
        if (HS == 64 && TQ > 64 && element_blocks >= 96 && element_blocks * ((T + 31) / 32) >= 1536 && !g_attention_f32_no_pieces) {
            const int cus = compute_units();
            if (cus <= 0) return SD3_ERR_HIP;
            const long long blocks = B * element_blocks;
            // How the two runs of keys are computed, which their results do not depend on: side by side in workgroups of 64 or of 128 queries as long as all of these
            // find a compute unit, then one after the other in workgroups of half the wavefronts, two to a unit and independent of each other's
            // barriers. us, 24 heads: 512 tokens 25 | 27 | 32; 700 58 | 34 | 42, a batch of two 86 | 69 | 60; 1178 90 | 57 | 67, a batch of two 178 | 113 | 106.
            if (2 * blocks <= cus) return launch_attn_pieces<2, 2, 1>(s, B, NH, scale2, a.out_pieces, st);
            if (blocks <= cus) return launch_attn_pieces<4, 2, 1>(s, B, NH, scale2, a.out_pieces, st);
            return launch_attn_pieces<4, 1, 2>(s, B, NH, scale2, a.out_pieces, st);
        }
        // 32 queries per workgroup; with so few (queries, heads) that this leaves compute units idle, 16. Four key runs in both: eight, or the keys over several
        // workgroups and a second kernel to merge, cost as much in starts and merging as they save in the runs (2 heads of 128, 1178 tokens: 36 and 36 us, four
        // runs 32).
        const bool few = (long long)NH * ((TQ + 31) / 32) < 192;
        if (a.ld_qkv[0] >= (1 << 22) || a.ld_qkv[1] >= (1 << 22)) {  // (tens of thousands of heads)
            if (a.out_pieces) return fail(SD3_ERR_INVALID_ARG, "attention (fp32): no outputs in pieces for rows as long as these");
            return HS == 64 ? launch_split_as<64, 2, 1, 4, true, false>(s, B, NH, scale2, st) : launch_split_as<128, 2, 1, 4, true, false>(s, B, NH, scale2, st);
        }
        if (HS == 64) return few ? launch_split<64, 1, 2, 4>(s, B, NH, scale2, a.out_pieces, st) : launch_split<64, 2, 1, 4>(s, B, NH, scale2, a.out_pieces, st);
        return few ? launch_split<128, 1, 1, 4>(s, B, NH, scale2, a.out_pieces, st) : launch_split<128, 2, 1, 4>(s, B, NH, scale2, a.out_pieces, st);
    }
    if (a.out_pieces) return fail(SD3_ERR_INVALID_ARG, "attention (fp32): no outputs in pieces for these heads, strides or alignments");
    dim3 grid((TQ + BQ - 1) / BQ, NH, B), block(256);
    const int hsp = HS <= 32 ? 32 : (HS <= 64 ? 64 : 128);
#define SD3_ATTN_LAUNCH(P)                                                                              \
    do {                                                                                                \
        if (vec) hipLaunchKernelGGL((attn_f32_kernel<P, true>), grid, block, 0, st, s, HS, scale);      \
        else hipLaunchKernelGGL((attn_f32_kernel<P, false>), grid, block, 0, st, s, HS, scale);         \
    } while (0)
    if (hsp == 32) SD3_ATTN_LAUNCH(32);
    else if (hsp == 64) SD3_ATTN_LAUNCH(64);
    else SD3_ATTN_LAUNCH(128);
#undef SD3_ATTN_LAUNCH
    return launch_status("attention_f32");
}

}  // namespace sd3
