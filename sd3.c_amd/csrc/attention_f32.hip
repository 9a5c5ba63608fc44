// fp32 multi-head attention on the fp32 matrix cores, for the fp32 parity path and the attention operator.
// Replaces multihead_attention (modules.cpp:766-831) and, through its two-segment addressing, the token
// concatenation / split around it (modules.cpp:1427-1432): keys/values/queries of the joint sequence are read
// straight from the context buffers (first T[0] tokens) and the latent buffers (next T[1] tokens).
//
// Two kernels: attn_f32_split_kernel for head_dim 64 and 128 with 16-byte aligned rows (below), attn_f32_kernel for any other head_dim up
// to 128. Formulation of both: everything is kept transposed so that the probabilities never leave registers.
//   S^T (keys x queries) = K . Q^T      -> C-layout: a lane owns ONE query column and 16 keys per 32-key block
//   O^T (d x queries)   += V^T . P^T    -> the lane's own S^T registers are exactly the P^T operand it must supply
// Online softmax statistics are per query = per lane (plus one exchange with lane^32).
#include <type_traits>

#include "common.hpp"

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
};

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

// ---- head_dim 64 and 128 ----
// The matrix unit (v_mfma_f32_16x16x4_f32: 64 FLOP per cycle and SIMD) is the bound, and everything it needs fits the registers of one
// wavefront: 16*QB queries and 16*KB keys at a time. So no LDS tiles and no barriers: the KS wavefronts of a workgroup share its queries
// and split the KEYS (tile t goes to wavefront t % KS); K and V rows come straight from memory (L2: all workgroups of a head run on one
// XCD) into registers, half a tile of matrix work ahead of their use; the KS partial results are merged in a fixed tree at the end.
// This gives every SIMD work also where there are few queries: 1178 tokens and 2 heads are 20 workgroups of 128 queries with the keys in
// one run (290 us), 592 wavefronts this way (30 us). 2 x 24 heads of 64, 1178 tokens: 244 -> 148 us, 70 -> 115 TFLOP/s of 155 (the matrix
// instructions alone about 127, the softmax 12, the loads 9).
//
// Contraction order: K and Q are read as float4 along d, so step s of 16-wide chunk c contracts d = 16c + 4g + s over the lane groups
// g = l/16. S^T registers r of a 16x16 block are keys 4g + r of query l%16: as they are, the operand of step r of O^T += V^T P^T, whose
// V rows 4g + r are read as float4 along d: block j of the four takes d = 4(l%16) + j, so a lane ends with 16 consecutive d of its query.
// LONG_ROWS: rows are 2^22 floats or more apart (and less than 2^24): four times the stride does not fit the 24-bit product of the row offsets. An
// instantiation of its own, since the shift behind the product, done in every case, costs the others up to 2 %. 65536 heads of 64, 2 queries, 40 keys:
// 691 us, with attn_f32_kernel 2204.
template <int HS, int QB, int KB, int KS, bool LONG_ROWS>
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
        float alpha[QB];
#pragma unroll
        for (int i = 0; i < QB; i++) {
            float mx = m_run[i];
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) mx = fmaxf(mx, sc[kb][i][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            alpha[i] = __builtin_amdgcn_exp2f(m_run[i] - mx);
            m_run[i] = mx;
            l_run[i] *= alpha[i];
#pragma unroll
            for (int kb = 0; kb < KB; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = __builtin_amdgcn_exp2f(sc[kb][i][r] - mx);
                    sc[kb][i][r] = p;
                    l_run[i] += p;
                }
        }
#pragma unroll
        for (int i = 0; i < QB; i++)
            if (__builtin_amdgcn_ballot_w64(alpha[i] != 1.0f))  // the maximum moves in few tiles
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int j = 0; j < 4; j++) o[i][u][j] *= alpha[i];
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
        float* p = s.out[seg] + ((long long)b * s.Tq[seg] + (seg ? qt - Tq0 : qt)) * s.ld_out[seg] + h * HS + 16 * lg;
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                *reinterpret_cast<f32x4_t*>(p + 64 * u + 4 * r) =
                    f32x4_t{o[i][u][0][r] * inv, o[i][u][1][r] * inv, o[i][u][2][r] * inv, o[i][u][3][r] * inv};
    }
}

template <int HS, int QB, int KB, int KS, bool LONG_ROWS = false>
int launch_split(const SegDev& s, int B, int NH, float scale, hipStream_t st) {
    const int TQ = s.Tq[0] + s.Tq[1], n_q = (TQ + 16 * QB - 1) / (16 * QB);
    const long long total = (long long)B * NH * n_q;
    if (total > 0x7fffffff) return fail(SD3_ERR_UNSUPPORTED, "attention (fp32): too many work items");
    hipLaunchKernelGGL((attn_f32_split_kernel<HS, QB, KB, KS, LONG_ROWS>), dim3((unsigned)total), dim3(KS * 64), 0, st, s, NH, n_q, (int)total, scale);
    return launch_status("attention_f32");
}
}  // namespace

int attention_f32(const AttnSegments& a, int B, int NH, int HS, hipStream_t st) {
    const int T = a.T[0] + a.T[1], TQ = a.Tq[0] + a.Tq[1];
    if (B <= 0 || NH <= 0 || TQ <= 0) return SD3_OK;
    if (T <= 0) return fail(SD3_ERR_INVALID_ARG, "attention: no keys");
    if (HS <= 0 || HS > 128) return fail(SD3_ERR_UNSUPPORTED, "attention (fp32): head_dim %d not in 1..128", HS);
    SegDev s;
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
        // 32 queries per workgroup; with so few (queries, heads) that this leaves compute units idle, 16. (Not by the batch: a batch
        // element's result stays what it is alone.) Four key runs in both: eight, or the keys over several workgroups and a second
        // kernel to merge, cost as much in starts and merging as they save in the runs (2 heads of 128, 1178 tokens: 36 and 36 us, four
        // runs 32).
        const bool few = (long long)NH * ((TQ + 31) / 32) < 192;
        if (a.ld_qkv[0] >= (1 << 22) || a.ld_qkv[1] >= (1 << 22))  // (tens of thousands of heads)
            return HS == 64 ? launch_split<64, 2, 1, 4, true>(s, B, NH, scale2, st) : launch_split<128, 2, 1, 4, true>(s, B, NH, scale2, st);
        if (HS == 64) return few ? launch_split<64, 1, 2, 4>(s, B, NH, scale2, st) : launch_split<64, 2, 1, 4>(s, B, NH, scale2, st);
        return few ? launch_split<128, 1, 1, 4>(s, B, NH, scale2, st) : launch_split<128, 2, 1, 4>(s, B, NH, scale2, st);
    }
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
