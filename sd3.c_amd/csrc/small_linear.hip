// Linear layers whose left operand has few rows (the batch; eight per launch): the adaLN modulation projections
// (modules.cpp:1384-1501 compute them one 1536-column chunk at a time with partial_linear), the timestep and
// pooled-text MLPs (modules.cpp:1664-1671). They are pure weight streaming, so one launch covers a whole list
// of weight matrices ("jobs") and reads every weight element exactly once, fp32 N-contiguous as the reference stores it or
// (bf16 modulation projections) as panels.
#include <vector>

#include "common.hpp"

namespace sd3 {

// Block = 256 threads = CG column groups (4 columns each) x 256 / CG slices of K. A launch is bound by the weights it streams once enough
// rows of them are requested at a time: 128 columns and 8 slices (CG = 32) per workgroup do where thousands of workgroups are resident.
// With fewer workgroups a thread's run of K is a chain of memory latencies, so the columns are cut finer and K into more slices.
// x is staged transposed in LDS (xs[k][m]) so that a thread reads its M inputs for one k with wide LDS loads.
// Jobs travel as a kernel argument (no device-side table to keep coherent with the host).
struct SmallLinearJobPack {
    SmallLinearJob j[SMALL_LINEAR_JOBS_PER_LAUNCH];  // 52 x 56 bytes of kernel arguments: the 49 projections of a 24-block forward in one launch
};

template <int M, bool VEC, int CG>
__global__ void __launch_bounds__(256) small_linear_kernel(const float* __restrict__ x_all, int m_real, int K_all, const SmallLinearJobPack jobs, int act) {
    extern __shared__ float smem[];
    const SmallLinearJob job = jobs.j[blockIdx.y];
    constexpr int COLS = CG * 4, SLICES = 256 / CG;
    const int col_base = blockIdx.x * COLS;
    if (col_base >= job.N) return;
    const float* __restrict__ x = job.x ? job.x : x_all;  // (uniform over the workgroup)
    const int K = job.x ? job.K : K_all;
    const int tid = threadIdx.x;
#pragma unroll
    for (int m = 0; m < M; m++)
        for (int k = tid; k < K; k += 256) smem[k * M + m] = (m < m_real) ? x[(long long)m * K + k] : 0.f;
    __syncthreads();

    const int cl = tid % CG, ks = tid / CG;
    const int c0 = col_base + cl * 4;
    const int kper = (K + SLICES - 1) / SLICES;
    const int kbeg = ks * kper, kend = min(K, kbeg + kper);  // (with few rows the last slices may be empty)
    const float* W = job.W + job.n0 + c0;
    float acc[M][4];
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[m][j] = 0.f;

    constexpr int UNROLL_K = M <= 2 ? 8 : 4;
    if (c0 < job.N) {
        // weight rows in flight per thread: eight with one or two rows of x (measured: 4 and 16 are slower), four with more rows (registers)
#pragma unroll UNROLL_K
        for (int k = kbeg; k < kend; k++) {
            float w[4];
            if (VEC) {
                const float4 v = *reinterpret_cast<const float4*>(W + (long long)k * job.ldw);
                w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = (c0 + j < job.N) ? W[(long long)k * job.ldw + j] : 0.f;
            }
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float xv = smem[k * M + m];
#pragma unroll
                for (int j = 0; j < 4; j++) acc[m][j] += xv * w[j];
            }
        }
    }
    __syncthreads();  // everyone is done with xs; reuse it for the cross-slice reduction: red[ks][m][COLS]
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) smem[(ks * M + m) * COLS + cl * 4 + j] = acc[m][j];
    __syncthreads();
    for (int e = tid; e < M * COLS; e += 256) {
        const int m = e / COLS, c = e % COLS;
        const int col = col_base + c;
        if (m < m_real && col < job.N) {
            float s = 0.f;
#pragma unroll
            for (int sl = 0; sl < SLICES; sl++) s += smem[(sl * M + m) * COLS + c];
            if (job.bias) s += job.bias[job.n0 + col];
            if (act == SD3_ACT_SILU) s = silu_precise(s);
            else if (act == SD3_ACT_GELU_TANH) s = gelu_tanh_precise(s);
            job.out[(long long)m * job.N + col] = s;
        }
    }
}

// The modulation projections of the bf16 path on their own (common.hpp: ada_panel): one workgroup per panel. Those of a block (216 or 360
// panels of 1536 x 64): 16 us; of all 24 blocks, 1.53 GB, one / four / eight rows: 266, 291, 520 us (5.8, 5.3, 3.0 TB/s; from (K,N) weights, 128
// columns x 8 slices a workgroup, eight rows took 840). Eight rows are neither the weights nor the vector units (40 % of the time) nor the LDS (41 %, of which 54 %
// bank conflicts: the four slices of a wavefront read xs a multiple of 64 banks apart): with 114 KB of LDS a unit has one workgroup, whose staging of y,
// streaming and summing up nothing else covers.
struct AdaJobPack {
    AdaJob j[SMALL_LINEAR_JOBS_PER_LAUNCH];
};
template <int M>
__global__ void __launch_bounds__(512) ada_panel_kernel(const float* __restrict__ y, int B, int K, const AdaJobPack jobs) {
    extern __shared__ float smem[];
    const AdaJob job = jobs.j[blockIdx.y];
    const int t = blockIdx.x;
    if (t * 64 >= job.N) return;
    ada_stage_rows<512, M>(y, B, K, smem);
    ada_panel<512, M, false>(job.W + (long long)t * 64 * K, job.bias + t * 64, job.out + t * 64, job.ld, B, K, smem, smem + M * K);
}
template <int M>
static int launch_panels(const float* y, int B, int K, const AdaJobPack& pack, int n, int max_N, hipStream_t st) {
    const int smem = ada_lds_bytes(M, K);
    static DynamicLds lds;
    SD3_TRY(lds.allow(reinterpret_cast<const void*>(ada_panel_kernel<M>), smem));
    hipLaunchKernelGGL((ada_panel_kernel<M>), dim3(max_N / 64, n), dim3(512), smem, st, y, B, K, pack);
    return launch_status("ada_panels");
}
int ada_panels(const float* y, int B, int K, const AdaJob* jobs, int n, hipStream_t st) {
    if (B <= 0 || n <= 0) return SD3_OK;
    if (K <= 0 || K > 4096 || K % ADA_SLICES) return fail(SD3_ERR_UNSUPPORTED, "ada_panels: K=%d out of range", K);
    // eight rows at a time, or as many as the transposed rows and the slices' sums leave LDS for
    const int group = ada_lds_bytes(8, K) <= 160 * 1024 ? 8 : 4;
    constexpr int PER = SMALL_LINEAR_JOBS_PER_LAUNCH;
    for (int m0 = 0; m0 < B; m0 += group)
        for (int base = 0; base < n; base += PER) {
            const int count = n - base < PER ? n - base : PER, rows = B - m0 < group ? B - m0 : group;
            AdaJobPack pack{};
            int max_N = 0;
            for (int i = 0; i < count; i++) {
                const AdaJob& j = jobs[base + i];
                if (j.N % 64 || (reinterpret_cast<uintptr_t>(j.W) & 7)) return fail(SD3_ERR_INVALID_ARG, "ada_panels: %d columns are not whole panels", j.N);
                pack.j[i] = AdaJob{j.W, j.bias, j.out + (long long)m0 * j.ld, j.N, j.ld};
                max_N = j.N > max_N ? j.N : max_N;
            }
            const float* x = y + (long long)m0 * K;
            if (rows == 1) SD3_TRY(launch_panels<1>(x, rows, K, pack, count, max_N, st));
            else if (rows == 2) SD3_TRY(launch_panels<2>(x, rows, K, pack, count, max_N, st));
            else if (rows <= 4) SD3_TRY(launch_panels<4>(x, rows, K, pack, count, max_N, st));
            else SD3_TRY(launch_panels<8>(x, rows, K, pack, count, max_N, st));
        }
    return SD3_OK;
}
// (K,N) fp32 -> bf16 panels (N/64, K, 64): 256 groups of four columns of 16 rows per workgroup
template <bool VEC>
__global__ void __launch_bounds__(256) pack_ada_panels_kernel(const float* __restrict__ W, bf16_t* __restrict__ out, int K, int N) {
    const int n = (blockIdx.x * 256 + threadIdx.x) * 4, k0 = blockIdx.y * 16;
    if (n >= N) return;
    const float* w = W + (long long)k0 * N + n;
    bf16_t* o = out + ((n >> 6) * (long long)K + k0) * 64 + (n & 63);
#pragma unroll 4
    for (int k = 0; k < min(16, K - k0); k++) {
        const float* r = w + (long long)k * N;
        const float4 v = VEC ? *reinterpret_cast<const float4*>(r) : make_float4(r[0], r[1], r[2], r[3]);
        *reinterpret_cast<uint2*>(o + k * 64) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
    }
}
int pack_ada_panels(const float* W, bf16_t* out, int K, int N, hipStream_t st) {
    if (N % 64) return fail(SD3_ERR_INVALID_ARG, "pack_ada_panels: %d columns are not whole panels", N);
    if (K <= 0 || N <= 0) return SD3_OK;
    const dim3 grid((N / 4 + 255) / 256, (K + 15) / 16);
    if ((reinterpret_cast<uintptr_t>(W) & 15) == 0) hipLaunchKernelGGL(pack_ada_panels_kernel<true>, grid, dim3(256), 0, st, W, out, K, N);
    else hipLaunchKernelGGL(pack_ada_panels_kernel<false>, grid, dim3(256), 0, st, W, out, K, N);
    return launch_status("pack_ada_panels");
}

template <int M, int CG>
static void launch_groups(const float* x, int m_real, int K, int K_max, const SmallLinearJobPack& jobs, int n_jobs, int max_N, bool vec, int act,
                          hipStream_t st) {
    dim3 grid((max_N + 4 * CG - 1) / (4 * CG), n_jobs), block(256);
    const int kk = K_max > 1024 ? K_max : 1024;
    const size_t smem = (size_t)kk * M * sizeof(float);
    if (vec) hipLaunchKernelGGL((small_linear_kernel<M, true, CG>), grid, block, smem, st, x, m_real, K, jobs, act);
    else hipLaunchKernelGGL((small_linear_kernel<M, false, CG>), grid, block, smem, st, x, m_real, K, jobs, act);
}

// The split is chosen from the weights of the launch alone, so that a row's result does not depend on how many rows there are: up to two
// wide workgroups per compute unit, runs of one cache line (32 columns, 32 slices). Wide and narrow, us: the timestep and text MLPs (2 x 12
// wide workgroups, K up to 2048) 24.0 and 11.8 with one row, 45 and 20 with four; the modulation vectors of one block of width 768, eight
// rows (90): 38 and 21 -- shorter runs than a line lose everywhere from 16 workgroups on.
template <int M>
static void launch_small(const float* x, int m_real, int K, int K_max, const SmallLinearJobPack& jobs, int n_jobs, int max_N, bool vec, int act,
                         hipStream_t st) {
    long long wide = 0;  // workgroups of 128 columns
    for (int i = 0; i < n_jobs; i++) wide += (jobs.j[i].N + 127) / 128;
    if (wide > 512) launch_groups<M, 32>(x, m_real, K, K_max, jobs, n_jobs, max_N, vec, act, st);
    else launch_groups<M, 8>(x, m_real, K, K_max, jobs, n_jobs, max_N, vec, act, st);
}

int small_linear_batched(const float* x, int M, int K, const SmallLinearJob* jobs_host, int n_jobs, int act, hipStream_t st) {
    if (M <= 0 || n_jobs <= 0) return SD3_OK;
    const int K_launch = K;  // depth of the launch's own x (jobs may bring theirs)
    for (int i = 0; i < n_jobs; i++) {
        if (!jobs_host[i].x && !x) return fail(SD3_ERR_INVALID_ARG, "small_linear: job %d has no left operand", i);
        if (jobs_host[i].x && jobs_host[i].K > K) K = jobs_host[i].K;  // from here on K is the largest depth of the launch (LDS size)
    }
    if (K <= 0 || K > 4096) return fail(SD3_ERR_UNSUPPORTED, "small_linear: K=%d out of range", K);
    // rows per launch: eight, or four when eight transposed rows of x do not fit the 64 KB of LDS a workgroup may use (K > 2048)
    const int group = ((size_t)(K > 1024 ? K : 1024) * 8 * sizeof(float) > 65536) ? 4 : 8;
    if (M > group) {
        // more rows than that (the reference's own block test runs a batch of 16, module_tests/dit_block.py:12): a group at a time, the
        // weights streamed once per group
        std::vector<SmallLinearJob> part(jobs_host, jobs_host + n_jobs);
        for (int m0 = 0; m0 < M; m0 += group) {
            for (int i = 0; i < n_jobs; i++) {
                part[i].out = jobs_host[i].out ? jobs_host[i].out + (long long)m0 * jobs_host[i].N : nullptr;
                part[i].x = jobs_host[i].x ? jobs_host[i].x + (long long)m0 * jobs_host[i].K : nullptr;
            }
            SD3_TRY(small_linear_batched(x ? x + (long long)m0 * K_launch : nullptr, M - m0 < group ? M - m0 : group, K_launch, part.data(), n_jobs, act, st));
        }
        return SD3_OK;
    }
    constexpr int PER = SMALL_LINEAR_JOBS_PER_LAUNCH;
    for (int base = 0; base < n_jobs; base += PER) {
        const int n = (n_jobs - base) < PER ? (n_jobs - base) : PER;
        SmallLinearJobPack pack;
        int max_N = 0;
        bool vec = true;
        for (int i = 0; i < n; i++) {
            pack.j[i] = jobs_host[base + i];
            const SmallLinearJob& j = pack.j[i];
            if (j.N > max_N) max_N = j.N;
            if ((j.N % 4) || (j.ldw % 4) || (j.n0 % 4) || ((reinterpret_cast<uintptr_t>(j.W) % 16) != 0)) vec = false;
        }
        for (int i = n; i < PER; i++) pack.j[i] = SmallLinearJob{nullptr, nullptr, nullptr, 0, 0, 0, nullptr, 0};
        if (max_N == 0) continue;
        if (M == 1) launch_small<1>(x, M, K_launch, K, pack, n, max_N, vec, act, st);
        else if (M == 2) launch_small<2>(x, M, K_launch, K, pack, n, max_N, vec, act, st);
        else if (M <= 4) launch_small<4>(x, M, K_launch, K, pack, n, max_N, vec, act, st);
        else launch_small<8>(x, M, K_launch, K, pack, n, max_N, vec, act, st);
        SD3_TRY(launch_status("small_linear"));
    }
    return SD3_OK;
}

}  // namespace sd3
