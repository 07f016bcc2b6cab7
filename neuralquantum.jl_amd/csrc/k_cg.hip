// Matrix-free SR: S v = (1/Ns) sum_s Oc(s) (Oc(s) . v) + shift, without S.
//
// Reference semantics: SrMatrixR (SR_notfull.jl:84-148): mul!(res, O, O' v)
// over the real and imaginary parts, res / N + shift v; solved by the
// iterative solvers of SRIterative.jl:71-152 (here conjugate gradients,
// sr_cg, with IterativeSolvers' relative-residual tolerance).
//
// The compact O rows Y (Ns x R, row per sample, P-order column blocks) hold
// block A = columns [0, nA) (the real parts) and block B = columns [nA, R)
// (the imaginary parts); column c belongs to parameter c (block A) or
// offB + c - nA (block B), so Re(Oc^H Oc) v = A^T (A v_A) + B^T (B v_B).
// One product:
//   k_sv      per workgroup, over its samples: w_A[s] = sum_{c < nA} Yc[s, c]
//             v[c], w_B[s] likewise over B, part[c] = sum_s Yc[s, c] w_blk(c)[s];
//   k_ytw_finish  q[k] = (sum of the workgroups' columns of k) / Ns
//             + shift(k) v[k].
// Yc = Y - mu (centred on the fly, FP64 arithmetic on FP32 or FP64 rows).
#include "nq_device.h"
#include "nq_kernels.h"

namespace {

// One product, one pass over Y: a workgroup takes RB rows of its samples at a time into registers
// (column t + 512 j in thread t), sums their products with v over the workgroup (RB rows, two blocks:
// one transposed wave reduction, one LDS exchange and barrier), and adds w_blk Yc to its columns' sums
// from the same registers while the next rows load.  Bound by HBM: 2 x Ns R bytes were read before, one
// pass for w = Yc v and one for Yc^T w (4x4 XYZ, FP64, 424 MB of rows: 122 + 128 us a product; now 79 us,
// 5.4 TB/s, and the sum over the workgroups 33 -> 12 us).
template <typename YT, int CT, int RB>
__global__ __launch_bounds__(512) void k_sv(const YT* Y, int64_t Ns, int R, int nA, int offB, const double* mu,
                                            const double* v, double* part) {
    __shared__ double red[2][8][8];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t per = (Ns + gridDim.x - 1) / gridDim.x;
    const int64_t s0 = (int64_t)blockIdx.x * per, s1 = (s0 + per < Ns) ? s0 + per : Ns;
    double vj[CT], mj[CT], acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int c = t + 512 * j;
        const bool in = c < R;
        vj[j] = in ? v[c < nA ? c : offB + c - nA] : 0.0;   // columns past R: 0 times a clamped load
        mj[j] = in ? mu[c] : 0.0;
        acc[j] = 0.0;
    }
    YT y[RB][CT], yn[RB][CT];
    auto load = [&](int64_t s, YT (&d)[RB][CT]) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const YT* row = Y + (s + r < s1 ? s + r : s1 - 1) * R;
#pragma unroll
            for (int j = 0; j < CT; ++j) d[r][j] = row[t + 512 * j < R ? t + 512 * j : R - 1];
        }
    };
    int buf = 0;
    if (s0 < s1) load(s0, y);
    for (int64_t s = s0; s < s1; s += RB, buf ^= 1) {
        load(s + RB < s1 ? s + RB : s, yn);
        double p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = 0.0;
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                const double x = ((double)y[r][j] - mj[j]) * vj[j];
                const bool first = t + 512 * j < nA;
                p[r] += first ? x : 0.0;
                p[4 + r] += first ? 0.0 : x;
            }
        const double tot = wave_totals<8>(p, lane);          // lane l: sum of p[l / 8]
        if ((lane & 7) == 0) red[buf][wave][lane >> 3] = tot;
        __syncthreads();
        double w = red[buf][lane >> 3][lane & 7];             // lane 8 wave + k, summed over the waves
        w += __shfl_xor(w, 8, 64);
        w += __shfl_xor(w, 16, 64);
        w += __shfl_xor(w, 32, 64);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const bool row = s + r < s1;
            const double wa = row ? rl_d(w, r) : 0.0, wb = row ? rl_d(w, 4 + r) : 0.0;
#pragma unroll
            for (int j = 0; j < CT; ++j)
                acc[j] += ((double)y[r][j] - mj[j]) * (t + 512 * j < nA ? wa : wb);
        }
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int j = 0; j < CT; ++j) y[r][j] = yn[r][j];
    }
#pragma unroll
    for (int j = 0; j < CT; ++j)
        if (t + 512 * j < R) part[(int64_t)blockIdx.x * R + t + 512 * j] = acc[j];
}

// q[k] = scale * (column sums of parameter k) + shift(k) v[k]; a parameter owns one column of A (k < nA),
// one of B (k >= offB, k - offB < nB) or both.  64 parameters per workgroup, the chunks over 16 thread
// groups (coalesced along the parameters), combined in a fixed order
__global__ __launch_bounds__(1024) void k_ytw_finish(const double* part, int chunks, int R, int nA, int offB, int np,
                                                     double scale, double eps, int kind, const double* diag,
                                                     const double* v, double* q) {
    __shared__ double red[16][64];
    const int x = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + x, nB = R - nA;
    const bool inA = k < np && k < nA, inB = k < np && k >= offB && k - offB < nB;
    double acc = 0.0;
    if (inA)
        for (int i = g; i < chunks; i += 16) acc += part[(int64_t)i * R + k];
    if (inB)
        for (int i = g; i < chunks; i += 16) acc += part[(int64_t)i * R + nA + (k - offB)];
    red[g][x] = acc;
    __syncthreads();
    if (g != 0 || k >= np) return;
    double sum = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum += red[i][x];
    double sh = 0.0;
    if (v) sh = ((kind == 0) ? eps : eps * diag[k]) * v[k];
    q[k] = scale * sum + sh;
}

// diag(S)[k] = (1/Ns) sum_s (sum over the columns of k of Yc[s, c]^2)
template <typename YT>
__global__ __launch_bounds__(256) void k_colsq(const YT* Y, int64_t Ns, int R, const double* mu, int chunks,
                                               double* part) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= R) return;
    const int64_t per = (Ns + chunks - 1) / chunks;
    const int64_t s0 = (int64_t)blockIdx.y * per, s1 = (s0 + per < Ns) ? s0 + per : Ns;
    const double m = mu[c];
    double acc = 0.0;
    for (int64_t s = s0; s < s1; ++s) {
        const double y = (double)Y[s * R + c] - m;
        acc += y * y;
    }
    part[(int64_t)blockIdx.y * R + c] = acc;
}

// out[slot] = sum_i x[i] y[i] (two stages: per-block partials, then one block)
__global__ __launch_bounds__(256) void k_dot_part(const double* x, const double* y, int n, double* part) {
    __shared__ double sh[4];
    double acc = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) acc += x[i] * y[i];
    acc = wave_total(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ __launch_bounds__(64) void k_dot_finish(const double* part, int nparts, double* out) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < nparts; i += 64) acc += part[i];
    acc = wave_total(acc);
    if (threadIdx.x == 0) *out = acc;
}

// CG scalars live in device memory: sc[0] = r.r, sc[1] = p.q, sc[2] = new r.r
// x += alpha p, r -= alpha q with alpha = sc[0] / sc[1]
__global__ __launch_bounds__(256) void k_cg_xr(double* x, double* r, const double* p, const double* q, int n,
                                               const double* sc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double alpha = sc[0] / sc[1];
    x[i] += alpha * p[i];
    r[i] -= alpha * q[i];
}

// p = r + beta p with beta = sc[2] / sc[0]
__global__ __launch_bounds__(256) void k_cg_p(double* p, const double* r, int n, const double* sc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    p[i] = r[i] + (sc[2] / sc[0]) * p[i];
}

__global__ void k_copy_scalar(const double* src, double* dst) { *dst = *src; }

// MINRES vectors (the Lanczos basis v and the directions w = V R^-1)
// y = a y
__global__ __launch_bounds__(256) void k_mr_scale(double* y, int n, double a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] *= a;
}

// v_next -= h v_prev (h on the host), then v_next -= sc[0] v_curr (the
// projection, on the device): the two orthogonalisations of one Lanczos step,
// the second applied by k_mr_orth after the dot product
__global__ __launch_bounds__(256) void k_mr_axpy(double* y, const double* x, int n, double a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += a * x[i];
}

__global__ __launch_bounds__(256) void k_mr_orth(double* vn, const double* vc, int n, const double* proj) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) vn[i] -= proj[0] * vc[i];
}

// v_next /= h4; w_next = (v_curr - h2 w_curr - h1 w_prev) / h3; x += rhs w_next
__global__ __launch_bounds__(256) void k_mr_step(double* vn, const double* vc, double* wn, const double* wc,
                                                 const double* wp, double* x, int n, double inv_h4, double h2,
                                                 double h1, double inv_h3, double rhs) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    vn[i] *= inv_h4;
    const double w = (vc[i] - h2 * wc[i] - h1 * wp[i]) * inv_h3;
    wn[i] = w;
    x[i] += rhs * w;
}

// LSQR: v *= inv_alfa (the new right vector); x += t1 w; w = v + t2 w
__global__ __launch_bounds__(256) void k_ls_step(double* v, double* w, double* x, int n, double inv_alfa, double t1,
                                                 double t2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double vi = v[i] * inv_alfa, wi = w[i];
    v[i] = vi;
    x[i] += t1 * wi;
    w[i] = vi + t2 * wi;
}

inline int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

hipError_t nq_launch_sv(const void* Y, int y_fp64, int64_t Ns, int R, int nA, int offB, int np, const double* mu,
                        const double* v, double eps, int kind, const double* diag, double* part, double* q,
                        hipStream_t st) {
    // one workgroup per CU; four rows at a time while they and the next four fit in the registers
    const int groups = (int)(Ns < 4 * NQ_SV_GROUPS ? (Ns + 3) / 4 : NQ_SV_GROUPS);
    const dim3 g(groups), b(512);
#define NQ_SV(CT, RB)                                                                                              \
    do {                                                                                                           \
        if (y_fp64) hipLaunchKernelGGL((k_sv<double, CT, RB>), g, b, 0, st, (const double*)Y, Ns, R, nA, offB, mu, v, part); \
        else hipLaunchKernelGGL((k_sv<float, CT, RB>), g, b, 0, st, (const float*)Y, Ns, R, nA, offB, mu, v, part);  \
    } while (0)
    if (R <= 1024) NQ_SV(2, 4);
    else if (R <= 2048) NQ_SV(4, 4);
    else if (R <= 3584) NQ_SV(7, 4);
    else if (R <= 6656) NQ_SV(13, 2);
    else return hipErrorInvalidValue;
#undef NQ_SV
    hipLaunchKernelGGL(k_ytw_finish, dim3(nblk(np, 64)), dim3(1024), 0, st, part, groups, R, nA, offB, np,
                       1.0 / (double)Ns, eps, kind, diag, v, q);
    return hipGetLastError();
}

hipError_t nq_launch_sdiag(const void* Y, int y_fp64, int64_t Ns, int R, int nA, int offB, int np, const double* mu,
                           double* part, int chunks, double* diag, hipStream_t st) {
    const dim3 g(nblk(R, 256), chunks);
    if (y_fp64)
        hipLaunchKernelGGL((k_colsq<double>), g, dim3(256), 0, st, (const double*)Y, Ns, R, mu, chunks, part);
    else
        hipLaunchKernelGGL((k_colsq<float>), g, dim3(256), 0, st, (const float*)Y, Ns, R, mu, chunks, part);
    // diag[k] = scale * column sums of k (the finish kernel without a shift term)
    hipLaunchKernelGGL(k_ytw_finish, dim3(nblk(np, 64)), dim3(1024), 0, st, part, chunks, R, nA, offB, np,
                       1.0 / (double)Ns, 0.0, 0, (const double*)nullptr, (const double*)nullptr, diag);
    return hipGetLastError();
}

hipError_t nq_launch_dot(const double* x, const double* y, int n, double* part, int nparts, double* out,
                         hipStream_t st) {
    hipLaunchKernelGGL(k_dot_part, dim3(nparts), dim3(256), 0, st, x, y, n, part);
    hipLaunchKernelGGL(k_dot_finish, dim3(1), dim3(64), 0, st, part, nparts, out);
    return hipGetLastError();
}

hipError_t nq_launch_cg_xr(double* x, double* r, const double* p, const double* q, int n, const double* sc,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_cg_xr, dim3(nblk(n, 256)), dim3(256), 0, st, x, r, p, q, n, sc);
    return hipGetLastError();
}

hipError_t nq_launch_cg_p(double* p, const double* r, int n, const double* sc, hipStream_t st) {
    hipLaunchKernelGGL(k_cg_p, dim3(nblk(n, 256)), dim3(256), 0, st, p, r, n, sc);
    return hipGetLastError();
}

hipError_t nq_launch_copy_scalar(const double* src, double* dst, hipStream_t st) {
    hipLaunchKernelGGL(k_copy_scalar, dim3(1), dim3(1), 0, st, src, dst);
    return hipGetLastError();
}

hipError_t nq_launch_mr_scale(double* y, int n, double a, hipStream_t st) {
    hipLaunchKernelGGL(k_mr_scale, dim3(nblk(n, 256)), dim3(256), 0, st, y, n, a);
    return hipGetLastError();
}

hipError_t nq_launch_mr_axpy(double* y, const double* x, int n, double a, hipStream_t st) {
    hipLaunchKernelGGL(k_mr_axpy, dim3(nblk(n, 256)), dim3(256), 0, st, y, x, n, a);
    return hipGetLastError();
}

hipError_t nq_launch_mr_orth(double* vn, const double* vc, int n, const double* proj, hipStream_t st) {
    hipLaunchKernelGGL(k_mr_orth, dim3(nblk(n, 256)), dim3(256), 0, st, vn, vc, n, proj);
    return hipGetLastError();
}

hipError_t nq_launch_mr_step(double* vn, const double* vc, double* wn, const double* wc, const double* wp, double* x,
                             int n, double inv_h4, double h2, double h1, double inv_h3, double rhs, hipStream_t st) {
    hipLaunchKernelGGL(k_mr_step, dim3(nblk(n, 256)), dim3(256), 0, st, vn, vc, wn, wc, wp, x, n, inv_h4, h2, h1,
                       inv_h3, rhs);
    return hipGetLastError();
}

hipError_t nq_launch_ls_step(double* v, double* w, double* x, int n, double inv_alfa, double t1, double t2,
                             hipStream_t st) {
    hipLaunchKernelGGL(k_ls_step, dim3(nblk(n, 256)), dim3(256), 0, st, v, w, x, n, inv_alfa, t1, t2);
    return hipGetLastError();
}
