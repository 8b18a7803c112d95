// Sparse linear algebra for gfx950: CSR SpMV (several lanes per row, wave64 reductions), dot
// products with fixed-order two-stage reductions, multicolour ILU(0), the SA-AMG V-cycle and the
// Krylov solvers of src/cfa/linalg.cuh.
//
// Krylov design: the reference copies every dot product to the host (three blocking transfers
// per CG iteration, linalg.cuh:172-177). Here all scalars stay on the device: a one-workgroup
// "final" kernel reduces the block partials in a fixed order and applies the scalar logic of the
// reference (coefficients, breakdown guards, stopping rules), and the iteration counter lives on
// the device too. Every vector kernel reads a device state word and returns at once when the
// solve has stopped. One iteration is therefore the same kernel sequence every time: it is
// captured once as a HIP graph and replayed (about 1.7 us per kernel node on MI355X against
// 2.5 us per stream launch), with the host a few iterations ahead, following a progress word
// that the final kernels write to mapped pinned memory, so the queue never drains.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <type_traits>
#include <vector>

#include "cfa_device.hpp"

using namespace cfa_dev;

namespace {

constexpr int RED_BLOCKS = 1024;   // partial sums per reduction (grid-stride kernels)
constexpr int OP_BLOCKS = 4096;    // partials that one segment of the workspace holds
constexpr int LOOKAHEAD = 3;       // iterations enqueued ahead of the last one known to have finished
constexpr int GRAPH_CACHE = 4;     // captured iteration graphs kept per solver kind

// Solve state (device ints after the scalar area of the workspace)
enum { ST_RUNNING = 0, ST_CONVERGED = 1, ST_STOPPED = 2, ST_TRIVIAL = 3 };

__device__ __forceinline__ bool halted(const int* state) { return state && state[0] != ST_RUNNING; }

// Loads a row's range [k0, k1) and the solve state together and reports whether the solve runs:
// both loads are in flight at once, so the state word does not add a round trip in front of the
// row's loads (measured: 0.25-0.3 us of a 3-4.4 us sweep on 18k-115k rows). The empty asm
// statement makes the three values complete before the early exit.
// Rows past the end get the empty range [ptr[rows], ptr[rows]); the loads are unconditional (and
// in bounds: ptr has rows + 1 entries) so that no branch separates them.
__device__ __forceinline__ bool running_with_range(const int* __restrict__ ptr, int row, int rows,
                                                   const int* __restrict__ state, int& k0, int& k1) {
    const int r = row < rows ? row : rows;
    k0 = ptr[r];
    k1 = ptr[r + (row < rows ? 1 : 0)];
    const int sv = state ? state[0] : ST_RUNNING;
    asm volatile("" ::"v"(k0), "v"(k1), "s"(sv));
    return sv == ST_RUNNING;
}

__device__ __forceinline__ void publish(int* status, int progress, int state) {
    if (!status) return;
    __hip_atomic_store(&status[1], state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&status[0], progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---- CSR products --------------------------------------------------------------------------------
enum CsrOp { OP_SPMV, OP_ADD, OP_RESID, OP_JACOBI };

// y = A x | y += A x | y = b - A x | y = x + omega dinv (b - A x)   (src/cfa/linalg.cuh:884-901).
// T = double, or float for the mixed-precision cycle (values, vectors and arithmetic in FP32).
template <int TPR, int OP, typename T = double>
__global__ void __launch_bounds__(BLOCK)
k_csr_op(int rows, const int* __restrict__ rp, const int* __restrict__ ci, const T* __restrict__ val,
         const T* __restrict__ x, const T* __restrict__ b, const T* __restrict__ dinv, T omega, T* __restrict__ y,
         const int* __restrict__ state) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = g / TPR, lane = g % TPR;
    int k0, k1;
    if (!running_with_range(rp, row, rows, state, k0, k1)) return;
    T s = 0;
    row_entries<TPR>(ci, val, k0, k1, lane, [&](T a, int j) { s += a * x[j]; });
    s = group_sum<TPR>(s);
    if (row >= rows || lane != 0) return;
    if (OP == OP_SPMV) y[row] = s;
    else if (OP == OP_ADD) y[row] += s;
    else if (OP == OP_RESID) y[row] = b[row] - s;
    else y[row] = x[row] + omega * dinv[row] * (b[row] - s);
}

// First two steps of the V-cycle smoother fused: x0 = omega dinv b (src/cfa/linalg.cuh:864-868),
// y = x0 + omega dinv (b - A x0), with x0 formed on the fly from b and dinv at the neighbours.
template <int TPR, typename T = double>
__global__ void __launch_bounds__(BLOCK)
k_jacobi_from_zero(int rows, const int* __restrict__ rp, const int* __restrict__ ci, const T* __restrict__ val,
                   const T* __restrict__ b, const T* __restrict__ dinv, T omega, T* __restrict__ y,
                   const int* __restrict__ state) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = g / TPR, lane = g % TPR;
    int k0, k1;
    if (!running_with_range(rp, row, rows, state, k0, k1)) return;
    T s = 0;
    row_entries<TPR>(ci, val, k0, k1, lane, [&](T a, int j) { s += a * (omega * dinv[j] * b[j]); });
    s = group_sum<TPR>(s);
    if (row >= rows || lane != 0) return;
    const T x0 = omega * dinv[row] * b[row];
    y[row] = x0 + omega * dinv[row] * (b[row] - s);
}

template <typename T = double>
__global__ void k_jacobi_init(int n, T omega, const T* __restrict__ dinv, const T* __restrict__ b, T* __restrict__ x,
                              const int* __restrict__ state) {
    if (halted(state)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = omega * dinv[i] * b[i];
}

// The lane's share of one row of a dense product, its loads eight at a time ahead of their uses
template <typename T>
__device__ __forceinline__ double dense_row(int n, const double* __restrict__ a, const T* __restrict__ x, int lane) {
    double s = 0.0;
#pragma unroll 8
    for (int j = lane; j < n; j += WAVE) s += a[j] * (double)x[j];
    return s;
}

// y = Ainv x with the dense coarse inverse, one wavefront per row (src/cfa/linalg.cuh:929-937);
// FP64 arithmetic also when x and y are FP32 (the coarse solve stays FP64 in the mixed cycle)
template <typename T = double>
__global__ void __launch_bounds__(BLOCK)
k_dense_matvec(int n, const double* __restrict__ A, const T* __restrict__ x, T* __restrict__ y,
               const int* __restrict__ state) {
    if (halted(state)) return;
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE, lane = threadIdx.x & (WAVE - 1);
    const double s = i < n ? wave_sum(dense_row(n, A + (size_t)i * n, x, lane)) : 0.0;
    if (i < n && lane == 0) y[i] = (T)s;
}

// Level data of the double or the float cycle
template <typename T> struct Lv;
template <> struct Lv<double> {
    __host__ __device__ static const double* a(const cfa_amg_level_t& L) { return L.a_v; }
    __host__ __device__ static const double* p(const cfa_amg_level_t& L) { return L.p_v; }
    __host__ __device__ static const double* r(const cfa_amg_level_t& L) { return L.r_v; }
    __host__ __device__ static const double* dinv(const cfa_amg_level_t& L) { return L.dinv; }
    __host__ __device__ static const double* sv(const cfa_amg_level_t& L) { return L.s_v; }
    static const double* w(const cfa_amg_level_t& L) { return L.w_v; }
    static const double* q(const cfa_amg_level_t& L) { return L.q_v; }
    __host__ __device__ static double* x(const cfa_amg_level_t& L) { return L.x; }
    __host__ __device__ static double* b(const cfa_amg_level_t& L) { return L.b; }
    __host__ __device__ static double* res(const cfa_amg_level_t& L) { return L.r; }
    __host__ __device__ static double* ax(const cfa_amg_level_t& L) { return L.ax; }
    static double* cb(const cfa_amg_t* a) { return a->cb; }
    static double* cx(const cfa_amg_t* a) { return a->cx; }
};
template <> struct Lv<float> {
    __host__ __device__ static const float* a(const cfa_amg_level_t& L) { return L.a_v32; }
    __host__ __device__ static const float* p(const cfa_amg_level_t& L) { return L.p_v32; }
    __host__ __device__ static const float* r(const cfa_amg_level_t& L) { return L.r_v32; }
    __host__ __device__ static const float* dinv(const cfa_amg_level_t& L) { return L.dinv32; }
    __host__ __device__ static const float* sv(const cfa_amg_level_t& L) { return L.s_v32; }
    static const float* w(const cfa_amg_level_t& L) { return L.w_v32; }
    static const float* q(const cfa_amg_level_t& L) { return L.q_v32; }
    __host__ __device__ static float* x(const cfa_amg_level_t& L) { return L.x32; }
    __host__ __device__ static float* b(const cfa_amg_level_t& L) { return L.b32; }
    __host__ __device__ static float* res(const cfa_amg_level_t& L) { return L.r32; }
    __host__ __device__ static float* ax(const cfa_amg_level_t& L) { return L.ax32; }
    static float* cb(const cfa_amg_t* a) { return a->cb32; }
    static float* cx(const cfa_amg_t* a) { return a->cx32; }
};

// ---- reductions ------------------------------------------------------------------------------------
// partial[b] = sum over the block's grid-stride share of x . y
__global__ void __launch_bounds__(BLOCK)
k_dot_partial(int n, const double* __restrict__ x, const double* __restrict__ y, double* __restrict__ part,
              const int* __restrict__ state) {
    __shared__ double lds[BLOCK / WAVE];
    if (halted(state)) return;
    double acc = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) acc += x[i] * y[i];
    acc = block_sum(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

__global__ void k_sum_to(int nb, const double* __restrict__ part, double* __restrict__ out, int take_sqrt) {
    __shared__ double lds[BLOCK / WAVE];
    const double s = sum_partials(part, nb, 1, lds);
    if (threadIdx.x == 0) *out = take_sqrt ? sqrt(s) : s;
}

// Workgroups of a vector kernel that leaves partial sums: every workgroup of the consumer reads them
// all again, so vectors that one workgroup per CU can stream (up to 2^20 entries) get no more than
// that, longer ones RED_BLOCKS for the bytes in flight. Time steps with 256 / 512 / 1024 workgroups at
// most on such vectors: 4.97 / 4.97 / 5.02 ms on 115k nodes, 15.6 / 15.8 / 15.8 ms on 461k.
inline int red_blocks(long long n) {
    return std::min(blocks_for(n > 0 ? n : 1), n <= (1 << 20) ? RED_BLOCKS / 4 : RED_BLOCKS);
}

// ---- elementwise ------------------------------------------------------------------------------------
__global__ void k_axpy(int n, double a, const double* __restrict__ x, double* __restrict__ y) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += a * x[i];
}
__global__ void k_xpay(int n, const double* __restrict__ x, double b, double* __restrict__ y) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = x[i] + b * y[i];
}
__global__ void k_vec_mul(int n, const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out,
                          const int* __restrict__ state) {
    if (halted(state)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] * b[i];
}
__global__ void k_fill_zero(int n, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = 0.0;
}
__global__ void k_copy(int n, const double* __restrict__ a, double* __restrict__ out, const int* __restrict__ state) {
    if (halted(state)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i];
}
// inverse diagonal, 1 where |d| <= eps (src/cfa/linalg.cuh:28-48 with eps 1e-14, :871-878 with
// eps 1e-300; a missing diagonal counts as 1 resp. 0, both giving 1)
__global__ void k_inv_diag(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                           const double* __restrict__ val, double eps, double* __restrict__ inv) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double d = eps > 1.0e-100 ? 1.0 : 0.0;
    for (int k = rp[i]; k < rp[i + 1]; ++k)
        if (ci[k] == i) { d = val[k]; break; }
    inv[i] = (fabs(d) > eps) ? (1.0 / d) : 1.0;
}

template <int TPR, int NRHS>
__global__ void __launch_bounds__(BLOCK)
k_spmv_multi(int n, const int* __restrict__ rp, const int* __restrict__ ci, const double* __restrict__ val,
             const double* __restrict__ x, double* __restrict__ y) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = g / TPR, lane = g % TPR;
    double s[NRHS];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) s[c] = 0.0;
    if (row < n)
        row_entries<TPR>(ci, val, rp[row], rp[row + 1], lane, [&](double a, int j) {
#pragma unroll
            for (int c = 0; c < NRHS; ++c) s[c] += a * x[(size_t)c * n + j];
        });
#pragma unroll
    for (int c = 0; c < NRHS; ++c) s[c] = group_sum<TPR>(s[c]);
    if (row < n && lane == 0)
#pragma unroll
        for (int c = 0; c < NRHS; ++c) y[(size_t)c * n + row] = s[c];
}

// ======================================================================================================
// PCG (src/cfa/linalg.cuh:183-256)
// ======================================================================================================
enum { S_BNORM = 0, S_RZ_OLD, S_PQ, S_ALPHA, S_RNORM, S_REL, S_BETA, S_TOL };
// ints: [0] state, [1] final iteration count, [2] current iteration

// Start of a solve from the b.b and r.r partials: ||b||, x = 0 and stop when ||b|| < 1e-14
// (linalg.cuh:205-209, the caller's k_zero_if_trivial), converged with 0 iterations when ||r|| < tol ||b||
// (linalg.cuh:217-218); the tolerance and the "not computed" relative residual -1
__global__ void k_pcg_init(int nb, const double* __restrict__ part_b, const double* __restrict__ part_r, double tol,
                           double* __restrict__ sc, int* __restrict__ st, int* __restrict__ status) {
    __shared__ double lds[2 * BLOCK / WAVE];
    double s[2];
    sum_partials_k<2>({part_b, part_r}, {nb, nb}, 1, s, lds);
    if (threadIdx.x != 0) return;
    const double b_norm = sqrt(s[0]);
    sc[S_BNORM] = b_norm;
    sc[S_TOL] = tol;
    sc[S_REL] = -1.0;
    st[1] = 0;
    st[2] = 0;
    const int state = b_norm < 1.0e-14 ? ST_TRIVIAL : sqrt(s[1]) < tol * b_norm ? ST_CONVERGED : ST_RUNNING;
    st[0] = state;
    publish(status, 0, state);
}

// The solve's outcome in the pinned status words [2..7]: state, iterations, relative residual(s) (as
// two words each), read by the host after it has waited for the stream
__device__ __forceinline__ void publish_double(int* status, double v) {
    const unsigned long long b = __double_as_longlong(v);
    __hip_atomic_store(&status[0], (int)(unsigned)b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&status[1], (int)(unsigned)(b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
double published_double(const volatile int* status) {
    const unsigned long long b = (unsigned)status[0] | ((unsigned long long)(unsigned)status[1] << 32);
    double v;
    std::memcpy(&v, &b, sizeof(v));
    return v;
}
__global__ void k_pcg_outcome(const double* __restrict__ sc, const int* __restrict__ st, int* __restrict__ status) {
    __hip_atomic_store(&status[2], st[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&status[3], st[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    publish_double(status + 4, sc[S_REL]);
}

__global__ void k_pcg_start(int* __restrict__ st) { st[0] = ST_RUNNING; }

__global__ void k_zero_if_trivial(int n, double* __restrict__ x, const int* __restrict__ st) {
    if (st[0] != ST_TRIVIAL) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = 0.0;
}

// r = b - q; partials b.b and r.r
__global__ void __launch_bounds__(BLOCK)
k_pcg_residual(int n, const double* __restrict__ b, const double* __restrict__ q, double* __restrict__ r,
               double* __restrict__ part_b, double* __restrict__ part_r) {
    __shared__ double lds[2 * BLOCK / WAVE];
    double acc[2] = {0.0, 0.0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const double bi = b[i], ri = bi + (-1.0) * q[i];
        r[i] = ri;
        acc[0] += bi * bi;
        acc[1] += ri * ri;
    }
    block_sum_k<2>(acc, lds);
    if (threadIdx.x == 0) {
        part_b[blockIdx.x] = acc[0];
        part_r[blockIdx.x] = acc[1];
    }
}

// alpha = rz_old / (p.q); breakdown when |p.q| < 1e-30
__global__ void k_pcg_final_alpha(int nb, const double* __restrict__ part, double* __restrict__ sc,
                                  int* __restrict__ st, int* __restrict__ status) {
    __shared__ double lds[BLOCK / WAVE];
    if (st[0] != ST_RUNNING) return;
    const double pq = sum_partials(part, nb, 1, lds);
    if (threadIdx.x != 0) return;
    sc[S_PQ] = pq;
    if (fabs(pq) < 1.0e-30) {
        st[0] = ST_STOPPED;
        st[1] = st[2];
        publish(status, st[2], ST_STOPPED);
        return;
    }
    sc[S_ALPHA] = sc[S_RZ_OLD] / pq;
}

// x += alpha p; r -= alpha q; partial r.r
__global__ void __launch_bounds__(BLOCK)
k_pcg_update_xr(int n, const double* __restrict__ sc, const double* __restrict__ p, const double* __restrict__ q,
                double* __restrict__ x, double* __restrict__ r, double* __restrict__ part, const int* __restrict__ st) {
    __shared__ double lds[BLOCK / WAVE];
    if (halted(st)) return;
    const double alpha = sc[S_ALPHA];
    double acc = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        x[i] += alpha * p[i];
        const double ri = r[i] + (-alpha) * q[i];
        r[i] = ri;
        acc += ri * ri;
    }
    acc = block_sum(acc, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// ||r|| < tol ||b|| -> converged after it + 1 iterations
__global__ void k_pcg_final_rnorm(int nb, const double* __restrict__ part, double* __restrict__ sc,
                                  int* __restrict__ st, int* __restrict__ status) {
    __shared__ double lds[BLOCK / WAVE];
    if (st[0] != ST_RUNNING) return;
    const double rr = sum_partials(part, nb, 1, lds);
    if (threadIdx.x != 0) return;
    const double r_norm = sqrt(rr);
    sc[S_RNORM] = r_norm;
    sc[S_REL] = r_norm / sc[S_BNORM];
    if (r_norm < sc[S_TOL] * sc[S_BNORM]) {
        st[0] = ST_CONVERGED;
        st[1] = st[2] + 1;
        publish(status, st[2] + 1, ST_CONVERGED);
    }
}

// beta = rz_new / (rz_old + 1e-30); rz_old = rz_new; next iteration (first: prologue, rz only)
__global__ void k_pcg_final_beta(int nb, const double* __restrict__ part, double* __restrict__ sc,
                                 int* __restrict__ st, int* __restrict__ status, int first) {
    __shared__ double lds[BLOCK / WAVE];
    if (st[0] != ST_RUNNING) return;
    const double rz = sum_partials(part, nb, 1, lds);
    if (threadIdx.x != 0) return;
    if (!first) {
        sc[S_BETA] = rz / (sc[S_RZ_OLD] + 1.0e-30);
        st[2] += 1;
    }
    sc[S_RZ_OLD] = rz;
    publish(status, st[2], ST_RUNNING);
}

// p = z + beta p
__global__ void k_pcg_p(int n, const double* __restrict__ z, const double* __restrict__ sc, double* __restrict__ p,
                        const int* __restrict__ st) {
    if (halted(st)) return;
    const double beta = sc[S_BETA];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = z[i] + beta * p[i];
}

// ---- Row runs through LDS ------------------------------------------------------------------------
// The entries of RB consecutive rows are one contiguous run of a CSR matrix. A workgroup loads such a
// run coalesced, every lane's column indices, values and gathers in flight together, leaves the
// products in LDS, and a lane per row and value array adds the row's products in CSR order. With
// lanes per row instead, one load instruction of a wavefront touches the entries of 32 rows scattered
// over 1.8 KB, and the operator's kernels (three and two value arrays) ran at 2.2-2.9 TB/s.
constexpr int RUN_SLOTS(int RB) { return RB / 32; }              // entries per lane and tile
constexpr int RUN_TILE(int RB) { return RUN_SLOTS(RB) * BLOCK; }   // 8 entries per row

template <int RB, int NV>
struct RunTile {
    int c[RUN_SLOTS(RB)];
    double v[RUN_SLOTS(RB)][NV];
    __device__ __forceinline__ void load(const int* __restrict__ ci, const RowValues<NV, double>& vals, int t, int end) {
#pragma unroll
        for (int u = 0; u < RUN_SLOTS(RB); ++u) {
            const int k = t + u * BLOCK + (int)threadIdx.x;
            const bool ok = k < end;
            c[u] = ok ? ci[k] : 0;
#pragma unroll
            for (int m = 0; m < NV; ++m) v[u][m] = ok ? vals.p[m][k] : 0.0;
        }
    }
};

// Adds the tile's products of the lane's row (entries k0..k1 of the run, tile from t) to acc, for the
// value arrays of the lane's part of the workgroup (BLOCK / RB parts, array m with part m mod parts)
template <int RB, int NV>
__device__ __forceinline__ void run_row_sums(const double* __restrict__ prod, int t, int k0, int k1, double (&acc)[NV]) {
    constexpr int PARTS = BLOCK / RB;
    const int part = threadIdx.x / RB;
    const int a = max(k0, t) - t, b = min(k1, t + RUN_TILE(RB)) - t;
#pragma unroll
    for (int m = 0; m < NV; ++m) {
        if (m % PARTS != part) continue;
        for (int k = a; k < b; ++k) acc[m] += prod[m * RUN_TILE(RB) + k];
    }
}
template <int RB>
__device__ __forceinline__ bool run_part_has(int m) { return m % (BLOCK / RB) == (int)threadIdx.x / RB; }

// Fused operator, stage 1: q = Kp p (CSR) and g = M^-1 B p, all on the same row pattern
template <int RB>
__global__ void __launch_bounds__(BLOCK)
k_apply_K_B(int n, const int* __restrict__ rp, const int* __restrict__ ci, const double* __restrict__ val,
            const double* __restrict__ oss, const double* __restrict__ inv_m, const double* __restrict__ in,
            double* __restrict__ q, double* __restrict__ gx, double* __restrict__ gy, const int* __restrict__ st) {
    __shared__ double prod[3 * RUN_TILE(RB)];
    if (halted(st)) return;
    const RowValues<3, double> kb{{val, oss, oss + (size_t)rp[n]}};
    for (int r0 = blockIdx.x * RB; r0 < n; r0 += gridDim.x * RB) {
        const int row = r0 + (int)threadIdx.x % RB, e0 = rp[r0], e1 = rp[min(r0 + RB, n)];
        const int k0 = row < n ? rp[row] : e1, k1 = row < n ? rp[row + 1] : e1;
        double s[3] = {0.0, 0.0, 0.0};
        for (int t = e0; t < e1; t += RUN_TILE(RB)) {
            RunTile<RB, 3> tile;
            tile.load(ci, kb, t, e1);
#pragma unroll
            for (int u = 0; u < RUN_SLOTS(RB); ++u) {
                const double xj = in[tile.c[u]];
#pragma unroll
                for (int m = 0; m < 3; ++m) prod[m * RUN_TILE(RB) + u * BLOCK + threadIdx.x] = tile.v[u][m] * xj;
            }
            __syncthreads();
            run_row_sums<RB, 3>(prod, t, k0, k1, s);
            __syncthreads();
        }
        if (row >= n) continue;
        if (run_part_has<RB>(0)) q[row] = s[0];
        if (run_part_has<RB>(1)) gx[row] = s[1] * inv_m[row];
        if (run_part_has<RB>(2)) gy[row] = s[2] * inv_m[row];
    }
}

// Fused operator, stage 2: q -= B^T g on non-Dirichlet rows; partial p.q per block. The grid is
// capped (grid-stride over row runs) so that the consumers' re-summation stays short.
template <int RB>
__global__ void __launch_bounds__(BLOCK)
k_apply_BT_dot(int n, const int* __restrict__ rp, const int* __restrict__ ci,
               const double* __restrict__ oss, const int* __restrict__ tag, OutletMode om,
               const double* __restrict__ gx, const double* __restrict__ gy, const double* __restrict__ p,
               double* __restrict__ q, double* __restrict__ part, const int* __restrict__ st) {
    __shared__ double prod[RUN_TILE(RB)];
    __shared__ double lds[BLOCK / WAVE];
    if (halted(st)) return;
    const size_t nnz = (size_t)rp[n];
    const RowValues<2, double> bt{{oss + 2 * nnz, oss + 3 * nnz}};
    double contrib = 0.0;
    for (int r0 = blockIdx.x * RB; r0 < n; r0 += gridDim.x * RB) {
        const int row = r0 + (int)threadIdx.x, e0 = rp[r0], e1 = rp[min(r0 + RB, n)];
        const bool own = (int)threadIdx.x < RB && row < n;
        const int k0 = own ? rp[row] : e1, k1 = own ? rp[row + 1] : e1;
        const double qi0 = own ? q[row] : 0.0, pi = own ? p[row] : 0.0;
        const int ti = own ? tag[row] : 0;
        double s[1] = {0.0};
        for (int t = e0; t < e1; t += RUN_TILE(RB)) {
            RunTile<RB, 2> tile;
            tile.load(ci, bt, t, e1);
#pragma unroll
            for (int u = 0; u < RUN_SLOTS(RB); ++u) {
                const int j = tile.c[u];
                prod[u * BLOCK + threadIdx.x] = tile.v[u][0] * gx[j] + tile.v[u][1] * gy[j];
            }
            __syncthreads();
            if (own) run_row_sums<RB, 1>(prod, t, k0, k1, s);
            __syncthreads();
        }
        if (!own) continue;
        double qi = qi0;
        if (!pressure_dirichlet(row, ti, om)) {
            qi -= s[0];
            q[row] = qi;
        }
        contrib += pi * qi;
    }
    contrib = block_sum(contrib, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = contrib;
}

// ======================================================================================================
// PCG with the scalar reductions folded into the kernels that consume them
// ======================================================================================================
// A kernel that needs a scalar (beta, alpha, the residual test) sums its producer's block
// partials itself, in the same fixed order in every block, so all blocks reach the same value
// and the same decision without a separate one-workgroup kernel; only block 0 writes the state
// words. The search direction alternates between two buffers so that the operator kernel can
// form p_k = z_k + beta_{k-1} p_{k-1} on the fly while it applies the operator (the reference's
// separate k_xpay, linalg.cuh:252). r.z partials alternate between two buffers as well: the
// operator of iteration k reads r_k.z_k and r_{k-1}.z_{k-1}, while the preconditioner of the same
// iteration writes r_{k+1}.z_{k+1} over the older one.
enum { ST_CAPPED = 4 };

struct PcgArgs {
    int n, max_iter;
    const int* rp; const int* ci; const double* val;
    const double* oss; const double* inv_m; const int* tag; double* gx; double* gy;
    OutletMode om;
    double* x; double* r; double* z; double* q; double* p[2];
    double* rbuf[2];   // residual by parity: r and the merged update's second buffer
    double* prz[2]; double* ppq; double* prr;
    int nb_rz, nb_rr;
    const double* inv_diag;
    double* sc; int* st; int* status;
};

// Operator of iteration k (parity h): p_k formed on the fly and stored to p[h]; q = Kp p_k, and
// with OSS g = M^-1 B p_k for the second stage, else the p.q partials here. Iteration cap check.
// Row runs through LDS; the first run's entries and both gathers are loaded before the barrier of
// the r.z sums, so the sums and the state word cost no round trip of their own.
template <int RB, bool OSS>
__global__ void __launch_bounds__(BLOCK)
k_fp_operator(PcgArgs a, int h) {
    constexpr int NV = OSS ? 3 : 1, U = RUN_SLOTS(RB), TILE = RUN_TILE(RB);
    __shared__ double prod[NV * TILE];
    __shared__ double lds[2 * BLOCK / WAVE];
    __shared__ int lds_st[2];
    const double* __restrict__ z = a.z;
    const double* __restrict__ po = a.p[1 - h];
    double* __restrict__ pn = a.p[h];
    const int* __restrict__ rp = a.rp;
    const int* __restrict__ ci = a.ci;
    RowValues<NV, double> kb;
    kb.p[0] = a.val;
    if constexpr (OSS) {
        kb.p[1] = a.oss;
        kb.p[2] = a.oss + (size_t)a.rp[a.n];
    }
    RunTile<RB, NV> tile;
    double zj[U], pj[U], zi = 0.0, pi = 0.0;
    int row, e0, e1, k0, k1;
    auto load_tile = [&](int t) {
        tile.load(ci, kb, t, e1);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            zj[u] = z[tile.c[u]];
            pj[u] = po[tile.c[u]];
        }
    };
    auto load_run = [&](int r0) {
        row = r0 + (int)threadIdx.x % RB;
        e0 = rp[r0];
        e1 = rp[min(r0 + RB, a.n)];
        load_tile(e0);
        k0 = row < a.n ? rp[row] : e1;
        k1 = row < a.n ? rp[row + 1] : e1;
        if (row < a.n) {
            zi = z[row];
            pi = po[row];
        }
    };
    int r0 = blockIdx.x * RB;   // the grid has no empty workgroups
    load_run(r0);
    double rz[2];   // r_k.z_k, r_{k-1}.z_{k-1}
    sum_partials_k<2, 2>({a.prz[h], a.prz[1 - h]}, {a.nb_rz, a.nb_rz}, 1, rz, lds, a.st, lds_st);
    const int it = lds_st[1];
    if (lds_st[0] != ST_RUNNING) return;
    if (it >= a.max_iter) {
        if (blockIdx.x == 0 && threadIdx.x == 0) { a.st[0] = ST_CAPPED; publish(a.status, it, ST_CAPPED); }
        return;
    }
    const bool first = it == 0;   // p and r_{k-1}.z_{k-1} are not set yet
    const double beta = first ? 0.0 : rz[0] / (rz[1] + 1.0e-30);
    double contrib = 0.0;
    for (;;) {
        double s[NV];
#pragma unroll
        for (int m = 0; m < NV; ++m) s[m] = 0.0;
        for (int t = e0;;) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double xj = first ? zj[u] : fma(beta, pj[u], zj[u]);
#pragma unroll
                for (int m = 0; m < NV; ++m) prod[m * TILE + u * BLOCK + threadIdx.x] = tile.v[u][m] * xj;
            }
            __syncthreads();
            run_row_sums<RB, NV>(prod, t, k0, k1, s);
            __syncthreads();
            t += TILE;
            if (t >= e1) break;
            load_tile(t);
        }
        if (row < a.n) {
            if (run_part_has<RB>(0)) {
                const double p = first ? zi : fma(beta, pi, zi);
                pn[row] = p;
                a.q[row] = s[0];
                if (!OSS) contrib += p * s[0];
            }
            if constexpr (OSS) {
                if (run_part_has<RB>(1)) a.gx[row] = s[1] * a.inv_m[row];
                if (run_part_has<RB>(2)) a.gy[row] = s[2] * a.inv_m[row];
            }
        }
        r0 += gridDim.x * RB;
        if (r0 >= a.n) break;
        load_run(r0);
    }
    if (!OSS) {
        contrib = block_sum(contrib, lds);
        if (threadIdx.x == 0) a.ppq[blockIdx.x] = contrib;
    }
}

// alpha = r_k.z_k / (p_k.q) with the breakdown guard, x += alpha p, r -= alpha q, r.r partials;
// the completed-iteration counter advances here.
__global__ void __launch_bounds__(BLOCK)
k_fp_update(PcgArgs a, int h, int nb_pq) {
    __shared__ double lds[2 * BLOCK / WAVE], lds_rr[BLOCK / WAVE];
    __shared__ int word[2];
    const double* __restrict__ p = a.p[h];
    const double* __restrict__ q = a.q;
    double* __restrict__ x = a.x;
    double* __restrict__ r = a.r;
    int i = blockIdx.x * BLOCK + threadIdx.x;
    double xi = 0.0, pi = 0.0, qi = 0.0, ri = 0.0;
    auto load = [&] {
        if (i >= a.n) return;
        xi = x[i];
        pi = p[i];
        qi = q[i];
        ri = r[i];
    };
    load();   // beside the sums
    double sums[2];   // p.q, r.z
    sum_partials_k<2, 2>({a.ppq, a.prz[h]}, {nb_pq, a.nb_rz}, 1, sums, lds, a.st, word);
    const int it = word[1];
    if (word[0] != ST_RUNNING) return;
    const double pq = sums[0];
    if (fabs(pq) < 1.0e-30) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            a.st[0] = ST_STOPPED;
            a.st[1] = it;
            publish(a.status, it, ST_STOPPED);
        }
        return;
    }
    const double alpha = sums[1] / pq;
    double acc = 0.0;
    while (i < a.n) {
        x[i] = xi + alpha * pi;
        const double rn = ri + (-alpha) * qi;
        r[i] = rn;
        acc += rn * rn;
        i += gridDim.x * BLOCK;
        load();
    }
    acc = block_sum(acc, lds_rr);
    if (threadIdx.x == 0) {
        a.prr[blockIdx.x] = acc;
        if (blockIdx.x == 0) a.st[2] = it + 1;
    }
}

// Residual test of the iteration (||r|| < tol ||b||, linalg.cuh:241-247) from the r.r partials, with
// the state word; true (in every thread of every block) when the solve goes on. Kernels compute their
// rows before it, so that its round trip runs beside theirs. lds: BLOCK / WAVE doubles.
__device__ __forceinline__ bool residual_test_running(const double* prr, int nb_rr, double* sc, int* st, int* status,
                                                      double* lds, int* lds_state) {
    const double bnorm = sc[S_BNORM], limit = sc[S_TOL] * bnorm;
    double rr[1];
    sum_partials_k<1, 1>({prr}, {nb_rr}, 1, rr, lds, st, lds_state);
    if (*lds_state != ST_RUNNING) return false;
    const double r_norm = sqrt(rr[0]);
    const bool done = r_norm < limit;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc[S_RNORM] = r_norm;
        sc[S_REL] = r_norm / bnorm;
        const int it = st[2];
        if (done) {
            st[0] = ST_CONVERGED;
            st[1] = it;
        }
        publish(status, it, done ? ST_CONVERGED : ST_RUNNING);
    }
    return !done;
}

// One-workgroup residual test, for preconditioners whose first kernel cannot take it
__global__ void k_fp_check(const double* prr, int nb_rr, double* sc, int* st, int* status) {
    __shared__ double lds[BLOCK / WAVE];
    __shared__ int word;
    (void)residual_test_running(prr, nb_rr, sc, st, status, lds, &word);
}

// First two V-cycle sweeps from x = 0 on level 0 (as k_jacobi_from_zero), preceded by the
// residual test of the iteration.
template <int TPR>
__global__ void __launch_bounds__(BLOCK)
k_jacobi_from_zero_check(int rows, const int* __restrict__ rp, const int* __restrict__ ci,
                         const double* __restrict__ val, const double* __restrict__ b,
                         const double* __restrict__ dinv, double omega, double* __restrict__ y,
                         const double* __restrict__ prr, int nb_rr, double* sc, int* st, int* status) {
    __shared__ double lds[BLOCK / WAVE];
    __shared__ int word;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = g / TPR, lane = g % TPR;
    double s = 0.0;
    if (row < rows)
        row_entries<TPR>(ci, val, rp[row], rp[row + 1], lane,
                         [&](double a, int j) { s += a * (omega * dinv[j] * b[j]); });
    s = group_sum<TPR>(s);
    if (!residual_test_running(prr, nb_rr, sc, st, status, lds, &word)) return;
    if (row >= rows || lane != 0) return;
    const double x0 = omega * dinv[row] * b[row];
    y[row] = x0 + omega * dinv[row] * (b[row] - s);
}

// Last V-cycle sweep on a level 0 without coupled transfers: y = x + omega dinv (b - A x) written as
// FP64 (the preconditioned residual z), with the r.z block partials when part is set (rdot = the FP64
// residual r; b itself in the FP64 cycle). Row runs through LDS; the grid is capped, so that the
// consumers' re-summation stays short. On 1.84 M rows 59 us for its 215 MB, 3.6 TB/s where a 1 GiB copy
// reaches 5.2; with lanes per row, whose loads scatter over the rows of a wavefront, 68 us.
template <int RB, typename T = double>
__global__ void __launch_bounds__(BLOCK)
k_jacobi_dot(int rows, const int* __restrict__ rp, const int* __restrict__ ci, const T* __restrict__ val,
             const T* __restrict__ x, const T* __restrict__ b, const T* __restrict__ dinv, T omega,
             double* __restrict__ y, const double* __restrict__ rdot, double* __restrict__ part,
             const int* __restrict__ st) {
    constexpr int U = RB / 32, CAP = U * BLOCK;
    __shared__ T prod[CAP];
    __shared__ double lds[BLOCK / WAVE];
    if (halted(st)) return;   // nothing writes the state while this kernel runs
    const int tid = threadIdx.x;
    double contrib = 0.0;
    for (int r0 = blockIdx.x * RB; r0 < rows; r0 += gridDim.x * RB) {
        const int row = r0 + tid, e0 = rp[r0], e1 = rp[min(r0 + RB, rows)];
        const bool own = tid < RB && row < rows;
        const int k0 = own ? rp[row] : 0, k1 = own ? rp[row + 1] : 0;
        const T xi = own ? x[row] : T(0), bi = own ? b[row] : T(0), di = own ? dinv[row] : T(0);
        const double ri = own && part ? rdot[row] : 0.0;
        T s = 0;
        for (int t = e0; t < e1; t += CAP) {
            int c[U];
            T v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = t + u * BLOCK + tid;
                c[u] = k < e1 ? ci[k] : 0;
                v[u] = k < e1 ? val[k] : T(0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) prod[u * BLOCK + tid] = v[u] * x[c[u]];
            __syncthreads();
            for (int k = max(k0, t), end = min(k1, t + CAP); k < end; ++k) s += prod[k - t];
            __syncthreads();
        }
        if (own) {
            const double yi = (double)(xi + omega * di * (bi - s));
            y[row] = yi;
            contrib += ri * yi;
        }
    }
    if (part) {
        contrib = block_sum(contrib, lds);
        if (tid == 0) part[blockIdx.x] = contrib;
    }
}

// ---- Sliced-ELL rows (the V-cycle's level-0 sweeps) --------------------------------------------
// The operator's rows in slices of 64 positions, one wavefront each, stored column-major inside a
// slice: entry k of the row at position p = 64 q + l sits at sp[q] + 64 k + l, a slice holds
// (sp[q + 1] - sp[q]) / 64 slots per position, and srow[p] names the row (-1 past the last row).
// Inside each window of SELL_WINDOW positions the rows are ordered by decreasing length (ties by
// row index), so the rows of a slice have nearly the same length and little is padded; padded
// slots hold column 0 and value 0. Each entry load of a wavefront is one contiguous run (512 bytes
// in FP64), where the CSR kernels' loads scatter over the rows of a lane group: on a 7.35 M-row
// matrix of the uniform meshes' 5- and 9-entry rows a Jacobi sweep takes 175 us against 257 us.
// One lane per row; the row's products are summed in the order of the CSR kernels with G lanes per
// row (G interleaved partial sums, joined by the lane group's tree), so the results are the CSR
// kernels' bit for bit. Each cache line of the copy is read by one load instruction, so a sweep
// whose bytes exceed the 256 MB Infinity Cache loads it non-temporally, leaving the caches to the
// gathered vector (uniform level 7: 188 -> 160-166 us); a smaller one keeps plain loads, so that
// the copy stays cached between sweeps (on the level-6 adaptive meshes the hint cost 8.0 -> 9.2 us).
constexpr int SELL_SLICE = 64;
constexpr int SELL_WINDOW = 256;
constexpr double SELL_STREAM_BYTES = 256.0 * 1024 * 1024;

__host__ __device__ inline int sell_positions(int rows) { return (rows + SELL_SLICE - 1) / SELL_SLICE * SELL_SLICE; }

// The position's row, the base of its slots and the slice's length; false when `state` says the
// solve has stopped (its word loaded together with the slice's offsets, as in running_with_range).
__device__ __forceinline__ bool sell_slot(const int* __restrict__ sp, const int* __restrict__ srow, int p,
                                          const int* __restrict__ state, int& row, int& base, int& len) {
    const int q = p / SELL_SLICE;
    const int k0 = sp[q], k1 = sp[q + 1];
    row = srow[p];
    const int sv = state ? state[0] : ST_RUNNING;
    asm volatile("" ::"v"(k0), "v"(k1), "v"(row), "s"(sv));
    base = k0 + p % SELL_SLICE;
    len = (k1 - k0) / SELL_SLICE;
    return sv == ST_RUNNING;
}

// sum over the row's entries k of a_k xv(j_k), every index and value loaded before any is used
// (slots past the slice's length give (0, column 0) without a load, so the gathers are
// unconditional and add exact zeros), in the order of row_entries<G> + group_sum<G>: entry k goes
// to partial k mod G, each partial in entry order, the partials joined as the lane tree joins them
// (G = 2: p0 + p1; G = 4: (p0 + p2) + (p1 + p3)). NT: non-temporal loads of the copy.
template <int MAXL, int G, bool NT, typename T, typename F>
__device__ __forceinline__ T sell_row_sum(const int* __restrict__ ci, const T* __restrict__ val, int base, int len,
                                         F xv) {
    int c[MAXL];
    T v[MAXL];
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
        const bool ok = k < len;
        const int at = base + SELL_SLICE * k;
        if constexpr (NT) {
            c[k] = ok ? __builtin_nontemporal_load(ci + at) : 0;
            v[k] = ok ? __builtin_nontemporal_load(val + at) : T(0);
        } else {
            c[k] = ok ? ci[at] : 0;
            v[k] = ok ? val[at] : T(0);
        }
    }
    T acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = 0;
#pragma unroll
    for (int k = 0; k < MAXL; ++k) acc[k % G] += v[k] * xv(c[k]);
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1)
#pragma unroll
        for (int g = 0; g < o; ++g) acc[g] += acc[g + o];
    return acc[0];
}

// y = b - A x (OP_RESID) | y = x + omega dinv (b - A x) (OP_JACOBI) on the sliced-ELL copy
template <int MAXL, int G, bool NT, int OP, typename T>
__global__ void __launch_bounds__(BLOCK)
k_sell_op(int positions, const int* __restrict__ sp, const int* __restrict__ srow, const int* __restrict__ ci,
          const T* __restrict__ val, const T* __restrict__ x, const T* __restrict__ b, const T* __restrict__ dinv,
          T omega, T* __restrict__ y, const int* __restrict__ state) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= positions) return;
    int row, base, len;
    if (!sell_slot(sp, srow, p, state, row, base, len)) return;
    const T s = sell_row_sum<MAXL, G, NT>(ci, val, base, len, [&](int j) { return x[j]; });
    if (row < 0) return;
    if (OP == OP_RESID) y[row] = b[row] - s;
    else y[row] = x[row] + omega * dinv[row] * (b[row] - s);
}

// k_jacobi_from_zero on the sliced-ELL copy
template <int MAXL, int G, bool NT, typename T>
__global__ void __launch_bounds__(BLOCK)
k_sell_from_zero(int positions, const int* __restrict__ sp, const int* __restrict__ srow, const int* __restrict__ ci,
                 const T* __restrict__ val, const T* __restrict__ b, const T* __restrict__ dinv, T omega,
                 T* __restrict__ y, const int* __restrict__ state) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= positions) return;
    int row, base, len;
    if (!sell_slot(sp, srow, p, state, row, base, len)) return;
    const T s = sell_row_sum<MAXL, G, NT>(ci, val, base, len, [&](int j) { return omega * dinv[j] * b[j]; });
    if (row < 0) return;
    const T x0 = omega * dinv[row] * b[row];
    y[row] = x0 + omega * dinv[row] * (b[row] - s);
}

// k_jacobi_from_zero_check on the sliced-ELL copy: the iteration's residual test, then the sweeps
template <int MAXL, int G, bool NT>
__global__ void __launch_bounds__(BLOCK)
k_sell_from_zero_check(int positions, const int* __restrict__ sp, const int* __restrict__ srow,
                       const int* __restrict__ ci, const double* __restrict__ val, const double* __restrict__ b,
                       const double* __restrict__ dinv, double omega, double* __restrict__ y,
                       const double* __restrict__ prr, int nb_rr, double* sc, int* st, int* status) {
    __shared__ double lds[BLOCK / WAVE];
    __shared__ int word;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    int row = -1;
    double s = 0.0;
    if (p < positions) {
        int base, len;
        (void)sell_slot(sp, srow, p, nullptr, row, base, len);
        s = sell_row_sum<MAXL, G, NT>(ci, val, base, len, [&](int j) { return omega * dinv[j] * b[j]; });
    }
    if (!residual_test_running(prr, nb_rr, sc, st, status, lds, &word)) return;
    if (row < 0) return;
    const double x0 = omega * dinv[row] * b[row];
    y[row] = x0 + omega * dinv[row] * (b[row] - s);
}

// ---- The coupled V(2,2) cycle --------------------------------------------------------------------
// With G = I - omega D^-1 A and W = G^2 P (set up once per hierarchy), a level's cycle is
//   x1 = two steps from zero on b,   b_coarse = W^T b,   x = two steps from x1 on b + W e_coarse:
// the restricted residual P^T (b - A x1) is P^T (G^T)^2 b for a symmetric A, and the two steps after
// the correction x1 + P e are linear, so they give two steps from x1 plus G^2 P e. Nothing the level
// smooths is then on the way down or up: its smoothing runs in the launches that carry the coarser
// levels, and a level costs two launches (one down, one up) instead of six. A cycle on the adaptive
// meshes is bound by its launches (3-4 us each below level 0, whatever their size), not by bytes;
// W has about as many entries per row as A, so the bytes moved are those of the residual,
// restriction and prolongation it replaces.
//
// One launch of the descent (stage l): from-zero steps of level l, the coarse right-hand side of
// level l + 1 (or the dense bottom product), and the first step of level l - 1, each on its own
// range of workgroups. RowSet: CSR rows with 2^shift lanes per row.
template <typename T, typename B>
struct RowSet {
    int blocks, rows, shift;
    const int* rp; const int* ci; const T* v;
    const T* x; const B* b; const T* dinv; T omega; T* y;
};
template <typename T, typename B, typename B2>
struct CoupledStage {
    RowSet<T, B> zero;     // y = two steps from zero on b
    RowSet<T, B> mul;      // y = v b, or the dense product
    RowSet<T, B2> step;    // y = x + omega dinv (b - A x)
    const double* dense;   // mul is this dense matrix (rows x rows) times x
    int sell;              // which row set runs on the stage's sliced-ELL copy: 0 zero, 2 step, -1 none
    const int* s_sp; const int* s_row; const int* s_ci; const T* s_v;
    const double* prr; int nb_rr; double* sc; int* st; int* status;   // the residual test (prr set)
};

// row_entries and group_sum with 2^shift lanes per row: the same entries in the same order
template <typename T, typename F>
__device__ __forceinline__ T lanes_row_sum(const int* __restrict__ ci, const T* __restrict__ v, int k0, int k1, int lane,
                                           int shift, F xv) {
    const int tpr = 1 << shift;
    T s = 0;
    for (int k = k0 + lane; k < k1; k += ROW_UNROLL * tpr) {
        int c[ROW_UNROLL];
        T a[ROW_UNROLL];
#pragma unroll
        for (int u = 0; u < ROW_UNROLL; ++u) {
            const int idx = k + u * tpr;
            const bool ok = idx < k1;
            c[u] = ok ? ci[idx] : 0;
            a[u] = ok ? v[idx] : T(0);
        }
#pragma unroll
        for (int u = 0; u < ROW_UNROLL; ++u) s += a[u] * xv(c[u]);
    }
    for (int o = tpr >> 1; o > 0; o >>= 1) s += __shfl_down(s, o, tpr);
    return s;
}

// MAXL, G: the stage's sliced-ELL copy (MAXL 0: none in this stage). Every value is computed
// before the residual test's barrier, so the test's reduction runs beside the row loads.
template <int MAXL, int G, typename T, typename B, typename B2>
__global__ void __launch_bounds__(BLOCK)
k_coupled_stage(CoupledStage<T, B, B2> a) {
    __shared__ double lds[BLOCK / WAVE];
    __shared__ int lds_state;
    int blk = blockIdx.x;
    T out = 0;
    T* dst = nullptr;
    int row = -1;
    const int sv = a.st ? a.st[0] : ST_RUNNING;
    if (blk < a.mul.blocks) {
        const RowSet<T, B>& r = a.mul;
        if (a.dense) {
            const int i = (blk * BLOCK + threadIdx.x) / WAVE, lane = threadIdx.x & (WAVE - 1);
            if (i < r.rows) {
                const double s = wave_sum(dense_row(r.rows, a.dense + (size_t)i * r.rows, r.x, lane));
                if (lane == 0) { out = (T)s; row = i; }
            }
        } else {
            const int g = blk * BLOCK + threadIdx.x, i = g >> r.shift, lane = g & ((1 << r.shift) - 1);
            const int k0 = i < r.rows ? r.rp[i] : 0, k1 = i < r.rows ? r.rp[i + 1] : 0;
            const B* __restrict__ b = r.b;
            out = lanes_row_sum(r.ci, r.v, k0, k1, lane, r.shift, [&](int j) { return (T)b[j]; });
            if (i < r.rows && lane == 0) row = i;
        }
        dst = r.y;
    } else if ((blk -= a.mul.blocks) < a.zero.blocks) {
        const RowSet<T, B>& r = a.zero;
        const B* __restrict__ b = r.b;
        const T* __restrict__ dinv = r.dinv;
        const T omega = r.omega;
        const auto x0 = [&](int j) { return omega * dinv[j] * (T)b[j]; };
        T s = 0;
        bool done = false;
        if constexpr (MAXL > 0) {
            if (a.sell == 0) {
                const int p = blk * BLOCK + threadIdx.x;
                if (p < sell_positions(r.rows)) {
                    int base, len;
                    (void)sell_slot(a.s_sp, a.s_row, p, nullptr, row, base, len);
                    s = sell_row_sum<MAXL, G, false>(a.s_ci, a.s_v, base, len, x0);
                }
                done = true;
            }
        }
        if (!done) {
            const int g = blk * BLOCK + threadIdx.x, i = g >> r.shift, lane = g & ((1 << r.shift) - 1);
            const int k0 = i < r.rows ? r.rp[i] : 0, k1 = i < r.rows ? r.rp[i + 1] : 0;
            s = lanes_row_sum(r.ci, r.v, k0, k1, lane, r.shift, x0);
            if (i < r.rows && lane == 0) row = i;
        }
        if (row >= 0) {
            const T bi = (T)b[row];
            const T xi = omega * dinv[row] * bi;
            out = xi + omega * dinv[row] * (bi - s);
        }
        dst = r.y;
    } else {
        blk -= a.zero.blocks;
        const RowSet<T, B2>& r = a.step;
        const T* __restrict__ x = r.x;
        T s = 0;
        bool done = false;
        if constexpr (MAXL > 0) {
            if (a.sell == 2) {
                const int p = blk * BLOCK + threadIdx.x;
                if (p < sell_positions(r.rows)) {
                    int base, len;
                    (void)sell_slot(a.s_sp, a.s_row, p, nullptr, row, base, len);
                    s = sell_row_sum<MAXL, G, false>(a.s_ci, a.s_v, base, len, [&](int j) { return x[j]; });
                }
                done = true;
            }
        }
        if (!done) {
            const int g = blk * BLOCK + threadIdx.x, i = g >> r.shift, lane = g & ((1 << r.shift) - 1);
            const int k0 = i < r.rows ? r.rp[i] : 0, k1 = i < r.rows ? r.rp[i + 1] : 0;
            s = lanes_row_sum(r.ci, r.v, k0, k1, lane, r.shift, [&](int j) { return x[j]; });
            if (i < r.rows && lane == 0) row = i;
        }
        if (row >= 0) out = x[row] + r.omega * r.dinv[row] * ((T)r.b[row] - s);
        dst = r.y;
    }
    bool running = sv == ST_RUNNING;
    if (a.prr) running = residual_test_running(a.prr, a.nb_rr, a.sc, a.st, a.status, lds, &lds_state);
    if (running && row >= 0) dst[row] = out;
}

// The PCG update and the first stage of the cycle on the new residual in one launch: alpha with the
// breakdown guard (k_fp_update), x += alpha p, r_new = r - alpha q into the other residual buffer, the
// r.r partials, and stage 0 of the descent on r_new, whose entries at the neighbours are not stored yet:
// the row sums are linear in it, so each row sums r's and q's terms apart (in FP64 also in the FP32
// cycle) and combines them once alpha is known. The residual test moves to the next stage. Saves a launch
// per iteration on small meshes: 4.6 + 8.0 us and a gap -> 9.6 us on 29k nodes; on 115k it is no faster
// (5.5 + 15.4 -> 21.6 us, and the next stage 10.2 -> 12.7 us).
constexpr int UPDATE_STAGE_ROWS = 1 << 16;
template <typename T>
struct UpdateStage {
    RowSet<T, double> zero, mul;   // as in CoupledStage; b unused
    int sell;
    const int* s_sp; const int* s_row; const int* s_ci; const T* s_v;
    const double* r; const double* q; const double* p;
    double* rn; double* x;
    const double* ppq; int nb_pq; const double* prz; int nb_rz;
    double* prr;
    int* st; int* status;
};
struct Pair {
    double r, q;
};
template <typename T, typename F>
__device__ __forceinline__ Pair lanes_row_sum2(const int* __restrict__ ci, const T* __restrict__ v, int k0, int k1,
                                               int lane, int shift, F term) {
    const int tpr = 1 << shift;
    Pair s = {0.0, 0.0};
    for (int k = k0 + lane; k < k1; k += ROW_UNROLL * tpr) {
        int c[ROW_UNROLL];
        T a[ROW_UNROLL];
#pragma unroll
        for (int u = 0; u < ROW_UNROLL; ++u) {
            const int idx = k + u * tpr;
            const bool ok = idx < k1;
            c[u] = ok ? ci[idx] : 0;
            a[u] = ok ? v[idx] : T(0);
        }
#pragma unroll
        for (int u = 0; u < ROW_UNROLL; ++u) term((double)a[u], c[u], s);
    }
    for (int o = tpr >> 1; o > 0; o >>= 1) {
        s.r += __shfl_down(s.r, o, tpr);
        s.q += __shfl_down(s.q, o, tpr);
    }
    return s;
}
template <int MAXL, typename T>
__global__ void __launch_bounds__(BLOCK)
k_update_stage(UpdateStage<T> a) {
    __shared__ double lds[2 * BLOCK / WAVE], lds_rr[BLOCK / WAVE];
    __shared__ int word[2];
    const double* __restrict__ r = a.r;
    const double* __restrict__ q = a.q;
    const bool first = (int)blockIdx.x >= a.mul.blocks;   // the rows of the from-zero steps and of r, x
    int row = -1;
    Pair s = {0.0, 0.0};
    T wd = 0;   // omega dinv of the row
    double ri = 0.0, qi = 0.0, pi = 0.0, xi = 0.0;
    if (!first) {
        const RowSet<T, double>& m = a.mul;
        const int g = blockIdx.x * BLOCK + threadIdx.x, i = g >> m.shift, lane = g & ((1 << m.shift) - 1);
        const int k0 = i < m.rows ? m.rp[i] : 0, k1 = i < m.rows ? m.rp[i + 1] : 0;
        s = lanes_row_sum2(m.ci, m.v, k0, k1, lane, m.shift, [&](double v, int j, Pair& t) {
            t.r += v * r[j];
            t.q += v * q[j];
        });
        if (i < m.rows && lane == 0) row = i;
    } else {
        const RowSet<T, double>& m = a.zero;
        const int blk = (int)blockIdx.x - a.mul.blocks;
        const T* __restrict__ dinv = m.dinv;
        const auto term = [&](double v, int j, Pair& t) {
            const double w = v * (double)(m.omega * dinv[j]);
            t.r += w * r[j];
            t.q += w * q[j];
        };
        bool done = false;
        if constexpr (MAXL > 0) {
            if (a.sell == 0) {
                const int pos = blk * BLOCK + threadIdx.x;
                if (pos < sell_positions(m.rows)) {
                    int base, len;
                    (void)sell_slot(a.s_sp, a.s_row, pos, nullptr, row, base, len);
                    int c[MAXL];
                    T v[MAXL];
#pragma unroll
                    for (int k = 0; k < MAXL; ++k) {
                        const bool ok = k < len;
                        c[k] = ok ? a.s_ci[base + SELL_SLICE * k] : 0;
                        v[k] = ok ? a.s_v[base + SELL_SLICE * k] : T(0);
                    }
#pragma unroll
                    for (int k = 0; k < MAXL; ++k) term((double)v[k], c[k], s);
                }
                done = true;
            }
        }
        if (!done) {
            const int g = blk * BLOCK + threadIdx.x, i = g >> m.shift, lane = g & ((1 << m.shift) - 1);
            const int k0 = i < m.rows ? m.rp[i] : 0, k1 = i < m.rows ? m.rp[i + 1] : 0;
            s = lanes_row_sum2(m.ci, m.v, k0, k1, lane, m.shift, term);
            if (i < m.rows && lane == 0) row = i;
        }
        if (row >= 0) {
            wd = m.omega * dinv[row];
            ri = r[row];
            qi = q[row];
            pi = a.p[row];
            xi = a.x[row];
        }
    }
    double sums[2];   // p.q, r.z
    sum_partials_k<2, 2>({a.ppq, a.prz}, {a.nb_pq, a.nb_rz}, 1, sums, lds, a.st, word);
    const int it = word[1];
    if (word[0] != ST_RUNNING) return;
    const double pq = sums[0];
    if (fabs(pq) < 1.0e-30) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            a.st[0] = ST_STOPPED;
            a.st[1] = it;
            publish(a.status, it, ST_STOPPED);
        }
        return;
    }
    const double alpha = sums[1] / pq;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.st[2] = it + 1;
    const T sum = (T)(s.r - alpha * s.q);
    if (!first) {
        if (row >= 0) a.mul.y[row] = sum;
        return;
    }
    double acc = 0.0;
    if (row >= 0) {
        const double rn = ri + (-alpha) * qi;
        a.rn[row] = rn;
        a.x[row] = xi + alpha * pi;
        acc = rn * rn;
        const T b = (T)rn, x0 = wd * b;
        a.zero.y[row] = x0 + wd * (b - sum);
    }
    acc = block_sum(acc, lds_rr);
    if (threadIdx.x == 0) a.prr[blockIdx.x - a.mul.blocks] = acc;
}

// The ascent of a level: second step and coarse correction, y = x + omega dinv (b - A x) + W e
template <typename T, typename B>
__global__ void __launch_bounds__(BLOCK)
k_coupled_up(RowSet<T, B> r, const int* __restrict__ w_rp, const int* __restrict__ w_ci, const T* __restrict__ w_v,
             const T* __restrict__ e, const int* __restrict__ state) {
    const int g = blockIdx.x * BLOCK + threadIdx.x, i = g >> r.shift, lane = g & ((1 << r.shift) - 1);
    const int sv = state ? state[0] : ST_RUNNING;
    const bool in = i < r.rows;
    const int a0 = in ? r.rp[i] : 0, a1 = in ? r.rp[i + 1] : 0, w0 = in ? w_rp[i] : 0, w1 = in ? w_rp[i + 1] : 0;
    if (sv != ST_RUNNING) return;
    const T* __restrict__ x = r.x;
    const T s = lanes_row_sum(r.ci, r.v, a0, a1, lane, r.shift, [&](int j) { return x[j]; });
    const T c = lanes_row_sum(w_ci, w_v, w0, w1, lane, r.shift, [&](int j) { return e[j]; });
    if (in && lane == 0) r.y[i] = x[i] + r.omega * r.dinv[i] * ((T)r.b[i] - s) + c;
}

// The ascent of level 0 into the FP64 output with the r.z block partials. The entries of RB
// consecutive rows are one contiguous run of each CSR matrix: the workgroup loads it coalesced, every
// lane's entries and gathers in flight together, leaves the products in LDS, and one lane per row
// adds its row's in CSR order. (With lanes per row the loads of a wavefront scatter over its rows:
// 2 lanes took 7.3 us for the step alone on 115k rows, 20 us on 460k.) A run longer than the LDS
// tile takes further passes.
template <int RB, typename T>
__global__ void __launch_bounds__(BLOCK)
k_coupled_up_dot(int rows, const int* __restrict__ a_rp, const int* __restrict__ a_ci, const T* __restrict__ a_v,
                 const T* __restrict__ x, const double* __restrict__ r, const T* __restrict__ dinv, T omega,
                 const int* __restrict__ w_rp, const int* __restrict__ w_ci, const T* __restrict__ w_v,
                 const T* __restrict__ e, double* __restrict__ y, double* __restrict__ part,
                 const int* __restrict__ state) {
    constexpr int U = RB / 32, CAP = U * BLOCK;
    __shared__ T pa[CAP], pw[CAP];
    __shared__ double lds[BLOCK / WAVE];
    if (state && state[0] != ST_RUNNING) return;
    const int tid = threadIdx.x;
    double contrib = 0.0;
    for (int r0 = blockIdx.x * RB; r0 < rows; r0 += gridDim.x * RB) {
        const int r1 = r0 + RB < rows ? r0 + RB : rows, row = r0 + tid;
        const int a0 = a_rp[r0], a1 = a_rp[r1], w0 = w_rp[r0], w1 = w_rp[r1];
        const bool own = tid < RB && row < rows;
        const int ra0 = own ? a_rp[row] : 0, ra1 = own ? a_rp[row + 1] : 0;
        const int rw0 = own ? w_rp[row] : 0, rw1 = own ? w_rp[row + 1] : 0;
        const double ri = own ? r[row] : 0.0;
        const T xi = own ? x[row] : T(0), di = own ? dinv[row] : T(0);
        T sa = 0, sw = 0;
        for (int ta = a0, tw = w0; ta < a1 || tw < w1; ta += CAP, tw += CAP) {
            int ca[U], cw[U];
            T va[U], vw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int ka = ta + u * BLOCK + tid, kw = tw + u * BLOCK + tid;
                ca[u] = ka < a1 ? a_ci[ka] : 0;
                va[u] = ka < a1 ? a_v[ka] : T(0);
                cw[u] = kw < w1 ? w_ci[kw] : 0;
                vw[u] = kw < w1 ? w_v[kw] : T(0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                pa[u * BLOCK + tid] = va[u] * x[ca[u]];
                pw[u * BLOCK + tid] = vw[u] * e[cw[u]];
            }
            __syncthreads();
            for (int k = max(ra0, ta), k1 = min(ra1, ta + CAP); k < k1; ++k) sa += pa[k - ta];
            for (int k = max(rw0, tw), k1 = min(rw1, tw + CAP); k < k1; ++k) sw += pw[k - tw];
            __syncthreads();
        }
        if (own) {
            const double z = (double)(xi + omega * di * ((T)ri - sa) + sw);
            y[row] = z;
            contrib += ri * z;
        }
    }
    if (part) {
        contrib = block_sum(contrib, lds);
        if (tid == 0) part[blockIdx.x] = contrib;
    }
}

// The positions of one window's rows (a workgroup per window of SELL_WINDOW rows): each row's rank
// among the window's rows by decreasing length, ties by row index; the slices' entry counts (64
// times the length of their first, longest row) and the longest row (atomic max into info[1]).
__global__ void __launch_bounds__(SELL_WINDOW)
k_sell_plan(int rows, int positions, const int* __restrict__ rp, int* __restrict__ srow, int* __restrict__ cnt,
            int* __restrict__ info) {
    __shared__ int len_of[SELL_WINDOW];
    __shared__ int len_at[SELL_WINDOW];
    const int t = threadIdx.x, w0 = blockIdx.x * SELL_WINDOW, r = w0 + t;
    const int L = r < rows ? rp[r + 1] - rp[r] : -1;
    len_of[t] = L;
    __syncthreads();
    int rank = 0;
    for (int u = 0; u < SELL_WINDOW; ++u) {
        const int Lu = len_of[u];
        rank += (Lu > L || (Lu == L && u < t)) ? 1 : 0;
    }
    len_at[rank] = L;
    if (w0 + rank < positions) srow[w0 + rank] = L >= 0 ? r : -1;
    if (L > 0) atomicMax(&info[1], L);
    __syncthreads();
    if (t < SELL_WINDOW / SELL_SLICE) {
        const int q = w0 / SELL_SLICE + t;
        if (q * SELL_SLICE < positions) cnt[q] = SELL_SLICE * max(len_at[t * SELL_SLICE], 0);
    }
}

// The slots of each position: its row's entries in CSR order, then (column 0, value 0) up to the
// slice's length
__global__ void k_sell_fill(int positions, const int* __restrict__ rp, const int* __restrict__ ci,
                            const double* __restrict__ val, const int* __restrict__ srow, const int* __restrict__ sp,
                            int* __restrict__ sci, double* __restrict__ sv) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= positions) return;
    const int q = p / SELL_SLICE;
    const int base = sp[q] + p % SELL_SLICE, len = (sp[q + 1] - sp[q]) / SELL_SLICE;
    const int row = srow[p];
    const int k0 = row >= 0 ? rp[row] : 0, rl = row >= 0 ? rp[row + 1] - k0 : 0;
    for (int k = 0; k < len; ++k) {
        const bool ok = k < rl;
        sci[base + SELL_SLICE * k] = ok ? ci[k0 + k] : 0;
        sv[base + SELL_SLICE * k] = ok ? val[k0 + k] : 0.0;
    }
}

// Entry of the FP32 cycle: b32 = (float) r, after the iteration's residual test when prr is set
__global__ void k_to_f32_check(int n, const double* __restrict__ r, float* __restrict__ b32,
                               const double* __restrict__ prr, int nb_rr, double* sc, int* st, int* status) {
    __shared__ double lds[BLOCK / WAVE];
    __shared__ int word;
    if (st && prr) {
        if (!residual_test_running(prr, nb_rr, sc, st, status, lds, &word)) return;
    } else if (halted(st)) {
        return;
    }
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) b32[i] = (float)r[i];
}

__global__ void k_f64_to_f32(size_t n, const double* __restrict__ in, float* __restrict__ out) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = (float)in[i];
}

// Jacobi preconditioner z = D^-1 r with the r.z partials, optionally after the residual test
__global__ void __launch_bounds__(BLOCK)
k_fp_jacobi_prec(PcgArgs a, int h_next, int check) {
    __shared__ double lds[BLOCK / WAVE], lds_rz[BLOCK / WAVE];
    __shared__ int word;
    if (check) {
        if (!residual_test_running(a.prr, a.nb_rr, a.sc, a.st, a.status, lds, &word)) return;
    } else if (halted(a.st)) {
        return;
    }
    double acc = 0.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += gridDim.x * blockDim.x) {
        const double zi = a.inv_diag[i] * a.r[i];
        a.z[i] = zi;
        acc += a.r[i] * zi;
    }
    acc = block_sum(acc, lds_rz);
    if (threadIdx.x == 0) a.prz[h_next][blockIdx.x] = acc;
}

// ======================================================================================================
// multicolour ILU(0) (src/cfa/linalg.cuh:361-568)
// ======================================================================================================
// Rows of one colour: for each elimination step of the row's schedule, l_ik = a_ik / u_kk and
// a_ij -= l_ik u_kj for the scheduled entries, in the schedule's order (colour by colour, CSR
// order inside a colour, then row k in column order: the order of linalg.cuh:366-392). Rows of
// one colour do not couple and rows k of earlier colours are final, so the update is in place.
__global__ void k_ilu_factor_rows(int m, int t0, const int* __restrict__ el_ptr, const int* __restrict__ el,
                                  const int* __restrict__ upd, double* __restrict__ lu) {
#pragma clang fp contract(off)   // separate multiply and subtract: the factors match a serial CPU run bit for bit
    const int t = t0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= t0 + m) return;
    for (int e = el_ptr[t]; e < el_ptr[t + 1]; ++e) {
        const int q = el[4 * e], kd = el[4 * e + 1], u0 = el[4 * e + 2], u1 = el[4 * e + 3];
        const double lik = lu[q] / lu[kd];
        lu[q] = lik;
        for (int u = u0; u < u1; ++u) lu[upd[2 * u]] -= lik * lu[upd[2 * u + 1]];
    }
}

__global__ void k_ilu_gather(int nl, int nu, int n, const int* __restrict__ l_src, const int* __restrict__ u_src,
                             const int* __restrict__ d_src, const double* __restrict__ lu, double* __restrict__ lv,
                             double* __restrict__ uv, double* __restrict__ dinv, float* __restrict__ lv32,
                             float* __restrict__ uv32, float* __restrict__ dinv32) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < nl) { const double v = lu[l_src[e]]; lv[e] = v; if (lv32) lv32[e] = (float)v; }
    if (e < nu) { const double v = lu[u_src[e]]; uv[e] = v; if (uv32) uv32[e] = (float)v; }
    if (e < n) { const double v = 1.0 / lu[d_src[e]]; dinv[e] = v; if (dinv32) dinv32[e] = (float)v; }
}

// The sliced-ELL values of the split rows after a factorization: slot k takes split entry src[k]
// (FP64 and, when kept, FP32 from the FP32 split values, so they equal the CSR path's), 0 for padding
__global__ void k_ilu_sell_values(int ls, int us, const int* __restrict__ lsrc, const int* __restrict__ usrc,
                                  const double* __restrict__ lv, const double* __restrict__ uv,
                                  const float* __restrict__ lv32, const float* __restrict__ uv32,
                                  double* __restrict__ slv, double* __restrict__ suv, float* __restrict__ slv32,
                                  float* __restrict__ suv32) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ls) {
        const int e = lsrc[k];
        slv[k] = e >= 0 ? lv[e] : 0.0;
        if (slv32) slv32[k] = e >= 0 ? lv32[e] : 0.0f;
    }
    if (k < us) {
        const int e = usrc[k];
        suv[k] = e >= 0 ? uv[e] : 0.0;
        if (suv32) suv32[k] = e >= 0 ? uv32[e] : 0.0f;
    }
}

// One colour's sweep on the sliced-ELL rows, one lane per row: forward (UPPER false: acc = r_i -
// sum l z, times dinv on the last colour) or backward (acc = z_i - sum u z, times dinv). All MAXL
// slots are loaded before the gathers; a padding slot gathers nothing and subtracts an exact +0,
// so each row's result is k_ilu_lower / k_ilu_upper's. mpos: the colour's positions (a multiple
// of 64) from global position p0.
template <int NRHS, int MAXL, bool UPPER, typename T>
__global__ void __launch_bounds__(BLOCK)
k_ilu_sweep_sell(int mpos, int n, int cs, int p0, const int* __restrict__ srow, const int* __restrict__ sp,
                 const int* __restrict__ sc, const T* __restrict__ sv, const T* __restrict__ dinv, int last,
                 const double* __restrict__ r, double* __restrict__ z, const int* __restrict__ st) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= mpos) return;
    int t, base, len;
    if (!sell_slot(sp, srow, p0 + p, st, t, base, len)) return;
    int c[MAXL];
    T v[MAXL];
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
        const bool ok = k < len;
        c[k] = ok ? sc[base + SELL_SLICE * k] : 0;
        v[k] = ok ? sv[base + SELL_SLICE * k] : T(0);
    }
    if (t < 0) return;
    const int i = cs + t;
    double acc[NRHS];
#pragma unroll
    for (int q = 0; q < NRHS; ++q) acc[q] = UPPER ? z[(size_t)q * n + i] : r[(size_t)q * n + i];
#pragma unroll
    for (int k = 0; k < MAXL; ++k) {
        const double a = (double)v[k];
        const bool ok = k < len;
#pragma unroll
        for (int q = 0; q < NRHS; ++q) {
            const double zj = ok ? z[(size_t)q * n + c[k]] : 0.0;
            acc[q] -= a * zj;
        }
    }
    const double d = (double)dinv[t];
#pragma unroll
    for (int q = 0; q < NRHS; ++q) z[(size_t)q * n + i] = (UPPER || last) ? acc[q] * d : acc[q];
}

// The ILU(0) apply runs in colour order: r is permuted there (read in row order, written into one
// run per colour), the sweeps then stream every colour's rows, vector entries and factor entries,
// and z is permuted back (written in row order). In row order a colour's rows are spread over the
// whole vector, so each colour's sweep touched every cache line of r and z: measured at U7, 2.2x
// the algorithmic bytes crossed HBM.
// z back to row order (one colour: no backward sweep)
template <int NRHS>
__global__ void k_ilu_unpermute(int n, const int* __restrict__ pos, const double* __restrict__ zp,
                                double* __restrict__ z, const int* __restrict__ st) {
    if (halted(st)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int q = pos[i];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) z[(size_t)c * n + i] = zp[(size_t)c * n + q];
}

// One entry's move into colour order with the forward sweep of colour 0: position q (at index k of
// the component's vectors) below m0 goes to z (times dinv when colour 0 is also the last), else to r
template <typename T>
__device__ __forceinline__ void ilu_permuted_entry(size_t k, int q, int m0, int last, const T* __restrict__ dinv,
                                                   double v, double* __restrict__ rp, double* __restrict__ zp) {
    if (q >= m0) rp[k] = v;
    else zp[k] = last ? v * (double)dinv[q] : v;
}

// The permutation into colour order fused with the forward sweep of colour 0. L holds the columns
// of earlier colours, so colour 0 has no L entries and its sweep is z = r (times dinv when it is
// also the last colour): its z entries are written here, and its r entries are not needed.
template <int NRHS, typename T>
__global__ void k_ilu_permute_first(int n, int m0, const int* __restrict__ pos, const double* __restrict__ r,
                                    const T* __restrict__ dinv, int last, double* __restrict__ rp,
                                    double* __restrict__ zp, const int* __restrict__ st) {
    if (halted(st)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int q = pos[i];
#pragma unroll
    for (int c = 0; c < NRHS; ++c)
        ilu_permuted_entry((size_t)c * n + q, q, m0, last, dinv, r[(size_t)c * n + i], rp, zp);
}

// The backward sweep of colour 0 fused with the permutation back to row order, one thread per
// row i in row order: the rows of colour 0 (positions below m0) finish their sweep and write z
// directly, every other row copies its final value from z_perm.
template <int NRHS, typename T>
__global__ void __launch_bounds__(BLOCK)
k_ilu_last_unpermute(int n, int m0, const int* __restrict__ pos, const int* __restrict__ up,
                     const int* __restrict__ uc, const T* __restrict__ uv, const T* __restrict__ dinv,
                     const double* __restrict__ zp, double* __restrict__ z, const int* __restrict__ st) {
    if (halted(st)) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int q = pos[i];
    if (q >= m0) {
#pragma unroll
        for (int c = 0; c < NRHS; ++c) z[(size_t)c * n + i] = zp[(size_t)c * n + q];
        return;
    }
    double acc[NRHS];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) acc[c] = zp[(size_t)c * n + q];
    row_entries<1>(uc, uv, up[q], up[q + 1], 0, [&](T ut, int j) {
        const double u = (double)ut;
#pragma unroll
        for (int c = 0; c < NRHS; ++c) acc[c] -= u * zp[(size_t)c * n + j];
    });
    const double d = (double)dinv[q];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) z[(size_t)c * n + i] = acc[c] * d;
}

// Forward sweep over the rows cs .. cs + m - 1 of one colour (colour order), all components per
// thread (the L row is read once). The row's entries are loaded ahead of their uses
// (row_entries) and subtracted in order, one lane per row: two lanes per row were 7-10 % faster
// at U6/U7 but sum in another order, which moves the reference's stored MMS error table in its
// last printed digit.
template <int NRHS, typename T>
__global__ void __launch_bounds__(BLOCK)
k_ilu_lower(int m, int n, int cs, const int* __restrict__ lp, const int* __restrict__ lc, const T* __restrict__ lv,
            const T* __restrict__ dinv, int last, const double* __restrict__ r, double* __restrict__ z,
            const int* __restrict__ st) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int e0, e1;
    if (!running_with_range(lp, t, m, st, e0, e1) || t >= m) return;
    const int i = cs + t;
    double acc[NRHS];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) acc[c] = r[(size_t)c * n + i];
    row_entries<1>(lc, lv, e0, e1, 0, [&](T lt, int j) {
        const double l = (double)lt;
#pragma unroll
        for (int c = 0; c < NRHS; ++c) acc[c] -= l * z[(size_t)c * n + j];
    });
    const double d = (double)dinv[t];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) z[(size_t)c * n + i] = last ? acc[c] * d : acc[c];
}

template <int NRHS, typename T>
__global__ void __launch_bounds__(BLOCK)
k_ilu_upper(int m, int n, int cs, const int* __restrict__ up, const int* __restrict__ uc, const T* __restrict__ uv,
            const T* __restrict__ dinv, double* __restrict__ z, const int* __restrict__ st) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    int e0, e1;
    if (!running_with_range(up, t, m, st, e0, e1) || t >= m) return;
    const int i = cs + t;
    double acc[NRHS];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) acc[c] = z[(size_t)c * n + i];
    row_entries<1>(uc, uv, e0, e1, 0, [&](T ut, int j) {
        const double u = (double)ut;
#pragma unroll
        for (int c = 0; c < NRHS; ++c) acc[c] -= u * z[(size_t)c * n + j];
    });
    const double d = (double)dinv[t];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) z[(size_t)c * n + i] = acc[c] * d;
}

// The forward sweep with TPR lanes per row, for the FP32 factors of the mixed-precision path (no
// reference order to keep there): each lane sums its entries' products, the group adds them, and
// the row takes r - sum.
template <int NRHS, int TPR>
__global__ void __launch_bounds__(BLOCK)
k_ilu_lower_lanes(int m, int n, int cs, const int* __restrict__ lp, const int* __restrict__ lc,
                  const float* __restrict__ lv, const float* __restrict__ dinv, int last, const double* __restrict__ r,
                  double* __restrict__ z, const int* __restrict__ st) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = g / TPR, lane = g % TPR;
    int e0, e1;
    if (!running_with_range(lp, t, m, st, e0, e1)) return;
    const int i = cs + t;
    double sum[NRHS];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) sum[c] = 0.0;
    row_entries<TPR>(lc, lv, e0, e1, lane, [&](float lt, int j) {
        const double l = (double)lt;
#pragma unroll
        for (int c = 0; c < NRHS; ++c) sum[c] += l * z[(size_t)c * n + j];
    });
#pragma unroll
    for (int c = 0; c < NRHS; ++c) sum[c] = group_sum<TPR>(sum[c]);
    if (t >= m || lane != 0) return;
    const double d = (double)dinv[t];
#pragma unroll
    for (int c = 0; c < NRHS; ++c) {
        const double acc = r[(size_t)c * n + i] - sum[c];
        z[(size_t)c * n + i] = last ? acc * d : acc;
    }
}

// The trailing colours of at most ILU_TAIL_ROWS rows each (greedy colouring leaves two or three of the
// five or six with few rows), forward t..nc-1 and backward nc-2..t, in one launch: one workgroup with
// a barrier between colours instead of a launch per colour and direction, since such a launch is all
// latency. Each row is k_ilu_lower's and k_ilu_upper's, in their order. Uniform level 4 (two colours of
// under 256 rows): 5.0 + 2.8 + 1.9 us and two gaps -> 7.9 us. A row per lane: with colours of 1280
// and 2560 rows the workgroup took 24 and 63 us for what separate launches do in 12 and 23.
constexpr int ILU_TAIL_ROWS = 1024;
constexpr int ILU_TAIL_THREADS = 1024;
constexpr int ILU_TAIL_COLOURS = 16;
struct IluTail {
    int first, nc;
    int start[ILU_TAIL_COLOURS + 1];   // colour_start of colours first .. nc
};
template <int NRHS, typename T>
__global__ void __launch_bounds__(ILU_TAIL_THREADS)
k_ilu_tail(int n, IluTail a, const int* __restrict__ lp, const int* __restrict__ lc, const T* __restrict__ lv,
           const int* __restrict__ up, const int* __restrict__ uc, const T* __restrict__ uv,
           const T* __restrict__ dinv, const double* __restrict__ r, double* z, const int* __restrict__ st) {
    if (halted(st)) return;
    const int colours = a.nc - a.first;
    for (int k = 0; k < 2 * colours - 1; ++k) {
        const bool lower = k < colours;
        const int c = lower ? k : 2 * colours - 2 - k;
        const bool last = c == colours - 1;
        const int* ptr = lower ? lp : up;
        const int* col = lower ? lc : uc;
        const T* val = lower ? lv : uv;
        const double* src = lower ? r : z;
        if (k > 0) __syncthreads();
        for (int i = a.start[c] + (int)threadIdx.x; i < a.start[c + 1]; i += ILU_TAIL_THREADS) {
            double acc[NRHS];
#pragma unroll
            for (int q = 0; q < NRHS; ++q) acc[q] = src[(size_t)q * n + i];
            row_entries<1>(col, val, ptr[i], ptr[i + 1], 0, [&](T vt, int j) {
                const double v = (double)vt;
#pragma unroll
                for (int q = 0; q < NRHS; ++q) acc[q] -= v * z[(size_t)q * n + j];
            });
            const double d = (double)dinv[i];
#pragma unroll
            for (int q = 0; q < NRHS; ++q) z[(size_t)q * n + i] = !lower || last ? acc[q] * d : acc[q];
        }
    }
}

// ======================================================================================================
// Two-component BiCGSTAB (src/cfa/linalg.cuh:642-779)
// ======================================================================================================
// Per-component scalars: slot(c) = base + c
enum {
    B_RN0 = 0, B_BD = 2, B_RHO = 4, B_RHO_OLD = 6, B_ALPHA = 8, B_OMEGA = 10, B_REL = 12,
    B_CB = 14, B_CO = 16, B_CA = 18, B_A1 = 20, B_A2 = 22, B_CW = 24, B_TOL = 26
};
// ints: [0] state (stopped when both components are inactive), [2 + c] active, [4 + c] iters,
// [6 + c] converged, [8 + c] half-step done, [10] current iteration, [11] iteration cap

// Two-component partial sums: part[b * 6 + 2 q + c]
// (lds: at least 2 nq * blockDim.x / 64 doubles)
template <int NQ>
__device__ __forceinline__ void write_partials2(double* part, double (&acc)[NQ][2], double* lds) {
    double v[2 * NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int c = 0; c < 2; ++c) v[2 * q + c] = acc[q][c];
    block_sum_k<2 * NQ>(v, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < 2 * NQ; ++k) part[(size_t)blockIdx.x * 6 + k] = v[k];
}

// Both components' products of a run of RB rows (one workgroup, k_apply_K_B's scheme): the lane's row
// and component (part 0 and 1 of the workgroup) and its sum; prod: 2 RUN_TILE(RB) doubles
template <int RB>
__device__ __forceinline__ double run_product2(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                               const double* __restrict__ val, const double* __restrict__ x_u,
                                               const double* __restrict__ x_v, int r0, double* prod) {
    const RowValues<1, double> av{{val}};
    const int row = r0 + (int)threadIdx.x % RB, e0 = rp[r0], e1 = rp[min(r0 + RB, n)];
    const int k0 = row < n ? rp[row] : e1, k1 = row < n ? rp[row + 1] : e1;
    double s[2] = {0.0, 0.0};
    for (int t = e0; t < e1; t += RUN_TILE(RB)) {
        RunTile<RB, 1> tile;
        tile.load(ci, av, t, e1);
#pragma unroll
        for (int u = 0; u < RUN_SLOTS(RB); ++u) {
            const int at = u * BLOCK + threadIdx.x, j = tile.c[u];
            prod[at] = tile.v[u][0] * x_u[j];
            prod[RUN_TILE(RB) + at] = tile.v[u][0] * x_v[j];
        }
        __syncthreads();
        run_row_sums<RB, 2>(prod, t, k0, k1, s);
        __syncthreads();
    }
    return run_part_has<RB>(0) ? s[0] : s[1];
}

// The iterate from the caller's guesses, r = b - A x (both components), r0 = p = r, v = 0; partial r.r
template <int RB>
__global__ void __launch_bounds__(BLOCK)
k_bicg_init(int n, const int* __restrict__ rp, const int* __restrict__ ci, const double* __restrict__ val,
            const double* __restrict__ b_u, const double* __restrict__ b_v, const double* __restrict__ x_u,
            const double* __restrict__ x_v, double* __restrict__ x, double* __restrict__ r, double* __restrict__ r0v,
            double* __restrict__ p, double* __restrict__ v, double* __restrict__ part) {
    __shared__ double prod[2 * RUN_TILE(RB)];
    __shared__ double lds[2 * BLOCK / WAVE];
    const int c = threadIdx.x / RB;
    double acc[1][2] = {{0.0, 0.0}};
    for (int r0 = blockIdx.x * RB; r0 < n; r0 += gridDim.x * RB) {
        const double s = run_product2<RB>(n, rp, ci, val, x_u, x_v, r0, prod);
        const int row = r0 + (int)threadIdx.x % RB;
        if (c > 1 || row >= n) continue;
        const int i = c * n + row;
        const double q = (c ? b_v : b_u)[row] - s;
        x[i] = (c ? x_v : x_u)[row];
        r[i] = q;
        r0v[i] = q;
        p[i] = q;
        v[i] = 0.0;
        if (c) acc[0][1] += q * q;
        else acc[0][0] += q * q;
    }
    write_partials2<1>(part, acc, lds);
}

__device__ __forceinline__ void bicg_stop(int* st, int c, int it, int ok) {
    st[2 + c] = 0;
    st[4 + c] = it;
    st[6 + c] = ok;
}

// Scalars and state of a solve from the r.r partials; the first iteration's p update takes no
// coefficients (p = r), and a component whose rho breaks down at once stops with 0 iterations
__global__ void k_bicg_final_init(int nb, const double* __restrict__ part, double tol, double* __restrict__ sc,
                                  int* __restrict__ st, int* __restrict__ status, int max_iter) {
    __shared__ double lds[2 * BLOCK / WAVE];
    double rr[2];
    sum_partials_k<2>({part, part + 1}, {nb, nb}, 6, rr, lds);
    if (threadIdx.x != 0) return;
    int act[2];
    sc[B_TOL] = tol;
    for (int c = 0; c < 2; ++c) {
        const double rn0 = sqrt(rr[c]), bd = 1.0e-30 * rn0 * rn0 + 1.0e-300;
        sc[B_RN0 + c] = rn0;
        sc[B_RHO + c] = rr[c];
        sc[B_BD + c] = bd;
        sc[B_RHO_OLD + c] = 1.0;
        sc[B_ALPHA + c] = 1.0;
        sc[B_OMEGA + c] = 1.0;
        sc[B_REL + c] = 0.0;
        sc[B_CB + c] = 0.0;
        sc[B_CO + c] = 0.0;
        act[c] = rn0 >= 1.0e-13 ? 1 : 0;
        st[2 + c] = act[c];
        st[4 + c] = 0;
        st[6 + c] = 1;
        st[8 + c] = 0;
    }
    st[10] = 0;
    st[11] = max_iter;
    int state = (act[0] || act[1]) && max_iter > 0 ? ST_RUNNING : ST_STOPPED;
    if (state == ST_RUNNING) {
        for (int c = 0; c < 2; ++c)
            if (act[c] && fabs(rr[c]) < sc[B_BD + c]) {
                bicg_stop(st, c, 0, 0);
                act[c] = 0;
            }
        if (!(act[0] || act[1])) state = ST_STOPPED;
    }
    st[0] = state;
    publish(status, 0, state);
}

// The solutions to the caller's vectors and the outcome (status [2..13]: active, iterations, converged
// and relative residual of both components)
__global__ void k_bicg_outcome(int n, const double* __restrict__ x, double* __restrict__ x_u, double* __restrict__ x_v,
                               const double* __restrict__ sc, const int* __restrict__ st, int* __restrict__ status) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        x_u[i] = x[i];
        x_v[i] = x[n + i];
    }
    if (i < 6) __hip_atomic_store(&status[2 + i], st[2 + i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (blockIdx.x == 0 && threadIdx.x < 2) publish_double(status + 8 + 2 * threadIdx.x, sc[B_REL + threadIdx.x]);
}

// p = r + cb (p - co v), from the second iteration on, and the permutation of p into colour order with
// the forward sweep of colour 0 (k_ilu_permute_first), one thread per row for both components
template <typename T>
__global__ void __launch_bounds__(BLOCK)
k_bicg_p(int n, const double* __restrict__ r, const double* __restrict__ v, const double* __restrict__ sc,
         double* __restrict__ p, int m0, const int* __restrict__ pos, const T* __restrict__ dinv, int last,
         double* __restrict__ rp, double* __restrict__ zp, const int* __restrict__ st) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    const int state = st[0], it = st[10];
    if (state != ST_RUNNING || i >= n) return;
    const int q = pos[i];
    double pv[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int k = c * n + i;
        pv[c] = it > 0 ? r[k] + sc[B_CB + c] * (p[k] - sc[B_CO + c] * v[k]) : p[k];
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        if (it > 0) p[c * n + i] = pv[c];
        ilu_permuted_entry(c * n + q, q, m0, last, dinv, pv[c], rp, zp);
    }
}

// y = A x for both components; with dots: partial y.w0 (mode 1) or y.y, y.w0 (mode 2). Row runs
// through LDS (k_apply_K_B's scheme; two lanes per row took 82 us on 1.84 M nodes, 20 us on 461k)
template <int RB>
__global__ void __launch_bounds__(BLOCK)
k_spmv2_dots(int n, const int* __restrict__ rp, const int* __restrict__ ci, const double* __restrict__ val,
             const double* __restrict__ x, double* __restrict__ y, const double* __restrict__ w0, int mode,
             double* __restrict__ part, const int* __restrict__ st) {
    __shared__ double prod[2 * RUN_TILE(RB)];
    __shared__ double lds[4 * BLOCK / WAVE];
    if (halted(st)) return;
    const int c = threadIdx.x / RB;
    double dot0 = 0.0, dot1 = 0.0;   // of the lane's component
    for (int r0 = blockIdx.x * RB; r0 < n; r0 += gridDim.x * RB) {
        const int row = r0 + (int)threadIdx.x % RB, i = c * n + row;
        const bool own = c < 2 && row < n;
        const double wi = own ? w0[i] : 0.0;
        const double s = run_product2<RB>(n, rp, ci, val, x, x + n, r0, prod);
        if (!own) continue;
        y[i] = s;
        if (mode == 1) {   // r0 . v
            dot0 += wi * s;
        } else {           // t . t, t . s
            dot0 += s * s;
            dot1 += s * wi;
        }
    }
    double acc[2][2] = {{c == 0 ? dot0 : 0.0, c == 1 ? dot0 : 0.0}, {c == 0 ? dot1 : 0.0, c == 1 ? dot1 : 0.0}};
    if (mode == 1) write_partials2<1>(part, reinterpret_cast<double(&)[1][2]>(acc), lds);
    else write_partials2<2>(part, acc, lds);
}

// The scalar steps between the vector kernels are folded into the kernels that consume them:
// every block sums the producer's partials in the same fixed order and takes the same decision;
// block 0 alone writes the state. A component stopped here is treated by a late block exactly
// as an already inactive one (zero coefficient), so a block that reads the state before or after
// block 0's write computes the same values.

// alpha = rho / (r0 . v) with the breakdown guard (from the r0.v partials), then s = r - alpha v, the
// s.s partials, and the permutation of s into colour order with the forward sweep of colour 0, one
// thread per row for both components
template <typename T>
__global__ void __launch_bounds__(BLOCK)
k_bicg_s(int n, const double* __restrict__ r, const double* __restrict__ v, double* __restrict__ sc,
         double* __restrict__ s, double* __restrict__ part, int nb_a, const double* __restrict__ part_a,
         int m0, const int* __restrict__ pos, const T* __restrict__ dinv, int last, double* __restrict__ rp,
         double* __restrict__ zp, int* __restrict__ st, int* __restrict__ status) {
    __shared__ double lds[2 * BLOCK / WAVE];
    __shared__ int word[3];
    int i = blockIdx.x * BLOCK + threadIdx.x, q = 0;
    double ri[2] = {0.0, 0.0}, vi[2] = {0.0, 0.0};
    auto load = [&] {
        if (i >= n) return;
        q = pos[i];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            ri[c] = r[c * n + i];
            vi[c] = v[c * n + i];
        }
    };
    load();   // beside the sums
    const double bd[2] = {sc[B_BD], sc[B_BD + 1]}, rho[2] = {sc[B_RHO], sc[B_RHO + 1]};
    double ca[2];
    bool act[2];
    double o2[2];
    sum_partials_k<2, 3>({part_a, part_a + 1}, {nb_a, nb_a}, 6, o2, lds, st, word);
    if (word[0] != ST_RUNNING) return;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        act[c] = word[1 + c] && !(fabs(o2[c]) < bd[c]);
        ca[c] = act[c] ? rho[c] / o2[c] : 0.0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const int it = st[10];
        for (int c = 0; c < 2; ++c) {
            sc[B_CA + c] = ca[c];
            if (word[1 + c] && !act[c]) bicg_stop(st, c, it, 0);
            if (act[c]) sc[B_ALPHA + c] = ca[c];
        }
        if (!(act[0] || act[1])) { st[0] = ST_STOPPED; publish(status, it, ST_STOPPED); }
    }
    if (!(act[0] || act[1])) return;
    double acc[1][2] = {{0.0, 0.0}};
    while (i < n) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double si = ri[c] - ca[c] * vi[c];
            s[c * n + i] = si;
            acc[0][c] += si * si;
            ilu_permuted_entry(c * n + q, q, m0, last, dinv, si, rp, zp);
        }
        i += gridDim.x * BLOCK;
        load();
    }
    write_partials2<1>(part, acc, lds);
}

// omega = (t . s) / (t . t) unless the half step already converged (from the s.s and t.t, t.s
// partials), then x += alpha phat + omega shat, r = s - omega t and the r.r, r0.r partials
__global__ void __launch_bounds__(BLOCK)
k_bicg_xr(int n, const double* __restrict__ ph, const double* __restrict__ sh, const double* __restrict__ s,
          const double* __restrict__ t, const double* __restrict__ r0, double* __restrict__ sc, double* __restrict__ x,
          double* __restrict__ r, double* __restrict__ part, int nb_s, const double* __restrict__ part_s, int nb_t,
          const double* __restrict__ part_t, int* __restrict__ st) {
    __shared__ double lds[6 * BLOCK / WAVE];
    __shared__ int word[3];
    int i = blockIdx.x * BLOCK + threadIdx.x;
    double xi = 0.0, pi = 0.0, hi = 0.0, si = 0.0, ti = 0.0, oi = 0.0;
    auto load = [&] {
        if (i >= 2 * n) return;
        xi = x[i];
        pi = ph[i];
        hi = sh[i];
        si = s[i];
        ti = t[i];
        oi = r0[i];
    };
    load();   // beside the sums
    const double tol = sc[B_TOL], rn0[2] = {sc[B_RN0], sc[B_RN0 + 1]}, bd[2] = {sc[B_BD], sc[B_BD + 1]},
                 alpha[2] = {sc[B_ALPHA], sc[B_ALPHA + 1]};
    double sums[6];   // s.s, t.t, t.s of both components
    sum_partials_k<6, 3>({part_s, part_s + 1, part_t, part_t + 1, part_t + 2, part_t + 3},
                         {nb_s, nb_s, nb_t, nb_t, nb_t, nb_t}, 6, sums, lds, st, word);
    if (word[0] != ST_RUNNING) return;
    double a1[2], a2[2];
    int half[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const double ss = sums[c], tt = sums[2 + c], ts = sums[4 + c];
        a1[c] = a2[c] = 0.0;
        half[c] = 0;
        if (!word[1 + c]) continue;
        a1[c] = alpha[c];
        const double s_norm = sqrt(ss);
        if (s_norm < tol * rn0[c] || s_norm < 1.0e-11) half[c] = 1;
        else a2[c] = (tt > bd[c]) ? (ts / tt) : 0.0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0)
        for (int c = 0; c < 2; ++c) {
            sc[B_A1 + c] = a1[c];
            sc[B_A2 + c] = a2[c];
            sc[B_CW + c] = a2[c];
            st[8 + c] = half[c];
            if (word[1 + c] && !half[c]) sc[B_OMEGA + c] = a2[c];
        }
    double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
    while (i < 2 * n) {
        const int c = i >= n;
        x[i] = xi + ((c ? a1[1] : a1[0]) * pi + (c ? a2[1] : a2[0]) * hi);
        const double ri = si - (c ? a2[1] : a2[0]) * ti;
        r[i] = ri;
        if (c) {
            acc[0][1] += ri * ri;
            acc[1][1] += oi * ri;
        } else {
            acc[0][0] += ri * ri;
            acc[1][0] += oi * ri;
        }
        i += gridDim.x * BLOCK;
        load();
    }
    write_partials2<2>(part, acc, lds);
}

// end of an iteration: half-step stops, residual test, rho update, iteration cap; then the start
// of the next one (breakdown check on rho, p-update coefficients). The scalars and state are loaded
// beside the partials, decided on in registers and written once.
__global__ void k_bicg_final_post(int nb, const double* __restrict__ part, double* __restrict__ sc,
                                  int* __restrict__ st, int* __restrict__ status) {
    __shared__ double lds[4 * BLOCK / WAVE];
    double rho[2], rn0[2], bd[2], alpha[2], omega[2];
    int act[2], half[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        rho[c] = sc[B_RHO + c];
        rn0[c] = sc[B_RN0 + c];
        bd[c] = sc[B_BD + c];
        alpha[c] = sc[B_ALPHA + c];
        omega[c] = sc[B_OMEGA + c];
        act[c] = st[2 + c];
        half[c] = st[8 + c];
    }
    const double tol = sc[B_TOL];
    const int state0 = st[0], it = st[10], max_iter = st[11];
    double sums[4];
    sum_partials_k<4>({part, part + 1, part + 2, part + 3}, {nb, nb, nb, nb}, 6, sums, lds);
    if (state0 != ST_RUNNING || threadIdx.x != 0) return;
    const double rr[2] = {sums[0], sums[1]}, r0r[2] = {sums[2], sums[3]};
    double rho_old[2];
    for (int c = 0; c < 2; ++c) {
        rho_old[c] = rho[c];
        if (half[c]) {
            bicg_stop(st, c, it + 1, 1);
            act[c] = 0;
        }
        if (!act[c]) continue;
        const double r_norm = sqrt(rr[c]);
        sc[B_REL + c] = r_norm / rn0[c];
        if (r_norm < tol * rn0[c] || r_norm < 1.0e-11) {
            bicg_stop(st, c, it + 1, 1);
            act[c] = 0;
            continue;
        }
        rho[c] = r0r[c];
        sc[B_RHO_OLD + c] = rho_old[c];
        sc[B_RHO + c] = rho[c];
        if (it + 1 == max_iter) {
            bicg_stop(st, c, max_iter, 0);
            act[c] = 0;
        }
    }
    st[10] = it + 1;
    if (act[0] || act[1])   // start of the next iteration
        for (int c = 0; c < 2; ++c) {
            double cb = 0.0, co = 0.0;
            if (act[c] && fabs(rho[c]) < bd[c]) {
                bicg_stop(st, c, it + 1, 0);
                act[c] = 0;
            }
            if (act[c]) {
                cb = (rho[c] / rho_old[c]) * (alpha[c] / (omega[c] + 1.0e-30));
                co = omega[c];
            }
            sc[B_CB + c] = cb;
            sc[B_CO + c] = co;
        }
    const int state = act[0] || act[1] ? ST_RUNNING : ST_STOPPED;
    st[0] = state;
    publish(status, it + 1, state);
}

// ======================================================================================================
// Host side
// ======================================================================================================
hipStream_t S(cfa_stream_t s) { return as_stream(s); }

#define CFA_TRY(expr) do { const hipError_t e_ = (expr); if (e_ != hipSuccess) return (int)e_; } while (0)

// Calls f with std::integral_constant<int, TPR> for the lanes-per-row value tpr (1..64)
template <typename F>
void tpr_dispatch(int tpr, F f) {
    switch (tpr) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        case 32: f(std::integral_constant<int, 32>{}); break;
        default: f(std::integral_constant<int, 64>{}); break;
    }
}

template <int OP, typename T = double>
void csr_op_launch(int tpr, int rows, const int* rp, const int* ci, const T* val, const T* x, const T* b,
                   const T* dinv, double omega, T* y, const int* st, hipStream_t s) {
    const int blocks = blocks_for((long long)rows * tpr);
    tpr_dispatch(tpr, [&](auto c) {
        constexpr int TPR = decltype(c)::value;
        hipLaunchKernelGGL((k_csr_op<TPR, OP, T>), dim3(blocks), dim3(BLOCK), 0, s, rows, rp, ci, val, x, b, dinv,
                           (T)omega, y, st);
    });
}

template <typename T = double>
void jacobi_from_zero_launch(int tpr, int rows, const int* rp, const int* ci, const T* val, const T* b, const T* dinv,
                             double omega, T* y, const int* st, hipStream_t s) {
    const int blocks = blocks_for((long long)rows * tpr);
    tpr_dispatch(tpr, [&](auto c) {
        constexpr int TPR = decltype(c)::value;
        hipLaunchKernelGGL((k_jacobi_from_zero<TPR, T>), dim3(blocks), dim3(BLOCK), 0, s, rows, rp, ci, val, b, dinv,
                           (T)omega, y, st);
    });
}

// Hooks of the fused PCG into the preconditioner: the iteration's residual test runs in the first
// level-0 kernel, and the last level-0 sweep emits the r.z partials.
struct PrecHooks {
    const double* prr = nullptr;   // r.r partials of the iteration (residual test when set)
    int nb_rr = 0;
    double* sc = nullptr;
    int* st_w = nullptr;
    int* status = nullptr;
    double* dot_part = nullptr;    // r.z partials out (when set)
    int dot_blocks = 0;            // set: number of r.z partials written
    // the iteration's update runs in the cycle's first launch (k_update_stage; a hierarchy coupled from
    // level 0 only): its arguments, and the parity of the iteration
    const PcgArgs* update = nullptr;
    int h = 0, nb_pq = 0;
};

// Rows per workgroup of the operator kernels and their workgroups (at most RED_BLOCKS, so that the
// consumers re-sum at most that many partials; 1536 and 2048 ran the same). 64 rows split a small mesh
// over the CUs; 128 leave room for six workgroups' LDS on a CU. Stage 1 with 64 / 128 / 256 rows:
// 6.0 / 6.3 / 8.9 us on 29k nodes; 64 / 128 rows: 11.3 / 11.2 us on 115k, 118 / 107 us on 1.84 M.
int run_rows(int n) {
    return n <= 64 * RED_BLOCKS ? 64 : 128;
}
int run_blocks(int n) { return std::min(blocks_for(n, run_rows(n)), RED_BLOCKS); }
template <typename F>
void run_dispatch(int n, F f) {
    if (run_rows(n) == 64) f(std::integral_constant<int, 64>{});
    else f(std::integral_constant<int, 128>{});
}

// last level-0 sweep into the FP64 output, with the r.z partials when part is set; returns the
// number of partials
template <typename T = double>
int jacobi_dot_launch(int rows, const int* rp, const int* ci, const T* val, const T* x, const T* b, const T* dinv,
                      double omega, double* y, const double* rdot, double* part, const int* st, hipStream_t s) {
    const int nb = run_blocks(rows);
    run_dispatch(rows, [&](auto rb) {
        constexpr int RB = decltype(rb)::value;
        hipLaunchKernelGGL((k_jacobi_dot<RB, T>), dim3(nb), dim3(BLOCK), 0, s, rows, rp, ci, val, x, b, dinv, (T)omega,
                           y, rdot, part, st);
    });
    return nb;
}

void jacobi_from_zero_check_launch(int tpr, int rows, const int* rp, const int* ci, const double* val,
                                   const double* b, const double* dinv, double omega, double* y,
                                   const PrecHooks& hk, hipStream_t s) {
    const int blocks = blocks_for((long long)rows * tpr);
    tpr_dispatch(tpr, [&](auto c) {
        constexpr int TPR = decltype(c)::value;
        hipLaunchKernelGGL(k_jacobi_from_zero_check<TPR>, dim3(blocks), dim3(BLOCK), 0, s, rows, rp, ci, val, b, dinv,
                           omega, y, hk.prr, hk.nb_rr, hk.sc, hk.st_w, hk.status);
    });
}

// MAXL (slots loaded per lane) of the sliced-ELL kernels for the level's longest row (at most
// CFA_SELL_MAX_LEN), G, the CSR lanes per row whose summation order they keep (1, 2 or 4), and NT,
// non-temporal loads when a sweep's bytes (values of vb bytes) exceed the Infinity Cache
template <typename F>
void sell_dispatch(const cfa_amg_level_t& L, int vb, F f) {
    const bool nt = (4.0 + vb) * L.a_nnz + (4.0 + 4.0 * vb) * L.rows > SELL_STREAM_BYTES;
    auto with_g = [&](auto m) {
        auto with_nt = [&](auto g) {
            if (nt) f(m, g, std::true_type{});
            else f(m, g, std::false_type{});
        };
        if (L.tpr_a == 1) with_nt(std::integral_constant<int, 1>{});
        else if (L.tpr_a == 2) with_nt(std::integral_constant<int, 2>{});
        else with_nt(std::integral_constant<int, 4>{});
    };
    const int maxl = L.s_len;
    if (maxl <= 8) with_g(std::integral_constant<int, 8>{});
    else if (maxl <= 12) with_g(std::integral_constant<int, 12>{});
    else with_g(std::integral_constant<int, 16>{});
}

// A level's sliced-ELL copy as the kernels take it
bool sell_usable(const cfa_amg_level_t& L) {
    return L.s_row && L.s_ci && L.s_v && L.s_len >= 0 && L.s_len <= CFA_SELL_MAX_LEN &&
           (L.tpr_a == 1 || L.tpr_a == 2 || L.tpr_a == 4);
}

// The level operator's sweeps and residual: on its sliced-ELL copy when it has one, else on its
// CSR rows
template <int OP, typename T>
void level_op_launch(const cfa_amg_level_t& L, const T* x, const T* b, const T* dinv, T* y, const int* st,
                     hipStream_t s) {
    static_assert(OP == OP_JACOBI || OP == OP_RESID, "the sliced-ELL copy serves the sweeps and the residual");
    if (!L.s_sp) {
        csr_op_launch<OP, T>(L.tpr_a, L.rows, L.a_rp, L.a_ci, Lv<T>::a(L), x, b, dinv, OP == OP_JACOBI ? L.omega : 0.0,
                             y, st, s);
        return;
    }
    const int pos = sell_positions(L.rows);
    sell_dispatch(L, sizeof(T), [&](auto m, auto g, auto nt) {
        constexpr int M = decltype(m)::value, G = decltype(g)::value;
        constexpr bool NT = decltype(nt)::value;
        hipLaunchKernelGGL((k_sell_op<M, G, NT, OP, T>), dim3(blocks_for(pos)), dim3(BLOCK), 0, s, pos, L.s_sp, L.s_row,
                           L.s_ci, Lv<T>::sv(L), x, b, dinv, (T)L.omega, y, st);
    });
}

template <typename T>
void level_from_zero_launch(const cfa_amg_level_t& L, const T* b, const T* dinv, T* y, const int* st, hipStream_t s) {
    if (!L.s_sp) {
        jacobi_from_zero_launch<T>(L.tpr_a, L.rows, L.a_rp, L.a_ci, Lv<T>::a(L), b, dinv, L.omega, y, st, s);
        return;
    }
    const int pos = sell_positions(L.rows);
    sell_dispatch(L, sizeof(T), [&](auto m, auto g, auto nt) {
        constexpr int M = decltype(m)::value, G = decltype(g)::value;
        constexpr bool NT = decltype(nt)::value;
        hipLaunchKernelGGL((k_sell_from_zero<M, G, NT, T>), dim3(blocks_for(pos)), dim3(BLOCK), 0, s, pos, L.s_sp,
                           L.s_row, L.s_ci, Lv<T>::sv(L), b, dinv, (T)L.omega, y, st);
    });
}

void level_from_zero_check_launch(const cfa_amg_level_t& L, const double* b, double* y, const PrecHooks& hk,
                                  hipStream_t s) {
    if (!L.s_sp) {
        jacobi_from_zero_check_launch(L.tpr_a, L.rows, L.a_rp, L.a_ci, L.a_v, b, L.dinv, L.omega, y, hk, s);
        return;
    }
    const int pos = sell_positions(L.rows);
    sell_dispatch(L, sizeof(double), [&](auto m, auto g, auto nt) {
        constexpr int M = decltype(m)::value, G = decltype(g)::value;
        constexpr bool NT = decltype(nt)::value;
        hipLaunchKernelGGL((k_sell_from_zero_check<M, G, NT>), dim3(blocks_for(pos)), dim3(BLOCK), 0, s, pos, L.s_sp,
                           L.s_row, L.s_ci, L.s_v, b, L.dinv, L.omega, y, hk.prr, hk.nb_rr, hk.sc, hk.st_w, hk.status);
    });
}

// The dense matrix is the V(2,2) cycle from its level down: other cycles go through the levels
bool dense_bottom(const cfa_amg_t* amg) { return amg->dense && amg->smooth_steps == 2; }

// The level index of the cycle's bottom: the dense level when there is one, else past the last level
int bottom_level(const cfa_amg_t* amg) { return dense_bottom(amg) ? amg->dense_level : amg->n_levels; }

// Level l and every level above the bottom carry the coupled transfers, for the V(2,2) cycle
bool coupled_from(const cfa_amg_t* amg, int l) {
    if (amg->smooth_steps != 2) return false;
    for (int k = l; k < bottom_level(amg); ++k)
        if (!amg->levels[k].w_rp) return false;
    return l < bottom_level(amg);
}

// right-hand side, result, size and matrix of the dense product at the cycle's bottom
template <typename T>
struct Bottom {
    int n;
    const double* m;
    T* b;
    T* x;
};
template <typename T>
Bottom<T> bottom_of(const cfa_amg_t* amg) {
    if (dense_bottom(amg)) {
        const cfa_amg_level_t& L = amg->levels[amg->dense_level];
        return {L.rows, amg->dense, Lv<T>::b(L), Lv<T>::x(L)};
    }
    return {amg->coarse_n, amg->coarse_inv, Lv<T>::cb(amg), Lv<T>::cx(amg)};
}

int log2_of(int tpr) {
    int s = 0;
    while ((1 << s) < tpr && s < 6) ++s;
    return s;
}

// workgroups of rows with 2^shift lanes each
int row_blocks(int rows, int shift) { return blocks_for((long long)rows << shift); }

template <typename T, typename B, typename B2>
void coupled_stage_launch(const CoupledStage<T, B, B2>& a, const cfa_amg_level_t* sell, hipStream_t s) {
    const int grid = a.zero.blocks + a.mul.blocks + a.step.blocks;
    if (grid == 0) return;
    auto go = [&](auto m, auto g) {
        constexpr int M = decltype(m)::value, G = decltype(g)::value;
        hipLaunchKernelGGL((k_coupled_stage<M, G, T, B, B2>), dim3(grid), dim3(BLOCK), 0, s, a);
    };
    if (!sell) {
        go(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
        return;
    }
    auto with_g = [&](auto m) {
        if (sell->tpr_a == 1) go(m, std::integral_constant<int, 1>{});
        else if (sell->tpr_a == 2) go(m, std::integral_constant<int, 2>{});
        else go(m, std::integral_constant<int, 4>{});
    };
    if (sell->s_len <= 8) with_g(std::integral_constant<int, 8>{});
    else if (sell->s_len <= 12) with_g(std::integral_constant<int, 12>{});
    else with_g(std::integral_constant<int, 16>{});
}

// Stage l of the descent, from level l0 (B0: the type of level l0's right-hand side b0, FP64 on level
// 0): from-zero steps of level l, its coarse right-hand side or the dense product, the first step of
// level l - 1.
template <typename T, typename B, typename B2, typename B0>
void coupled_stage(const cfa_amg_t* amg, int l0, int l, const B0* b0, const int* st, hipStream_t s, PrecHooks* hk) {
    CoupledStage<T, B, B2> a;
    std::memset(&a, 0, sizeof(a));
    const cfa_amg_level_t* sell = nullptr;
    auto use_sell = [&](const cfa_amg_level_t& L, int slot) {
        sell = &L;
        a.sell = slot;
        a.s_sp = L.s_sp; a.s_row = L.s_row; a.s_ci = L.s_ci; a.s_v = Lv<T>::sv(L);
        return blocks_for(sell_positions(L.rows));
    };
    a.sell = -1;
    a.st = const_cast<int*>(st);
    const int bottom = bottom_level(amg);
    if (l == bottom) {
        const Bottom<T> e = bottom_of<T>(amg);
        a.dense = e.m;
        a.mul.rows = e.n;
        a.mul.x = e.b;
        a.mul.y = e.x;
        a.mul.blocks = blocks_for((long long)e.n * WAVE);
    } else {
        const cfa_amg_level_t& L = amg->levels[l];
        const B* b;
        if constexpr (std::is_same<B, B0>::value) b = l == l0 ? b0 : (const B*)(const void*)Lv<T>::b(L);
        else b = (const B*)(const void*)Lv<T>::b(L);
        const int sh = log2_of(L.tpr_a), shq = log2_of(L.tpr_q);
        a.zero = {row_blocks(L.rows, sh), L.rows, sh, L.a_rp, L.a_ci, Lv<T>::a(L), nullptr, b, Lv<T>::dinv(L),
                  (T)L.omega, Lv<T>::x(L)};
        // one copy per stage: the finer level's, when both have one (the CSR rows give the same bits)
        if (L.s_sp && !(l > l0 && amg->levels[l - 1].s_sp)) a.zero.blocks = use_sell(L, 0);
        T* cb = l + 1 < bottom ? Lv<T>::b(amg->levels[l + 1]) : bottom_of<T>(amg).b;
        a.mul = {row_blocks(L.cols, shq), L.cols, shq, L.q_rp, L.q_ci, Lv<T>::q(L), nullptr, b, nullptr, T(0), cb};
    }
    if (l == (hk && hk->update ? 1 : 0) && hk && hk->prr) {
        a.prr = hk->prr; a.nb_rr = hk->nb_rr; a.sc = hk->sc; a.st = hk->st_w; a.status = hk->status;
    }
    if (l > l0) {
        const cfa_amg_level_t& F = amg->levels[l - 1];
        const B2* b;
        if constexpr (std::is_same<B2, B0>::value) b = l - 1 == l0 ? b0 : (const B2*)(const void*)Lv<T>::b(F);
        else b = (const B2*)(const void*)Lv<T>::b(F);
        const int sh = log2_of(F.tpr_a);
        a.step = {row_blocks(F.rows, sh), F.rows, sh, F.a_rp, F.a_ci, Lv<T>::a(F), Lv<T>::x(F), b, Lv<T>::dinv(F),
                  (T)F.omega, Lv<T>::ax(F)};
        if (F.s_sp) a.step.blocks = use_sell(F, 2);
    }
    coupled_stage_launch(a, sell, s);
}

// Workgroups of the from-zero rows of level 0, whose r.r partials k_update_stage leaves
int update_blocks(const cfa_amg_level_t& L) {
    return L.s_sp ? blocks_for(sell_positions(L.rows)) : row_blocks(L.rows, log2_of(L.tpr_a));
}

template <typename T>
void update_stage(const cfa_amg_t* amg, const PrecHooks& hk, hipStream_t s) {
    const cfa_amg_level_t& L = amg->levels[0];
    const PcgArgs& g = *hk.update;
    UpdateStage<T> a;
    std::memset(&a, 0, sizeof(a));
    const int sh = log2_of(L.tpr_a), shq = log2_of(L.tpr_q);
    T* cb = bottom_level(amg) > 1 ? Lv<T>::b(amg->levels[1]) : bottom_of<T>(amg).b;
    a.zero = {update_blocks(L), L.rows, sh, L.a_rp, L.a_ci, Lv<T>::a(L), nullptr, nullptr, Lv<T>::dinv(L), (T)L.omega,
              Lv<T>::x(L)};
    a.mul = {row_blocks(L.cols, shq), L.cols, shq, L.q_rp, L.q_ci, Lv<T>::q(L), nullptr, nullptr, nullptr, T(0), cb};
    a.sell = L.s_sp ? 0 : -1;
    a.s_sp = L.s_sp; a.s_row = L.s_row; a.s_ci = L.s_ci; a.s_v = L.s_sp ? Lv<T>::sv(L) : nullptr;
    a.r = g.rbuf[hk.h]; a.q = g.q; a.p = g.p[hk.h];
    a.rn = g.rbuf[1 - hk.h]; a.x = g.x;
    a.ppq = g.ppq; a.nb_pq = hk.nb_pq; a.prz = g.prz[hk.h]; a.nb_rz = g.nb_rz;
    a.prr = g.prr; a.st = g.st; a.status = g.status;
    auto go = [&](auto m) {
        hipLaunchKernelGGL((k_update_stage<decltype(m)::value, T>), dim3(a.mul.blocks + a.zero.blocks), dim3(BLOCK), 0, s,
                           a);
    };
    if (!L.s_sp) go(std::integral_constant<int, 0>{});
    else if (L.s_len <= 8) go(std::integral_constant<int, 8>{});
    else if (L.s_len <= 12) go(std::integral_constant<int, 12>{});
    else go(std::integral_constant<int, 16>{});
}

// The coupled cycle from level l0 with right-hand side b0 (FP64 on level 0, also in the FP32 cycle);
// the result in level l0's x buffer, or on level 0 in the FP64 `out`, with the r.z partials.
template <typename T, typename B0>
T* coupled_vcycle(const cfa_amg_t* amg, int l0, const B0* b0, double* out, const int* st, hipStream_t s,
                  PrecHooks* hk) {
    const int bottom = bottom_level(amg);
    for (int l = l0; l <= bottom; ++l) {
        if (l == 0 && hk && hk->update) update_stage<T>(amg, *hk, s);
        else if (l == l0) coupled_stage<T, B0, T, B0>(amg, l0, l, b0, st, s, hk);
        else if (l == l0 + 1) coupled_stage<T, T, B0, B0>(amg, l0, l, b0, st, s, hk);
        else coupled_stage<T, T, T, B0>(amg, l0, l, b0, st, s, hk);
    }
    for (int l = bottom - 1; l >= l0; --l) {
        const cfa_amg_level_t& L = amg->levels[l];
        const T* e = l + 1 < bottom ? Lv<T>::x(amg->levels[l + 1]) : bottom_of<T>(amg).x;
        if constexpr (std::is_same<B0, double>::value) {
            if (out && l == 0) {
                // rows per workgroup: one pass of at most RED_BLOCKS workgroups as long as that takes no
                // more than 256 rows each
                auto go = [&](auto rb) {
                    constexpr int RB = decltype(rb)::value;
                    const int nb = std::min(blocks_for(L.rows, RB), RED_BLOCKS);
                    hipLaunchKernelGGL((k_coupled_up_dot<RB, T>), dim3(nb), dim3(BLOCK), 0, s, L.rows, L.a_rp, L.a_ci,
                                       Lv<T>::a(L), Lv<T>::ax(L), b0, Lv<T>::dinv(L), (T)L.omega, L.w_rp, L.w_ci,
                                       Lv<T>::w(L), e, out, hk ? hk->dot_part : nullptr, st);
                    if (hk && hk->dot_part) hk->dot_blocks = nb;
                };
                if (L.rows <= 64 * RED_BLOCKS) go(std::integral_constant<int, 64>{});
                else if (L.rows <= 128 * RED_BLOCKS) go(std::integral_constant<int, 128>{});
                else go(std::integral_constant<int, 256>{});
                return nullptr;
            }
        }
        const int sh = log2_of(L.tpr_a);
        auto up = [&](auto* b) {
            using B = typename std::remove_cv<typename std::remove_pointer<decltype(b)>::type>::type;
            RowSet<T, B> r = {row_blocks(L.rows, sh), L.rows, sh, L.a_rp, L.a_ci, Lv<T>::a(L), Lv<T>::ax(L), b,
                              Lv<T>::dinv(L), (T)L.omega, Lv<T>::x(L)};
            hipLaunchKernelGGL((k_coupled_up<T, B>), dim3(r.blocks), dim3(BLOCK), 0, s, r, L.w_rp, L.w_ci, Lv<T>::w(L),
                               e, st);
        };
        if (l == l0) up(b0);
        else up((const T*)Lv<T>::b(L));
    }
    return Lv<T>::x(amg->levels[l0]);
}

// One V-cycle (src/cfa/linalg.cuh:1184-1206) for level l with right-hand side b, in FP64 or FP32
// (T). Each level's x / ax buffers form a ping-pong pair; the function returns the buffer holding
// the level's iterate. On level 0 the last smoothing step writes straight into the FP64 `out`
// when given (rdot: the FP64 residual for the r.z partials).
template <typename T>
T* vcycle(const cfa_amg_t* amg, int l, const T* b, double* out, const double* rdot, const int* st, hipStream_t s,
          PrecHooks* hk = nullptr) {
    if (coupled_from(amg, l) && (l > 0 || std::is_same<T, double>::value))
        return coupled_vcycle<T, T>(amg, l, b, l == 0 ? out : nullptr, st, s, hk);
    const cfa_amg_level_t& L = amg->levels[l];
    const int n = L.rows;
    const int ss = amg->smooth_steps;
    T* xa = Lv<T>::x(L);
    T* xb = Lv<T>::ax(L);
    const T* dv = Lv<T>::dinv(L);
    // the residual test of a fused PCG iteration (the FP32 cycle takes it in its entry kernel)
    const bool check_here = std::is_same<T, double>::value && hk && hk->prr && l == 0;
    if (ss >= 2) {
        bool done = false;
        if constexpr (std::is_same<T, double>::value) {
            if (check_here) {
                level_from_zero_check_launch(L, b, xa, *hk, s);
                done = true;
            }
        }
        if (!done) level_from_zero_launch<T>(L, b, dv, xa, st, s);
        for (int k = 2; k < ss; ++k) {
            level_op_launch<OP_JACOBI, T>(L, xa, b, dv, xb, st, s);
            std::swap(xa, xb);
        }
    } else {   // x = omega dinv b is always taken, also for fewer than one smoothing step
        if (check_here)
            hipLaunchKernelGGL(k_fp_check, dim3(1), dim3(BLOCK), 0, s, hk->prr, hk->nb_rr, hk->sc, hk->st_w, hk->status);
        hipLaunchKernelGGL(k_jacobi_init<T>, dim3(blocks_for(n)), dim3(BLOCK), 0, s, n, (T)L.omega, dv, b, xa, st);
    }
    level_op_launch<OP_RESID, T>(L, xa, b, nullptr, Lv<T>::res(L), st, s);
    const bool deeper = l + 1 < bottom_level(amg);
    const Bottom<T> bot = bottom_of<T>(amg);
    T* cb = deeper ? Lv<T>::b(amg->levels[l + 1]) : bot.b;
    csr_op_launch<OP_SPMV, T>(L.tpr_r, L.cols, L.r_rp, L.r_ci, Lv<T>::r(L), Lv<T>::res(L), nullptr, nullptr, 0.0, cb,
                              st, s);
    const T* cx;
    if (deeper) {
        cx = vcycle<T>(amg, l + 1, Lv<T>::b(amg->levels[l + 1]), nullptr, nullptr, st, s);
    } else {
        hipLaunchKernelGGL(k_dense_matvec<T>, dim3(blocks_for((long long)bot.n * WAVE)), dim3(BLOCK), 0, s, bot.n, bot.m,
                           bot.b, bot.x, st);
        cx = bot.x;
    }
    csr_op_launch<OP_ADD, T>(L.tpr_p, n, L.p_rp, L.p_ci, Lv<T>::p(L), cx, nullptr, nullptr, 0.0, xa, st, s);
    for (int k = 0; k < ss; ++k) {
        if (out && k == ss - 1) {
            // on the CSR rows: its r.z block partials keep their grouping by rows
            const int nb = jacobi_dot_launch<T>(n, L.a_rp, L.a_ci, Lv<T>::a(L), xa, b, dv, L.omega, out,
                                                rdot, hk ? hk->dot_part : nullptr, st, s);
            if (hk && hk->dot_part) hk->dot_blocks = nb;
            return nullptr;   // the result is in out
        }
        level_op_launch<OP_JACOBI, T>(L, xa, b, dv, xb, st, s);
        std::swap(xa, xb);
    }
    return xa;
}

// A hierarchy descriptor the V-cycle can run: sizes, and the FP32 arrays when use_f32 is set
bool amg_valid(const cfa_amg_t* amg) {
    if (amg->n_levels < 0 || (amg->n_levels > 0 && !amg->levels) || amg->coarse_n < 0 || amg->smooth_steps < 0)
        return false;
    if (amg->use_f32) {
        if (amg->n_levels > 0 && (!amg->cb32 || !amg->cx32)) return false;
        for (int l = 0; l < amg->n_levels; ++l) {
            const cfa_amg_level_t& L = amg->levels[l];
            if (!L.a_v32 || !L.p_v32 || !L.r_v32 || !L.dinv32 || !L.x32 || !L.b32 || !L.r32 || !L.ax32) return false;
            if (L.s_sp && !L.s_v32) return false;
        }
    }
    for (int l = 0; l < amg->n_levels; ++l) {
        const cfa_amg_level_t& L = amg->levels[l];
        if (L.s_sp && !sell_usable(L)) return false;
        if (L.w_rp && (!L.w_ci || !L.w_v || !L.q_rp || !L.q_ci || !L.q_v)) return false;
        if (L.w_rp && amg->use_f32 && (!L.w_v32 || !L.q_v32)) return false;
    }
    return !amg->dense || (amg->dense_level >= 1 && amg->dense_level < amg->n_levels);
}

// z = V-cycle(r); with hooks, the residual test first and the r.z partials last. The FP32 cycle
// (amg->use_f32) reads r through b32 and writes z in FP64.
void amg_apply_enqueue(const cfa_amg_t* amg, const double* r, double* z, const int* st, hipStream_t s,
                       PrecHooks* hk = nullptr) {
    const int n = amg->n_levels ? amg->levels[0].rows : amg->coarse_n;
    const bool f32 = amg->use_f32 && amg->n_levels > 0 && amg->smooth_steps >= 1;
    bool wrote_z = false;
    if (amg->n_levels == 0) {
        if (hk && hk->prr)
            hipLaunchKernelGGL(k_fp_check, dim3(1), dim3(BLOCK), 0, s, hk->prr, hk->nb_rr, hk->sc, hk->st_w, hk->status);
        hipLaunchKernelGGL(k_dense_matvec<double>, dim3(blocks_for((long long)amg->coarse_n * WAVE)), dim3(BLOCK), 0, s,
                           amg->coarse_n, amg->coarse_inv, r, z, st);
    } else if (f32 && coupled_from(amg, 0)) {   // r is read in FP64 where the level-0 kernels use it
        (void)coupled_vcycle<float, double>(amg, 0, r, z, st, s, hk);
        wrote_z = true;
    } else if (f32) {
        float* b32 = amg->levels[0].b32;
        hipLaunchKernelGGL(k_to_f32_check, dim3(red_blocks(n)), dim3(BLOCK), 0, s, n, r, b32,
                           hk ? hk->prr : nullptr, hk ? hk->nb_rr : 0, hk ? hk->sc : nullptr,
                           hk && hk->prr ? hk->st_w : const_cast<int*>(st), hk ? hk->status : nullptr);
        (void)vcycle<float>(amg, 0, b32, z, r, st, s, hk);
        wrote_z = true;
    } else {
        double* res = vcycle<double>(amg, 0, r, z, r, st, s, hk);
        wrote_z = res == nullptr;
        if (!wrote_z) hipLaunchKernelGGL(k_copy, dim3(blocks_for(n)), dim3(BLOCK), 0, s, n, res, z, st);
    }
    if (hk && hk->dot_part && !wrote_z) {
        hk->dot_blocks = red_blocks(n);
        hipLaunchKernelGGL(k_dot_partial, dim3(hk->dot_blocks), dim3(BLOCK), 0, s, n, r, z, hk->dot_part, st);
    }
}

// First colour of the trailing run that k_ilu_tail takes (n_colours when fewer than two colours qualify)
int ilu_tail_first(const cfa_ilu_t* ilu) {
    const int nc = ilu->n_colours;
    int t = nc;
    while (t > 1 && nc - t < ILU_TAIL_COLOURS && ilu->colour_start[t] - ilu->colour_start[t - 1] <= ILU_TAIL_ROWS) --t;
    return nc - t >= 2 ? t : nc;
}

// The sweeps after the permutation into colour order (r_perm, and colour 0 in z_perm): colours 1..
// forward, colours nc-2..1 backward (the trailing small ones in one launch), colour 0 backward with the
// permutation back (the last colour has no U entries)
template <int NRHS, typename T>
void ilu_sweeps(const cfa_ilu_t* ilu, const T* lv, const T* uv, const T* dinv, double* z, const int* st,
                hipStream_t s) {
    const int nc = ilu->n_colours, n = ilu->n;
    if (nc == 0) return;
    double* rp = ilu->r_perm;
    double* zp = ilu->z_perm;
    const int m0 = ilu->colour_start[1] - ilu->colour_start[0];
    // forward sweeps with the FP32 factors (mixed precision): two lanes per row; FP64: one lane, the
    // reference's order (the backward sweeps take one lane either way: two were no faster)
    constexpr bool lanes = std::is_same<T, float>::value;
    // the one-lane sweeps on the sliced-ELL rows when the factor has them
    const T* slv = std::is_same<T, float>::value ? (const T*)(const void*)ilu->s_lv32 : (const T*)(const void*)ilu->s_lv;
    const T* suv = std::is_same<T, float>::value ? (const T*)(const void*)ilu->s_uv32 : (const T*)(const void*)ilu->s_uv;
    const bool sell_l = ilu->s_lrow && slv && ilu->s_pos0, sell_u = ilu->s_urow && suv && ilu->s_pos0;
    auto sell_sweep = [&](auto upper, int c, int len, const int* srow, const int* sp, const int* sc, const T* sv) {
        const int cs = ilu->colour_start[c], mpos = (ilu->colour_start[c + 1] - cs + 63) / 64 * 64;
        auto go = [&](auto mx) {
            constexpr int M = decltype(mx)::value;
            constexpr bool U = decltype(upper)::value;
            hipLaunchKernelGGL((k_ilu_sweep_sell<NRHS, M, U, T>), dim3(blocks_for(mpos)), dim3(BLOCK), 0, s, mpos, n,
                               cs, ilu->s_pos0[c], srow, sp, sc, sv, dinv + cs, (!U && c == nc - 1) ? 1 : 0, rp, zp,
                               st);
        };
        if (len <= 8) go(std::integral_constant<int, 8>{});
        else if (len <= 12) go(std::integral_constant<int, 12>{});
        else go(std::integral_constant<int, 16>{});
    };
    const int tail = ilu_tail_first(ilu);
    for (int c = 1; c < tail; ++c) {
        const int cs = ilu->colour_start[c], m = ilu->colour_start[c + 1] - cs;
        if (m == 0) continue;
        if (!lanes && sell_l)
            sell_sweep(std::false_type{}, c, ilu->s_llen, ilu->s_lrow, ilu->s_lsp, ilu->s_lc, slv);
        else if constexpr (lanes)
            hipLaunchKernelGGL((k_ilu_lower_lanes<NRHS, 2>), dim3(blocks_for(2LL * m)), dim3(BLOCK), 0, s, m, n, cs,
                               ilu->lp + cs, ilu->lc, lv, dinv + cs, c == nc - 1 ? 1 : 0, rp, zp, st);
        else
            hipLaunchKernelGGL((k_ilu_lower<NRHS, T>), dim3(blocks_for(m)), dim3(BLOCK), 0, s, m, n, cs, ilu->lp + cs,
                               ilu->lc, lv, dinv + cs, c == nc - 1 ? 1 : 0, rp, zp, st);
    }
    if (tail < nc) {
        IluTail a;
        a.first = tail;
        a.nc = nc;
        for (int c = tail; c <= nc; ++c) a.start[c - tail] = ilu->colour_start[c];
        hipLaunchKernelGGL((k_ilu_tail<NRHS, T>), dim3(1), dim3(ILU_TAIL_THREADS), 0, s, n, a, ilu->lp, ilu->lc, lv,
                           ilu->up, ilu->uc, uv, dinv, rp, zp, st);
    }
    for (int c = std::min(nc - 2, tail - 1); c >= 1; --c) {
        const int cs = ilu->colour_start[c], m = ilu->colour_start[c + 1] - cs;
        if (m == 0) continue;
        if (sell_u) {
            sell_sweep(std::true_type{}, c, ilu->s_ulen, ilu->s_urow, ilu->s_usp, ilu->s_uc, suv);
            continue;
        }
        hipLaunchKernelGGL((k_ilu_upper<NRHS, T>), dim3(blocks_for(m)), dim3(BLOCK), 0, s, m, n, cs, ilu->up + cs,
                           ilu->uc, uv, dinv + cs, zp, st);
    }
    if (nc >= 2)
        hipLaunchKernelGGL((k_ilu_last_unpermute<NRHS, T>), dim3(blocks_for(n)), dim3(BLOCK), 0, s, n, m0, ilu->pos,
                           ilu->up, ilu->uc, uv, dinv, zp, z, st);
    else
        hipLaunchKernelGGL((k_ilu_unpermute<NRHS>), dim3(blocks_for(n)), dim3(BLOCK), 0, s, n, ilu->pos, zp, z, st);
}

// Calls f with the factor's values in the precision applied: (lv, uv, dinv)
template <typename F>
void ilu_values(const cfa_ilu_t* ilu, int use_f32, F f) {
    if (use_f32 && ilu->lv32) f((const float*)ilu->lv32, (const float*)ilu->uv32, (const float*)ilu->dinv32);
    else f((const double*)ilu->lv, (const double*)ilu->uv, (const double*)ilu->dinv);
}

template <int NRHS>
void ilu_apply_impl(const cfa_ilu_t* ilu, const double* r, double* z, hipStream_t s) {
    const int nc = ilu->n_colours, n = ilu->n;
    if (n == 0 || nc == 0) return;
    ilu_values(ilu, 0, [&](auto lv, auto uv, auto dinv) {
        using T = typename std::remove_const<typename std::remove_pointer<decltype(lv)>::type>::type;
        hipLaunchKernelGGL((k_ilu_permute_first<NRHS, T>), dim3(blocks_for(n)), dim3(BLOCK), 0, s, n,
                           ilu->colour_start[1] - ilu->colour_start[0], ilu->pos, r, dinv, nc == 1 ? 1 : 0, ilu->r_perm,
                           ilu->z_perm, nullptr);
        ilu_sweeps<NRHS, T>(ilu, lv, uv, dinv, z, nullptr, s);
    });
}

// Host wait on the progress word: returns when progress >= target, the solve stopped, or the
// stream is idle.
void wait_progress(const cfa_krylov_ws_t* ws, int target, hipStream_t s) {
    volatile int* st = ws->status_host;
    for (int spin = 0;; ++spin) {
        if (st[0] >= target || st[1] != ST_RUNNING) return;
        if ((spin & 63) == 63) {
            if (hipStreamQuery(s) == hipSuccess) return;
            std::this_thread::yield();
        }
    }
}

int* state_words(cfa_krylov_ws_t* ws) { return reinterpret_cast<int*>(ws->scal + 40); }

// Captured iteration graphs, keyed by everything the captured launches depend on
struct IterGraph {
    std::vector<unsigned char> key;
    hipGraphExec_t exec = nullptr;
    unsigned long long used = 0;
};
struct WsInternal {
    hipStream_t cap = nullptr;
    IterGraph pcg[GRAPH_CACHE], bicg[GRAPH_CACHE];
    unsigned long long clock = 0;
    bool capture_broken = false;
};

WsInternal* internal_of(cfa_krylov_ws_t* ws) {
    if (!ws->internal) ws->internal = new WsInternal();
    return static_cast<WsInternal*>(ws->internal);
}

struct KeyBuilder {
    std::vector<unsigned char> k;
    template <typename T>
    void add(const T& v) {
        const unsigned char* p = reinterpret_cast<const unsigned char*>(&v);
        k.insert(k.end(), p, p + sizeof(T));
    }
    void add_bytes(const void* p, size_t n) {
        const unsigned char* q = static_cast<const unsigned char*>(p);
        k.insert(k.end(), q, q + n);
    }
};

// The cached graph for `key` (least recently used slot replaced), captured from `enqueue`;
// nullptr when capture is unavailable (the caller then launches directly).
template <typename F>
hipGraphExec_t iteration_graph(cfa_krylov_ws_t* ws, IterGraph* cache, const std::vector<unsigned char>& key,
                               F enqueue) {
    WsInternal* in = internal_of(ws);
    if (!ws->use_graphs || in->capture_broken) return nullptr;
    IterGraph* slot = &cache[0];
    for (int k = 0; k < GRAPH_CACHE; ++k) {
        if (cache[k].exec && cache[k].key == key) {
            cache[k].used = ++in->clock;
            return cache[k].exec;
        }
        if (cache[k].used < slot->used) slot = &cache[k];
    }
    if (slot->exec) { (void)hipGraphExecDestroy(slot->exec); slot->exec = nullptr; }
    if (!in->cap && hipStreamCreateWithFlags(&in->cap, hipStreamNonBlocking) != hipSuccess) {
        in->cap = nullptr;
        in->capture_broken = true;
        (void)hipGetLastError();
        return nullptr;
    }
    hipGraph_t graph = nullptr;
    bool ok = hipStreamBeginCapture(in->cap, hipStreamCaptureModeRelaxed) == hipSuccess;
    if (ok) {
        enqueue(in->cap);
        ok = hipStreamEndCapture(in->cap, &graph) == hipSuccess && graph;
    }
    if (ok) ok = hipGraphInstantiate(&slot->exec, graph, nullptr, nullptr, 0) == hipSuccess;
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    if (!ok) {
        slot->exec = nullptr;
        in->capture_broken = true;
        return nullptr;
    }
    slot->key = key;
    slot->used = ++in->clock;
    return slot->exec;
}

// The iteration loop shared by both solvers: enqueue iterations (graph replay or direct
// launches), staying LOOKAHEAD iterations ahead of the progress the device has published.
template <typename F>
int run_iterations(cfa_krylov_ws_t* ws, hipGraphExec_t graph, int max_iter, F enqueue, hipStream_t s) {
    for (int it = 0; it < max_iter; ++it) {
        if (it >= LOOKAHEAD) {
            wait_progress(ws, it - LOOKAHEAD + 1, s);
            if (ws->status_host[1] != ST_RUNNING) break;
        }
        if (graph) CFA_TRY(hipGraphLaunch(graph, s));
        else enqueue(s);
    }
    return launch_status();
}

}  // namespace

extern "C" {

int cfa_krylov_ws_release(cfa_krylov_ws_t* ws) {
    if (!ws || !ws->internal) return CFA_OK;
    WsInternal* in = static_cast<WsInternal*>(ws->internal);
    for (int k = 0; k < GRAPH_CACHE; ++k) {
        if (in->pcg[k].exec) (void)hipGraphExecDestroy(in->pcg[k].exec);
        if (in->bicg[k].exec) (void)hipGraphExecDestroy(in->bicg[k].exec);
    }
    if (in->cap) (void)hipStreamDestroy(in->cap);
    delete in;
    ws->internal = nullptr;
    return CFA_OK;
}

int cfa_spmv(int n, const int* rp, const int* ci, const double* val, const double* x, double* y, int nrhs,
             cfa_stream_t stream) {
    if (n < 0 || !rp || !ci || !val || !x || !y || nrhs < 1 || nrhs > 2) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    // the mesh matrices (5-9 entries per row): two lanes per row from 20k rows (measured fastest
    // for the level-0 sweeps of the same pattern), a group of eight on small, latency-bound meshes
    auto launch = [&](auto c) {
        constexpr int TPR = decltype(c)::value;
        const int blocks = blocks_for((long long)n * TPR);
        if (nrhs == 1)
            hipLaunchKernelGGL((k_spmv_multi<TPR, 1>), dim3(blocks), dim3(BLOCK), 0, S(stream), n, rp, ci, val, x, y);
        else
            hipLaunchKernelGGL((k_spmv_multi<TPR, 2>), dim3(blocks), dim3(BLOCK), 0, S(stream), n, rp, ci, val, x, y);
    };
    if (n >= 20000) launch(std::integral_constant<int, 2>{});
    else launch(std::integral_constant<int, 8>{});
    return launch_status();
}

int cfa_dot(int n, const double* x, const double* y, double* result, double* ws, cfa_stream_t stream) {
    if (n < 0 || !x || !y || !result || !ws) return CFA_E_ARG;
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(BLOCK), 0, S(stream), n, x, y, ws, nullptr);
    hipLaunchKernelGGL(k_sum_to, dim3(1), dim3(BLOCK), 0, S(stream), nb, ws, ws + RED_BLOCKS, 0);
    const int rc = launch_status();
    if (rc) return rc;
    CFA_TRY(hipMemcpyAsync(result, ws + RED_BLOCKS, sizeof(double), hipMemcpyDeviceToHost, S(stream)));
    CFA_TRY(hipStreamSynchronize(S(stream)));
    return CFA_OK;
}

int cfa_axpy(int n, double a, const double* x, double* y, cfa_stream_t stream) {
    if (n < 0 || !x || !y) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    hipLaunchKernelGGL(k_axpy, dim3(blocks_for(n)), dim3(BLOCK), 0, S(stream), n, a, x, y);
    return launch_status();
}

int cfa_xpay(int n, const double* x, double b, double* y, cfa_stream_t stream) {
    if (n < 0 || !x || !y) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    hipLaunchKernelGGL(k_xpay, dim3(blocks_for(n)), dim3(BLOCK), 0, S(stream), n, x, b, y);
    return launch_status();
}

int cfa_vec_mul(int n, const double* a, const double* b, double* out, cfa_stream_t stream) {
    if (n < 0 || !a || !b || !out) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    hipLaunchKernelGGL(k_vec_mul, dim3(blocks_for(n)), dim3(BLOCK), 0, S(stream), n, a, b, out, nullptr);
    return launch_status();
}

int cfa_inv_diag(int n, const int* rp, const int* ci, const double* val, double eps, double* inv_diag,
                 cfa_stream_t stream) {
    if (n < 0 || !rp || !ci || !val || !inv_diag) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    hipLaunchKernelGGL(k_inv_diag, dim3(blocks_for(n)), dim3(BLOCK), 0, S(stream), n, rp, ci, val, eps, inv_diag);
    return launch_status();
}

int cfa_amg_apply(const cfa_amg_t* amg, const double* r, double* z, cfa_stream_t stream) {
    if (!amg || !r || !z || !amg_valid(amg)) return CFA_E_ARG;
    amg_apply_enqueue(amg, r, z, nullptr, S(stream));
    return launch_status();
}

}  // extern "C"

namespace {

// PCG with the reductions folded into the consuming kernels (k_fp_*), two iterations per
// captured graph (the search direction and the r.z partials alternate between two buffers).
// Same algorithm, guards and stopping rules as the reference (src/cfa/linalg.cuh:183-256).
void launch_fp_operator(bool oss, hipStream_t s, const PcgArgs& a, int h) {
    run_dispatch(a.n, [&](auto rb) {
        constexpr int RB = decltype(rb)::value;
        if (oss) hipLaunchKernelGGL((k_fp_operator<RB, true>), dim3(run_blocks(a.n)), dim3(BLOCK), 0, s, a, h);
        else hipLaunchKernelGGL((k_fp_operator<RB, false>), dim3(run_blocks(a.n)), dim3(BLOCK), 0, s, a, h);
    });
}
void launch_apply_K_B(hipStream_t s, int n, const int* rp, const int* ci, const double* val,
                      const double* oss, const double* inv_m, const double* in, double* q, double* gx, double* gy,
                      const int* st) {
    run_dispatch(n, [&](auto rb) {
        constexpr int RB = decltype(rb)::value;
        hipLaunchKernelGGL(k_apply_K_B<RB>, dim3(run_blocks(n)), dim3(BLOCK), 0, s, n, rp, ci, val, oss, inv_m, in,
                           q, gx, gy, st);
    });
}
// returns the number of partials
int launch_apply_BT_dot(hipStream_t s, int n, const int* rp, const int* ci, const double* oss,
                        const int* tag, OutletMode om, const double* gx, const double* gy, const double* p, double* q,
                        double* part, const int* st) {
    run_dispatch(n, [&](auto rb) {
        constexpr int RB = decltype(rb)::value;
        hipLaunchKernelGGL(k_apply_BT_dot<RB>, dim3(run_blocks(n)), dim3(BLOCK), 0, s, n, rp, ci, oss, tag, om, gx,
                           gy, p, q, part, st);
    });
    return run_blocks(n);
}

// pressure-Dirichlet rows of the operator: node p_pin with the outlet Dirichlet condition, else outlet nodes
OutletMode outlet_of(const cfa_oss_op_t* oss) {
    return OutletMode{oss->outlet_dirichlet, oss->p_pin, 0.0};
}

// Where the outcome kernels write: the mapped words, or the head of the (then idle) partials for a
// workspace without a device view of them, from where outcome_arrived copies them
int* outcome_words(const cfa_krylov_ws_t* ws) {
    return ws->status_dev ? ws->status_dev : reinterpret_cast<int*>(ws->part);
}
int outcome_arrived(const cfa_krylov_ws_t* ws, hipStream_t s) {
    if (!ws->status_dev)
        CFA_TRY(hipMemcpyAsync(ws->status_host + 2, outcome_words(ws) + 2, 12 * sizeof(int), hipMemcpyDeviceToHost, s));
    CFA_TRY(hipStreamSynchronize(s));
    return CFA_OK;
}

// k_pcg_outcome's words as the solve's result
void pcg_outcome(const cfa_krylov_ws_t* ws, int max_iter, cfa_solve_result_t* result) {
    const volatile int* w = ws->status_host;
    const int state = w[2];
    const bool capped = state == ST_RUNNING || state == ST_CAPPED;   // iteration cap
    result->iters[0] = capped ? max_iter : w[3];
    result->converged[0] = !capped && state != ST_STOPPED;
    result->rel_residual[0] = published_double(w + 4);
}

int pcg_fused(int n, const int* rp, const int* ci, const double* val, const double* b, double* x, int max_iter,
              double tol, const cfa_oss_op_t* oss, const cfa_amg_t* amg, cfa_krylov_ws_t* ws,
              cfa_solve_result_t* result, hipStream_t s) {
    PcgArgs a;
    std::memset(&a, 0, sizeof(a));   // the graph key compares the bytes, padding included
    a.n = n;
    a.max_iter = max_iter;
    a.rp = rp; a.ci = ci; a.val = val;
    a.r = ws->vec[0]; a.z = ws->vec[1]; a.p[0] = ws->vec[2]; a.q = ws->vec[3]; a.p[1] = ws->vec[5];
    double* inv_diag = ws->vec[4];
    a.inv_diag = inv_diag;
    a.x = x;
    a.rbuf[0] = a.r;
    a.rbuf[1] = ws->vec[6];
    // The update in the cycle's first launch where a launch costs more than what it adds: both gathers of
    // every level-0 entry of A and W^T, and the residual test's sums in every workgroup of the next stage.
    // Time steps merged / apart: 2.53 / 2.60 ms on 29k nodes, 4.85 / 4.74 ms on 115k; the line between them
    // is not measured. Its partials, one per workgroup of tpr_a lanes a row, can be up to 16384: the check is
    // what keeps them in their segment.
    const bool merged = amg && amg->n_levels > 0 && coupled_from(amg, 0) && n <= UPDATE_STAGE_ROWS &&
                        update_blocks(amg->levels[0]) <= OP_BLOCKS;
    // block partials: four segments of OP_BLOCKS doubles, then the prologue's (5 * 4096 of the
    // workspace's 8 * 4096)
    a.prz[0] = ws->part; a.prz[1] = ws->part + OP_BLOCKS; a.ppq = ws->part + 2 * OP_BLOCKS;
    a.prr = ws->part + 3 * OP_BLOCKS;
    double* scratch = ws->part + 4 * OP_BLOCKS;
    a.sc = ws->scal; a.st = state_words(ws); a.status = ws->status_dev;
    if (oss) {
        a.oss = oss->oss_val; a.inv_m = oss->inv_m; a.tag = oss->bc_tag; a.gx = oss->gx; a.gy = oss->gy;
        a.om = outlet_of(oss);
    }
    ws->status_host[0] = 0;
    ws->status_host[1] = ST_RUNNING;
    const int nb = red_blocks(n);
    const int blocks = blocks_for(n);
    const int nb_op = run_blocks(n);
    const int* st_r = a.st;

    // prologue (linalg.cuh:205-227): r = b - A x, ||b||, x = 0 when trivial, initial test, z = M^-1 r
    if (!amg) hipLaunchKernelGGL(k_inv_diag, dim3(blocks), dim3(BLOCK), 0, s, n, rp, ci, val, 1.0e-14, inv_diag);
    if (oss) {
        launch_apply_K_B(s, n, rp, ci, val, a.oss, a.inv_m, x, a.q, a.gx, a.gy, nullptr);
        (void)launch_apply_BT_dot(s, n, rp, ci, a.oss, a.tag, a.om, a.gx, a.gy, a.q, a.q, scratch, nullptr);
    } else {
        csr_op_launch<OP_SPMV, double>(2, n, rp, ci, val, x, nullptr, nullptr, 0.0, a.q, nullptr, s);
    }
    hipLaunchKernelGGL(k_pcg_residual, dim3(nb), dim3(BLOCK), 0, s, n, b, a.q, a.r, scratch, a.prr);
    hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(BLOCK), 0, s, nb, scratch, a.prr, tol, a.sc, a.st, a.status);
    hipLaunchKernelGGL(k_zero_if_trivial, dim3(blocks), dim3(BLOCK), 0, s, n, x, st_r);
    auto apply_prec = [&](int h_next, bool check, hipStream_t q_s) {
        if (amg) {
            PrecHooks hk;
            if (check) {
                hk.prr = a.prr; hk.nb_rr = nb; hk.sc = a.sc; hk.st_w = a.st; hk.status = a.status;
            }
            hk.dot_part = a.prz[h_next];
            amg_apply_enqueue(amg, a.r, a.z, st_r, q_s, &hk);
            return hk.dot_blocks;
        }
        hipLaunchKernelGGL(k_fp_jacobi_prec, dim3(nb), dim3(BLOCK), 0, q_s, a, h_next, check ? 1 : 0);
        return nb;
    };
    a.nb_rz = apply_prec(0, false, s);
    a.nb_rr = merged ? update_blocks(amg->levels[0]) : nb;
    int rc = launch_status();
    if (rc) return rc;

    // iteration k with parity h (linalg.cuh:231-253)
    auto iteration = [&](int h, hipStream_t q_s) {
        launch_fp_operator(oss != nullptr, q_s, a, h);
        if (oss)
            (void)launch_apply_BT_dot(q_s, n, rp, ci, a.oss, a.tag, a.om, a.gx, a.gy, a.p[h], a.q, a.ppq, st_r);
        if (merged) {
            PrecHooks hk;
            hk.prr = a.prr; hk.nb_rr = a.nb_rr; hk.sc = a.sc; hk.st_w = a.st; hk.status = a.status;
            hk.dot_part = a.prz[1 - h];
            hk.update = &a; hk.h = h; hk.nb_pq = nb_op;
            amg_apply_enqueue(amg, a.rbuf[1 - h], a.z, st_r, q_s, &hk);
            return;
        }
        hipLaunchKernelGGL(k_fp_update, dim3(nb), dim3(BLOCK), 0, q_s, a, h, nb_op);
        (void)apply_prec(1 - h, true, q_s);
    };
    auto two_iterations = [&](hipStream_t q_s) {
        iteration(0, q_s);
        iteration(1, q_s);
    };
    hipGraphExec_t graph = nullptr;
    if (max_iter > 0) {
        // graph key: every pointer, size and constant the launches bake in
        KeyBuilder kb;
        kb.add(a);
        kb.add(oss != nullptr);
        kb.add(amg != nullptr);
        if (amg) {
            kb.add(amg->n_levels); kb.add(amg->coarse_n); kb.add(amg->coarse_inv); kb.add(amg->cb); kb.add(amg->cx);
            kb.add(amg->smooth_steps); kb.add(amg->cb32); kb.add(amg->cx32); kb.add(amg->use_f32);
            kb.add(amg->dense_level); kb.add(amg->dense);
            if (amg->n_levels > 0) kb.add_bytes(amg->levels, sizeof(cfa_amg_level_t) * (size_t)amg->n_levels);
        }
        graph = iteration_graph(ws, internal_of(ws)->pcg, kb.k, two_iterations);
    }
    for (int g = 0; 2 * g < max_iter; ++g) {
        if (g >= 2) {
            wait_progress(ws, 2 * g - 3, s);
            if (ws->status_host[1] != ST_RUNNING) break;
        }
        if (graph) CFA_TRY(hipGraphLaunch(graph, s));
        else two_iterations(s);
    }
    hipLaunchKernelGGL(k_pcg_outcome, dim3(1), dim3(1), 0, s, a.sc, a.st, outcome_words(ws));
    rc = launch_status();
    if (rc) return rc;
    rc = outcome_arrived(ws, s);
    if (rc) return rc;
    pcg_outcome(ws, max_iter, result);
    return launch_status();
}

}  // namespace

extern "C" {

int cfa_to_f32(size_t n, const double* in, float* out, cfa_stream_t stream) {
    if ((n > 0 && (!in || !out))) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    const int blocks = (int)std::min<size_t>((n + BLOCK - 1) / BLOCK, 4096);
    hipLaunchKernelGGL(k_f64_to_f32, dim3(blocks), dim3(BLOCK), 0, S(stream), n, in, out);
    return launch_status();
}

int cfa_amg_smooth(const cfa_amg_t* amg, int level, const double* x, const double* b, double* y,
                   cfa_stream_t stream) {
    if (!amg || !x || !b || !y || level < 0 || level >= amg->n_levels || !amg->levels) return CFA_E_ARG;
    const cfa_amg_level_t& L = amg->levels[level];
    if (L.s_sp && !sell_usable(L)) return CFA_E_ARG;
    level_op_launch<OP_JACOBI, double>(L, x, b, L.dinv, y, nullptr, S(stream));
    return launch_status();
}

int cfa_amg_smooth_f32(const cfa_amg_t* amg, int level, const float* x, const float* b, float* y,
                       cfa_stream_t stream) {
    if (!amg || !x || !b || !y || level < 0 || level >= amg->n_levels || !amg->levels) return CFA_E_ARG;
    const cfa_amg_level_t& L = amg->levels[level];
    if (!amg->use_f32 || !L.a_v32 || !L.dinv32 || (L.s_sp && !L.s_v32)) return CFA_E_NOTREADY;
    if (L.s_sp && !sell_usable(L)) return CFA_E_ARG;
    level_op_launch<OP_JACOBI, float>(L, x, b, L.dinv32, y, nullptr, S(stream));
    return launch_status();
}

size_t cfa_sell_ws_bytes(int rows) {
    if (rows < 0) return 0;
    const int slices = sell_positions(rows) / SELL_SLICE;
    const size_t scan = cfa_scan_counts_ws_bytes(slices);
    return scan ? ((size_t)slices * sizeof(int) + 255) / 256 * 256 + scan : 0;
}

int cfa_sell_plan(int rows, const int* rp, int* sell_row, int* sell_sp, int* info, void* ws, size_t ws_bytes,
                  cfa_stream_t stream) {
    if (rows < 0 || !info || !sell_sp) return CFA_E_ARG;
    if (rows > 0 && (!rp || !sell_row)) return CFA_E_ARG;
    const size_t need = cfa_sell_ws_bytes(rows);
    if (need == 0 || !ws || ws_bytes < need) return CFA_E_ARG;
    const hipStream_t s = S(stream);
    const int positions = sell_positions(rows), slices = positions / SELL_SLICE;
    int* cnt = static_cast<int*>(ws);
    const size_t cnt_bytes = ((size_t)slices * sizeof(int) + 255) / 256 * 256;
    CFA_TRY(hipMemsetAsync(info, 0, 2 * sizeof(int), s));
    if (rows > 0)
        hipLaunchKernelGGL(k_sell_plan, dim3(blocks_for(rows, SELL_WINDOW)), dim3(SELL_WINDOW), 0, s, rows, positions,
                           rp, sell_row, cnt, info);
    const int e = launch_status();
    if (e != CFA_OK) return e;
    return cfa_scan_counts(slices, cnt, sell_sp, info, static_cast<unsigned char*>(ws) + cnt_bytes, need - cnt_bytes,
                           stream);
}

int cfa_sell_fill(int rows, const int* rp, const int* ci, const double* val, const int* sell_row,
                  const int* sell_sp, int* sell_ci, double* sell_v, cfa_stream_t stream) {
    if (rows < 0) return CFA_E_ARG;
    if (rows == 0) return CFA_OK;
    if (!rp || !ci || !val || !sell_row || !sell_sp || !sell_ci || !sell_v) return CFA_E_ARG;
    const int positions = sell_positions(rows);
    hipLaunchKernelGGL(k_sell_fill, dim3(blocks_for(positions)), dim3(BLOCK), 0, S(stream), positions, rp, ci, val,
                       sell_row, sell_sp, sell_ci, sell_v);
    return launch_status();
}

int cfa_pcg_operator(int n, const int* rp, const int* ci, const double* val, const cfa_oss_op_t* oss,
                     const double* in, double* out, double* part, int stage, cfa_stream_t stream) {
    if (n < 0 || !rp || !ci || !val || !oss || !in || !out || !part || stage < 0 || stage > 2) return CFA_E_ARG;
    if (!oss->oss_val || !oss->inv_m || !oss->bc_tag || !oss->gx || !oss->gy) return CFA_E_ARG;
    if (oss->outlet_dirichlet && n > 0 && (oss->p_pin < 0 || oss->p_pin >= n)) return CFA_E_ARG;
    if (n == 0) return CFA_OK;
    hipStream_t s = S(stream);
    if (stage != 2)
        launch_apply_K_B(s, n, rp, ci, val, oss->oss_val, oss->inv_m, in, out, oss->gx, oss->gy, nullptr);
    if (stage != 1)
        (void)launch_apply_BT_dot(s, n, rp, ci, oss->oss_val, oss->bc_tag, outlet_of(oss), oss->gx, oss->gy, in,
                                  out, part, nullptr);
    return launch_status();
}

int cfa_pcg(int n, const int* rp, const int* ci, const double* val, const double* b, double* x, int max_iter,
            double tol, const cfa_oss_op_t* oss, cfa_op_cb extra_cb, void* extra_ctx, const cfa_amg_t* amg,
            cfa_op_cb prec_cb, void* prec_ctx, cfa_krylov_ws_t* ws, cfa_solve_result_t* result,
            cfa_stream_t stream) {
    if (n < 0 || !rp || !ci || !val || !b || !x || !ws || !result || ws->cap < n || !ws->status_host || max_iter < 0)
        return CFA_E_ARG;
    if (oss && (!oss->oss_val || !oss->inv_m || !oss->bc_tag || !oss->gx || !oss->gy)) return CFA_E_ARG;
    if (oss && oss->outlet_dirichlet && n > 0 && (oss->p_pin < 0 || oss->p_pin >= n)) return CFA_E_ARG;
    if (amg && !amg_valid(amg)) return CFA_E_ARG;
    hipStream_t s = S(stream);
    result->iters[0] = 0;
    result->converged[0] = 1;
    result->rel_residual[0] = -1.0;   // no residual computed (trivial or initial convergence)
    if (n == 0) return CFA_OK;
    if (!extra_cb && !prec_cb) return pcg_fused(n, rp, ci, val, b, x, max_iter, tol, oss, amg, ws, result, s);
    // solves with host callbacks: the iteration as separate kernels with one-workgroup finals
    double* r = ws->vec[0];
    double* z = ws->vec[1];
    double* p = ws->vec[2];
    double* q = ws->vec[3];
    double* inv_diag = ws->vec[4];
    double* part = ws->part;
    double* sc = ws->scal;
    int* st = state_words(ws);
    int* status = ws->status_dev;
    const int nb = red_blocks(n);
    const int blocks = blocks_for(n);
    constexpr int TPR = 4;
    ws->status_host[0] = 0;
    ws->status_host[1] = ST_RUNNING;

    auto apply_op = [&](const double* in, double* out, hipStream_t q_s) {
        if (oss) {
            launch_apply_K_B(q_s, n, rp, ci, val, oss->oss_val, oss->inv_m, in, out, oss->gx, oss->gy, st);
        } else {
            csr_op_launch<OP_SPMV, double>(TPR, n, rp, ci, val, in, nullptr, nullptr, 0.0, out, st, q_s);
            if (extra_cb) extra_cb(in, out, extra_ctx);
        }
    };
    // second stage of the fused operator (q -= B^T g) with the p.q partials, or a plain dot
    auto finish_op_dot = [&](const double* pv, double* qv, hipStream_t q_s) {
        if (oss) {
            return launch_apply_BT_dot(q_s, n, rp, ci, oss->oss_val, oss->bc_tag, outlet_of(oss), oss->gx, oss->gy,
                                       pv, qv, part, st);
        }
        hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(BLOCK), 0, q_s, n, pv, qv, part, st);
        return nb;
    };
    auto apply_prec = [&](const double* rv, double* zv, hipStream_t q_s) {
        if (amg) amg_apply_enqueue(amg, rv, zv, st, q_s);
        else if (prec_cb) prec_cb(rv, zv, prec_ctx);
        else hipLaunchKernelGGL(k_vec_mul, dim3(blocks), dim3(BLOCK), 0, q_s, n, inv_diag, rv, zv, st);
    };

    // prologue (src/cfa/linalg.cuh:205-227), all decisions on the device (the state is set by k_pcg_init;
    // until then the kernels run whatever an earlier solve left there)
    hipLaunchKernelGGL(k_pcg_start, dim3(1), dim3(1), 0, s, st);
    if (!amg && !prec_cb)
        hipLaunchKernelGGL(k_inv_diag, dim3(blocks), dim3(BLOCK), 0, s, n, rp, ci, val, 1.0e-14, inv_diag);
    apply_op(x, q, s);
    if (oss) (void)finish_op_dot(q, q, s);   // q -= B^T g (its dot is not used)
    hipLaunchKernelGGL(k_pcg_residual, dim3(nb), dim3(BLOCK), 0, s, n, b, q, r, part, part + OP_BLOCKS);
    hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(BLOCK), 0, s, nb, part, part + OP_BLOCKS, tol, sc, st, status);
    hipLaunchKernelGGL(k_zero_if_trivial, dim3(blocks), dim3(BLOCK), 0, s, n, x, st);
    apply_prec(r, z, s);
    hipLaunchKernelGGL(k_copy, dim3(blocks), dim3(BLOCK), 0, s, n, z, p, st);
    hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(BLOCK), 0, s, n, r, z, part, st);
    hipLaunchKernelGGL(k_pcg_final_beta, dim3(1), dim3(BLOCK), 0, s, nb, part, sc, st, status, 1);
    int rc = launch_status();
    if (rc) return rc;

    // one iteration (src/cfa/linalg.cuh:231-253)
    auto iteration = [&](hipStream_t q_s) {
        apply_op(p, q, q_s);
        const int npart = finish_op_dot(p, q, q_s);
        hipLaunchKernelGGL(k_pcg_final_alpha, dim3(1), dim3(BLOCK), 0, q_s, npart, part, sc, st, status);
        hipLaunchKernelGGL(k_pcg_update_xr, dim3(nb), dim3(BLOCK), 0, q_s, n, sc, p, q, x, r, part, st);
        hipLaunchKernelGGL(k_pcg_final_rnorm, dim3(1), dim3(BLOCK), 0, q_s, nb, part, sc, st, status);
        apply_prec(r, z, q_s);
        hipLaunchKernelGGL(k_dot_partial, dim3(nb), dim3(BLOCK), 0, q_s, n, r, z, part, st);
        hipLaunchKernelGGL(k_pcg_final_beta, dim3(1), dim3(BLOCK), 0, q_s, nb, part, sc, st, status, 0);
        hipLaunchKernelGGL(k_pcg_p, dim3(blocks), dim3(BLOCK), 0, q_s, n, z, sc, p, st);
    };
    rc = run_iterations(ws, nullptr, max_iter, iteration, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_pcg_outcome, dim3(1), dim3(1), 0, s, sc, st, outcome_words(ws));
    rc = outcome_arrived(ws, s);
    if (rc) return rc;
    pcg_outcome(ws, max_iter, result);
    return launch_status();
}

int cfa_ilu0_factor(const cfa_ilu_t* ilu, const double* val, cfa_stream_t stream) {
    if (!ilu || !val || !ilu->lu || !ilu->colour_start || !ilu->el_ptr || !ilu->el || !ilu->upd) return CFA_E_ARG;
    hipStream_t s = S(stream);
    if (ilu->n == 0) return CFA_OK;
    CFA_TRY(hipMemcpyAsync(ilu->lu, val, (size_t)ilu->nnz * sizeof(double), hipMemcpyDeviceToDevice, s));
    for (int c = 1; c < ilu->n_colours; ++c) {   // colour 0 has no L entries
        const int t0 = ilu->colour_start[c], m = ilu->colour_start[c + 1] - t0;
        if (m == 0) continue;
        hipLaunchKernelGGL(k_ilu_factor_rows, dim3(blocks_for(m, 128)), dim3(128), 0, s, m, t0, ilu->el_ptr, ilu->el,
                           ilu->upd, ilu->lu);
    }
    const int len = std::max(ilu->n, std::max(ilu->nl, ilu->nu));
    hipLaunchKernelGGL(k_ilu_gather, dim3(blocks_for(len)), dim3(BLOCK), 0, s, ilu->nl, ilu->nu, ilu->n, ilu->l_src,
                       ilu->u_src, ilu->d_src, ilu->lu, ilu->lv, ilu->uv, ilu->dinv, ilu->lv32, ilu->uv32, ilu->dinv32);
    if (ilu->s_lrow && ilu->s_urow && ilu->s_lsrc && ilu->s_usrc && ilu->s_lv && ilu->s_uv) {
        const int slots = std::max(std::max(ilu->s_lslots, ilu->s_uslots), 1);
        hipLaunchKernelGGL(k_ilu_sell_values, dim3(blocks_for(slots)), dim3(BLOCK), 0, s, ilu->s_lslots, ilu->s_uslots,
                           ilu->s_lsrc, ilu->s_usrc, ilu->lv, ilu->uv, ilu->lv32 ? ilu->lv32 : nullptr,
                           ilu->uv32 ? ilu->uv32 : nullptr, ilu->s_lv, ilu->s_uv, ilu->lv32 ? ilu->s_lv32 : nullptr,
                           ilu->uv32 ? ilu->s_uv32 : nullptr);
    }
    return launch_status();
}

int cfa_ilu0_apply(const cfa_ilu_t* ilu, const double* r, double* z, int nrhs, cfa_stream_t stream) {
    if (!ilu || !r || !z || nrhs < 1 || nrhs > 2 || !ilu->colour_start || !ilu->pos || !ilu->r_perm ||
        !ilu->z_perm)
        return CFA_E_ARG;
    if (ilu->n == 0) return CFA_OK;
    if (nrhs == 2) ilu_apply_impl<2>(ilu, r, z, S(stream));
    else ilu_apply_impl<1>(ilu, r, z, S(stream));
    return launch_status();
}

int cfa_bicgstab2(int n, const int* rp, const int* ci, const double* val, const double* b_u, const double* b_v,
                  double* x_u, double* x_v, int max_iter, double tol, const cfa_ilu_t* ilu, int use_f32,
                  cfa_krylov_ws_t* ws, cfa_solve_result_t* result, cfa_stream_t stream) {
    if (n < 0 || !rp || !ci || !val || !b_u || !b_v || !x_u || !x_v || !ilu || !ws || !result || ws->cap < n ||
        !ws->status_host || max_iter < 0 || !ilu->colour_start || ilu->n != n || !ilu->pos || !ilu->r_perm ||
        !ilu->z_perm)
        return CFA_E_ARG;
    hipStream_t s = S(stream);
    for (int c = 0; c < 2; ++c) { result->iters[c] = 0; result->converged[c] = 1; result->rel_residual[c] = 0.0; }
    if (n == 0) return CFA_OK;
    double* x = ws->vec[0];
    double* r = ws->vec[2];
    double* r0 = ws->vec[3];
    double* p = ws->vec[4];
    double* v = ws->vec[5];
    double* sv = ws->vec[6];
    double* t = ws->vec[7];
    double* ph = ws->vec[8];
    double* sh = ws->vec[9];
    double* part_a = ws->part;                 // 6 * RED_BLOCKS each
    double* part_b = ws->part + 6 * RED_BLOCKS;
    double* part_c = ws->part + 12 * RED_BLOCKS;
    double* part_d = ws->part + 18 * RED_BLOCKS;
    double* sc = ws->scal;
    int* st = state_words(ws);
    int* status = ws->status_dev;
    ws->status_host[0] = 0;
    ws->status_host[1] = ST_RUNNING;

    const int nb_rows = run_blocks(n), nb1 = red_blocks(n), nb2 = red_blocks(2LL * n);
    auto spmv2_dots = [&](const double* xin, double* yout, const double* w0, int mode, double* partials,
                          hipStream_t q_s) {
        run_dispatch(n, [&](auto rb) {
            constexpr int RB = decltype(rb)::value;
            hipLaunchKernelGGL(k_spmv2_dots<RB>, dim3(nb_rows), dim3(BLOCK), 0, q_s, n, rp, ci, val, xin, yout, w0,
                               mode, partials, st);
        });
    };
    run_dispatch(n, [&](auto rb) {
        constexpr int RB = decltype(rb)::value;
        hipLaunchKernelGGL(k_bicg_init<RB>, dim3(nb_rows), dim3(BLOCK), 0, s, n, rp, ci, val, b_u, b_v, x_u, x_v, x, r, r0,
                           p, v, part_a);
    });
    hipLaunchKernelGGL(k_bicg_final_init, dim3(1), dim3(BLOCK), 0, s, nb_rows, part_a, tol, sc, st, status, max_iter);
    int rc = launch_status();
    if (rc) return rc;

    // one iteration for both components (src/cfa/linalg.cuh:700-775)
    auto iteration = [&](hipStream_t q_s) {
        ilu_values(ilu, use_f32, [&](auto lv, auto uv, auto dinv) {
            using T = typename std::remove_const<typename std::remove_pointer<decltype(lv)>::type>::type;
            const int m0 = ilu->n_colours ? ilu->colour_start[1] - ilu->colour_start[0] : 0,
                      last = ilu->n_colours == 1 ? 1 : 0;
            hipLaunchKernelGGL(k_bicg_p<T>, dim3(blocks_for(n)), dim3(BLOCK), 0, q_s, n, r, v, sc, p, m0, ilu->pos, dinv,
                               last, ilu->r_perm, ilu->z_perm, st);
            ilu_sweeps<2, T>(ilu, lv, uv, dinv, ph, st, q_s);
            spmv2_dots(ph, v, r0, 1, part_a, q_s);
            hipLaunchKernelGGL(k_bicg_s<T>, dim3(nb1), dim3(BLOCK), 0, q_s, n, r, v, sc, sv, part_b, nb_rows, part_a, m0,
                               ilu->pos, dinv, last, ilu->r_perm, ilu->z_perm, st, status);
            ilu_sweeps<2, T>(ilu, lv, uv, dinv, sh, st, q_s);
        });
        spmv2_dots(sh, t, sv, 2, part_c, q_s);
        hipLaunchKernelGGL(k_bicg_xr, dim3(nb2), dim3(BLOCK), 0, q_s, n, ph, sh, sv, t, r0, sc, x, r, part_d, nb1,
                           part_b, nb_rows, part_c, st);
        hipLaunchKernelGGL(k_bicg_final_post, dim3(1), dim3(BLOCK), 0, q_s, nb2, part_d, sc, st, status);
    };
    hipGraphExec_t graph = nullptr;
    if (max_iter > 0) {
        KeyBuilder kb;
        kb.add(n); kb.add(rp); kb.add(ci); kb.add(val); kb.add(use_f32); kb.add(ilu->n_colours);
        kb.add_bytes(ilu->colour_start, sizeof(int) * (size_t)(ilu->n_colours + 1));
        kb.add(ilu->pos); kb.add(ilu->r_perm); kb.add(ilu->z_perm);
        kb.add(ilu->rows); kb.add(ilu->lp); kb.add(ilu->up); kb.add(ilu->lc); kb.add(ilu->uc); kb.add(ilu->lv);
        kb.add(ilu->uv); kb.add(ilu->dinv); kb.add(ilu->lv32); kb.add(ilu->uv32); kb.add(ilu->dinv32);
        kb.add(ilu->s_lrow); kb.add(ilu->s_lsp); kb.add(ilu->s_lc); kb.add(ilu->s_lv); kb.add(ilu->s_lv32);
        kb.add(ilu->s_urow); kb.add(ilu->s_usp); kb.add(ilu->s_uc); kb.add(ilu->s_uv); kb.add(ilu->s_uv32);
        kb.add(ilu->s_llen); kb.add(ilu->s_ulen);
        for (int k = 0; k < 10; ++k) kb.add(ws->vec[k]);
        kb.add(ws->part); kb.add(sc); kb.add(status);
        graph = iteration_graph(ws, internal_of(ws)->bicg, kb.k, iteration);
    }
    rc = run_iterations(ws, graph, max_iter, iteration, s);
    if (rc) return rc;
    // at least 8 lanes in the first workgroup for the outcome's words
    hipLaunchKernelGGL(k_bicg_outcome, dim3(blocks_for(n)), dim3(BLOCK), 0, s, n, x, x_u, x_v, sc, st,
                       outcome_words(ws));
    rc = launch_status();
    if (rc) return rc;
    rc = outcome_arrived(ws, s);
    if (rc) return rc;
    const volatile int* w = ws->status_host;
    for (int c = 0; c < 2; ++c) {
        const bool active = w[2 + c] != 0;   // still so when the loop ended: cap reached without the in-kernel stop
        result->iters[c] = active ? max_iter : w[4 + c];
        result->converged[c] = active ? 0 : w[6 + c];
        result->rel_residual[c] = published_double(w + 8 + 2 * c);
    }
    return launch_status();
}

int cfa_bicgstab_jacobi(int n, const int* rp, const int* ci, const double* val, const double* b, double* x,
                        int max_iter, double tol, cfa_krylov_ws_t* ws, cfa_solve_result_t* result,
                        cfa_stream_t stream) {
    // Host-side scalar logic with one transfer per dot product, as the reference's one-component
    // solver (src/cfa/linalg.cuh:261-347); it is off the default path (--momentum-precond jacobi).
    if (n < 0 || !rp || !ci || !val || !b || !x || !ws || !result || ws->cap < n) return CFA_E_ARG;
    hipStream_t s = S(stream);
    result->iters[0] = 0;
    result->converged[0] = 1;
    result->rel_residual[0] = 0.0;
    if (n == 0) return CFA_OK;
    double* r = ws->vec[0];
    double* r0 = ws->vec[1];
    double* p = ws->vec[2];
    double* v = ws->vec[3];
    double* sv = ws->vec[4];
    double* t = ws->vec[5];
    double* ph = ws->vec[6];
    double* sh = ws->vec[7];
    double* dinv = ws->vec[8];
    const int blocks = blocks_for(n);
    auto dot = [&](const double* a, const double* bb) {
        double out = 0.0;
        cfa_dot(n, a, bb, &out, ws->part, stream);
        return out;
    };
    auto spmv = [&](const double* in, double* out) { cfa_spmv(n, rp, ci, val, in, out, 1, stream); };
    hipLaunchKernelGGL(k_inv_diag, dim3(blocks), dim3(BLOCK), 0, s, n, rp, ci, val, 1.0e-14, dinv);
    spmv(x, v);
    CFA_TRY(hipMemcpyAsync(r, b, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, -1.0, v, r);
    CFA_TRY(hipMemcpyAsync(r0, r, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, s));
    CFA_TRY(hipMemcpyAsync(p, r, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(k_fill_zero, dim3(blocks), dim3(BLOCK), 0, s, n, v);
    const double rn0 = std::sqrt(dot(r, r));
    if (rn0 < 1.0e-13) return launch_status();
    double rho_old = 1.0, alpha = 1.0, omega = 1.0;
    const double bd = 1.0e-30 * rn0 * rn0 + 1.0e-300;
    int iter = 0;
    bool done = false;
    for (; iter < max_iter; ++iter) {
        const double rho_new = dot(r0, r);
        if (std::fabs(rho_new) < bd) break;
        if (iter > 0) {
            const double beta = (rho_new / rho_old) * (alpha / (omega + 1.0e-30));
            hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, -omega, v, p);
            hipLaunchKernelGGL(k_xpay, dim3(blocks), dim3(BLOCK), 0, s, n, r, beta, p);
        }
        hipLaunchKernelGGL(k_vec_mul, dim3(blocks), dim3(BLOCK), 0, s, n, dinv, p, ph, nullptr);
        spmv(ph, v);
        const double r0v = dot(r0, v);
        if (std::fabs(r0v) < bd) break;
        alpha = rho_new / r0v;
        CFA_TRY(hipMemcpyAsync(sv, r, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, -alpha, v, sv);
        const double s_norm = std::sqrt(dot(sv, sv));
        if (s_norm < tol * rn0 || s_norm < 1.0e-11) {
            hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, alpha, ph, x);
            ++iter;
            done = true;
            break;
        }
        hipLaunchKernelGGL(k_vec_mul, dim3(blocks), dim3(BLOCK), 0, s, n, dinv, sv, sh, nullptr);
        spmv(sh, t);
        const double tt = dot(t, t);
        omega = (tt > bd) ? (dot(t, sv) / tt) : 0.0;
        hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, alpha, ph, x);
        hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, omega, sh, x);
        CFA_TRY(hipMemcpyAsync(r, sv, (size_t)n * sizeof(double), hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(BLOCK), 0, s, n, -omega, t, r);
        const double r_norm = std::sqrt(dot(r, r));
        result->rel_residual[0] = r_norm / rn0;
        if (r_norm < tol * rn0 || r_norm < 1.0e-11) {
            ++iter;
            done = true;
            break;
        }
        rho_old = rho_new;
    }
    result->iters[0] = iter;
    result->converged[0] = done ? 1 : 0;
    CFA_TRY(hipStreamSynchronize(s));
    return launch_status();
}

}  // extern "C"
