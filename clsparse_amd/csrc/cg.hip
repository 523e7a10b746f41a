// Conjugate Gradients on gfx950 with a device-resident iteration loop.
//
// Algorithm and stopping rule follow the reference exactly
// (src/library/solvers/conjugate-gradients.hpp L47-229,
//  src/library/solvers/solver-control.hpp L47-64):
//   r = b - A x;  residuum = ||r||_1 / ||b||_1;  stop if finished(residuum);
//   z = M r; p = z; rz = <r, z>
//   loop: y = A p; alpha = rz / <y, p>; x += alpha p; r -= alpha y; z = M r;
//         beta = <r, z>_new / rz; p = z + beta p; residuum = ||r||_1/||b||_1;
//         finished = residuum <= relTol || residuum <= absTol * initial
//                    || nIters >= maxIters   (nIters = index of this iteration)
// The reference drives ~17 launches and 3 blocking host reads per iteration.
// Here the scalars never leave the device. Stencil systems whose vectors fit the
// registers and the LDS of the chip (2.1 M FP64, 4.2 M FP32 rows; with the learned
// factor 2.1 M) run many iterations in one cooperative launch
// (cg_persist_kernel.hpp, fsai_persist.hip). The others run one iteration as four
// kernels (SpMV, <y,p>, fused x/r/z update with <r,z> and ||r|| partials, fused p
// update with the convergence test), fewer with A in diagonal storage; chunks of
// iterations are captured once in a hipGraph and replayed, and the host reads a
// small state block after each chunk. After convergence the remaining kernels of
// a chunk return at once.
//
// Reductions are two-stage and fixed-order (per-workgroup partials; every
// consumer re-adds the same partials in the same order), so a solve is
// bit-reproducible. Dots and norms accumulate in FP64 for both precisions.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "cg_persist.hpp"
#include "fsai_persist.hpp"
#include "cg_state.hpp"
#include "common.hpp"
#include "solver_common.hpp"
#include "dia.hpp"

namespace {

// Iterations of one persistent launch at most: milliseconds, so that the host
// looks at the state now and then (a multiple of kChunk).
constexpr int kMaxRun = 16 * kChunk;
// Rows per thread per step of the grid-stride loops: the loads of kRows rows
// are issued together (the grid is capped at kReducePartialsMax workgroups,
// so one row at a time leaves the kernels waiting on memory latency). Rows
// are still visited, and partial sums formed, in grid-stride order.
constexpr int kRows = 4;

__device__ __forceinline__ double norm_term(int crit, double r)
{
    return crit == kCritL2 ? r * r : fabs(r);
}

// r = b - y (or b when x == 0); z = M r; p = z; partials of ||r|| and <r, z>.
template <typename T>
__global__ __launch_bounds__(256) void cg_init_kernel(size_t n, const T* __restrict__ b,
                                                      const T* __restrict__ y, T* __restrict__ r,
                                                      T* __restrict__ z, T* __restrict__ p,
                                                      const T* __restrict__ invD, int prec,
                                                      int x_zero, int crit,
                                                      double* __restrict__ part_nr,
                                                      double* __restrict__ part_rz)
{
    __shared__ double sh[4];
    double nr = 0.0, rz = 0.0;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        const T ri = x_zero ? b[i] : b[i] - y[i];
        r[i] = ri;
        nr += norm_term(crit, static_cast<double>(ri));
        if (prec == kPrecFsai) continue;  // z, p and <r, z> follow the G G^T apply
        const T zi = (prec == kPrecJacobi) ? ri * invD[i] : ri;
        z[i] = zi;
        p[i] = zi;
        rz += static_cast<double>(ri) * static_cast<double>(zi);
    }
    nr = block_sum256(nr, sh);
    rz = block_sum256(rz, sh);
    if (threadIdx.x == 0) {
        part_nr[blockIdx.x] = nr;
        part_rz[blockIdx.x] = rz;
    }
}

__global__ __launch_bounds__(256) void cg_init_finalize(CgDevState* __restrict__ st,
                                                        const double* __restrict__ part_nr,
                                                        uint32_t g, double* __restrict__ init_out)
{
    __shared__ double sh[4];
    const double s = sum_partials(part_nr, g, sh);
    if (threadIdx.x == 0) {
        const double norm = st->crit == kCritL2 ? sqrt(s) : s;
        st->init_res = norm / st->norm_ref;
        st->cur_res = st->init_res;
        st->first = 1;  // p = z
        st->pending = 0;
        if (init_out != nullptr) *init_out = st->init_res;
    }
}

// part_yp[block] = sum y_i p_i
template <typename T>
__global__ __launch_bounds__(256) void cg_dot_kernel(size_t n, const T* __restrict__ y,
                                                     const T* __restrict__ p,
                                                     double* __restrict__ part_yp,
                                                     const CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    if (st->done) return;
    double a = 0.0;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i0 = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i0 < n; i0 += kRows * stride) {
        T yv[kRows], pv[kRows];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i < n) {
                yv[u] = y[i];
                pv[u] = p[i];
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u)
            if (i0 + u * stride < n) a += static_cast<double>(yv[u]) * static_cast<double>(pv[u]);
    }
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) part_yp[blockIdx.x] = a;
}

// alpha = rz / yp; x += alpha p; r -= alpha y; z = M r; partials <r,z>, ||r||.
// x may be held in a wider type than the other vectors (FP64 solution update).
// PN: p is first brought up to date, p = z + beta_f p as the SpMV kernel of
// this iteration formed it on the fly (cg_spmv_pn_kernel), and stored.
template <typename T, typename TX, bool PN = false>
__global__ __launch_bounds__(256) void cg_update_kernel(
    size_t n, TX* __restrict__ x, T* __restrict__ r, T* __restrict__ z, T* __restrict__ p,
    const T* __restrict__ y, const T* __restrict__ invD, int prec,
    const double* __restrict__ part_yp, const double* __restrict__ part_rz_prev,
    double* __restrict__ part_rz, double* __restrict__ part_nr, uint32_t g,
    CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    const int done = st->done;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->stop = done;
    if (done) return;
    const double yp = sum_partials(part_yp, g, sh);
    const double rz = sum_partials(part_rz_prev, g, sh);
    const T alpha = static_cast<T>(rz / yp);
    const TX alpha_x = static_cast<TX>(rz / yp);
    const int crit = st->crit;
    const T beta = PN ? static_cast<T>(st->beta_f) : T(0);
    double nr = 0.0, rzn = 0.0;
    // FP32: an eighth of the rows per XCD, as the learned factor's kernels walk
    // them (5.4 M rows, 71.0 -> 69.7 us an iteration); FP64: sweeps over all rows
    // (3.4 M rows, 94.9 us an iteration; by eighths 98.4).
    constexpr bool kWalk = sizeof(T) == 4;
    const uint32_t blk = kWalk ? xcd_remap(blockIdx.x, gridDim.x) : blockIdx.x;
    const RowWalk rw = kWalk ? row_walk(n, blk, gridDim.x, threadIdx.x) : row_sweep(n, blk, gridDim.x, threadIdx.x);
    const size_t stride = rw.stride;
    for (size_t i0 = rw.first; i0 < rw.end; i0 += kRows * stride) {
        T pv[kRows], rv[kRows], yv[kRows], dv[kRows], zv[kRows];
        TX xv[kRows];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i < rw.end) {
                pv[u] = p[i];
                if (PN) zv[u] = z[i];
                xv[u] = x[i];
                rv[u] = r[i];
                yv[u] = y[i];
                if (prec == kPrecJacobi) dv[u] = invD[i];
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= rw.end) continue;
            if (PN) {
                pv[u] = fma(beta, pv[u], zv[u]);  // p (beta 0 and z == p while `first`)
                p[i] = pv[u];
            }
            x[i] = xv[u] + alpha_x * static_cast<TX>(pv[u]);
            const T ri = rv[u] - alpha * yv[u];
            r[i] = ri;
            nr += norm_term(crit, static_cast<double>(ri));
            if (prec == kPrecFsai) continue;  // z and <r, z> follow the G G^T apply
            const T zi = (prec == kPrecJacobi) ? ri * dv[u] : ri;
            z[i] = zi;
            rzn += static_cast<double>(ri) * static_cast<double>(zi);
        }
    }
    nr = block_sum256(nr, sh);
    rzn = block_sum256(rzn, sh);
    if (threadIdx.x == 0) {
        part_nr[blk] = nr;
        part_rz[blk] = rzn;
    }
    if (PN && blockIdx.x == 0 && threadIdx.x == 0) {
        st->pending = 1;  // the convergence test of this iteration follows
        st->first = 0;    // p now lags z by one update
    }
}

// End of an iteration: workgroup 0 of the p update evaluates finished()
// from the ||r|| partials.
__device__ void cg_finish(CgDevState* __restrict__ st, const double* __restrict__ part_nr, uint32_t g,
                          double* sh)
{
    if (blockIdx.x != 0) return;
    const double s = sum_partials(part_nr, g, sh);
    if (threadIdx.x == 0) {
        const double norm = st->crit == kCritL2 ? sqrt(s) : s;
        const double res = norm / st->norm_ref;
        const int it = st->iter;
        st->cur_res = res;
        st->hist[it % kHist] = res;
        const bool conv = (res <= st->rel_tol) || (res <= st->abs_tol * st->init_res);
        if (conv || it >= st->max_iters) {
            st->done = 1;
            st->n_iters = it;
            st->converged = conv ? 1 : 0;
        }
        st->iter = it + 1;
    }
}

// beta = rz_new / rz_old; p = z + beta p; workgroup 0 evaluates finished().
template <typename T>
__global__ __launch_bounds__(256) void cg_pupdate_kernel(size_t n, T* __restrict__ p,
                                                         const T* __restrict__ z,
                                                         const double* __restrict__ part_rz,
                                                         const double* __restrict__ part_rz_prev,
                                                         const double* __restrict__ part_nr,
                                                         uint32_t g, CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    if (st->stop) return;
    const double rz_new = sum_partials(part_rz, g, sh);
    const double rz_old = sum_partials(part_rz_prev, g, sh);
    const T beta = static_cast<T>(rz_new / rz_old);
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i0 = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i0 < n; i0 += kRows * stride) {
        T zv[kRows], pv[kRows];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i < n) {
                zv[u] = z[i];
                pv[u] = p[i];
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i < n) p[i] = zv[u] + beta * pv[u];
        }
    }

    cg_finish(st, part_nr, g, sh);
}

// The convergence test of the last iteration of a chunk (the fused SpMV
// kernel of the next iteration would run it otherwise): one workgroup.
__global__ __launch_bounds__(256) void cg_test_kernel(CgDevState* __restrict__ st,
                                                      const double* __restrict__ part_nr, uint32_t g)
{
    __shared__ double sh[4];
    if (st->done || !st->pending) return;
    cg_finish(st, part_nr, g, sh);
    if (threadIdx.x == 0) st->pending = 0;
}

// p = z + beta p with beta = rz_new / rz_old unless p is already current
// (`first`): the p update a fused iteration leaves to the next SpMV, made
// explicit before a residual replacement re-bases p.
template <typename T>
__global__ __launch_bounds__(256) void cg_materialize_p(size_t n, T* __restrict__ p, const T* __restrict__ z,
                                                        const double* __restrict__ part_rz_new,
                                                        const double* __restrict__ part_rz_old, uint32_t g,
                                                        const CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    if (st->first) return;
    const double rz_new = sum_partials(part_rz_new, g, sh);
    const double rz_old = sum_partials(part_rz_old, g, sh);
    const T beta = static_cast<T>(rz_new / rz_old);
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
        p[i] = fma(beta, p[i], z[i]);
}

// R rows iu[0..R) of y = A p' (p' = fma(b, p, z) formed at each operand)
// from diagonal storage, their <y, p'> terms added to a; rows with live[u]
// false are computed from in-range loads and dropped, as in dia_rows.
template <int K, bool SYM, typename T, int R>
__device__ __forceinline__ void pn_rows(uint32_t n, const DiaOffsets& off, __amdgpu_buffer_rsrc_t rv,
                                        __amdgpu_buffer_rsrc_t rp, __amdgpu_buffer_rsrc_t rz, T b,
                                        T* __restrict__ y, const uint32_t (&iu)[R], const bool (&live)[R], double& a)
{
    constexpr int KL = SYM ? (K + 1) / 2 : K;
    constexpr uint32_t S = sizeof(T);
    T v[R][K], xv[R][K], pi[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const uint32_t i = iu[u];
#pragma unroll
        for (int d = 0; d < K; ++d) {
            const uint32_t j = i + static_cast<uint32_t>(off.o[d]);  // wraps below 0: out of range
            xv[u][d] = fma(b, buf_load<T>(rp, j * S, 0), buf_load<T>(rz, j * S, 0));
            if (d < KL) {
                const uint32_t il = i < n ? i : n - 1;
                v[u][d] = buf_load<T>(rv, il * S, static_cast<uint32_t>(d) * n * S);
            } else {
                const uint32_t at = j < n ? (static_cast<uint32_t>(K - 1 - d) * n + j) * S : 0xFFFFFFFFu;
                v[u][d] = buf_load<T>(rv, at, 0);
            }
        }
        pi[u] = fma(b, buf_load<T>(rp, i * S, 0), buf_load<T>(rz, i * S, 0));
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
        double sum = 0.0;  // FP32 products summed in FP64, as the CSR SpMV sums them
#pragma unroll
        for (int d = 0; d < K; ++d)
            if (v[u][d] != T(0)) sum += static_cast<double>(mul_rounded_t(v[u][d], xv[u][d]));
        const T acc = static_cast<T>(sum);
        if (live[u]) y[iu[u]] = acc;
        a += live[u] ? static_cast<double>(acc) * static_cast<double>(pi[u]) : 0.0;
    }
}

// y = A p' with p' = fma(beta, p, z), formed at every row the stencil reads,
// from diagonal storage as dia_spmv_dot_buf_kernel does (while `first`,
// beta = 0 and z holds p, so p' = p), in the same row order (line > 0: lanes
// walk rows c, c + line, ...);
// <y, p'> partials; workgroup 0 first runs the convergence test of the
// previous iteration and publishes beta and the choice for the x / r update.
// beta = rz_new / rz_old is what cg_pupdate_kernel would have used, and
// p' = fma(beta, p, z) here and in the update, so both see the same p'.
template <int K, bool SYM, typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4))) void cg_spmv_pn_kernel(
    uint32_t n, DiaOffsets off, const T* __restrict__ vals, const T* __restrict__ p, const T* __restrict__ z,
    T* __restrict__ y, double* __restrict__ part_yp, const double* __restrict__ part_rz_new,
    const double* __restrict__ part_rz_old, const double* __restrict__ part_nr, uint32_t g,
    CgDevState* __restrict__ st, uint32_t line)
{
    constexpr uint32_t S = sizeof(T);
    constexpr int R = 2;  // rows per step (launched for FP32; 4 ran slower)
    __shared__ double sh[4];
    if (st->done) return;
    const int first = st->first;
    const int pending = st->pending;
    double beta = 0.0;
    if (!first) beta = sum_partials(part_rz_new, g, sh) / sum_partials(part_rz_old, g, sh);
    const T b = static_cast<T>(beta);
    if (blockIdx.x == 0) {
        if (pending) cg_finish(st, part_nr, g, sh);
        if (threadIdx.x == 0) {
            st->pending = 0;
            st->beta_f = beta;
        }
    }
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(vals), 0, K * n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(z), 0, n * S, 0x00020000);
    const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
    double a = 0.0;
    if (line == 0) {
        const uint32_t stride = gridDim.x * 256;
        for (uint32_t i0 = blk * 256 + threadIdx.x; i0 < n; i0 += R * stride) {
            uint32_t iu[R];
            bool live[R];
#pragma unroll
            for (int u = 0; u < R; ++u) {
                iu[u] = i0 + u * stride;
                live[u] = iu[u] < n;
            }
            pn_rows<K, SYM, T, R>(n, off, rv, rp, rz, b, y, iu, live, a);
        }
    } else {
        const uint32_t threads = gridDim.x * 256;
        const LinePart lp = line_part(n, line, threads);
        for (uint32_t q = blk * 256 + threadIdx.x; q < lp.items; q += threads) {
            uint32_t c, k_beg, k_end;
            line_item(lp, q, c, k_beg, k_end);
            for (uint32_t k0 = k_beg; k0 < k_end; k0 += R) {
                uint32_t iu[R];
                bool live[R];
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    iu[u] = c + (k0 + u) * line;
                    live[u] = k0 + u < k_end && iu[u] < n;
                    if (!live[u]) iu[u] = c;  // a row in range, computed and dropped
                }
                pn_rows<K, SYM, T, R>(n, off, rv, rp, rz, b, y, iu, live, a);
            }
        }
    }
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) part_yp[blk] = a;
}

// ---- learned-FSAI factor in diagonal storage (BF16 values, FP32 compute) ----
// Row i of G holds G(i, i + off[d]) = vals[d n + i]; entries outside the
// pattern are zero and skipped, so they never read the input vector. Each
// product is rounded on its own and the row is summed in ascending column
// order: the same sums as the CSR SpMV of the factor.

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(static_cast<uint32_t>(h) << 16); }

__device__ __forceinline__ float mul_rounded_f(float a, float b)
{
#pragma clang fp contract(off)
    return a * b;
}

// y = G^T r and partials of ||y||^2 (one per workgroup, g workgroups).
// Row i of G^T holds G(i - off[d], i) at column i - off[d]: ascending column
// order walks the diagonals from off = 0 down.
template <int K>
__global__ __launch_bounds__(256) void fsai_gt_dia_kernel(size_t n, DiaOffsets off,
                                                          const uint16_t* __restrict__ vals,
                                                          const float* __restrict__ r,
                                                          float* __restrict__ y,
                                                          double* __restrict__ part,
                                                          const int* __restrict__ done)
{
    __shared__ double sh[4];
    if (done != nullptr && *done != 0) return;
    const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);  // contiguous rows per XCD
    double a = 0.0;
    const RowWalk rw = row_walk(n, blk, gridDim.x, threadIdx.x);
    const size_t stride = rw.stride;
    for (size_t i0 = rw.first; i0 < rw.end; i0 += kRows * stride) {
        uint16_t h[kRows][K];
        float rv[kRows][K];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
#pragma unroll
            for (int d = 0; d < K; ++d) {
                const size_t j = i - static_cast<int64_t>(off.o[d]);
                const bool in = i < rw.end && j < n;
                h[u][d] = in ? vals[static_cast<size_t>(d) * n + j] : uint16_t(0);
                rv[u][d] = in ? r[j] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= rw.end) continue;
            double sum = 0.0;  // products summed in FP64, as the CSR SpMV sums them
#pragma unroll
            for (int d = K - 1; d >= 0; --d)
                if (h[u][d] != 0) sum += static_cast<double>(mul_rounded_f(bf16_to_f32(h[u][d]), rv[u][d]));
            const float acc = static_cast<float>(sum);
            y[i] = acc;
            a += static_cast<double>(acc) * static_cast<double>(acc);
        }
    }
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) part[blk] = a;
}

// z = G y.
template <int K>
__global__ __launch_bounds__(256) void fsai_g_dia_kernel(size_t n, DiaOffsets off,
                                                         const uint16_t* __restrict__ vals,
                                                         const float* __restrict__ y,
                                                         float* __restrict__ z,
                                                         const int* __restrict__ done)
{
    if (done != nullptr && *done != 0) return;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i0 = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i0 < n; i0 += kRows * stride) {
        uint16_t h[kRows][K];
        float yv[kRows][K];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
#pragma unroll
            for (int d = 0; d < K; ++d) {
                const int64_t j = static_cast<int64_t>(i) + off.o[d];
                const bool in = i < n && j >= 0;
                h[u][d] = in ? vals[static_cast<size_t>(d) * n + i] : uint16_t(0);
                yv[u][d] = in ? y[j] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= n) continue;
            double sum = 0.0;  // products summed in FP64, as the CSR SpMV sums them
#pragma unroll
            for (int d = 0; d < K; ++d)
                if (h[u][d] != 0) sum += static_cast<double>(mul_rounded_f(bf16_to_f32(h[u][d]), yv[u][d]));
            z[i] = static_cast<float>(sum);
        }
    }
}

constexpr int kPupdateRows = 2;  // rows per lane in flight in the factor's p update (4: 0.8 % slower)

// p = G y + beta p with beta = ||y||^2_new / <r, z>_old (the p update of
// cg_pupdate_kernel with z = G y formed in registers, never stored), then
// the convergence test.
template <int K, int R = kPupdateRows>
__global__ __launch_bounds__(256) void fsai_g_pupdate_dia_kernel(
    size_t n, DiaOffsets off, const uint16_t* __restrict__ vals, const float* __restrict__ y,
    float* __restrict__ p, const double* __restrict__ part_rz, const double* __restrict__ part_rz_prev,
    const double* __restrict__ part_nr, uint32_t g, CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    if (st->stop) return;
    const double rz_new = sum_partials(part_rz, g, sh);
    const double rz_old = sum_partials(part_rz_prev, g, sh);
    const float beta = static_cast<float>(rz_new / rz_old);
    const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);  // contiguous rows per XCD
    const RowWalk rw = row_walk(n, blk, gridDim.x, threadIdx.x);
    const size_t stride = rw.stride;
    for (size_t i0 = rw.first; i0 < rw.end; i0 += R * stride) {
        uint16_t h[R][K];
        float yv[R][K], pv[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const size_t i = i0 + u * stride;
#pragma unroll
            for (int d = 0; d < K; ++d) {
                const int64_t j = static_cast<int64_t>(i) + off.o[d];
                const bool in = i < rw.end && j >= 0;
                h[u][d] = in ? vals[static_cast<size_t>(d) * n + i] : uint16_t(0);
                yv[u][d] = in ? y[j] : 0.f;
            }
            pv[u] = i < rw.end ? p[i] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= rw.end) continue;
            double sum = 0.0;  // products summed in FP64, as the CSR SpMV sums them
#pragma unroll
            for (int d = 0; d < K; ++d)
                if (h[u][d] != 0) sum += static_cast<double>(mul_rounded_f(bf16_to_f32(h[u][d]), yv[u][d]));
            p[i] = static_cast<float>(sum) + beta * pv[u];
        }
    }
    cg_finish(st, part_nr, g, sh);
}

// One iteration's preconditioner and p update: y = G^T r with <r, z>
// partials, then p = G y + beta p and the convergence test.
template <int K>
void launch_dia_iteration(size_t n, uint32_t g, const DiaOffsets& off, const uint16_t* vals, const float* r,
                          float* y, float* p, double* part_rz, const double* part_rz_prev,
                          const double* part_nr, CgDevState* st, hipStream_t s)
{
    hipLaunchKernelGGL((fsai_gt_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, vals, r, y, part_rz,
                       &st->done);
    hipLaunchKernelGGL((fsai_g_pupdate_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, vals, y, p,
                       part_rz, part_rz_prev, part_nr, g, st);
}

constexpr int kFuseRows = 2;  // rows per lane in flight in the fused update (registers)

// The x / r update of cg_update_kernel (learned FSAI: no z) fused with
// w = G^T r_new, the ||r_new|| partials of the convergence test and the
// ||w||^2 partials (<r, z>). G^T's row i reads r_new at rows i - off[d]; this
// workgroup forms r_new there from r and y exactly as the row's owner forms
// it, so r_new goes to the other buffer (r_out) and r stays whole for the
// other workgroups; w goes to a buffer of its own for the same reason (y is
// read at other rows). Partials are indexed by the XCD-remapped workgroup,
// whose rows are those of cg_update_kernel's workgroup of that index, so
// the sums are those of the separate kernels.
template <int K, typename TX, int R = kFuseRows>
__global__ __launch_bounds__(256) void fsai_update_gt_dia_kernel(
    size_t n, DiaOffsets off, const uint16_t* __restrict__ vals, TX* __restrict__ x,
    const float* __restrict__ r, float* __restrict__ r_out, const float* __restrict__ p,
    const float* __restrict__ y, float* __restrict__ w, const double* __restrict__ part_yp,
    const double* __restrict__ part_rz_prev, double* __restrict__ part_rz, double* __restrict__ part_nr,
    uint32_t g, CgDevState* __restrict__ st)
{
    __shared__ double sh[4];
    const int done = st->done;
    if (blockIdx.x == 0 && threadIdx.x == 0) st->stop = done;
    if (done) return;
    const double yp = sum_partials(part_yp, g, sh);
    const double rz = sum_partials(part_rz_prev, g, sh);
    const float alpha = static_cast<float>(rz / yp);
    const TX alpha_x = static_cast<TX>(rz / yp);
    const int crit = st->crit;
    const uint32_t blk = xcd_remap(blockIdx.x, gridDim.x);
    double nr = 0.0, a = 0.0;
    const RowWalk rw = row_walk(n, blk, gridDim.x, threadIdx.x);
    const size_t stride = rw.stride;
    for (size_t i0 = rw.first; i0 < rw.end; i0 += R * stride) {
        uint16_t h[R][K];
        float rv[R][K], yv[R][K], pv[R];
        TX xv[R];
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const size_t i = i0 + u * stride;
#pragma unroll
            for (int d = 0; d < K; ++d) {
                const size_t j = i - static_cast<int64_t>(off.o[d]);
                const bool in = i < rw.end && j < n;
                h[u][d] = in ? vals[static_cast<size_t>(d) * n + j] : uint16_t(0);
                rv[u][d] = in ? r[j] : 0.f;
                yv[u][d] = in ? y[j] : 0.f;
            }
            pv[u] = i < rw.end ? p[i] : 0.f;
            xv[u] = i < rw.end ? x[i] : TX(0);
        }
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= rw.end) continue;
            x[i] = xv[u] + alpha_x * static_cast<TX>(pv[u]);
            double sum = 0.0;  // products summed in FP64, as the CSR SpMV sums them
#pragma unroll
            for (int d = K - 1; d >= 0; --d) {
                const float rn = rv[u][d] - alpha * yv[u][d];  // as cg_update_kernel forms r
                if (d == K - 1) {  // off[K - 1] = 0: row i itself
                    r_out[i] = rn;
                    nr += norm_term(crit, static_cast<double>(rn));
                }
                if (h[u][d] != 0) sum += static_cast<double>(mul_rounded_f(bf16_to_f32(h[u][d]), rn));
            }
            const float acc = static_cast<float>(sum);
            w[i] = acc;
            a += static_cast<double>(acc) * static_cast<double>(acc);
        }
    }
    nr = block_sum256(nr, sh);
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) {
        part_nr[blk] = nr;
        part_rz[blk] = a;
    }
}

// One learned-FSAI iteration after y = A p: the fused x / r update and
// w = G^T r_new (r from r_in to r_out), then p = G w + beta p and the
// convergence test.
template <int K, typename TX>
void launch_dia_update_iteration(size_t n, uint32_t g, const DiaOffsets& off, const uint16_t* vals, TX* x,
                                 const float* r_in, float* r_out, const float* p_in, const float* y, float* w,
                                 float* p, const double* part_yp, double* part_rz, const double* part_rz_prev,
                                 double* part_nr, CgDevState* st, hipStream_t s)
{
    hipLaunchKernelGGL((fsai_update_gt_dia_kernel<K, TX>), dim3(g), dim3(256), 0, s, n, off, vals, x, r_in, r_out,
                       p_in, y, w, part_yp, part_rz_prev, part_rz, part_nr, g, st);
    hipLaunchKernelGGL((fsai_g_pupdate_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, vals, w, p, part_rz,
                       part_rz_prev, part_nr, g, st);
}

template <int K>
void launch_dia_apply(size_t n, uint32_t g, const DiaOffsets& off, const uint16_t* vals, const float* r,
                      float* tmp, float* out, double* part, const int* done, hipStream_t s)
{
    hipLaunchKernelGGL((fsai_gt_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, vals, r, tmp, part,
                       done);
    hipLaunchKernelGGL((fsai_g_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, vals, tmp, out, done);
}

template <typename T>
struct CgBuffers
{
    T* r;
    T* z;
    T* p;
    T* y;
    T* invD;
    T* one;
    T* zero;
    double* part_yp;
    double* part_rz[2];
    double* part_nr[2];
    CgDevState* st;
    unsigned long long* slots;  // grid-wide sums of the persistent iteration

    static size_t bytes(size_t n)
    {
        return 5 * align_up(n * sizeof(T)) + 2 * align_up(sizeof(T)) +
               5 * align_up(kReducePartialsMax * sizeof(double)) + align_up(sizeof(CgDevState)) +
               align_up(persist_slot_words() * sizeof(unsigned long long));
    }
    void carve(Carve& c, size_t n)
    {
        r = c.take<T>(n);
        z = c.take<T>(n);
        p = c.take<T>(n);
        y = c.take<T>(n);
        invD = c.take<T>(n);
        one = c.take<T>(1);
        zero = c.take<T>(1);
        part_yp = c.take<double>(kReducePartialsMax);
        part_rz[0] = c.take<double>(kReducePartialsMax);
        part_rz[1] = c.take<double>(kReducePartialsMax);
        part_nr[0] = c.take<double>(kReducePartialsMax);
        part_nr[1] = c.take<double>(kReducePartialsMax);
        st = c.take<CgDevState>(1);
        slots = c.take<unsigned long long>(persist_slot_words());
    }
};

// CLSPARSE_AMD_CG_FUSE=0: the Jacobi / unpreconditioned iteration keeps its
// separate p update kernel.
bool cg_fuse_enabled()
{
    const char* e = std::getenv("CLSPARSE_AMD_CG_FUSE");
    return !(e && e[0] == '0');
}

// cg_spmv_pn_kernel for the stencil's diagonal count and storage.
template <typename T>
clsparseStatus launch_spmv_pn(const DiaMatrix<T>& A, size_t n, uint32_t g, const T* p, const T* z, T* y,
                              double* part_yp, const double* rz_new, const double* rz_old, const double* nr,
                              CgDevState* st, hipStream_t s)
{
    const uint32_t line = dia_line(A.off, A.ndiag, n);
#define CLS_PN(K, S)                                                                                     \
    hipLaunchKernelGGL((cg_spmv_pn_kernel<K, S, T>), dim3(g), dim3(256), 0, s, static_cast<uint32_t>(n), \
                       A.off, A.vals, p, z, y, part_yp, rz_new, rz_old, nr, g, st, line)
    if (A.sym) {
        switch (A.ndiag) {
        case 3: CLS_PN(3, true); break;
        case 5: CLS_PN(5, true); break;
        case 7: CLS_PN(7, true); break;
        case 9: CLS_PN(9, true); break;
        default: return clsparseInvalidValue;
        }
    } else {
        switch (A.ndiag) {
        case 1: CLS_PN(1, false); break;
        case 2: CLS_PN(2, false); break;
        case 3: CLS_PN(3, false); break;
        case 4: CLS_PN(4, false); break;
        case 5: CLS_PN(5, false); break;
        case 6: CLS_PN(6, false); break;
        case 7: CLS_PN(7, false); break;
        case 8: CLS_PN(8, false); break;
        case 9: CLS_PN(9, false); break;
        default: return clsparseInvalidValue;
        }
    }
#undef CLS_PN
    CLS_HIP_TRY(hipGetLastError());
    return clsparseSuccess;
}

// Residual of the starting point: r = b - A x (b itself when x == 0), and for
// the elementwise preconditioners z = M r, p = z, <r, z>; writes init_res into
// the device state and to init_out if given.
template <typename T>
clsparseStatus cg_setup(const clsparseCsrMatrix* A, const T* x, const T* b, size_t n, int prec, int crit,
                        CgBuffers<T>& buf, hipStream_t s, bool ext, bool x_zero, double* init_out)
{
    const uint32_t g = grid_for(n);
    if (!x_zero) CLS_TRY(launch_csrmv<T>(buf.one, A, x, buf.zero, buf.y, s, ext, nullptr));
    hipLaunchKernelGGL((cg_init_kernel<T>), dim3(g), dim3(256), 0, s, n, b, buf.y, buf.r, buf.z, buf.p, buf.invD, prec,
                       x_zero ? 1 : 0, crit, buf.part_nr[1], buf.part_rz[1]);
    hipLaunchKernelGGL(cg_init_finalize, dim3(1), dim3(256), 0, s, buf.st, buf.part_nr[1], g, init_out);
    CLS_HIP_TRY(hipGetLastError());
    return clsparseSuccess;
}

__global__ void state_recover(CgDevState* st, double init_res, int iter)
{
    if (threadIdx.x == 0) cg_recover(*st, init_res, iter);
}

// The device-resident PCG loop on one system. x, b are T vectors of length n.
template <typename T, typename TX = T>
class CgEngine
{
public:
    // G, GT: the factor of M = G G^T and its transpose (kPrecFsai only);
    // g_bf16: their values are BF16 bit patterns (FP32 engines only);
    // dia: the BF16 factor in diagonal storage, used instead of G and GT.
    // r_alt: n values the engine may keep r in between iterations (the
    // learned factor in diagonal storage fuses the x / r update into G^T r
    // with it); their contents are not kept.
    CgEngine(const clsparseCsrMatrix* A, TX* x, const T* b, size_t n, int prec, int crit,
             CgBuffers<T>& buf, hipStream_t s, bool ext, const clsparseCsrMatrix* G = nullptr,
             const clsparseCsrMatrix* GT = nullptr, bool g_bf16 = false,
             const FsaiDia* dia = nullptr, const DiaMatrix<T>* adia = nullptr, T* r_alt = nullptr,
             int num_cus = 0, int device = 0, clsparseAmdSolverLaunches* launches = nullptr)
        : A_(A), x_(x), b_(b), n_(n), prec_(prec), crit_(crit), buf_(buf), s_(s), ext_(ext),
          g_(grid_for(n)), G_(G), GT_(GT), g_bf16_(g_bf16), r_alt_(r_alt), device_(device), launches_(launches)
    {
        if (adia != nullptr && adia->vals != nullptr) adia_ = *adia;
        if (std::is_same_v<T, TX> && prec_ != kPrecFsai && adia_.vals != nullptr)
            plan_ = cg_persist_plan(n, adia_.ndiag, adia_.off.o, sizeof(T), num_cus);
        if (dia != nullptr && std::is_same_v<T, float> && g_bf16) {
            use_dia_ = true;
            dia_ = *dia;
            for (int d = 0; d < kFsaiMaxDiags; ++d) dia_off_.o[d] = dia->off[d];
        }
        if (std::is_same_v<T, TX> && prec_ == kPrecFsai && use_dia_ && adia_.vals != nullptr)
            plan_ = fsai_persist_plan(n, adia_.ndiag, adia_.off.o, dia_.ndiag, dia_off_.o, num_cus);
        persist_ = plan_.rows != 0;
        // FP32 only: in FP64 the fused SpMV (p and z at every stencil offset)
        // ran slower than the separate p update (128^3 Jacobi-PCG 39.4-40.5
        // against 37.2-37.3 ms), in FP32 faster (mixed 22.3-22.6 against
        // 23.2 ms, clsparseScsrcg 13.6-13.7 against 14.1 ms, the same iterates).
        // Its buffer resources take K n sizeof(T) bytes in 32 bits; larger
        // systems keep the separate kernels (whose SpMV then takes flat loads).
        can_fuse_ = std::is_same_v<T, float> && prec_ != kPrecFsai && adia_.vals != nullptr && cg_fuse_enabled() &&
                    dia_buf_fits(adia_.ndiag, n, sizeof(T));
        // CLSPARSE_AMD_CG_FUSE=0 keeps the separate x / r update (the same iterates).
        can_fuse_gt_ = prec_ == kPrecFsai && use_dia_ && r_alt_ != nullptr && cg_fuse_enabled();
        start_kernels();
    }
    ~CgEngine()
    {
        if (exec_) (void)hipGraphExecDestroy(exec_);
        if (graph_) (void)hipGraphDestroy(graph_);
    }

    // cg_setup and, for the learned factor, z = M r, p = z, <r, z>.
    clsparseStatus setup(bool x_zero)
    {
        if constexpr (std::is_same_v<T, TX>) {
            CLS_TRY(cg_setup<T>(A_, x_, b_, n_, prec_, crit_, buf_, s_, ext_, x_zero, nullptr));
        } else {
            if (!x_zero) return clsparseInvalidValue;  // the wide-x engine starts from a given residual
            CLS_TRY(cg_setup<T>(A_, nullptr, b_, n_, prec_, crit_, buf_, s_, ext_, true, nullptr));
        }
        start_kernels();
        if (prec_ == kPrecFsai) {
            CLS_TRY(apply_fsai(buf_.part_rz[1], nullptr));
            hipLaunchKernelGGL((cast_kernel<T, T>), dim3(ew_grid(n_)), dim3(256), 0, s_, n_, buf_.z,
                               buf_.p);
            CLS_HIP_TRY(hipGetLastError());
        }
        return clsparseSuccess;
    }

    // One chunk of kChunk iterations (captured once in a graph, then
    // replayed); afterwards the host copy of the device state is current.
    // Iterations after the device state says done return at once. The
    // persistent iteration runs several chunks in one launch, at most max_run
    // iterations, while the residual after each is above go_on; where a launch
    // gave up (host_state->failed) the caller starts again from x, in separate
    // launches from then on. A device that refuses the launch has run nothing of
    // it: the chunk runs in separate launches.
    // With the learned factor it also returns after a chunk that does not
    // halve the best residual, best to start with, of the chunks before
    // (host_state->best_res then).
    clsparseStatus run_chunk(CgDevState* host_state, int max_run = kChunk, double go_on = -1.0, double best = 0.0)
    {
        if (persistent()) {
            bool refused = false;
            if (prec_ == kPrecFsai) CLS_TRY(run_persistent_fsai(host_state, max_run, go_on, best, &refused));
            else CLS_TRY(run_persistent(host_state, max_run, go_on, &refused));
            if (!refused) return clsparseSuccess;
        }
        const bool use_graph = graphs_enabled();
        if (use_graph && exec_ == nullptr) {
            CLS_HIP_TRY(hipStreamBeginCapture(s_, hipStreamCaptureModeThreadLocal));
            clsparseStatus st = clsparseSuccess;
            for (int k = 0; k < kChunk && st == clsparseSuccess; ++k) st = enqueue_iteration(k & 1);
            if (st == clsparseSuccess) st = enqueue_chunk_end();
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(s_, &g);
            if (st != clsparseSuccess) {
                if (g) (void)hipGraphDestroy(g);
                return st;
            }
            CLS_HIP_TRY(e);
            graph_ = g;
            CLS_HIP_TRY(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0));
        }
        if (use_graph) {
            CLS_HIP_TRY(hipGraphLaunch(exec_, s_));
        } else {
            for (int k = 0; k < kChunk; ++k) CLS_TRY(enqueue_iteration(k & 1));
            CLS_TRY(enqueue_chunk_end());
        }
        CLS_HIP_TRY(hipMemcpyAsync(host_state, buf_.st, sizeof(CgDevState), hipMemcpyDeviceToHost,
                                   s_));
        CLS_HIP_TRY(hipStreamSynchronize(s_));
        return clsparseSuccess;
    }

    // Runs chunks until the device state says done. `on_chunk` sees the host
    // copy of the state after every chunk. init_res: of the set-up.
    template <typename F>
    clsparseStatus run(CgDevState* host_state, double init_res, int max_run, F&& on_chunk)
    {
        for (int iter = 0;;) {
            CLS_TRY(run_chunk(host_state, max_run));
            if (host_state->failed) {
                CLS_TRY(cg_setup<T>(A_, x_, b_, n_, prec_, crit_, buf_, s_, ext_, false, nullptr));
                hipLaunchKernelGGL(state_recover, dim3(1), dim3(64), 0, s_, buf_.st, init_res, iter);
                CLS_HIP_TRY(hipGetLastError());
                start_kernels();
                continue;
            }
            iter = host_state->iter;
            on_chunk(*host_state);
            if (host_state->done) break;
        }
        return clsparseSuccess;
    }

    // z_new = G (G^T r) into `out` through `tmp`, for the residual replacement
    // of the reliable solver (learned factor only: rr_precondition forms the
    // elementwise ones).
    clsparseStatus precondition(T* out, T* tmp)
    {
        if (use_dia_) return dia_apply(buf_.r, tmp, out, buf_.part_yp, nullptr);
        CLS_TRY(spmv_g(GT_, buf_.r, tmp, nullptr));
        return spmv_g(G_, tmp, out, nullptr);
    }
    int prec() const { return prec_; }
    bool fused() const { return fused_; }
    // A launch of the solve that gave up, of this engine or of another one on the
    // same buffers, leaves the slots with the sums it published and the count of
    // its sums behind: no launch of either runs on them again.
    bool persistent() const { return persist_ && launches_->gave_up == 0; }
    bool persistent_fsai() const { return persistent() && prec_ == kPrecFsai; }

    // After a chunk that ran `ran` iterations: r back in buf_.r when the
    // fused learned-FSAI iteration left it in r_alt (an odd count).
    clsparseStatus settle_r(int ran)
    {
        if (!fuse_gt_ || (ran & 1) == 0) return clsparseSuccess;
        CLS_HIP_TRY(hipMemcpyAsync(buf_.r, r_alt_, n_ * sizeof(T), hipMemcpyDeviceToDevice, s_));
        return clsparseSuccess;
    }

    // The fused iteration leaves p one update behind z: bring it up to date
    // (before a residual replacement re-bases it). ran: iterations the last
    // chunk executed.
    clsparseStatus materialize_p(int ran)
    {
        if (!fused_ || ran <= 0) return clsparseSuccess;
        const int j = (ran - 1) & 1;  // partials of the last executed x / r update
        hipLaunchKernelGGL((cg_materialize_p<T>), dim3(g_), dim3(256), 0, s_, n_, buf_.p, buf_.z,
                           buf_.part_rz[j], buf_.part_rz[j ^ 1], g_, buf_.st);
        CLS_HIP_TRY(hipGetLastError());
        return clsparseSuccess;
    }

    // z = M r of the current recurrence residual into the z buffer, where the
    // iterations keep z in registers only (the residual replacement re-bases
    // p on it). tmp: n values of scratch.
    clsparseStatus materialize_z(T* tmp)
    {
        if (prec_ == kPrecFsai && use_dia_) return dia_apply(buf_.r, tmp, buf_.z, buf_.part_yp, nullptr);
        return clsparseSuccess;
    }

private:
    // The kernels of the iterations after a set-up. Those that fuse the p update or
    // G^T r go on from their own state only, not from a persistent launch's.
    void start_kernels()
    {
        fused_ = can_fuse_ && !persistent();
        fuse_gt_ = can_fuse_gt_ && !persistent();
        at_start_ = true;
    }

    clsparseStatus run_persistent(CgDevState* host_state, int max_run, double go_on, bool* refused)
    {
        if constexpr (std::is_same_v<T, TX>) {
            CgPersistArgs<T> a{};
            a.n = static_cast<uint32_t>(n_);
            a.plan = plan_;
            a.vals = adia_.vals;
            a.sym = adia_.sym ? 1 : 0;
            a.x = x_;
            a.r = buf_.r;
            a.p = buf_.p;
            a.z = buf_.z;
            a.p2 = buf_.y;
            a.invD = prec_ == kPrecJacobi ? buf_.invD : nullptr;
            a.rz_in = buf_.part_rz[1];
            a.rz_out[0] = buf_.part_rz[0];
            a.rz_out[1] = buf_.part_rz[1];
            a.g_in = g_;
            a.st = buf_.st;
            a.slots = buf_.slots;
            a.max_run = max_run;
            a.go_on = go_on;
            a.spin_limit = persist_spin_limit();
            return run_alone(host_state, refused, [&] { return launch_cg_persist<T>(a, s_); });
        }
        return clsparseInvalidValue;
    }

    clsparseStatus run_persistent_fsai(CgDevState* host_state, int max_run, double go_on, double best, bool* refused)
    {
        if constexpr (std::is_same_v<T, float> && std::is_same_v<TX, float>) {
            FsaiPersistArgs a{};
            a.n = static_cast<uint32_t>(n_);
            a.plan = plan_;
            a.vals = adia_.vals;
            a.sym = adia_.sym ? 1 : 0;
            a.g = dia_.vals;
            a.x = x_;
            a.r = buf_.r;
            a.p = buf_.p;
            a.y = buf_.y;
            a.w = buf_.z;
            a.rz_in = buf_.part_rz[1];
            a.rz_out[0] = buf_.part_rz[0];
            a.rz_out[1] = buf_.part_rz[1];
            a.g_in = g_;
            a.st = buf_.st;
            a.slots = buf_.slots;
            a.max_run = max_run;
            a.go_on = go_on;
            a.best = best;
            a.spin_limit = persist_spin_limit();
            return run_alone(host_state, refused, [&] { return launch_fsai_persist(a, s_); });
        }
        return clsparseInvalidValue;
    }

    // One persistent kernel per device at a time: two that shared the CUs
    // could each hold some the other waits for.
    template <typename F>
    clsparseStatus run_alone(CgDevState* host_state, bool* refused, F&& launch)
    {
        std::lock_guard<std::mutex> one(persist_mutex(device_));
        if (persist_refused() || launch() != clsparseSuccess) {  // e.g. fewer CUs than the device has: nothing ran
            (void)hipGetLastError();
            ++launches_->refused;
            persist_ = false;
            if (at_start_) start_kernels();
            *refused = true;  // (and host_state is not written)
            return clsparseSuccess;
        }
        at_start_ = false;
        ++launches_->started;
        CLS_HIP_TRY(hipMemcpyAsync(host_state, buf_.st, sizeof(CgDevState), hipMemcpyDeviceToHost, s_));
        CLS_HIP_TRY(hipStreamSynchronize(s_));
        if (host_state->failed) ++launches_->gave_up;
        return clsparseSuccess;
    }

    // After the last iteration of a chunk: its convergence test, which the
    // next fused SpMV would otherwise run.
    clsparseStatus enqueue_chunk_end()
    {
        if (!fused_) return clsparseSuccess;
        hipLaunchKernelGGL(cg_test_kernel, dim3(1), dim3(256), 0, s_, buf_.st, buf_.part_nr[(kChunk - 1) & 1], g_);
        CLS_HIP_TRY(hipGetLastError());
        return clsparseSuccess;
    }

    clsparseStatus enqueue_iteration(int par)
    {
        const int* done = &buf_.st->done;
        if constexpr (std::is_same_v<T, float>) {
        if (fused_) {
            // y = A p' (p' = z + beta p on the fly) with <y, p'> and the previous
            // iteration's test; then p = p', x, r, z and their partials.
            CLS_TRY(launch_spmv_pn<T>(adia_, n_, g_, buf_.p, buf_.z, buf_.y, buf_.part_yp, buf_.part_rz[par ^ 1],
                                      buf_.part_rz[par], buf_.part_nr[par ^ 1], buf_.st, s_));
            hipLaunchKernelGGL((cg_update_kernel<T, TX, true>), dim3(g_), dim3(256), 0, s_, n_, x_, buf_.r,
                               buf_.z, buf_.p, buf_.y, buf_.invD, prec_, buf_.part_yp, buf_.part_rz[par ^ 1],
                               buf_.part_rz[par], buf_.part_nr[par], g_, buf_.st);
            CLS_HIP_TRY(hipGetLastError());
            return clsparseSuccess;
        }
        }
        if (adia_.vals != nullptr) {
            CLS_TRY(launch_dia_spmv(adia_, n_, g_, buf_.p, buf_.y, buf_.p, buf_.part_yp, done, s_));
        } else {
            CLS_TRY(launch_csrmv<T>(buf_.one, A_, buf_.p, buf_.zero, buf_.y, s_, ext_, done));
            hipLaunchKernelGGL((cg_dot_kernel<T>), dim3(g_), dim3(256), 0, s_, n_, buf_.y, buf_.p,
                               buf_.part_yp, buf_.st);
        }
        if (fuse_gt_) return dia_update_iteration(par);
        hipLaunchKernelGGL((cg_update_kernel<T, TX>), dim3(g_), dim3(256), 0, s_, n_, x_, buf_.r,
                           buf_.z, buf_.p, buf_.y, buf_.invD, prec_, buf_.part_yp,
                           buf_.part_rz[par ^ 1], buf_.part_rz[par], buf_.part_nr[par], g_,
                           buf_.st);
        if (prec_ == kPrecFsai && use_dia_) return dia_iteration(par);
        if (prec_ == kPrecFsai) CLS_TRY(apply_fsai(buf_.part_rz[par], done));
        hipLaunchKernelGGL((cg_pupdate_kernel<T>), dim3(g_), dim3(256), 0, s_, n_, buf_.p, buf_.z,
                           buf_.part_rz[par], buf_.part_rz[par ^ 1], buf_.part_nr[par], g_,
                           buf_.st);
        CLS_HIP_TRY(hipGetLastError());
        return clsparseSuccess;
    }

    // The FSAI preconditioner and p update of one iteration from diagonal
    // storage (z stays in registers: materialize_z forms it when needed).
    clsparseStatus dia_iteration(int par)
    {
        if constexpr (std::is_same_v<T, float>) {
            const uint16_t* v = dia_.vals;
            double* rz = buf_.part_rz[par];
            const double* rz0 = buf_.part_rz[par ^ 1];
            const double* nr = buf_.part_nr[par];
#define CLS_DIA_ITER(K) \
    launch_dia_iteration<K>(n_, g_, dia_off_, v, buf_.r, buf_.y, buf_.p, rz, rz0, nr, buf_.st, s_)
            switch (dia_.ndiag) {
            case 1: CLS_DIA_ITER(1); break;
            case 2: CLS_DIA_ITER(2); break;
            case 3: CLS_DIA_ITER(3); break;
            case 4: CLS_DIA_ITER(4); break;
            case 5: CLS_DIA_ITER(5); break;
            case 6: CLS_DIA_ITER(6); break;
            case 7: CLS_DIA_ITER(7); break;
            case 8: CLS_DIA_ITER(8); break;
            default: return clsparseInvalidValue;
            }
#undef CLS_DIA_ITER
            CLS_HIP_TRY(hipGetLastError());
            return clsparseSuccess;
        }
        return clsparseInvalidValue;
    }

    // The learned-FSAI iteration after y = A p with the x / r update fused
    // into w = G^T r: iteration k of a chunk reads r from r_[k & 1] and
    // writes it to the other buffer (chunks are of even length, so a whole
    // chunk ends with r in buf_.r; settle_r moves it back after a short
    // one); w lives in z, which this engine keeps in registers otherwise.
    clsparseStatus dia_update_iteration(int par)
    {
        if constexpr (std::is_same_v<T, float>) {
            const uint16_t* v = dia_.vals;
            const T* r_in = par ? r_alt_ : buf_.r;
            T* r_out = par ? buf_.r : r_alt_;
            double* rz = buf_.part_rz[par];
            const double* rz0 = buf_.part_rz[par ^ 1];
            double* nr = buf_.part_nr[par];
#define CLS_DIA_UPD(K)                                                                                          \
    launch_dia_update_iteration<K, TX>(n_, g_, dia_off_, v, x_, r_in, r_out, buf_.p, buf_.y, buf_.z, buf_.p,    \
                                       buf_.part_yp, rz, rz0, nr, buf_.st, s_)
            switch (dia_.ndiag) {
            case 1: CLS_DIA_UPD(1); break;
            case 2: CLS_DIA_UPD(2); break;
            case 3: CLS_DIA_UPD(3); break;
            case 4: CLS_DIA_UPD(4); break;
            case 5: CLS_DIA_UPD(5); break;
            case 6: CLS_DIA_UPD(6); break;
            case 7: CLS_DIA_UPD(7); break;
            case 8: CLS_DIA_UPD(8); break;
            default: return clsparseInvalidValue;
            }
#undef CLS_DIA_UPD
            CLS_HIP_TRY(hipGetLastError());
            return clsparseSuccess;
        }
        return clsparseInvalidValue;
    }

    // z = G (G^T r) through y (free between the r update and the next A p);
    // partials of <r, z> = ||G^T r||^2, read from y alone.
    clsparseStatus apply_fsai(double* part_rz, const int* done)
    {
        if (use_dia_) return dia_apply(buf_.r, buf_.y, buf_.z, part_rz, done);
        CLS_TRY(spmv_g(GT_, buf_.r, buf_.y, done));
        CLS_TRY(spmv_g(G_, buf_.y, buf_.z, done));
        hipLaunchKernelGGL((cg_dot_kernel<T>), dim3(g_), dim3(256), 0, s_, n_, buf_.y, buf_.y,
                           part_rz, buf_.st);
        CLS_HIP_TRY(hipGetLastError());
        return clsparseSuccess;
    }

    // tmp = G^T r (with ||tmp||^2 partials), out = G tmp, diagonal storage.
    clsparseStatus dia_apply(const T* r, T* tmp, T* out, double* part, const int* done)
    {
        if constexpr (std::is_same_v<T, float>) {
            switch (dia_.ndiag) {
            case 1: launch_dia_apply<1>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 2: launch_dia_apply<2>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 3: launch_dia_apply<3>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 4: launch_dia_apply<4>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 5: launch_dia_apply<5>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 6: launch_dia_apply<6>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 7: launch_dia_apply<7>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            case 8: launch_dia_apply<8>(n_, g_, dia_off_, dia_.vals, r, tmp, out, part, done, s_); break;
            default: return clsparseInvalidValue;
            }
            CLS_HIP_TRY(hipGetLastError());
            return clsparseSuccess;
        }
        return clsparseInvalidValue;
    }

    // out = M_ in for one factor of M, in its stored precision.
    clsparseStatus spmv_g(const clsparseCsrMatrix* M_, const T* in, T* out, const int* done)
    {
        if constexpr (std::is_same_v<T, float>) {
            if (g_bf16_) return launch_csrmv_bf16(buf_.one, M_, in, buf_.zero, out, s_, done);
        }
        return launch_csrmv<T>(buf_.one, M_, in, buf_.zero, out, s_, false, done);
    }

    const clsparseCsrMatrix* A_;
    TX* x_;
    const T* b_;
    size_t n_;
    int prec_;
    int crit_;
    bool fused_ = false;  // Jacobi / none with A in diagonal storage: fused p update
    CgBuffers<T>& buf_;
    hipStream_t s_;
    bool ext_;
    uint32_t g_;
    const clsparseCsrMatrix* G_;
    const clsparseCsrMatrix* GT_;
    bool g_bf16_;
    T* r_alt_;
    int device_;
    clsparseAmdSolverLaunches* launches_;  // of the solve
    PersistPlan plan_{};
    bool persist_ = false;      // whole chunks in one cooperative launch (cg_persist.hpp)
    bool can_fuse_ = false, can_fuse_gt_ = false;  // where no persistent launch runs
    bool at_start_ = true;      // no persistent launch since the set-up
    bool fuse_gt_ = false;  // learned factor in diagonal storage: x / r update fused into G^T r
    bool use_dia_ = false;
    FsaiDia dia_{};
    DiaMatrix<T> adia_{};
    DiaOffsets dia_off_{};
    hipGraph_t graph_ = nullptr;
    hipGraphExec_t exec_ = nullptr;
};

template <typename T>
clsparseStatus cg_solve(cldenseVector* x, const clsparseCsrMatrix* A, const cldenseVector* b,
                        clSParseSolverControl sc, clsparseControl control)
{
    // Size rule of conjugate-gradients.hpp L57-62; CG also needs a square A
    // (the reference would overrun its length-N temporaries otherwise).
    if (A->num_cols != b->num_values || A->num_rows != x->num_values ||
        A->num_rows != A->num_cols)
        return clsparseInvalidSystemSize;
    const size_t n = A->num_cols;
    hipStream_t s = control->solver_stream;
    T* xp = dev_ptr<T>(x->values, x->off_values);
    const T* bp = dev_ptr<T>(b->values, b->off_values);
    if (n > 0 && (xp == nullptr || bp == nullptr)) return clsparseInvalidMemObject;

    // Stencil matrices: A's values in diagonal storage for the iterations
    // (same row sums as the CSR-Adaptive SpMV; not with extended precision).
    // The kernels write what the host decides by into pinned memory: one wait
    // for ||b|| and the sampled offsets, one for the checks of the diagonal
    // storage and the first residual (a wait and a copy for each of the six
    // took 0.25 ms of a small solve).
    void* pinned = nullptr;
    CLS_TRY(control_pinned(control, align_up(sizeof(CgDevState)) + sizeof(SolverHost), &pinned));
    CgDevState* hs = static_cast<CgDevState*>(pinned);
    SolverHost* hp = reinterpret_cast<SolverHost*>(static_cast<char*>(pinned) + align_up(sizeof(CgDevState)));
    CLS_TRY(enter_solver_stream(control));
    // ||b||_1 (conjugate-gradients.hpp L77-81)
    CLS_TRY(launch_reduce<T, double>(RedOp::Abs, bp, nullptr, n, &hp->norm_b, false, control->red_partials, s));
    const bool sampled = !control->extended_precision && dia_sample(A, hp->samples, s);
    CLS_HIP_TRY(hipGetLastError());
    CLS_HIP_TRY(hipStreamSynchronize(s));
    const double norm_b = hp->norm_b;

    if (norm_b == 0) {
        // b == 0: x = b and zero tolerances (L87-95).
        sc->nIters = 0;
        sc->absoluteTolerance = 0.0;
        sc->relativeTolerance = 0.0;
        if (n > 0)
            CLS_HIP_TRY(hipMemcpyAsync(xp, bp, n * sizeof(T), hipMemcpyDeviceToDevice, s));
        sc->stats = clsparseAmdSolverStats{};
        sc->launches = clsparseAmdSolverLaunches{};
        CLS_TRY(leave_solver_stream(control));
        return clsparseSuccess;
    }

    const auto t0 = std::chrono::steady_clock::now();
    DiaOffsets a_off{};
    int a_ndiag = sampled ? dia_from_samples(A, hp->samples, &a_off) : 0;
    void* work = nullptr;
    CLS_TRY(control_workspace(control, CgBuffers<T>::bytes(n) + (a_ndiag ? align_up(a_ndiag * n * sizeof(T)) : 0),
                              &work));
    Carve c{static_cast<char*>(work)};
    CgBuffers<T> buf;
    buf.carve(c, n);
    T* a_dia = a_ndiag ? c.take<T>(a_ndiag * n) : nullptr;

    // Device state: tolerances of the solver control (solver-control.hpp L52-64).
    CgDevState init{};
    init.norm_ref = norm_b;
    init.rel_tol = sc->relativeTolerance;
    init.abs_tol = sc->absoluteTolerance;
    init.max_iters = sc->maxIters;
    init.crit = kCritL1Ref;
    const int prec = (sc->preconditioner == DIAGONAL) ? kPrecJacobi : kPrecNone;
    hipLaunchKernelGGL((solver_prepare_kernel<T, CgDevState>), dim3(ew_grid(persist_slot_words())),
                       dim3(256), 0, s, init, buf.st, buf.one, buf.zero, static_cast<double*>(nullptr), buf.slots,
                       static_cast<uint32_t>(persist_slot_words()), persist_slot_empty());
    CLS_HIP_TRY(hipGetLastError());
    if (a_ndiag) {
        CLS_TRY((dia_fill<T, T>(A, n, a_ndiag, a_off, a_dia, prec == kPrecJacobi ? buf.invD : nullptr, hp, s)));
    } else if (prec == kPrecJacobi) {
        hipLaunchKernelGGL((extract_inv_diag<T, T>), dim3((A->num_rows + 255) / 256), dim3(256), 0,
                           s, A->num_rows, dev_ptr<uint32_t>(A->row_pointer, A->off_row_pointer),
                           dev_ptr<uint32_t>(A->col_indices, A->off_col_indices),
                           dev_ptr<T>(A->values, A->off_values), buf.invD);
        CLS_HIP_TRY(hipGetLastError());
    }
    CLS_TRY(cg_setup<T>(A, xp, bp, n, prec, kCritL1Ref, buf, s, control->extended_precision, false, &hp->init_res));
    CLS_HIP_TRY(hipStreamSynchronize(s));
    DiaMatrix<T> adia{};
    if (a_ndiag && hp->dia_bad) a_ndiag = 0;
    if (a_ndiag) adia = DiaMatrix<T>{a_dia, a_ndiag, hp->dia_unsym == 0, a_off};
    CgEngine<T> eng(A, xp, bp, n, prec, kCritL1Ref, buf, s, control->extended_precision, nullptr, nullptr,
                    false, nullptr, &adia, nullptr, control->num_cus, control->device, &sc->launches);

    sc->initialResidual = hp->init_res;  // L127-129
    sc->stats = clsparseAmdSolverStats{};
    sc->launches = clsparseAmdSolverLaunches{};
    if (sc->finished(sc->initialResidual)) {  // L134-138 (uses the stored nIters)
        sc->nIters = 0;
        sc->stats.l1_residual = sc->initialResidual;
        CLS_TRY(leave_solver_stream(control));
        return clsparseSuccess;
    }

    int printed = 0;
    // VERBOSE prints every residual from the history ring: kChunk at a time.
    const int max_run = sc->printMode == VERBOSE ? kChunk : kMaxRun;
    CLS_TRY(eng.run(hs, sc->initialResidual, max_run, [&](const CgDevState& st) {
        const int upto = st.done ? st.n_iters + 1 : st.iter;
        if (sc->printMode == VERBOSE) {
            for (int k = printed; k < upto; ++k) {
                sc->nIters = k;
                sc->currentResidual = st.hist[k % kHist];
                sc->print();
            }
        }
        printed = upto;
    }));
    sc->nIters = hs->n_iters;
    sc->currentResidual = hs->cur_res;
    CLS_TRY(leave_solver_stream(control));

    const auto t1 = std::chrono::steady_clock::now();
    sc->stats.iterations = hs->n_iters + 1;
    sc->stats.l1_residual = hs->cur_res;
    sc->stats.seconds = std::chrono::duration<double>(t1 - t0).count();
    sc->stats.status_detail = hs->converged ? 0 : 1;
    sc->stats.a_diagonals = a_ndiag;
    return clsparseSuccess;
}

template <typename T>
clsparseStatus cg_entry(cldenseVector* x, const clsparseCsrMatrix* A, const cldenseVector* b,
                        clSParseSolverControl solverControl, clsparseControl control)
{
    // Check order of conjugate-gradients.cpp L28-41.
    if (!clsparseInitialized) return clsparseNotInitialized;
    if (control == nullptr) return clsparseInvalidControlObject;
    if (solverControl == nullptr) return clsparseInvalidSolverControlObject;
    if (x == nullptr || A == nullptr || b == nullptr) return clsparseInvalidValue;
    const clsparseStatus status = cg_solve<T>(x, A, b, solverControl, control);
    solverControl->printSummary(status);  // L59
    return status;
}

// y = A x through the diagonal storage the CG solvers move a stencil matrix's
// values to: the plain SpMV (fused == 0) or the FP32-solver kernel that forms
// its operand as p' = fma(0, x, x) on the first iteration (fused != 0).
template <typename T>
clsparseStatus csrmv_diag(const clsparseCsrMatrix* A, const cldenseVector* x, cldenseVector* y, int fused,
                          cl_int* ndiag, clsparseControl control)
{
    CLS_TRY(check_init_control(control));
    if (A == nullptr || x == nullptr || y == nullptr || ndiag == nullptr) return clsparseInvalidValue;
    *ndiag = 0;
    if (A->num_rows != A->num_cols || x->num_values < A->num_cols || y->num_values < A->num_rows)
        return clsparseInvalidSize;
    const size_t n = A->num_rows;
    const T* xp = dev_ptr<T>(x->values, x->off_values);
    T* yp = dev_ptr<T>(y->values, y->off_values);
    if (n > 0 && (xp == nullptr || yp == nullptr)) return clsparseInvalidMemObject;
    hipStream_t s = control->solver_stream;
    CLS_TRY(enter_solver_stream(control));
    void* pinned = nullptr;
    CLS_TRY(control_pinned(control, sizeof(SolverHost), &pinned));
    SolverHost* hp = static_cast<SolverHost*>(pinned);
    if (!dia_sample(A, hp->samples, s)) return leave_solver_stream(control);
    CLS_HIP_TRY(hipGetLastError());
    CLS_HIP_TRY(hipStreamSynchronize(s));
    DiaOffsets off{};
    const int nd = dia_from_samples(A, hp->samples, &off);
    if (nd == 0) return leave_solver_stream(control);
    void* work = nullptr;
    CLS_TRY(control_workspace(control,
                              align_up(nd * n * sizeof(T)) + align_up(sizeof(CgDevState)) +
                                  align_up(kReducePartialsMax * sizeof(double)),
                              &work));
    Carve c{static_cast<char*>(work)};
    T* vals = c.take<T>(nd * n);
    CgDevState* st = c.take<CgDevState>(1);
    double* part = c.take<double>(kReducePartialsMax);
    CLS_TRY((dia_fill<T, T>(A, n, nd, off, vals, nullptr, hp, s)));
    CLS_HIP_TRY(hipStreamSynchronize(s));
    if (hp->dia_bad) return leave_solver_stream(control);
    const bool sym = hp->dia_unsym == 0;
    const DiaMatrix<T> D{vals, nd, sym, off};
    const uint32_t g = grid_for(n);
    if (fused && dia_buf_fits(nd, n, sizeof(T))) {
        CgDevState init{};
        init.first = 1;  // beta = 0 and z = p: p' = p
        CLS_HIP_TRY(hipMemcpyAsync(st, &init, sizeof(CgDevState), hipMemcpyHostToDevice, s));
        CLS_TRY(launch_spmv_pn<T>(D, n, g, xp, xp, yp, part, part, part, part, st, s));
    } else {
        CLS_TRY(launch_dia_spmv<T>(D, n, g, xp, yp, nullptr, nullptr, nullptr, s));
    }
    CLS_HIP_TRY(hipStreamSynchronize(s));
    *ndiag = nd;
    CLS_TRY(leave_solver_stream(control));
    return finish_op(control);
}

}  // namespace

extern "C" clsparseStatus clsparseAmdScsrmvDiag(const clsparseCsrMatrix* A, const cldenseVector* x,
                                                cldenseVector* y, cl_int fused, cl_int* ndiag,
                                                const clsparseControl control)
{
    return csrmv_diag<float>(A, x, y, fused, ndiag, control);
}

extern "C" clsparseStatus clsparseAmdDcsrmvDiag(const clsparseCsrMatrix* A, const cldenseVector* x,
                                                cldenseVector* y, cl_int fused, cl_int* ndiag,
                                                const clsparseControl control)
{
    return csrmv_diag<double>(A, x, y, fused, ndiag, control);
}

// src/library/solvers/conjugate-gradients.cpp L18-64
extern "C" clsparseStatus clsparseScsrcg(cldenseVector* x, const clsparseCsrMatrix* A,
                                         const cldenseVector* b,
                                         clSParseSolverControl solverControl,
                                         clsparseControl control)
{
    return cg_entry<float>(x, A, b, solverControl, control);
}

// src/library/solvers/conjugate-gradients.cpp L66-116
extern "C" clsparseStatus clsparseDcsrcg(cldenseVector* x, const clsparseCsrMatrix* A,
                                         const cldenseVector* b,
                                         clSParseSolverControl solverControl,
                                         clsparseControl control)
{
    return cg_entry<double>(x, A, b, solverControl, control);
}

// ---- mixed-precision CG with reliable updates (no reference counterpart) -----
//
// One preconditioned CG run in precision TI (values of A, r, z, p, y) with the
// solution x held and updated in FP64 and every dot product and norm
// accumulated in FP64. Whenever the recurrence residual has fallen by a factor
// `delta` since the last replacement, or claims convergence, the residual is
// replaced by the FP64 true residual b - A x (FP64 CSR-Adaptive SpMV) -- the
// reliable-update scheme of van der Vorst and Ye ("Residual replacement
// strategies for Krylov subspace iterative methods", SIAM J. Sci. Comput.
// 22(3), 2000) -- and the search direction is re-based on the new residual
// (p' = z' + (<r',z'>/<r,z>) (p - z), z' = M r'), so the Krylov process goes on
// without a restart. The FP64 true relative residual ||b - A x||_2 / ||b||_2
// decides convergence. TI = float is the mixed-precision solver; TI = double
// is FP64 PCG judged by the same FP64 true residual (the baseline).

namespace {

constexpr int kStagnationChunks = 16;  // learned FSAI must halve ||r|| within this many chunks
constexpr int kPilotChunks = 2;        // chunks per preconditioner in the pilot race

// Jacobi wins the pilot race only when its rate beats the learned factor's by
// this factor (CLSPARSE_AMD_RACE_MARGIN overrides): over the pilot's window
// (iterations 33-64) Jacobi's residual falls faster than over a whole solve
// -- its first iterations damp the components it handles well -- while the
// learned factor's rate there is about its whole-solve rate (160^3
// anisotropic problem: Jacobi 0.0228 per iteration in the window, 0.0183
// over the solve; learned factor 0.0322 and 0.033). A factor that is exactly
// Jacobi but dearer per iteration (a zero network) still loses: its rate is
// below Jacobi's by the cost ratio, about 1.27.
double race_margin()
{
    const char* e = std::getenv("CLSPARSE_AMD_RACE_MARGIN");
    const double m = e ? std::atof(e) : 1.15;
    return m > 0 ? m : 1.15;
}

// CLSPARSE_AMD_FSAI_POLICY=always keeps the learned factor unless it breaks
// down or stagnates; "race" runs the pilot race on every new factor; the
// default runs it only when a loss estimate leaves the factor's lead over
// Jacobi in doubt (estimate_enabled, factor_losses).
bool race_enabled()
{
    const char* e = std::getenv("CLSPARSE_AMD_FSAI_POLICY");
    return !(e && std::strcmp(e, "always") == 0);
}
bool estimate_enabled()
{
    const char* e = std::getenv("CLSPARSE_AMD_FSAI_POLICY");
    return !(e && (std::strcmp(e, "always") == 0 || std::strcmp(e, "race") == 0));
}
// A new factor whose estimated ||G^T A G - I||_F^2 is at most this fraction
// of Jacobi's (G = D^-1/2) is kept without the pilot race. Measured ratios:
// 0.25-0.44 for the trained network on the held-out 3-D problems, 0.33 on
// the 2-D training family; 1 for the zero network, 8-140 for a network with
// a wrong output layer.
constexpr double kLossRatioKeep = 0.5;
constexpr int kLossProbes = 1;  // within 0.5 % of eight probes at n >= 10^5

// z_i = +-1 from a hash of (seed, i): a Rademacher probe.
__global__ __launch_bounds__(256) void probe_kernel(size_t n, uint64_t seed, float* __restrict__ z)
{
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        uint64_t x = (seed + 1) * 0x9E3779B97F4A7C15ull ^ (static_cast<uint64_t>(i) * 0xD1B54A32D192ED03ull);
        x ^= x >> 31;
        x *= 0xBF58476D1CE4E5B9ull;
        x ^= x >> 29;
        z[i] = (x & 1) ? 1.f : -1.f;
    }
}

// out = D^-1/2 in (invD = 1 / a_ii), and the partials of ||out||^2 (one
// per workgroup) when part is given.
__global__ __launch_bounds__(256) void jacobi_factor_kernel(size_t n, const float* __restrict__ invD,
                                                            const float* __restrict__ in, float* __restrict__ out,
                                                            double* __restrict__ part)
{
    __shared__ double sh[4];
    double a = 0.0;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        const float v = sqrtf(invD[i]) * in[i];
        out[i] = v;
        a += static_cast<double>(v) * static_cast<double>(v);
    }
    a = block_sum256(a, sh);
    if (part != nullptr && threadIdx.x == 0) part[blockIdx.x] = a;
}

// Hutchinson estimates, over `probes` Rademacher vectors z, of
// ||F^T A F - I||_F^2 / n for the learned factor F = G (diagonal storage,
// as the solver applies it) and for Jacobi's F = D^-1/2, with A in diagonal
// storage: t = F z, y = A t with <y, t>, w = F^T y with ||w||^2, and
// ||F^T A F z - z||^2 = ||w||^2 - 2 <y, t> + n. z, t, y, w: n values each;
// part_a, part_b: one double per workgroup of grid_for(n).
clsparseStatus factor_losses(const FsaiDia& dia, const DiaMatrix<float>& adia, const float* invD, size_t n,
                             int probes, float* z, float* t, float* y, float* w, double* part_a, double* part_b,
                             hipStream_t s, double* loss_fsai, double* loss_jacobi)
{
    const uint32_t g = grid_for(n);
    DiaOffsets off{};
    for (int d = 0; d < kFsaiMaxDiags; ++d) off.o[d] = dia.off[d];
    std::vector<double> ha(g), hb(g);
    double acc[2] = {0.0, 0.0};
    for (int k = 0; k < probes; ++k) {
        hipLaunchKernelGGL(probe_kernel, dim3(g), dim3(256), 0, s, n, static_cast<uint64_t>(k), z);
        for (int f = 0; f < 2; ++f) {
            if (f == 0) {
                switch (dia.ndiag) {
#define CLS_G(K) hipLaunchKernelGGL((fsai_g_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, dia.vals, z, t, nullptr)
                case 1: CLS_G(1); break;
                case 2: CLS_G(2); break;
                case 3: CLS_G(3); break;
                case 4: CLS_G(4); break;
                case 5: CLS_G(5); break;
                case 6: CLS_G(6); break;
                case 7: CLS_G(7); break;
                case 8: CLS_G(8); break;
                default: return clsparseInvalidValue;
#undef CLS_G
                }
            } else {
                hipLaunchKernelGGL(jacobi_factor_kernel, dim3(g), dim3(256), 0, s, n, invD, z, t,
                                   static_cast<double*>(nullptr));
            }
            CLS_TRY(launch_dia_spmv(adia, n, g, t, y, t, part_a, nullptr, s));
            if (f == 0) {
                switch (dia.ndiag) {
#define CLS_GT(K) \
    hipLaunchKernelGGL((fsai_gt_dia_kernel<K>), dim3(g), dim3(256), 0, s, n, off, dia.vals, y, w, part_b, nullptr)
                case 1: CLS_GT(1); break;
                case 2: CLS_GT(2); break;
                case 3: CLS_GT(3); break;
                case 4: CLS_GT(4); break;
                case 5: CLS_GT(5); break;
                case 6: CLS_GT(6); break;
                case 7: CLS_GT(7); break;
                case 8: CLS_GT(8); break;
                default: return clsparseInvalidValue;
#undef CLS_GT
                }
            } else {
                hipLaunchKernelGGL(jacobi_factor_kernel, dim3(g), dim3(256), 0, s, n, invD, y, w, part_b);
            }
            CLS_HIP_TRY(hipGetLastError());
            CLS_HIP_TRY(hipMemcpyAsync(ha.data(), part_a, g * sizeof(double), hipMemcpyDeviceToHost, s));
            CLS_HIP_TRY(hipMemcpyAsync(hb.data(), part_b, g * sizeof(double), hipMemcpyDeviceToHost, s));
            CLS_HIP_TRY(hipStreamSynchronize(s));
            double yt = 0.0, ww = 0.0;
            for (uint32_t i = 0; i < g; ++i) {
                yt += ha[i];
                ww += hb[i];
            }
            acc[f] += (ww - 2.0 * yt + static_cast<double>(n)) / static_cast<double>(n);
        }
    }
    *loss_fsai = acc[0] / probes;
    *loss_jacobi = acc[1] / probes;
    return clsparseSuccess;
}

// r = (T) r64
template <typename T>
__global__ __launch_bounds__(256) void rr_cast(size_t n, const double* __restrict__ r64,
                                               T* __restrict__ r)
{
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
        r[i] = static_cast<T>(r64[i]);
}

// x += xd, xd = 0 (where an increment is kept), r64 = b: what the true residual
// starts from.
template <typename T>
__global__ __launch_bounds__(256) void flush_and_copy(size_t n, double* __restrict__ x, T* __restrict__ xd,
                                                      const double* __restrict__ b, double* __restrict__ r64)
{
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        if (xd != nullptr) {
            x[i] += static_cast<double>(xd[i]);
            xd[i] = T(0);
        }
        r64[i] = b[i];
    }
}

// x += (double) xd; xd = 0: folds the low-precision solution increment of
// the inner iterations into the FP64 solution.
template <typename T>
__global__ __launch_bounds__(256) void flush_increment(size_t n, double* __restrict__ x, T* __restrict__ xd)
{
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        x[i] += static_cast<double>(xd[i]);
        xd[i] = T(0);
    }
}

// s = <r', z'> / <r, z>;  p = z' + s (p - z);  z = z'.
// z_is_p: z takes the new p instead (an engine with the fused p update reads
// z only to form p' = fma(beta, p, z), with beta = 0 right after this).
template <typename T>
__global__ __launch_bounds__(256) void rr_rebase(size_t n, T* __restrict__ p, T* __restrict__ z,
                                                 const T* __restrict__ znew,
                                                 const double* __restrict__ part_old,
                                                 const double* __restrict__ part_new, uint32_t g, int z_is_p)
{
    __shared__ double sh[4];
    const double rz_old = sum_partials(part_old, g, sh);
    const double rz_new = sum_partials(part_new, g, sh);
    const T sc = static_cast<T>(rz_old != 0.0 ? rz_new / rz_old : 0.0);
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) {
        const T zn = znew[i];
        const T pn = zn + sc * (p[i] - z[i]);
        p[i] = pn;
        z[i] = z_is_p ? pn : zn;
    }
}

__global__ __launch_bounds__(256) void copy_partials(const double* __restrict__ src,
                                                     double* __restrict__ dst, uint32_t g)
{
    for (uint32_t i = threadIdx.x; i < g; i += 256) dst[i] = src[i];
}

// Lets the loop go on after a residual replacement: clears done / converged
// and sets the recurrence residual to the replaced one.
__device__ void resume(CgDevState* st, const double* __restrict__ rnorm)
{
    st->done = 0;
    st->converged = 0;
    st->cur_res = *rnorm / st->norm_ref;
    st->first = 1;  // p is current (set up or re-based)
    st->pending = 0;
    st->failed = 0;
}

__global__ void state_resume(CgDevState* st, const double* __restrict__ rnorm)
{
    if (threadIdx.x == 0) resume(st, rnorm);
}

// The replaced residual of an elementwise preconditioner in one kernel: r =
// (T) r64, z' = M r, partials of <r, z'> (summed as cg_dot_kernel sums them), and
// state_resume.
template <typename T>
__global__ __launch_bounds__(256) void rr_precondition(size_t n, const double* __restrict__ r64, T* __restrict__ r,
                                                       T* __restrict__ znew, const T* __restrict__ invD, int prec,
                                                       double* __restrict__ part, CgDevState* st,
                                                       const double* __restrict__ rnorm)
{
    __shared__ double sh[4];
    if (blockIdx.x == 0 && threadIdx.x == 0) resume(st, rnorm);
    double a = 0.0;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256;
    for (size_t i0 = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x; i0 < n; i0 += kRows * stride) {
        double rv[kRows];
        T dv[kRows];
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= n) continue;
            rv[u] = r64[i];
            dv[u] = prec == kPrecJacobi ? invD[i] : T(1);
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const size_t i = i0 + u * stride;
            if (i >= n) continue;
            const T ri = static_cast<T>(rv[u]), zi = prec == kPrecJacobi ? ri * dv[u] : ri;
            r[i] = ri;
            znew[i] = zi;
            a += static_cast<double>(ri) * static_cast<double>(zi);
        }
    }
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = a;
}

// CLSPARSE_AMD_MIXED_X64=1: the mixed solvers keep the solution in FP64 and
// update it every iteration (default: an FP32 increment, folded into the FP64
// x at each residual replacement).
bool mixed_x64()
{
    const char* e = std::getenv("CLSPARSE_AMD_MIXED_X64");
    return e && e[0] == '1';
}

// X64 (mixed only): the inner iterations update the caller's FP64 x in every
// iteration instead of an FP32 increment folded in at each replacement.
template <typename TI, bool X64 = false>
clsparseStatus reliable_solve(cldenseVector* x, const clsparseCsrMatrix* A, const cldenseVector* b,
                              clSParseSolverControl sc, clsparseControl control,
                              clsparseAmdFsai fsai = nullptr)
{
    if (!clsparseInitialized) return clsparseNotInitialized;
    if (control == nullptr) return clsparseInvalidControlObject;
    if (sc == nullptr) return clsparseInvalidSolverControlObject;
    if (x == nullptr || A == nullptr || b == nullptr) return clsparseInvalidValue;
    if (A->num_cols != b->num_values || A->num_rows != x->num_values ||
        A->num_rows != A->num_cols)
        return clsparseInvalidSystemSize;

    constexpr bool kMixed = sizeof(TI) == sizeof(float);
    constexpr bool kIncr = kMixed && !X64;  // FP32 solution increment
    const size_t n = A->num_rows;
    const size_t nnz = A->num_nonzeros;
    if (fsai && fsai_n(fsai) != n) return clsparseInvalidSystemSize;
    hipStream_t s = control->solver_stream;
    double* xp = dev_ptr<double>(x->values, x->off_values);
    const double* bp = dev_ptr<double>(b->values, b->off_values);
    if (n > 0 && (xp == nullptr || bp == nullptr)) return clsparseInvalidMemObject;

    // Residual replacement once the recurrence residual has fallen by delta
    // since the last one: two decades keep the FP32 recurrence far above its
    // drift (about sqrt(eps32) = 3e-4 of the replacement point's residual);
    // 0.01 against 0.1 halves the replacements at the same iteration counts
    // (160^3 learned FSAI and Jacobi to 1e-8, 128^3 Jacobi to 1e-10), and
    // 0.003 began to add iterations.
    double delta = 0.01;
    if (const char* e = std::getenv("CLSPARSE_AMD_RELIABLE_DELTA")) delta = std::atof(e);

    const auto t0 = std::chrono::steady_clock::now();
    // (after the caller's queued work: A's arrays and the partials buffer)
    CLS_TRY(enter_solver_stream(control));
    // The factor first: creating its metadata uses the control's pinned buffer.
    int prec = (sc->preconditioner == DIAGONAL) ? kPrecJacobi : kPrecNone;
    int used = prec;  // statistics: 0 none, 1 Jacobi, 2 FSAI, 3 FSAI -> Jacobi
    const clsparseCsrMatrix* G = nullptr;
    const clsparseCsrMatrix* GT = nullptr;
    bool g_bf16 = false;
    FsaiDia dia{};
    bool have_dia = false;
    if (fsai) {
        CLS_TRY(fsai_prepare(fsai, s));
        if constexpr (kMixed) {
            // The factor's values in BF16 (CLSPARSE_AMD_FSAI_BF16=0: FP32):
            // M = G G^T stays symmetric positive definite for any rounding of
            // a nonsingular G, and the SpMVs with G move fewer bytes.
            const char* e = std::getenv("CLSPARSE_AMD_FSAI_BF16");
            g_bf16 = !(e && e[0] == '0');
            G = g_bf16 ? fsai_G16(fsai) : fsai_G32(fsai);
            GT = g_bf16 ? fsai_GT16(fsai) : fsai_GT32(fsai);
            // Diagonal storage of the BF16 factor where its pattern allows
            // (CLSPARSE_AMD_FSAI_DIA=0: always the CSR SpMVs).
            const char* ed = std::getenv("CLSPARSE_AMD_FSAI_DIA");
            have_dia = g_bf16 && !(ed && ed[0] == '0') && fsai_dia(fsai, &dia);
        } else {
            G = fsai_G64(fsai);
            GT = fsai_GT64(fsai);
        }
        prec = fsai_valid(fsai) ? kPrecFsai : kPrecJacobi;
        used = fsai_valid(fsai) ? 2 : 3;
        if (!have_dia) CLS_TRY(fsai_ensure_meta(fsai, control));  // CSR SpMVs with G and G^T
    }

    // Candidate diagonals of A from rows spread over it (a stencil's interior
    // rows hold all of them); the fill kernel below checks every row against
    // them. CLSPARSE_AMD_DIA=0: CSR always. ||b|| comes with the same wait.
    void* pinned = nullptr;
    CLS_TRY(control_pinned(control, align_up(sizeof(CgDevState)) + sizeof(SolverHost), &pinned));
    CgDevState* hs = static_cast<CgDevState*>(pinned);
    SolverHost* hp = reinterpret_cast<SolverHost*>(static_cast<char*>(pinned) + align_up(sizeof(CgDevState)));
    CLS_TRY(launch_reduce<double, double>(RedOp::Sqr, bp, nullptr, n, &hp->norm_b, true, control->red_partials, s));
    const bool sampled = dia_sample(A, hp->samples, s);
    CLS_HIP_TRY(hipGetLastError());
    CLS_HIP_TRY(hipStreamSynchronize(s));
    const double norm_b = hp->norm_b;
    sc->stats = clsparseAmdSolverStats{};
    sc->launches = clsparseAmdSolverLaunches{};
    if (norm_b == 0) {
        sc->nIters = 0;
        if (n > 0) CLS_HIP_TRY(hipMemcpyAsync(xp, bp, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        CLS_TRY(leave_solver_stream(control));
        return clsparseSuccess;
    }
    DiaOffsets a_off{};
    int a_ndiag = sampled ? dia_from_samples(A, hp->samples, &a_off) : 0;

    // Workspace: TI values of A (mixed only), FP64 residual, the solution
    // increment since the last residual replacement (mixed: an FP32 vector
    // folded into the FP64 x at every true residual, so the inner iterations
    // move 4-byte x values; FP64: a copy of x restored if a preconditioner
    // breaks down), scalars, TI start residual, then the CG buffers; with a
    // factor also the pilot race's start point and the learned factor's
    // pilot end point.
    const size_t bytes = (kMixed ? align_up(nnz * sizeof(TI)) : 0) + align_up(n * sizeof(double)) +
                         align_up(n * (kIncr ? sizeof(TI) : sizeof(double))) +
                         align_up(2 * sizeof(double)) + align_up(n * sizeof(TI)) +
                         CgBuffers<TI>::bytes(n) + (fsai ? 2 * align_up(n * sizeof(double)) : 0) +
                         (a_ndiag ? align_up(a_ndiag * n * sizeof(TI)) : 0);
    void* work = nullptr;
    CLS_TRY(control_workspace(control, bytes, &work));
    Carve c{static_cast<char*>(work)};
    TI* valsI = kMixed ? c.take<TI>(nnz) : nullptr;
    double* r64 = c.take<double>(n);
    TI* xd = kIncr ? c.take<TI>(n) : nullptr;              // mixed: increment since the last flush
    double* xsave = kIncr ? nullptr : c.take<double>(n);  // FP64 x: last replacement point
    double* sc64 = c.take<double>(2);  // -1, +1
    TI* rI = c.take<TI>(n);            // TI start residual; FSAI temporary afterwards
    CgBuffers<TI> buf;
    buf.carve(c, n);
    double* xstart = fsai ? c.take<double>(n) : nullptr;
    double* xpilot = fsai ? c.take<double>(n) : nullptr;
    TI* a_dia = a_ndiag ? c.take<TI>(a_ndiag * n) : nullptr;

    // Device state of the TI loop: L2 recurrence residual relative to ||b||.
    CgDevState init{};
    init.norm_ref = norm_b;
    init.rel_tol = sc->relativeTolerance;
    init.abs_tol = 0.0;
    init.max_iters = sc->maxIters - 1;
    init.crit = kCritL2;
    hipLaunchKernelGGL((solver_prepare_kernel<TI, CgDevState>), dim3(ew_grid(persist_slot_words())),
                       dim3(256), 0, s, init, buf.st, buf.one, buf.zero, sc64, buf.slots,
                       static_cast<uint32_t>(persist_slot_words()), persist_slot_empty());
    CLS_HIP_TRY(hipGetLastError());

    // TI-precision A on the same pattern (shares col_indices, row_pointer, meta).
    clsparseCsrMatrix AI = *A;
    if constexpr (kMixed) {
        hipLaunchKernelGGL((cast_kernel<double, TI>), dim3(ew_grid(nnz)), dim3(256), 0, s, nnz,
                           dev_ptr<double>(A->values, A->off_values), valsI);
        AI.values = valsI;
        AI.off_values = 0;
    }
    TI* const invD = prec != kPrecNone ? buf.invD : nullptr;
    if (a_ndiag) {
        CLS_TRY((dia_fill<double, TI>(A, n, a_ndiag, a_off, a_dia, invD, hp, s)));
    } else if (invD != nullptr) {
        hipLaunchKernelGGL((extract_inv_diag<double, TI>), dim3((n + 255) / 256), dim3(256), 0, s,
                           static_cast<uint32_t>(n),
                           dev_ptr<uint32_t>(A->row_pointer, A->off_row_pointer),
                           dev_ptr<uint32_t>(A->col_indices, A->off_col_indices),
                           dev_ptr<double>(A->values, A->off_values), invD);
    }
    // The increment starts at zero (every true residual below folds it in).
    if constexpr (kIncr) hipLaunchKernelGGL((fill_kernel<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, xd, TI(0));
    CLS_HIP_TRY(hipGetLastError());

    // Mixed: x += xd, xd = 0 (flush) or xd = 0 (discard, back to the last
    // flush point); FP64 engines update x itself.
    auto flush = [&]() -> clsparseStatus {
        if constexpr (kIncr) {
            hipLaunchKernelGGL((flush_increment<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, xp, xd);
            CLS_HIP_TRY(hipGetLastError());
        }
        return clsparseSuccess;
    };
    auto discard = [&]() -> clsparseStatus {
        if constexpr (kIncr) {
            hipLaunchKernelGGL((fill_kernel<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, xd, TI(0));
            CLS_HIP_TRY(hipGetLastError());
        }
        return clsparseSuccess;
    };
    // Back to the last replacement point after a breakdown.
    auto restore = [&]() -> clsparseStatus {
        if constexpr (kIncr)
            return discard();
        else
            CLS_HIP_TRY(hipMemcpyAsync(xp, xsave, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        return clsparseSuccess;
    };
    // x += xd; r64 = b - A x; ||r64||_2 -> hp->res; returns the true relative residual.
    auto true_residual = [&](double* rel) -> clsparseStatus {
        hipLaunchKernelGGL((flush_and_copy<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, xp, xd, bp, r64);
        CLS_HIP_TRY(hipGetLastError());
        CLS_TRY(launch_csrmv<double>(sc64, A, xp, sc64 + 1, r64, s, control->extended_precision,
                                     nullptr));
        CLS_TRY(launch_reduce<double, double>(RedOp::Sqr, r64, nullptr, n, &hp->res, true,
                                              control->red_partials, s));
        CLS_HIP_TRY(hipStreamSynchronize(s));
        *rel = hp->res / norm_b;
        return clsparseSuccess;
    };

    // (its wait also makes the checks of the diagonal storage known)
    double rel = 0.0, first_rel = 0.0;
    CLS_TRY(true_residual(&rel));
    first_rel = rel;
    DiaMatrix<TI> adia{};
    if (a_ndiag && hp->dia_bad) a_ndiag = 0;
    if (a_ndiag) adia = DiaMatrix<TI>{a_dia, a_ndiag, hp->dia_unsym == 0, a_off};

    using Engine = CgEngine<TI, std::conditional_t<kIncr, TI, double>>;
    auto* xe = [&] {
        if constexpr (kIncr)
            return xd;
        else
            return xp;
    }();
    // rI holds the inner right-hand side for each set-up only: the learned
    // factor's fused iteration may keep r in it between iterations.
    Engine eng_main(&AI, xe, rI, n, prec, kCritL2, buf, s, false, G, GT, g_bf16, have_dia ? &dia : nullptr,
                    &adia, rI, control->num_cus, control->device, &sc->launches);
    Engine eng_jac(&AI, xe, rI, n, kPrecJacobi, kCritL2, buf, s, false, nullptr, nullptr, false, nullptr,
                   &adia, nullptr, control->num_cus, control->device, &sc->launches);
    Engine* eng = &eng_main;
    // A pilot race already run for this factor decides without a new one
    // (the factor object forgets it when G changes).
    int race_known = 0;
    double known_rf = 0.0, known_rj = 0.0;
    if (fsai && prec == kPrecFsai && race_enabled()) {
        race_known = fsai_race(fsai, &known_rf, &known_rj);
        if (race_known == 2) {
            eng = &eng_jac;
            used = 3;
        }
    }

    // (Re)starts the TI loop from the current x: r = (TI)(b - A x), z = M r, p = z.
    auto restart = [&]() -> clsparseStatus {
        hipLaunchKernelGGL((rr_cast<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, r64, rI);
        CLS_HIP_TRY(hipGetLastError());
        CLS_TRY(eng->setup(true));
        hipLaunchKernelGGL(state_resume, dim3(1), dim3(64), 0, s, buf.st, &hp->res);
        CLS_HIP_TRY(hipGetLastError());
        return clsparseSuccess;
    };

    int replacements = 0;
    int detail = 1;
    int iters = 0;
    double rate_fsai_out = 0.0, rate_jac_out = 0.0;
    double loss_fsai = 0.0, loss_jac = 0.0;
    if (rel <= sc->relativeTolerance) {
        detail = 0;
    } else {
        if constexpr (!kIncr)
            CLS_HIP_TRY(hipMemcpyAsync(xsave, xp, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        // A new factor clearly ahead of Jacobi by the loss estimate is kept
        // without the pilot race (the factor keeps that outcome as a race's);
        // otherwise the race decides. The iteration buffers are free here.
        if constexpr (kMixed) {
            if (eng->prec() == kPrecFsai && race_enabled() && race_known == 0 && estimate_enabled() && have_dia &&
                adia.vals != nullptr) {
                CLS_TRY(factor_losses(dia, adia, buf.invD, n, kLossProbes, buf.z, buf.p, buf.y, buf.r, buf.part_yp,
                                      buf.part_rz[0], s, &loss_fsai, &loss_jac));
                if (std::isfinite(loss_fsai) && loss_fsai <= kLossRatioKeep * loss_jac) {
                    race_known = 1;
                    known_rf = known_rj = 0.0;  // no race was run
                    fsai_set_race(fsai, 1, 0.0, 0.0);
                }
            }
        }
        CLS_TRY(restart());
        double res_at_replace = rel;
        double best_res = rel;
        int chunks_since_best = 0;
        int iter_at_chunk = 0;
        // Pilot race of the learned factor against Jacobi: kPilotChunks chunks
        // of each from the same starting point (FSAI first; its end point is
        // kept, x goes back to the start for Jacobi); the rate
        // -ln(res_end / res_start) / seconds is measured over all chunks but
        // the first of each (which captures the graph), i.e. over the second
        // chunk of 32 iterations. The learned factor goes on from its own
        // end point unless Jacobi's rate beats it by race_margin(), then Jacobi
        // goes on from its own. (Jacobi started where FSAI stopped would
        // meet a residual whose easily damped components are already gone.)
        enum Phase { kPilotFsai, kPilotJacobi, kMain };
        Phase phase = (eng->prec() == kPrecFsai && race_enabled() && race_known == 0) ? kPilotFsai : kMain;
        if (phase == kPilotFsai)
            CLS_HIP_TRY(hipMemcpyAsync(xstart, xp, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        int phase_chunks = 0;
        double phase_res0 = 0.0, rate_fsai = 0.0, rate_jac = 0.0;
        auto phase_t0 = std::chrono::steady_clock::now();
        // Switches to engine e from the current x (true residual, restart);
        // *over is set when the solve has ended (converged or out of iterations).
        auto switch_to = [&](Engine* e, bool* over) -> clsparseStatus {
            eng = e;
            CLS_TRY(true_residual(&rel));
            *over = true;
            if (rel <= sc->relativeTolerance) {
                detail = 0;
                return clsparseSuccess;
            }
            if (iters >= sc->maxIters) return clsparseSuccess;
            *over = false;
            CLS_TRY(restart());
            res_at_replace = rel;
            best_res = rel;
            chunks_since_best = 0;
            iter_at_chunk = hs->iter;
            phase_chunks = 0;
            return clsparseSuccess;
        };
        for (;;) {
            // The pilot race counts and times single chunks.
            CLS_TRY(eng->run_chunk(hs, phase == kMain ? kMaxRun : kChunk, delta * res_at_replace, best_res));
            if (hs->failed) {  // a persistent launch gave up: from x again, in separate launches
                bool over = false;
                hs->iter = iter_at_chunk;
                hipLaunchKernelGGL(state_recover, dim3(1), dim3(64), 0, s, buf.st, 0.0, iter_at_chunk);
                CLS_HIP_TRY(hipGetLastError());
                CLS_TRY(switch_to(eng, &over));
                if (over) break;
                continue;
            }
            if (eng->persistent_fsai() && hs->best_res < best_res) {  // chunks of the launch before its last one
                best_res = hs->best_res;
                chunks_since_best = 0;
            }
            const int ran = hs->iter - iter_at_chunk;
            CLS_TRY(eng->settle_r(ran));
            iter_at_chunk = hs->iter;
            iters = hs->iter;
            const double cur = hs->cur_res;
            const bool finite = std::isfinite(cur);
            if (phase != kMain && finite && !hs->done) {
                const auto now = std::chrono::steady_clock::now();
                if (++phase_chunks == 1) {
                    phase_res0 = cur;
                    phase_t0 = now;
                } else if (phase_chunks == kPilotChunks) {
                    const double dt = std::chrono::duration<double>(now - phase_t0).count();
                    const double rate = dt > 0 ? std::log(phase_res0 / cur) / dt : 0.0;
                    bool over = false;
                    if (phase == kPilotFsai) {
                        rate_fsai = rate;
                        phase = kPilotJacobi;
                        used = 3;
                        CLS_TRY(flush());  // the learned factor's end point, whole
                        CLS_HIP_TRY(hipMemcpyAsync(xpilot, xp, n * sizeof(double), hipMemcpyDeviceToDevice, s));
                        CLS_HIP_TRY(hipMemcpyAsync(xp, xstart, n * sizeof(double), hipMemcpyDeviceToDevice, s));
                        CLS_TRY(switch_to(&eng_jac, &over));
                    } else {
                        rate_jac = rate;
                        phase = kMain;
                        const bool keep = rate_jac <= race_margin() * rate_fsai;
                        fsai_set_race(fsai, keep ? 1 : 2, rate_fsai, rate_jac);
                        if (keep) {
                            used = 2;
                            CLS_TRY(discard());  // Jacobi's progress is dropped
                            CLS_HIP_TRY(hipMemcpyAsync(xp, xpilot, n * sizeof(double), hipMemcpyDeviceToDevice, s));
                            CLS_TRY(switch_to(&eng_main, &over));
                        }
                    }
                    if (over) break;
                    continue;
                }
            } else if (phase != kMain && !finite) {
                phase = kMain;  // the stagnation / breakdown rule below takes over
            }
            // Breakdown or stagnation of the learned preconditioner: back to
            // the last saved x and on with Jacobi.
            if (eng->prec() == kPrecFsai) {
                if (finite && cur < 0.5 * best_res) {
                    best_res = cur;
                    chunks_since_best = 0;
                } else {
                    ++chunks_since_best;
                }
                if (!finite || chunks_since_best >= kStagnationChunks) {
                    if (!finite) CLS_TRY(restore());
                    used = 3;
                    phase = kMain;
                    bool over = false;
                    CLS_TRY(switch_to(&eng_jac, &over));
                    if (over) break;
                    continue;
                }
            }
            if (!finite) {  // Jacobi or none broke down: stop at the last replacement point
                CLS_TRY(restore());
                break;
            }
            const bool out_of_iters = hs->done && !hs->converged;
            if (!hs->done && cur > delta * res_at_replace) continue;

            // Residual replacement (or the final check).
            CLS_TRY(true_residual(&rel));
            ++replacements;
            if (rel <= sc->relativeTolerance) {
                detail = 0;
                break;
            }
            if (out_of_iters || iters >= sc->maxIters) break;
            if constexpr (!kIncr)
                CLS_HIP_TRY(hipMemcpyAsync(xsave, xp, n * sizeof(double), hipMemcpyDeviceToDevice, s));
            // r = (TI) r64; z' = M r into y; <r, z'> partials -> part_yp;
            // re-base p and z; the new <r, z> becomes the previous one.
            CLS_TRY(eng->materialize_p(ran));
            CLS_TRY(eng->materialize_z(rI));
            const uint32_t g = grid_for(n);
            // Sets of partials: the last executed iteration of the chunk wrote
            // <r, z> to part_rz[(ran - 1) & 1].
            const double* old_part = buf.part_rz[(ran - 1) & 1];
            if (eng->prec() == kPrecFsai) {
                hipLaunchKernelGGL((rr_cast<TI>), dim3(ew_grid(n)), dim3(256), 0, s, n, r64, buf.r);
                CLS_HIP_TRY(hipGetLastError());
                CLS_TRY(eng->precondition(buf.y, rI));
                // cg_dot_kernel is a no-op once done is set: clear it first.
                hipLaunchKernelGGL(state_resume, dim3(1), dim3(64), 0, s, buf.st, &hp->res);
                hipLaunchKernelGGL((cg_dot_kernel<TI>), dim3(g), dim3(256), 0, s, n, buf.r, buf.y,
                                   buf.part_yp, buf.st);
            } else {
                hipLaunchKernelGGL((rr_precondition<TI>), dim3(g), dim3(256), 0, s, n, r64, buf.r, buf.y, buf.invD,
                                   eng->prec(), buf.part_yp, buf.st, &hp->res);
            }
            hipLaunchKernelGGL((rr_rebase<TI>), dim3(g), dim3(256), 0, s, n, buf.p, buf.z, buf.y,
                               old_part, buf.part_yp, g, eng->fused() ? 1 : 0);
            hipLaunchKernelGGL(copy_partials, dim3(1), dim3(256), 0, s, buf.part_yp, buf.part_rz[1], g);
            CLS_HIP_TRY(hipGetLastError());
            res_at_replace = rel;
        }
        rate_fsai_out = race_known ? known_rf : rate_fsai;
        rate_jac_out = race_known ? known_rj : rate_jac;
    }
    CLS_TRY(leave_solver_stream(control));
    const auto t1 = std::chrono::steady_clock::now();
    sc->nIters = iters;
    sc->initialResidual = first_rel;
    sc->currentResidual = rel;
    sc->stats.iterations = iters;
    sc->stats.outer_iterations = replacements;
    sc->stats.true_residual = rel;
    sc->stats.seconds = std::chrono::duration<double>(t1 - t0).count();
    sc->stats.status_detail = detail;
    sc->stats.preconditioner = used;
    sc->stats.pilot_rate_fsai = rate_fsai_out;
    sc->stats.pilot_rate_jacobi = rate_jac_out;
    sc->stats.loss_fsai = loss_fsai;
    sc->stats.loss_jacobi = loss_jac;
    sc->stats.a_diagonals = a_ndiag;
    sc->stats.g_diagonals = have_dia ? dia.ndiag : 0;
    return clsparseSuccess;
}

}  // namespace

extern "C" clsparseStatus clsparseAmdDcsrcgMixed(cldenseVector* x, const clsparseCsrMatrix* A,
                                                 const cldenseVector* b,
                                                 clSParseSolverControl sc,
                                                 clsparseControl control)
{
    if (mixed_x64()) return reliable_solve<float, true>(x, A, b, sc, control);
    return reliable_solve<float>(x, A, b, sc, control);
}

extern "C" clsparseStatus clsparseAmdDcsrcgRefined(cldenseVector* x, const clsparseCsrMatrix* A,
                                                   const cldenseVector* b,
                                                   clSParseSolverControl sc,
                                                   clsparseControl control)
{
    return reliable_solve<double>(x, A, b, sc, control);
}

extern "C" clsparseStatus clsparseAmdDcsrcgFsai(cldenseVector* x, const clsparseCsrMatrix* A,
                                                const cldenseVector* b, clsparseAmdFsai fsai,
                                                clSParseSolverControl sc, clsparseControl control)
{
    if (fsai == nullptr) return clsparseInvalidValue;
    if (mixed_x64()) return reliable_solve<float, true>(x, A, b, sc, control, fsai);
    return reliable_solve<float>(x, A, b, sc, control, fsai);
}

extern "C" clsparseStatus clsparseAmdDcsrcgFsai64(cldenseVector* x, const clsparseCsrMatrix* A,
                                                  const cldenseVector* b, clsparseAmdFsai fsai,
                                                  clSParseSolverControl sc, clsparseControl control)
{
    if (fsai == nullptr) return clsparseInvalidValue;
    return reliable_solve<double>(x, A, b, sc, control, fsai);
}
