// CG iterations of a stencil matrix in one cooperative launch.
//
// The launch-per-step iteration (cg.hip) moves every vector through memory in
// each of its two or three kernels and pays a kernel boundary for each. Here
// one workgroup per CU stays resident for the whole run: every thread owns R
// rows and keeps x, r and 1/diagonal of them in registers (p in registers or
// LDS), so an iteration moves A (not even that when the rows are few: A stays
// in registers too) and the p that workgroups read of each other. The
// recurrence, the products and the order of a row's sum are those of cg.hip;
// the dot products are added in another (also fixed) order.
//
// One iteration: the operands into LDS; y = A p with <y, p>; grid sum; alpha,
// x, r, z = M r with <r, z> and ||r||; grid sum; the convergence test (every
// workgroup forms the same decision from the same sums). p = z + beta p is
// published after that for the next iteration, with a third grid barrier; or
// (TWO, few rows per thread) z is published before the second sum and every
// workgroup forms p = z + beta p of the rows that it reads itself: one barrier
// fewer, but two values read and written per shared row.
//
// Per iteration against the launch-per-step kernels (whose bytes, launches and
// gaps it saves): FP64 Jacobi 93 x 101 Poisson 17.0 -> 4.7 us, 40^3 21.6 -> 6.0,
// 64^3 21.2 -> 6.9, 100^3 35.1 -> 15.4, 128^3 57.2 -> 23.1 us; FP32 64^3 18.0 ->
// 6.9, 160^3 57.4 -> 32 us. What is left of a small iteration is the two grid
// sums (1.5-2 us each) and a memory latency for the operands; at 128^3 it
// streams A (67 MB) and the shared p at about 4.5 TB/s beside three barriers.
#pragma once

#include <algorithm>
#include <cstdlib>

#include "cg_persist.hpp"
#include "persist_tile.hpp"

namespace {

template <typename T>
__device__ __forceinline__ double abs_term(int crit, T r)
{
    const double d = static_cast<double>(r);
    return crit == kCritL2 ? d * d : fabs(d);
}

// AREG: the thread's K R values of A stay in registers (SYM is then only how
// they are read in); else A is read from memory in every iteration, in half
// storage if SYM.
template <int K, bool SYM, typename T, int R, bool AREG, bool TWO, bool LINE>
__global__ __launch_bounds__(kGridThreads) void cg_persist_kernel(CgPersistArgs<T> a)
{
    constexpr uint32_t S = sizeof(T);
    constexpr bool PREG = R * S < 64;  // p in registers beside the tile
    constexpr int N = R == 4 && !LINE ? 12 : 8;  // tile copies in flight per thread
    extern __shared__ __align__(16) char tile_bytes[];
    __shared__ GridShared sh;
    T* const tile = reinterpret_cast<T*>(tile_bytes);
    CgDevState* st = a.st;
    if (st->done) return;
    const PersistPlan& pl = a.plan;
    const uint32_t n = a.n, nd = pl.ndiag;
    const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t first = persist_first_row(pl, wg);
    const uint32_t tid = threadIdx.x;
    const uint32_t live_threads = LINE ? persist_live_threads(pl, wg) : kGridThreads;
    const bool mine = tid < live_threads;
    uint32_t step = LINE ? pl.row_step : kGridThreads;
    uint32_t tstep = LINE ? pl.tile_step : kGridThreads;

    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.vals), 0, nd * n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rz_ = __builtin_amdgcn_make_buffer_rsrc(a.z, 0, n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rp0 = __builtin_amdgcn_make_buffer_rsrc(a.p, 0, n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rp1 = __builtin_amdgcn_make_buffer_rsrc(a.p2, 0, n * S, 0x00020000);
    const uint32_t dead = LINE ? persist_dead_bits(mine) : 0u;
    auto row_of = [&](uint32_t t, int k) { return (first + t + k * step) | dead; };
    const StencilValues<K, T> values{rv, n, nd, pl};

    T x[R], r[R], p[PREG ? R : 1], z[TWO ? R : 1], m[R];
    T v[AREG ? R : 1][K];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t i = row_of(tid, k);
        const bool live = i < n;
        x[k] = live ? a.x[i] : T(0);
        const T pi = live ? a.p[i] : T(0);
        if constexpr (PREG) p[k] = pi;
        tile[pl.own + k * tstep + tid] = pi;
        r[k] = live ? a.r[i] : T(0);
        m[k] = (live && a.invD != nullptr) ? a.invD[i] : T(1);
        if constexpr (TWO) z[k] = pi;
        if constexpr (AREG) {
#pragma unroll
            for (int d = 0; d < K; ++d) v[k][d] = values(i, d, a.sym != 0);
        }
    }
    // <r, z> of the state handed over: the same sum of the same partials in
    // every workgroup.
    double rz = 0.0;
    {
        double s = 0.0;
        for (uint32_t i = tid; i < a.g_in; i += kGridThreads) s += a.rz_in[i];
        s = wave_sum(s);
        if ((tid & 63) == 0) sh.w[tid >> 6][0] = s;
        __syncthreads();
#pragma unroll
        for (uint32_t w = 0; w < kGridWaves; ++w) rz += sh.w[w][0];
        __syncthreads();
    }
    FillSlots<LINE ? 1 : N> where;
    if constexpr (!LINE) {
        where.find(pl, first, tid);
    }
    const bool shared = gridDim.x > 1;  // some other workgroup reads this one's rows
    const double norm_ref = st->norm_ref, rel_tol = st->rel_tol, abs_stop = st->abs_tol * st->init_res;
    const int max_iters = st->max_iters, crit = st->crit;
    int iter = st->iter;
    uint32_t epoch = st->epoch;
    double res = st->cur_res;
    bool conv = false, done = false, ok = true;
    double sums[2];
    T beta = T(0);
    for (int ran = 0;;) {
        // Opaque, anew for every step: keeps the address arithmetic with it (kept
        // across, it takes more registers than the rows themselves), and the tests of A's
        // values in registers for 0 (their masks more scalar ones than there are).
        uint32_t t = tid;
        auto anew = [&] {
            asm volatile("" : "+v"(t));
            if constexpr (LINE) asm volatile("" : "+s"(step), "+s"(tstep));
        };
        anew();
        if constexpr (AREG) {
#pragma unroll
            for (int k = 0; k < R; ++k)
#pragma unroll
                for (int d = 0; d < K; ++d) asm volatile("" : "+v"(v[k][d]));
        }
        // The operands. TWO: p = z + beta p; in the first iteration of a
        // launch p is whole in a.p.
        if constexpr (TWO) {
            const bool whole = ran == 0;
            T g0[N], g1[N];
            fill_tile<R, LINE, N>(
                pl, first, t, live_threads, where,
                [&](uint32_t j, int u) {
                    g0[u] = load_shared<T>(whole ? rp0 : rz_, j, n);
                    g1[u] = load_shared<T>((ran & 1) ? rp1 : rp0, j, n);
                },
                [&](uint32_t at, int u) { tile[at] = whole ? g0[u] : fma(beta, g1[u], g0[u]); });
            T* pout = (ran & 1) ? a.p : a.p2;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t at = pl.own + k * tstep + t, i = row_of(t, k);
                const T pk = PREG ? p[PREG ? k : 0] : tile[at];
                const T pn = whole ? pk : fma(beta, pk, z[k]);
                if constexpr (PREG) p[k] = pn;
                if (mine) tile[at] = pn;
                if (shared && i < n) store_shared(pout + i, pn);
            }
        } else {
            T g0[N];
            fill_tile<R, LINE, N>(
                pl, first, t, live_threads, where, [&](uint32_t j, int u) { g0[u] = load_shared<T>(rp0, j, n); },
                [&](uint32_t at, int u) { tile[at] = g0[u]; });
        }
        __syncthreads();
        // y = A p, <y, p>
        T y[R];
        double yp = 0.0;
        constexpr int U = persist_group<T, R>();
#pragma unroll
        for (int k0 = 0; k0 < R; k0 += U) {
            anew();
            T av[U][K];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int d = 0; d < K; ++d) av[u][d] = AREG ? v[AREG ? k0 + u : 0][d] : values(row_of(t, k0 + u), d, SYM);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t at = pl.own + (k0 + u) * tstep + t;
                double sum = 0.0;  // FP32 products summed in FP64, as the CSR SpMV sums them
#pragma unroll
                for (int d = 0; d < K; ++d) {
                    const T pj = tile[at + static_cast<uint32_t>(pl.delta[d])];
                    sum += stencil_term(av[u][d], pj);
                }
                y[k0 + u] = static_cast<T>(sum);
                yp += static_cast<double>(y[k0 + u]) * static_cast<double>(tile[at]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        sums[0] = yp;
        if (!(ok = grid_sum<1>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        anew();
        const T alpha = static_cast<T>(rz / sums[0]);
        double rzn = 0.0, nr = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const T pk = PREG ? p[PREG ? k : 0] : tile[pl.own + k * tstep + t];
            x[k] = x[k] + alpha * pk;
            r[k] = r[k] - alpha * y[k];
            nr += abs_term(crit, r[k]);
            const T zk = r[k] * m[k];
            rzn += static_cast<double>(r[k]) * static_cast<double>(zk);
            if constexpr (TWO) {
                z[k] = zk;
                const uint32_t i = row_of(t, k);
                if (shared && i < n) store_shared(a.z + i, zk);
            }
        }
        sums[0] = rzn;
        sums[1] = nr;
        if (!(ok = grid_sum<2>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        beta = static_cast<T>(sums[0] / rz);
        rz = sums[0];
        res = (crit == kCritL2 ? sqrt(sums[1]) : sums[1]) / norm_ref;
        conv = res <= rel_tol || res <= abs_stop;
        done = conv || iter >= max_iters;
        if (wg == 0 && tid == 0) st->hist[iter % kHist] = res;
        ++iter;
        ++ran;
        const bool end = done || ran >= a.max_run || (ran % kChunk == 0 && !(res > a.go_on && res <= 1e300));
        anew();
        if constexpr (!TWO) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t at = pl.own + k * tstep + t, i = row_of(t, k);
                const T pn = fma(beta, PREG ? p[PREG ? k : 0] : tile[at], r[k] * m[k]);
                if constexpr (PREG) p[k] = pn;
                if (mine) tile[at] = pn;
                if (shared && i < n) store_shared(a.p + i, pn);
            }
        }
        if (end) break;
        if constexpr (!TWO)
            if (!(ok = grid_sum<0>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
    }
    if (!ok) {
        if (tid == 0) st->failed = 1;
        return;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t i = row_of(tid, k);
        if (i < n) {
            const T zk = r[k] * m[k];
            a.x[i] = x[k];
            a.r[i] = r[k];
            a.z[i] = zk;
            const T pk = PREG ? p[PREG ? k : 0] : tile[pl.own + k * tstep + tid];
            a.p[i] = TWO ? fma(beta, pk, zk) : pk;
        }
    }
    // The state as the launch-per-step kernels leave it: <r, z> as the first
    // of g_in partials, in both sets.
    if (wg == 0) {
        for (uint32_t i = tid; i < a.g_in; i += kGridThreads) {
            a.rz_out[0][i] = i == 0 ? rz : 0.0;
            a.rz_out[1][i] = i == 0 ? rz : 0.0;
        }
        if (tid == 0) {
            st->cur_res = res;
            st->iter = iter;
            st->epoch = epoch;
            if (done) {
                st->done = 1;
                st->n_iters = iter - 1;
                st->converged = conv ? 1 : 0;
            }
        }
    }
}

// A stays in registers while a thread's values take at most this many
// (7 diagonals, 8 FP64 rows: 112; read from memory instead, a 100^3 iteration
// takes 17.9 instead of 16.5 us, and 16 FP32 rows at 128^3 24.5 instead of 22.8).
constexpr int kAregMax = 112;
template <int K, typename T, int R>
constexpr bool areg()
{
    return K * R * static_cast<int>(sizeof(T) / 4) <= kAregMax;
}

template <int K, bool SYM, typename T, int R, bool LINE>
hipError_t launch(CgPersistArgs<T>& a, hipStream_t s)
{
    constexpr bool kAreg = areg<K, T, R>();
    auto* f = &cg_persist_kernel<K, SYM && !kAreg, T, R, kAreg, R <= 4, LINE>;
    const size_t lds = a.plan.tile_size * sizeof(T);
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(f),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kPersistLds);
    if (e != hipSuccess) return e;
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(f), dim3(a.plan.wgs), dim3(kGridThreads), args,
                                      static_cast<uint32_t>(lds), s);
}

template <int K, typename T, int R, bool LINE>
hipError_t launch_sym(CgPersistArgs<T>& a, hipStream_t s)
{
    // Half storage needs the diagonal's exact count (odd, mirrored).
    if (a.sym && a.plan.ndiag == K) return launch<K, true, T, R, LINE>(a, s);
    a.sym = 0;
    return launch<K, false, T, R, LINE>(a, s);
}

template <int K, typename T>
hipError_t launch_rows(CgPersistArgs<T>& a, hipStream_t s)
{
    const bool lines = a.plan.line != 0;
    switch (a.plan.rows) {
    case 1: return launch_sym<K, T, 1, false>(a, s);
    case 2: return launch_sym<K, T, 2, false>(a, s);
    case 4: return lines ? launch_sym<K, T, 4, true>(a, s) : launch_sym<K, T, 4, false>(a, s);
    case 8: return lines ? launch_sym<K, T, 8, true>(a, s) : launch_sym<K, T, 8, false>(a, s);
    case 16: return lines ? launch_sym<K, T, 16, true>(a, s) : launch_sym<K, T, 16, false>(a, s);
    default: break;
    }
    if constexpr (sizeof(T) == 4)
        if (a.plan.rows == 32 && lines) return launch_sym<K, T, 32, true>(a, s);
    return hipErrorInvalidValue;
}

}  // namespace

template <typename T>
clsparseStatus launch_cg_persist(CgPersistArgs<T> a, hipStream_t s)
{
    if (a.plan.rows == 0) return clsparseInvalidValue;
    // Even counts take the next odd kernel (the missing diagonal reads 0).
    hipError_t e = hipErrorInvalidValue;
    if (a.plan.ndiag <= 3) e = launch_rows<3, T>(a, s);
    else if (a.plan.ndiag <= 5) e = launch_rows<5, T>(a, s);
    else if (a.plan.ndiag <= 7) e = launch_rows<7, T>(a, s);
    else if (a.plan.ndiag <= 9) e = launch_rows<9, T>(a, s);
    // (refused, for instance while another process runs cooperative launches: the
    // caller goes on without, and without a word)
    return e == hipSuccess ? clsparseSuccess : clsparseInvalidKernelExecution;
}
