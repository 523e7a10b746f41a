// BiCGStab iterations of a stencil matrix in one cooperative launch: the
// recurrence and checks of bicgstab.hip with a thread's rows of x, r, r*, p,
// A M p and 1/diagonal in registers (see cg_persist_kernel.hpp for the layout
// and what bounds it). s takes r's registers, and M p and M s are formed again
// where they are needed, so two vectors a row move between workgroups, and A.
//
// One iteration: M p into the tiles; v = A M p, <r*, v>; sum; s, M s
// published, ||s||; sum; first check; M s into the tiles; t = A M s, <t, s>,
// <t, t>; sum; x, r, ||r||, <r*, r>; sum; second check; p, M p published;
// barrier. Five grid-wide sums against five to seven kernels.
//
// FP64 Jacobi, convection-diffusion, per iteration against the launch-per-step
// kernels: 12^3 45.7 -> 15 us (solve set-up included in both), 40^3 44 -> 13.1,
// 64^3 45 -> 15.6, 96^3 71 -> 24 us (32 while it streamed the seven diagonals
// twice, 99 MB; six of them now stay on the chip).
#pragma once

#include "bicg_persist.hpp"
#include "persist_tile.hpp"

namespace {

// REGS, KEPT: so many of the thread's diagonals of A stay in registers, the next
// KEPT in LDS behind the tile; the rest is read for every product. (SYM: in half
// storage; REGS = K: SYM is then only how they are read in.)
template <int K, bool SYM, typename T, int R, int REGS, int KEPT, bool LINE>
__global__ __launch_bounds__(kGridThreads) void bicg_persist_kernel(BiPersistArgs<T> a)
{
    constexpr uint32_t S = sizeof(T);
    constexpr int N = LINE ? line_slots<R>() : R == 4 ? 12 : 8;  // tile copies in flight per thread
    extern __shared__ __align__(16) char tile_bytes[];
    __shared__ GridShared sh;
    T* const tile = reinterpret_cast<T*>(tile_bytes);
    BiDevState* st = a.st;
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
    const bool shared = gridDim.x > 1;

    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.vals), 0, nd * n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rMp = __builtin_amdgcn_make_buffer_rsrc(a.Mp, 0, n * S, 0x00020000);
    const __amdgpu_buffer_rsrc_t rMs = __builtin_amdgcn_make_buffer_rsrc(a.Ms, 0, n * S, 0x00020000);
    const uint32_t dead = LINE ? persist_dead_bits(mine) : 0u;
    auto row_of = [&](uint32_t t, int k) { return (first + t + k * step) | dead; };
    const StencilValues<K, T> values{rv, n, nd, pl};

    T x[R], r[R], rs[R], p[R], m[R];
    T v[REGS > 0 ? R : 1][REGS > 0 ? REGS : 1];
    T* const kept = tile + pl.tile_size;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t i = row_of(tid, k);
        const bool live = i < n;
        x[k] = live ? a.x[i] : T(0);
        r[k] = live ? a.r[i] : T(0);
        rs[k] = live ? a.rs[i] : T(0);
        p[k] = live ? a.p[i] : T(0);
        m[k] = (live && a.invD != nullptr) ? a.invD[i] : T(1);
        if (mine) tile[pl.own + k * tstep + tid] = p[k] * m[k];
#pragma unroll
        for (int d = 0; d < REGS; ++d) v[k][d] = values(i, d, REGS == K ? a.sym != 0 : SYM);
#pragma unroll
        for (int d = 0; d < KEPT; ++d) kept[(d * R + k) * kGridThreads + tid] = values(i, REGS + d, SYM);
    }
    double rr = 0.0;  // <r*, r> handed over: the same sum in every workgroup
    {
        double s = 0.0;
        for (uint32_t i = tid; i < a.g_in; i += kGridThreads) s += a.rr[i];
        s = wave_sum(s);
        if ((tid & 63) == 0) sh.w[tid >> 6][0] = s;
        __syncthreads();
#pragma unroll
        for (uint32_t w = 0; w < kGridWaves; ++w) rr += sh.w[w][0];
        __syncthreads();
    }
    FillSlots<LINE ? 1 : N> where;
    if constexpr (!LINE) where.find(pl, first, tid);
    const double norm_b = st->norm_b;
    int iter = st->iter, stop = 0;
    uint32_t epoch = st->epoch;
    double res = st->cur_res;
    bool ok = true;
    double sums[2];
    // Opaque, anew for every step: keeps the address arithmetic with it, and the
    // tests of A's values in registers for 0 inside the loop.
    // out = A (tile) with <out, w> and, for the second product, <out, out>.
    uint32_t t = tid;
    auto anew = [&] {
        asm volatile("" : "+v"(t));
        if constexpr (LINE) asm volatile("" : "+s"(step), "+s"(tstep));
    };
    auto product = [&](T (&out)[R], const T (&w)[R], double& ow, double& oo) {
        constexpr int U = persist_group<T, R>();
#pragma unroll
        for (int k = 0; k < (REGS > 0 ? R : 0); ++k)
#pragma unroll
            for (int d = 0; d < REGS; ++d) asm volatile("" : "+v"(v[k][d]));
#pragma unroll
        for (int k0 = 0; k0 < R; k0 += U) {
            anew();
            T av[U][K];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int d = 0; d < K; ++d) {
                    if (d < REGS) av[u][d] = v[REGS > 0 ? k0 + u : 0][d < REGS ? d : 0];
                    else if (d < REGS + KEPT) av[u][d] = kept[((d - REGS) * R + k0 + u) * kGridThreads + t];
                    else av[u][d] = values(row_of(t, k0 + u), d, SYM);
                }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t at = pl.own + (k0 + u) * tstep + t;
                double sum = 0.0;  // FP32 products summed in FP64, as the CSR SpMV sums them
#pragma unroll
                for (int d = 0; d < K; ++d) {
                    const T pj = tile[at + static_cast<uint32_t>(pl.delta[d])];
                    sum += stencil_term(av[u][d], pj);
                }
                out[k0 + u] = static_cast<T>(sum);
                ow += static_cast<double>(out[k0 + u]) * static_cast<double>(w[k0 + u]);
                oo += static_cast<double>(out[k0 + u]) * static_cast<double>(out[k0 + u]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int ran = 0;;) {
        anew();
        T Av[R], At[R];  // A M p, A M s
        T g0[N];
        fill_tile<R, LINE, N>(
            pl, first, t, live_threads, where, [&](uint32_t j, int u) { g0[u] = load_shared<T>(rMp, j, n); },
            [&](uint32_t at, int u) { tile[at] = g0[u]; });
        __syncthreads();
        double ra = 0.0, unused = 0.0;
        product(Av, rs, ra, unused);
        sums[0] = ra;
        if (!(ok = grid_sum<1>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        anew();
        const T alpha = static_cast<T>(rr / sums[0]);
        double ns = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t i = row_of(t, k);
            r[k] = r[k] - alpha * Av[k];  // s
            const T ms = r[k] * m[k];
            if (mine) tile[pl.own + k * tstep + t] = ms;
            if (shared && i < n) store_shared(a.Ms + i, ms);
            ns += fabs(static_cast<double>(r[k]));
        }
        sums[0] = ns;
        if (!(ok = grid_sum<1>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        res = sums[0] / norm_b;
        if (bi_finished(st, res, iter)) {
            stop = 1;
#pragma unroll
            for (int k = 0; k < R; ++k) x[k] = x[k] + alpha * (p[k] * m[k]);
            break;
        }
        anew();
        fill_tile<R, LINE, N>(
            pl, first, t, live_threads, where, [&](uint32_t j, int u) { g0[u] = load_shared<T>(rMs, j, n); },
            [&](uint32_t at, int u) { tile[at] = g0[u]; });
        __syncthreads();
        double us = 0.0, ww = 0.0;
        product(At, r, us, ww);
        sums[0] = us;
        sums[1] = ww;
        if (!(ok = grid_sum<2>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        anew();
        const T omega = static_cast<T>(sums[0] / sums[1]);
        double nr = 0.0, rrn = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            T xi = x[k] + alpha * (p[k] * m[k]);
            x[k] = xi + omega * (r[k] * m[k]);
            r[k] = r[k] - omega * At[k];
            nr += fabs(static_cast<double>(r[k]));
            rrn += static_cast<double>(rs[k]) * static_cast<double>(r[k]);
        }
        sums[0] = rrn;
        sums[1] = nr;
        if (!(ok = grid_sum<2>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        T beta = static_cast<T>(sums[0] / rr);
        beta = beta * alpha;
        beta = beta / omega;
        const T bo = beta * omega;
        rr = sums[0];
        res = sums[1] / norm_b;
        anew();
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t i = row_of(t, k);
            const T pi = beta * p[k] + r[k];
            p[k] = pi - bo * Av[k];
            const T mp = p[k] * m[k];
            if (mine) tile[pl.own + k * tstep + t] = mp;
            if (shared && i < n) store_shared(a.Mp + i, mp);
        }
        if (bi_finished(st, res, iter)) {
            stop = 2;
            break;
        }
        ++iter;
        if (++ran >= a.max_run) break;
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
            a.x[i] = x[k];
            a.r[i] = r[k];
            a.p[i] = p[k];
            a.Mp[i] = p[k] * m[k];
        }
    }
    if (wg == 0) {
        for (uint32_t i = tid; i < a.g_in; i += kGridThreads) a.rr[i] = i == 0 ? rr : 0.0;
        if (tid == 0) {
            st->cur_res = res;
            st->iter = iter;
            st->epoch = epoch;
            if (stop) {
                st->done = 1;
                st->stop_kind = stop;
                st->n_iters = iter;
                st->converged = (res <= st->rel_tol || res <= st->abs_tol * st->init_res) ? 1 : 0;
            }
        }
    }
}

// A stays in registers while a thread's values take at most this many (the
// vectors take 14 per FP64 row).
constexpr int kBiAregMax = 60;

// Beyond that, three diagonals in LDS where the tile leaves room for them, and of
// a plan by lines (whose kernel has registers left) this many in registers:
// 96^3 32.0 -> 24.1 us an iteration.
template <typename T>
constexpr int kBiRegs = sizeof(T) == 8 ? 3 : 1;
constexpr int kBiKept = 3;

template <int K, bool SYM, typename T, int R, int REGS, int KEPT, bool LINE>
hipError_t launch_bi_kernel(BiPersistArgs<T>& a, hipStream_t s)
{
    auto* f = &bicg_persist_kernel<K, SYM, T, R, REGS, KEPT, LINE>;
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(f),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kPersistLds);
    if (e != hipSuccess) return e;
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(f), dim3(a.plan.wgs), dim3(kGridThreads), args,
                                      static_cast<uint32_t>((a.plan.tile_size + KEPT * R * kGridThreads) * sizeof(T)), s);
}

template <int K, bool SYM, typename T, int R, bool LINE>
hipError_t launch_bi(BiPersistArgs<T>& a, hipStream_t s)
{
    constexpr bool kAll = K * R * static_cast<int>(sizeof(T) / 4) <= kBiAregMax;
    if constexpr (kAll) return launch_bi_kernel<K, false, T, R, K, 0, LINE>(a, s);
    else {
        constexpr int kRegs = LINE ? std::min(kBiRegs<T>, K - kBiKept) : 0;
        if ((a.plan.tile_size + kBiKept * R * kGridThreads) * sizeof(T) <= kPersistLds) {
            // (what is left is read in full storage: one or a few diagonals)
            return launch_bi_kernel<K, false, T, R, kRegs, kBiKept, LINE>(a, s);
        }
        return launch_bi_kernel<K, SYM, T, R, 0, 0, LINE>(a, s);
    }
}

template <int K, typename T, int R, bool LINE>
hipError_t launch_bi_sym(BiPersistArgs<T>& a, hipStream_t s)
{
    // Half storage needs the diagonal's exact count (odd, mirrored).
    if (a.sym && a.plan.ndiag == K) return launch_bi<K, true, T, R, LINE>(a, s);
    a.sym = 0;
    return launch_bi<K, false, T, R, LINE>(a, s);
}

template <int K, typename T>
hipError_t launch_bi_rows(BiPersistArgs<T>& a, hipStream_t s)
{
    const bool lines = a.plan.line != 0;
    switch (a.plan.rows) {
    case 1: return launch_bi_sym<K, T, 1, false>(a, s);
    case 2: return launch_bi_sym<K, T, 2, false>(a, s);
    case 4: return lines ? launch_bi_sym<K, T, 4, true>(a, s) : launch_bi_sym<K, T, 4, false>(a, s);
    case 8: return lines ? launch_bi_sym<K, T, 8, true>(a, s) : launch_bi_sym<K, T, 8, false>(a, s);
    default: break;
    }
    if constexpr (sizeof(T) == 4)
        if (a.plan.rows == 16)
            return lines ? launch_bi_sym<K, T, 16, true>(a, s) : launch_bi_sym<K, T, 16, false>(a, s);
    return hipErrorInvalidValue;
}

}  // namespace

template <typename T>
clsparseStatus launch_bicg_persist(BiPersistArgs<T> a, hipStream_t s)
{
    if (a.plan.rows == 0) return clsparseInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    if (a.plan.ndiag <= 3) e = launch_bi_rows<3, T>(a, s);
    else if (a.plan.ndiag <= 5) e = launch_bi_rows<5, T>(a, s);
    else if (a.plan.ndiag <= 7) e = launch_bi_rows<7, T>(a, s);
    else if (a.plan.ndiag <= 9) e = launch_bi_rows<9, T>(a, s);
    // (refused, for instance while another process runs cooperative launches: the
    // caller goes on without, and without a word)
    return e == hipSuccess ? clsparseSuccess : clsparseInvalidKernelExecution;
}
