// Learned-FSAI CG iterations of a stencil matrix in one cooperative launch.
//
// As cg_persist_kernel.hpp: one workgroup per CU stays resident, a thread keeps
// x, r and p of its R rows in registers (A and G too when the rows are few),
// and the products and the order of a row's sum are those of the launch-per-
// step kernels (cg.hip). One LDS tile holds in turn what the three products
// read: p and y = A p, <y, p>, grid sum; r and w = G^T r with ||w||^2 = <r, z>
// and ||r||, grid sum; w and z = G w, p = z + beta p, grid barrier. G^T reads
// rows above the workgroup's and G rows below it only, so those fills copy one
// side. r of other workgroups' rows is formed from their last r and y, as the
// owner forms it: a barrier between the r update and G^T r would cost 2 us.
//
// Per iteration against the launch-per-step kernels: 30 x 40 x 28 24.1 -> 13.2
// us, 64^3 23.3 -> 13.6, 100 x 90 x 110 31.4 -> 22.2, 120^3 40.7 -> 27.5, 128^3
// 41.9 -> 28.4 (the solver's residual replacements included: 1-3 us). What is
// left is three grid sums and three fills (store, barrier, load: 3 us each) and
// with 16 rows the rest of A from memory.
#include "dia.hpp"
#include "fsai_persist.hpp"
#include "persist_tile.hpp"

namespace {

__device__ __forceinline__ float bf16_low(uint32_t two) { return __uint_as_float(two << 16); }
__device__ __forceinline__ float bf16_high(uint32_t two) { return __uint_as_float(two & 0xFFFF0000u); }

// The KG values of G's (or G^T's) row i, two to a register; 0 outside.
template <int KG>
struct FactorRow
{
    uint32_t two[(KG + 1) / 2];
    __device__ __forceinline__ float operator[](int d) const { return (d & 1) ? bf16_high(two[d / 2]) : bf16_low(two[d / 2]); }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t n, const PersistPlan& pl, uint32_t i, bool transposed)
    {
        uint32_t h[KG + 1];
        h[KG] = 0;
#pragma unroll
        for (int d = 0; d < KG; ++d) {
            const uint32_t j = transposed ? i - static_cast<uint32_t>(pl.off[d]) : i;
            h[d] = __builtin_amdgcn_raw_buffer_load_b16(rs, i < n && j < n ? (d * n + j) * 2 : 0xFFFFFFFFu, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < (KG + 1) / 2; ++q) two[q] = h[2 * q] | h[2 * q + 1] << 16;
    }
};

// Place of diagonal d of K among those that stay on the chip: the main one, then
// a lower one and its mirror image, which are read from the same memory.
template <int K>
constexpr int place(int d)
{
    return d == K / 2 ? 0 : d < K / 2 ? 1 + 2 * d : 2 * (K - d);
}

// REGS, KEPT: so many diagonals of A stay in registers, the next KEPT in LDS
// behind the tile; the rest is read in every iteration (SYM: in half storage). G
// and G^T stay in registers.
template <int K, bool SYM, int R, int REGS, int KEPT, bool LINE>
__global__ __launch_bounds__(kGridThreads) void fsai_persist_kernel(FsaiPersistArgs a)
{
    constexpr int KG = (K + 1) / 2;
    constexpr int N = LINE ? line_slots<R>() : R == 4 ? 12 : 8;  // tile copies in flight per thread
    extern __shared__ __align__(16) char tile_bytes[];
    __shared__ GridShared sh;
    float* const tile = reinterpret_cast<float*>(tile_bytes);
    CgDevState* st = a.st;
    if (st->done) return;
    const PersistPlan& pl = a.plan;
    const uint32_t n = a.n;
    const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t first = persist_first_row(pl, wg);
    const uint32_t tid = threadIdx.x;
    const uint32_t live_threads = LINE ? persist_live_threads(pl, wg) : kGridThreads;
    const bool mine = tid < live_threads;
    uint32_t step = LINE ? pl.row_step : kGridThreads;
    uint32_t tstep = LINE ? pl.tile_step : kGridThreads;
    auto buffer = [&](const void* q, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(q), 0, bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rv = buffer(a.vals, K * n * 4), rg = buffer(a.g, KG * n * 2);
    const __amdgpu_buffer_rsrc_t rp = buffer(a.p, n * 4), rr = buffer(a.r, n * 4);
    const __amdgpu_buffer_rsrc_t ry = buffer(a.y, n * 4), rw = buffer(a.w, n * 4);
    const uint32_t dead = LINE ? persist_dead_bits(mine) : 0u;
    auto row_of = [&](uint32_t t, int k) { return (first + t + k * step) | dead; };
    const StencilValues<K, float> values{rv, n, K, pl};

    float x[R], r[R], p[R], v[REGS > 0 ? R : 1][REGS > 0 ? REGS : 1];
    FactorRow<KG> g[R], gt[R];
    float* const kept = tile + pl.tile_size;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t i = row_of(tid, k);
        const bool live = i < n;
        x[k] = live ? a.x[i] : 0.f;
        r[k] = live ? a.r[i] : 0.f;
        p[k] = live ? a.p[i] : 0.f;
#pragma unroll
        for (int d = 0; d < K; ++d) {
            const int at = place<K>(d);
            if (at < REGS) v[k][at] = values(i, d, a.sym != 0);
            else if (at < REGS + KEPT) kept[((at - REGS) * R + k) * kGridThreads + tid] = values(i, d, a.sym != 0);
        }
        g[k].load(rg, n, pl, i, false);
        gt[k].load(rg, n, pl, i, true);
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
    if constexpr (!LINE) where.find(pl, first, tid);
    const bool shared = gridDim.x > 1;  // some other workgroup reads this one's rows
    const double norm_ref = st->norm_ref, rel_tol = st->rel_tol, abs_stop = st->abs_tol * st->init_res;
    const int max_iters = st->max_iters, crit = st->crit;
    int iter = st->iter;
    uint32_t epoch = st->epoch;
    double res = st->cur_res, best = a.best;
    bool conv = false, done = false, ok = true;
    double sums[2];
    for (int ran = 0;;) {
        // Opaque, anew for every product: keeps the address arithmetic with it
        // (kept from one to the next, it takes more registers than the rows).
        uint32_t t = tid;
        auto anew = [&] {
            asm volatile("" : "+v"(t));
            if constexpr (LINE) asm volatile("" : "+s"(step), "+s"(tstep));
        };
        anew();
        // (and the tests of the registers' values for 0: hoisted, their masks
        // take more scalar registers than there are)
#pragma unroll
        for (int k = 0; k < (REGS > 0 ? R : 0); ++k)
#pragma unroll
            for (int d = 0; d < REGS; ++d) asm volatile("" : "+v"(v[k][d]));
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int q = 0; q < (KG + 1) / 2; ++q) asm volatile("" : "+v"(g[k].two[q]), "+v"(gt[k].two[q]));
        float c0[N], c1[N];
        auto own = [&](const float (&q)[R]) {
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (mine) tile[pl.own + k * tstep + t] = q[k];
        };
        auto publish = [&](float* to, const float (&q)[R]) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t i = row_of(t, k);
                if (shared && i < n) store_shared(to + i, q[k]);
            }
        };
        // p; y = A p, <y, p>
        own(p);
        fill_tile<R, LINE, N>(
            pl, first, t, live_threads, where, [&](uint32_t j, int u) { c0[u] = load_shared<float>(rp, j, n); },
            [&](uint32_t at, int u) { tile[at] = c0[u]; });
        __syncthreads();
        float y[R];
        double yp = 0.0;
        constexpr int U = persist_group<float, R>();
#pragma unroll
        for (int k0 = 0; k0 < R; k0 += U) {
            if (k0 > 0) anew();
            float av[U][K];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int d = 0; d < K; ++d) {
                    const int in = place<K>(d);
                    if (in < REGS) av[u][d] = v[REGS > 0 ? k0 + u : 0][in < REGS ? in : 0];
                    else if (in < REGS + KEPT) av[u][d] = kept[((in - REGS) * R + k0 + u) * kGridThreads + t];
                    else av[u][d] = values(row_of(t, k0 + u), d, SYM);
                }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t at = pl.own + (k0 + u) * tstep + t;
                double sum = 0.0;  // FP32 products summed in FP64, as the CSR SpMV sums them
#pragma unroll
                for (int d = 0; d < K; ++d) {
                    const float pj = tile[at + static_cast<uint32_t>(pl.delta[d])];
                    sum += stencil_term(av[u][d], pj);
                }
                y[k0 + u] = static_cast<float>(sum);
                yp += static_cast<double>(y[k0 + u]) * static_cast<double>(p[k0 + u]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        anew();
        publish(a.y, y);
        sums[0] = yp;
        if (!(ok = grid_sum<1>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        // x, r; w = G^T r, <r, z> = ||w||^2, ||r||
        anew();
        const float alpha = static_cast<float>(rz / sums[0]);
        double rzn = 0.0, nr = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            x[k] = x[k] + alpha * p[k];
            r[k] = r[k] - alpha * y[k];
            const double d = static_cast<double>(r[k]);
            nr += crit == kCritL2 ? d * d : fabs(d);
        }
        own(r);
        fill_tile<R, LINE, N, kUpper>(
            pl, first, t, live_threads, where,
            [&](uint32_t j, int u) {
                c0[u] = load_shared<float>(rr, j, n);
                c1[u] = load_shared<float>(ry, j, n);
            },
            [&](uint32_t at, int u) { tile[at] = c0[u] - alpha * c1[u]; });
        __syncthreads();
        float w[R];
#pragma unroll
        for (int k0 = 0; k0 < R; k0 += U) {
            if (k0 > 0) anew();
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t at = pl.own + (k0 + u) * tstep + t;
                double sum = 0.0;
#pragma unroll
                for (int d = KG - 1; d >= 0; --d) {
                    const float rj = tile[at + static_cast<uint32_t>(pl.delta[K - 1 - d])], gv = gt[k0 + u][d];
                    sum += stencil_term(gv, rj);
                }
                w[k0 + u] = static_cast<float>(sum);
                rzn += static_cast<double>(w[k0 + u]) * static_cast<double>(w[k0 + u]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        anew();
        publish(a.w, w);
        sums[0] = rzn;
        sums[1] = nr;
        if (!(ok = grid_sum<2>(a.slots, wg, epoch, sums, sh, a.spin_limit))) break;
        const float beta = static_cast<float>(sums[0] / rz);
        rz = sums[0];
        res = (crit == kCritL2 ? sqrt(sums[1]) : sums[1]) / norm_ref;
        conv = res <= rel_tol || res <= abs_stop;
        done = conv || iter >= max_iters;
        if (wg == 0 && tid == 0) st->hist[iter % kHist] = res;
        ++iter;
        ++ran;
        bool end = done || ran >= a.max_run;
        if (!end && ran % kChunk == 0) {
            end = !(res > a.go_on && res < 0.5 * best);
            if (!end) best = res;
        }
        // p = G w + beta p
        anew();
        own(w);
        fill_tile<R, LINE, N, kLower>(
            pl, first, t, live_threads, where, [&](uint32_t j, int u) { c0[u] = load_shared<float>(rw, j, n); },
            [&](uint32_t at, int u) { tile[at] = c0[u]; });
        __syncthreads();
#pragma unroll
        for (int k0 = 0; k0 < R; k0 += U) {
            if (k0 > 0) anew();
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t at = pl.own + (k0 + u) * tstep + t;
                double sum = 0.0;
#pragma unroll
                for (int d = 0; d < KG; ++d) {
                    const float wj = tile[at + static_cast<uint32_t>(pl.delta[d])], gv = g[k0 + u][d];
                    sum += stencil_term(gv, wj);
                }
                p[k0 + u] = static_cast<float>(sum) + beta * p[k0 + u];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (end) break;
        anew();
        publish(a.p, p);
        publish(a.r, r);
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
            st->best_res = best;
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

// A stays in registers up to 8 rows per thread; with 16, three diagonals in LDS
// where the tile leaves room for them, and of a plan by lines (whose kernel has
// registers left) up to two in registers: 128^3 30.4 -> 28.4 us. 120^3 gained as
// much, 35.5 -> 33.6, before other changes took it to 27.5.
constexpr int kRegRows = 8, kFsaiRegs = 2, kFsaiKept = 3;
// With 32 rows the eight waves of a CU wait for memory that the 32 of the
// launch-per-step kernels overlap: 160^3 72 us an iteration against 65.7.
constexpr uint32_t kMostRows = 16;

template <int K, bool SYM, int R, int REGS, int KEPT, bool LINE>
hipError_t launch_kernel(FsaiPersistArgs& a, hipStream_t s)
{
    auto* f = &fsai_persist_kernel<K, SYM, R, REGS, KEPT, LINE>;
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(f),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize, kPersistLds);
    if (e != hipSuccess) return e;
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(f), dim3(a.plan.wgs), dim3(kGridThreads), args,
                                      static_cast<uint32_t>((a.plan.tile_size + KEPT * R * kGridThreads) * sizeof(float)), s);
}

template <int K, bool SYM, int R, bool LINE>
hipError_t launch(FsaiPersistArgs& a, hipStream_t s)
{
    if constexpr (R <= kRegRows) return launch_kernel<K, false, R, K, 0, LINE>(a, s);
    else {
        constexpr int kKept = std::min(kFsaiKept, K), kRegs = LINE ? std::min(kFsaiRegs, K - kKept) : 0;
        if ((a.plan.tile_size + kKept * R * kGridThreads) * sizeof(float) <= kPersistLds)
            return launch_kernel<K, SYM, R, kRegs, kKept, LINE>(a, s);
        return launch_kernel<K, SYM, R, 0, 0, LINE>(a, s);
    }
}

template <int K, int R, bool LINE>
hipError_t launch_sym(FsaiPersistArgs& a, hipStream_t s)
{
    return a.sym ? launch<K, true, R, LINE>(a, s) : launch<K, false, R, LINE>(a, s);
}

template <int K>
hipError_t launch_rows(FsaiPersistArgs& a, hipStream_t s)
{
    const bool lines = a.plan.line != 0;
    switch (a.plan.rows) {
    case 1: return launch_sym<K, 1, false>(a, s);
    case 2: return launch_sym<K, 2, false>(a, s);
    case 4: return lines ? launch_sym<K, 4, true>(a, s) : launch_sym<K, 4, false>(a, s);
    case 8: return lines ? launch_sym<K, 8, true>(a, s) : launch_sym<K, 8, false>(a, s);
    case 16: return lines ? launch_sym<K, 16, true>(a, s) : launch_sym<K, 16, false>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

PersistPlan fsai_persist_plan(size_t n, int ndiag, const int32_t* off, int g_ndiag, const int32_t* g_off, int num_cus)
{
    if (!persist_enabled() || ndiag < 3 || ndiag > kPersistDiags || ndiag % 2 == 0 || g_ndiag != (ndiag + 1) / 2)
        return PersistPlan{};
    for (int d = 0; d < g_ndiag; ++d)
        if (g_off[d] != off[d] || off[ndiag - 1 - d] != -off[d]) return PersistPlan{};
    // 32-bit byte offsets into the diagonals.
    if (!dia_buf_fits(kPersistDiags, n, sizeof(float))) return PersistPlan{};
    const PersistPlan p = persist_plan(n, ndiag, off, sizeof(float), static_cast<uint32_t>(std::max(num_cus, 0)));
    return p.rows <= kMostRows ? p : PersistPlan{};
}

clsparseStatus launch_fsai_persist(FsaiPersistArgs a, hipStream_t s)
{
    hipError_t e = hipErrorInvalidValue;
    switch (a.plan.ndiag) {
    case 3: e = launch_rows<3>(a, s); break;
    case 5: e = launch_rows<5>(a, s); break;
    case 7: e = launch_rows<7>(a, s); break;
    case 9: e = launch_rows<9>(a, s); break;
    default: break;
    }
    // (refused, for instance while another process runs cooperative launches: the
    // caller goes on without, and without a word)
    return e == hipSuccess ? clsparseSuccess : clsparseInvalidKernelExecution;
}
