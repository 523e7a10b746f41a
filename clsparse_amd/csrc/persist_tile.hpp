// What the persistent solver kernels share: the operand tile in LDS and the
// reads of A's diagonal storage.
#pragma once

#include "common.hpp"
#include "grid_sync.hpp"
#include "persist_plan.hpp"

namespace {

template <typename T>
__device__ __forceinline__ T rounded_mul(T a, T b)
{
#pragma clang fp contract(off)
    return a * b;
}

// All bits set for a thread that owns no rows: or'ed to a row index it makes
// one past every matrix. Opaque: as `mine ? row : ~0` the compiler splits the
// kernel by `mine` and spills hundreds of registers (32 FP32 rows per thread).
__device__ __forceinline__ uint32_t persist_dead_bits(bool mine)
{
    uint32_t dead = mine ? 0u : 0xFFFFFFFFu;
    asm volatile("" : "+v"(dead));
    return dead;
}

// Rows of a product in flight: their values of A from memory, their operands
// from the tile.
template <typename T, int R>
constexpr int persist_group()
{
    return R < 4 ? R : R * sizeof(T) <= 32 ? 4 : 2;
}

// v x of a row's sum, 0 where v is 0 (whatever x is). A select, not a branch:
// within `if (v != 0)` the compiler reads x from the LDS one value at a time
// (with it, the dead bits and the groups of rows below, 64^3 FP64 CG 8.1 -> 6.9
// us an iteration, 128^3 25.8 -> 23.1, FP32 128^3 21.6 -> 16.2, 160^3 36.9 -> 32.0).
template <typename T>
__device__ __forceinline__ double stencil_term(T v, T x)
{
    const T product = rounded_mul(v, x);
    return static_cast<double>(v != T(0) ? product : T(0));
}

// Copies the rows of other workgroups that this one's operands need into its
// tile, N of them per thread in flight: get(row, slot) starts a load and
// put(tile index, slot) stores its value. Chunks: the plan's copies as one
// list (their loads overlap: one memory latency for all of them, not one per
// copy), `where` its first N entries of this thread. side: only the rows below
// the workgroup's own ones (kLower), only those above (kUpper), or both.
constexpr uint32_t kNoRow = 0xFFFFFFFFu;

__device__ __forceinline__ void fill_where(const PersistPlan& pl, uint32_t first, uint32_t e, uint32_t& row, uint32_t& at)
{
    row = kNoRow;
    at = 0;
    for (uint32_t c = 0; c < pl.ncopy; ++c) {
        const uint32_t len = pl.copy_len[c];
        if (e < len) {
            row = first + static_cast<uint32_t>(pl.copy_from[c]) + e;
            at = pl.copy_at[c] + e;
            e = kNoRow;
        } else if (e != kNoRow) {
            e -= len;
        }
    }
    if (e != kNoRow) at = kNoRow;
}

template <int N>
struct FillSlots
{
    uint32_t row[N], at[N];
    __device__ __forceinline__ void find(const PersistPlan& pl, uint32_t first, uint32_t tid)
    {
#pragma unroll
        for (int u = 0; u < N; ++u) fill_where(pl, first, tid + u * kGridThreads, row[u], at[u]);
    }
};

// Slots of a plan by lines that take the two whole levels and up to eight levels
// of a column at once.
template <int R>
constexpr int line_slots()
{
    return 2 + (R < 8 ? R : 8);
}

template <int R, bool LINE, int N, Side SIDE = kBoth, typename Get, typename Put>
__device__ __forceinline__ void fill_tile(const PersistPlan& pl, uint32_t first, uint32_t tid, uint32_t live,
                                          const FillSlots<LINE ? 1 : N>& where, Get get, Put put)
{
    if constexpr (!LINE) {
        auto wanted = [&](int32_t from) { return SIDE == kBoth || (from < 0) == (SIDE == kLower); };
        if (pl.copy_total <= N * kGridThreads) {
            auto live = [&](int u) {
                return where.at[u] != kNoRow && wanted(static_cast<int32_t>(where.row[u] - first));
            };
#pragma unroll
            for (int u = 0; u < N; ++u)
                if (live(u)) get(where.row[u], u);
#pragma unroll
            for (int u = 0; u < N; ++u)
                if (live(u)) put(where.at[u], u);
            return;
        }
        for (uint32_t c = 0; c < pl.ncopy; ++c) {
            if (!wanted(pl.copy_from[c])) continue;
            const uint32_t len = pl.copy_len[c], at = pl.copy_at[c];
            const uint32_t row = first + static_cast<uint32_t>(pl.copy_from[c]);
            for (uint32_t e0 = tid; e0 < len; e0 += N * kGridThreads) {
#pragma unroll
                for (int u = 0; u < N; ++u)
                    if (e0 + u * kGridThreads < len) get(row + e0 + u * kGridThreads, u);
#pragma unroll
                for (int u = 0; u < N; ++u)
                    if (e0 + u * kGridThreads < len) put(at + e0 + u * kGridThreads, u);
            }
        }
    } else {
        // The levels before the first and after the last, and of every level the
        // columns beside the workgroup's own (persist_columns). One column a thread,
        // M of its levels at a time: the slowest workgroup's memory latencies
        // hold up all others. The first of them together with the two whole
        // levels where the caller has the slots for it (BiCGStab 85 x 90 x 80
        // 21.6 -> 20.6 us an iteration, learned FSAI 60^3 14.8 -> 14.1; CG with 16
        // FP32 rows has no registers for them: 15.9 -> 16.6).
        constexpr bool kTogether = N == line_slots<R>();
        constexpr int M = kTogether ? N - 2 : N < R ? N : R;
        const PersistColumns column = persist_columns(pl, SIDE, live);
        const uint32_t columns = column.count();
        const uint32_t c = column(tid);
        if (SIDE != kUpper) get(first - pl.line + tid, 0);
        if (SIDE != kLower) get(first + R * pl.line + tid, 1);
        if (kTogether && tid < columns) {
#pragma unroll
            for (int u = 0; u < M; ++u) get(first + u * pl.line + c, (2 + u) % N);
        }
        if (SIDE != kUpper) put(pl.own - pl.tile_step + tid, 0);
        if (SIDE != kLower) put(pl.own + R * pl.tile_step + tid, 1);
        if (kTogether && tid < columns) {
#pragma unroll
            for (int u = 0; u < M; ++u) put(pl.own + u * pl.tile_step + c, (2 + u) % N);
        }
        auto levels = [&](uint32_t col, int k_first) {
#pragma unroll 1
            for (int k0 = k_first; k0 < R; k0 += M) {
#pragma unroll
                for (int u = 0; u < M; ++u) get(first + (k0 + u) * pl.line + col, u);
#pragma unroll
                for (int u = 0; u < M; ++u) put(pl.own + (k0 + u) * pl.tile_step + col, u);
            }
        };
        if (tid < columns) levels(c, kTogether ? M : 0);
        if (columns > kGridThreads)
            for (uint32_t e = tid + kGridThreads; e < columns; e += kGridThreads) levels(column(e), 0);
    }
}

// A in diagonal storage: values(i, d, half) is A(i, i + off[d]), 0 outside the
// matrix and for the diagonals past the nd stored ones; half: the upper
// diagonals are read from the lower ones, mirrored to row i + off[d].
template <int K, typename T>
struct StencilValues
{
    __amdgpu_buffer_rsrc_t rs;
    uint32_t n, nd;
    const PersistPlan& pl;

    // The diagonal's start is the load's scalar offset, so all diagonals of a row
    // share one vector offset; no row: 2 GB, past the end (a plan's 2^22 rows
    // at most take 9 x 16 MB).
    __device__ __forceinline__ T lower(uint32_t i, uint32_t d) const
    {
        const uint32_t S = sizeof(T);
        return buf_load<T>(rs, i < n ? i * S : 0x80000000u, d * n * S);
    }
    __device__ __forceinline__ T operator()(uint32_t i, int d, bool half) const
    {
        if (half && d >= (K + 1) / 2)
            return lower(i < n ? i + static_cast<uint32_t>(pl.off[d]) : n, K - 1 - d);
        return lower(d < static_cast<int>(nd) ? i : n, d);
    }
};

}  // namespace
