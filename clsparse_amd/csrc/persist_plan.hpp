// How the rows of a stencil matrix are laid out over the resident workgroups
// of a persistent solver kernel, and which rows of the other workgroups each
// one copies into its LDS per iteration. Plain C++ (host and device): the host
// tests compile this header with g++ and walk the plan.
#pragma once

#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define PP_HD __host__ __device__
#else
#define PP_HD
#endif

constexpr int kPersistDiags = 9;
constexpr uint32_t kPersistThreads = 512;  // threads per workgroup
constexpr uint32_t kPersistWgs = 256;      // workgroups at most (one per CU)
constexpr uint32_t kPersistLds = 158 * 1024;  // bytes of LDS for the operand tile

// Thread t of workgroup w owns rows first(w) + t + k * row_step, k < rows.
//
// Chunks (line == 0): a workgroup owns 512 * rows consecutive rows
// (row_step 512). Its LDS tile holds, for every group of nearby offsets
// [lo, hi], the rows [first + lo, first + hi + 512 rows): consecutive rows of
// the vector, the own ones among them for the group around 0.
// Lines (line > 0: the largest offset, a z line of a 3-D grid): a workgroup
// owns 512 consecutive columns of `rows` levels (row_step = line), so the far
// neighbours of all but its first and last level are its own rows. The tile
// holds levels -1 .. rows of 512 columns with `side` more on both sides of
// each (side: the largest offset other than the far ones).
//
// The operand of diagonal d for a row is at tile index
//   own + k * tile_step + t + delta[d].
struct PersistPlan
{
    uint32_t rows;       // per thread; 0: no plan
    uint32_t wgs;
    uint32_t row_step;
    uint32_t line, side, col_tiles;  // lines only
    int ndiag;
    uint32_t own, tile_step, tile_size;
    int32_t off[kPersistDiags];
    int32_t delta[kPersistDiags];
    // Chunks: copies of [first + from, first + from + len) to tile index at
    // (the own rows are not copied: they are written from registers).
    uint32_t ncopy, copy_total;
    int32_t copy_from[kPersistDiags + 1];
    uint32_t copy_len[kPersistDiags + 1], copy_at[kPersistDiags + 1];
};

PP_HD inline uint32_t persist_first_row(const PersistPlan& p, uint32_t wg)
{
    if (p.line == 0) return wg * kPersistThreads * p.rows;
    const uint32_t lev = wg / p.col_tiles;
    return lev * p.rows * p.line + (wg - lev * p.col_tiles) * kPersistThreads;
}

// The threads of workgroup wg whose rows are rows of the matrix's lines (the
// last column tile of a line may be partial).
PP_HD inline uint32_t persist_live_threads(const PersistPlan& p, uint32_t wg)
{
    if (p.line == 0) return kPersistThreads;
    const uint32_t left = p.line - (wg % p.col_tiles) * kPersistThreads;
    return left < kPersistThreads ? left : kPersistThreads;
}

PP_HD inline bool persist_live_thread(const PersistPlan& p, uint32_t wg, uint32_t t)
{
    return t < persist_live_threads(p, wg);
}

// Lines: the columns that a workgroup with `live` columns copies for each of its own
// levels (each column's place there; below 0 they wrap): `side` ones on both sides of
// its 512, and in the last column tile of a line the `side` ones past its end that
// are not among those (rows of the next line, which diagonals that run across line
// ends read). Only the rows below the workgroup's own ones (kLower: left), only those
// above (kUpper), or both.
enum Side : int { kBoth, kLower, kUpper };

struct PersistColumns
{
    uint32_t left, right, past, live;
    PP_HD uint32_t count() const { return left + right + past; }
    PP_HD uint32_t operator()(uint32_t e) const
    {
        return e < left ? e - left : e < left + right ? kPersistThreads + e - left : live + e - left - right;
    }
};

PP_HD inline PersistColumns persist_columns(const PersistPlan& p, Side side, uint32_t live)
{
    const uint32_t idle = kPersistThreads - live;
    return {side != kUpper ? p.side : 0, side != kLower ? p.side : 0,
            side != kLower ? (p.side < idle ? p.side : idle) : 0, live};
}

inline void persist_copy(PersistPlan* p, int64_t from, int64_t len, int64_t at)
{
    if (len <= 0) return;
    p->copy_from[p->ncopy] = static_cast<int32_t>(from);
    p->copy_len[p->ncopy] = static_cast<uint32_t>(len);
    p->copy_at[p->ncopy] = static_cast<uint32_t>(at);
    p->copy_total += static_cast<uint32_t>(len);
    ++p->ncopy;
}

// Chunks of `rows` rows per thread for offsets off[0..nd) in ascending order,
// 0 among them or not; rows = 0 when the tile does not fit.
inline PersistPlan persist_plan_chunks(size_t n, int nd, const int32_t* off, uint32_t rows, size_t value_size)
{
    PersistPlan p{};
    const int64_t tile = int64_t(kPersistThreads) * rows;
    const size_t wgs = (n + tile - 1) / tile;
    p.ndiag = nd;
    p.row_step = p.tile_step = kPersistThreads;
    p.wgs = static_cast<uint32_t>(wgs);
    // Own rows first; groups of offsets whose intervals touch share one.
    int64_t at = 0;
    bool have_own = false;
    auto group = [&](int64_t lo, int64_t hi, int d0, int d1) {
        const bool own = lo <= 0 && hi >= 0;
        const int64_t base = at - lo;  // tile index of offset 0 of row first
        for (int d = d0; d < d1; ++d) p.delta[d] = static_cast<int32_t>(base + off[d]);
        if (own) {
            p.own = static_cast<uint32_t>(base);
            have_own = true;
            persist_copy(&p, lo, -lo, at);
            persist_copy(&p, tile, hi, base + tile);
        } else {
            persist_copy(&p, lo, hi - lo + tile, at);
        }
        at += hi - lo + tile;
    };
    // Offsets near 0 (|o| <= tile) and 0 itself form the own group; the
    // others are joined while they are within a tile of each other.
    int d = 0;
    while (d < nd && off[d] < -tile) {
        int e = d + 1;
        while (e < nd && off[e] < -tile && int64_t(off[e]) - off[e - 1] <= tile) ++e;
        group(off[d], off[e - 1], d, e);
        d = e;
    }
    int e = d;
    while (e < nd && off[e] <= tile) ++e;
    group(e > d && off[d] < 0 ? off[d] : 0, e > d && off[e - 1] > 0 ? off[e - 1] : 0, d, e);
    d = e;
    while (d < nd) {
        e = d + 1;
        while (e < nd && int64_t(off[e]) - off[e - 1] <= tile) ++e;
        group(off[d], off[e - 1], d, e);
        d = e;
    }
    if (!have_own || at * int64_t(value_size) > int64_t(kPersistLds) || wgs > kPersistWgs) return PersistPlan{};
    for (int k = 0; k < nd; ++k) {
        p.off[k] = off[k];
        p.delta[k] -= static_cast<int32_t>(p.own);
    }
    p.tile_size = static_cast<uint32_t>(at);
    p.rows = rows;
    return p;
}

// Lines: offsets -line, ..., line with every other offset of at most 256 in
// size; rows = 0 when the matrix has no such form or the tile does not fit.
inline PersistPlan persist_plan_lines(size_t n, int nd, const int32_t* off, uint32_t rows, size_t value_size)
{
    PersistPlan p{};
    if (nd < 3 || off[0] >= 0 || off[0] != -off[nd - 1]) return p;
    const int64_t line = off[nd - 1];
    int64_t side = 0;
    for (int d = 1; d < nd - 1; ++d) {
        const int64_t o = off[d] < 0 ? -int64_t(off[d]) : off[d];
        if (o > side) side = o;
    }
    if (line < 2 * int64_t(kPersistThreads) || 2 * side > int64_t(kPersistThreads)) return p;
    const uint64_t tiles = (line + kPersistThreads - 1) / kPersistThreads;
    const uint64_t levels = (n + line - 1) / line;
    const uint64_t wgs = tiles * ((levels + rows - 1) / rows);
    const uint64_t width = kPersistThreads + 2 * side, size = width * (rows + 2);
    if (wgs > kPersistWgs || size * value_size > kPersistLds) return p;
    p.ndiag = nd;
    p.wgs = static_cast<uint32_t>(wgs);
    p.row_step = p.line = static_cast<uint32_t>(line);
    p.side = static_cast<uint32_t>(side);
    p.col_tiles = static_cast<uint32_t>(tiles);
    p.tile_step = static_cast<uint32_t>(width);
    p.own = static_cast<uint32_t>(width + side);
    p.tile_size = static_cast<uint32_t>(size);
    for (int d = 0; d < nd; ++d) {
        p.off[d] = off[d];
        p.delta[d] = off[d] == line ? int32_t(width) : off[d] == -line ? -int32_t(width) : off[d];
    }
    p.rows = rows;
    return p;
}

// The plan of an n-row matrix on the ascending offsets off[0..nd) with one
// workgroup per CU; rows = 0 when no plan covers it (more than 16 FP64 or 32
// FP32 rows per thread, or a tile larger than the LDS).
//
// The fewest rows per thread that cover the matrix: an iteration of a small
// system is latency, and one row's chain is the shortest (9,393 rows, FP64:
// 5.2 us with 1 row on 19 workgroups, 6.3 with 4, 8.9 with 8). One or two rows
// only on at most half of the CUs: with the sums and the halos of 256
// workgroups 262,144 rows take 9.3 us, with 4 rows on 128 workgroups 8.6
// (125,000 rows: 9.1 us with 1 row, 7.8 with 2). From 4 rows on lines are
// preferred to chunks, whose workgroups read two far values per row from each
// other (262,144 rows 8.6 against 9.0 us; 16 FP64 rows of three groups do not
// fit the LDS at all).
inline PersistPlan persist_plan(size_t n, int nd, const int32_t* off, size_t value_size, uint32_t num_cus)
{
    if (n == 0 || n >= (size_t(1) << 30) || nd < 1 || nd > kPersistDiags) return PersistPlan{};
    const uint32_t most = value_size == 4 ? 32 : 16;
    for (uint32_t r = 1; r <= most; r *= 2) {
        PersistPlan p{};
        if (r >= 4) p = persist_plan_lines(n, nd, off, r, value_size);
        if ((p.rows == 0 || p.wgs > num_cus) && r <= 16) p = persist_plan_chunks(n, nd, off, r, value_size);
        if (p.rows != 0 && p.wgs <= (r <= 2 ? num_cus / 2 : num_cus)) return p;
    }
    return PersistPlan{};
}
