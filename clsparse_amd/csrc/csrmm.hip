// Sparse times dense: C = alpha * A * B + beta * C (clsparse[S/D]csrmm).
//
// Semantics of the reference (src/library/blas3/clsparse-csrmm.cpp L25-76,
// clsparse-csrmm.hpp L84-179, kernels/csrmm_general.cl L59-167): B and C are
// row-major with lead_dim as the row stride (the major field is not read),
// element (k, c) of B at off_values + k * lead_dim + c; alpha == 0 gives
// beta * C without reading B, beta == 0 never reads C, beta == 1 adds C.
// The reference runs one CSR-Vector SpMV per column of C (A re-read for every
// column). Here each lane owns V consecutive columns (16 bytes of them wherever
// they start: the hardware needs only an element's alignment), W lanes (a power
// of two >= the column groups, up to 64) form a row slot, and a wave runs 64 / W
// rows of C at once: each slot loads W or 4 W nonzeros of its row, hands each
// nonzero's value and column to its lanes through lane permutes, and keeps 4 or
// 8 B row segments in flight per step, every one a coalesced read. What bounds
// it is the texture data path (busy for most of the kernel) and, for long rows
// on few waves, the latency of a slot's chain of trips; so a group of columns
// takes as few lanes as its bytes allow, also where V does not divide the
// columns (81 entries a row times 13 FP32 columns: 16 one-column lanes per row
// 52 us, 4 four-column lanes with four nonzeros each 36 us; one FP64 column
// 68 -> 30 us), rows far longer than the mean are shared by the slots of their wave,
// and rows past kLongRow entries by the workgroup (a power-law matrix with
// 75,000-entry rows times 13 FP64 columns: 7.5 ms -> 0.41).
// Waves walk consecutive rows and workgroups are remapped so each XCD covers
// one contiguous range of rows (neighbouring rows share B rows in its L2). Each
// element of C is summed in an order fixed by the shapes, so results are
// deterministic.
#include <algorithm>

#include "common.hpp"

namespace {

// B row segments in flight per lane: 8; 4 of 16 bytes where a mean row is one
// trip (short rows want the waves that fewer registers allow: 7 entries times
// 24 FP64 columns 97 against 105 us; 81 entries times 13 FP32 columns 43
// against 36 us with 8).
template <int V, int Q>
constexpr int b_in_flight() { return V > 1 && Q == 1 ? 4 : 8; }

// Rows longer than this are left to the whole workgroup: one slot alone walks
// them at a few nonzeros per memory latency.
constexpr uint32_t kLongRow = 512;
constexpr uint32_t kLongList = 16;  // per wave, in the wave's row order; rows past it stay with their slot

// V consecutive columns of a row of B or C per lane, read and written with one
// access of V * sizeof(T) bytes wherever they start (an element's alignment is
// enough for the hardware).
template <typename T, int V>
struct Cols
{
    T e[V];
};

template <typename T, int V>
__device__ __forceinline__ Cols<T, V> load_cols(const T* p)
{
    Cols<T, V> r;
    if constexpr (V > 1) {
        typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
        const vec x = *reinterpret_cast<const vec*>(p);
#pragma unroll
        for (int k = 0; k < V; ++k) r.e[k] = x[k];
    } else {
        r.e[0] = p[0];
    }
    return r;
}

template <typename T, int V>
__device__ __forceinline__ void store_cols(T* p, const Cols<T, V>& r)
{
    if constexpr (V > 1) {
        typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
        vec x;
#pragma unroll
        for (int k = 0; k < V; ++k) x[k] = r.e[k];
        *reinterpret_cast<vec*>(p) = x;
    } else {
        p[0] = r.e[0];
    }
}

// A place in the entries, `by` further on. TOP: entries may lie less than a step below
// 2^32, where a place that wrapped would be one before its row's end again; it stays at
// 2^32 - 1, which no entry has.
template <bool TOP>
__device__ __forceinline__ uint32_t further(uint32_t at, uint32_t by)
{
    return TOP ? __builtin_elementwise_add_sat(at, by) : at + by;
}
constexpr uint32_t kMostStep = 1024;  // nonzeros that a workgroup of Q = 4 takes in turn

// sum += the nonzeros j of [beg, end) with (j - beg) % step < W Q, Q consecutive
// ones per lane of the slot and W Q per trip, times the lane's V columns at Bc.
template <typename T, int W, int V, int Q, bool TOP>
__device__ __forceinline__ void slot_sum(Cols<T, V>& sum, uint32_t beg, uint32_t end, uint32_t step, uint32_t nnz,
                                         const uint32_t* __restrict__ ci, const T* __restrict__ v,
                                         const T* __restrict__ Bc, uint32_t ldb, T alpha, bool colok, uint32_t t, int base)
{
    constexpr int kIn = b_in_flight<V, Q>();
    static_assert(kIn % Q == 0, "a group of loads starts at a lane's first nonzero");
    // Lane t of the slot holds nonzeros j0 + Q t .. + Q - 1 of a trip; with Q > 1
    // (rows of several trips) the next trip's are loaded before this one's B rows.
    T an[Q];
    uint32_t cn[Q];
    auto load = [&](uint32_t j0) {
        const uint32_t jj = j0 + Q * t;
        if constexpr (Q > 1) {
            typedef uint32_t cvec __attribute__((ext_vector_type(Q), aligned(4)));
            typedef T tvec __attribute__((ext_vector_type(Q), aligned(sizeof(T))));
            if (jj < end && nnz - jj >= Q) {
                const cvec c4 = *reinterpret_cast<const cvec*>(ci + jj);
                const tvec v4 = *reinterpret_cast<const tvec*>(v + jj);
#pragma unroll
                for (int u = 0; u < Q; ++u) {
                    cn[u] = c4[u];
                    an[u] = v4[u];
                }
                return;
            }
        }
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            an[u] = jj + u < end ? v[jj + u] : T(0);
            cn[u] = jj + u < end ? ci[jj + u] : 0u;
        }
    };
    if (Q > 1) load(beg);
    for (uint32_t j0 = beg; j0 < end; j0 = further<TOP>(j0, step)) {
        if (Q == 1) load(j0);
        T av[Q];
        uint32_t cc[Q];
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            av[u] = alpha * an[u];
            cc[u] = cn[u];
        }
        if (Q > 1 && further<TOP>(j0, step) < end) load(further<TOP>(j0, step));
        const uint32_t cnt = min(static_cast<uint32_t>(W * Q), end - j0);
        for (uint32_t q = 0; q < cnt; q += kIn) {
            T a8[kIn];
            Cols<T, V> b8[kIn];
#pragma unroll
            for (int u = 0; u < kIn; ++u) {
                const int src = base + static_cast<int>(min((q + u) / Q, static_cast<uint32_t>(W - 1)));
                a8[u] = __shfl(av[u % Q], src, 64);
                const uint32_t col = __shfl(cc[u % Q], src, 64);
#pragma unroll
                for (int k = 0; k < V; ++k) b8[u].e[k] = T(0);
                if (colok && q + u < cnt) b8[u] = load_cols<T, V>(Bc + static_cast<size_t>(col) * ldb);
            }
            // No branch around the products (b8 is 0 past cnt): 1024^2 rows of 3 entries
            // near the diagonal times 32 FP64 columns 59 -> 53 us. Not so with four nonzeros a
            // lane in wide slots, whose loads then all arrive before the first product: random
            // rows of 200 times 16 FP64 columns 40 us with branches, 52 without.
            constexpr bool kBranch = Q > 1 && W >= 8;
#pragma unroll
            for (int u = 0; u < kIn; ++u) {
                if (kBranch && q + u >= cnt) continue;
                const T a = q + u < cnt ? a8[u] : T(0);
#pragma unroll
                for (int k = 0; k < V; ++k) sum.e[k] = fma(a, b8[u].e[k], sum.e[k]);
            }
        }
    }
}

// The sum of a lane's columns over the slots of its wave, in every one of them.
template <int W, typename T, int V>
__device__ __forceinline__ void add_slots(Cols<T, V>& sum)
{
#pragma unroll
    for (int d = W; d < 64; d *= 2)
#pragma unroll
        for (int k = 0; k < V; ++k) sum.e[k] += __shfl_xor(sum.e[k], d, 64);
}

// The lane's columns of one row of C: out = beta out + sum; only the columns
// from `skip` on are the lane's to store.
template <bool RAGGED, typename T, int V>
__device__ __forceinline__ void finish_cols(T* out, Cols<T, V> sum, T beta, uint32_t skip)
{
    if (beta != T(0)) {
        const Cols<T, V> old = load_cols<T, V>(out);
#pragma unroll
        for (int k = 0; k < V; ++k) sum.e[k] = beta == T(1) ? sum.e[k] + old.e[k] : sum.e[k] + beta * old.e[k];
    }
    if (!RAGGED || skip == 0) {
        store_cols<T, V>(out, sum);
    } else {
#pragma unroll
        for (int k = 0; k < V; ++k)
            if (static_cast<uint32_t>(k) >= skip) out[k] = sum.e[k];
    }
}

// W lanes per row slot, V columns per lane, Q nonzeros per lane and trip.
// RAGGED (V does not divide ncols, ncols >= V): the last group of a row starts
// early and stores the columns that are its own. Rows of more than wave_row entries
// are taken by all slots of the wave. Eight waves per SIMD with one nonzero a lane,
// four with four, are the most that the loads in flight leave registers for.
template <typename T, int W, int V, int Q, bool RAGGED, bool TOP>
__global__ __launch_bounds__(256, Q == 1 ? 8 : 4) void csrmm_kernel(uint32_t num_rows, uint32_t ncols, uint32_t nnz,
                                                    uint32_t wave_row,
                                                    const uint32_t* __restrict__ rp,
                                                    const uint32_t* __restrict__ ci,
                                                    const T* __restrict__ v, const T* __restrict__ B,
                                                    uint32_t ldb, T* __restrict__ C, uint32_t ldc,
                                                    const T* __restrict__ pAlpha,
                                                    const T* __restrict__ pBeta)
{
    constexpr uint32_t kSlots = 64 / W;
    static_assert(4 * kSlots * W * Q <= kMostStep, "the largest step");
    __shared__ uint32_t long_rows[4][kLongList];
    __shared__ uint32_t long_count[4];
    __shared__ T part[4][W * V];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t slot = lane / W;
    const uint32_t t = lane % W;
    const int base = static_cast<int>(slot * W);  // first lane of this slot
    const T alpha = *pAlpha;
    const T beta = *pBeta;
    const uint32_t wv = threadIdx.x >> 6;
    uint32_t nlong = 0;  // of this wave
    // Each XCD (gridDim.x is a multiple of 8; logical workgroups [x G/8,
    // (x+1) G/8) run on XCD x) owns one contiguous eighth of the rows and its
    // waves sweep it in steps of waves * kSlots rows: a B row shared by
    // nearby rows is then fetched into one L2, not one per XCD.
    const uint32_t lb = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t per_xcd = gridDim.x / 8;
    const uint32_t xcd = lb / per_xcd;
    const uint32_t rows_per_xcd = (num_rows + 7) / 8;
    const uint32_t first = min(num_rows, xcd * rows_per_xcd);
    const uint32_t stop = min(num_rows, first + rows_per_xcd);
    const uint32_t wave = (lb - xcd * per_xcd) * 4 + (threadIdx.x >> 6);
    const uint32_t waves = per_xcd * 4;
    // The next step's row bounds are loaded at the top of each step, so their
    // latency hides behind this step's nonzeros and B rows.
    uint32_t row0 = first + wave * kSlots;
    uint32_t nbeg = 0, nend = 0;
    if (row0 + slot < stop) {
        nbeg = rp[row0 + slot];
        nend = rp[row0 + slot + 1];
    }
    for (; row0 < stop; row0 += waves * kSlots) {
        const uint32_t row = row0 + slot;
        bool live = row < stop;
        uint32_t beg = nbeg, end = nend;
        const uint32_t next = row0 + waves * kSlots + slot;
        if (next < stop) {
            nbeg = rp[next];
            nend = rp[next + 1];
        }
        const unsigned long long is_long = __ballot(live && end - beg > kLongRow);
        if (is_long != 0) {
            // One bit per slot (its first lane), in slot order.
            unsigned long long firsts = 0;
#pragma unroll
            for (uint32_t q = 0; q < kSlots; ++q) firsts |= 1ull << (q * W);
            const unsigned long long bits = is_long & firsts;
            const uint32_t at = nlong + __popcll(bits & ((1ull << base) - 1));
            if ((bits >> base & 1) != 0 && at < kLongList) {  // the workgroup takes it below
                if (t == 0) long_rows[wv][at] = row;
                live = false;
                end = beg;
            }
            nlong += __popcll(bits);
        }
        // Rows far longer than the mean follow after the others, one by one, W Q
        // nonzeros to each slot of the wave in turn (200,000 rows of 4 entries, every 50th
        // of 300, times 13 FP32 columns: the wave waited 86 us for those slots; 37).
        unsigned long long wave_rows = 0;
        const uint32_t first_beg = beg, first_end = end;
        uint32_t at = row, step = W * Q;
        if constexpr (W < 64) {
            const bool far = live && end - beg > wave_row;
            wave_rows = __ballot(far && t == 0);
            if (far) {
                live = false;
                end = beg;
            }
        }
        for (bool shared = false;; shared = true) {
            for (uint32_t c0 = 0; c0 < ncols; c0 += W * V) {
                const uint32_t c = c0 + t * V;
                const uint32_t cs = RAGGED ? min(c, ncols - V) : c;
                Cols<T, V> sum;
#pragma unroll
                for (int k = 0; k < V; ++k) sum.e[k] = T(0);
                if (alpha != T(0))
                    slot_sum<T, W, V, Q, TOP>(sum, beg, end, step, nnz, ci, v, B + cs, ldb, alpha, c < ncols, t, base);
                if (shared) add_slots<W>(sum);
                if (live && c < ncols)
                    finish_cols<RAGGED, T, V>(C + static_cast<size_t>(at) * ldc + cs, sum, beta, c - cs);
            }
            if (wave_rows == 0) break;
            const int owner = __builtin_ctzll(wave_rows);
            wave_rows &= wave_rows - 1;
            beg = further<TOP>(__shfl(first_beg, owner, 64), slot * (W * Q));
            end = __shfl(first_end, owner, 64);
            step = kSlots * W * Q;
            at = row0 + static_cast<uint32_t>(owner) / W;
            live = slot == 0;
        }
    }
    if (lane == 0) long_count[wv] = min(nlong, kLongList);
    __syncthreads();
    // Long rows: all slots of the workgroup take turns at W Q nonzeros, then
    // their sums are added in slot order.
    if ((long_count[0] | long_count[1] | long_count[2] | long_count[3]) == 0) return;
    for (uint32_t i = 0; i < 4 * kLongList; ++i) {
        if (i % kLongList >= long_count[i / kLongList]) continue;
        const uint32_t row = long_rows[i / kLongList][i % kLongList];
        const uint32_t beg = rp[row], end = rp[row + 1];
        const uint32_t mine = further<TOP>(beg, (wv * kSlots + slot) * (W * Q));
        for (uint32_t c0 = 0; c0 < ncols; c0 += W * V) {
            const uint32_t c = c0 + t * V;
            const uint32_t cs = RAGGED ? min(c, ncols - V) : c;
            Cols<T, V> sum;
#pragma unroll
            for (int k = 0; k < V; ++k) sum.e[k] = T(0);
            if (alpha != T(0))
                slot_sum<T, W, V, Q, TOP>(sum, mine, end, 4 * kSlots * W * Q, nnz, ci, v, B + cs, ldb, alpha, c < ncols, t,
                                     base);
            add_slots<W>(sum);
            if (slot == 0)
#pragma unroll
                for (int k = 0; k < V; ++k) part[wv][t * V + k] = sum.e[k];
            __syncthreads();
            if (threadIdx.x < W && c < ncols) {
#pragma unroll
                for (int k = 0; k < V; ++k)
                    sum.e[k] = ((part[0][t * V + k] + part[1][t * V + k]) + part[2][t * V + k]) + part[3][t * V + k];
                finish_cols<RAGGED, T, V>(C + static_cast<size_t>(row) * ldc + cs, sum, beta, c - cs);
            }
            __syncthreads();
        }
    }
}

// Launches csrmm_kernel on at most as many workgroups as the chip holds at
// once: the kernel's resident workgroups per CU (queried once) times the CUs, a
// multiple of 8 (one equal share per XCD). The resident waves of an XCD then
// work on one compact window of its rows that advances together, so the B rows
// that neighbouring rows share stay in its L2.
template <typename T, int W, int V, int Q, bool RAGGED, bool TOP = false>
clsparseStatus launch_csrmm(int num_cus, hipStream_t s, uint32_t n, uint32_t ncols, uint32_t nnz, const uint32_t* rp,
                            const uint32_t* ci, const T* v, const T* B, uint32_t ldb, T* C, uint32_t ldc, const T* pa,
                            const T* pb)
{
    static const int per_cu = [] {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, csrmm_kernel<T, W, V, Q, RAGGED, TOP>, 256, 0) != hipSuccess) b = 0;
        return std::max(b, 1);
    }();
    constexpr uint32_t kRows = 4 * (64 / W);  // rows a workgroup has in hand
    const uint32_t want = (n + kRows - 1) / kRows;
    const uint32_t resident = std::max<uint32_t>(8u, static_cast<uint32_t>(per_cu * std::max(num_cus, 1)) / 8 * 8);
    const uint32_t grid = std::min<uint32_t>(resident, (want + 7) / 8 * 8);
    // Far longer than the mean: a row of eight times as many, and of sixteen trips.
    const uint32_t wave_row = std::max<uint32_t>(16u * W * Q, 8 * (nnz / n));
    hipLaunchKernelGGL((csrmm_kernel<T, W, V, Q, RAGGED, TOP>), dim3(grid), dim3(256), 0, s, n, ncols, nnz, wave_row, rp, ci, v, B, ldb, C,
                       ldc, pa, pb);
    CLS_HIP_TRY(hipGetLastError());
    return clsparseSuccess;
}

template <typename T>
clsparseStatus csrmm_entry(const clsparseScalar* alpha, const clsparseCsrMatrix* A,
                           const cldenseMatrix* B, const clsparseScalar* beta, cldenseMatrix* C,
                           clsparseControl control)
{
    CLS_TRY(check_init_control(control));
    if (alpha == nullptr || A == nullptr || B == nullptr || beta == nullptr || C == nullptr)
        return clsparseInvalidValue;
    // Shapes the reference reads without checking: B has A's columns as rows,
    // C has A's rows, and the leading dimensions cover the used columns.
    if (B->num_rows != A->num_cols || C->num_rows != A->num_rows || C->num_cols > B->num_cols ||
        B->lead_dim < C->num_cols || C->lead_dim < C->num_cols)
        return clsparseInvalidSize;
    const uint32_t n = A->num_rows, ncols = C->num_cols;
    if (n == 0 || ncols == 0) return finish_op(control);
    const T* pa = dev_ptr<T>(alpha->value, alpha->off_value);
    const T* pb = dev_ptr<T>(beta->value, beta->off_value);
    const T* Bp = dev_ptr<T>(B->values, B->off_values);
    T* Cp = dev_ptr<T>(C->values, C->off_values);
    if (Bp == nullptr || Cp == nullptr || pa == nullptr || pb == nullptr) return clsparseInvalidMemObject;
    CLS_TRY(launch_csrmm_rows<T>(A, ncols, Bp, B->lead_dim, Cp, C->lead_dim, pa, pb, control->num_cus,
                                 control->stream));
    return finish_op(control);
}

}  // namespace

template <typename T>
clsparseStatus launch_csrmm_rows(const clsparseCsrMatrix* A, uint32_t ncols, const T* Bp, uint32_t ldb, T* Cp,
                                 uint32_t ldc, const T* pa, const T* pb, int num_cus, hipStream_t s)
{
    const uint32_t n = A->num_rows;
    if (n == 0 || ncols == 0) return clsparseSuccess;
    const uint32_t* rp = dev_ptr<uint32_t>(A->row_pointer, A->off_row_pointer);
    const uint32_t* ci = dev_ptr<uint32_t>(A->col_indices, A->off_col_indices);
    const T* v = dev_ptr<T>(A->values, A->off_values);
    if (rp == nullptr) return clsparseInvalidMemObject;
    // V columns per lane, 16 bytes of them where there are as many; W lanes per
    // row slot (a power of two >= the column groups, at most 64). A count that V
    // does not divide takes one column a lane where the slots of all rows are fewer
    // than 512 waves: each row is then one slot's chain of trips, and more lanes make
    // it shorter (1,850 rows of 81 times 13 FP32 columns 10.5 -> 9.2 us).
    constexpr uint32_t kVec = 16 / sizeof(T);
    auto lanes = [](uint32_t groups) {
        return groups > 32 ? 64u : groups > 16 ? 32u : groups > 8 ? 16u : groups > 4 ? 8u : groups > 2 ? 4u
                                                                                   : groups > 1 ? 2u : 1u;
    };
    uint32_t V = ncols >= kVec ? kVec : (ncols >= 2 ? 2u : 1u);
    uint32_t W = lanes((ncols + V - 1) / V);
    if (ncols % V != 0 && static_cast<uint64_t>(n) * W < 512 * 64) {
        V = 1;
        W = lanes(ncols);
    }
    const uint32_t nnz = A->num_nonzeros;
    // Four nonzeros per lane and trip for rows of several trips (FP64, 8 columns,
    // W = 4: 5 entries a row 11.5 us with one and 15.2 with four, 9 entries 16.8 and
    // 19.5; 81 entries 31 and 26). With W = 16 rows of three to eight trips only where the
    // half of the waves that four leave a CU hold all slots, or many times as many
    // would be needed: 18,500 rows of 81 (4,600 waves, twice around) times 64 FP32
    // columns 21 us with one and 28 with four; 1,850 rows 11.5 and 10.0, 74,000 random
    // rows 170 and 150.
    const bool ragged = ncols % V != 0;
    const uint64_t waves = static_cast<uint64_t>(n) * W / 64;
    const bool twice = W == 16 && nnz <= 8 * static_cast<uint64_t>(n) * W &&
                       waves > 16 * static_cast<uint64_t>(num_cus) && waves <= 64 * static_cast<uint64_t>(num_cus);
    const bool quads = nnz > 3 * static_cast<uint64_t>(n) * W && !twice;
#define CLS_CSRMM(WW, VV, QQ, RR) \
    CLS_TRY((launch_csrmm<T, WW, VV, QQ, RR>(num_cus, s, n, ncols, nnz, rp, ci, v, Bp, ldb, Cp, ldc, pa, pb)))
    // Rows may end less than a step below 2^32: one kernel for all counts of columns.
    // (The additions that saturate cost the others up to 10 %: rows of 9 entries,
    // 6 M of them, one FP64 column 18.8 -> 20.7 us; 0.2 % in the mean of 722 products.)
    if (nnz > 0u - kMostStep)
        return launch_csrmm<T, 64, 1, 1, false, true>(num_cus, s, n, ncols, nnz, rp, ci, v, Bp, ldb, Cp, ldc, pa, pb);
#define CLS_CSRMM_Q(WW, VV)                  \
    do {                                     \
        if (quads && ragged)                 \
            CLS_CSRMM(WW, VV, 4, ((VV) > 1));\
        else if (quads)                      \
            CLS_CSRMM(WW, VV, 4, false);     \
        else if (ragged)                     \
            CLS_CSRMM(WW, VV, 1, ((VV) > 1));\
        else                                 \
            CLS_CSRMM(WW, VV, 1, false);     \
    } while (0)
    if (V == kVec) {
        switch (W) {
        case 64: CLS_CSRMM_Q(64, kVec); break;
        case 32: CLS_CSRMM_Q(32, kVec); break;
        case 16: CLS_CSRMM_Q(16, kVec); break;
        case 8: CLS_CSRMM_Q(8, kVec); break;
        case 4: CLS_CSRMM_Q(4, kVec); break;
        case 2: CLS_CSRMM_Q(2, kVec); break;
        default: CLS_CSRMM_Q(1, kVec); break;
        }
    } else if (V == 2) {
        if (W == 1) CLS_CSRMM_Q(1, 2);
        else CLS_CSRMM_Q(2, 2);
    } else {
        switch (W) {
        case 64: CLS_CSRMM_Q(64, 1); break;
        case 32: CLS_CSRMM_Q(32, 1); break;
        case 16: CLS_CSRMM_Q(16, 1); break;
        case 8: CLS_CSRMM_Q(8, 1); break;
        case 4: CLS_CSRMM_Q(4, 1); break;
        case 2: CLS_CSRMM_Q(2, 1); break;
        default: CLS_CSRMM_Q(1, 1); break;
        }
    }
#undef CLS_CSRMM_Q
#undef CLS_CSRMM
    CLS_HIP_TRY(hipGetLastError());
    return clsparseSuccess;
}

template clsparseStatus launch_csrmm_rows<float>(const clsparseCsrMatrix*, uint32_t, const float*, uint32_t, float*,
                                                 uint32_t, const float*, const float*, int, hipStream_t);
template clsparseStatus launch_csrmm_rows<double>(const clsparseCsrMatrix*, uint32_t, const double*, uint32_t,
                                                  double*, uint32_t, const double*, const double*, int, hipStream_t);

// src/library/blas3/clsparse-csrmm.cpp L25-49
extern "C" clsparseStatus clsparseScsrmm(const clsparseScalar* alpha, const clsparseCsrMatrix* sparseMatA,
                                         const cldenseMatrix* denseMatB, const clsparseScalar* beta,
                                         cldenseMatrix* denseMatC, const clsparseControl control)
{
    return csrmm_entry<float>(alpha, sparseMatA, denseMatB, beta, denseMatC, control);
}

// src/library/blas3/clsparse-csrmm.cpp L51-76
extern "C" clsparseStatus clsparseDcsrmm(const clsparseScalar* alpha, const clsparseCsrMatrix* sparseMatA,
                                         const cldenseMatrix* denseMatB, const clsparseScalar* beta,
                                         cldenseMatrix* denseMatC, const clsparseControl control)
{
    return csrmm_entry<double>(alpha, sparseMatA, denseMatB, beta, denseMatC, control);
}
