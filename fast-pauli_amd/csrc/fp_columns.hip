// fp_columns.hip — host side of the column kernels (fp_columns.hpp): which operators run on
// state columns, the transposed slabs and the launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>

#include "fast_pauli_hip.h"
#include "fp_apply_columns.hpp"
#include "fp_columns.hpp"
#include "fp_runtime.hpp"

using fprt::fail;

namespace
{

// Transposed states kept at a time (an apply keeps as much of outputs again).  The slab of an
// expectation is still in the Infinity Cache (256 MB) when its kernel reads it; an apply's two fill
// that cache.  us with 32 / 64 / 128 / 256 MiB: expectation n = 14, 1000 complex128 states, 1024
// strings 1744 / 1661 / 1594 / 1571, n = 20, 20 states, 1000 strings 5138 / 5087 / 4484 / 4369;
// apply n = 14, 1000 states, 500 strings 3277 / 3222 / 3162 / 3177, n = 20, 19 complex64 states, 512
// strings 5959 / 5842 / 5762 / 5680.
constexpr size_t kSlabBytes = size_t(128) << 20;
// Tiles per column: at most 2^8 (a class pairs every tile with another one).
constexpr uint32_t kMaxTileBits = 8;

size_t round256(size_t v)
{
    return (v + 255) / 256 * 256;
}

// Of an expectation: columns per tile and bytes per column.
struct ColGeom
{
    uint32_t per_group;
    size_t col_bytes;
};

ColGeom col_geom(fp_hip_ops const *ops, int dtype)
{
    bool const c64 = dtype != FP_C128;
    uint32_t const w = fpc::tile_bits(c64), n = uint32_t(ops->n_qubits);
    return ColGeom{n < w ? 1u << (w - n) : 1u, (size_t(1) << n) * (c64 ? 8u : 16u)};
}

// Columns of a slab that has room for `room`: whole tiles, and as many columns on every XCD.
uint32_t slab_columns(ColGeom const &g, size_t n_states, size_t room)
{
    size_t cols = std::min(room, n_states);
    if (cols < n_states)
    {
        size_t const whole = cols >= 8 * g.per_group ? 8 * g.per_group : g.per_group;
        cols = std::max<size_t>(cols / whole * whole, std::min<size_t>(cols, g.per_group));
    }
    return uint32_t(std::min<size_t>(cols, 0x7fffffffu));
}

template <class T, int NS, bool IN>
void launch_columns(typename fpk::VecOf<T, 1>::type *batch, typename fpk::VecOf<T, NS>::type *cols, uint64_t rows,
                    uint64_t ld, uint64_t c0, uint32_t n_cols, hipStream_t st)
{
    dim3 const grid(uint32_t((rows + 31) / 32), (n_cols + 31) / 32);
    hipLaunchKernelGGL((fpc::k_columns<T, NS, IN>), grid, dim3(256), 0, st, batch, cols, rows, ld, c0, n_cols);
}

} // namespace

namespace fprt
{

// The column kernel reads every tile once per class of strings (x >> tile bits), as a leader
// or as a partner, and pays a transposed copy of the batch; the coset-tiled kernel reads the
// batch once per group of about 9 strings.  So columns win when the classes are full: from
// about 3 strings per class (complex64: 4; 5 with a power-of-two state count, where the tiled
// kernel takes its paired lanes), and for several states from 64 strings, which pay the copy.
// One state needs no copy: from 8 strings.  Measured (us, tiled / columns; strings per class q):
//   complex128, n = 14 S = 16: N = 32 (q 8) 14.8 / 20.9, N = 256 91.8 / 28.6;
//   n = 16 S = 16: N = 32 (q 2) 24.8 / 39.9, N = 256 (q 16) 211 / 67.7;
//   n = 18: S = 16 N = 128 (q 2) 170 / 229, S = 13 N = 300 (q 4.7) 399 / 253, S = 1 N = 1000 236 / 53;
//   n = 20: S = 16 N = 512 (q 2) 2388 / 3604, S = 20 N = 1000 (q 3.9) 9364 / 5259;
//   complex64, n = 18 S = 16 N = 128 (q 4) 81 / 98, S = 13 N = 300 (q 9.4) 400 / 130;
//   n = 20 S = 16 N = 512 (q 4) 1126 / 1185, S = 1 N = 1000 (q 7.8) 281 / 119.
// FAST_PAULI_EV_KERNEL=columns forces it (where the shape allows), any other value forbids it.
bool ev_columns_eligible(fp_hip_ops const *ops, int dtype, size_t n_states)
{
    bool const c64 = dtype != FP_C128;
    uint32_t const w = fpc::tile_bits(c64), n = uint32_t(ops->n_qubits);
    if (n < fpc::low_bits(c64) || n > w + kMaxTileBits || n_states > 0x7fffffffu)
        return false;
    char const *v = std::getenv("FAST_PAULI_EV_KERNEL");
    if (v && *v)
        return std::strcmp(v, "columns") == 0;
    uint32_t const c = n > w ? n - w : 0u;
    double const q = double(ops->n_strings) / double(uint32_t(1) << c);
    if (n_states == 1)
        return ops->n_strings >= 8 && q >= (c <= 6 ? 0.5 : 3.0);
    bool const pow2 = (n_states & (n_states - 1)) == 0;
    return ops->n_strings >= 64 && q >= (c64 ? (pow2 ? 5.0 : 4.0) : 3.0);
}

fp_status run_op_expect_columns(fp_hip_ops const *ops, int dtype, void const *states, void *out, size_t dim,
                                size_t n_states, int accumulate, hipStream_t st, Workspace const *ws, bool *done)
{
    *done = false;
    bool const c64 = dtype != FP_C128;
    // one aligned state is a column already
    bool const in_place = n_states == 1 && (reinterpret_cast<uintptr_t>(states) & 15u) == 0;
    ColGeom const g = col_geom(ops, dtype);
    uint32_t slab = slab_columns(g, n_states, std::max<size_t>(1, kSlabBytes / g.col_bytes));
    // (a workspace takes the same items on smaller slabs: the same sums)
    uint32_t const per = column_item_size(c64, uint32_t(ops->n_qubits), ops->n_strings, n_states, slab);
    TileTables *tt = nullptr;
    fp_status s = tile_tables(ops, kTilesEvColumns, per, c64 ? 1u : 0u, &tt);
    if (s != FP_OK)
        return s;
    uint32_t const n_items = tt->n_groups;
    size_t const table_bytes = round256(tt->h.size());
    if (ws)
    {
        size_t const per_column = (in_place ? 0 : g.col_bytes) + size_t(n_items) * sizeof(fpk::Dbl2);
        if (ws->bytes < table_bytes + 256 + per_column)
            return FP_OK;
        slab = std::min(slab, slab_columns(g, n_states, (ws->bytes - table_bytes - 256) / per_column));
    }
    size_t const slab_bytes = in_place ? 0 : round256(slab * g.col_bytes);
    size_t const part_bytes = round256(size_t(n_items) * slab * sizeof(fpk::Dbl2));
    unsigned char *base = nullptr;
    unsigned char const *d_tables = nullptr;
    if (ws)
    {
        std::lock_guard<std::mutex> lock(ops->tiles_mu);
        FP_HIP(hipMemcpyAsync(ws->base, tt->h.data(), tt->h.size(), hipMemcpyHostToDevice, st));
        if (!stream_capturing(st)) // the host image may be rebuilt only once this copy has read it
            FP_HIP(hipEventRecord(tt->uploaded, st));
        d_tables = static_cast<unsigned char *>(ws->base);
        base = static_cast<unsigned char *>(ws->base) + table_bytes;
    }
    else
    {
        void *scratch = nullptr;
        s = scratch_get(st, slab_bytes + part_bytes, &scratch);
        if (s == FP_ERR_OUT_OF_MEMORY)
        {
            (void)hipGetLastError();
            return FP_OK; // no room for the slab: the kernels that read the batch as it is
        }
        TileAddr at;
        if (s != FP_OK || (s = tile_device(ops, tt, st, &at)) != FP_OK)
            return s;
        d_tables = at.base;
        base = static_cast<unsigned char *>(scratch);
    }
    auto *partial = reinterpret_cast<fpk::Dbl2 *>(base + slab_bytes);
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute(reinterpret_cast<void const *>(&fpc::k_ev_columns<double>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, int(fpc::kTileBytes));
        hipError_t const e = hipFuncSetAttribute(reinterpret_cast<void const *>(&fpc::k_ev_columns<float>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(fpc::kTileBytes));
        attr = attr == hipSuccess ? e : attr;
    });
    if (attr != hipSuccess)
        return fail(FP_ERR_RUNTIME, "hipFuncSetAttribute failed: %s", hipGetErrorString(attr));
    auto run = [&](auto T_tag) -> fp_status {
        typedef decltype(T_tag) T;
        typedef typename fpk::VecOf<T, 1>::type V;
        typedef typename fpc::Piece<T>::type P;
        for (size_t c0 = 0; c0 < n_states; c0 += slab)
        {
            uint32_t const nc = uint32_t(std::min<size_t>(slab, n_states - c0));
            P const *cols = static_cast<P const *>(states);
            if (!in_place)
            {
                launch_columns<T, 1, true>(const_cast<V *>(static_cast<V const *>(states)),
                                           reinterpret_cast<V *>(base), dim, n_states, c0, nc, st);
                FP_LAUNCHED();
                cols = reinterpret_cast<P const *>(base);
            }
            uint32_t const groups = (nc + g.per_group - 1) / g.per_group;
            uint64_t const blocks = uint64_t(n_items) * groups;
            hipLaunchKernelGGL(fpc::k_ev_columns<T>, dim3(uint32_t(blocks)), dim3(fpc::kThreads), fpc::kTileBytes, st,
                               cols, uint32_t(ops->n_qubits), nc, n_items, groups,
                               reinterpret_cast<fpc::ColItem const *>(d_tables),
                               reinterpret_cast<fpc::ColEntry const *>(d_tables + tt->o_chunks),
                               reinterpret_cast<fpc::ColStr const *>(d_tables + tt->o_strs), partial);
            FP_LAUNCHED();
            hipLaunchKernelGGL(fpk::k_reduce_partials<T>, dim3(nc), dim3(fpk::kBlock), 0, st, partial,
                               uint64_t(n_items), uint64_t(nc), static_cast<T *>(out) + 2 * c0, accumulate, 1.0, 0.0);
            FP_LAUNCHED();
        }
        return FP_OK;
    };
    s = dtype == FP_C128 ? run(double{}) : run(float{});
    *done = s == FP_OK;
    return s;
}

// ---------------------------------------------------------------------------
// Apply on columns
// ---------------------------------------------------------------------------

namespace
{

// Configurations of k_apply_columns: one row a thread and four or eight partner rows in flight,
// straight from the column; or 2^13-row tiles in LDS, eight rows a thread.
template <class T, int NS, bool WTD>
fp_status launch_apply_columns(void const *cols, void *out, uint32_t n, uint32_t n_cols, uint32_t n_states,
                               uint32_t const *xs, uint32_t const *zs, T const *cf, uint64_t cf_stride,
                               uint32_t n_strings, uint32_t shift, int accumulate, bool lds, hipStream_t st)
{
    typedef typename fpk::VecOf<T, NS>::type V;
    auto go = [&](auto e_tag, auto u_tag, auto th_tag, auto lds_tag) -> fp_status {
        constexpr int E = decltype(e_tag)::value, U = decltype(u_tag)::value, TH = decltype(th_tag)::value;
        constexpr bool LDS = decltype(lds_tag)::value;
        constexpr uint32_t kTile = 6u + fpc::log2c(E) + fpc::log2c(TH / 64);
        constexpr size_t kLds = LDS ? sizeof(V) * E * TH : 0;
        // rows in flight: complex128 one batch ahead, complex64, whose terms take half the time, two
        // (n = 16, one state, 500 strings: 20.1 us with one, 17.7 with two; complex128 19.3 / 23.2)
        constexpr int D = LDS ? 1 : sizeof(T) == 4 && !WTD ? 3 : 2;
        auto const kfn = &fpc::k_apply_columns<T, NS, E, U, TH, LDS, D, WTD>;
        if constexpr (LDS)
        {
            static std::once_flag once;
            static hipError_t attr = hipSuccess;
            static hipFuncAttributes fa{};
            std::call_once(once, [&] {
                attr = hipFuncSetAttribute(reinterpret_cast<void const *>(kfn),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds));
                if (attr == hipSuccess)
                    attr = hipFuncGetAttributes(&fa, reinterpret_cast<void const *>(kfn));
            });
            if (attr != hipSuccess)
                return fail(FP_ERR_RUNTIME, "apply kernel attributes: %s", hipGetErrorString(attr));
            if (fa.sharedSizeBytes != 0)
                return fail(FP_ERR_RUNTIME, "the apply kernel's tile does not start its LDS: %zu static bytes",
                            fa.sharedSizeBytes);
        }
        uint32_t const tiles = n > kTile ? 1u << (n - kTile) : 1u, per = n < kTile ? 1u << (kTile - n) : 1u;
        uint32_t const groups = (n_cols + per - 1) / per;
        hipLaunchKernelGGL(kfn, dim3(tiles * groups), dim3(TH), kLds, st, static_cast<V const *>(cols),
                           static_cast<V *>(out), n, n_cols, groups, tiles, xs, zs, cf, cf_stride, n_states, n_strings,
                           shift, accumulate);
        FP_LAUNCHED();
        return FP_OK;
    };
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 4> I4;
    typedef std::integral_constant<int, 8> I8;
    typedef std::integral_constant<int, 256> I256;
    typedef std::integral_constant<int, 1024> I1024;
    return lds ? go(I8{}, I1{}, I1024{}, std::true_type{}) : go(I1{}, I4{}, I256{}, std::false_type{});
}

// The LDS tiles (one block per CU): columns of 2^9 to 2^14 rows, at least half of whose partner
// rows they hold, when whole rounds of them fill the chip.  us, LDS / direct: complex128, 500
// strings, 1000 states n = 14 3180 / 4310, n = 12 716 / 1061, n = 14 300 states (600 tiles) 1131 /
// 1300; but complex64 n = 14, 300 states (300 tiles) 816 / 670, and beyond, complex128 n = 18,
// 30 states 2880 / 2520 (13 states 1575 / 1180, complex64 1630 / 846).
bool apply_lds_tiles(uint32_t n, uint64_t n_cols)
{
    uint64_t const tiles = n > 13 ? n_cols << (n - 13) : n_cols >> (13 - n);
    uint64_t const rounds = (tiles + 255) / 256;
    return n >= 9 && n <= 14 && tiles >= 192 && 10 * tiles >= 7 * 256 * rounds &&
           lds_bytes() >= (size_t(1) << 17);
}

} // namespace

// How an apply runs: 0 on the row-major batch (streaming or coset-tiled kernels), 1 as one
// column made of the whole batch, 2 on transposed columns.
//  1: a power-of-two state count (weighted: one state, whose weights are then one row) and a
//     batch of at most 8 MiB (one state: 32 MiB), which the L2s and the Infinity Cache serve;
//     beyond 4 MiB from 64 strings (n = 20, one complex128 state: N = 24 41.6 us streaming /
//     45.9, N = 64 113 / 112).  Below it from 2 strings, where both forms are one launch (n = 14,
//     16 states: N = 2 3.6 / 3.6, N = 8 4.2 / 3.8, N = 16 6.4 / 5.2), but weighted from 8 (n = 14:
//     N = 2..5 6.8 / 7.2, N = 8 7.6 / 7.3), and one complex64 state past 2 MiB, whose rows are 8
//     bytes, from 16 (n = 19: N = 2 3.3 / 4.1, N = 12 5.6 / 6.5, N = 16 6.8 / 6.6, N = 24 10.9 /
//     9.4; n = 18: N = 12 4.0 / 4.2, N = 24 6.3 / 5.5).  us, streaming / column: n = 10, 128 states,
//     64 strings 18.6 / 8.1; n = 18, one state, 1000 strings 287 / 141.
//  2: columns of at most 4 MiB (an XCD's L2), 8 MiB where the state count is not a power of two
//     (the coset-tiled kernel is then at its slowest); enough work to pay the two transposed
//     copies: from 32 strings and 3e7 (string, element) terms.  us, streaming or tiled / columns:
//     n = 14, 1000 complex128 states, 500 strings 8500 / 3160; n = 20, 19 complex64 states, 512
//     strings 10990 / 5640; but n = 12, 100 complex64 states, 64 strings (2.6e7 terms) 16.2 / 21.3
//     and n = 20, 16 complex64 states, 64 strings 619 / 733.
//     Weighted, whose row-major form reads a weight per string and element: also from 48 strings
//     on fewer than 2^19 elements.  n = 10, 2 states, 89 strings 43.8 / 17.2; n = 12, 100 states, 48
//     strings 42.7 / 36.7; n = 9, 50 states, 200 strings 122 / 45; but n = 9, 2 states, 32 strings,
//     200 operators 37.7 / 49.7 and n = 18, 2 states, 40 strings 30.4 / 42.2.
// FAST_PAULI_APPLY_KERNEL=columns forces 1 or 2 where the shape allows, other values forbid them.
int apply_columns_route(fp_hip_ops const *ops, int dtype, size_t n_states, bool weighted)
{
    size_t const n = ops->n_qubits, N = ops->n_strings, esz = dtype == FP_C128 ? 16 : 8;
    if (N < 2 || n > 24 || n_states > (size_t(1) << 24))
        return 0;
    char const *v = std::getenv("FAST_PAULI_APPLY_KERNEL");
    bool const forced = v && std::strcmp(v, "columns") == 0;
    if (v && *v && !forced)
        return 0;
    size_t const elements = (size_t(1) << n) * n_states;
    bool const pow2 = (n_states & (n_states - 1)) == 0;
    size_t const bytes = elements * esz;
    if (pow2 && (!weighted || n_states == 1) && elements >= 64 &&
        bytes <= (n_states == 1 ? size_t(32) << 20 : size_t(8) << 20))
    {
        size_t const narrow = dtype != FP_C128 && n_states == 1 && bytes > (size_t(2) << 20) ? 16 : 2;
        if (forced || N >= (bytes > (size_t(4) << 20) ? 64 : std::max<size_t>(narrow, weighted ? 8 : 2)))
            return 1;
    }
    size_t const col_bytes = (size_t(1) << n) * esz;
    if (n < 6 || col_bytes > (size_t(8) << 20))
        return 0;
    if (forced)
        return 2;
    if (col_bytes > (size_t(4) << 20) && pow2)
        return 0;
    if (weighted && N >= 48 && elements < (size_t(1) << 19))
        return 2;
    return N >= 32 && double(N) * double(elements) >= 3e7 ? 2 : 0;
}

fp_status run_apply_columns(fp_hip_ops const *ops, int dtype, int kind, void const *states, void const *data,
                            void *out, size_t dim, size_t n_states, int accumulate, hipStream_t st, bool *done)
{
    *done = false;
    bool const weighted = kind == kTilesWeightedApply, c64 = dtype != FP_C128;
    int const route = apply_columns_route(ops, dtype, n_states, weighted);
    if (route == 0 || ((route == 2 || weighted) && stream_capturing(st)))
        return FP_OK;
    uint32_t const n = uint32_t(ops->n_qubits), N = uint32_t(ops->n_strings);
    size_t const esz = c64 ? 8 : 16;
    uint32_t const *xs = ops->d_x32, *zs = ops->d_z32;
    bool const aligned16 = ((reinterpret_cast<uintptr_t>(states) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    // scratch: [transposed states | transposed outputs | weights]
    bool const pairs = c64 && n <= 18 && n_states > 1;
    uint32_t const ns = pairs ? 2u : 1u;
    size_t const col_bytes = dim * esz * ns;
    size_t const all_cols = (n_states + ns - 1) / ns;
    size_t cols = route == 2 ? std::max<size_t>(1, std::min(kSlabBytes / col_bytes, all_cols)) : 0;
    if (cols < all_cols && cols >= 8)
        cols = cols / 8 * 8; // as many columns on every XCD
    size_t const slab = round256(cols * col_bytes);
    size_t const w_bytes = weighted ? round256(n_states * size_t(N) * esz + fpc::kXzPad * esz) : 0;
    unsigned char *base = nullptr;
    std::unique_ptr<StreamGuard> guard; // held until the kernels that use the scratch are enqueued
    if (2 * slab + w_bytes > 0)
    {
        guard = std::make_unique<StreamGuard>(st);
        void *scratch = nullptr;
        fp_status const s = scratch_get(st, 2 * slab + w_bytes, &scratch);
        if (s == FP_ERR_OUT_OF_MEMORY)
        {
            (void)hipGetLastError();
            return FP_OK; // no room: the kernels that read the batch as it is
        }
        if (s != FP_OK)
            return s;
        base = static_cast<unsigned char *>(scratch);
    }
    auto run = [&](auto T_tag, auto const *coef) -> fp_status {
        typedef decltype(T_tag) T;
        typedef typename fpk::VecOf<T, 1>::type V1;
        T *w = nullptr;
        if (weighted)
        {
            w = reinterpret_cast<T *>(base + 2 * slab);
            constexpr int R = 8;
            dim3 const grid(uint32_t((n_states + 255) / 256), (N + R - 1) / R);
            hipLaunchKernelGGL((fpc::k_weights<T, R>), grid, dim3(256), 0, st, coef, static_cast<T const *>(data),
                               ops->d_ny, w, uint64_t(N), uint64_t(ops->n_operators), uint64_t(n_states));
            FP_LAUNCHED();
        }
        if (route == 1)
        {
            uint32_t shift = 0;
            while ((size_t(1) << shift) < n_states)
                ++shift;
            // complex64: two states a row where that leaves enough waves
            bool const two = c64 && shift > 0 && aligned16 && dim * n_states >= (size_t(1) << 19);
            if constexpr (sizeof(T) == 4)
                if (two)
                    return launch_apply_columns<T, 2, false>(states, out, n + shift - 1, 1, 1, xs, zs, coef, 0, N,
                                                             shift - 1, accumulate, false, st);
            return weighted ? launch_apply_columns<T, 1, true>(states, out, n, 1, 1, xs, zs, w, N, N, 0, accumulate,
                                                               false, st)
                            : launch_apply_columns<T, 1, false>(states, out, n + shift, 1, 1, xs, zs, coef, 0, N, shift,
                                                                accumulate, false, st);
        }
        auto slabs = [&](auto ns_tag) -> fp_status {
            constexpr int NS = decltype(ns_tag)::value;
            typedef typename fpk::VecOf<T, NS>::type V;
            auto *ic = reinterpret_cast<V *>(base), *oc = reinterpret_cast<V *>(base + slab);
            for (size_t c0 = 0; c0 < n_states; c0 += cols * NS)
            {
                uint32_t const nst = uint32_t(std::min<size_t>(cols * NS, n_states - c0));
                uint32_t const nc = (nst + NS - 1) / NS;
                launch_columns<T, NS, true>(const_cast<V1 *>(static_cast<V1 const *>(states)), ic, dim, n_states, c0,
                                            nst, st);
                if (accumulate)
                    launch_columns<T, NS, true>(static_cast<V1 *>(out), oc, dim, n_states, c0, nst, st);
                FP_LAUNCHED();
                bool const lds = apply_lds_tiles(n, nc);
                fp_status const s =
                    weighted ? launch_apply_columns<T, NS, true>(ic, oc, n, nc, nst, xs, zs, w + 2 * c0 * N, N, N, 0,
                                                                 accumulate, lds, st)
                             : launch_apply_columns<T, NS, false>(ic, oc, n, nc, nst, xs, zs, coef, 0, N, 0, accumulate,
                                                                  lds, st);
                if (s != FP_OK)
                    return s;
                launch_columns<T, NS, false>(static_cast<V1 *>(out), oc, dim, n_states, c0, nst, st);
                FP_LAUNCHED();
            }
            return FP_OK;
        };
        if constexpr (sizeof(T) == 4)
            if (pairs)
                return slabs(std::integral_constant<int, 2>{});
        return slabs(std::integral_constant<int, 1>{});
    };
    fp_status s;
    if (dtype == FP_C128)
        s = run(double{}, weighted ? ops->d_h128 : kind == kTilesSummedApply ? ops->d_rowsum128 : ops->d_cf128);
    else
        s = run(float{}, weighted ? ops->d_h64 : kind == kTilesSummedApply ? ops->d_rowsum64 : ops->d_cf64);
    *done = s == FP_OK;
    return s;
}

// Entries of a batch: columns as in apply_columns_route, but from 16 strings and 64 KiB of states,
// as the copies and launches are shared.  256 complex64 entries, n = 8..18, 16..512 strings, 1..64
// states, ms: from 32 strings and 4 MiB 26.2, 16 strings and 4 MiB 25.5, 1 MiB 24.2, 256 KiB 23.5,
// 64 KiB 23.25, 16 KiB 23.2; 8 strings and 64 KiB 23.2.
bool batch_columns_eligible(fp_hip_ops const *ops, int dtype, size_t n_states)
{
    size_t const n = ops->n_qubits, esz = dtype == FP_C128 ? 16 : 8;
    char const *v = std::getenv("FAST_PAULI_APPLY_KERNEL");
    if ((v && *v && std::strcmp(v, "columns") != 0) || n < 6 || n > 20 || n_states > (size_t(1) << 24))
        return false;
    size_t const col_bytes = (size_t(1) << n) * esz;
    bool const pow2 = (n_states & (n_states - 1)) == 0;
    return ops->n_strings >= 16 && col_bytes * n_states >= (size_t(64) << 10) &&
           col_bytes <= (pow2 ? size_t(4) << 20 : size_t(8) << 20);
}

namespace
{

// f(type, states a row) for a variant of columns
template <class F> fp_status with_columns(uint32_t variant, F f)
{
    if (!(variant & kColsC64))
        return f(double{}, std::integral_constant<int, 1>{});
    if (variant & kColsPairs)
        return f(float{}, std::integral_constant<int, 2>{});
    return f(float{}, std::integral_constant<int, 1>{});
}

} // namespace

fp_status launch_column_round(ColumnRound const &r, unsigned char const *tables, unsigned char *in,
                              unsigned char *out, hipStream_t st)
{
    auto const *jobs = reinterpret_cast<fpc::ColJob const *>(tables + r.o_jobs);
    auto const *ends = reinterpret_cast<uint32_t const *>(tables + r.o_ends);
    auto const *segs = reinterpret_cast<fpc::ColSeg const *>(tables + r.o_segs);
    auto copies = [&](size_t o) { return reinterpret_cast<fpc::ColCopy const *>(tables + o); };
    auto copy_ends = [&](size_t o) { return reinterpret_cast<uint32_t const *>(tables + o); };
    return with_columns(r.variant, [&](auto T_tag, auto ns_tag) -> fp_status {
        typedef decltype(T_tag) T;
        constexpr int NS = decltype(ns_tag)::value;
        hipLaunchKernelGGL((fpc::k_columns_batch<T, NS, true>), dim3(r.in_blocks), dim3(256), 0, st, in, out,
                           copies(r.o_in), copy_ends(r.o_in_ends), r.n_in);
        FP_LAUNCHED();
        hipLaunchKernelGGL((fpc::k_apply_columns_batch<T, NS>), dim3(r.blocks), dim3(256), 0, st, in, out, jobs, ends,
                           segs, r.n_segs);
        FP_LAUNCHED();
        hipLaunchKernelGGL((fpc::k_columns_batch<T, NS, false>), dim3(r.out_blocks), dim3(256), 0, st, in, out,
                           copies(r.o_out), copy_ends(r.o_out_ends), r.n_out);
        FP_LAUNCHED();
        return FP_OK;
    });
}

} // namespace fprt

extern "C" fp_status fp_hip_op_apply_columns(fp_hip_ops const *ops, int dtype, size_t dim, size_t n_states, int weighted,
                                             int *columns)
{
    if (!ops || !columns)
        return fail(FP_ERR_INVALID_ARGUMENT, "NULL ops or result");
    if (dtype != FP_C128 && dtype != FP_C64)
        return fail(FP_ERR_INVALID_ARGUMENT, "unknown dtype %d", dtype);
    if (n_states == 0 || dim != (size_t(1) << ops->n_qubits))
        return fail(FP_ERR_INVALID_ARGUMENT, "shape (%zu, %zu) does not match %zu qubits", dim, n_states,
                    ops->n_qubits);
    *columns = fprt::apply_columns_route(ops, dtype, n_states, weighted != 0) != 0 ? 1 : 0;
    return FP_OK;
}

extern "C" fp_status fp_hip_op_expectation_columns(fp_hip_ops const *ops, int dtype, size_t dim, size_t n_states,
                                                   int *columns)
{
    if (!ops || !columns)
        return fail(FP_ERR_INVALID_ARGUMENT, "NULL ops or result");
    if (dtype != FP_C128 && dtype != FP_C64)
        return fail(FP_ERR_INVALID_ARGUMENT, "unknown dtype %d", dtype);
    if (n_states == 0 || dim != (size_t(1) << ops->n_qubits))
        return fail(FP_ERR_INVALID_ARGUMENT, "shape (%zu, %zu) does not match %zu qubits", dim, n_states,
                    ops->n_qubits);
    *columns = fprt::ev_columns_eligible(ops, dtype, n_states) ? 1 : 0;
    return FP_OK;
}
