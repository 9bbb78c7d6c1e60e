// fp_columns.hip — host side of the column kernels (fp_columns.hpp): which operators run on
// state columns, the transposed slabs and the launches.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "fast_pauli_hip.h"
#include "fp_columns.hpp"
#include "fp_runtime.hpp"

using fprt::fail;

namespace
{

// Transposed states kept at a time: a slab this size is still in the Infinity Cache
// (256 MB) when the column kernel reads it.
constexpr size_t kSlabBytes = size_t(128) << 20;
// Tiles per column: at most 2^8 (a class pairs every tile with another one).
constexpr uint32_t kMaxTileBits = 8;
constexpr double kTargetItems = 2000.0;

size_t round256(size_t v)
{
    return (v + 255) / 256 * 256;
}

bool capturing(hipStream_t st)
{
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &s) != hipSuccess)
    {
        (void)hipGetLastError();
        return true;
    }
    return s != hipStreamCaptureStatusNone;
}

// Columns per tile of the expectation kernel and columns per slab.
struct ColGeom
{
    uint32_t per_group, slab;
    size_t col_bytes;
};

ColGeom col_geom(fp_hip_ops const *ops, int dtype, size_t n_states, size_t slab_bytes)
{
    bool const c64 = dtype != FP_C128;
    uint32_t const w = fpc::tile_bits(c64), n = uint32_t(ops->n_qubits);
    ColGeom g{};
    g.per_group = n < w ? 1u << (w - n) : 1u;
    g.col_bytes = (size_t(1) << n) * (c64 ? 8u : 16u);
    size_t cols = std::max<size_t>(1, std::min<size_t>(slab_bytes / g.col_bytes, n_states));
    if (cols < n_states) // whole tiles, and as many columns on every XCD
        cols = std::max<size_t>(cols / (8 * g.per_group) * (8 * g.per_group), std::min<size_t>(cols, g.per_group));
    g.slab = uint32_t(std::min<size_t>(cols, 0x7fffffffu));
    return g;
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
    if (!ws && capturing(st)) // the slab may have to be allocated
        return FP_OK;
    // one aligned state is a column already
    bool const in_place = n_states == 1 && (reinterpret_cast<uintptr_t>(states) & 15u) == 0;
    ColGeom const g = col_geom(ops, dtype, n_states, ws ? ws->bytes / 2 : kSlabBytes);
    if (ws && !in_place && g.slab * g.col_bytes > ws->bytes / 2)
        return FP_OK;
    uint32_t const n_groups_max = (g.slab + g.per_group - 1) / g.per_group;
    // String evaluations per item: about kTargetItems blocks (four per resident slot), and at
    // least 16 so that the tile loads of an item are paid by its strings.  Steps of a quarter
    // keep the tables cached per set few.  Measured around it (500 to 6000 blocks wanted):
    // n = 12 S = 100 N = 1024 complex128 72.7 / 64.5 at 1500 / 67.3 at 2000 / 77.5 us at 6000,
    // n = 18 S = 13 N = 300 complex64 156 / 133 / 127 / 125; n = 14 S = 1000 is flat.
    uint32_t const w = fpc::tile_bits(c64), n = uint32_t(ops->n_qubits);
    double const work = double(ops->n_strings) * double(n_groups_max) *
                        (n > w ? 0.5 * double(uint32_t(1) << (n - w)) : 0.6);
    uint32_t per = 16;
    while (per < 256 && work > kTargetItems * per)
        per += per / 4;
    TileTables *tt = nullptr;
    fp_status s = tile_tables(ops, kTilesEvColumns, per, c64 ? 1u : 0u, &tt);
    if (s != FP_OK)
        return s;
    uint32_t const n_items = tt->n_groups;
    // from 4 column groups per XCD: their items stay on one XCD, whose L2 then serves the tiles
    // (n = 16 S = 40 N = 300 complex64: 82 us against 86)
    bool const xcd = n_groups_max >= 32;
    if (uint64_t(n_items) * (n_groups_max + 8) > 0x7fffffffu)
        return FP_OK;
    size_t const slab_bytes = in_place ? 0 : round256(size_t(g.slab) * g.col_bytes);
    size_t const part_bytes = round256(size_t(n_items) * g.slab * sizeof(fpk::Dbl2));
    unsigned char *base = nullptr;
    unsigned char const *d_tables = nullptr;
    if (ws)
    {
        size_t const table_bytes = round256(tt->h.size());
        if (table_bytes + slab_bytes + part_bytes > ws->bytes)
            return FP_OK;
        std::lock_guard<std::mutex> lock(ops->tiles_mu);
        FP_HIP(hipMemcpyAsync(ws->base, tt->h.data(), tt->h.size(), hipMemcpyHostToDevice, st));
        FP_HIP(hipEventRecord(tt->uploaded, st)); // the host image may be rebuilt only once this copy has read it
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
        if (s != FP_OK || (s = tile_device(ops, tt, st)) != FP_OK)
            return s;
        d_tables = static_cast<unsigned char const *>(tt->d_mem);
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
        for (size_t c0 = 0; c0 < n_states; c0 += g.slab)
        {
            uint32_t const nc = uint32_t(std::min<size_t>(g.slab, n_states - c0));
            P const *cols = static_cast<P const *>(states);
            if (!in_place)
            {
                dim3 const tg(uint32_t((dim + 31) / 32), (nc + 31) / 32);
                hipLaunchKernelGGL(fpc::k_columns_in<V>, tg, dim3(256), 0, st, static_cast<V const *>(states),
                                   reinterpret_cast<V *>(base), uint64_t(dim), uint64_t(n_states), uint64_t(c0), nc);
                FP_LAUNCHED();
                cols = reinterpret_cast<P const *>(base);
            }
            uint32_t const groups = (nc + g.per_group - 1) / g.per_group;
            uint64_t const blocks = uint64_t(n_items) * (xcd ? (groups + 7) / 8 * 8 : groups);
            hipLaunchKernelGGL(fpc::k_ev_columns<T>, dim3(uint32_t(blocks)), dim3(fpc::kThreads), fpc::kTileBytes, st,
                               cols, uint32_t(ops->n_qubits), nc, n_items, groups, xcd ? 1 : 0,
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

} // namespace fprt

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
