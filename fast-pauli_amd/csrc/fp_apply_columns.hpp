// fp_apply_columns.hpp — PauliOp::apply (and SummedPauliOp::apply / apply_weighted) on state
// columns, bit-exact with the sequential string order.
//
// A column is a contiguous array of 2^n rows of one state (complex64: of two neighbouring
// states, 16 bytes a row): a transposed copy of the batch, or the batch itself when its row
// length is a power of two (a row-major batch of 2^k states is one column of 2^(n + k) rows on
// which every mask is shifted by k).  Each thread owns E rows, 64 apart, keeps their sums in
// registers and adds the strings in order, so every element sees the sequential loop's
// operations (cmul_exact, one rounding per sum) in its order: one launch for all strings, the
// column read once per string from L2 or LDS and written once.
//
// The partner of row (g, i, lane) (wave, slot, lane parts) is (g ^ x_g, i ^ x_i, lane ^ x_l):
// a per-lane offset (one XOR per string), a scalar offset per slot.  The sign is a per-lane bit,
// a wave-uniform bit and one flip per slot, applied as the factor of the final multiply-add.
//
// Bound: 10 (LDS) to 12 vector instructions per (string, 64 rows), 8 of them the unfused product
// and sums, against 16 clocks of L1 for a gathered KiB (64 bytes a clock; 4 clocks from LDS) and
// the scalar unit, which all four SIMDs share: whole rounds of strings run without a branch, on
// structure-of-arrays masks (wide scalar loads), and with one row a thread only a shift a string
// is scalar.  Tests between the strings and masks split by scalar instructions made every wave
// wait for its loads (n = 16, one complex128 state, 500 strings 40.6 us, now 19.3; n = 10, 128
// states, 64 strings 10.9, now 8.1; n = 18, 13 complex64 states, 300 strings 524, now 397).  Two
// shapes are built: one row a thread, partner rows gathered from L2 four or eight strings ahead;
// and 2^13 rows a block in LDS (fp_columns.hip says which runs where).  By its counters: n = 18,
// one complex128 state, L1 76 % and vector issue 57 % busy; n = 14 with weights, from LDS,
// vector issue 81 %; n = 20 complex64, half of the gathers miss the L2, whose 4 MiB hold half of
// a column.  Measured, row-major kernels / columns, us: n = 10, 128 complex128 states, 64
// strings 18.6 / 8.1; n = 18, one complex128 state, 1000 strings 287 / 141; n = 20, 19 complex64
// states, 512 strings 10990 / 5640; n = 14, 1000 complex128 states, 2000 strings, a weight per
// string and state 29130 / 10930.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fp_columns.hpp"
#include "fp_kernels.hpp"

namespace fpc
{

// A uniform pointer held in scalar registers (the compiler cannot always tell).
template <class P> __device__ __forceinline__ P const *uniform(P const *p)
{
    uint64_t const v = reinterpret_cast<uint64_t>(p);
    uint32_t const lo = __builtin_amdgcn_readfirstlane(uint32_t(v));
    uint32_t const hi = __builtin_amdgcn_readfirstlane(uint32_t(v >> 32));
    return reinterpret_cast<P const *>((uint64_t(hi) << 32) | lo);
}

// Buffer over one column of `rows` pieces; reads past its end return zero.
template <class V> __device__ __forceinline__ __amdgpu_buffer_rsrc_t column_rsrc(V const *col, uint64_t rows)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<V *>(uniform(col)), short(0),
                                             int(uint32_t(rows * sizeof(V))), 0x00027000);
}

template <class V> __device__ __forceinline__ V buffer_load(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff)
{
    if constexpr (sizeof(V) == 16)
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, int(voff), int(soff), 0));
    else
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rsrc, int(voff), int(soff), 0));
}

// +-1 with the sign in bit 31 of `bits` (other bits clear)
template <class T> __device__ __forceinline__ T unit_sign(uint32_t bits)
{
    if constexpr (sizeof(T) == 8)
        return __hiloint2double(int(bits | 0x3ff00000u), 0);
    else
        return __uint_as_float(bits | 0x3f800000u);
}
// v with its sign flipped by bit 31 of `bits`
template <class T> __device__ __forceinline__ T flip(T v, uint32_t bits)
{
    if constexpr (sizeof(T) == 8)
        return __hiloint2double(__double2hiint(v) ^ int(bits), __double2loint(v));
    else
        return __uint_as_float(__float_as_uint(v) ^ bits);
}

constexpr uint32_t log2c(uint32_t v)
{
    return v <= 1 ? 0 : 1 + log2c(v / 2);
}

// Records read past the last string (the tables are padded by as many).
constexpr uint32_t kXzPad = 64;

// Constant memory: uniform reads are scalar loads, also through pointers that come from a table.
template <class P> using Const = __attribute__((address_space(4))) P const;

// One block's part of an apply: group bo.group, tile bo.index of n_cols columns of 2^n rows
// (cols to out), NS states a row.  A block of TH threads owns a tile of TH * E rows of a column,
// or the columns that fill it.
// LDS: the tile's rows are kept in LDS, and strings whose partner rows lie in it read them there.
// D: partner rows of D - 1 batches of U strings are in flight while one batch is added.
// cf: complex coefficients with (-i)^{nY} folded in; WTD: those of state t at cf + 2 * cf_stride * t.
// shift: masks are shifted by this many bits (one column made of a whole batch).
template <class T, int NS, int E, int U, int TH, bool LDS, int D, bool WTD>
__device__ __forceinline__ void apply_columns(BlockOf bo, typename fpk::VecOf<T, NS>::type const *__restrict__ cols,
                                              typename fpk::VecOf<T, NS>::type *__restrict__ out, uint32_t n,
                                              uint32_t n_cols, Const<uint32_t> *xs, Const<uint32_t> *zs, Const<T> *cf, uint64_t cf_stride,
                                              uint32_t n_states, uint32_t n_strings, uint32_t shift, int accumulate)
{
    typedef typename fpk::VecOf<T, NS>::type V; // one row of NS states
    constexpr uint32_t kLe = log2c(E), kLv = log2c(sizeof(V));
    constexpr uint32_t kLow = 6u + kLe;                // row bits inside a wave
    constexpr uint32_t kTile = kLow + log2c(TH / 64u); // log2 rows of a tile
    constexpr uint32_t kSlot = 64u * sizeof(V);        // bytes from one slot to the next
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t const lane = threadIdx.x & 63u;
    uint32_t const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t const grp = bo.group, p = bo.index;
    uint32_t const per = n < kTile ? 1u << (kTile - n) : 1u; // columns in a tile
    uint64_t const rows = uint64_t(1) << n;
    uint32_t const t = grp * per + (n < kTile ? (wave << kLow) >> n : 0u);
    if (!LDS && t >= n_cols)
        return;
    bool const live = t < n_cols; // a ragged last group has dead waves
    uint32_t const tc = live ? t : n_cols - 1u;
    V const *col = cols + uint64_t(tc) * rows;
    // this thread's rows of the column: row0 + 64 i
    uint32_t const g = n < kTile ? wave & ((1u << (n - kLow)) - 1u) : (p << (kTile - kLow)) | wave; // row >> kLow
    uint32_t const row0 = (g << kLow) | lane;
    V *oc = out + uint64_t(tc) * rows + row0;
    // LDS address of slot 0: the tile starts the workgroup's LDS, as the kernel has no static shared
    // arrays (the launch checks it; adding the tile's address instead costs an instruction a read)
    uint32_t const a0 = ((wave << kLow) | lane) << kLv;
    if constexpr (LDS)
    {
#pragma unroll
        for (int i = 0; i < E; ++i)
            *reinterpret_cast<V *>(smem + a0 + uint32_t(i) * kSlot) = col[row0 + uint32_t(i) * 64u];
    }
    V acc[E];
#pragma unroll
    for (int i = 0; i < E; ++i)
        acc[i] = accumulate && live ? oc[i * 64] : V(0);
    if constexpr (LDS)
        __syncthreads();
    // WTD: the coefficients of this column's states (the last state again past the end)
    Const<T> *c[WTD ? NS : 1];
#pragma unroll
    for (int w = 0; w < (WTD ? NS : 1); ++w)
        c[w] = cf + 2 * cf_stride * (WTD ? (tc * NS + w < n_states ? tc * NS + w : n_states - 1u) : 0u);
    __amdgpu_buffer_rsrc_t const rsrc = column_rsrc(col, rows);
    uint32_t const lv = lane << kLv, gv = g << (kLow + kLv);
    uint32_t const rv = row0 << kLv, rz = row0 >> shift; // one row a thread: its offset, its bits for z
    // Batches of U strings in a pipeline: while batch k is added, the partner rows of the next
    // D - 1 batches are in flight, and the scalar loads of x for batch k + D and of z and the
    // coefficients for k + 1.  Masks and coefficients are read past the end (the tables are
    // padded), and rows with them (inside the column, or zero), but add nothing.
    constexpr int Q = D == 3 ? 3 : 2; // batches a round, and buffers of scalars
    uint32_t x[Q][U], z[Q][U];
    T cr[Q][U][WTD ? NS : 1], ci[Q][U][WTD ? NS : 1];
    V R[D][U][E];
    auto fetch_x = [&](int k, uint32_t(&v)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            v[u] = xs[k * U + u];
    };
    auto fetch_c = [&](int k, uint32_t(&v)[U], T(&r)[U][WTD ? NS : 1], T(&i)[U][WTD ? NS : 1]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            v[u] = zs[k * U + u];
#pragma unroll
            for (int w = 0; w < (WTD ? NS : 1); ++w)
            {
                r[u][w] = c[w][2 * (k * U + u)];
                i[u][w] = c[w][2 * (k * U + u) + 1];
            }
        }
    };
    auto load = [&](uint32_t const(&xv)[U], V(&v)[U][E]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            // one row a thread: its whole offset in a vector register (one scalar instruction a
            // string; the lane and wave parts take several, which E rows share)
            if constexpr (E == 1)
                v[u][0] = buffer_load<V>(rsrc, rv ^ (xv[u] << (shift + kLv)), 0);
            else if (uint32_t const xu = xv[u] << shift; LDS && (xu >> kTile) == 0)
            {
                uint32_t const a = a0 ^ (xu << kLv);
#pragma unroll
                for (int i = 0; i < E; ++i)
                    v[u][i] =
                        *reinterpret_cast<__attribute__((address_space(3))) V const *>(a ^ (uint32_t(i) * kSlot));
            }
            else
            {
                uint32_t const vo = lv ^ ((xu & 63u) << kLv), so = gv ^ ((xu >> 6) << (6u + kLv));
#pragma unroll
                for (int i = 0; i < E; ++i)
                    v[u][i] = buffer_load<V>(rsrc, vo, so ^ (uint32_t(i) * kSlot));
            }
        }
    };
    auto eval = [&](uint32_t count, uint32_t const(&zv)[U], T const(&r)[U][WTD ? NS : 1],
                    T const(&im)[U][WTD ? NS : 1], V(&v)[U][E]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (uint32_t(u) < count)
            {
                // sign of the row: per-lane bits, wave-uniform bits, then one flip per slot
                uint32_t const zu = zv[u] << shift;
                uint32_t const neg = E == 1 ? uint32_t(__popc(rz & zv[u]))
                                            : uint32_t(__popc(lane & zu)) + uint32_t(__popc(g & (zu >> kLow)));
                uint32_t zb[kLe + 1];
#pragma unroll
                for (uint32_t b = 0; b < kLe; ++b)
                    zb[b] = (zu << (25u - b)) & 0x80000000u;
                T sg = unit_sign<T>(neg << 31);
                // slots in Gray-code order: one sign flip from each to the next
#pragma unroll
                for (int j = 0; j < E; ++j)
                {
                    int const i = j ^ (j >> 1);
                    if (j)
                        sg = flip<T>(sg, zb[__builtin_ctz(uint32_t(j))]);
#pragma unroll
                    for (int h = 0; h < NS; ++h)
                    {
                        // the signed term: products and their sum rounded as cmul_exact does, then
                        // one rounding in the sum, which a multiply-add by +-1 gives exactly
                        int const w = WTD ? h : 0;
                        T tr, ti;
                        fpk::cmul_exact<T>(r[u][w], im[u][w], v[u][i][2 * h], v[u][i][2 * h + 1], tr, ti);
                        acc[i][2 * h] = fma(sg, tr, acc[i][2 * h]);
                        acc[i][2 * h + 1] = fma(sg, ti, acc[i][2 * h + 1]);
                    }
                }
            }
    };
    auto step = [&](int k) {
        fetch_c(k + 1, z[(k + 1) % Q], cr[(k + 1) % Q], ci[(k + 1) % Q]);
        fetch_x(k + D, x[(k + D) % Q]);
        load(x[(k + D - 1) % Q], R[(k + D - 1) % D]);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int k = 0; k < D - 1; ++k)
    {
        fetch_x(k, x[0]);
        load(x[0], R[k]);
    }
    fetch_x(D - 1, x[(D - 1) % Q]);
    fetch_c(0, z[0], cr[0], ci[0]);
    uint32_t left = n_strings;
    for (; left >= uint32_t(Q * U); left -= Q * U) // whole rounds: no tests inside
    {
#pragma unroll
        for (int k = 0; k < Q; ++k)
        {
            step(k);
            eval(U, z[k % Q], cr[k % Q], ci[k % Q], R[k % D]);
            __builtin_amdgcn_sched_barrier(0);
        }
        xs += Q * U;
        zs += Q * U;
#pragma unroll
        for (int w = 0; w < (WTD ? NS : 1); ++w)
            c[w] += 2 * Q * U;
    }
#pragma unroll
    for (int k = 0; k < Q; ++k)
    {
        if (left <= uint32_t(k * U))
            break;
        step(k);
        eval(left - uint32_t(k * U), z[k % Q], cr[k % Q], ci[k % Q], R[k % D]);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < E; ++i)
        if (live)
            __builtin_nontemporal_store(acc[i], oc + i * 64);
}

// One operator on n_cols columns: n_groups * tiles blocks.
template <class T, int NS, int E, int U, int TH, bool LDS, int D, bool WTD>
__global__ __launch_bounds__(TH) void k_apply_columns(typename fpk::VecOf<T, NS>::type const *__restrict__ cols,
                                                      typename fpk::VecOf<T, NS>::type *__restrict__ out, uint32_t n,
                                                      uint32_t n_cols, uint32_t n_groups, uint32_t tiles,
                                                      uint32_t const *__restrict__ xs, uint32_t const *__restrict__ zs, T const *__restrict__ cf,
                                                      uint64_t cf_stride, uint32_t n_states, uint32_t n_strings, uint32_t shift,
                                                      int accumulate)
{
    apply_columns<T, NS, E, U, TH, LDS, D, WTD>(block_of(blockIdx.x, tiles, n_groups), cols, out, n, n_cols,
                                                   (Const<uint32_t> *)xs, (Const<uint32_t> *)zs, (Const<T> *)cf, cf_stride, n_states, n_strings,
                                                   shift, accumulate);
}

// Index of the first of `count` ascending ends that `pos` lies below, else >= count.  `ends` is
// padded with its last entry to a multiple of 64: one load and a ballot for 64 of them.
__device__ __forceinline__ uint32_t find_segment(uint32_t const *ends, uint32_t count, uint32_t pos)
{
    for (uint32_t base = 0; base < count; base += 64)
    {
        uint32_t const below = uint32_t(__popcll(__ballot(pos >= ends[base + (threadIdx.x & 63u)])));
        if (below < 64)
            return base + below;
    }
    return count;
}

// Many operators on columns of one slab (byte offsets into `in` and `out`): XCD k (blockIdx % 8)
// works through its own n_segs segments, so the blocks of a column follow each other on one XCD
// and every XCD gets the same number of string terms, whatever the operators' sizes.  One row a
// thread, straight from the columns: 256 complex64 operators of n = 8..18 (3 GB of states, 5.5e10
// terms) take 18.0 ms, 57.3 as streaming items and coset-tiled launches; LDS tiles
// made it 4.4 ms slower for n = 9..14 and 18 (0.3 ms for n = 9..14, whose blocks are too few to
// fill their rounds).
template <class T, int NS>
__global__ __launch_bounds__(256) void k_apply_columns_batch(unsigned char const *__restrict__ in,
                                                             unsigned char *__restrict__ out,
                                                             ColJob const *__restrict__ jobs,
                                                             uint32_t const *__restrict__ ends,
                                                             ColSeg const *__restrict__ segs, uint32_t n_segs)
{
    typedef typename fpk::VecOf<T, NS>::type V;
    constexpr uint32_t kTile = 8; // log2 rows of a block
    uint32_t const xcd = blockIdx.x & 7u, pos = blockIdx.x >> 3;
    uint32_t const at = __builtin_amdgcn_readfirstlane(find_segment(ends + xcd * n_segs, n_segs, pos));
    if (at >= n_segs)
        return;
    ColSeg const sg = segs[xcd * n_segs + at];
    ColJob const j = jobs[sg.job];
    uint32_t const b = sg.block0 + (pos - sg.start);
    uint32_t const lt = j.n > kTile ? j.n - kTile : 0u; // log2 tiles of a column
    apply_columns<T, NS, 1, 4, 256, false, 2, false>(
        BlockOf{b >> lt, b & ((1u << lt) - 1u)}, reinterpret_cast<V const *>(in + j.cols),
        reinterpret_cast<V *>(out + j.cols), j.n, j.n_cols, (Const<uint32_t> *)j.xs, (Const<uint32_t> *)j.zs, (Const<T> *)j.cf, 0, 0, j.n_strings, 0,
        int(j.accumulate));
}

// The copies of a slab's columns in (from the states, and from outputs that are added to) or out.
template <class T, int NS, bool IN>
__global__ __launch_bounds__(256) void k_columns_batch(unsigned char *__restrict__ in, unsigned char *__restrict__ out,
                                                       ColCopy const *__restrict__ copies,
                                                       uint32_t const *__restrict__ ends, uint32_t n_copies)
{
    typedef typename fpk::VecOf<T, 1>::type V1;
    typedef typename fpk::VecOf<T, NS>::type V;
    uint32_t const at = __builtin_amdgcn_readfirstlane(find_segment(ends, n_copies, blockIdx.x));
    if (at >= n_copies)
        return;
    ColCopy const c = copies[at];
    uint32_t const b = blockIdx.x - c.start, lb = c.n > 5u ? c.n - 5u : 0u; // log2 blocks of 32 rows
    move_columns<T, NS, IN>((__attribute__((address_space(1))) V1 *)c.batch,
                            reinterpret_cast<V *>((c.out ? out : in) + c.cols), uint64_t(1) << c.n, c.ld, c.c0,
                            c.n_states, b & ((1u << lb) - 1u), b >> lb);
}

// w(s, t) = sum_k h(s, k) x(k, t), k in order, product then add (no contraction: the reference's
// sequential loop, fast_pauli/cpp/include/__summed_pauli_op.hpp:378-503), times (-i)^{nY_s} (an
// exact swap and negation), one row of n_strings per state.  A thread takes one state and R
// strings, whose h are scalar loads: x is read once for R sums (one string a thread read it N
// times: 406 us at 2000 strings, 200 operators, 1000 states).
template <class T, int R>
__global__ __launch_bounds__(256) void k_weights(T const *__restrict__ h, T const *__restrict__ x,
                                                 uint32_t const *__restrict__ nys, T *__restrict__ w,
                                                 uint64_t n_strings, uint64_t n_ops, uint64_t n_states)
{
#pragma clang fp contract(off)
    uint64_t const t = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    uint64_t const s0 = uint64_t(blockIdx.y) * R;
    if (t >= n_states)
        return;
    T wr[R], wi[R];
    T const *hp[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
    {
        wr[r] = wi[r] = T(0);
        hp[r] = h + 2 * n_ops * (s0 + r < n_strings ? s0 + r : n_strings - 1);
    }
    for (uint64_t k = 0; k < n_ops; ++k)
    {
        T const d = x[k * n_states + t];
#pragma unroll
        for (int r = 0; r < R; ++r)
        {
            T const pr = hp[r][2 * k] * d;
            T const pi = hp[r][2 * k + 1] * d;
            wr[r] = wr[r] + pr;
            wi[r] = wi[r] + pi;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (s0 + r < n_strings)
        {
            uint32_t const ny = nys[s0 + r] & 3u;
            T const a = wr[r], b = wi[r];
            w[2 * (t * n_strings + s0 + r)] = ny == 0 ? a : ny == 1 ? b : ny == 2 ? -a : -b;
            w[2 * (t * n_strings + s0 + r) + 1] = ny == 0 ? b : ny == 1 ? -a : ny == 2 ? -b : a;
        }
}

} // namespace fpc
