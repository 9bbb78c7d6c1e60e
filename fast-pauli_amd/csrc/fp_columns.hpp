// fp_columns.hpp — PauliOp expectation values on state columns.
//
// Each state is one contiguous column of 2^n rows (a transposed copy of the batch; the
// batch itself when it holds one state).  A block owns one leader tile of 2^w consecutive
// rows of a column: its threads hold the tile's rows in registers (8 16-byte slots each),
// and the partner tile of a class of strings (equal x >> w) goes through LDS.  A string
// then costs one 16-byte LDS read per slot: leaders are never re-read, and strings whose
// partner rows lie in the same tile lead their pairs from half of the slots.
//
// Row index within a tile: [wave | slot (3 bits) | lane (6 bits) | sub (complex64)].  The
// partner of (wave, slot, lane) is (wave ^ x_w, slot ^ x_s, lane ^ x_l): one XOR per string
// for the lane and wave parts, the slot part an immediate offset of the body specialised
// on x_s; the sign parity(row & z) is a per-lane bit, a wave-uniform bit, and +-1 factors
// for the three slot bits (and the sub bit), applied in a tree of FMAs.  The string's
// coefficient is known, so its sum stays in the thread: no cross-lane sum per string.
//
// Bound: LDS reads (one wave read of 16 bytes per lane takes 4 clocks of a CU) and vector issue
// (about 33 instructions per string and 8 slots); at n = 14 they are 62 % and 64 % busy, scalar
// issue 56 %, without bank conflicts, and a second pair of strings in flight gains nothing
// there.  With few strings per class the tile loads are the larger part (n = 18, 13 complex64
// states: vector issue 54 %, LDS 30 %).  Shares are of issue counters over the kernel's cycles,
// an instruction taking four of its SIMD or of its CU's LDS.  Tiles of 64 KiB in 512-thread
// blocks, two to a CU, so that one block's loads overlap the other's strings; 8 slots of 16
// bytes keep 95 (complex64 99) VGPRs, four waves per SIMD.  Measured against the coset-tiled
// kernel (us): n = 14, 1024 strings, 1000 complex128 states 6200 -> 1610; n = 16, 1024 strings,
// one state 70 -> 15.4; n = 18, 300 strings, 13 complex64 states 373 -> 114.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fp_kernels.hpp"
#include "fp_tile_types.hpp"

namespace fpc
{

// 16 bytes of a column: one complex128 row or two complex64 rows
template <class T> struct Piece;
template <> struct Piece<double>
{
    typedef fpk::VecOf<double, 1>::type type;
};
template <> struct Piece<float>
{
    typedef fpk::VecOf<float, 2>::type type;
};

// The leader slots of a body: all 8, or (HALF) the 4 whose bit kSel, the highest of XS, is clear.
template <int XS, bool HALF> struct Lead
{
    static constexpr int kSel = !HALF ? -1 : (XS & 4) ? 2 : (XS & 2) ? 1 : 0;
    static constexpr bool leads(int i)
    {
        return kSel < 0 || !((i >> (kSel < 0 ? 0 : kSel)) & 1);
    }
};

// The partner pieces of the leader slots; `part` is the LDS address of slot 0's partner when XS = 0.
template <class T, int XS, bool HALF>
__device__ __forceinline__ void load_partners(typename Piece<T>::type (&R)[8], unsigned char const *part)
{
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (Lead<XS, HALF>::leads(i))
            R[i] = *reinterpret_cast<typename Piece<T>::type const *>(part + ((i ^ XS) << 10));
}

// Block `b` of per_group blocks for each of n_groups column groups.  Block ids are dealt to the
// 8 XCDs round-robin: the blocks of a group follow each other on one XCD, whose L2 then serves
// the columns' repeated reads; the last n_groups % 8 groups are spread over all of them.
struct BlockOf
{
    uint32_t group, index;
};
__device__ __forceinline__ BlockOf block_of(uint32_t b, uint32_t per_group, uint32_t n_groups)
{
    uint32_t const whole = n_groups & ~7u;
    if (b < whole * per_group)
    {
        uint32_t const slot = b >> 3;
        return BlockOf{(slot / per_group) * 8u + (b & 7u), slot % per_group};
    }
    uint32_t const r = b - whole * per_group;
    return BlockOf{whole + r / per_group, r % per_group};
}

// One string on the leader slots L and their partners R.  sg[k]: sign factor of slot bit k,
// s0: of the sub bit.
template <class T, int XS, bool SUB, bool IM, bool HALF>
__device__ __forceinline__ T pair_sum(typename Piece<T>::type const (&L)[8], typename Piece<T>::type const (&R)[8],
                                      T const (&sg)[3], T s0)
{
    constexpr int kNp = sizeof(T) == 4 ? 2 : 1;
    constexpr int kSel = Lead<XS, HALF>::kSel;
    auto leads = [](int i) { return Lead<XS, HALF>::leads(i); };
    T v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (leads(i))
        {
            T g[kNp];
#pragma unroll
            for (int c = 0; c < kNp; ++c)
            {
                int const d = (SUB && kNp == 2) ? 1 - c : c;
                T const lr = L[i][2 * c], li = L[i][2 * c + 1], rr = R[i][2 * d], ri = R[i][2 * d + 1];
                g[c] = IM ? fma(lr, ri, -(li * rr)) : fma(lr, rr, li * ri);
            }
            v[i] = kNp == 2 ? fma(s0, g[kNp - 1], g[0]) : g[0];
        }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k != kSel)
        {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (leads(i) && !((i >> k) & 1) && (i & ((1 << k) - 1) & ~(kSel >= 0 ? 1 << kSel : 0)) == 0)
                    v[i] = fma(sg[k], v[i | (1 << k)], v[i]);
        }
    return v[0];
}

// x = 0: |psi|^2 over the 8 slots
template <class T>
__device__ __forceinline__ T self_sum(typename Piece<T>::type const (&L)[8], T const (&sg)[3], T s0)
{
    T v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
    {
        T const a = fma(L[i][0], L[i][0], L[i][1] * L[i][1]);
        if constexpr (sizeof(T) == 4)
            v[i] = fma(s0, fma(L[i][2], L[i][2], L[i][3] * L[i][3]), a);
        else
            v[i] = a;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int i = 0; i < 8; i += 2 << k)
            v[i] = fma(sg[k], v[i | (1 << k)], v[i]);
    return v[0];
}

// cols: n_cols columns of 2^n rows, back to back.  A block runs one item on one column group:
// one column, or the 2^(tile_bits - n) columns that fill a tile.  partial[item * n_cols + t]:
// FP64 sums.
template <class T>
__global__ __launch_bounds__(kThreads, 4) void k_ev_columns(typename Piece<T>::type const *__restrict__ cols, uint32_t n,
                                                         uint32_t n_cols, uint32_t n_items, uint32_t n_groups,
                                                         ColItem const *__restrict__ items,
                                                         ColEntry const *__restrict__ entries,
                                                         ColStr const *__restrict__ strs,
                                                         fpk::Dbl2 *__restrict__ partial)
{
    typedef typename Piece<T>::type P;
    constexpr bool kC64 = sizeof(T) == 4;
    constexpr uint32_t kSub = sub_bits(kC64), kW = tile_bits(kC64);
    extern __shared__ __align__(16) unsigned char smem[];
    P *tile = reinterpret_cast<P *>(smem);
    __shared__ double red[2][kThreads / 64];

    BlockOf const bo = block_of(blockIdx.x, n_items, n_groups);
    uint32_t const grp = bo.group, it = bo.index;
    ColItem const item = items[it];
    uint32_t const tid = threadIdx.x, lane = tid & 63u;
    uint32_t const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t const e0 = wave * 512u + lane; // slot 0 of this thread, in pieces of the tile
    // pieces of a column group and of the tile; a ragged last group has dead columns
    uint64_t const col_pieces = (uint64_t(1) << n) >> kSub;
    uint32_t const per_group = n < kW ? 1u << (kW - n) : 1u;
    uint64_t const first_piece = uint64_t(grp) * per_group * col_pieces;
    uint64_t const n_pieces = uint64_t(n_cols) * col_pieces - first_piece; // live pieces from here
    P const *base = cols + first_piece;

    P L[8];
    {
        uint64_t const t0 = uint64_t(item.p) * (kThreads * 8u) + e0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            L[i] = t0 + uint32_t(i) * 64u < n_pieces ? base[t0 + uint32_t(i) * 64u] : P(0);
    }
    uint32_t const g = (item.p << kWaveBits) | wave; // row bits above the slots
    uint32_t const la = (wave << 13) | (lane << 4);
    double acc_re = 0.0, acc_im = 0.0;
    // An entry's partner rows are asked for before the barrier that ends the previous one, and
    // its first records with them: a wave that is done early waits for its loads meanwhile.
    ColEntry next = entries[item.entry_first];
    ColStr first = strs[next.first];
    for (uint32_t e = 0; e < item.entry_count; ++e)
    {
        ColEntry const en = next;
        ColStr st = first;
        if (en.u == 0)
        {
            __syncthreads(); // the previous partner tile is no longer read
#pragma unroll
            for (int i = 0; i < 8; ++i)
                tile[e0 + uint32_t(i) * 64u] = L[i];
        }
        else
        {
            P const *src = base + uint64_t(item.p ^ en.u) * (kThreads * 8u) + e0; // n > kW: whole tiles, all live
            P r[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                r[i] = src[uint32_t(i) * 64u];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 8; ++i)
                tile[e0 + uint32_t(i) * 64u] = r[i];
        }
        next = entries[item.entry_first + (e + 1 < item.entry_count ? e + 1 : e)];
        first = strs[next.first];
        __syncthreads();
        uint32_t const end = en.first + en.count;
        for (uint32_t s = en.first; s < end;)
        {
            // strings of one case follow each other: one branch to their body, which then
            // runs the whole stretch with the next record in flight (a branch per string:
            // 2174 us instead of 1603 at n = 14, 1024 strings, 1000 complex128 states)
            uint32_t const stretch = st.code >> kColRunShift;
            uint32_t const stop = stretch < end - s ? s + stretch : end;
            auto signs = [&](ColStr const &r, T(&sg)[3], T &s0) {
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    sg[k] = (r.code >> (kColZShift + uint32_t(k))) & 1u ? T(-1) : T(1);
                s0 = kC64 && ((r.code >> (kColZShift + 3u)) & 1u) ? T(-1) : T(1);
            };
            auto add = [&](ColStr const &r, T v) {
                // row sign: this lane's bits of z plus the wave-uniform ones
                uint32_t const neg = uint32_t(__popc(lane & r.zl)) + uint32_t(__popc(g & r.zg));
                double const d = double(v);
                double const ds =
                    __longlong_as_double(__double_as_longlong(d) ^ (static_cast<long long>(neg & 1u) << 63));
                acc_re = fma(r.sre, ds, acc_re);
                acc_im = fma(r.sim, ds, acc_im);
            };
            auto run = [&](auto xs_tag, auto sub_tag, auto im_tag, auto half_tag) {
                constexpr int XS = decltype(xs_tag)::value;
                constexpr bool SUB = decltype(sub_tag)::value, IM = decltype(im_tag)::value,
                               HALF = decltype(half_tag)::value;
                if constexpr (HALF)
                {
                    // two strings at a time: 8 LDS reads in flight, as in the other bodies (one-tile
                    // columns gain 2 %, n = 14 nothing)
                    for (; s + 1 < stop; s += 2)
                    {
                        ColStr const a = st, b = strs[s + 1];
                        st = strs[s + 2]; // one record follows the last
                        P Ra[8], Rb[8];
                        load_partners<T, XS, HALF>(Ra, smem + (la ^ a.px));
                        load_partners<T, XS, HALF>(Rb, smem + (la ^ b.px));
                        T sg[3], s0;
                        signs(a, sg, s0);
                        add(a, pair_sum<T, XS, SUB, IM, HALF>(L, Ra, sg, s0));
                        signs(b, sg, s0);
                        add(b, pair_sum<T, XS, SUB, IM, HALF>(L, Rb, sg, s0));
                    }
                    if (s >= stop)
                        return;
                }
                while (true)
                {
                    ColStr const nx = strs[s + 1];
                    P R[8];
                    load_partners<T, XS, HALF>(R, smem + (la ^ st.px));
                    T sg[3], s0;
                    signs(st, sg, s0);
                    add(st, pair_sum<T, XS, SUB, IM, HALF>(L, R, sg, s0));
                    st = nx;
                    if (++s >= stop)
                        break;
                }
            };
#define FP_COL_CASE(XS, SUB, IM, HALF)                                                                                 \
    case (XS) | ((SUB) ? kColSub : 0u) | ((IM) ? kColImag : 0u) | ((HALF) ? kColHalf : 0u):                            \
        run(std::integral_constant<int, XS>{}, std::integral_constant<bool, SUB>{},                                    \
            std::integral_constant<bool, IM>{}, std::integral_constant<bool, HALF>{});                                 \
        break;
#define FP_COL_XS(SUB, IM)                                                                                             \
    FP_COL_CASE(0, SUB, IM, false)                                                                                     \
    FP_COL_CASE(1, SUB, IM, false)                                                                                     \
    FP_COL_CASE(2, SUB, IM, false)                                                                                     \
    FP_COL_CASE(3, SUB, IM, false)                                                                                     \
    FP_COL_CASE(4, SUB, IM, false)                                                                                     \
    FP_COL_CASE(5, SUB, IM, false)                                                                                     \
    FP_COL_CASE(6, SUB, IM, false)                                                                                     \
    FP_COL_CASE(7, SUB, IM, false)                                                                                     \
    FP_COL_CASE(1, SUB, IM, true)                                                                                      \
    FP_COL_CASE(2, SUB, IM, true)                                                                                      \
    FP_COL_CASE(3, SUB, IM, true)                                                                                      \
    FP_COL_CASE(4, SUB, IM, true)                                                                                      \
    FP_COL_CASE(5, SUB, IM, true)                                                                                      \
    FP_COL_CASE(6, SUB, IM, true)                                                                                      \
    FP_COL_CASE(7, SUB, IM, true)
            uint32_t const kase = st.code & kColCase;
            if (kase == kColSelf)
            {
                for (; s < stop; ++s)
                {
                    ColStr const nx = strs[s + 1];
                    T sg[3], s0;
                    signs(st, sg, s0);
                    add(st, self_sum<T>(L, sg, s0));
                    st = nx;
                }
            }
            else if constexpr (kC64)
            {
                switch (kase)
                {
                    FP_COL_XS(false, false)
                    FP_COL_XS(false, true)
                    FP_COL_XS(true, false)
                    FP_COL_XS(true, true)
                default: __builtin_unreachable();
                }
            }
            else
            {
                switch (kase)
                {
                    FP_COL_XS(false, false)
                    FP_COL_XS(false, true)
                default: __builtin_unreachable();
                }
            }
#undef FP_COL_XS
#undef FP_COL_CASE
        }
    }
    // a wave's rows belong to one column: wave sums, then the waves of a column in order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
    {
        acc_re += __shfl_xor(acc_re, off, 64);
        acc_im += __shfl_xor(acc_im, off, 64);
    }
    if (lane == 0)
    {
        red[0][wave] = acc_re;
        red[1][wave] = acc_im;
    }
    __syncthreads();
    uint32_t const t = grp * per_group + tid;
    if (tid < per_group && t < n_cols)
    {
        uint32_t const waves = (kThreads / 64u) / per_group;
        double sr = 0.0, si = 0.0;
        for (uint32_t j = 0; j < waves; ++j)
        {
            sr += red[0][tid * waves + j];
            si += red[1][tid * waves + j];
        }
        partial[uint64_t(it) * n_cols + t] = fpk::Dbl2{sr, si};
    }
}

// Columns [c0, c0 + n_cols) of a row-major (rows x ld) batch to columns of NS states a row, and
// back (IN = false): block (bx, by) moves 32 rows of 32 states through LDS; an odd last state is
// paired with zeros, which are not written back.
template <class T, int NS, bool IN>
__device__ __forceinline__ void move_columns(__attribute__((address_space(1))) typename fpk::VecOf<T, 1>::type *batch,
                                             typename fpk::VecOf<T, NS>::type *__restrict__ cols, uint64_t rows,
                                             uint64_t ld, uint64_t c0, uint32_t n_cols, uint32_t bx, uint32_t by)
{
    typedef typename fpk::VecOf<T, 1>::type V1;
    typedef typename fpk::VecOf<T, NS>::type V;
    __shared__ V1 tile[32][33];
    uint64_t const r0 = uint64_t(bx) * 32;
    uint32_t const cb = by * 32u;
    uint32_t const tx = threadIdx.x & 31u, ty = threadIdx.x >> 5;
    auto batch_side = [&] {
#pragma unroll
        for (uint32_t k = ty; k < 32; k += 8)
            if (r0 + k < rows)
            {
                auto *at = batch + (r0 + k) * ld + c0 + cb + tx;
                bool const live = cb + tx < n_cols;
                if constexpr (IN)
                    tile[k][tx] = live ? *at : V1(0);
                else if (live)
                    __builtin_nontemporal_store(tile[k][tx], at);
            }
    };
    auto column_side = [&] {
#pragma unroll
        for (uint32_t k = ty; k < 32 / NS; k += 8)
            if (r0 + tx < rows && cb + k * NS < n_cols)
            {
                V *at = cols + uint64_t(cb / NS + k) * rows + r0 + tx;
                if constexpr (IN)
                {
                    V v;
#pragma unroll
                    for (int h = 0; h < NS; ++h)
                    {
                        v[2 * h] = tile[tx][k * NS + h][0];
                        v[2 * h + 1] = tile[tx][k * NS + h][1];
                    }
                    *at = v;
                }
                else
                {
                    V const v = *at;
#pragma unroll
                    for (int h = 0; h < NS; ++h)
                        tile[tx][k * NS + h] = V1{v[2 * h], v[2 * h + 1]};
                }
            }
    };
    if constexpr (IN)
        batch_side();
    else
        column_side();
    __syncthreads();
    if constexpr (IN)
        column_side();
    else
        batch_side();
}

template <class T, int NS, bool IN>
__global__ __launch_bounds__(256) void k_columns(typename fpk::VecOf<T, 1>::type *__restrict__ batch,
                                                 typename fpk::VecOf<T, NS>::type *__restrict__ cols, uint64_t rows,
                                                 uint64_t ld, uint64_t c0, uint32_t n_cols)
{
    typedef typename fpk::VecOf<T, 1>::type V1;
    move_columns<T, NS, IN>((__attribute__((address_space(1))) V1 *)batch, cols, rows, ld, c0, n_cols, blockIdx.x,
                            blockIdx.y);
}

} // namespace fpc
