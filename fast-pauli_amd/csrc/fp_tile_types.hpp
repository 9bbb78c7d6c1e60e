// fp_tile_types.hpp — the host-built records that the tiled kernels read: string
// groups over coset tiles, their chunks and per-string records, and the
// per-string EV matrix's chunks.  Plain data with no HIP dependency, so that the
// host-side table builder also compiles as ordinary C++ (and under the address
// and undefined-behaviour sanitizers in its unit test).
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define FP_HD __host__ __device__
#else
#define FP_HD
#endif

namespace fpt
{

constexpr int kMaxDh = 13; // string-span dimensions per tile (B table of 2^13 entries, read once per block)

struct TileGroup
{
    uint32_t n_chunks;
    uint32_t chunk_first;
    uint32_t n_piv;    // dh: pivots (high dimensions of V)
    uint32_t btab_off; // first entry of this group's B table (2^dh entries)
    uint64_t piv_lo;   // pivot bit positions 0..7, ascending, 8 bits each
    uint64_t piv_hi;   // pivot bit positions 8..15
    uint32_t hoist;     // bit hoist_bit(W, U1, r): every wave of a block has at most one
                        // unit and it takes the one-string fast path (expectation tables)
    uint32_t shared;    // bit shared_bit(W, c64, rr): the group runs the shared-leader
                        // form (expectation tables)
    uint32_t str_first; // first ShStr of the group (expectation tables)
    uint32_t n_str;     // strings of the group
    uint32_t n_wht;     // per-string EV matrix tables: the first n_wht chunks are transform classes
    uint32_t pad;
};

// Strings of a shared-leader group: every local x mask has bit k set, so the
// leader rows (local bit k clear) are common to all of them.  At most
// max_shared(W) strings for the instance with W waves per block (its per-string
// registers), kMaxShared over all instances.
constexpr int kMaxShared = 10;
FP_HD constexpr int max_shared(uint32_t W)
{
    return W == 16 ? 10 : 9;
}

struct ShStr
{
    uint64_t zc;   // z compressed onto the coset-index bits: coset sign = parity(q & zc)
    uint32_t A;    // local x mask (bit k set)
    uint32_t Z;    // local z mask
    uint32_t imag; // 1: Im w (odd nY), 0: Re w
    uint32_t pad;
    double sre; // scale c_s * kappa_s
    double sim;
};

// Bit of TileGroup::shared for W waves per block, complex64 (two states per
// lane) or not, and 2^rr leader rows per pass.
FP_HD constexpr uint32_t shared_bit(uint32_t W, bool c64, uint32_t rr)
{
    return (W == 16 ? 16u : 0u) + (c64 ? 8u : 0u) + rr;
}

// Bit of TileGroup::hoist for W waves per block, U1 passes per fast-path step and
// 2^r leader rows per pass (r = 6 - log2 S_blk).
FP_HD constexpr uint32_t hoist_bit(uint32_t W, uint32_t U1, uint32_t r)
{
    return (W == 16 ? 16u : 0u) + (U1 == 8 ? 8u : 0u) + r;
}

struct TileChunk
{
    uint32_t A;     // local x mask; 0: every row, kappa 1
    uint32_t h;     // top bit of A
    uint32_t count; // strings in this chunk (1..kChunk), all with local mask A
    uint32_t first; // first TileStr
    uint32_t need;  // bit 0: some string uses Re w, bit 1: some string uses Im w
    uint32_t pad[3];
};

struct TileStr
{
    uint64_t zc;   // z compressed onto the coset-index bits: coset sign = parity(q & zc)
    uint32_t zt;   // local z with bit h removed: row sign of leader p = parity(p & zt)
    uint32_t imag; // 1: Im w (odd nY), 0: Re w
    double sre;    // scale c_s * kappa_s
    double sim;
};

constexpr int kChunk = 4;

} // namespace fpt

namespace fpa
{

struct ApplyStr
{
    uint64_t zc;  // z compressed onto the coset-index bits: coset sign = parity(q & zc)
    uint32_t A;   // local x mask
    uint32_t Z;   // local z mask
    double cr;    // folded coefficient c_s (-i)^{nY_s}, complex128
    double ci;
    float fr;     // the same, complex64 (rounded as the streaming kernel's table)
    float fi;
    uint32_t s;   // the string's index in the operator
    uint32_t pad;
};

} // namespace fpa

namespace fpl
{

constexpr int kChunk = 8;

// A class of strings with equal x and equal half of w is evaluated by one
// Walsh-Hadamard transform of G over the leader rows when it holds at least
// kWhtMin strings (split into classes of at most kWhtMax):
//     ev_s = scale_s * sum_leaders (-1)^{parity(a & Z_s)} G(a) = scale_s * W[compress(Z_s)],
// one pass over the rows and (d-1) butterfly levels instead of one pass per string.
// One wave transforms a class on its own, in parts of kWhtPartBytes of G held in
// a private LDS slice (no block barrier); the parts are combined per string by
// their top index bits.
constexpr uint32_t kWhtMin = 12;
constexpr uint32_t kWhtMax = 256;        // 4 strings per lane
constexpr uint32_t kWhtMinRowsLog2 = 10; // columns shorter than this keep the per-string loop
constexpr uint32_t kWhtPartBytes = 2048;
constexpr uint32_t kWhtWaves = 15;       // waves with a slice (the last wave takes per-string chunks only)
constexpr uint32_t kWhtLdsBytes = kWhtWaves * kWhtPartBytes;

enum : uint32_t
{
    kAllRows = 0,
    kPairs = 1,
    kPairsLane = 2
};

struct EvChunk
{
    uint32_t x;     // x mask (n <= 14: fits 32 bits)
    uint32_t h;     // highest set bit of x (pair modes)
    uint32_t mode;  // kAllRows / kPairs / kPairsLane
    uint32_t count; // strings in this chunk (1..kChunk)
    uint32_t first; // index of the first EvStr
    uint32_t imag;  // 1: every string of the chunk takes Im w (odd nY), 0: Re w
    uint32_t pad[2];
};

// Mode of a string with x mask x (highest set bit h) over `rows` rows.
FP_HD constexpr uint32_t ev_mode(uint64_t x, uint32_t h, uint64_t rows)
{
    return x == 0 ? kAllRows : (h >= 6 ? kPairs : (rows >= 128 ? kPairsLane : kAllRows));
}

struct EvStr
{
    uint32_t z;
    uint32_t imag; // 1: G = Im w, 0: G = Re w
    uint32_t out;  // output row (original string index)
    uint32_t zc;   // coset kernel: z compressed onto the coset-index bits (0 otherwise)
    double scale;  // eps (kAllRows) or 2 eps (kPairs)
};

} // namespace fpl

// PauliOp expectation on state columns (the column kernel).  A column's rows are cut
// into tiles of 2^w consecutive rows; within a tile a row index is
//   [wave bits | 3 slot bits | 6 lane bits | sub bit (complex64 only)],
// the slots being the 8 16-byte pieces (one complex128 or two complex64 rows) a thread owns.
// Strings are filed by class u = x >> w: a class pairs leader tile p with tile p ^ u.
namespace fpc
{

constexpr uint32_t kSlotBits = 3;
constexpr uint32_t kLaneBits = 6;
constexpr uint32_t kThreads = 512;
constexpr uint32_t kWaveBits = 3;
constexpr uint32_t kTileBytes = kThreads * 8u * 16u;

FP_HD constexpr uint32_t sub_bits(bool c64)
{
    return c64 ? 1u : 0u;
}
// row bits below the wave bits
FP_HD constexpr uint32_t low_bits(bool c64)
{
    return kSlotBits + kLaneBits + sub_bits(c64);
}
FP_HD constexpr uint32_t tile_bits(bool c64)
{
    return kWaveBits + low_bits(c64);
}

// One block's work on a column: leader tile p, entries [entry_first, entry_first + entry_count).
struct ColItem
{
    uint32_t p;
    uint32_t entry_first;
    uint32_t entry_count;
    uint32_t pad;
};

// Strings [first, first + count) of class u: the partner tile is p ^ u.
struct ColEntry
{
    uint32_t u;
    uint32_t first;
    uint32_t count;
    uint32_t pad;
};

// ColStr::code: bits 0-2 the slot bits of x, bit 3 its sub bit, bit 4 Im w, and one of
//   bit 5: x = 0 (every row, |psi|^2),
//   bit 6: partner in the same tile, pairs led by the slots whose bit (the highest slot
//          bit of x) is clear;
// bits 8-10 the slot bits of z, bit 11 its sub bit.  A same-tile string whose slot bits are
// all clear visits each pair from both sides (its scale is halved).
constexpr uint32_t kColSub = 8, kColImag = 16, kColSelf = 32, kColHalf = 64, kColCase = 127;
constexpr uint32_t kColZShift = 8;
// bits 16 up: how many strings of the class, from this one on, share its case
constexpr uint32_t kColRunShift = 16, kColRunMax = 0xffff;

struct ColStr
{
    uint32_t px;   // byte offset of x's lane and wave bits within the tile (XOR)
    uint32_t zl;   // z's lane bits
    uint32_t zg;   // z's bits above the slot bits
    uint32_t code;
    double sre; // scale c_s * kappa_s (times 1/2 where pairs are visited twice)
    double sim;
};

// Many operators on the columns of one slab (k_apply_columns_batch, k_columns_batch).
struct ColJob
{
    uint64_t cols;   // byte offset of the first column in both slabs
    uint64_t xs, zs, cf; // device addresses of the operator's masks and folded coefficients
    uint32_t n, n_cols, n_strings, accumulate;
};
// Blocks [block0, ...) of a job, from position `start` of an XCD's queue on.
struct ColSeg
{
    uint32_t start, job, block0, pad;
};
// States [c0, c0 + n_states) of a row-major (2^n x ld) batch and their columns.
struct ColCopy
{
    uint64_t batch; // device address
    uint64_t cols;  // byte offset of the first column in its slab
    uint64_t ld, c0;
    uint32_t n, n_states;
    uint32_t start; // first block
    uint32_t out;   // the output slab's columns
};

} // namespace fpc

