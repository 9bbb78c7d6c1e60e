// Unit test of the column kernel's host tables (build_column_image in
// fast-pauli_amd/csrc/fp_tiles_host.cpp), built with the address and
// undefined-behaviour sanitizers.  It walks every item, entry and string record
// the way the kernel does (tiles, waves, slots, lanes, leaders, partner offsets
// and signs) on a random column and compares the sum with
//     sum_s c_s sum_j m_s(j) conj(psi_j) psi_{j ^ x_s}
// evaluated row by row, for columns shorter than a tile, of one tile and of
// several, random and structured string sets and several item sizes.
//
// Both sums are FP64 over the same terms in another order: N 2^n terms of size
// |c| |psi|^2, so 1e-12 relative to sum_s |c_s| <psi|psi> leaves a margin over
// the 1e-16 sqrt(N 2^n) expected.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <utility>
#include <vector>

#include "fp_tiles_host.hpp"

namespace
{

int g_failures = 0;

struct Rng
{
    uint64_t s;
    uint64_t next()
    {
        uint64_t z = (s += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }
    double unit()
    {
        return double(next() >> 11) * 0x1.0p-52 - 1.0;
    }
};

typedef std::complex<double> cplx;

uint32_t parity(uint64_t v)
{
    return uint32_t(__builtin_popcountll(v) & 1);
}

struct Set
{
    size_t n;
    std::vector<uint64_t> x, z;
    std::vector<uint32_t> ny;
    std::vector<double> coeffs;
    fprt::StringTable table() const
    {
        return fprt::StringTable{n, x.size(), x.data(), z.data(), ny.data(), coeffs.data(), nullptr, nullptr};
    }
};

// kind 0: uniform letters; 1: at most three X/Y bits; 2: diagonal; 3: four x masks; 4: X/Y on the low 3 bits
Set make(size_t n, size_t N, int kind, Rng &r)
{
    Set s{n, {}, {}, {}, {}};
    uint64_t const mask = (uint64_t(1) << n) - 1;
    for (size_t i = 0; i < N; ++i)
    {
        uint64_t x = r.next() & mask;
        if (kind == 1)
            x = (uint64_t(1) << (r.next() % n)) | (uint64_t(1) << (r.next() % n)) | (uint64_t(1) << (r.next() % n));
        else if (kind == 2)
            x = 0;
        else if (kind == 3)
            x = (0x9e3779b97f4a7c15ull * (i % 4)) & mask;
        else if (kind == 4)
            x &= 7;
        uint64_t const z = r.next() & mask;
        s.x.push_back(x);
        s.z.push_back(z);
        s.ny.push_back(uint32_t(__builtin_popcountll(x & z)));
        s.coeffs.push_back(r.unit());
        s.coeffs.push_back(r.unit());
    }
    return s;
}

cplx direct(Set const &s, std::vector<cplx> const &psi, double &scale)
{
    static cplx const unit[4] = {{1, 0}, {0, -1}, {-1, 0}, {0, 1}}; // (-i)^nY
    cplx sum = 0;
    scale = 0;
    double norm = 0;
    for (cplx const &v : psi)
        norm += std::norm(v);
    for (size_t k = 0; k < s.x.size(); ++k)
    {
        cplx e = 0;
        for (size_t j = 0; j < psi.size(); ++j)
        {
            cplx const w = std::conj(psi[j]) * psi[j ^ s.x[k]];
            e += parity(j & s.z[k]) ? -w : w;
        }
        cplx const c(s.coeffs[2 * k], s.coeffs[2 * k + 1]);
        sum += c * (unit[s.ny[k] & 3] * e).real(); // the expectation value of a string is real
        scale += std::abs(c) * norm;
    }
    return sum;
}

cplx through_tables(Set const &s, bool c64, uint32_t per_item, std::vector<cplx> const &psi)
{
    fprt::TileImage im;
    if (fprt::build_column_image(s.table(), c64, per_item, im) != FP_OK)
    {
        ++g_failures;
        return 0;
    }
    auto const *items = reinterpret_cast<fpc::ColItem const *>(im.h.data());
    auto const *entries = reinterpret_cast<fpc::ColEntry const *>(im.h.data() + im.o_chunks);
    auto const *strs = reinterpret_cast<fpc::ColStr const *>(im.h.data() + im.o_strs);
    uint32_t const sb = fpc::sub_bits(c64), w = fpc::tile_bits(c64), low = fpc::low_bits(c64);
    uint32_t const waves = s.n < w ? 1u << (s.n - low) : 1u << fpc::kWaveBits;
    cplx sum = 0;
    for (uint32_t i = 0; i < im.n_groups; ++i)
        for (uint32_t e = 0; e < items[i].entry_count; ++e)
        {
            fpc::ColEntry const &en = entries[items[i].entry_first + e];
            for (uint32_t k = en.first; k < en.first + en.count; ++k)
            {
                fpc::ColStr const &st = strs[k];
                uint32_t const xs = st.code & 7u, kase = st.code & fpc::kColCase;
                // the stretch of one case reaches at least this string and stays in its case
                uint32_t const run = st.code >> fpc::kColRunShift;
                if (run == 0)
                    ++g_failures;
                for (uint32_t m = 1; m < run; ++m)
                    g_failures += (strs[k + m].code & fpc::kColCase) != kase;
                uint32_t const sel = xs & 4 ? 2 : xs & 2 ? 1 : 0;
                double v = 0;
                for (uint32_t wave = 0; wave < waves; ++wave)
                    for (uint32_t slot = 0; slot < 8; ++slot)
                    {
                        if ((kase & fpc::kColHalf) && ((slot >> sel) & 1u))
                            continue;
                        for (uint32_t lane = 0; lane < 64; ++lane)
                            for (uint32_t sub = 0; sub <= sb; ++sub)
                            {
                                auto row = [&](uint32_t tile, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
                                    return (uint64_t(tile) << w) | (uint64_t(a) << low) | (uint64_t(b) << (6 + sb)) |
                                           (uint64_t(c) << sb) | d;
                                };
                                uint32_t const byte = ((wave << 13) | (lane << 4)) ^ st.px;
                                uint64_t const j = row(items[i].p, wave, slot, lane, sub);
                                uint64_t const q = row(items[i].p ^ en.u, byte >> 13, slot ^ xs, (byte >> 4) & 63u,
                                                       sub ^ ((kase & fpc::kColSub) ? 1u : 0u));
                                uint32_t const zs = (st.code >> fpc::kColZShift) & 7u;
                                uint32_t const z0 = (st.code >> (fpc::kColZShift + 3)) & 1u;
                                uint32_t const g = (items[i].p << fpc::kWaveBits) | wave;
                                uint32_t const neg = parity(lane & st.zl) ^ parity(g & st.zg) ^ parity(slot & zs) ^
                                                     (sub & z0);
                                cplx const wv = std::conj(psi.at(j)) * psi.at(q);
                                double const t = kase == fpc::kColSelf ? std::norm(psi.at(j))
                                                 : (kase & fpc::kColImag) ? wv.imag()
                                                                          : wv.real();
                                v += neg ? -t : t;
                            }
                    }
                sum += cplx(st.sre, st.sim) * v;
            }
        }
    return sum;
}

// Rounds of a batch: through the tables, as the kernels walk them, every state of every entry is
// copied in once (outputs too when accumulating), computed by exactly the blocks that cover its
// column, and copied out once; columns of a round stay apart and inside the slab.
int check_rounds(std::vector<fprt::ColumnEntry> const &es, size_t slab)
{
    std::vector<fprt::ColumnRound> rounds;
    std::vector<unsigned char> im;
    size_t used = 0;
    fprt::build_column_rounds(es, slab, rounds, im, used);
    int bad = 0;
    std::vector<std::vector<int>> in(es.size()), acc(es.size()), out(es.size());
    for (size_t i = 0; i < es.size(); ++i)
        for (auto *v : {&in[i], &acc[i], &out[i]})
            v->assign(es[i].n_states, 0);
    auto find = [](uint32_t const *ends, uint32_t count, uint32_t pos) {
        uint32_t i = 0;
        while (i < count && pos >= ends[i])
            ++i;
        return i;
    };
    for (fprt::ColumnRound const &r : rounds)
    {
        auto const *jobs = reinterpret_cast<fpc::ColJob const *>(im.data() + r.o_jobs);
        bool const pairs = r.variant & fprt::kColsPairs;
        uint32_t const tile = 8;
        uint64_t const row = (r.variant & fprt::kColsC64) && !pairs ? 8 : 16;
        // copies: block by block
        struct Span
        {
            uint64_t at, size;
            size_t entry;
        };
        std::vector<Span> spans;
        for (int dir = 0; dir < 2; ++dir)
        {
            auto const *c = reinterpret_cast<fpc::ColCopy const *>(im.data() + (dir ? r.o_out : r.o_in));
            auto const *ends = reinterpret_cast<uint32_t const *>(im.data() + (dir ? r.o_out_ends : r.o_in_ends));
            uint32_t const count = dir ? r.n_out : r.n_in, blocks = dir ? r.out_blocks : r.in_blocks;
            std::vector<uint32_t> seen(count, 0);
            for (uint32_t b = 0; b < blocks; ++b)
            {
                uint32_t const at = find(ends, count, b);
                if (at >= count)
                {
                    ++bad;
                    continue;
                }
                bad += b - c[at].start != seen[at]++;
            }
            for (uint32_t k = 0; k < count; ++k)
            {
                fpc::ColCopy const &k_ = c[k];
                size_t e = 0;
                while (e < es.size() && (k_.out ? es[e].out : es[e].states) != k_.batch)
                    ++e;
                if (e == es.size())
                {
                    ++bad;
                    continue;
                }
                bad += k_.n != es[e].n || k_.ld != es[e].n_states;
                bad += seen[k] != ((uint64_t(1) << k_.n) + 31) / 32 * ((k_.n_states + 31) / 32);
                auto &v = dir ? out[e] : k_.out ? acc[e] : in[e];
                for (uint64_t t = 0; t < k_.n_states; ++t)
                    ++v.at(k_.c0 + t);
                uint64_t const cols = pairs ? (k_.n_states + 1) / 2 : k_.n_states;
                bad += pairs && k_.c0 % 2 != 0;
                bad += k_.cols + cols * (row << k_.n) > used || k_.cols % 16 != 0;
                if (dir)
                    spans.push_back(Span{k_.cols, cols * (row << k_.n), e});
            }
        }
        for (size_t a = 0; a < spans.size(); ++a)
            for (size_t b = 0; b < a; ++b)
                bad += spans[a].at < spans[b].at + spans[b].size && spans[b].at < spans[a].at + spans[a].size;
        // apply blocks
        auto const *ends = reinterpret_cast<uint32_t const *>(im.data() + r.o_ends);
        auto const *segs = reinterpret_cast<fpc::ColSeg const *>(im.data() + r.o_segs);
        bad += r.n_segs % 64 != 0 || r.blocks % 8 != 0;
        std::vector<std::vector<int>> hit(spans.size());
        for (size_t j = 0; j < spans.size(); ++j)
        {
            fprt::ColumnEntry const &e = es[spans[j].entry];
            bad += jobs[j].cols != spans[j].at || jobs[j].n != e.n || jobs[j].n_strings != e.n_strings ||
                   jobs[j].xs != e.xs || jobs[j].zs != e.zs || jobs[j].cf != e.cf || (jobs[j].accumulate != 0) != e.accumulate ||
                   jobs[j].n_cols * (row << e.n) != spans[j].size;
            uint64_t const per = e.n < tile ? 1u << (tile - e.n) : 1u, tiles = e.n > tile ? 1u << (e.n - tile) : 1u;
            hit[j].assign((jobs[j].n_cols + per - 1) / per * tiles, 0);
        }
        for (uint32_t b = 0; b < r.blocks; ++b)
        {
            uint32_t const x = b & 7, pos = b >> 3, at = find(ends + x * r.n_segs, r.n_segs, pos);
            if (at >= r.n_segs)
                continue;
            fpc::ColSeg const &s = segs[x * r.n_segs + at];
            ++hit.at(s.job).at(s.block0 + pos - s.start);
        }
        for (auto const &h : hit)
            for (int v : h)
                bad += v != 1;
    }
    for (size_t i = 0; i < es.size(); ++i)
        for (size_t t = 0; t < es[i].n_states; ++t)
            bad += in[i][t] != 1 || out[i][t] != 1 || acc[i][t] != (es[i].accumulate ? 1 : 0);
    bad += used > slab && es.size() > 1; // (a lone column may be larger than the slab)
    return bad;
}

int round_cases(Rng &r)
{
    int n_cases = 0;
    for (size_t slab : {size_t(1) << 14, size_t(1) << 18, size_t(1) << 22})
        for (int rep = 0; rep < 2; ++rep)
            for (size_t count : {size_t(1), size_t(2), size_t(9), size_t(150)})
            {
                std::vector<fprt::ColumnEntry> es;
                for (size_t i = 0; i < count; ++i)
                {
                    fprt::ColumnEntry e{};
                    e.n = 6 + uint32_t(r.next() % (slab >= (size_t(1) << 22) ? 13 : 5));
                    e.n_strings = 1 + uint32_t(r.next() % 600);
                    e.c64 = r.next() % 2;
                    e.accumulate = r.next() % 3 == 0;
                    e.n_states = 1 + r.next() % (count > 9 ? 9 : 70);
                    e.states = 0x1000 * (4 * i + 1);
                    e.out = 0x1000 * (4 * i + 2);
                    e.xs = 0x1000 * (4 * i + 3);
                    e.zs = e.xs + 0x800;
                    e.cf = 0x1000 * (4 * i + 4);
                    es.push_back(e);
                }
                ++n_cases;
                if (int const bad = check_rounds(es, slab))
                {
                    ++g_failures;
                    std::fprintf(stderr, "FAIL rounds slab=%zu count=%zu: %d faults\n", slab, count,
                                 bad);
                }
            }
    return n_cases;
}

// A launch on `slab` columns stays below 2^32 threads of 512-thread blocks, and its partials, one
// an item and column, below 64 MiB: counted in the tables, and bounded for the largest sets.
int item_cases(Rng &r)
{
    int n_cases = 0;
    auto launch = [&](bool c64, size_t n, size_t N, size_t slab, uint64_t n_items) {
        uint32_t const w = fpc::tile_bits(c64);
        uint64_t const per_group = n < w ? uint64_t(1) << (w - n) : 1, groups = (slab + per_group - 1) / per_group;
        ++n_cases;
        if (n_items * groups * fpc::kThreads >= uint64_t(1) << 32 || n_items * slab > fprt::kMaxColumnItems)
        {
            ++g_failures;
            std::fprintf(stderr, "FAIL launch c64=%d n=%zu strings=%zu slab=%zu: %llu items\n", int(c64), n, N, slab,
                         static_cast<unsigned long long>(n_items));
        }
    };
    for (auto const &[n, N] : {std::pair<size_t, size_t>{9, 2200000}, {12, 3000}, {15, 700}})
    {
        size_t const slab = (size_t(128) << 20) / (size_t(16) << n);
        Set const s = make(n, N, 0, r);
        fprt::TileImage im;
        uint32_t const per = fprt::column_item_size(false, uint32_t(n), N, 100000, slab);
        g_failures += fprt::build_column_image(s.table(), false, per, im) != FP_OK;
        launch(false, n, N, slab, im.n_groups);
        uint64_t const tiles = n > fpc::tile_bits(false) ? uint64_t(1) << (n - fpc::tile_bits(false)) : 1;
        g_failures += im.n_groups > tiles * (N / per + 1);
    }
    for (bool c64 : {false, true})
        for (size_t n = fpc::low_bits(c64); n <= fpc::tile_bits(c64) + 8; ++n)
            for (size_t N = 8; N < (size_t(1) << 31); N = N * 3 + 1)
                for (size_t states : {size_t(1), size_t(100), size_t(100000)})
                {
                    size_t const slab = std::min((size_t(128) << 20) / ((c64 ? size_t(8) : size_t(16)) << n), states);
                    uint64_t const tiles = n > fpc::tile_bits(c64) ? uint64_t(1) << (n - fpc::tile_bits(c64)) : 1;
                    uint32_t const per = fprt::column_item_size(c64, uint32_t(n), N, states, slab);
                    launch(c64, n, N, slab, tiles * (N / per + 1));
                }
    return n_cases;
}

} // namespace

int main()
{
    Rng r{11};
    int n_cases = 0;
    for (bool c64 : {false, true})
        for (uint32_t n = fpc::low_bits(c64); n <= fpc::tile_bits(c64) + 3; ++n)
        {
            std::vector<cplx> psi(size_t(1) << n);
            for (cplx &v : psi)
                v = cplx(r.unit(), r.unit());
            for (int kind = 0; kind < 5; ++kind)
                for (uint32_t per_item : {1u, 7u, 256u})
                {
                    Set const s = make(n, kind == 3 ? 24 : 13, kind, r);
                    double scale = 0;
                    cplx const want = direct(s, psi, scale), got = through_tables(s, c64, per_item, psi);
                    ++n_cases;
                    if (!(std::abs(got - want) <= 1e-12 * scale))
                    {
                        ++g_failures;
                        std::fprintf(stderr, "FAIL c64=%d n=%u kind=%d per_item=%u: off by %g of %g\n", int(c64), n,
                                     kind, per_item, std::abs(got - want), scale);
                    }
                }
        }
    n_cases += round_cases(r);
    n_cases += item_cases(r);
    // sizes the kernel does not take
    Set const small = make(fpc::low_bits(false) - 1, 4, 0, r), large = make(fpc::tile_bits(false) + 13, 4, 0, r);
    fprt::TileImage im;
    g_failures += fprt::build_column_image(small.table(), false, 16, im) == FP_OK;
    g_failures += fprt::build_column_image(large.table(), false, 16, im) == FP_OK;
    std::printf("column tables: %d cases, %d failures\n", n_cases, g_failures);
    return g_failures == 0 ? 0 : 1;
}
