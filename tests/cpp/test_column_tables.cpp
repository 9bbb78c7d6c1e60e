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
#include <cmath>
#include <complex>
#include <cstdio>
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
    // sizes the kernel does not take
    Set const small = make(fpc::low_bits(false) - 1, 4, 0, r), large = make(fpc::tile_bits(false) + 13, 4, 0, r);
    fprt::TileImage im;
    g_failures += fprt::build_column_image(small.table(), false, 16, im) == FP_OK;
    g_failures += fprt::build_column_image(large.table(), false, 16, im) == FP_OK;
    std::printf("column tables: %d cases, %d failures\n", n_cases, g_failures);
    return g_failures == 0 ? 0 : 1;
}
