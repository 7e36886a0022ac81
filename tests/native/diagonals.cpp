// Driver for the diagonals of a matrix (csrc/format.cpp): built by
// tests/test_diagonals.py with g++ and the sanitizers and run on the CPU.
// Whatever rows a diagonal appears in, build_format finds what a plain count of
// col - row finds, and every row's word says which it holds and where its
// second lane's part begins. Prints "done, N failures".
#include "dim_internal.h"

#include <algorithm>
#include <cstdio>
#include <random>
#include <set>
#include <vector>

using namespace dimgpu;

namespace {

int g_fail = 0;

#define EXPECT(cond, ...)                                                                                    \
    do {                                                                                                     \
        if (!(cond)) {                                                                                       \
            std::printf(__VA_ARGS__);                                                                        \
            std::printf("\n");                                                                               \
            ++g_fail;                                                                                        \
        }                                                                                                    \
    } while (0)

struct Csr {
    uint32_t rows = 0;
    std::vector<uint32_t> rp{0}, ci;
};

Csr banded(uint32_t rows, const std::vector<int64_t>& offs, double drop, std::mt19937& g) {
    std::uniform_real_distribution<double> u(0.0, 1.0);
    Csr m;
    m.rows = rows;
    for (uint32_t r = 0; r < rows; ++r) {
        for (int64_t o : offs)
            if (r + o >= 0 && r + o < rows && (o == 0 || u(g) >= drop))
                m.ci.push_back(static_cast<uint32_t>(r + o));
        m.rp.push_back(static_cast<uint32_t>(m.ci.size()));
    }
    return m;
}

void check(const char* name, const Csr& m, uint32_t sigma, bool ordered) {
    HostFormat f;
    const std::vector<double> v(m.ci.size(), 1.0);
    const std::string err = build_format(m.rows, m.rows, m.ci.size(), m.rp.data(), m.ci.data(), v.data(), sigma, f);
    EXPECT(err.empty(), "%s: %s", name, err.c_str());
    std::set<int64_t> all;
    bool empty = false;
    for (uint32_t r = 0; r < m.rows; ++r) {
        empty = empty || m.rp[r] == m.rp[r + 1];
        for (uint32_t k = m.rp[r]; k < m.rp[r + 1]; ++k)
            all.insert(int64_t{m.ci[k]} - r);
    }
    const uint32_t nd = all.size() <= kDiaMax ? dia_kernel_diagonals(static_cast<uint32_t>(all.size())) : 0;
    const bool keep = !empty && ordered && nd && !all.empty() && uint64_t{nd} * m.rows * 4 <= m.ci.size() * 5;
    EXPECT(f.dia_nd == (keep ? nd : 0), "%s sigma %u: %u diagonals kept, %u expected", name, sigma, f.dia_nd,
           keep ? nd : 0);
    EXPECT(f.dia_meta.size() == (keep ? m.rows : 0), "%s sigma %u: %zu words", name, sigma, f.dia_meta.size());
    const bool codes = !empty && !all.empty() && sigma <= kMaxCodedSigma && all.size() <= (1u << code_bits(sigma));
    EXPECT(f.col_dict.size() == (codes ? all.size() : 0), "%s sigma %u: %zu codes", name, sigma, f.col_dict.size());
    if (codes)
        EXPECT(std::equal(all.begin(), all.end(), f.col_dict.begin()), "%s sigma %u: dictionary", name, sigma);
    if (!f.dia_nd || !keep)
        return;
    const std::vector<int64_t> offs(all.begin(), all.end());
    for (size_t d = 0; d < kDiaMax; ++d)
        EXPECT(f.dia_off[d] == (d < offs.size() ? offs[d] : 0), "%s sigma %u: offset %zu", name, sigma, d);
    for (uint32_t r = 0; r < m.rows; ++r) {
        uint32_t held = 0, split = kDiaNoSplit;
        for (uint32_t k = m.rp[r]; k < m.rp[r + 1]; ++k) {
            const uint32_t d = static_cast<uint32_t>(
              std::lower_bound(offs.begin(), offs.end(), int64_t{m.ci[k]} - r) - offs.begin());
            held |= 1u << d;
            // the first element in another lane than the row's first
            if (split == kDiaNoSplit && k / sigma != m.rp[r] / sigma && m.rp[r + 1] - m.rp[r] <= sigma)
                split = d;
        }
        EXPECT(f.dia_meta[r] == (held | split << kDiaSplitShift), "%s sigma %u: row %u has %x, not %x", name, sigma, r,
               f.dia_meta[r], held | split << kDiaSplitShift);
    }
}

} // namespace

int main() {
    std::mt19937 g(1);
    const std::vector<std::vector<int64_t>> forms = {
      {0}, {-1, 0, 1}, {-64, -1, 0, 1}, {-64, -1, 0, 1, 64}, {-300, -17, -1, 0, 1, 17, 300}, {-9, -5, -2, -1, 0, 1, 2, 5},
      {-33, -32, -31, -1, 0, 1, 31, 32, 33}, {-40, -30, -20, -10, 0, 10, 20, 30, 40, 50},
      {-8, -7, -6, -5, -4, -3, -2, -1, 0, 1, 2, 3, 4, 5, 6, 7}, {-9, -8, -7, -6, -5, -4, -3, -2, -1, 0, 1, 2, 3, 4, 5, 6, 7}};
    for (uint32_t sigma : {4u, 7u, 16u})
        for (uint32_t rows : {1u, 63u, 4096u, 20011u})
            for (size_t i = 0; i < forms.size(); ++i)
                for (double drop : {0.0, 0.1}) {
                    if (rows == 20011 && sigma != 7)
                        continue;
                    char name[64];
                    std::snprintf(name, sizeof name, "form %zu rows %u drop %g", i, rows, drop);
                    Csr m = banded(rows, forms[i], drop, g);
                    check(name, m, sigma, true);
                    if (rows < 4096)
                        continue;
                    // a diagonal that one row has, anywhere
                    for (int q = 0; q < 2; ++q) {
                        Csr one = m;
                        const uint32_t r = g() % (rows - 1000);
                        one.ci.insert(one.ci.begin() + one.rp[r + 1], r + 900);
                        for (uint32_t k = r + 1; k <= rows; ++k)
                            ++one.rp[k];
                        check("one more", one, sigma, true);
                        if (q == 0 && i) { // columns of one row out of order
                            Csr mixed = m;
                            std::swap(mixed.ci[mixed.rp[r]], mixed.ci[mixed.rp[r + 1] - 1]);
                            check("out of order", mixed, sigma, mixed.rp[r + 1] - mixed.rp[r] < 2);
                        }
                    }
                }
    std::printf("done, %d failures\n", g_fail);
    return g_fail != 0;
}
