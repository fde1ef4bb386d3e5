// Compares line_reach with the offsets of every group, over random arrays; prints the number compared.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "line_reach.h"

using namespace ifft;

static long long offset(const LineMap &m, long long line)
{
    long long off = 0;
    for (int d = m.nd - 1; d >= 0; --d) {
        off += (line % m.cnt[d]) * m.st[d];
        line /= m.cnt[d];
    }
    return off;
}

int main()
{
    std::mt19937 rng(1);
    auto pick = [&](int n) { return (int)(rng() % (unsigned)n); };
    int n = 0;
    for (int trial = 0; trial < 40000; ++trial) {
        LineMap m{};
        m.nd = pick(5);
        long long lines = 1, next = 1 + pick(3);
        for (int d = m.nd - 1; d >= 0; --d) {
            m.cnt[d] = pick(4) ? 1 + pick(12) : 1;
            // packed, padded, broadcast or anything, of either sign
            const int kind = pick(8);
            m.st[d] = kind < 4 ? next : kind < 6 ? next + 1 + pick(5) : kind < 7 ? 0 : pick(50);
            if (pick(6) == 0) m.st[d] = -m.st[d];
            next = std::llabs(m.st[d]) * m.cnt[d] + (m.st[d] ? 0 : next);
            lines *= m.cnt[d];
        }
        const int tbs[] = {1, 2, 3, 4, 5, 8, 16, 42, 64};
        const long long tb = tbs[pick(9)];
        long long lo, hi, span_lo = 0, span_hi = 0;
        line_reach(m, tb, lo, hi);
        for (long long l0 = 0; l0 < lines; l0 += tb)
            for (long long l = l0; l < lines && l < l0 + tb; ++l) {
                const long long o = offset(m, l) - offset(m, l0);
                span_lo = std::min(span_lo, o);
                span_hi = std::max(span_hi, o);
            }
        bool even = true;   // one dimension left after merging: the bounds are exact
        int left = 0;
        for (int d = 0; d < m.nd; ++d) left += m.cnt[d] > 1;
        even = left <= 1;
        if (lo > span_lo || hi < span_hi || (even && (lo != span_lo || hi != span_hi))) {
            std::printf("trial %d tb %lld: [%lld, %lld] holds [%lld, %lld]\n", trial, tb, lo, hi, span_lo, span_hi);
            return 1;
        }
        ++n;
    }
    std::printf("%d\n", n);
    return 0;
}
