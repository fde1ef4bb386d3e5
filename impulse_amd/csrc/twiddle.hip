// Host FP64 twiddle generation.
//
// exp(-2 pi i k / n) is evaluated in long double after an exact integer
// reduction of the angle to the first octant, then rounded to double.  Angles
// that are multiples of pi/4 therefore come out exactly (0, +-1, +-sqrt(1/2)),
// which the reference's exact known-answer tests rely on
// (tests/test_fft2.nim:7-15); PocketFFT obtains the same property by its own
// octant reduction (impulse/fft/cpp_pocketfft/pocketfft_hdronly.h:277-349).
#include <algorithm>
#include <cmath>

#include "engine.h"

namespace ifft {

static const long double kPiL = 3.141592653589793238462643383279502884L;

double2 twiddle_at(uint64_t k, uint64_t n)
{
    k %= n;
    const unsigned __int128 x = (unsigned __int128)8u * k;
    const uint64_t oct = (uint64_t)(x / n);
    const uint64_t r = (uint64_t)(x - (unsigned __int128)oct * n);
    long double c, s;
    if ((oct & 1u) == 0) {
        const long double a = (kPiL / 4.0L) * ((long double)r / (long double)n);
        c = cosl(a);
        s = sinl(a);
    } else if (r == 0) {
        c = s = sqrtl(0.5L);
    } else {
        const long double a = (kPiL / 4.0L) * ((long double)(n - r) / (long double)n);
        c = cosl(a);
        s = sinl(a);
    }
    long double re, im;  // cos / sin of 2 pi k / n
    switch (oct) {
        case 0: re = c; im = s; break;
        case 1: re = s; im = c; break;
        case 2: re = -s; im = c; break;
        case 3: re = -c; im = s; break;
        case 4: re = -c; im = -s; break;
        case 5: re = -s; im = -c; break;
        case 6: re = s; im = -c; break;
        default: re = c; im = -s; break;
    }
    return make_double2((double)re, (double)-im);
}

// out[j] = W_n^{j * step}, j < count
void twiddle_table(std::vector<double2> &out, uint64_t n, uint64_t count, uint64_t step)
{
    out.resize(count);
    for (uint64_t j = 0; j < count; ++j)
        out[j] = twiddle_at((uint64_t)(((unsigned __int128)j * step) % n), n);
}

// ---------------------------------------------------------------------------
// mixed-radix shapes (mix_fft.h)
// ---------------------------------------------------------------------------

// VALU operations of one radix-R butterfly, counted from the code
int mix_ops(int R)
{
    static const int ops[17] = {0, 0, 4, 16, 16, 40, 44, 72, 60, 120, 100, 160, 112, 216, 172, 200, 170};
    return ops[R];
}

// Factors N into min_stages .. 6 radices of 2 .. 16 and the threads per transform they take, or returns
// false.  The cheapest order by operation count wins (of equals the one with the smaller radices first): butterflies,
// twiddle products, the LDS accesses of each stage with the bank conflicts of the first stage's writes
// (their stride is the radix: 16-byte words fall on 8 bank groups, so an odd first radix has none), and
// the per-stage overhead of every thread.  A plan tries many lengths: the search leaves
// a branch as soon as the rest needs more stages than are left or, by a bound from below, costs more
// than the best (8 us a length on average and 40 at most, 62 and 1,200 without).
bool mix_factor(int N, int max_threads, std::vector<int> &radices, int &threads, double *cost_out,
                int min_stages)
{
    if (N < (min_stages > 1 ? 4 : 2)) return false;
    double best = -1.0;
    std::vector<int> cur;
    auto nb_of = [](int R) { return R > 8 ? 1 : 16 / R; };   // mix_nb
    int most = 2;   // two stages over the fewest there could be reach every 13-smooth length (5^5, 7^4, ...)
    for (long long v = 1; v < N; v *= 16) ++most;
    most = std::min(most, 6);   // kMixMaxStages
    // a stage past the first costs its butterflies at least this per bit of its radix and point
    static const double per_bit = [] {
        double least = 1e300;
        for (int R = 2; R <= 16; ++R)
            least = std::min(least, (double)(mix_ops(R) + 4 * (R - 1) + 10 * R) / (R * std::log2((double)R)));
        return least * (1.0 - 1e-9);
    }();
    // n: what is left to factor; ops, nt: of the stages so far, their costs whole numbers
    auto rec = [&](auto &&self, int n, double ops, int nt) -> void {
        const int k = (int)cur.size();
        if (n == 1 && k >= min_stages) {
            int g = cur[0];
            g = (g & 1) ? 1 : (g & 2) ? 2 : (g & 4) ? 4 : 8;   // gcd with the 8 bank groups
            const double cost = ops + 60.0 * nt * k + 4.0 * N * (g - 1);
            if (best < 0.0 || cost < best || (cost == best && cur < radices)) {
                best = cost;
                radices = cur;
                threads = nt;
            }
            return;
        }
        const int left = most - k;
        if (left <= 0 || n > 1LL << (4 * left)) return;
        if (best >= 0.0 && k && ops + 60.0 * nt * k + per_bit * N * std::log2((double)n) > best) return;
        // past the first stage the order costs nothing: ascending radices stand for all orders
        for (int R = 16; R >= (k > 1 ? cur.back() : 2); --R)
            if (n % R == 0) {
                const int t = std::max(nt, (N / R + nb_of(R) - 1) / nb_of(R));
                if (t > max_threads) continue;
                cur.push_back(R);
                self(self, n / R, ops + (double)(N / R) * (mix_ops(R) + (k ? 4 * (R - 1) : 0) + 10 * R), t);
                cur.pop_back();
            }
    };
    rec(rec, N, 0.0, 1);
    if (cost_out) *cost_out = best;
    return best >= 0.0;
}

// the twiddles of stages 1, 2, ... in stage order: W_{pR}^{qk} at (q - 1) p + k, q = 1 .. R - 1,
// k < p, p the product of the earlier radices; conjugated for sign > 0
void mix_table(std::vector<double2> &out, const std::vector<int> &radices, int sign)
{
    out.clear();
    int p = radices[0];
    for (size_t s = 1; s < radices.size(); ++s) {
        const int R = radices[s];
        for (int q = 1; q < R; ++q)
            for (int k = 0; k < p; ++k) {
                double2 w = twiddle_at((uint64_t)q * (uint64_t)k, (uint64_t)p * (uint64_t)R);
                if (sign > 0) w.y = -w.y;
                out.push_back(w);
            }
        p *= R;
    }
}

}  // namespace ifft
