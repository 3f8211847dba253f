// Host check of the FP64 stage's division policy (vh::DivTry): whatever it
// accepts has the division operator's bits, and it accepts what it says it
// does.  Prints one line per part, "mismatches M refused R of N".
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../cpu-vh_amd/csrc/vh_device.hpp"

namespace {

std::mt19937_64 rng(2024);

// sign and mantissa at random (some mantissas all zeros or all ones), |x| in [2^k, 2^(k+1)), k >= -1074
double make(int k, bool positive) {
    uint64_t m = rng() & ((1ull << 52) - 1);
    const unsigned pick = rng() & 15;
    if (pick == 0) m = 0;
    if (pick == 1) m = (1ull << 52) - 2;
    uint64_t u;
    if (k >= -1022) u = ((uint64_t)(k + 1023) << 52) | m;
    else u = (1ull << (k + 1074)) | (m & ((1ull << (k + 1074)) - 1));
    if (!positive && (rng() & 1)) u |= 1ull << 63;
    double x;
    std::memcpy(&x, &u, 8);
    return x;
}
int between(int lo, int hi) { return lo + (int)(rng() % (uint64_t)(hi - lo + 1)); }

bool same(double x, double y) { return std::memcmp(&x, &y, 8) == 0; }

// numerators of exponents [alo, ahi], divisors of [blo, bhi]
long part(const char *name, long n, int alo, int ahi, int blo, int bhi, bool all_accepted) {
    long bad = 0, refused = 0;
    for (long i = 0; i < n; ++i) {
        const double a = alo > ahi ? (rng() & 1 ? 0.0 : -0.0) : make(between(alo, ahi), false);
        const double b = make(between(blo, bhi), true);
        vh::DivTry d;
        const double q = d(a, d.recip(b));
        d.see(q);
        if (d.fails()) ++refused;
        else if (!same(q, a / b)) ++bad;
    }
    const bool wrong = bad || (all_accepted && refused);
    std::printf("%s: mismatches %ld refused %ld of %ld%s\n", name, bad, refused, n, wrong ? " WRONG" : "");
    return wrong;
}

// quotients by 3 and 5: nothing refused
long by_integers(const char *name, long n, int alo, int ahi) {
    const vh::IntRecip r3{3.0, 1.0 / 3.0}, r5{5.0, 1.0 / 5.0};
    long bad = 0, refused = 0;
    for (long i = 0; i < n; ++i) {
        const double a = i < 4096 ? (i & 1 ? -1 : 1) * (double)(i >> 1) * 0x1p-1074 : make(between(alo, ahi), false);
        vh::DivTry d;
        const double q3 = d(a, r3), q5 = d(a, r5);
        d.see(q3);
        d.see(q5);
        refused += d.fails();
        bad += !same(q3, a / 3.0) || !same(q5, a / 5.0);
    }
    std::printf("%s: mismatches %ld refused %ld of %ld%s\n", name, bad, refused, n, bad || refused ? " WRONG" : "");
    return bad || refused;
}

}  // namespace

int main(int argc, char **argv) {
    const long n = argc > 1 ? std::atol(argv[1]) : 1000000;
    long wrong = 0;
    wrong += part("ordinary", n, -960, 800, -16, 49, true);
    wrong += part("smallest accepted numerators", n, -969, -960, -16, 49, true);
    wrong += part("zero numerators", n, 1, 0, -16, 49, true);
    // t^3 at t = 0.001, dt = 1e-9: the time's powers and the step are divisors too
    wrong += part("small divisors", n, -900, 800, -100, -16, true);
    wrong += part("small numerators", n, -1000, -950, -16, 49, false);
    wrong += part("subnormal quotients", n, -1074, -1000, -16, 49, false);
    wrong += part("quotients of the last bits", n, -1074, -1060, -4, 8, false);
    wrong += part("overflowing quotients", n, 1000, 1023, -16, 20, false);
    wrong += part("divisors outside", n, -960, 800, -140, 140, false);
    wrong += by_integers("thirds and fifths", n, -1022, 1023);
    wrong += by_integers("subnormal thirds and fifths", n, -1074, -1000);
    return wrong ? 1 : 0;
}
