// Host model of two vh_fo_flag_noalloc calls that overlap in the fixed
// scratch: their passes' blocks in random order, each call's own order kept.
// The ids either writes stay inside its arrays, and one call after the other
// gives exactly its cut cubes.
#include <cstdio>
#include <random>
#include <vector>

#include "../cpu-vh_amd/csrc/vh_kernels.hpp"

namespace {

constexpr long MAX_CUBES = 1 << 15;  // of the model's scratch
std::vector<unsigned long long> scratch(vh::fo_flag_scratch(MAX_CUBES));
unsigned long long *const counts = scratch.data(), *const masks = scratch.data() + vh::fo_flag_blocks(MAX_CUBES);

struct Call {
    long M, cap;
    std::vector<bool> cut;
    std::vector<long long> ids;
    unsigned long long count = 0;
    long next = 0;  // step: the blocks of pass 1, the scan, the blocks of pass 3
    bool ok = true;
    Call(long cubes, long room, double share, std::mt19937 &r) : M(cubes), cap(room), cut(cubes), ids(room, -1) {
        for (long c = 0; c < M; ++c) cut[c] = r() < share * 4294967296.0;
    }
    long blocks() const { return vh::fo_flag_blocks(M); }
    bool done() const { return next == 2 * blocks() + 1; }
    void step() {
        const long nb = blocks(), k = next++;
        if (k < nb) {
            unsigned long long n = 0;
            for (int w = 0; w < 4; ++w) {
                unsigned long long m = 0;
                for (int l = 0; l < 64; ++l) {
                    const long c = k * 256 + w * 64 + l;
                    if (c < M && cut[c]) m |= 1ull << l;
                }
                masks[k * 4 + w] = m;
                n += (unsigned long long)__builtin_popcountll(m);
            }
            counts[k] = n;
        } else if (k == nb) {
            unsigned long long sum = 0;
            for (long i = 0; i < nb; ++i) {
                const unsigned long long v = counts[i];
                counts[i] = sum;
                sum += v;
            }
            count = sum;
            ok = ok && count < (1ull << 62);
        } else {
            const long b = k - nb - 1;
            const unsigned long long *m = masks + b * 4;
            for (int w = 0; w < 4; ++w)
                for (int l = 0; l < 64; ++l) {
                    const long long pos = vh::fo_flag_place(counts[b], m[0], m[1], m[2], m[3], w, l, b * 256, M, cap);
                    if (pos < 0) continue;
                    const long long c = b * 256 + w * 64 + l;
                    if (pos >= cap || c >= M) ok = false;
                    else ids[(size_t)pos] = c;
                }
        }
    }
    bool exact() const {
        long n = 0;
        for (long c = 0; c < M; ++c)
            if (cut[c]) {
                if (n < cap && ids[(size_t)n] != c) return false;
                ++n;
            }
        for (long k = n; k < cap; ++k)
            if (ids[(size_t)k] != -1) return false;
        return count == (unsigned long long)n;
    }
};

}  // namespace

int main() {
    std::mt19937 r(7);
    const long sizes[] = {1, 63, 255, 256, 257, 4096, 5000, MAX_CUBES};
    long bad = 0, cases = 0;
    for (long Ma : sizes)
        for (long Mb : sizes)
            for (int trial = 0; trial < 60; ++trial) {
                const double share = trial % 3 == 0 ? 1.0 : 0.3;
                Call a(Ma, trial % 2 ? Ma : Ma / 2, share, r), b(Mb, Mb, trial % 5 == 0 ? 0.99 : 0.2, r);
                while (!a.done() || !b.done()) {
                    Call &c = a.done() ? b : (b.done() ? a : (r() & 1 ? a : b));
                    for (long run = 1 + (long)(r() % 40); run > 0 && !c.done(); --run) c.step();
                }
                bad += !a.ok || !b.ok;
                Call s(Ma, a.cap, share, r);
                while (!s.done()) s.step();
                bad += !s.ok || !s.exact();
                ++cases;
            }
    std::printf("cases %ld bad %ld\n", cases, bad);
    return bad ? 1 : 0;
}
