// Host build of the column division (limbforge_amd/csrc/div_core.hpp) against Knuth's division of limb_core.hpp over
// structured and random mantissas, exponents at their limits, zeros and statuses: where it decides, the same bits;
// and among random operands it decides all but a few.  Test infrastructure: compiled by tests/test_div_core_cpu.py
// with LF_HOST_BUILD defined.
#include "div_core.hpp"
#include <cstdio>
#include <random>

static long failures = 0;

template <int N> lf::Num<N> value(std::mt19937_64& rng, int kind)
{
    static const uint32_t edge[8] = {0, 1, 2, 0x7fffffff, 0x80000000, 0x80000001, 0xfffffffe, 0xffffffff};
    lf::Num<N> x;
    for (int i = 0; i < N; ++i) {
        const uint32_t r = (uint32_t)rng();
        x.w[i] = kind == 1 ? ((r & 1) ? 0xffffffffu : 0u) : kind == 2 ? 0u : kind == 3 ? 0xffffffffu : kind == 4 ? edge[r & 7] : r;
    }
    x.w[N - 1] |= 0x80000000u;
    if (kind == 2 && (rng() & 1)) x.w[0] |= 1;
    x.e = (int)(rng() % 1000) - 500;
    if (rng() % 50 == 0) x.e = 1000000000 - (int)(rng() % 3);
    if (rng() % 50 == 0) x.e = -1000000000 + (int)(rng() % 3);
    x.s = (rng() & 1) ? 1 : -1;
    x.st = 0;
    if (rng() % 40 == 0) x = lf::zero<N>(0);
    if (rng() % 60 == 0) x.st = 1 + rng() % 7;
    return x;
}

template <int N> void run(int cases)
{
    std::mt19937_64 rng(1000 + N);
    long undecided = 0, plain = 0;
    for (int c = 0; c < cases; ++c) {
        const int ka = (int)(rng() % 5), kb = (int)(rng() % 5);
        auto a = value<N>(rng, ka);
        const auto b = value<N>(rng, kb);
        const bool near = rng() % 10 == 0;
        if (near) {
            for (int i = 0; i < N; ++i) a.w[i] = b.w[i];
            a.w[0] ^= (uint32_t)(rng() % 3);
        }
        lf::Num<N> z;
        const bool ok = lf::cd_div<N>(a, b, lf::cd_divisor<N>(b.w), z);
        if (!ka && !kb && !near) {
            ++plain;
            undecided += !ok;
        }
        if (!ok) continue;
        const auto want = lf::div<N>(a, b);
        bool same = z.e == want.e && z.s == want.s && z.st == want.st;
        for (int i = 0; i < N; ++i) same = same && z.w[i] == want.w[i];
        if (!same && ++failures <= 10) std::printf("MISMATCH bits=%d case=%d kinds %d %d\n", 32 * N, c, ka, kb);
    }
    if (undecided > 2) { // expected: plain * 2^-24
        ++failures;
        std::printf("bits=%d: %ld of %ld random quotients undecided\n", 32 * N, undecided, plain);
    }
}

template <int N> void all(int cases)
{
    run<N>(cases);
    if constexpr (N < 32) all<N + 1>(cases);
}

int main()
{
    all<2>(20000);
    std::printf("%ld failures\n", failures);
    return failures ? 1 : 0;
}
