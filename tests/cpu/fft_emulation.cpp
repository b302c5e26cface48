// The in-place transforms of fft_small.h run by one thread, for every length 2^a 3^b 5^c from 8 to
// 256: modes against a direct DFT in 64 bits, forward then inverse against the input, the places of
// the modes a permutation, and no access outside the sequences.  Prints the largest error.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "fft_small.h"

int main()
{
    double worst = 0.0;
    int lengths = 0, deepest = 0;
    for (int n = 8; n <= 256; ++n) {
        int m = n;
        for (int p : {2, 3, 5})
            while (m % p == 0) m /= p;
        if (m != 1) continue;
        ++lengths;
        FftAxis ax;
        ax.n = n;
        if (!fft::split(n, &ax.ns, ax.f)) { std::printf("no radices for %d\n", n); return 1; }
        deepest = ax.ns > deepest ? ax.ns : deepest;
        std::vector<float2> tw(n);
        std::vector<int> seen(n, 0), place(n);
        for (int k = 0; k < n; ++k) {
            const double t = -2.0 * M_PI * k / n;
            tw[k] = make_float2((float)std::cos(t), (float)std::sin(t));
            place[k] = fft::place_of(n, ax.ns, ax.f, k);
            if (place[k] < 0 || place[k] >= n || seen[place[k]]++) { std::printf("places of %d\n", n); return 1; }
        }
        // three sequences with their elements `stride` apart, a guard on both sides
        const int nseq = 3, stride = 5, guard = 64;
        std::vector<float2> in(nseq * n), buf(guard * 2 + nseq * n * stride, make_float2(7.f, 7.f));
        std::srand(n);
        for (auto &v : in) v = make_float2(std::rand() / (float)RAND_MAX - 0.5f, std::rand() / (float)RAND_MAX - 0.5f);
        auto at = [&](int s, int j) -> float2 & { return buf[guard + s * n * stride + j * stride]; };
        for (int s = 0; s < nseq; ++s)
            for (int j = 0; j < n; ++j) at(s, j) = in[s * n + j];
        struct Place {
            fft::FastDiv per;
            int seq;
            int operator()(int idx, int &t) const { return per(idx, t) * seq; }
        };
        auto make = [&](int tasks) { return Place{fft::FastDiv(tasks), n * stride}; };
        fft::transform<false, 1>(buf.data() + guard, ax, nseq, make, stride, tw.data());
        for (int s = 0; s < nseq; ++s)
            for (int k = 0; k < n; ++k) {
                double re = 0, im = 0;
                for (int j = 0; j < n; ++j) {
                    const double t = -2.0 * M_PI * ((long)j * k % n) / n;
                    re += in[s * n + j].x * std::cos(t) - in[s * n + j].y * std::sin(t);
                    im += in[s * n + j].x * std::sin(t) + in[s * n + j].y * std::cos(t);
                }
                const float2 v = at(s, place[k]);
                worst = std::fmax(worst, std::hypot(v.x - re, v.y - im) / std::sqrt((double)n));
            }
        fft::transform<true, 1>(buf.data() + guard, ax, nseq, make, stride, tw.data());
        for (int s = 0; s < nseq; ++s)
            for (int j = 0; j < n; ++j)
                worst = std::fmax(worst, std::hypot(at(s, j).x / n - in[s * n + j].x, at(s, j).y / n - in[s * n + j].y));
        for (size_t q = 0; q < buf.size(); ++q) {
            const long r = (long)q - guard;
            const bool element = r >= 0 && r < nseq * n * stride && r % stride == 0;
            if (!element && (buf[q].x != 7.f || buf[q].y != 7.f)) { std::printf("write outside at %d\n", n); return 1; }
        }
    }
    std::printf("lengths %d stages %d worst %.3e\n", lengths, deepest, worst);
    return 0;
}
