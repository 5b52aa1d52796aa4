// The sharing of splits in a ragged attention batch, on the CPU: reads lines "B S tiles...", prints "L sums linear" for each,
// where `sums` is how many sums the search took and `linear` what a search one by one takes; then the split counts.
#include <cmath>
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>
#include <vector>

#include "../../swiftlm_amd/csrc/sdpa_shares.h"

int main() {
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        int B, S;
        in >> B >> S;
        std::vector<int> nt(B);
        long total = 0;
        int longest = 0;
        for (int& t : nt) { in >> t; total += t; longest = t > longest ? t : longest; }
        const int W = B * S, least = (longest + 511) / 512, even = (int)((total + W - 1) / W), loose = (int)(total / (W - B)) + 1;
        int sums = 0;
        auto fits = [&](int L) {
            ++sums;
            long s = 0;
            for (int t : nt) s += (t + L - 1) / L;
            return s <= W;
        };
        const int lo = even < least ? least : even;
        const int L = dflash::tiles_per_share(lo, longest < loose ? longest : loose, fits);
        const int took = sums;
        int want = lo;
        sums = 0;
        while (!fits(want)) ++want;
        if (want != L) { std::printf("wrong %d %d\n", L, want); return 1; }
        // a reciprocal that is off by two units in the last place either way gives the same counts
        for (int u = -2; u <= 2; ++u) {
            float inv = 1.f / (float)L;
            for (int i = 0; i < (u < 0 ? -u : u); ++i) inv = std::nextafter(inv, u < 0 ? 0.f : 2.f);
            for (int t : nt)
                if ((int)std::floor(dflash::share_quotient((float)t, inv)) + 1 != (t + L - 1) / L) { std::printf("counts %d %d\n", t, L); return 1; }
        }
        std::printf("%d %d %d\n", L, took, sums);
    }
    return 0;
}
