// The draws of dxg::Normals against std::normal_distribution<float> on the same
// generator, through restarts after an odd and an even number of draws.
#include "normals.hpp"

#include <cstdio>

int main()
{
    for (unsigned long long seed : { 0ull, 1ull, 7ull, 12345ull, 0xfedcba9876543210ull }) {
        dxg::Normals ours;
        ours.rng.seed(seed);
        std::mt19937_64 rng(seed);
        for (int draws : { 3456, 27648, 27647, 1, 2 }) {
            const float sd = std::sqrt(2.0f / static_cast<float>(draws));
            ours.has_kept = false;
            std::normal_distribution<float> theirs(0.0f, sd);
            for (int k = 0; k < draws; ++k) {
                const float a = ours.draw() * sd, b = theirs(rng);
                if (a != b) {
                    std::printf("seed %llu, draw %d of %d: %.9g, standard library %.9g\n", seed, k, draws, a, b);
                    return 1;
                }
            }
        }
    }
    return 0;
}
