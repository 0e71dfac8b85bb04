// Standard normal draws of the denoiser's initial weights.
#pragma once

#include <algorithm>
#include <cmath>
#include <random>

namespace dxg {

// Standard normals by Marsaglia's polar method in FP32 from 64-bit draws: the
// values std::normal_distribution<float> gives here, without its two long
// double logarithms per pair (444,000 draws: 31 ms with it, 9 ms without).
struct Normals {
    std::mt19937_64 rng;
    float kept = 0.0f;
    bool has_kept = false;
    float uniform() { return std::min(static_cast<float>(rng()) * 0x1p-64f, 0x1.fffffep-1f); }
    float draw()
    {
        if (has_kept) {
            has_kept = false;
            return kept;
        }
        float x, y, r2;
        do {
            x = 2.0f * uniform() - 1.0f;
            y = 2.0f * uniform() - 1.0f;
            r2 = x * x + y * y;
        } while (r2 > 1.0f || r2 == 0.0f);
        const float m = std::sqrt(-2.0f * std::log(r2) / r2);
        kept = x * m;
        has_kept = true;
        return y * m;
    }
};

}  // namespace dxg
