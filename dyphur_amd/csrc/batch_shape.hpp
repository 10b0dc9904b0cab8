// batch_shape.hpp — which scenes of a batch get a workgroup of their own
// (host code only).
#pragma once

#include <algorithm>
#include <cstdint>
#include <functional>
#include <vector>

namespace dy {

// Default of the launch shape's wave_scene_max for scenes of off[i + 1] - off[i]
// bodies, when the device holds `slots` workgroups of 256 threads at once: 32
// (scenes past 32 bodies a workgroup each) or 128 (a wavefront each up to 128).
//
// A workgroup steps a scene sooner (10 frames of settled columns: 33 bodies
// 820 against 890 us, 64 1 165 / 1 530, 128 1 560 / 2 750; below, in units of 2 us),
// but takes the place of four wavefronts.  So it is worth it where the longest
// scene decides, and not where the workgroups need the chip twice over: the
// estimate is the longest scene's time, and with more workgroups than slots
// that of two in a row at the place where the second round starts.
//
// Workgroup over wavefront form, measured at 512 slots: 512 scenes of 33, 64, 128
// bodies 1.11, 1.21, 1.55, 600 scenes 0.66, 0.77, 0.95; of lognormal sizes around
// 48, at most 257: 300 scenes 1.02, 768 1.08, 1 024 1.04, 1 500 0.94; around 64,
// at most 513 (whose workgroups decide in both forms): 0.96 to 1.00 at any
// count.  Recording, at 256 slots: 256 scenes of 33, 64, 128 bodies 1.16, 1.37,
// 1.78, 300 scenes 0.70, 0.84, 1.03; lognormal around 48: 600 scenes 1.17, 768 0.98,
// 1 024 0.77.
inline uint32_t batch_wave_max(const uint32_t *off, uint32_t n_scenes, uint32_t slots) {
    constexpr uint32_t kFew = 32, kMany = 128;
    const auto wave = [](uint32_t n) { return 10u * n + 120u; };
    const auto group = [](uint32_t n) { return 4u * n + 290u; };
    std::vector<uint32_t> big;
    uint32_t longest_wave = 0;
    for (uint32_t i = 0; i < n_scenes; ++i) {
        const uint32_t n = off[i + 1] - off[i];
        if (n <= kFew) continue;
        big.push_back(n);
        if (n <= kMany) longest_wave = std::max(longest_wave, n);
    }
    if (longest_wave == 0 || slots == 0 || big.size() > 2ull * slots) return kMany;
    std::sort(big.begin(), big.end(), std::greater<uint32_t>());
    const uint32_t as_waves = std::max(wave(longest_wave), big[0] > kMany ? group(big[0]) : 0u);
    uint32_t as_groups = group(big[0]);
    if (big.size() > slots) as_groups = std::max(as_groups, group(big[slots - 1]) + group(big[slots]));
    return as_groups < as_waves ? kFew : kMany;
}

}  // namespace dy
