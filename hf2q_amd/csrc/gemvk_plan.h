// How the products of a few rows with the activations in registers (gemvk.h) are dealt out: slices of k, waves, super-blocks per wave.
// Host arithmetic alone, no HIP.
#pragma once

#include <stdint.h>

namespace hq {

// Slices of k, a launch each: as many super-blocks as the registers of a workgroup hold, 16 with two operands (six to eight f32 rows), else 36.
// The super-blocks are spread evenly: a short last slice would have too few waves to add up the parts of its rows.
inline uint32_t krows_slices(uint32_t nsb, bool f32, uint32_t m) {
    const uint32_t cap = f32 && m > 5u ? 16u : 36u;
    return (nsb + cap - 1u) / cap;
}
inline uint32_t krows_slice_blocks(uint32_t nsb, uint32_t slices, uint32_t i) { return nsb / slices + (i < nsb % slices ? 1u : 0u); }

// How nsb super-blocks are dealt out: kp waves to a group of sixteen rows, rg groups side by side, at most s super-blocks to a wave and w
// waves.  What counts is the work of the busiest SIMD (wave i runs on SIMD i % 4) per group, then the waves that hide the latencies.
struct KSplit {
    uint32_t s, w, kp, rg, load;  // kp 0: none; load: super-blocks of the busiest SIMD
};
inline KSplit krows_split(uint32_t nsb, uint32_t units, uint32_t m, uint32_t cus, uint32_t s, uint32_t w) {
    KSplit best{s, w, 0, 0, 0};
    for (uint32_t kp = (nsb + s - 1u) / s; kp <= w && kp <= nsb; ++kp) {
        if (m > 2u * kp) continue;  // (a wave adds up the parts of at most two rows of a group)
        const uint32_t base = nsb / kp, extra = nsb % kp;
        for (uint32_t rg = 1; rg <= 4u && rg * kp <= w && (rg == 1u || units >= 2u * rg * cus); ++rg) {
            uint32_t simd[4] = {0, 0, 0, 0}, load = 0;
            for (uint32_t i = 0; i < rg * kp; ++i) simd[i % 4u] += base + (i % kp < extra ? 1u : 0u);
            for (uint32_t i = 0; i < 4u; ++i) load = simd[i] > load ? simd[i] : load;
            const uint32_t mine = load * (best.kp ? best.rg : 1u), theirs = best.load * rg;
            if (!best.kp || mine < theirs || (mine == theirs && rg * kp > best.rg * best.kp)) best = KSplit{s, w, kp, rg, load};
        }
    }
    return best;
}

// The form of a launch over nsb super-blocks, by super-blocks per wave and the waves that the registers then allow (512 per SIMD lane; 32 to 34 per
// super-block and operand and about sixty others; Q6_K has no room for sixteen waves of two).  Sixteen waves of two only where twelve would
// all have two: k = 5120 over 17408 rows 21.2 us with sixteen, 19.8 with twelve, slices of 24 super-blocks of 4096 x 12288 21.0 and 23.2.
inline KSplit krows_form(bool q6k, bool f32, uint32_t m, uint32_t nsb, uint32_t units, uint32_t cus) {
    const KSplit one = krows_split(nsb, units, m, cus, 1, 16);
    if (f32 && m > 5u) return one;  // two operands
    const KSplit two = krows_split(nsb, units, m, cus, 2, 12), three = krows_split(nsb, units, m, cus, 3, 12);
    if (one.kp && one.load * two.rg <= two.load * one.rg && one.load * three.rg <= three.load * one.rg) return one;
    if (!q6k && nsb > 20u && nsb <= 24u) return krows_split(nsb, units, m, cus, 2, 16);
    return two.kp && two.load * three.rg <= three.load * two.rg ? two : three;
}

}  // namespace hq
