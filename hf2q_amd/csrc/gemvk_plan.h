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
inline uint32_t krows_load(uint32_t nsb, uint32_t kp, uint32_t rg) {
    uint32_t simd[4] = {0, 0, 0, 0}, load = 0;
    for (uint32_t i = 0; i < rg * kp; ++i) simd[i % 4u] += nsb / kp + (i % kp < nsb % kp ? 1u : 0u);
    for (uint32_t i = 0; i < 4u; ++i) load = simd[i] > load ? simd[i] : load;
    return load;
}
inline KSplit krows_split(uint32_t nsb, uint32_t units, uint32_t m, uint32_t cus, uint32_t s, uint32_t w) {
    KSplit best{s, w, 0, 0, 0};
    for (uint32_t kp = (nsb + s - 1u) / s; kp <= w && kp <= nsb; ++kp) {
        if (m > 2u * kp) continue;  // (a wave adds up the parts of at most two rows of a group)
        for (uint32_t rg = 1; rg <= 4u && rg * kp <= w && (rg == 1u || units >= 2u * rg * cus); ++rg) {
            const uint32_t load = krows_load(nsb, kp, rg), mine = load * (best.kp ? best.rg : 1u), theirs = best.load * rg;
            if (!best.kp || mine < theirs || (mine == theirs && rg * kp > best.rg * best.kp)) best = KSplit{s, w, kp, rg, load};
        }
    }
    return best;
}

// The form of a launch over nsb super-blocks, which waves share a group's k, by super-blocks per wave and the waves that the registers then allow (512 per SIMD lane; 32 to 34 per
// super-block and operand and about sixty others; Q6_K has no room for sixteen waves of two).  Sixteen waves of two only where twelve would
// all have two: k = 5120 over 17408 rows 21.2 us with sixteen, 19.8 with twelve, slices of 24 super-blocks of 4096 x 12288 21.0 and 23.2.
inline KSplit krows_form_of(bool q6k, bool f32, uint32_t m, uint32_t nsb, uint32_t units, uint32_t cus) {
    const KSplit one = krows_split(nsb, units, m, cus, 1, 16);
    if (f32 && m > 5u) return one;  // two operands
    const KSplit two = krows_split(nsb, units, m, cus, 2, 12), three = krows_split(nsb, units, m, cus, 3, 12);
    if (one.kp && one.load * two.rg <= two.load * one.rg && one.load * three.rg <= three.load * one.rg) return one;
    if (!q6k && nsb > 20u && nsb <= 24u) return krows_split(nsb, units, m, cus, 2, 16);
    return two.kp && two.load * three.rg <= three.load * two.rg ? two : three;
}

// And how many groups side by side: more than that where it takes fewer rounds, by the work of the busiest SIMD over all rounds, and for four waves to a
// group, one to a SIMD with nothing to hide its latencies behind, also where the work is the same.  Which waves add up a group stays that of
// the form, and so do the bits.  us, one group / two or three: 8192 x 1024 bf16 Q5_K at five rows 6.3 / 5.7, 12288 x 1024 f32 Q4_0 at four 8.5 / 7.3, 12288 x 1280 f32 Q6_K at
// eight 16.0 / 13.8, 14336 x 1024 bf16 Q4_K at five 8.2 / 6.8, 20480 x 1280 (two / three) 0.91 of the time over all types.  (Four for two of four waves,
// 16384 x 1024: up to 1.07 of it.)
inline KSplit krows_form(bool q6k, bool f32, uint32_t m, uint32_t nsb, uint32_t units, uint32_t cus) {
    KSplit p = krows_form_of(q6k, f32, m, nsb, units, cus);
    if (!p.kp) return p;
    uint32_t least = (units + p.rg * cus - 1u) / (p.rg * cus) * p.load;
    for (uint32_t rg = p.rg + 1u; rg <= 4u && rg * p.kp <= p.w && units >= rg * cus; ++rg) {
        const uint32_t load = krows_load(nsb, p.kp, rg), all = (units + rg * cus - 1u) / (rg * cus) * load;
        if (all < least || (all == least && p.rg * p.kp <= 4u)) least = all, p.rg = rg, p.load = load;
    }
    return p;
}

}  // namespace hq
