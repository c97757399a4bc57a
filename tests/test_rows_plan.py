"""CPU checks of the plan behind the products of a few rows with the activations in registers: the host arithmetic is compiled by itself."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <initializer_list>
#include <stdio.h>
#include "gemvk_plan.h"
int main() {
    using namespace hq;
    unsigned long launches = 0;
    for (uint32_t nsb = 4; nsb <= 400; ++nsb)
        for (uint32_t m = 2; m <= 8; ++m)
            for (int f32 = 0; f32 < 2; ++f32) {
                const uint32_t slices = krows_slices(nsb, f32, m);
                uint32_t all = 0;
                for (uint32_t i = 0; i < slices; ++i) {
                    const uint32_t n = krows_slice_blocks(nsb, slices, i);
                    all += n;
                    for (uint32_t units : {1u, 3u, 256u, 1023u, 2048u, 16416u})
                        for (int q6k = 0; q6k < 2; ++q6k, ++launches) {
                            const KSplit p = krows_form(q6k, f32, m, n, units, 256);
                            const bool two = f32 && m > 5;  // operands: the kernel has one super-block to a wave then
                            if (!p.kp || !p.rg || p.kp * p.rg > p.w || (n + p.kp - 1) / p.kp > p.s || n < p.kp || p.rg * m > 2 * p.kp * p.rg || p.rg > 4 ||
                                (p.s == 1 ? p.w != 16 : p.w != 12 && (q6k || p.s != 2)) || (two && p.s != 1) || p.s > 3) {
                                printf("%u rows, %u super-blocks (%u of them, slice %u), f32 %d, %u groups: kp %u rg %u s %u w %u\n", m, nsb, n, i, f32, units, p.kp, p.rg, p.s, p.w);
                                return 1;
                            }
                        }
                }
                if (all != nsb) return printf("%u super-blocks in %u slices are %u\n", nsb, slices, all), 1;
            }
    printf("%lu launches\n", launches);
    return 0;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")

    def run(program):
        src, exe = d / "plan.cpp", d / "plan"
        src.write_text(program)
        subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "hf2q_amd", "csrc"), str(src), "-o", str(exe)], check=True)
        return subprocess.run([str(exe)], capture_output=True, text=True)

    return run


def test_every_slice_of_every_length_has_a_split(plan):
    """Rows of up to 400 super-blocks, two to eight of them: no slice is left without waves to add up its rows (54016 weights over eight f32
    rows once ended in a slice of three super-blocks, for which there is none), and every split is one that the kernel has a form for."""
    r = plan(PROGRAM)
    assert r.returncode == 0, r.stdout + r.stderr


GROUPS = r"""
#include <stdio.h>
#include "gemvk_plan.h"
int main() {
    using namespace hq;
    const uint32_t cus = 256;
    unsigned more = 0;
    for (uint32_t nsb = 4; nsb <= 36; ++nsb)
        for (uint32_t m = 2; m <= 8; ++m)
            for (uint32_t units = 1; units <= 4200; ++units)
                for (int f32 = 0; f32 < 2; ++f32) {
                    if (f32 && m > 5 && nsb > 16) continue;
                    const KSplit p = krows_form_of(false, f32, m, nsb, units, cus), q = krows_form(false, f32, m, nsb, units, cus);
                    more += q.rg != p.rg;
                    auto all = [&](const KSplit& x) { return (units + x.rg * cus - 1) / (x.rg * cus) * krows_load(nsb, x.kp, x.rg); };
                    if (q.kp != p.kp || q.s != p.s || q.w != p.w || q.rg < p.rg || q.rg > 4 || q.rg * q.kp > q.w || all(q) > all(p) || q.load != krows_load(nsb, q.kp, q.rg) ||
                        (q.rg > p.rg && units < q.rg * cus))
                        return printf("%u super-blocks, %u rows, %u groups: kp %u rg %u -> kp %u rg %u\n", nsb, m, units, p.kp, p.rg, q.kp, q.rg), 1;
                }
    return more == 0;
}
"""


def test_groups_side_by_side_leave_the_sums_alone(plan):
    """More groups side by side: the same waves to a group, no more work on a SIMD over all rounds, no CU without a group, within the kernel's waves."""
    r = plan(GROUPS)
    assert r.returncode == 0, r.stdout + r.stderr
