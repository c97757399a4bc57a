// Host side of the kernel in gemvk.h: which products it takes, and its launches.
#include "gemvk.h"

namespace hq {

// Where it is ahead of the kernels that serve a few rows otherwise (and no less exact: 0.9 .. 2e-7 of the result, Q8_0 and Q4_0 rows in bf16 8e-8), or
// behind them and ten to fifty times as exact: k below 2048 and up to 3584 from two rounds of groups on, where the groups' hand-overs are much of the
// product, and heads of K-quants and Q8_0 up to 131072 rows with k up to 4096.  us and error of the result, the others / here: bf16 Q4_K at five rows 4096 x 1024 3.6, 2.6e-6 / 4.9, 1.5e-7,
// 65536 x 1280 16.6 / 18.8; f32 Q6_K at eight 12288 x 1280 9.7, 2.8e-6 / 13.8, 9e-8, 24576 x 2816 22.3 / 30.3; f32 Q4_0 at four 5120 x 1280 5.4, 4.2e-6 / 7.5, 7e-8; f32 Q8_0 at
// three 32768 x 2048 17.5, 2.4e-6 / 22.7, 7e-8, 4352 x 10240 17.4 / 27.8.  In all 17 000 products of two to sixteen rows: 0.90 of the time in the geometric mean.
// n of whole groups of sixteen rows, k of whole super-blocks; the rest of the rule is measured, us before / here:
//   bf16 rows at 3, 5, 8: Q4_K 4096 x 2816 6.6 / 5.2, 9.7 / 5.7, 9.9 / 6.2, 17408 x 5120 20.9 / 16.4, 21.0 / 16.8, 20.9 / 17.8, 152064 x 5120 94 / 81, 96 / 85,
//   97 / 91; Q5_K 4096 x 4096 8.7 / 6.5, 8.8 / 7.0, 8.8 / 7.4; Q6_K at 5 4096 x 4096 12.0 / 7.1, 17408 x 5120 40 / 24, 152064 x 5120 164 / 133; Q8_0 at 5 4096 x 4096
//   12.3 / 6.7, 152064 x 5120 343 / 142; Q4_0 at 3, 5 4096 x 4096 8.4 / 5.7, 11.8 / 6.4.  Behind: two rows over K-quants (4096 x 12288 10 / 16), three over
//   Q6_K below 32768 rows (17408 x 5120 22.7 / 23.9), Q4_0 heads (151936 x 3584 68 / 88), Q8_0 and Q4_0 of 16384 x 4096 (16.7 / 17.5).
//   f32 rows at 4, 5: Q4_K 8192 x 2816 10.6 / 8.7, 11.9 / 9.3; Q6_K at 5 12288 x 4096 18.4 / 16.8, 17408 x 5120 33.8 / 25.6, 152064 x 5120 167 / 146, 5120 x 17408 55.6 /
//   45.6; Q8_0 at 5 4096 x 4096 12.2 / 8.4, 152064 x 5120 354 / 150; Q4_0 at 3, 5 4096 x 4096 8.8 / 7.6, 12.2 / 8.3.  Behind: fewer rows (an f32 row costs a cut
//   into parts ahead of the first product, 2 us in all), matrices below 4096 rows (2048 x 4096 Q6_K at five 7.7 / 8.9), groups that fill the CUs
//   badly (5120 x 6144 Q6_K, 1.25 rounds, 15.7 / 16.8).  Six to eight f32 rows take two operands: ahead over Q8_0 and Q4_0 (152064 x 5120 at eight
//   388 / 206, 8192 x 2816 21 / 14) and Q6_K of seven and eight rows (4096 x 4096 17.6 / 12.9), behind over Q4_K and Q5_K (12288 x 4096 16.2 / 18.0).
// Long k in slices (a launch each, about 4 us ahead of the first product): 4096 x 12288 at five rows f32 Q4_K 28.4 / 21.4, Q6_K 39.8 / 25.9, Q8_0 36 / 22, bf16 Q5_K
//   22.1 / 18.9; behind for fewer rows over K-quants (Q6_K bf16 at four 17.6 / 21.3) and at six to eight f32 rows (Q4_K 28.8 / 37.6).
// Rounds: one group of sixteen rows per CU.  K-quants under four f32 rows are ahead in a round that is whole or nearly so and from one and a half rounds
// on, not with a few more groups than CUs, which take a second round for themselves: four f32 rows, 3840 and 4080 x 5120 Q4_K 10.9 / 9.1, 11.0 / 9.2, x 2816 Q6_K
// 9.5 / 7.9 (x 1024 6.0 / 6.2).
bool gemv_krows_takes(hq_ggml_type t, hq_act_dtype xdt, uint32_t m, uint32_t n, uint32_t k, const void* w) {
    uint32_t cus = 0;
    if (m < 2 || m > 8 || n % 16u || k % 256u || k < 1024 || !is_aligned(w, 16) || cu_count(&cus)) return false;
    const bool f32 = xdt != HQ_BF16, head = n >= 32768, sliced = krows_slices(k / 256u, f32, m) > 1u;
    const bool b32 = t == HQ_Q8_0 || t == HQ_Q4_0;
    if (!b32 && t != HQ_Q4_K && t != HQ_Q5_K && t != HQ_Q6_K) return false;
    const bool odd_k = k % 1024u != 0;  // k for which the K-quants have no chunked small-batch kernel
    if (t == HQ_Q8_0 && (uint64_t)n * k < 10u << 20) return false;  // (small ones: gemv_q80_rows_walked, gemvr32.hip)
    const uint32_t units = n / 16u;
    const bool whole_round = units <= cus && units * 16u >= (t == HQ_Q6_K && k < 2048 ? 16u : 15u) * cus, overhang = units > cus && 2u * units < 3u * cus;
    if (!f32) {
        if (t == HQ_Q4_0) return !head && (n < 16384 || k > 4096) && (m >= 3 || (uint64_t)n * k >= 6u << 20);
        if (t == HQ_Q8_0) return head ? true : sliced ? m >= 4 || (m == 3 && !odd_k) : n >= 16384 && k <= 4096 ? false : m >= 4 || (n >= 8192 && n >= k);
        if (sliced) return (m >= 6 || (m == 5 && !odd_k)) && (t != HQ_Q4_K || odd_k || k <= 12288);
        if (head) return m >= 3 && (t != HQ_Q6_K || k >= 4096);
        if (odd_k && n >= 8192 && n <= 16384 && k <= 4096) return true;
        return m >= (t == HQ_Q6_K || (t == HQ_Q5_K && n >= 12288 && k <= 4096) || (t == HQ_Q4_K && n >= 12288 && k <= 4096) ? 4u : 3u);
    }
    if (m >= 6) {  // two operands
        if (sliced && !(head && t == HQ_Q8_0)) return false;
        if (b32) return head || n >= 4096 || (t == HQ_Q4_0 && (uint64_t)n * k >= 6u << 20);
        return t == HQ_Q6_K && m >= 7 && !head;
    }
    if (t == HQ_Q4_0) return head ? m == 5 : m == 5 || (m >= 3 && (uint64_t)n * k >= 6u << 20);
    if (t == HQ_Q8_0) return head || (sliced ? m >= 4 || (m == 3 && !odd_k) : n >= 16384 && k <= 4096 ? m >= 5 : m == 5 || (m == 4 && n >= 4096) || (n >= 8192 && n >= k));
    if (head) return k >= (t == HQ_Q5_K ? 5120u : 4096u);
    if (n >= 16384 && k <= 4096) return t == HQ_Q6_K && m >= 4;
    if (units <= cus && !whole_round) return sliced ? m >= 4 : m == 5 && k > 4096;
    if (odd_k && n >= 8192 && k <= 4096) return m >= 3;
    if (t == HQ_Q6_K && !sliced && overhang) return false;
    return m >= (n >= 16384 && t == HQ_Q4_K ? 3u : t == HQ_Q5_K && sliced && !whole_round ? 5u : 4u) && (m == 5 || !overhang || sliced);
}

// Gate + up + SwiGLU of a few rows (n rows a matrix, one slice of k): both matrices' groups by the same workgroup, gate then up.  us, the walk of
// both matrices (launch_gemv_swiglu) / here: f32 rows at 4, 5, 8 17408 x 5120 Q5_K 43.9 / 35.0, 51.4 / 37.1, 12288 x 4096 Q4_K 24.1 / 21.0, 27.2 / 21.8, 47 / 26, Q8_0 30.2 / 24.9,
// 35.8 / 25.4, 48 / 28; bf16 rows at 4, 8 12288 x 4096 Q4_K 22.0 / 18.5, 34.6 / 17.2, Q6_K 25.7 / 22.9, 41.6 / 23.4, 2304 x 2816 Q5_K 9.2 / 7.8, 13.9 / 8.1.  Behind: two and three rows
// (12288 x 4096 Q4_K f32 17.5 / 20.2, 20.2 / 20.6), six f32 rows over Q5_K and Q6_K (14336 x 4096 37.9 / 39.5), four over small ones (8192 x 2048 Q6_K 13.5 / 14.3).
bool gemv_krows_swiglu_takes(hq_ggml_type t, hq_act_dtype xdt, uint32_t m, uint32_t n, uint32_t k, const void* wg, const void* wu) {
    if (m < 3 || m > 8 || n % 16u || k % 256u || k < 1024 || !is_aligned(wg, 16) || !is_aligned(wu, 16) || (uint64_t)n * k < 6u << 20) return false;
    if (t != HQ_Q8_0 && t != HQ_Q4_0 && t != HQ_Q4_K && t != HQ_Q5_K && t != HQ_Q6_K) return false;
    const bool f32 = xdt != HQ_BF16, b32 = t == HQ_Q8_0 || t == HQ_Q4_0;
    if (krows_slices(k / 256u, f32, m) > 1u) return false;
    if (!f32) return m >= 4;
    if (m >= 6) return m >= 7 || b32 || (t == HQ_Q4_K && n >= 8192 && k > 2048);
    if (t == HQ_Q4_0 && n >= 4096) return true;
    return m == 5 || (m == 4 && (b32 || t == HQ_Q4_K || (n >= 8192 && k > 2048)));
}

// A batch of products of the same rows (q, k, v), N weight rows in all.  us, the launches of launch_gemv_jobs / here: 4096 + 1024 + 1024 x 2816 at 3, 5, 8 rows bf16 Q4_K 8.0 / 7.1,
// 10.2 / 7.5, 13.7 / 7.7, Q5_K 8.6 / 7.9, 10.7 / 8.4, 14.3 / 8.6, Q4_0 13.7 / 7.4, 14.2 / 7.8, 18.1 / 7.9; f32 at 4, 5, 8 Q5_K 10.6 / 9.8, 12.1 / 10.4, 16.0 / 14.1, Q8_0 11.2 / 9.8, 12.4 / 10.4, 16.8 / 12.7;
// 6144 + 1024 + 1024 x 5120 at five f32 rows Q6_K 22.0 / 15.8, Q4_K 18.3 / 13.1.  Behind: fewer rows (f32 Q4_K at three 8.5 / 8.4, Q6_K at two 8.4 / 10.0), small batches under f32 rows
// (4096 + 512 + 512 x 2048 Q8_0 at five 8.1 / 9.0), six to eight f32 rows over K-quants of k = 4096 (Q5_K at six 14.7 / 16.5).
bool gemv_krows_batch_takes(hq_ggml_type t, hq_act_dtype xdt, uint32_t m, uint32_t N, uint32_t k) {
    const bool f32 = xdt != HQ_BF16, b32 = t == HQ_Q8_0 || t == HQ_Q4_0;
    if (m < 2 || m > 8 || k % 256u || k < 1024 || (uint64_t)N * k < (f32 ? 12u << 20 : 8u << 20)) return false;
    if (t != HQ_Q8_0 && t != HQ_Q4_0 && t != HQ_Q4_K && t != HQ_Q5_K && t != HQ_Q6_K) return false;
    if (krows_slices(k / 256u, f32, m) > 1u) return false;
    if (!f32) return m >= (t == HQ_Q4_K ? 2u : t == HQ_Q8_0 && k <= 2048 ? 4u : 3u);
    if (m >= 6) return b32 || (k % 1024u != 0 && (m >= 7 || t != HQ_Q5_K)) || (m >= 7 && t == HQ_Q4_K);
    return m == 5 || (m == 4 && (b32 || t == HQ_Q4_K || k % 1024u != 0 || N >= 8192));
}

int launch_gemv_krows(hipStream_t s, const void* x, hq_act_dtype xdt, uint32_t m, uint32_t k, hq_ggml_type t, const KRowsSeg* seg, uint32_t nseg,
                      bool swiglu, const float* gate, uint32_t perm_hd, uint32_t perm_rows, bool whole) {
    uint32_t cus = 0;
    if (int rc = cu_count(&cus)) return rc;
    if (nseg == 0 || nseg > kKMaxSegs || (swiglu && nseg != 2)) return fail(HQ_ERR_INVALID_ARGUMENT, "k rows: %u matrices", nseg);
    KRowsArgs a{};
    a.x = x;
    a.xstride = perm_hd ? perm_hd : k;
    a.hd = perm_hd;
    a.xplane = perm_rows * perm_hd;
    a.m = m;
    a.k = k;
    const uint32_t nsb = k / 256u;
    a.rowb = k / hq_block_elems(t) * hq_block_bytes(t);
    a.nseg = nseg;
    a.swiglu = swiglu;
    a.gate = gate;
    a.whole = whole;
    for (uint32_t i = 0; i < nseg; ++i) {
        a.w[i] = static_cast<const uint8_t*>(seg[i].w);
        a.y[i] = seg[i].y;
        a.n[i] = seg[i].n;
        a.units = a.end[i] = (i && !swiglu ? a.end[i - 1] : 0u) + seg[i].n / 16u;
    }
    const bool f32 = xdt != HQ_BF16;
    const uint32_t slices = krows_slices(nsb, f32, m);
    if ((swiglu || gate) && slices > 1u) return fail(HQ_ERR_INVALID_ARGUMENT, "k rows: gating in slices of k");
    a.nsb = 0;
    for (uint32_t i = 0; i < slices; ++i) {
        a.sb0 += a.nsb;
        a.nsb = krows_slice_blocks(nsb, slices, i);
        a.add = i != 0;
        int rc = HQ_ERR_UNSUPPORTED;
        switch (t) {
            case HQ_Q4_K: rc = launch_krows_q4k(s, a, f32, cus); break;
            case HQ_Q5_K: rc = launch_krows_q5k(s, a, f32, cus); break;
            case HQ_Q6_K: rc = launch_krows_q6k(s, a, f32, cus); break;
            case HQ_Q8_0: rc = launch_krows_q80(s, a, f32, cus); break;
            case HQ_Q4_0: rc = launch_krows_q40(s, a, f32, cus); break;
        }
        if (rc) return rc;
    }
    return HQ_OK;
}

// Nine to sixteen rows of Q8_0 / Q4_0 / Q6_K (Q4_K and Q5_K take passes of eight anyway) as two passes of half of them: no tile of 64 rows is
// filled with 16, and where the matrix fits them the second pass finds the weights in the device's caches (up to 256 MB; a head is read twice).  us, a tile / two passes, as the calls follow each other (about 24 us is what the
// host takes for a call): bf16 Q8_0 at 12 rows 4096 x 4096 27.3 / 23.9, 17408 x 5120 60.6 / 45.2, 151936 x 4096 325 / 234, Q4_0 5120 x 5120 30.3 / 24.0, 17408 x 5120 47.6 /
// 42.3 (14336 x 5120 36.4 / 39.5), Q6_K 4096 x 4096 30.0 / 24.9 (14336 x 5120 37.8 / 45.4, 18944 x 3584 37.3 / 43.8); f32 at 9 / 16 Q8_0 4096 x 4096 27.9 / 25.5, 29.3 / 25.4,
// 151936 x 4096 327 / 235, 327 / 257 (12288 x 4096 38.4 / 42.3), Q4_0 4096 x 4096 29.7 / 22.5, 29.5 / 26.3 (12288 x 4096 32 / 40), Q6_K 4096 x 4096 29.8 / 24.2, 27.8 / 29.7.
// No less exact: these kernels' error is 2e-7 of the result at most, a tile rounds its weights to f16.
bool gemv_krows_passes(hq_ggml_type t, hq_act_dtype xdt, uint32_t m, uint32_t n, uint32_t k, const void* w) {
    if (m <= 8 || m > 16 || (t != HQ_Q8_0 && t != HQ_Q4_0 && t != HQ_Q6_K)) return false;
    const uint32_t half = (m + 1u) / 2u;
    if (!gemv_krows_takes(t, xdt, half, n, k, w) || !gemv_krows_takes(t, xdt, m - half, n, k, w)) return false;
    if (krows_slices(k / 256u, xdt != HQ_BF16, half) > 1u) return false;
    const uint64_t weights = (uint64_t)n * k, M = 1u << 20;
    if (xdt == HQ_BF16) return t == HQ_Q8_0 || (t == HQ_Q4_0 ? n <= 12288 || n > 16384 : weights <= 25 * M);
    if (t == HQ_Q8_0) return n >= 32768 || (n >= 4096 && weights <= 16 * M);
    return weights <= (t == HQ_Q4_0 && m <= 10 ? 25 : 16) * M && (t == HQ_Q4_0 || m <= 12);
}

int launch_gemv_krows_passes(hipStream_t s, const void* x, hq_act_dtype xdt, const void* w, float* y, uint32_t m, uint32_t n, uint32_t k, hq_ggml_type t,
                             const float* gate, uint32_t perm_hd) {
    const uint32_t half = (m + 1u) / 2u;
    for (uint32_t r0 = 0; r0 < m; r0 += half) {
        const KRowsSeg seg{w, y + (size_t)r0 * n, n};
        const uint8_t* xr = static_cast<const uint8_t*>(x) + (size_t)r0 * (perm_hd ? perm_hd : k) * (xdt == HQ_BF16 ? 2 : 4);
        if (int rc = launch_gemv_krows(s, xr, xdt, m - r0 < half ? m - r0 : half, k, t, &seg, 1, false, gate ? gate + (size_t)r0 * n : nullptr, perm_hd, m, true)) return rc;
    }
    return HQ_OK;
}

}  // namespace hq
