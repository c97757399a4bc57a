// The MoE FFN block of a decode step (1..8 tokens) as ONE launch: router and shared-gate logits, softmax / top-k,
// gate and up projections of the routed and the shared expert with their SwiGLU, the down projections, and the
// weighted reduction (+ sigmoid-gated shared expert, + residual).  build_moe_ffn_layer_gpu_q_into
// (src/inference/models/qwen35/gpu_ffn.rs:2313-2802) encodes these as phases A-F of one command buffer;
// moe_ffn_cpu_ref (src/inference/models/qwen35/ffn.rs:179-336) is the specification.
//
// As separate launches the block costs four to five launch latencies in series (each small kernel spends 3-4 us
// before its first result whatever it computes).  Here one workgroup per CU walks the phases and hands results
// to the other workgroups through memory:
//   * every hand-over is a relaxed device-scope atomic store / load (write-through, cache-bypassing accesses) and no
//     fence is ever executed: a device-scope release fence writes a whole L2 back on this multi-XCD part;
//   * a consumer recognises fresh data by a TAG = (calls so far on this scratch) + 1: router logits and SwiGLU
//     activations travel as 64-bit (tag, value) words, so a value and its freshness arrive in one store, no store has
//     to be ordered behind another, and nothing has to be cleared between calls; workgroup 0 stores the new call count
//     when it leaves, and not before every workgroup has read the old one;
//   * after the logits a workgroup works for one token (token b % T): it polls that token's logits only, routes it,
//     takes gate / up rows and down columns of that token;
//   * the down projections are cut by output columns, not by expert: a workgroup computes its 8 .. 64 columns for every
//     slot of a token and sums them itself, so the outputs never cross workgroups.
// A workgroup fills its CU, so the workgroups of a launch are not always resident together: another launch (a second such
// block on another stream, a second process) may hold some of the CUs until its own are through.  So a workgroup that has
// polled `patience` times without success stops waiting for the others and works out what it misses by itself -- the
// logits for its own use, the activations of its token for everybody -- with the same arithmetic: duplicates have the same
// bits.  Started workgroups therefore always finish, whatever else is resident; only workgroup 0 then stays until all have
// started, which takes one CU from the others.  (What that costs where nobody runs out of patience cannot be told
// from the runs' spread: one token of Q5_K + Q6_K, f32, 17.0 us without and with it, eight of Q4_K, bf16, 32.2.)
//
// Row arithmetic is that of the separate dispatches — the same piece dot products, the same reduction order, the
// same SwiGLU rounding, the same order of the weighted sum — so the block's output has the bits of
// hq_dense_gemv_bf16_pair + hq_qmatmul_batch_ggml x 2 + hq_moe_weighted_reduce.
//
// Shapes: K-quant experts (Q4_K, Q5_K or Q6_K; gate / up of one type, down of the same or -- the mix GGUF files of the
// reference's model hold, docs/ADR-028...:4942-4946 -- Q4_K / Q5_K gate / up with a Q6_K down), hidden = 2048 (32 lanes
// per gate / up row: a wave step is one gate row and the up row of the same index), expert FFN = shared FFN = 512 (8
// lanes per down row), <= 256 experts, bf16 or f32 activations (f32: the dot products of the separate dispatches over f32
// activations, a lane's 64 of them in registers; one token of the Q5_K + Q6_K block 28 us as four launches, 16 as one; eight: 67 and 44).
#include <math.h>

#include "hq_internal.h"
#include "moe_topk.h"

#include "gemv_pieces.h"

namespace hq {
namespace {

constexpr uint32_t FH = 2048, FI = 512;               // hidden, expert FFN width
template <int TYPE>
constexpr uint32_t kRowBytesH = FH / 256 * kBlockBytes<TYPE>;  // bytes of a gate / up row
template <int TYPE>
constexpr uint32_t kRowBytesI = FI / 256 * kBlockBytes<TYPE>;  // bytes of a down row
constexpr uint32_t MAX_T = 8;                         // tokens per call
// Two shapes of workgroup (template arguments WAVES_, RING_ of the kernel): 8 waves with four weight fetches in flight
// each -- one token: the phases are round trips, few rows per wave -- and 12 waves with two -- several tokens: the
// phases are bound by VALU issue, and three waves per SIMD keep it a little busier than two (16 waves leave 128
// registers per lane and spill 60 .. 200 of them).
// A logit is stored LG_COPIES times and a workgroup polls copy (its index among its token's workgroups) % LG_COPIES: at
// one token 256 workgroups would otherwise poll the same 2 KB (sixteen cache lines, a few memory channels).
constexpr uint32_t LG_COPIES = 8;
constexpr uint32_t PATIENCE = 256;       // polls (about 1 us each) before a workgroup helps itself: waits end after a few by themselves
constexpr uint32_t START_POLLS = 1u << 20;  // polls of workgroup 0 for the last workgroup to start

struct FusedArgs {
    const void* x;           // [T][H] bf16 or f32
    const uint16_t* router;  // [E][H] bf16
    const uint16_t* sh_lw;   // [H] bf16 or null: shared-expert gate logit
    const uint8_t *eg, *eu, *ed, *sg, *su, *sd;
    const float* residual;
    float* out;
    uint32_t* route_ids;
    float* route_w;
    uint8_t* scratch;
    uint32_t T, E, K;
    uint64_t stride_gu, stride_d;
    uint32_t m4, m2, magic, patience;
};

// Scratch layout (byte offsets), the same on host and device: call counter and error word, then the two hand-over
// areas, both of (tag << 32 | value bits) words.
struct Layout {
    uint32_t T, E, K;
    __host__ __device__ uint32_t slots() const { return K + 1; }  // routed slots + the shared expert
    __host__ __device__ size_t logits() const { return 64; }  // u64 [LG_COPIES][T][E + 1]
    __host__ __device__ size_t act() const { return logits() + (size_t)LG_COPIES * T * (E + 1) * 8; }  // u64 [T][K + 1][I]
    __host__ __device__ size_t total() const { return act() + (size_t)T * slots() * FI * 8; }
};

template <typename V>
__device__ __forceinline__ void st_dev(V* p, V v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ V ld_dev(const V* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether the tag of a (tag, value) word is `tag` within `polls` polls; its value.
__device__ __forceinline__ bool wait_tagged(const uint64_t* p, uint32_t tag, uint32_t polls, uint32_t* value) {
    uint64_t got = ld_dev(p);
    for (uint32_t n = 0; (uint32_t)(got >> 32) != tag && n < polls; ++n) {
        __builtin_amdgcn_s_sleep(1);
        got = ld_dev(p);
    }
    *value = (uint32_t)got;
    return (uint32_t)(got >> 32) == tag;
}

// LDS bytes of a token's staged activations and their per-16 sums.
__host__ __device__ constexpr uint32_t staged_x_bytes(bool x_bf16) { return FH * (x_bf16 ? 2 : 4) + FH / 16 * 4; }

// LDS slot of 16-byte chunk ch of the staged activations.  Lanes that read together differ in the piece index (ch / 8)
// or, Q6_K, whose lane reads four runs of sixteen at a stride of 32 inside one half of a super-block, in bits 1, 4, 5, 6.
template <int TYPE>
__device__ __forceinline__ uint32_t swz8(uint32_t ch) {
    if constexpr (TYPE == HQ_Q6_K) return ch ^ (((ch >> 4) & 1u) | (((ch >> 5) & 3u) << 2));
    return ch ^ ((ch >> 4) & 7u);
}
// First float4 of run r (sixteen activations) of a lane's 64 activations of a row of FI: lane li = (super-block, quarter).
template <int TYPE>
__device__ __forceinline__ uint32_t act_run(uint32_t li, uint32_t r) {
    if constexpr (TYPE == HQ_Q6_K) return (li >> 2) * 64u + ((li >> 1) & 1u) * 32u + (li & 1u) * 4u + 8u * r;
    return li * 16u + 4u * r;
}

// What a workgroup knows and where it finds things, from the arguments and its place in the launch.
// TG, TD: types of gate / up and of down; WAVES per workgroup; activation type.
template <int TG, int TD, int WAVES_, bool X_BF16>
struct FusedBlock {
    static constexpr uint32_t WAVES = WAVES_, THREADS = 64 * WAVES, ROWB_H = kRowBytesH<TG>, ROWB_I = kRowBytesI<TD>;
    static constexpr uint32_t XQ = X_BF16 ? 1 : 2;  // 16-byte pieces of eight activations
    FusedArgs a;
    uint32_t T, E, K, S, P, n_rows;
    uint32_t tid, lane, b, G, wv;
    // After phase 1 a workgroup works for ONE token, token b % T: it needs that token's logits, activations and routing
    // only (eight tokens: an eighth of the words to poll for).
    uint32_t tok, jb, nb;        // the token, this workgroup among its nb workgroups
    uint32_t tw, NTW;            // this wave among the token's waves
    uint32_t groups, cols;       // output columns of a unit, in groups of eight: about one unit per workgroup
    // LDS: [the token's staged activations | later: its SwiGLU activations of all slots] | logits | ids | weights | partials
    uint4* lds_x;        // H/8 chunks (paired bf16 words) or H/4 (f32)
    float* lds_sx;       // H/16 per-16 sums
    float4* lds_act;     // S * I floats (over the activations, after phase 2)
    float* lds_as;       // S * I/16 sums
    float* lds_lg;       // E + 1
    uint32_t* lds_id;    // K
    float* lds_w;        // K + 1: slot K = shared gate
    float* lds_part;     // S * 64 down partials of one unit
    uint32_t* lds_gath;  // 64 * WAVES: the workgroup's SwiGLU activations
    uint32_t* lds_late;  // whether a thread ran out of patience; the call's tag
    uint32_t *s_epoch, *s_err;
    uint64_t *s_lg, *s_act;

    __device__ __forceinline__ FusedBlock(const FusedArgs& args, uint4* smem, uint32_t tid_, uint32_t b_, uint32_t G_) : a(args), tid(tid_), b(b_), G(G_) {
        const Layout L{a.T, a.E, a.K};
        T = a.T, E = a.E, K = a.K, S = K + 1, P = S * FI, n_rows = E + (a.sh_lw ? 1u : 0u);
        lane = tid & 63u;
        wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));  // known to be the same in a wave: scalar branches
        tok = b % T, jb = b / T, nb = (G - tok + T - 1u) / T;
        tw = jb * WAVES + wv, NTW = nb * WAVES;
        groups = T <= 1 ? 1u : T <= 2 ? 2u : T <= 4 ? 4u : 8u, cols = 8u * groups;
        lds_x = smem;
        lds_sx = reinterpret_cast<float*>(lds_x + (X_BF16 ? FH / 8 : FH / 4));
        const uint32_t area = staged_x_bytes(X_BF16), act_bytes = S * (FI * 4 + FI / 16 * 4);
        lds_act = reinterpret_cast<float4*>(smem);
        lds_as = reinterpret_cast<float*>(lds_act + (size_t)S * (FI / 4));
        lds_lg = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(smem) + (area > act_bytes ? area : act_bytes));
        lds_id = reinterpret_cast<uint32_t*>(lds_lg + (E + 1));
        lds_w = reinterpret_cast<float*>(lds_id + K);
        lds_part = lds_w + S;
        lds_gath = reinterpret_cast<uint32_t*>(lds_part + S * 64);
        lds_late = lds_gath + 64 * WAVES;
        s_epoch = reinterpret_cast<uint32_t*>(a.scratch);
        s_err = s_epoch + 1;
        s_lg = reinterpret_cast<uint64_t*>(a.scratch + L.logits());
        s_act = reinterpret_cast<uint64_t*>(a.scratch + L.act());
    }

    // A router row and a token's activations, 32 elements per lane, and their product with the arithmetic of dense_gemv_bf16_kernel.
    struct LogitIn {
        uint4 w[FH / 8 / 64], x[FH / 8 / 64 * XQ];
    };
    __device__ __forceinline__ void fetch_logit(LogitIn& in, uint32_t r, uint32_t t) const {
        const uint4* wr = reinterpret_cast<const uint4*>(r < E ? a.router + (size_t)r * FH : a.sh_lw);
        const uint4* xr = reinterpret_cast<const uint4*>(static_cast<const uint8_t*>(a.x) + (size_t)t * FH * (X_BF16 ? 2 : 4));
#pragma unroll
        for (uint32_t c = 0; c < FH / 8 / 64; ++c) {
            in.w[c] = wr[lane + 64 * c];
#pragma unroll
            for (uint32_t i = 0; i < XQ; ++i) in.x[XQ * c + i] = xr[XQ * (lane + 64 * c) + i];
        }
    }
    static __device__ __forceinline__ float dot_logit(const LogitIn& in) {
        float acc = 0.f;
#pragma unroll
        for (uint32_t c = 0; c < FH / 8 / 64; ++c) {
            const uint32_t ww[4] = {in.w[c].x, in.w[c].y, in.w[c].z, in.w[c].w};
            float xv[8];
            if constexpr (X_BF16) {
                const uint32_t tw[4] = {in.x[c].x, in.x[c].y, in.x[c].z, in.x[c].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) xv[2 * i] = bf16_bits_to_f32(tw[i] & 0xffffu), xv[2 * i + 1] = bf16_bits_to_f32(tw[i] >> 16);
            } else {
                const uint32_t tw[8] = {in.x[2 * c].x, in.x[2 * c].y, in.x[2 * c].z, in.x[2 * c].w, in.x[2 * c + 1].x, in.x[2 * c + 1].y, in.x[2 * c + 1].z, in.x[2 * c + 1].w};
#pragma unroll
                for (int i = 0; i < 8; ++i) xv[i] = __uint_as_float(tw[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc = fmaf(bf16_bits_to_f32(ww[i] & 0xffffu), xv[2 * i], acc);
                acc = fmaf(bf16_bits_to_f32(ww[i] >> 16), xv[2 * i + 1], acc);
            }
        }
        return wave_sum(acc);
    }

    __device__ __forceinline__ void fetch_x(XRaw<X_BF16>& raw) const {  // sixteen activations per thread, one pass
        static_assert(FH / 16 <= THREADS, "one pass stages a token");
        raw.fetch(static_cast<const uint8_t*>(a.x) + (size_t)tok * FH * (X_BF16 ? 2 : 4), tid < FH / 16 ? tid : 0u);  // (no branch around the load)
    }
    // The layout and sums of stage_store.
    __device__ __forceinline__ void stage_x(const XRaw<X_BF16>& raw) const {
        const uint32_t j = tid;
        if (j >= FH / 16) return;
        if constexpr (!X_BF16) {
            float sum = 0.f;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t f = 4 * j + i;
                lds_x[f ^ (f >> 4)] = raw.r[i];  // (the layout of the SwiGLU activations below, FH / 4 slots)
                sum += __uint_as_float(raw.r[i].x);
                sum += __uint_as_float(raw.r[i].y);
                sum += __uint_as_float(raw.r[i].z);
                sum += __uint_as_float(raw.r[i].w);
            }
            lds_sx[j] = sum;
        } else {
            const uint4 p = raw.r[0], q = raw.r[1];
            const uint32_t w[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
            uint4 o0, o1;
            o0.x = (w[0] & 0xffffu) | (w[1] << 16);
            o0.y = (w[0] >> 16) | (w[1] & 0xffff0000u);
            o0.z = (w[2] & 0xffffu) | (w[3] << 16);
            o0.w = (w[2] >> 16) | (w[3] & 0xffff0000u);
            o1.x = (w[4] & 0xffffu) | (w[5] << 16);
            o1.y = (w[4] >> 16) | (w[5] & 0xffff0000u);
            o1.z = (w[6] & 0xffffu) | (w[7] << 16);
            o1.w = (w[6] >> 16) | (w[7] & 0xffff0000u);
            lds_x[swz8<TG>(2 * j)] = o0;
            lds_x[swz8<TG>(2 * j + 1)] = o1;
            float sum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sum += bf16_bits_to_f32(w[e] & 0xffffu);
                sum += bf16_bits_to_f32(w[e] >> 16);
            }
            lds_sx[j] = sum;
        }
    }

    // The token's routing from its logits (every workgroup of the token for itself, one wave), and a barrier.
    __device__ __forceinline__ void route() const {
        if (wv == 0) {
            uint32_t id;
            float wt;
            softmax_topk_lane<4>(lds_lg, E, K, lane, id, wt);
            if (lane < K) {
                id = id < E ? id : E - 1u;  // (the selection only yields indices below E; a bound the fetch addresses can rely on)
                lds_id[lane] = id;
                lds_w[lane] = wt;
                if (jb == 0 && a.route_ids) {
                    a.route_ids[tok * K + lane] = id;
                    a.route_w[tok * K + lane] = wt;
                }
            }
            if (lane == 0) lds_w[K] = a.sh_lw ? 1.f / (1.f + expf(-lds_lg[E])) : 1.f;  // ffn.rs:28-30
        }
        __syncthreads();
    }

    // a lane's 64 staged activations and their sums
    __device__ __forceinline__ void load_x(uint32_t (&xp)[X_BF16 ? 32 : 64], float (&sx)[4]) const {
        const uint32_t li = lane & 31u;
        if constexpr (!X_BF16) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t f0 = act_run<TG>(li, (uint32_t)r);
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const uint4 v = lds_x[(f0 + j) ^ ((f0 + j) >> 4)];
                    xp[16 * r + 4 * j] = v.x;
                    xp[16 * r + 4 * j + 1] = v.y;
                    xp[16 * r + 4 * j + 2] = v.z;
                    xp[16 * r + 4 * j + 3] = v.w;
                }
                sx[r] = lds_sx[f0 / 4];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t ch = act_run<TG>(li, (uint32_t)r) / 2u;  // two chunks of eight per run
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint4 v = lds_x[swz8<TG>(ch + u)];
                    xp[8 * r + 4 * u] = v.x;
                    xp[8 * r + 4 * u + 1] = v.y;
                    xp[8 * r + 4 * u + 2] = v.z;
                    xp[8 * r + 4 * u + 3] = v.w;
                }
                sx[r] = lds_sx[ch / 2];
            }
        }
    }
    // Gate and up row p % I of slot p / I of the token: lanes 0-31 the gate row, 32-63 the up row.
    __device__ __forceinline__ void fetch_gu(Piece<TG>& pc, uint32_t p) const {
        const uint32_t li = lane & 31u, hf = lane >> 5, r = p % FI, s = p / FI;
        const uint8_t* base = s < K ? (hf ? a.eu : a.eg) + (size_t)lds_id[s] * a.stride_gu : (hf ? a.su : a.sg);
        pc.load(base + (size_t)r * ROWB_H + (li >> 2) * kBlockBytes<TG>, (int)(li & 3u));
    }

    // a lane's 64 SwiGLU activations of slot s and their sums
    __device__ __forceinline__ void load_act(float (&xf)[64], float (&sx)[4], uint32_t s) const {
        const uint32_t li = lane & 7u;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t f0 = act_run<TD>(li, (uint32_t)r);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t f = f0 + (uint32_t)j;
                const float4 v = lds_act[s * (FI / 4) + (f ^ (f >> 4))];
                xf[16 * r + 4 * j] = v.x;
                xf[16 * r + 4 * j + 1] = v.y;
                xf[16 * r + 4 * j + 2] = v.z;
                xf[16 * r + 4 * j + 3] = v.w;
            }
            sx[r] = lds_as[s * (FI / 16) + f0 / 4];
        }
    }
    // The down rows of column group g of unit c in slot s, eight lanes per row.
    __device__ __forceinline__ void fetch_d(Piece<TD>& pc, uint32_t c, uint32_t s, uint32_t g) const {
        const uint32_t li = lane & 7u, sub = lane >> 3;
        const uint8_t* base = s < K ? a.ed + (size_t)lds_id[s] * a.stride_d : a.sd;
        pc.load(base + (size_t)(cols * c + 8 * g + sub) * ROWB_I + (li >> 2) * kBlockBytes<TD>, (int)(li & 3u));
    }
    __device__ __forceinline__ void sum_acts() const {
        for (uint32_t e = tid; e < S * (FI / 16); e += THREADS) {  // per-16 sums in the order one thread adds them (stage_swiglu)
            const uint32_t s = e / (FI / 16), j = e % (FI / 16);
            float sum = 0.f;
#pragma unroll
            for (uint32_t k = 0; k < 16; ++k) {
                const uint32_t q = (j * 16 + k) >> 2;
                sum += reinterpret_cast<float*>(lds_act)[s * FI + (((q ^ (q >> 4)) << 2) | (k & 3u))];
            }
            lds_as[e] = sum;
        }
    }
    // The weighted sum over the slots of a unit's columns in slot order, the shared expert last (the order of moe_weighted_reduce_kernel).
    __device__ __forceinline__ void store_unit(uint32_t c) const {
        if (tid < cols) {
            const uint32_t col = cols * c + tid;
            float acc = 0.f;
            for (uint32_t s = 0; s < S; ++s) acc = fmaf(lds_w[s], lds_part[s * cols + tid], acc);
            if (a.residual) acc += a.residual[(size_t)tok * FH + col];
            a.out[(size_t)tok * FH + col] = acc;
        }
    }
};
template <int TG, bool X_BF16>
__device__ __forceinline__ float dot_gu(Piece<TG>& pc, uint32_t lane, uint32_t (&xp)[X_BF16 ? 32 : 64], float (&sx)[4], uint32_t m4, uint32_t m2, uint32_t magic) {
    float part;
    if constexpr (X_BF16)
        part = dot_pair(pc, (int)(lane & 3u), xp, sx, m4, m2, magic);
    else
        part = dot_f32(pc, (int)(lane & 3u), reinterpret_cast<const float*>(xp), sx);
    return group_sum(part, 5);
}

// A workgroup out of patience (see the header): everything that its outputs still need, by itself.  Nothing of the phases of
// the kernel is used but what lies in memory, and the arguments are read again, so that the kernel holds no register for this.
template <int TG, int TD, int WAVES, bool X_BF16>
__device__ __forceinline__ void finish_alone(uint4* smem, uint32_t tid, uint32_t b, uint32_t G, uint32_t tag) {
    union {
        FusedArgs args;
        uint32_t words[sizeof(FusedArgs) / 4];
    };
    auto ka = (const __attribute__((address_space(4))) uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka), "+v"(tid), "+s"(b), "+s"(G));
#pragma unroll
    for (uint32_t i = 0; i < sizeof(FusedArgs) / 4; ++i) words[i] = ka[i];
    const FusedBlock<TG, TD, WAVES, X_BF16> k(args, smem, tid, b, G);
    const uint32_t lane = k.lane, wv = k.wv;
    const uint64_t tag_hi = (uint64_t)tag << 32;
    __syncthreads();
    for (uint32_t r = wv; r < k.n_rows; r += WAVES) {
        typename FusedBlock<TG, TD, WAVES, X_BF16>::LogitIn in;
        k.fetch_logit(in, r, k.tok);
        const float v = k.dot_logit(in);
        if (lane == 0) k.lds_lg[r] = v;
    }
    XRaw<X_BF16> raw;
    k.fetch_x(raw);
    k.stage_x(raw);
    __syncthreads();
    k.route();
    {
        // gate / up rows whose activation has not arrived, from a place of the workgroup's own on: workgroups that do this at the
        // same time divide the rows
        const uint32_t count = (k.P - wv + WAVES - 1u) / WAVES, start = (uint32_t)((uint64_t)k.jb * count / k.nb);
        uint32_t xp[X_BF16 ? 32 : 64];
        float sx[4];
        k.load_x(xp, sx);
        for (uint32_t i = 0; i < count; ++i) {
            const uint32_t p = wv + (start + i < count ? start + i : start + i - count) * WAVES;
            uint64_t* word = k.s_act + (size_t)k.tok * k.P + p;
            if ((uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(ld_dev(word) >> 32)) == tag) continue;
            Piece<TG> pc;
            k.fetch_gu(pc, p);
            const float v = dot_gu<TG, X_BF16>(pc, lane, xp, sx, k.a.m4, k.a.m2, k.a.magic);
            const float gate = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
            const float up = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
            if (lane == 0) st_dev(word, tag_hi | __float_as_uint(silu_mul_f32(gate, up)));
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // every activation of the token is in place, seen or stored by this workgroup; the staged x is dead
    for (uint32_t i = k.tid; i < k.P; i += 64u * WAVES) {
        const uint32_t sl = i / FI, e = i % FI, q = e >> 2;
        reinterpret_cast<uint32_t*>(k.lds_act)[sl * FI + (((q ^ (q >> 4)) << 2) | (e & 3u))] = (uint32_t)ld_dev(k.s_act + (size_t)k.tok * k.P + i);
    }
    __syncthreads();
    k.sum_acts();
    __syncthreads();
    for (uint32_t c = k.jb; c < FH / k.cols; c += k.nb) {
        for (uint32_t st = wv; st < k.S * k.groups; st += WAVES) {
            const uint32_t s = st / k.groups, g = st % k.groups;
            Piece<TD> pc;
            k.fetch_d(pc, c, s, g);
            float xf[64], sx[4];
            k.load_act(xf, sx, s);
            const float v = group_sum(dot_f32(pc, (int)(lane & 3u), xf, sx), 3);
            if ((lane & 7u) == 0) k.lds_part[s * k.cols + 8 * g + (lane >> 3)] = v;
        }
        __syncthreads();
        k.store_unit(c);
        __syncthreads();
    }
    // Workgroup 0 leaves behind the start of all others: one that read the new call count would take it for its own.  Every
    // workgroup has stored its logits only when it had read the old one.
    if (b == 0 && tid < 64u)
        for (uint32_t r = lane; r < k.n_rows; r += 64u) {
            uint32_t v;
            if (!wait_tagged(&k.s_lg[r], tag, START_POLLS, &v)) st_dev(k.s_err, 1u);
        }
    __syncthreads();
}

// WAVES_ waves per workgroup, RING_ fetches in flight per wave.
template <int TG, int TD, int WAVES_, int RING_, bool X_BF16>
__global__ __launch_bounds__(64 * WAVES_) void moe_fused_kernel(FusedArgs a) {
    constexpr uint32_t WAVES = WAVES_, THREADS = 64 * WAVES;
    constexpr int RING = RING_;
    // activation loads of a thread per polling pass: (8 + 1) slots x 512 / 2 words = 4.5 per thread of 512, 2.25 of 1024
    constexpr int POLL = WAVES_ == 8 ? 5 : 3;
    extern __shared__ uint4 smem[];
    const FusedBlock<TG, TD, WAVES_, X_BF16> k(a, smem, threadIdx.x, blockIdx.x, gridDim.x);
    const uint32_t T = k.T, E = k.E, S = k.S, P = k.P, tid = k.tid, lane = k.lane, wv = k.wv, b = k.b, G = k.G;
    const uint32_t tok = k.tok, jb = k.jb, nb = k.nb, tw = k.tw, NTW = k.NTW;
    uint64_t *const s_lg = k.s_lg, *const s_act = k.s_act;
    float* const lds_lg = k.lds_lg;
    uint32_t* const lds_gath = k.lds_gath;

    // One wave reads the call count for the workgroup (2048 reads of that word instead of 256 take longer, and every wave would have
    // to have its own before the logits may leave).
    uint32_t tag0 = 0;
    if (wv == 0) tag0 = ld_dev(k.s_epoch) + 1u;

    // the token's activations, requested first and staged while the logits travel
    XRaw<X_BF16> xraw;
    k.fetch_x(xraw);

    // ---- phase 1: router logits and the shared-gate logit, one (row, token) per wave and turn ----
    // Workgroup b takes the rows b, b + G, ... for every token (G <= n_rows: it has at least one row), its waves the
    // (row, token) pairs in turn.  It delivers logits of EVERY token, and none before it has read the call count: once a
    // token's logits are complete, every workgroup has read it, and workgroup 0 may store the new one.
    const uint32_t pairs1 = (k.n_rows - b + G - 1u) / G * T;
    uint32_t tag;
    uint64_t tag_hi;
    auto logit = [&](uint32_t q) {
        typename FusedBlock<TG, TD, WAVES_, X_BF16>::LogitIn in;
        k.fetch_logit(in, b + G * (q / T), q % T);
        return k.dot_logit(in);
    };
    auto store_logit = [&](uint32_t q, float v) {
        if (lane < LG_COPIES) st_dev(&s_lg[((size_t)lane * T + q % T) * (E + 1) + b + G * (q / T)], tag_hi | __float_as_uint(v));
    };
    float first = 0.f;
    if (wv < pairs1) first = logit(wv);
    if (tid == 0) k.lds_late[0] = 0, k.lds_late[1] = tag0;
    __syncthreads();
    tag = (uint32_t)__builtin_amdgcn_readfirstlane((int)k.lds_late[1]);
    tag_hi = (uint64_t)tag << 32;
    if (wv < pairs1) store_logit(wv, first);
    for (uint32_t q = wv + WAVES; q < pairs1; q += WAVES) store_logit(q, logit(q));

    // ---- while the logits travel: the staged activations go to LDS ----
    k.stage_x(xraw);

    // ---- the token's logits ----
    for (uint32_t i = tid; i < E + 1; i += THREADS) {
        uint32_t v = 0;
        if (i < k.n_rows && !wait_tagged(&s_lg[((size_t)(jb % LG_COPIES) * T + tok) * (E + 1) + i], tag, a.patience, &v)) *k.lds_late = 1u;
        lds_lg[i] = __uint_as_float(v);
    }
    __syncthreads();
    // (lds_late is looked at where something is to leave the workgroup: until then the phases run on with what there is, whatever it
    // is.  It is read ahead of a barrier behind which it may be set again, so all waves read the same.)
    k.route();
    uint32_t m4, m2, magic;
    asm volatile("v_mov_b32 %0, %3\n\tv_mov_b32 %1, %4\n\tv_mov_b32 %2, %5"
                 : "=v"(m4), "=v"(m2), "=v"(magic)
                 : "s"(a.m4), "s"(a.m2), "s"(a.magic));

    // ---- phase 2: gate and up row p % I of slot p / I of the token, lanes 0-31 the gate row and 32-63 the up row, then
    // the SwiGLU; the waves of the token's workgroups take the rows in turn, RING fetches ahead ----
    // The activations are not stored where they arise.  Loads and stores are counted by one counter and return in order,
    // and a write-through store is acknowledged by memory a microsecond or more after its issue (several under load): a
    // store among the fetches holds back every fetch behind it.  Lane n keeps the activation of the wave's row n; after
    // the phase the waves put theirs together in LDS and ONE wave stores the workgroup's rows (eight consecutive words
    // per row index: 64-byte pieces instead of 8-byte ones), after the next phase's first weight fetches have been issued.
    // (A wave with more than 64 rows, which takes a small grid and many slots, stores for itself.)
    uint32_t keep = 0;
    const uint32_t rows2 = tw < P ? (P - tw + NTW - 1u) / NTW : 0u;
    const uint32_t rows2_wg = jb * WAVES < P ? (P - jb * WAVES + NTW - 1u) / NTW : 0u;  // of the workgroup's first wave: the most
    const bool gather = rows2_wg <= 64u;
    auto flush = [&](uint32_t first, uint32_t count) {
        if (lane < count && !*k.lds_late) st_dev(&s_act[(size_t)tok * P + tw + (first + lane) * NTW], tag_hi | keep);
    };
    {
        const uint32_t mine = rows2;
        constexpr int RG = !X_BF16 && TG == HQ_Q5_K && RING > 3 ? 3 : RING;  // (as for the down phase's ring)
        Piece<TG> ring[RG];
#pragma unroll
        for (int i = 0; i < RG; ++i)
            if ((uint32_t)i < mine) k.fetch_gu(ring[i], tw + (uint32_t)i * NTW);
        uint32_t xp[X_BF16 ? 32 : 64];
        float sx[4];
        k.load_x(xp, sx);
        float keep_g = 0.f, keep_u = 0.f;
        for (uint32_t i0 = 0; i0 < mine; i0 += RG) {
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const uint32_t n = i0 + (uint32_t)i;
                if (n < mine) {
                    const uint32_t p = tw + n * NTW;
                    const float v = dot_gu<TG, X_BF16>(ring[i], lane, xp, sx, m4, m2, magic);
                    const float gate = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
                    const float up = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
                    if (n + RG < mine) {
                        float tie = v;
                        asm volatile("" : "+v"(tie));
                        k.fetch_gu(ring[i], p + RG * NTW);
                    }
                    keep_g = lane == (n & 63u) ? gate : keep_g;  // the SwiGLU of up to 64 rows is one pass at the end
                    keep_u = lane == (n & 63u) ? up : keep_u;
                    if ((n & 63u) == 63u && n + 1u < mine) {
                        keep = __float_as_uint(silu_mul_f32(keep_g, keep_u));
                        flush(n - 63u, 64u);
                    }
                }
            }
        }
        keep = __float_as_uint(silu_mul_f32(keep_g, keep_u));
    }
    if (gather && lane < rows2) lds_gath[lane * WAVES + wv] = keep;
    // The workgroup's activations go out by its last wave (or by every wave for itself), which then waits for the stores'
    // acknowledgement while the other waves issue the next phase's first weight fetches; nobody polls before that: the
    // other workgroups' stores were issued at about the same time, so the first poll finds nearly everything, and polls
    // that start earlier only get in the way of the stores.
    const bool storing = !gather || wv == WAVES - 1u;
    auto store_acts = [&]() {
        if (gather) {
            if (storing)
                for (uint32_t idx = lane; idx < rows2_wg * WAVES; idx += 64u) {
                    const uint32_t p = jb * WAVES + idx % WAVES + idx / WAVES * NTW;
                    if (p < P) st_dev(&s_act[(size_t)tok * P + p], tag_hi | lds_gath[idx]);
                }
        } else if (rows2) {
            flush((rows2 - 1u) & ~63u, ((rows2 - 1u) & 63u) + 1u);
        }
    };
    auto await_acts_stored = [&]() {
        if (storing) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (gather) __syncthreads();
    };
    // Every fetch of the phase has been consumed: a wait that costs nothing and tells the compiler so (it cannot see it
    // from the loop's conditions), or it would make the next phase's fetches wait for each other for the sake of the
    // registers they share with these.
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    bool late = __builtin_amdgcn_readfirstlane((int)*k.lds_late) != 0;
    __syncthreads();  // the staged activations are dead from here on: their LDS holds the SwiGLU activations next

    // ---- phases 3 + 4: unit (column slice c of the token): the down rows of the slice for every slot of the token, then
    // the weighted sum over the slots in slot order, the shared expert last (the order of moe_weighted_reduce_kernel) ----
    if (!late) {
        constexpr int RD = TD == HQ_Q5_K && RING > 3 ? 3 : RING;  // (a ring of four Q5_K pieces beside the 64 activations spills)
        const uint32_t li = lane & 7u, sub = lane >> 3, groups = k.groups, cols = k.cols, units_per_t = FH / cols;
        store_acts();
        if (jb >= units_per_t) await_acts_stored();  // a workgroup without a unit
        for (uint32_t c = jb; c < units_per_t; c += nb) {
            // steps (slot s, row group g) = step index s * groups + g.  With several row groups a wave takes a run of
            // consecutive steps, so that it changes slot (and reloads the slot's activations from LDS) as seldom as
            // possible; with one row group (one token) every step is another slot and the waves take the steps in turn.
            const uint32_t n_steps = S * groups;
            const bool runs = groups > 1;
            const uint32_t st0 = runs ? wv * n_steps / WAVES : wv, stp = runs ? 1u : WAVES;
            const uint32_t mine = runs ? (wv + 1u) * n_steps / WAVES - st0 : wv < n_steps ? (n_steps - wv + WAVES - 1u) / WAVES : 0u;
            auto fetch = [&](Piece<TD>& pc, uint32_t n) {
                const uint32_t st = st0 + n * stp;
                k.fetch_d(pc, c, st / groups, st % groups);
            };
            Piece<TD> ring[RD];
            auto prefetch = [&]() {
#pragma unroll
                for (int i = 0; i < RD; ++i)
                    if ((uint32_t)i < mine) fetch(ring[i], (uint32_t)i);
            };
            if (c == jb && storing) {  // (a storing wave's fetches would stand in the queue in front of the acknowledgement's wait)
                await_acts_stored();
                prefetch();
            } else {
                prefetch();
                if (c == jb) await_acts_stored();
            }
            // the token's SwiGLU activations of every slot: (tag, value) words, two per 16-byte load, all of a thread's
            // loads of a pass in flight at once; a thread whose words are not all fresh asks for them again
            {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                const uint64_t* src = s_act + (size_t)tok * P;
                const uint32_t n2 = S * FI / 2;
                for (uint32_t base = 0; base < n2; base += POLL * THREADS) {
                    u32x4 got[POLL];
                    uint32_t off[POLL];
#pragma unroll
                    for (int i = 0; i < POLL; ++i) {
                        const uint32_t e2 = base + tid + (uint32_t)i * THREADS;
                        off[i] = 16u * (e2 < n2 ? e2 : n2 - 1u);  // past the end: the token's last words, not used
                    }
                    // (the wait stands in the block of the loads: no register of theirs is touched before they are back)
                    if constexpr (POLL == 5)
                        asm volatile("global_load_dwordx4 %0, %5, %10 sc0 sc1\n\tglobal_load_dwordx4 %1, %6, %10 sc0 sc1\n\t"
                                     "global_load_dwordx4 %2, %7, %10 sc0 sc1\n\tglobal_load_dwordx4 %3, %8, %10 sc0 sc1\n\t"
                                     "global_load_dwordx4 %4, %9, %10 sc0 sc1\n\ts_waitcnt vmcnt(0)"
                                     : "=&v"(got[0]), "=&v"(got[1]), "=&v"(got[2]), "=&v"(got[3]), "=&v"(got[4])
                                     : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "s"(src) : "memory");
                    else
                        asm volatile("global_load_dwordx4 %0, %3, %6 sc0 sc1\n\tglobal_load_dwordx4 %1, %4, %6 sc0 sc1\n\t"
                                     "global_load_dwordx4 %2, %5, %6 sc0 sc1\n\ts_waitcnt vmcnt(0)"
                                     : "=&v"(got[0]), "=&v"(got[1]), "=&v"(got[2])
                                     : "v"(off[0]), "v"(off[1]), "v"(off[2]), "s"(src) : "memory");
                    for (uint32_t tries = 0;; ++tries) {
                        bool fresh = true;
#pragma unroll
                        for (int i = 0; i < POLL; ++i) fresh &= got[i].y == tag && got[i].w == tag;
                        if (fresh) break;
                        if (tries >= a.patience) {
                            *k.lds_late = 1u;
                            break;
                        }
#pragma unroll
                        for (int i = 0; i < POLL; ++i)
                            if (got[i].y != tag || got[i].w != tag)
                                asm volatile("global_load_dwordx4 %0, %1, %2 sc0 sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(got[i]) : "v"(off[i]), "s"(src) : "memory");
                    }
#pragma unroll
                    for (int i = 0; i < POLL; ++i) {
                        const uint32_t e2 = base + tid + (uint32_t)i * THREADS;
                        if (e2 < n2) {
                            const uint32_t e = 2 * e2, sl = e / FI, ei = e % FI, q = ei >> 2;  // piece p = q / 16 reads float4 slot q ^ p
                            float* dst = reinterpret_cast<float*>(k.lds_act) + sl * FI + (((q ^ (q >> 4)) << 2) | (ei & 3u));
                            dst[0] = __uint_as_float(got[i].x);
                            dst[1] = __uint_as_float(got[i].z);
                        }
                    }
                }
            }
            __syncthreads();
            k.sum_acts();
            __syncthreads();
            float xf[64], sx[4];
            uint32_t cur_s = ~0u;
            for (uint32_t i0 = 0; i0 < mine; i0 += RD) {
#pragma unroll
                for (int i = 0; i < RD; ++i) {
                    const uint32_t n = i0 + (uint32_t)i;
                    if (n < mine) {
                        const uint32_t st = st0 + n * stp, s = st / groups, g = st % groups;
                        if (s != cur_s) {  // uniform
                            cur_s = s;
                            k.load_act(xf, sx, s);
                        }
                        const float v = group_sum(dot_f32(ring[i], (int)(li & 3u), xf, sx), 3);
                        if (n + RD < mine) {
                            float tie = v;
                            asm volatile("" : "+v"(tie));
                            fetch(ring[i], n + RD);
                        }
                        if (li == 0) k.lds_part[s * cols + 8 * g + sub] = v;
                    }
                }
            }
            // (every fetch has been consumed: a free wait that tells the compiler so, or it would make the next unit's first
            // fetches wait for the output store below)
            __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
            late = __builtin_amdgcn_readfirstlane((int)*k.lds_late) != 0;
            __syncthreads();
            if (late) break;
            k.store_unit(c);
            __syncthreads();  // lds_act / lds_part are rewritten by the next unit
        }
    }
    if (late) finish_alone<TG, TD, WAVES_, X_BF16>(smem, tid, b, G, tag);
    if (b == 0 && tid == 0) st_dev(k.s_epoch, tag);
}

}  // namespace

size_t moe_fused_scratch_bytes(uint32_t n_tokens, uint32_t n_experts, uint32_t top_k) {
    return (Layout{n_tokens, n_experts, top_k}.total() + 255) & ~(size_t)255;
}

namespace {
// The kernel instantiated for (gate / up type, down type), or null: one K-quant for all three, or Q4_K / Q5_K gate / up
// with a Q6_K down.
template <int W, int R, bool X_BF16>
void (*fused_kernel_of(hq_ggml_type t, hq_ggml_type td))(FusedArgs) {
    if (t == HQ_Q4_K && td == HQ_Q4_K) return moe_fused_kernel<HQ_Q4_K, HQ_Q4_K, W, R, X_BF16>;
    if (t == HQ_Q5_K && td == HQ_Q5_K) return moe_fused_kernel<HQ_Q5_K, HQ_Q5_K, W, R, X_BF16>;
    if (t == HQ_Q6_K && td == HQ_Q6_K) return moe_fused_kernel<HQ_Q6_K, HQ_Q6_K, W, R, X_BF16>;
    if (t == HQ_Q4_K && td == HQ_Q6_K) return moe_fused_kernel<HQ_Q4_K, HQ_Q6_K, W, R, X_BF16>;
    if (t == HQ_Q5_K && td == HQ_Q6_K) return moe_fused_kernel<HQ_Q5_K, HQ_Q6_K, W, R, X_BF16>;
    return nullptr;
}
// wide: the 12-wave form
void (*fused_kernel_for(hq_ggml_type t, hq_ggml_type td, bool bf16, bool wide = false))(FusedArgs) {
    if (bf16) return wide ? fused_kernel_of<12, 2, true>(t, td) : fused_kernel_of<8, 4, true>(t, td);
    return wide ? fused_kernel_of<12, 2, false>(t, td) : fused_kernel_of<8, 4, false>(t, td);
}
// Two tokens or more take the 12-wave form.
constexpr uint32_t fused_waves(uint32_t n_tokens) { return n_tokens >= 2u ? 12u : 8u; }
size_t fused_lds_bytes(uint32_t n_tokens, uint32_t n_experts, uint32_t top_k, bool bf16) {
    const size_t S = (size_t)top_k + 1, area = staged_x_bytes(bf16), act_bytes = S * (FI * 4 + FI / 16 * 4);
    return (area > act_bytes ? area : act_bytes) + (size_t)(n_experts + 1) * 4 + (size_t)top_k * 4 + S * 4 + S * 64 * 4 +
           (size_t)64 * fused_waves(n_tokens) * 4 + (size_t)fused_waves(n_tokens) * 4;
}
constexpr size_t kFusedMaxLds = 64 * 1024;
}  // namespace

// (A top-k whose activations do not fit -- 25 and more of 256 experts -- is not taken: callers run the separate dispatches.)
bool moe_fused_supported(uint32_t n_tokens, uint32_t hidden, uint32_t n_experts, uint32_t top_k, uint32_t inter,
                         uint32_t shared_inter, hq_ggml_type t, hq_ggml_type t_down, hq_act_dtype xdt) {
    return fused_kernel_for(t, t_down, xdt == HQ_BF16) != nullptr && (xdt == HQ_BF16 || xdt == HQ_F32) && hidden == FH && inter == FI && shared_inter == FI && n_tokens >= 1 &&
           n_tokens <= MAX_T && n_experts >= n_tokens && n_experts <= 256 && top_k >= 1 && top_k <= 64 && top_k <= n_experts &&
           fused_lds_bytes(n_tokens, n_experts, top_k, xdt == HQ_BF16) <= kFusedMaxLds;
}

int launch_moe_fused(hipStream_t s, const MoeFusedArgs& m) {
    FusedArgs a{};
    a.x = m.x;
    a.router = static_cast<const uint16_t*>(m.router);
    a.sh_lw = static_cast<const uint16_t*>(m.shared_gate_logit);
    a.eg = static_cast<const uint8_t*>(m.expert_gate);
    a.eu = static_cast<const uint8_t*>(m.expert_up);
    a.ed = static_cast<const uint8_t*>(m.expert_down);
    a.sg = static_cast<const uint8_t*>(m.shared_gate);
    a.su = static_cast<const uint8_t*>(m.shared_up);
    a.sd = static_cast<const uint8_t*>(m.shared_down);
    a.residual = m.residual;
    a.out = m.out;
    a.route_ids = m.route_ids;
    a.route_w = m.route_weights;
    a.scratch = static_cast<uint8_t*>(m.scratch);
    a.T = m.n_tokens;
    a.E = m.n_experts;
    a.K = m.top_k;
    a.stride_gu = m.stride_gate_up;
    a.stride_d = m.stride_down;
    a.m4 = m.t_gate_up == HQ_Q6_K ? N4 : M4;
    a.m2 = m.t_gate_up == HQ_Q5_K ? M1 : m.t_gate_up == HQ_Q6_K ? N2 : M2;
    a.magic = MAGIC;
    a.patience = m.spin_limit && m.spin_limit < PATIENCE ? m.spin_limit : PATIENCE;
    // from two tokens on the 12-wave form (17.8 / 22.5 / 34.3 us at 2 / 4 / 8 tokens against 19.0 / 24.2 / 34.8; one token: the same)
    const bool wide = m.n_tokens >= 2u;
    const uint32_t WAVES = fused_waves(m.n_tokens), THREADS = 64u * WAVES;
    auto kern = fused_kernel_for(m.t_gate_up, m.t_down, m.xdt == HQ_BF16, wide);
    if (!kern) return fail(HQ_ERR_UNSUPPORTED, "fused MoE block: gate / up type %d with down type %d", (int)m.t_gate_up, (int)m.t_down);
    uint32_t cus = 0;
    if (int rc = cu_count(&cus)) return rc;
    // every workgroup delivers at least one logit row, and one workgroup per CU
    const uint32_t rows = m.n_experts + (m.shared_gate_logit ? 1u : 0u);
    const uint32_t grid = cus < rows ? cus : rows;
    if (grid < m.n_tokens)  // after the logits a workgroup works for one token: every token needs a workgroup
        return fail(HQ_ERR_UNSUPPORTED, "fused MoE block: %u tokens over %u router rows", m.n_tokens, rows);
    const size_t lds = fused_lds_bytes(m.n_tokens, m.n_experts, m.top_k, m.xdt == HQ_BF16);
    if (lds > kFusedMaxLds) return fail(HQ_ERR_UNSUPPORTED, "fused MoE block: %zu bytes of LDS", lds);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(THREADS), lds, s, a);
    return check_launch("fused MoE block launch");
}

}  // namespace hq
