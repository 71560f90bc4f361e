// MoE routing for gfx950: per token row, top-k experts and their weights
// from the router's logits (the step before sorting).
//
// Modes (reference interface in parentheses):
//   * softmax top-k (topk_softmax, csrc/kernels/topk_softmax_kernels.cu:
//     380-500; fused_topk, aiter/fused_moe.py:1853-1923): experts ranked by
//     logit; weight exp(x - rowmax), divided by the sum over the k chosen
//     (renormalise) or over the whole row (plain softmax); optionally with
//     shared experts after the routed ones in each gating row, whose sigmoid
//     scores follow the k weights (topk_softmax_kernels.cu:326-353, 760-810);
//   * sigmoid top-k (topk_sigmoid, op_tests/test_moe_topk_sigmoid.py:28-32):
//     ranked by logit, weight sigmoid(x);
//   * grouped top-k (grouped_topk, aiter/ops/topk.py:163-197): softmax or
//     sigmoid scores; groups ranked by their best score; experts of the
//     topk_group best groups ranked by score;
//   * biased grouped top-k (biased_grouped_topk, aiter/ops/topk.py:116-160):
//     sigmoid scores; choice = score + correction bias; groups ranked by the
//     sum of their two best choices; experts of the chosen groups ranked by
//     choice; the weight is the unbiased score.
// Grouped modes multiply the weights by routed_scaling_factor (after the
// renormalisation when it is on). Ties go to the lower expert / group
// index. Weights come out in rank order.
//
// Two kernels. moe_route_wave_kernel gives a row a whole wave; lane l holds
// experts l*V .. l*V+V-1 (E <= 64 V <= 1024) and each rank is one maximum over
// the wave and a ballot. moe_route_kernel takes any grouping, with 16 or 64
// lanes per row and a (value, index) arg-max over them for each rank.
#include <type_traits>

#include "common.h"

namespace aiter_amd {

namespace route {

constexpr int kWaves = 4;         // waves per workgroup
constexpr int kMaxK = 32;
constexpr int kMaxGroups = 32;

enum Mode : int { SOFTMAX = 0, SIGMOID = 1, GROUPED = 2, BIASED = 3 };

struct Args {
    const void* gating;
    int dtype;
    int64_t M;
    int E;
    int k;
    int mode;
    int need_renorm;
    int softmax_scores;           // grouped: softmax (1) or sigmoid (0) scores
    int n_group;
    int topk_group;
    float scaling;
    const float* bias;
    float* w;
    int64_t ws;                   // row strides (elements) of the outputs
    int32_t* ids;
    int64_t is;
    int32_t* tei;                 // optional token_expert_indices [M, k]
    int64_t gs;                   // gating row stride (elements, >= E + ns)
    int ns;                       // shared experts: gating columns E .. E+ns-1
    int vec;                      // rows aligned for 4-element loads of a lane's logits
};

__device__ __forceinline__ float load_logit(const void* p, int dtype, int64_t i) {
    if (dtype == DT_FP32) return reinterpret_cast<const float*>(p)[i];
    const uint16_t b = reinterpret_cast<const uint16_t*>(p)[i];
    if (dtype == DT_BF16) return bf16_bits_to_f32(b);
    return (float)__builtin_bit_cast(_Float16, b);
}

// Reductions over the LPR lanes of one row: LPR = 64 uses cross-lane
// shuffles; LPR = 16 (four rows per wave) uses DPP row rotations, which stay
// in the VALU (no LDS round trip per step).
template <int LPR>
__device__ __forceinline__ float lane_xchg(float v, int step) {
    if constexpr (LPR == 64) {
        return __shfl_xor(v, step, 64);
    } else {
        int r;
        const int b = __builtin_bit_cast(int, v);
        switch (step) {   // row_ror:step within each 16-lane row
            case 8: r = __builtin_amdgcn_update_dpp(b, b, 0x128, 0xF, 0xF, false); break;
            case 4: r = __builtin_amdgcn_update_dpp(b, b, 0x124, 0xF, 0xF, false); break;
            case 2: r = __builtin_amdgcn_update_dpp(b, b, 0x122, 0xF, 0xF, false); break;
            default: r = __builtin_amdgcn_update_dpp(b, b, 0x121, 0xF, 0xF, false); break;
        }
        return __builtin_bit_cast(float, r);
    }
}

template <int LPR>
__device__ __forceinline__ int lane_xchg_i(int v, int step) {
    return __builtin_bit_cast(int, lane_xchg<LPR>(__builtin_bit_cast(float, v), step));
}

template <int LPR>
__device__ __forceinline__ float row_max(float v) {
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) v = __builtin_fmaxf(v, lane_xchg<LPR>(v, o));
    return v;
}

template <int LPR>
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) v += lane_xchg<LPR>(v, o);
    return v;
}

// (value, index) arg-max over the row's lanes: larger value, then lower index
template <int LPR>
__device__ __forceinline__ void row_argmax(float& v, int& i) {
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) {
        const float ov = lane_xchg<LPR>(v, o);
        const int oi = lane_xchg_i<LPR>(i, o);
        if (ov > v || (ov == v && oi < i)) {
            v = ov;
            i = oi;
        }
    }
}

// top-2 of the row's (a1 >= a2) pairs
template <int LPR>
__device__ __forceinline__ void row_top2(float& a1, float& a2) {
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) {
        const float b1 = lane_xchg<LPR>(a1, o);
        const float b2 = lane_xchg<LPR>(a2, o);
        const float hi = __builtin_fmaxf(a1, b1);
        const float lo = __builtin_fminf(a1, b1);
        a2 = __builtin_fmaxf(lo, __builtin_fmaxf(a2, b2));
        a1 = hi;
    }
}

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + expf(-x)); }

template <int V, int LPR>
__global__ __launch_bounds__(64 * kWaves) void moe_route_kernel(Args g) {
    constexpr int RPW = 64 / LPR;                     // rows per wave
    const int lane = threadIdx.x & (LPR - 1);         // lane within the row
    const int64_t row = ((int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6)) * RPW +
                        ((threadIdx.x & 63) / LPR);
    // rows past M still run (their loads are clamped, their stores skipped)
    // so every lane of a wave takes part in the row reductions
    const bool live = row < g.M;
    const int64_t lrow = live ? row : g.M - 1;
    const int E = g.E, k = g.k;
    const float NEG = -__builtin_inff();
    // ungrouped rows come here only with few experts (lanes16)
    constexpr bool kUngrouped = LPR == 16 && V <= 8;
    const bool softmax = kUngrouped && g.mode == SOFTMAX;
    const bool sigmoid = kUngrouped && g.mode == SIGMOID;

    float x[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int e = lane * V + j;
        x[j] = e < E ? load_logit(g.gating, g.dtype, lrow * g.gs + e) : NEG;
    }

    // score s (what the weight is taken from) and ranking key per expert
    float s[V], key[V];
    float m = NEG;
    if (softmax || (g.mode == GROUPED && g.softmax_scores)) {
        float lm = NEG;
#pragma unroll
        for (int j = 0; j < V; ++j) lm = __builtin_fmaxf(lm, x[j]);
        m = row_max<LPR>(lm);
    }
    if (softmax || sigmoid) {
#pragma unroll
        for (int j = 0; j < V; ++j) key[j] = x[j];
    } else {
        if (g.softmax_scores && g.mode == GROUPED) {
            float ls = 0.0f;
#pragma unroll
            for (int j = 0; j < V; ++j) {
                s[j] = lane * V + j < E ? expf(x[j] - m) : 0.0f;
                ls += s[j];
            }
            const float sum = row_sum<LPR>(ls);
#pragma unroll
            for (int j = 0; j < V; ++j) s[j] /= sum;
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) s[j] = lane * V + j < E ? sigmoid_f32(x[j]) : 0.0f;
        }
        // choice values, then the group scores
        float c[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const int e = lane * V + j;
            c[j] = e < E ? (g.mode == BIASED ? s[j] + g.bias[e] : s[j]) : NEG;
        }
        const int G = E / g.n_group;
        int ge[V];                    // group of each held expert (n_group: none)
#pragma unroll
        for (int j = 0; j < V; ++j) ge[j] = lane * V + j < E ? (lane * V + j) / G : g.n_group;
        float gsc[kMaxGroups];
#pragma unroll
        for (int gi = 0; gi < kMaxGroups; ++gi) {
            if (gi >= g.n_group) break;
            float a1 = NEG, a2 = NEG;
#pragma unroll
            for (int j = 0; j < V; ++j) {
                if (ge[j] == gi) {
                    if (c[j] > a1) {
                        a2 = a1;
                        a1 = c[j];
                    } else if (c[j] > a2) {
                        a2 = c[j];
                    }
                }
            }
            if (g.mode == BIASED) {
                row_top2<LPR>(a1, a2);
                gsc[gi] = a1 + a2;
            } else {
                gsc[gi] = row_max<LPR>(a1);
            }
        }
        // the topk_group best groups (lane-uniform)
        uint32_t chosen = 0;
        for (int t = 0; t < g.topk_group; ++t) {
            int best = -1;
            float bv = NEG;
#pragma unroll
            for (int gi = 0; gi < kMaxGroups; ++gi) {
                if (gi >= g.n_group) break;
                if (!((chosen >> gi) & 1u) && (best < 0 || gsc[gi] > bv)) {
                    best = gi;
                    bv = gsc[gi];
                }
            }
            chosen |= 1u << best;
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
            key[j] = ge[j] < g.n_group && ((chosen >> ge[j]) & 1u) ? c[j] : NEG;
        }
    }

    // ---- k ranks: wave arg-max, the owner retires the winner ----
    float sel_v[kMaxK];
    int sel_i[kMaxK];
    float sum_sel = 0.0f;
#pragma unroll
    for (int t = 0; t < kMaxK; ++t) {
        if (t >= k) break;
        float v = NEG;
        int i = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < V; ++j)
            if (key[j] > v) {          // ascending index: the lower one wins a tie
                v = key[j];
                i = lane * V + j;
            }
        row_argmax<LPR>(v, i);
        float w;
        if (softmax) {
            w = expf(v - m);
        } else if (sigmoid) {
            w = sigmoid_f32(v);
        } else {
            // the unbiased score of expert i, from its owner
            float own = 0.0f;
#pragma unroll
            for (int j = 0; j < V; ++j)
                if (lane * V + j == i) own = s[j];
            w = __shfl(own, (threadIdx.x & 63 & ~(LPR - 1)) + i / V, 64);
        }
#pragma unroll
        for (int j = 0; j < V; ++j)
            if (lane * V + j == i) key[j] = NEG, x[j] = NEG;
        sel_v[t] = w;
        sel_i[t] = i;
        sum_sel += w;
    }

    float scale = 1.0f;
    if (softmax) {
        if (g.need_renorm) {
            if (sum_sel != 0.0f) scale = 1.0f / sum_sel;
        } else {
            float rest = 0.0f;
#pragma unroll
            for (int j = 0; j < V; ++j)
                if (lane * V + j < E && x[j] != NEG) rest += expf(x[j] - m);
            const float Z = sum_sel + row_sum<LPR>(rest);
            if (Z != 0.0f) scale = 1.0f / Z;
        }
    } else if (!sigmoid) {
        scale = g.need_renorm ? g.scaling / sum_sel : g.scaling;
    }
#pragma unroll
    for (int t = 0; t < kMaxK; ++t) {
        if (t >= k) break;
        if (lane == t % LPR && live) {                  // top-17 and up: more ranks than 16 lanes
            g.w[row * g.ws + t] = sel_v[t] * scale;
            g.ids[row * g.is + t] = sel_i[t];
            if (g.tei) g.tei[row * k + t] = (int32_t)((int64_t)t * g.M + row);
        }
    }
    // shared experts (topk_softmax's fusion, topk_softmax_kernels.cu:326-353):
    // weight column k + j is sigmoid of gating column E + j, outside the
    // ranking and the renormalisation
    for (int j = lane; j < g.ns; j += LPR)
        if (live)
            g.w[row * g.ws + k + j] =
                sigmoid_f32(load_logit(g.gating, g.dtype, row * g.gs + E + j));
}

// ---- one row per wave, ranks picked by ballot ----
// A rank is one maximum over the wave's keys. The keys are the scores as
// order-preserving u32 (0: not a candidate -- NaN, -inf, past E, retired or
// in a group that was not kept), so the maximum needs one v_max per DPP step
// and no index beside it: the winner is the first lane whose own maximum
// equals the wave's (a ballot), and the expert its first key that does, the
// lower index on ties. The chosen value and expert of rank t stay in lane t,
// where the weights are computed once, side by side, after the last rank.
constexpr uint32_t kNoKey = 0;

__device__ __forceinline__ uint32_t order_key(float v) {
    // v + 0 turns -0 into +0, which ranks equal to it
    const uint32_t u = __builtin_bit_cast(uint32_t, v + 0.0f);
    const uint32_t k = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
    return v > -__builtin_inff() ? k : kNoKey;          // false for NaN and -inf
}

__device__ __forceinline__ float key_value(uint32_t k) {
    return __builtin_bit_cast(float, (k & 0x80000000u) ? k ^ 0x80000000u : ~k);
}

// v of another lane by a DPP control (row_mask: the 16-lane rows that take it;
// the others keep v)
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xF, false);
}

template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, dpp_u<CTRL, ROWS>(__builtin_bit_cast(uint32_t, v)));
}

__device__ __forceinline__ float lane_f(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Wave-wide reduction in registers: rotations within the 16-lane rows, then
// the two row broadcasts, which leave the result in lane 63. The broadcasts
// combine a row's result with the rows before it only where it is taken.
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
    auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
    v = mx(v, dpp_u<0x128>(v));
    v = mx(v, dpp_u<0x124>(v));
    v = mx(v, dpp_u<0x122>(v));
    v = mx(v, dpp_u<0x121>(v));
    v = mx(v, dpp_u<0x142, 0xA>(v));
    v = mx(v, dpp_u<0x143, 0xC>(v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_f<0x128>(v);
    v += dpp_f<0x124>(v);
    v += dpp_f<0x122>(v);
    v += dpp_f<0x121>(v);
    // the rows' sums sit in every lane of their row
    return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}

// The row's logits of this lane, experts lane * V ..; a lane's V logits come
// in aligned vector loads where the host found the rows aligned for them.
template <int V>
__device__ __forceinline__ void load_logits(const Args& g, int64_t row, int lane, float (&x)[V]) {
    const int64_t i0 = row * g.gs + lane * V;
    const float NEG = -__builtin_inff();
    if constexpr (V % 4 == 0) {
        if (g.vec) {
            const bool in = lane * V < g.E;              // E % V == 0
#pragma unroll
            for (int j = 0; j < V; j += 4) {
                if (g.dtype == DT_FP32) {
                    v4f q = {NEG, NEG, NEG, NEG};
                    if (in)
                        q = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(g.gating) +
                                                          i0 + j);
#pragma unroll
                    for (int u = 0; u < 4; ++u) x[j + u] = q[u];
                } else {
                    v2i q = {0, 0};
                    if (in)
                        q = *reinterpret_cast<const v2i*>(
                            reinterpret_cast<const uint16_t*>(g.gating) + i0 + j);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const uint16_t b = (uint16_t)((uint32_t)q[u >> 1] >> (16 * (u & 1)));
                        x[j + u] = !in                  ? NEG
                                   : g.dtype == DT_BF16 ? bf16_bits_to_f32(b)
                                                        : fp16_bits_to_f32(b);
                    }
                }
            }
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j)
        x[j] = lane * V + j < g.E ? load_logit(g.gating, g.dtype, i0 + j) : NEG;
}

// Ranking keys and scores of the grouped modes. E = 64 V and n_group a power
// of two, so a group is LG = 64 / n_group whole lanes: every lane finds the
// best (two) of its own experts, a butterfly over the LG lanes gives all the
// groups' scores at once, and a lane counts the groups that beat its own
// instead of picking the kept groups one after another.
template <int V>
__device__ __forceinline__ void group_keys(const Args& g, int lane, const float (&x)[V],
                                           float (&s)[V], uint32_t (&key)[V]) {
    const float NEG = -__builtin_inff();
    const bool biased = g.mode == BIASED;
    float b[V];
#pragma unroll
    for (int j = 0; j < V; ++j) b[j] = biased ? g.bias[lane * V + j] : 0.0f;
    if (g.softmax_scores && !biased) {
        float m = x[0];
#pragma unroll
        for (int j = 1; j < V; ++j) m = __builtin_fmaxf(m, x[j]);
        m = __builtin_fmaxf(m, dpp_f<0x128>(m));
        m = __builtin_fmaxf(m, dpp_f<0x124>(m));
        m = __builtin_fmaxf(m, dpp_f<0x122>(m));
        m = __builtin_fmaxf(m, dpp_f<0x121>(m));
        m = __builtin_fmaxf(__builtin_fmaxf(lane_f(m, 0), lane_f(m, 16)),
                            __builtin_fmaxf(lane_f(m, 32), lane_f(m, 48)));
        float ls = 0.0f;
#pragma unroll
        for (int j = 0; j < V; ++j) {
            s[j] = expf(x[j] - m);
            ls += s[j];
        }
        const float sum = wave_sum(ls);
#pragma unroll
        for (int j = 0; j < V; ++j) s[j] /= sum;
    } else {
#pragma unroll
        for (int j = 0; j < V; ++j) s[j] = sigmoid_f32(x[j]);
    }
    float c[V], a1 = NEG, a2 = NEG;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        c[j] = biased ? s[j] + b[j] : s[j];
        const float v = c[j] > NEG ? c[j] : NEG;         // NaN never leads a group
        a2 = __builtin_fmaxf(a2, __builtin_fminf(a1, v));
        a1 = __builtin_fmaxf(a1, v);
    }
    auto merge = [&](float o1, float o2) {
        a2 = __builtin_fmaxf(__builtin_fminf(a1, o1), __builtin_fmaxf(a2, o2));
        a1 = __builtin_fmaxf(a1, o1);
    };
    // lanes 1, 2, 4 and 8 apart; the mirrors stand for 4 and 8 apart, as the
    // quads (eights) are uniform by then
    const int LG = 64 / g.n_group;
    if (LG >= 2) merge(dpp_f<0xB1>(a1), dpp_f<0xB1>(a2));
    if (LG >= 4) merge(dpp_f<0x4E>(a1), dpp_f<0x4E>(a2));
    if (LG >= 8) merge(dpp_f<0x141>(a1), dpp_f<0x141>(a2));
    if (LG >= 16) merge(dpp_f<0x140>(a1), dpp_f<0x140>(a2));
    if (LG >= 32) merge(__shfl_xor(a1, 16, 64), __shfl_xor(a2, 16, 64));
    if (LG >= 64) merge(__shfl_xor(a1, 32, 64), __shfl_xor(a2, 32, 64));
    const float gsc = biased ? a1 + a2 : a1;
    const int mine = lane / LG;
    bool kept;
    if (__builtin_amdgcn_ballot_w64(gsc != gsc) == 0) {
        int better = 0;
        for (int h = 0; h < g.n_group; ++h) {
            const float o = lane_f(gsc, h * LG);
            better += o > gsc || (o == gsc && h < mine);
        }
        kept = better < g.topk_group;
    } else {
        // a NaN group score (inf - inf, from infinite biases) keeps the place
        // it has in a scan for the first larger score
        uint32_t chosen = 0;
        for (int t = 0; t < g.topk_group; ++t) {
            int best = -1;
            float bv = NEG;
            for (int h = 0; h < g.n_group; ++h) {
                const float o = lane_f(gsc, h * LG);
                if (!((chosen >> h) & 1u) && (best < 0 || o > bv)) {
                    best = h;
                    bv = o;
                }
            }
            chosen |= 1u << best;
        }
        kept = (chosen >> mine) & 1u;
    }
#pragma unroll
    for (int j = 0; j < V; ++j) key[j] = kept ? order_key(c[j]) : kNoKey;
}

// Bound by latency up to a few thousand rows (a serial chain of k ranks) and
// by VALU issue beyond. Measured on MI355X, launches back to back in a graph,
// E = 256, top-8, against the arg-max kernel: softmax T=1 8.1 -> 3.0 us, T=32
// 8.5 -> 3.3, T=8192 11.5 -> 7.2, T=16384 21.4 -> 11.6; biased grouped (8
// groups) T=32 14.5 -> 4.6, T=8192 28.9 -> 10.7, T=16384 53.8 -> 17.9.
template <int V, bool GROUP>
__global__ __launch_bounds__(64 * kWaves) void moe_route_wave_kernel(Args g) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= g.M) return;                              // whole waves, no barrier below
    const int k = g.k;
    const float NEG = -__builtin_inff();
    float x[V], s[V];
    uint32_t key[V];
    load_logits<V>(g, row, lane, x);
    if constexpr (GROUP) {
        group_keys<V>(g, lane, x, s, key);
    } else {
#pragma unroll
        for (int j = 0; j < V; ++j) key[j] = order_key(x[j]);
    }

    float sel_v = 0.0f, m = NEG;      // rank `lane`: its logit (grouped: score) and expert
    int sel_i = 0;
    for (int t = 0; t < k; ++t) {
        uint32_t lm = key[0];
#pragma unroll
        for (int j = 1; j < V; ++j) lm = key[j] > lm ? key[j] : lm;
        int first = V - 1;
        float own = GROUP ? s[V - 1] : 0.0f;
#pragma unroll
        for (int j = V - 2; j >= 0; --j) {
            const bool is = key[j] == lm;
            first = is ? j : first;
            if (GROUP) own = is ? s[j] : own;
        }
        const uint32_t top = wave_max_u(lm);
        const int win = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lm == top));
        const int j = __builtin_amdgcn_readlane(first, win);
        const bool any = top != kNoKey;
        const float v = any ? (GROUP ? lane_f(own, win) : key_value(top)) : (GROUP ? 0.0f : NEG);
        if (t == 0) m = v;
        if (lane == t) {
            sel_v = v;
            sel_i = any ? win * V + j : 0x7fffffff;
        }
#pragma unroll
        for (int u = 0; u < V; ++u)
            if (lane == win && u == j) key[u] = kNoKey;
    }

    float w = sel_v;
    if (g.mode == SOFTMAX)
        w = expf(sel_v - m);                             // m: the row's maximum, rank 0
    else if (g.mode == SIGMOID)
        w = sigmoid_f32(sel_v);
    float sum_sel = 0.0f;
    for (int t = 0; t < k; ++t) sum_sel += lane_f(w, t);
    float scale = 1.0f;
    if (g.mode == SOFTMAX) {
        float Z = sum_sel;
        if (!g.need_renorm) {
            // the rest of the row: what was not chosen (a NaN has no key)
            float rest = 0.0f;
#pragma unroll
            for (int u = 0; u < V; ++u)
                if (key[u] != kNoKey || x[u] != x[u]) rest += expf(x[u] - m);
            Z += wave_sum(rest);
        }
        if (Z != 0.0f) scale = 1.0f / Z;
    } else if (g.mode != SIGMOID) {
        scale = g.need_renorm ? g.scaling / sum_sel : g.scaling;
    }
    if (lane < k) {
        g.w[row * g.ws + lane] = w * scale;
        g.ids[row * g.is + lane] = sel_i;
        if (g.tei) g.tei[row * k + lane] = (int32_t)((int64_t)lane * g.M + row);
    }
    for (int u = lane; u < g.ns; u += 64)
        g.w[row * g.ws + k + u] =
            sigmoid_f32(load_logit(g.gating, g.dtype, row * g.gs + g.E + u));
}

// Experts per lane of the one-row-per-wave kernel.
static int wave_v(int64_t E) {
    const int64_t v = ceil_div(E, 64);
    return (int)(v <= 6 ? v : v <= 8 ? 8 : v <= 12 ? 12 : 16);
}

// Grouped rows that kernel takes: every lane full, whole lanes per group.
static bool wave_groups(int64_t E, int64_t n_group) {
    return E == 64 * wave_v(E) && n_group >= 1 && n_group <= 32 && 64 % n_group == 0;
}

// Ungrouped rows that 16 lanes take faster than a wave: many rows of few
// experts, whose 64 lanes are mostly empty. Measured on MI355X, launches back
// to back in a graph, us on 16 lanes / on the wave (bf16, top-8):
//   E = 8, top-2, any mode: T=4096 3.0 / 2.6, T=8192 3.2 / 3.3, T=16384 4.1 / 4.7;
//   softmax over the whole row, whose second pass of exponentials a wave's lanes
//   pay for however few experts they hold: E = 64 T=14336 9.4 / 9.0, T=16384
//   9.4 / 9.9, T=65536 30.0 / 31.9; E = 72 T=32768 20.5 / 20.9, T=65536 36.7 /
//   38.8; E = 96 T=32768 21.1 / 20.9, T=65536 37.7 / 38.3; E = 128 T=65536 37.5 /
//   38.5, but 39.3 / 39.2 with fp32 logits and top-4 faster on the wave;
//   softmax over the chosen: E = 64 T=32768 15.8 / 15.7, T=65536 27.9 / 28.2,
//   T=131072 51.9 / 53.1; E = 72 and up level;
//   sigmoid: E = 64 T=65536 28.7 / 27.2.
static bool lanes16(int64_t M, int64_t E, int mode, int need_renorm) {
    if (E <= 16) return M >= 8192;
    if (mode != SOFTMAX) return false;
    if (need_renorm) return E <= 64 && M >= 65536;
    return E <= 64 ? M >= 16384 : E <= 96 && M >= 65536;
}

// Grouped rows of whole lanes that 16 lanes take faster: softmax scores, one or
// two groups of 64 experts (a lane holds one expert and the groups cost the
// general kernel little). us on 16 lanes / on the wave, top-4: one group T=10240
// 7.8 / 7.2, T=12288 7.9 / 8.1, T=16384 8.9 / 9.8, T=65536 26.8 / 30.8; two groups
// T=12288 8.0 / 8.0, T=16384 9.5 / 9.6, T=65536 28.2 / 30.6; four groups T=65536
// 32.9 / 30.9.
static bool lanes16_grouped(int64_t M, int64_t E, int64_t n_group, int mode, int softmax_scores) {
    return mode == GROUPED && softmax_scores && E == 64 && n_group <= 2 &&
           M >= (n_group == 1 ? 12288 : 16384);
}

}  // namespace route

bool route_supported(int64_t E, int64_t k) {
    return E >= 1 && E <= 1024 && k >= 1 && k <= route::kMaxK && k <= E;
}

void launch_moe_route(const void* gating, int dtype, int64_t M, int64_t E, int64_t k, int mode,
                      int need_renorm, int softmax_scores, int64_t n_group, int64_t topk_group,
                      float scaling, const float* bias, float* w, int64_t ws, int32_t* ids,
                      int64_t is, int32_t* tei, hipStream_t stream, int64_t gating_stride,
                      int64_t num_shared) {
    route::Args g{};
    g.gs = gating_stride > 0 ? gating_stride : E;
    g.ns = (int)num_shared;
    g.gating = gating;
    g.dtype = dtype;
    g.M = M;
    g.E = (int)E;
    g.k = (int)k;
    g.mode = mode;
    g.need_renorm = need_renorm;
    g.softmax_scores = softmax_scores;
    g.n_group = (int)n_group;
    g.topk_group = (int)topk_group;
    g.scaling = scaling;
    g.bias = bias;
    g.w = w;
    g.ws = ws;
    g.ids = ids;
    g.is = is;
    g.tei = tei;
    const bool grouped = mode >= route::GROUPED;
    const dim3 block(64 * route::kWaves);
    const dim3 g16((unsigned)ceil_div(M, 4 * route::kWaves));
    const dim3 g64((unsigned)ceil_div(M, route::kWaves));
    // one row per wave with ballot-picked ranks, where the row suits it
    if (grouped ? route::wave_groups(E, n_group) && !route::lanes16_grouped(M, E, n_group, mode,
                                                                            softmax_scores)
                : !route::lanes16(M, E, mode, need_renorm)) {
        g.vec = g.gs % 4 == 0 && reinterpret_cast<uintptr_t>(gating) % 16 == 0;
        auto go = [&](auto v) {
            constexpr int V = decltype(v)::value;
            g.vec = g.vec && E % V == 0;
            if (grouped)
                hipLaunchKernelGGL((route::moe_route_wave_kernel<V, true>), g64, block, 0, stream,
                                   g);
            else
                hipLaunchKernelGGL((route::moe_route_wave_kernel<V, false>), g64, block, 0,
                                   stream, g);
        };
        switch (route::wave_v(E)) {
            case 1: go(std::integral_constant<int, 1>{}); break;
            case 2: go(std::integral_constant<int, 2>{}); break;
            case 3: go(std::integral_constant<int, 3>{}); break;
            case 4: go(std::integral_constant<int, 4>{}); break;
            case 5: go(std::integral_constant<int, 5>{}); break;
            case 6: go(std::integral_constant<int, 6>{}); break;
            case 8: go(std::integral_constant<int, 8>{}); break;
            case 12: go(std::integral_constant<int, 12>{}); break;
            default: go(std::integral_constant<int, 16>{}); break;
        }
        AMD_HIP_CHECK(hipGetLastError());
        return;
    }
    // The others: 16 lanes per row up to E = 256 (four rows per wave); wider
    // rows, and the grouped modes under 1024 tokens (a per-group pass over
    // each lane's experts, latency-bound when there are few rows), the whole
    // wave per row.
    if (grouped && M < 1024) {
        if (E <= 64)
            hipLaunchKernelGGL((route::moe_route_kernel<1, 64>), g64, block, 0, stream, g);
        else if (E <= 128)
            hipLaunchKernelGGL((route::moe_route_kernel<2, 64>), g64, block, 0, stream, g);
        else if (E <= 256)
            hipLaunchKernelGGL((route::moe_route_kernel<4, 64>), g64, block, 0, stream, g);
        else if (E <= 512)
            hipLaunchKernelGGL((route::moe_route_kernel<8, 64>), g64, block, 0, stream, g);
        else
            hipLaunchKernelGGL((route::moe_route_kernel<16, 64>), g64, block, 0, stream, g);
    } else if (E <= 16)
        hipLaunchKernelGGL((route::moe_route_kernel<1, 16>), g16, block, 0, stream, g);
    else if (E <= 64)
        hipLaunchKernelGGL((route::moe_route_kernel<4, 16>), g16, block, 0, stream, g);
    else if (E <= 128)
        hipLaunchKernelGGL((route::moe_route_kernel<8, 16>), g16, block, 0, stream, g);
    else if (E <= 256)
        hipLaunchKernelGGL((route::moe_route_kernel<16, 16>), g16, block, 0, stream, g);
    else if (E <= 512)
        hipLaunchKernelGGL((route::moe_route_kernel<8, 64>), g64, block, 0, stream, g);
    else
        hipLaunchKernelGGL((route::moe_route_kernel<16, 64>), g64, block, 0, stream, g);
    AMD_HIP_CHECK(hipGetLastError());
}

}  // namespace aiter_amd
