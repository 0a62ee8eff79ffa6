// Routed experts for a flat batch of tokens.  The router's logits, the choice of the `top` largest and their softmax
// are 32-bit.  The experts' products pick every (token, chosen expert) pair's matrices on the device from the list
// the router wrote: a pair streams its expert's gate and up rows against the token's row and applies silu(gate) * up;
// a token's output row is the weighted sum over its pairs of the expert's down rows against the pair's hidden row.
// Sums are 32-bit; the hidden row is rounded once to the activations' type; the output is float32.
//
// Experts without a gate (`plain`) have one matrix that reads the token, and max(up, 0)^2 in place of silu(gate) * up.
//
// Beside the experts that have matrices there may be identity experts: choices from `experts` on, whose output is the token's
// row itself.  And there may be a shared expert that every token uses, possibly weighted by a gate of one number a token: its
// products are made inside the same two kernels (steps of few tokens), or its output comes ready made.
#include "common.hpp"
#include "lds_loads.hpp"
#include "wide_product.hpp"

#include <math.h>

using namespace lsa;

constexpr float NEG_INF = -__builtin_huge_valf();

// The experts' activation.  limit <= 0: silu(gate) * up.  limit > 0: the clamped form g * sigmoid(1.702 g) * (u + 1) with
// g = min(gate, limit), u = clamp(up, -limit, limit).
__device__ __forceinline__ float gated_activation(float g, float u, float limit) {
    if (limit > 0.f) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
    }
    return g / (1.f + expf(-g)) * u;
}

__device__ __forceinline__ float rectified_square(float u) {
    u = fmaxf(u, 0.f);
    return u * u;
}

// Dot product of a weight row with a vector in LDS, a wavefront wide: 16-byte pieces where the length allows.
template <typename T>
__device__ inline float wave_dot(const T* __restrict__ w, const T* x_lds, int n, int lane) {
    constexpr int V = Elem<T>::kVec;
    float acc = 0.f;
    if (n % V == 0 && ((reinterpret_cast<size_t>(w) | reinterpret_cast<size_t>(x_lds)) & 15) == 0) {
        for (int i = lane * V; i < n; i += 64 * V) {
            const Vec16<T> a = load_vec16(w + i);
            const Vec16<T> b = *reinterpret_cast<const Vec16<T>*>(x_lds + i);
#pragma unroll
            for (int k = 0; k < V; ++k) acc += (float)a.v[k] * (float)b.v[k];
        }
    } else {
        for (int i = lane; i < n; i += 64) acc += (float)w[i] * (float)x_lds[i];
    }
    return wave_sum(acc);
}

// Two rows at once against the same vector (a gate row and its up row): their loads are in flight together.
template <typename T>
__device__ inline void wave_dot2(const T* __restrict__ w0, const T* __restrict__ w1, const T* x_lds, int n, int lane, float& r0, float& r1) {
    constexpr int V = Elem<T>::kVec;
    float a0 = 0.f, a1 = 0.f;
    if (n % V == 0 && ((reinterpret_cast<size_t>(w0) | reinterpret_cast<size_t>(w1) | reinterpret_cast<size_t>(x_lds)) & 15) == 0) {
        for (int i = lane * V; i < n; i += 64 * V) {
            const Vec16<T> p = load_vec16(w0 + i);
            const Vec16<T> q = load_vec16(w1 + i);
            const Vec16<T> b = *reinterpret_cast<const Vec16<T>*>(x_lds + i);
#pragma unroll
            for (int k = 0; k < V; ++k) {
                a0 += (float)p.v[k] * (float)b.v[k];
                a1 += (float)q.v[k] * (float)b.v[k];
            }
        }
    } else {
        for (int i = lane; i < n; i += 64) {
            a0 += (float)w0[i] * (float)x_lds[i];
            a1 += (float)w1[i] * (float)x_lds[i];
        }
    }
    r0 = wave_sum(a0);
    r1 = wave_sum(a1);
}

// Router logits for steps of few tokens, where a library product would be a launch of 11 us for a few thousand
// multiplications: grid (tokens, experts / 4), a wavefront per expert; the rows are widened as they are read, the rest is float32.
template <typename T>
__global__ __launch_bounds__(256) void route_logits_kernel(const T* __restrict__ x, const float* __restrict__ router,
                                                           float* __restrict__ logits, int experts, int width) {
    const int lane = threadIdx.x & 63, e = blockIdx.y * 4 + (threadIdx.x >> 6), t = blockIdx.x;
    if (e >= experts) return;
    const float* r = router + (size_t)e * width;
    const T* row = x + (size_t)t * width;
    float acc = 0.f;
    if (width % 4 == 0) {
        struct alignas(4 * sizeof(T)) Four { T v[4]; };
        for (int i = lane * 4; i < width; i += 256) {
            const float4 a = *reinterpret_cast<const float4*>(r + i);
            const Four b = *reinterpret_cast<const Four*>(row + i);
            acc += a.x * (float)b.v[0] + a.y * (float)b.v[1] + a.z * (float)b.v[2] + a.w * (float)b.v[3];
        }
    } else {
        for (int i = lane; i < width; i += 64) acc += r[i] * (float)row[i];
    }
    acc = wave_sum(acc);
    if (lane == 0) logits[(size_t)t * experts + e] = acc;
}

// Router logits for steps of up to a few hundred tokens, as partial sums [parts][tokens][experts] over ranges of the width that whoever
// chooses adds up: on 64-bit MFMA (two scores can lie a rounding apart; the kernel waits for memory either way), 16 tokens x 16 experts a workgroup, its four wavefronts a quarter of the range each.  A router
// has few rows, so what bounds the product is one walk over the width by few workgroups: cut into ranges of about 512 numbers a
// wavefront asks for all it reads at once (32 rows of 2048: 7.1 us, 6.0 with 32-bit sums, against 5 us for widening the rows and 12 us for the library's
// product).  Rows are widened as they are read; the width is a multiple of 8.
constexpr int ROUTE_PARTS = 8;           // most ranges
typedef double route_d4 __attribute__((ext_vector_type(4)));

template <typename T>
__global__ __launch_bounds__(256) void route_logits_parts_kernel(const T* __restrict__ x, const float* __restrict__ router,
                                                                 float* __restrict__ logits, int tokens, int experts, int width, int range) {
    __shared__ double s_sum[4][16][17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int begin = blockIdx.z * range + wave * (range / 4), end = min(width, begin + range / 4);
    const T* row = x + (size_t)min((int)blockIdx.x * 16 + r, tokens - 1) * width;
    const float* weights = router + (size_t)min((int)blockIdx.y * 16 + r, experts - 1) * width;
    struct alignas(16) Eight { T v[8]; };
    route_d4 part[2] = {};
#pragma unroll 4
    for (int k0 = begin; k0 < end; k0 += 32) {
        // (a piece behind the range's end is read from the width's last eight numbers and counts nothing)
        const int k = min(k0 + 8 * g, width - 8);
        const bool counts = k0 + 8 * g < end;
        const Eight a = *reinterpret_cast<const Eight*>(row + k);
        const float4 low = *reinterpret_cast<const float4*>(weights + k), high = *reinterpret_cast<const float4*>(weights + k + 4);
        const float b[8] = {low.x, low.y, low.z, low.w, high.x, high.y, high.z, high.w};
#pragma unroll
        for (int u = 0; u < 8; ++u)
            part[u & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(counts ? (double)(float)a.v[u] : 0.0, counts ? (double)b[u] : 0.0, part[u & 1], 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s_sum[wave][4 * e + g][r] = part[0][e] + part[1][e];
    __syncthreads();
    const int m = threadIdx.x >> 4, c = threadIdx.x & 15, t = blockIdx.x * 16 + m, e = blockIdx.y * 16 + c;
    if (t < tokens && e < experts)
        logits[((size_t)blockIdx.z * tokens + t) * experts + e] =
            (float)((s_sum[0][m][c] + s_sum[1][m][c]) + (s_sum[2][m][c] + s_sum[3][m][c]));
}

// The largest (smallest) of 64 lanes' numbers, in every lane: inside rows of 16 lanes by data-parallel moves, the four rows as scalars.
template <int CTRL>
__device__ __forceinline__ int from_across(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, true); }
__device__ __forceinline__ float largest_of_64(float v) {
    v = fmaxf(v, __int_as_float(from_across<0xB1>(__float_as_int(v))));         // quad_perm [1, 0, 3, 2]
    v = fmaxf(v, __int_as_float(from_across<0x4E>(__float_as_int(v))));         // quad_perm [2, 3, 0, 1]
    v = fmaxf(v, __int_as_float(from_across<0x141>(__float_as_int(v))));        // row_half_mirror
    v = fmaxf(v, __int_as_float(from_across<0x140>(__float_as_int(v))));        // row_mirror
    const int bits = __float_as_int(v);
    return fmaxf(fmaxf(__int_as_float(__builtin_amdgcn_readlane(bits, 0)), __int_as_float(__builtin_amdgcn_readlane(bits, 16))),
                 fmaxf(__int_as_float(__builtin_amdgcn_readlane(bits, 32)), __int_as_float(__builtin_amdgcn_readlane(bits, 48))));
}
__device__ __forceinline__ int smallest_of_64(int v) {
    v = min(v, from_across<0xB1>(v));
    v = min(v, from_across<0x4E>(v));
    v = min(v, from_across<0x141>(v));
    v = min(v, from_across<0x140>(v));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// One wavefront per token: the `top` largest of the token's float32 logits (the lowest index among equal ones) and
// their softmax.  The logits themselves are a float32 matrix product made before this kernel, rows of `stride` numbers, in `parts` partial
// sums [parts][tokens][stride].  A lane keeps the weight of the choice of its own number, so that the weights are divided by their sum
// and written once (one lane that reads its own writes again waits for memory `top` times: 32 rows, 8 of 128 experts 11.3 -> 7.8 us).
// scoring 0: that; 1: sigmoid(logits) are scores, choice values and weights; 2: the scores are the softmax over all experts,
// the choice values scores + correction, the weights the chosen scores divided by (their sum + 1e-20), times weight_scale.
// gate_out (or nullptr): sigmoid of the logit behind the experts', a gate of one number a token.  A lane keeps the logits
// of experts lane, lane + 64, ... in LDS (its own entries only: nothing crosses lanes through LDS), and every lane ends
// each round with the same (best, where).
__global__ __launch_bounds__(256) void route_top_kernel(const float* __restrict__ all_logits, int experts, int top,
                                                        int* __restrict__ chosen, float* __restrict__ weights, int n_tokens,
                                                        int scoring, int groups, int keep, const float* __restrict__ bias,
                                                        const float* __restrict__ correction, float weight_scale, int stride,
                                                        float* __restrict__ gate_out, int parts) {
    extern __shared__ float lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * (blockDim.x >> 6) + wave;
    if (t >= n_tokens) return;
    // (two arrays a wavefront: the values the choice is made among, and, for sigmoid scores, the scores themselves)
    float* logits = lds + (size_t)wave * 2 * experts;
    float* scores = logits + experts;
    const bool sigmoid_scores = scoring == 1;
    // (the partial sums' loads are issued together, those behind the last one of the last one again)
    const auto logit = [&](int e) {
        const float* first = all_logits + (size_t)t * stride + e;
        if (parts == 1) return first[0];
        float piece[ROUTE_PARTS];
        double sum = 0.0;
#pragma unroll
        for (int part = 0; part < ROUTE_PARTS; ++part) piece[part] = first[(size_t)min(part, parts - 1) * n_tokens * stride];
#pragma unroll
        for (int part = 0; part < ROUTE_PARTS; ++part) sum += part < parts ? (double)piece[part] : 0.0;
        return (float)sum;
    };
    if (gate_out && lane == 0) gate_out[t] = 1.f / (1.f + expf(-logit(experts)));
    float most = NEG_INF;
    for (int e = lane; e < experts; e += 64) {
        float v = logit(e);
        if (bias) v += bias[e];                            // (a bias per expert joins the logits)
        most = fmaxf(most, v);
        if (sigmoid_scores) v = 1.f / (1.f + expf(-v));
        scores[e] = v;
        logits[e] = v;
    }
    if (scoring == 2) {                                    // the softmax over all experts (a lane meets its own entries only)
        most = wave_max(most);
        float all = 0.f;
        for (int e = lane; e < experts; e += 64) {
            const float v = expf(scores[e] - most);
            scores[e] = v;
            all += v;
        }
        all = wave_sum(all);
        for (int e = lane; e < experts; e += 64) {
            const float v = scores[e] / all;
            scores[e] = v;
            logits[e] = correction ? v + correction[e] : v;
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (sigmoid_scores && groups > 1) {
        // A group's score is the sum of its two largest scores; the `keep` best groups stay (the first of equal ones),
        // the experts of the others cannot be chosen.  Lane g (and g + 64, ...) scores group g; entries of other lanes
        // are read here (a wavefront's LDS operations complete in the order they were issued).
        __builtin_amdgcn_wave_barrier();
        const int per = experts / groups;
        {
            const int base = 0, g = lane;             // (at most 64 groups: the host refuses more)
            float mine = NEG_INF;
            if (g < groups) {
                float first = NEG_INF, second = NEG_INF;
                for (int i = 0; i < per; ++i) {
                    const float v = scores[g * per + i];
                    if (v > first) { second = first; first = v; }
                    else if (v > second) second = v;
                }
                mine = per > 1 ? first + second : first;
            }
            // rank of my group among all: groups with a larger score, or an equal one and a smaller index, come first
            int before = 0;
            for (int other = 0; other < min(64, groups - base); ++other) {
                const float theirs = __shfl(mine, other, 64);
                before += (theirs > mine || (theirs == mine && other < lane)) ? 1 : 0;
            }
            if (g < groups && before >= keep)
                for (int i = 0; i < per; ++i) logits[g * per + i] = NEG_INF;
        }
        __builtin_amdgcn_wave_barrier();
    }
    float largest = 0.f, total = 0.f, mine = 0.f;
    for (int k = 0; k < top; ++k) {
        float best = NEG_INF;
        int where = 0x7fffffff;
        for (int e = lane; e < experts; e += 64) {
            const float v = logits[e];
            if (v > best || (v == best && e < where)) { best = v; where = e; }
        }
        const float most_left = largest_of_64(best);
        where = smallest_of_64(best == most_left ? where : 0x7fffffff);
        best = most_left;
        if (where >= experts) where = k < experts ? k : 0;        // (only if every logit left is NaN or -inf)
        if (k == 0) largest = best;
        float weight = sigmoid_scores ? best : expf(best - largest);
        // (a score stands in the entries of the lane that owns the expert; the wavefront's LDS operations keep their order)
        if (scoring == 2) weight = scores[where];
        total += weight;
        if (lane == 0) chosen[(size_t)t * top + k] = where;
        if (lane == (k & 63)) mine = weight;
        if ((k & 63) == 63 || k + 1 == top) {                     // (choices beyond the lanes' number wait in memory)
            const int at = (k & ~63) + lane;
            if (at <= k) weights[(size_t)t * top + at] = mine;
        }
        if ((where & 63) == lane) logits[where] = NEG_INF;
    }
    if (scoring == 1) return;
    for (int k = lane; k < top; k += 64) {                        // (a lane's own writes)
        const float weight = top <= 64 ? mine : weights[(size_t)t * top + k];
        weights[(size_t)t * top + k] = scoring == 0 ? weight / total : weight / (total + 1e-20f) * weight_scale;
    }
}

// The same for up to 64 * E experts in one group and up to 64 choices, which is what decoding steps of most models have: a lane keeps its experts'
// values in registers and its choice of its own number until the end, so that a round is two exchanges between lanes without LDS or memory, and a
// round's stores wait for nothing.  The same numbers bit by bit.  us a launch behind 64 MB of other reads, that kernel and this one: 6 of 64 of one token 4.9 and
// 3.1, 6 of 72 of 32 tokens in eight partial sums 6.5 and 3.9, of 8,192 tokens 11.5 and 8.3.  (PARTS: with the loads of partial sums under a condition on their number
// those of 32 tokens took 6.9, for the compiler then waits for them one by one.)
template <int E, bool PARTS>
__global__ __launch_bounds__(64) void route_top_registers_kernel(const float* __restrict__ all_logits, int experts, int top,
                                                                 int* __restrict__ chosen, float* __restrict__ weights, int n_tokens,
                                                                 int scoring, const float* __restrict__ bias, const float* __restrict__ correction,
                                                                 float weight_scale, int stride, float* __restrict__ gate_out, int parts) {
    const int lane = threadIdx.x, t = blockIdx.x;
    // Everything is asked for at once: lane's experts, the gate's logit (its partial sums in lanes of their own), bias and correction.
    const float* first = all_logits + (size_t)t * stride;
    const size_t part_stride = (size_t)n_tokens * stride;
    constexpr int MOST = PARTS ? ROUTE_PARTS : 1;                 // (partial sums behind the last are the last one's again: no load under a condition)
    float piece[E][MOST], add[E], gate_piece = 0.f;
    const float* added = bias ? bias : correction ? correction : first;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int e = min(lane + 64 * j, experts - 1);
#pragma unroll
        for (int part = 0; part < MOST; ++part) piece[j][part] = first[(PARTS ? (size_t)min(part, parts - 1) * part_stride : 0) + e];
        add[j] = added[e];
    }
    if (gate_out) gate_piece = first[(size_t)min(lane, parts - 1) * part_stride + experts];
    float value[E], score[E], most = NEG_INF;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        float v = piece[j][0];
        if constexpr (PARTS) {
            double sum = 0.0;
#pragma unroll
            for (int part = 0; part < MOST; ++part) sum += part < parts ? (double)piece[j][part] : 0.0;
            v = (float)sum;
        }
        if (bias) v += add[j];
        const bool there = lane + 64 * j < experts;
        if (there) most = fmaxf(most, v);
        if (scoring == 1) v = 1.f / (1.f + expf(-v));
        score[j] = v;
        value[j] = there ? v : NEG_INF;
    }
    if (gate_out) {
        double sum = 0.0;
#pragma unroll
        for (int part = 0; part < MOST; ++part) {
            const double one = (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(gate_piece), part));
            sum += part < parts ? one : 0.0;
        }
        if (lane == 0) gate_out[t] = 1.f / (1.f + expf(-(float)sum));
    }
    if (scoring == 2) {
        most = largest_of_64(most);
        float all = 0.f;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            if (lane + 64 * j < experts) {
                score[j] = expf(score[j] - most);
                all += score[j];
            }
        }
        all = wave_sum(all);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            score[j] /= all;
            if (lane + 64 * j < experts) value[j] = correction ? score[j] + add[j] : score[j];
        }
    }
    float largest = 0.f, total = 0.f, mine = 0.f;
    int my_choice = 0;
    for (int k = 0; k < top; ++k) {
        float best = NEG_INF;
        int where = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const int e = lane + 64 * j;
            if (e < experts && (value[j] > best || (value[j] == best && e < where))) { best = value[j]; where = e; }
        }
        const float most_left = largest_of_64(best);
        where = smallest_of_64(best == most_left ? where : 0x7fffffff);
        best = most_left;
        if (where >= experts) where = k < experts ? k : 0;        // (only if every logit left is NaN or -inf)
        if (k == 0) largest = best;
        float weight = scoring == 1 ? best : expf(best - largest);
        if (scoring == 2) {                                       // (the chosen expert's score, from the lane and place that keep it)
            weight = 0.f;
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const float kept = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(score[j]), where & 63));
                if (where >> 6 == j) weight = kept;
            }
        }
        total += weight;
        if (lane == k) {
            mine = weight;
            my_choice = where;
        }
#pragma unroll
        for (int j = 0; j < E; ++j)
            if (where == lane + 64 * j) value[j] = NEG_INF;
    }
    if (lane >= top) return;
    chosen[(size_t)t * top + lane] = my_choice;
    weights[(size_t)t * top + lane] = scoring == 1 ? mine : scoring == 0 ? mine / total : mine / (total + 1e-20f) * weight_scale;
}

// Where a workgroup of the two kernels below stands.  Together (several tokens, which may share experts; grid (XCDS * units, blocks / XCDS)): the tokens' or
// pairs' workgroups of one block of columns follow one another on one XCD (workgroups go round the eight in turn), so that what two of them read of one expert
// comes out of that XCD's cache the second time; with a block's workgroups all over the chip each reads it once on an XCD of its own.  48 pairs of about 35 of
// 64 experts of 1,408 at width 2,048: 86 -> 76 us for the first product, 44.5 -> 40.3 for the second (behind cold caches); 96 pairs 148 -> 120, 83 -> 77.  Two
// dimensions, because dividing by the number of units costs the workgroups of few tokens 0.4 us (the second product of two tokens, 2 of 8 experts of
// 1,024 at 1,024: 4.8 -> 5.3), and because one holds 2^24 workgroups only.  The pairs of one token share nothing and go one after another, grid (units,
// blocks): 8 of 128 experts of 768 at 2,048 14.0 us so, 14.8 in the other order, 6 of 64 of 1,408 15.2, 15.8.
constexpr int XCDS = 8;
__device__ __forceinline__ void shared_columns(bool together, int& unit, int& block) {
    unit = together ? (int)blockIdx.x / XCDS : (int)blockIdx.x;
    block = together ? (int)blockIdx.y * XCDS + ((int)blockIdx.x & (XCDS - 1)) : (int)blockIdx.y;
}
// The grid, or false where a launch does not hold it.
static bool shared_grid(bool together, long units, int blocks, dim3& grid) {
    const long wide = together ? units * XCDS : units, rounds = together ? (blocks + XCDS - 1) / XCDS : blocks;
    if (wide * 256 > 0xffffffffL || rounds > 65535) return false;
    grid = dim3((unsigned)wide, (unsigned)rounds);
    return true;
}

// workgroups (pairs x blocks of hidden columns, as shared_columns lays them): hidden[pair][f] = silu(G[f] . x) * (U[f] . x) for the pair's expert.  With a shared
// expert a token has one more pair, the last: the shared expert's matrices and its own hidden row [tokens][shared_inter].
// Pairs of identity experts (choices from `experts` on, where `identity`) have nothing to multiply.
template <typename T>
__global__ __launch_bounds__(256) void experts_gate_up_kernel(const T* __restrict__ x, const T* __restrict__ gate_up,
                                                              const int* __restrict__ chosen, T* __restrict__ hidden, int top,
                                                              int inter, int width, int experts, int columns_per_block, bool in_lds,
                                                              float limit, int identity, const T* __restrict__ shared_gate_up,
                                                              T* __restrict__ shared_hidden, int shared_inter, int plain, bool together) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    const int slots = top + (shared_gate_up ? 1 : 0);
    int unit, block;
    shared_columns(together, unit, block);
    const int t = unit / slots, slot = unit - t * slots;
    const bool shared = slot == top;
    const int pair = t * top + slot;
    int expert = shared ? 0 : chosen[pair];
    if (identity && expert >= experts) return;               // (the whole workgroup)
    if (block * columns_per_block >= (shared ? shared_inter : inter)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const T* x_lds = x + (size_t)t * width;                  // (a row too long for LDS is read where it lies)
    if (in_lds) {
        T* staged = reinterpret_cast<T*>(lds_bytes);
        for (int i = threadIdx.x; i < width; i += blockDim.x) staged[i] = x_lds[i];
        __syncthreads();
        x_lds = staged;
    }
    expert = expert < 0 ? 0 : expert >= experts ? experts - 1 : expert;
    const T* base = shared ? shared_gate_up : gate_up + (size_t)expert * (plain ? 1 : 2) * inter * width;
    T* result = shared ? shared_hidden + (size_t)t * shared_inter : hidden + (size_t)pair * inter;
    if (shared) inter = shared_inter;
    const int f0 = block * columns_per_block, f1 = min(inter, f0 + columns_per_block);
    if (plain) {                                             // two columns at once, so that as many loads are in flight
        for (int f = f0 + wave; f < f1; f += 2 * waves) {
            const int other = min(f + waves, f1 - 1);
            float a, b;
            wave_dot2(base + (size_t)f * width, base + (size_t)other * width, x_lds, width, lane, a, b);
            if (lane == 0) result[f] = (T)rectified_square(a);
            if (lane == 0 && f + waves < f1) result[f + waves] = (T)rectified_square(b);
        }
        return;
    }
    for (int f = f0 + wave; f < f1; f += waves) {
        float g, u;
        wave_dot2(base + (size_t)f * width, base + (size_t)(inter + f) * width, x_lds, width, lane, g, u);
        if (lane == 0) result[f] = (T)gated_activation(g, u, limit);
    }
}

// workgroups (tokens x blocks of output columns, as shared_columns lays them): out[t][c] = sum_s weights[t][s] * (D_s[c] . hidden[t * top + s]).
// A wavefront owns a column: every lane adds up its share of all `top` dot products, weighted, and the lanes' sums meet
// once at the end; the loads of all pairs' rows are independent of one another.  Added to that: the token's row x times the
// weights of its identity experts (choices from `experts` on, where x is given), and the shared expert's output times the
// token's gate: shared_y ready made, or shared_down[c] . shared_hidden[t].
template <typename T> struct BesideExperts {
    const T* x;                     // [tokens][width], or nullptr: no identity experts
    const float* gate;              // [tokens]: what the shared expert's output is multiplied by, or nullptr: one
    const T* y;                     // [tokens][width]: its output, or nullptr: the two below
    const T* down;                  // [width][inter], or nullptr (and y nullptr): no shared expert
    const T* hidden;                // [tokens][inter]
    int inter;
};

// AHEAD: how many pieces of 16 bytes of the matrix a lane asks for before it uses the first.  With all conditions between them (a division, the expert and a wait a
// piece) a launch took, us, before and now: 6 of 64 experts of 1,408 at 2,048, 1 token 12.2, 8.9, 4 tokens 27.6, 21.7, 8 tokens 45.9, 39.6; 4 of 32 of 2,048 at 4,096, 2 tokens
// 25.7, 20.7, 8 tokens 78, 69.5; 8 of 128 of 768 at 2,048, 1 token 9.3, 7.2.  (Eight ahead leave too few wavefronts: 8 tokens 50.)
template <typename T, int AHEAD>
__global__ __launch_bounds__(256) void experts_down_kernel(const T* __restrict__ hidden, const T* __restrict__ down,
                                                           const int* __restrict__ chosen, const float* __restrict__ weights,
                                                           float* __restrict__ out, int top, int inter, int width, int experts,
                                                           int columns_per_block, bool in_lds, BesideExperts<T> beside, bool together) {
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    constexpr int V = Elem<T>::kVec;
    int t, block;
    shared_columns(together, t, block);
    if (block * columns_per_block >= width) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const T* h_lds = hidden + (size_t)t * top * inter;
    if (in_lds) {
        T* staged = reinterpret_cast<T*>(lds_bytes);
        for (int i = threadIdx.x; i < top * inter; i += blockDim.x) staged[i] = h_lds[i];
        __syncthreads();
        h_lds = staged;
    }
    const bool vectors = inter % V == 0 && ((reinterpret_cast<size_t>(down) | reinterpret_cast<size_t>(h_lds)) & 15) == 0;
    // the token's experts and weights, read once (a lookup per piece below would be a trip to memory each)
    constexpr int MOST = 128;
    __shared__ int expert_of[MOST];
    __shared__ float weight_of[MOST];
    __shared__ float identity_weight;
    for (int s = threadIdx.x; s < min(top, MOST); s += blockDim.x) {
        const int expert = chosen[(size_t)t * top + s];
        expert_of[s] = beside.x && expert >= experts ? -1 : expert < 0 ? 0 : expert >= experts ? experts - 1 : expert;
        weight_of[s] = weights[(size_t)t * top + s];
    }
    if (threadIdx.x == 0 && beside.x) {
        float total = 0.f;
        for (int s = 0; s < top; ++s)
            if (chosen[(size_t)t * top + s] >= experts) total += weights[(size_t)t * top + s];
        identity_weight = total;
    }
    const float gate = beside.gate ? beside.gate[t] : 1.f;
    const bool shared_vectors = beside.inter % V == 0 && ((reinterpret_cast<size_t>(beside.down) | reinterpret_cast<size_t>(beside.hidden)) & 15) == 0;
    __syncthreads();
    const int c0 = block * columns_per_block, c1 = min(width, c0 + columns_per_block);
    for (int c = c0 + wave; c < c1; c += waves) {
        float acc = 0.f;
        if (vectors && top <= MOST && (size_t)top * (inter / V) * (inter / V) < 0xFFFFFFFFu) {
            // The pairs' rows end to end are one long vector of top * inter / V pieces, spread over the lanes: every
            // lane is busy whatever the experts' size, and its loads do not wait for one another.
            const int pieces = inter / V, all = top * pieces;
            const unsigned inverse = 0xFFFFFFFFu / (unsigned)pieces + 1;      // p / pieces = p * inverse >> 32 while p * pieces < 2^32 and pieces > 1 (2^32 has no place here)
            for (int p0 = lane; p0 < all; p0 += 64 * AHEAD) {
                Vec16<T> a[AHEAD], b[AHEAD];
                float weight[AHEAD];
                bool counts[AHEAD];
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {                // (no load under a condition: the compiler would wait for each)
                    const int p = min(p0 + 64 * u, all - 1), s = pieces == 1 ? p : (int)__umulhi((unsigned)p, inverse), i = (p - s * pieces) * V, expert = expert_of[s];
                    weight[u] = weight_of[s];
                    counts[u] = p0 + 64 * u < all && expert >= 0;    // (not behind the last piece, no identity expert)
                    a[u] = load_vec16(down + ((size_t)max(expert, 0) * width + c) * inter + i);
                    b[u] = *reinterpret_cast<const Vec16<T>*>(h_lds + (size_t)s * inter + i);
                }
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    float part = 0.f;
#pragma unroll
                    for (int k = 0; k < V; ++k) part += (float)a[u].v[k] * (float)b[u].v[k];
                    acc = counts[u] ? acc + weight[u] * part : acc;
                }
            }
        } else {
            for (int s = 0; s < top; ++s) {
                int expert = chosen[(size_t)t * top + s];
                if (beside.x && expert >= experts) continue;
                expert = expert < 0 ? 0 : expert >= experts ? experts - 1 : expert;
                const T* row = down + ((size_t)expert * width + c) * inter;
                const T* h = h_lds + (size_t)s * inter;
                float part = 0.f;
                for (int i = lane; i < inter; i += 64) part += (float)row[i] * (float)h[i];
                acc += weights[(size_t)t * top + s] * part;
            }
        }
        if (beside.down) {
            const T* row = beside.down + (size_t)c * beside.inter;
            const T* h = beside.hidden + (size_t)t * beside.inter;
            float part = 0.f;
            if (shared_vectors) {
                for (int i = lane * V; i < beside.inter; i += 64 * V) {
                    const Vec16<T> a = load_vec16(row + i), b = load_vec16(h + i);
#pragma unroll
                    for (int k = 0; k < V; ++k) part += (float)a.v[k] * (float)b.v[k];
                }
            } else {
                for (int i = lane; i < beside.inter; i += 64) part += (float)row[i] * (float)h[i];
            }
            acc += gate * part;
        }
        acc = wave_sum(acc);
        if (lane == 0) {
            if (beside.y) acc += gate * (float)beside.y[(size_t)t * width + c];
            if (beside.x) acc += identity_weight * (float)beside.x[(size_t)t * width + c];
            out[(size_t)t * width + c] = acc;
        }
    }
}

LSA_EXPORT int lsa_route_logits(int code, const void* x, const float* router, float* logits, int n, int experts, int width, hipStream_t stream) {
    if (n <= 0) return 0;
    const dim3 grid(n, (experts + 3) / 4);
    if (code) route_logits_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, router, logits, experts, width);
    else route_logits_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, router, logits, experts, width);
    LSA_LAUNCH_CHECK();
}

// Numbers of the width a part of lsa_route_logits_parts sums over: a wavefront of its four takes a multiple of 32.
static int route_range(int width) {
    const int parts = width >= 512 * ROUTE_PARTS ? ROUTE_PARTS : (width + 511) / 512;
    return ((width + parts - 1) / parts + 127) / 128 * 128;
}

// Partial sums that lsa_route_logits_parts writes for a width, or 0 if it does not take it.
LSA_EXPORT int lsa_route_logits_parts_count(int width) { return width < 8 || width % 8 ? 0 : (width + route_range(width) - 1) / route_range(width); }

LSA_EXPORT int lsa_route_logits_parts(int code, const void* x, const float* router, float* logits, int n, int experts, int width, hipStream_t stream) {
    if (n <= 0) return 0;
    const int parts = lsa_route_logits_parts_count(width);
    if (parts < 1 || experts < 1 || ((size_t)x | (size_t)router) % 16) return -1;
    const dim3 grid((n + 15) / 16, (experts + 15) / 16, parts);
    if (code) route_logits_parts_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, router, logits, n, experts, width, route_range(width));
    else route_logits_parts_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, router, logits, n, experts, width, route_range(width));
    LSA_LAUNCH_CHECK();
}

// scoring 1: the choice is made among sigmoid(logits), which are the weights as they are; groups > 1: only the
// experts of the `keep` best of `groups` equal groups of neighbours can be chosen (at most 64 groups).  scoring 2: see the kernel.
LSA_EXPORT int lsa_route_top(const float* logits, int experts, int top, int* chosen, float* weights, int n, int scoring,
                             int groups, int keep, const float* bias, const float* correction, float weight_scale, int stride, float* gate_out,
                             int parts, hipStream_t stream) {
    if (n <= 0) return 0;
    if (parts < 1 || parts > ROUTE_PARTS) return -1;
    const bool sigmoid_scores = scoring == 1;
    if (scoring < 0 || scoring > 2 || (correction != nullptr && scoring != 2) || stride < experts + (gate_out ? 1 : 0)) return -1;
    if (top < 1 || top > experts || (size_t)experts * 32 > 60000) return -1;
    if (groups > 1 && (!sigmoid_scores || groups > 64 || experts % groups || keep < 1 || keep > groups || top > keep * (experts / groups))) return -1;
    if (experts <= 128 && top <= 64 && groups <= 1 && !(bias != nullptr && correction != nullptr)) {
#define LSA_TOP(E, P) route_top_registers_kernel<E, P><<<n, 64, 0, stream>>>(logits, experts, top, chosen, weights, n, scoring, bias, correction, weight_scale, stride, gate_out, parts)
        if (experts <= 64) { if (parts > 1) LSA_TOP(1, true); else LSA_TOP(1, false); }
        else if (parts > 1) LSA_TOP(2, true);
        else LSA_TOP(2, false);
#undef LSA_TOP
        LSA_LAUNCH_CHECK();
    }
    route_top_kernel<<<(n + 3) / 4, 256, (size_t)experts * 8 * sizeof(float), stream>>>(logits, experts, top, chosen, weights, n,
                                                                                       scoring, groups, keep, bias, correction, weight_scale, stride, gate_out, parts);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_experts_gate_up(int code, const void* x, const void* gate_up, const int* chosen, void* hidden, int n, int top,
                                   int inter, int width, int experts, float limit, int identity, const void* shared_gate_up,
                                   void* shared_hidden, int shared_inter, int plain, hipStream_t stream) {
    if (n <= 0) return 0;
    if (shared_gate_up != nullptr && (shared_hidden == nullptr || shared_inter < 1)) return -1;
    const int most_inter = shared_gate_up && shared_inter > inter ? shared_inter : inter;
    size_t lds = (size_t)width * (code ? 2 : 4);
    const bool in_lds = lds <= 64000;
    if (!in_lds) lds = 0;
    const int columns = 16;
    dim3 grid;
    if (!shared_grid(n > 1, (long)n * (top + (shared_gate_up ? 1 : 0)), (most_inter + columns - 1) / columns, grid)) return -1;
    if (code) experts_gate_up_kernel<bf16_t><<<grid, 256, lds, stream>>>((const bf16_t*)x, (const bf16_t*)gate_up, chosen, (bf16_t*)hidden, top, inter, width, experts, columns, in_lds, limit, identity, (const bf16_t*)shared_gate_up, (bf16_t*)shared_hidden, shared_inter, plain, n > 1);
    else experts_gate_up_kernel<float><<<grid, 256, lds, stream>>>((const float*)x, (const float*)gate_up, chosen, (float*)hidden, top, inter, width, experts, columns, in_lds, limit, identity, (const float*)shared_gate_up, (float*)shared_hidden, shared_inter, plain, n > 1);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_experts_down(int code, const void* hidden, const void* down, const int* chosen, const float* weights, float* out,
                                int n, int top, int inter, int width, int experts, const void* x, const float* shared_gate, const void* shared_y,
                                const void* shared_down, const void* shared_hidden, int shared_inter, hipStream_t stream) {
    if (n <= 0) return 0;
    if ((shared_gate != nullptr && shared_y == nullptr && shared_down == nullptr) || (shared_down != nullptr && shared_hidden == nullptr)) return -1;
    // (a block takes four columns: staging the token's hidden rows in LDS would cost as much as it reads of the weights)
    const size_t lds = 0;
    const bool in_lds = false;
    const int columns = 4;
    dim3 grid;
    if (!shared_grid(n > 1, n, (width + columns - 1) / columns, grid)) return -1;
#define LSA_BESIDE(T) BesideExperts<T>{(const T*)x, shared_gate, (const T*)shared_y, (const T*)shared_down, (const T*)shared_hidden, shared_inter}
    // (trips of a lane: in fours or threes, whichever leaves fewer behind the last piece; a handful one by one)
    const int trips = (int)(((size_t)top * inter / (code ? 8 : 4) + 63) / 64), ahead = trips < 3 ? 1 : trips % 4 == 0 ? 4 : 3;
#define LSA_DOWN(T, AHEAD) experts_down_kernel<T, AHEAD><<<grid, 256, lds, stream>>>((const T*)hidden, (const T*)down, chosen, weights, out, top, inter, width, experts, columns, in_lds, LSA_BESIDE(T), n > 1)
    if (code && ahead == 4) LSA_DOWN(bf16_t, 4);
    else if (code && ahead == 3) LSA_DOWN(bf16_t, 3);
    else if (code) LSA_DOWN(bf16_t, 1);
    else if (ahead == 4) LSA_DOWN(float, 4);
    else if (ahead == 3) LSA_DOWN(float, 3);
    else LSA_DOWN(float, 1);
#undef LSA_DOWN
#undef LSA_BESIDE
    LSA_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------------------------------------
// Many tokens (portions of prompts, large batches): the pairs are sorted by expert, each expert's pairs padded to whole
// tiles of TILE_M rows, and one MFMA product per tile multiplies the tile's rows with its expert's matrix, so an expert's
// weights are read once per tile of 64 pairs instead of once per pair.  bfloat16 only (the float32 path keeps the
// kernels above).
//
// sort: one workgroup.  sorted[i] = pair at padded place i (-1: padding), tiles[j] = {expert of tile j, the expert's first tile and number of tiles},
// tiles[max_tiles].expert the number of tiles; places and tiles behind the last one are not written.  The order of an expert's pairs among themselves is whatever the atomics
// give; every pair's row is computed on its own, so the results do not depend on it.  The choices are read four a
// thread at a time; an expert's first place is a sum over 64 lanes and not a walk by one thread (12,288 pairs of 64 experts: 20.7 -> 11.7
// us; 32,760 pairs: 43 -> 24 us; 192 pairs: 8.8 -> 4.6 us).
constexpr int TILE_M = 64, WIDE_M = WIDE_TILE;                        // pairs a tile: see below
struct Tile { int expert, first, count; };

__global__ __launch_bounds__(1024) void experts_sort_kernel(const int* __restrict__ chosen, int n_pairs, int experts, int tile_rows,
                                                            int* __restrict__ sorted, Tile* __restrict__ tiles_of, int max_tiles) {
    extern __shared__ int lds_ints[];
    int* counts = lds_ints;
    int* offsets = lds_ints + experts;
    const int tid = threadIdx.x;
    for (int e = tid; e < experts; e += 1024) counts[e] = 0;
    __syncthreads();
    for (int p0 = 0; p0 < n_pairs; p0 += 4096) {
        int e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = chosen[min(p0 + 1024 * u + tid, n_pairs - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (p0 + 1024 * u + tid < n_pairs && e[u] >= 0 && e[u] < experts) atomicAdd(&counts[e[u]], 1);
    }
    __syncthreads();
    if (tid < 64) {
        int running = 0;                         // tiles in front of these 64 experts
        for (int e0 = 0; e0 < experts; e0 += 64) {
            const int e = e0 + tid, mine = e < experts ? (counts[e] + tile_rows - 1) / tile_rows : 0;
            int sum = mine;
#pragma unroll
            for (int step = 1; step < 64; step <<= 1) {
                const int other = __shfl_up(sum, step, 64);
                if (tid >= step) sum += other;
            }
            if (e < experts) offsets[e] = running + sum - mine;
            running += __shfl(sum, 63, 64);
        }
        if (tid == 0) tiles_of[max_tiles].expert = running;
    }
    __syncthreads();
    for (int e = tid >> 4; e < experts; e += 64) {               // sixteen threads an expert: its tiles, and the places behind its last pair
        const int count = counts[e], first = offsets[e], tiles = (count + tile_rows - 1) / tile_rows;
        for (int j = tid & 15; j < tiles; j += 16) tiles_of[first + j] = Tile{e, first, tiles};
        for (int i = count + (tid & 15); i < tiles * tile_rows; i += 16) sorted[first * tile_rows + i] = -1;
    }
    __syncthreads();
    for (int e = tid; e < experts; e += 1024) offsets[e] *= tile_rows;       // from here on: the next pair's place
    __syncthreads();
    for (int p0 = 0; p0 < n_pairs; p0 += 4096) {
        int e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = chosen[min(p0 + 1024 * u + tid, n_pairs - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int p = p0 + 1024 * u + tid;
            if (p < n_pairs && e[u] >= 0 && e[u] < experts) sorted[atomicAdd(&offsets[e[u]], 1)] = p;
        }
    }
}


// C = A . B^T for one tile of 64 sorted pairs and 128 rows of the expert's matrix (K contiguous in both).
// FORM 0: the products themselves.  FORM 2: max(product, 0)^2.  FORM 1 is GATED:
//   GATED: B's 128 rows are 64 gate rows f0 .. f0 + 63 and their 64 up rows; the result is silu(gate) * up, 64 columns.
//   Rows of A: a[(sorted[i] / pair_div)] (pair_div = top for the tokens' rows, 1 for the pairs' hidden rows).
// Four wavefronts, each 32 rows x 16 NT columns (GATED: half of them gate columns, half their up columns): 2 x NT MFMA
// tiles of 16 x 16, k in steps of 32.  A slab of BK columns of K of both operands goes through LDS (rows padded by 16
// bytes).  NT = 4 where an expert has few pairs (its weights bound the time), 8 where it has many (every operand read
// from LDS then feeds more products, which is what bounds a tile of 4).
template <int BK, int FORM, typename O, int NT>
__global__ __launch_bounds__(256) void experts_tile_kernel(const bf16_t* __restrict__ a, int a_stride, int pair_div,
                                                           const bf16_t* __restrict__ b, long expert_stride, int b_rows, int b_up_offset,
                                                           const int* __restrict__ sorted, const Tile* __restrict__ tiles_of,
                                                           O* __restrict__ out, int out_stride, int n_out, int k, float limit) {
    constexpr bool GATED = FORM == 1;
    constexpr int ROW = BK + 8;                                    // elements of a padded row in LDS
    __shared__ __align__(16) bf16_t a_lds[TILE_M * ROW];
    constexpr int BN = 32 * NT;                                    // rows of B a block takes
    __shared__ __align__(16) bf16_t b_lds[BN * ROW];
    __shared__ int rows_of[TILE_M];
    // Workgroups go to the eight XCDs in turn by their number.  The tiles of one expert stand next to each other in the
    // list; numbered so that neighbours in the list get numbers eight apart, they run on one XCD at about the same time
    // and the expert's rows are fetched into one L2 instead of several.
    const int total = gridDim.x * gridDim.y, number = blockIdx.y * gridDim.x + blockIdx.x, share = total / 8;
    const int place = number < share * 8 ? (number % 8) * share + number / 8 : number;
    const int tile = place % gridDim.x, block_n = place / gridDim.x;
    if (tile >= tiles_of[gridDim.x].expert) return;
    const int expert = tiles_of[tile].expert;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, quad = lane >> 4;
    const int wave_m = wave >> 1, wave_n = wave & 1;
    if (threadIdx.x < TILE_M) rows_of[threadIdx.x] = sorted[tile * TILE_M + threadIdx.x];
    __syncthreads();
    const int n0 = block_n * (GATED ? BN / 2 : BN);                // first output column of the block
    const bf16_t* bm = b + (size_t)expert * expert_stride;
    // which rows of B the block's LDS rows are: GATED: the first half gate rows n0 + r, the second half their up rows
    auto b_row = [&](int r) {
        int row = GATED ? (r < BN / 2 ? n0 + r : b_up_offset + n0 + r - BN / 2) : n0 + r;
        const int last = GATED ? (r < BN / 2 ? n_out - 1 : b_up_offset + n_out - 1) : n_out - 1;
        return row > last ? last : row;                            // (columns beyond the matrix repeat its last row; never stored)
    };
    f32x4 acc[2][NT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int PIECES = BK / 8;                                 // 16-byte pieces of a row of a slab
    constexpr int A_LOADS = TILE_M * PIECES / 256, B_LOADS = BN * PIECES / 256;      // 16-byte loads of a thread per slab
    // A thread's pieces of a slab: the same rows and places in every slab, so their addresses are made once.  The next
    // slab's pieces travel into registers while this slab is multiplied, and go to LDS when everybody is through with it.
    const bf16_t* a_src[A_LOADS];
    const bf16_t* b_src[B_LOADS];
    int a_dst[A_LOADS], b_dst[B_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u) {
        const int i = threadIdx.x + 256 * u, r = i / PIECES, piece = i - r * PIECES;
        const int pair = rows_of[r];
        a_src[u] = a + (size_t)(pair < 0 ? 0 : pair / pair_div) * a_stride + 8 * piece;
        a_dst[u] = r * ROW + 8 * piece;
    }
#pragma unroll
    for (int u = 0; u < B_LOADS; ++u) {
        const int i = threadIdx.x + 256 * u, r = i / PIECES, piece = i - r * PIECES;
        b_src[u] = bm + (size_t)b_row(r) * k + 8 * piece;
        b_dst[u] = r * ROW + 8 * piece;
    }
    bf16x8 a_next[A_LOADS], b_next[B_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u) a_next[u] = *reinterpret_cast<const bf16x8*>(a_src[u]);
#pragma unroll
    for (int u = 0; u < B_LOADS; ++u) b_next[u] = *reinterpret_cast<const bf16x8*>(b_src[u]);
    for (int k0 = 0; k0 < k; k0 += BK) {
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) *reinterpret_cast<bf16x8*>(a_lds + a_dst[u]) = a_next[u];
#pragma unroll
        for (int u = 0; u < B_LOADS; ++u) *reinterpret_cast<bf16x8*>(b_lds + b_dst[u]) = b_next[u];
        __syncthreads();
        if (k0 + BK < k) {
#pragma unroll
            for (int u = 0; u < A_LOADS; ++u) a_next[u] = *reinterpret_cast<const bf16x8*>(a_src[u] + k0 + BK);
#pragma unroll
            for (int u = 0; u < B_LOADS; ++u) b_next[u] = *reinterpret_cast<const bf16x8*>(b_src[u] + k0 + BK);
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            bf16x8 av[2], bv[NT];
#pragma unroll
            for (int i = 0; i < 2; ++i) av[i] = *reinterpret_cast<const bf16x8*>(a_lds + (wave_m * 32 + 16 * i + col) * ROW + kk + 8 * quad);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                // GATED: the first half of a wavefront's tiles are its gate columns, the second half their up columns
                const int r = GATED ? (j < NT / 2 ? wave_n * (BN / 4) + 16 * j : BN / 2 + wave_n * (BN / 4) + 16 * (j - NT / 2))
                                    : wave_n * (BN / 2) + 16 * j;
                bv[j] = *reinterpret_cast<const bf16x8*>(b_lds + (r + col) * ROW + kk + 8 * quad);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // lane holds rows 4 * quad + r of each 16 x 16 tile, column col
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int pair = rows_of[wave_m * 32 + 16 * i + 4 * quad + r];
            if (pair < 0) continue;
            O* o = out + (size_t)pair * out_stride;
            if (GATED) {
#pragma unroll
                for (int j = 0; j < NT / 2; ++j) {
                    const int f = n0 + wave_n * (BN / 4) + 16 * j + col;
                    const float g = acc[i][j][r], u = acc[i][j + NT / 2][r];
                    if (f < n_out) o[f] = (O)gated_activation(g, u, limit);
                }
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int c = n0 + wave_n * (BN / 2) + 16 * j + col;
                    if (c < n_out) o[c] = (O)(FORM == 2 ? rectified_square(acc[i][j][r]) : acc[i][j][r]);
                }
            }
        }
}

// ---- few pairs an expert ----------------------------------------------------------------------------------------------------
// C = A . B^T as above for tiles of 64 sorted pairs and 128 rows of the expert's matrix (GATED: for each 32 of them sixteen gate rows and their up rows), where k
// is a multiple of 64 and all rows begin at multiples of 16 bytes: eight wavefronts of 32 x 32, slabs of 64 of k through three buffers of LDS that loads fill
// without registers, two workgroups a compute unit.  Rows and columns of padding are neither loaded nor multiplied.
//   What bounds it is the experts' way from memory, which those loads keep fuller than the tiles above do with a slab in registers: 32 tokens, 6 of 64 experts of 1,408 at
// width 2,048 (56 of them chosen), all launches 213 -> 193 us (5.3 TB/s in the two products); 330 tokens 268 -> 246; 8 experts, 100 tokens 87 -> 56; 16 of 768, 64 tokens
// 77 -> 51; 32 of 2,048 at 4,096, 250 tokens 449 -> 360.  No faster: tiles of 64 or 256 rows of the matrix, four wavefronts, 32 rows of pairs, four to six buffers.
constexpr int STREAM_ROWS = 128, STREAM_BUFFERS = 3, STREAM_THREADS = 512;
template <int FORM, typename O>
__global__ __launch_bounds__(STREAM_THREADS) void experts_stream_kernel(const bf16_t* __restrict__ a, int a_stride, int pair_div, const bf16_t* __restrict__ b,
                                                                        long expert_stride, int b_up_offset, const int* __restrict__ sorted,
                                                                        const Tile* __restrict__ tiles_of, int max_tiles, O* __restrict__ out, int out_stride, int n_out,
                                                                        int k, float limit, int blocks) {
    constexpr bool GATED = FORM == 1;
    constexpr int COLUMNS = GATED ? STREAM_ROWS / 2 : STREAM_ROWS, SLAB = 64, BUFFER = (TILE_M + STREAM_ROWS) * SLAB * 2;
    __shared__ __attribute__((aligned(1024))) unsigned char buffers[STREAM_BUFFERS * BUFFER];
    __shared__ int rows_of[TILE_M];
    // Workgroups go to the eight XCDs in turn by their number (there are a multiple of eight): an XCD has neighbours of an order that walks the list of tiles for one
    // block of columns after the other, so that an expert's tiles run on one XCD at about the same time and its rows are fetched into one L2.
    const int place = (int)(blockIdx.x % XCDS) * (int)(gridDim.x / XCDS) + (int)(blockIdx.x / XCDS), tile = place % max_tiles, block_n = place / max_tiles;
    if (block_n >= blocks || tile >= tiles_of[max_tiles].expert) return;
    const int expert = tiles_of[tile].expert;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), col = lane & 15, quad = lane >> 4;
    const int wave_m = wave >> 2, wave_n = wave & 3, n0 = block_n * COLUMNS;
    if (threadIdx.x < TILE_M) rows_of[threadIdx.x] = sorted[tile * TILE_M + threadIdx.x];
    __syncthreads();
    // A load of a wavefront is 8 rows: wavefront w's are rows 8 w on of A, 8 w and 64 + 8 w on of B.  The eight 16-byte pieces of row r stand at places
    // piece ^ f(r), so that sixteen lanes whose reads are served together meet all 64 banks (wide_product.hpp).
    const buffer_t a_buffer = buffer_at(a), b_buffer = buffer_at(b + (size_t)expert * expert_stride);
    const int line = 8 * wave + (lane >> 3), pair = rows_of[line];
    const unsigned a_at = pair < 0 ? NOWHERE : 2u * ((unsigned)(pair / pair_div) * (unsigned)a_stride) + 16 * ((lane & 7) ^ (line >> 1 & 7));
    unsigned b_at[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int r = 64 * u + line, c = n0 + (GATED ? 16 * (r >> 5) + (r & 15) : r);
        b_at[u] = c >= n_out ? NOWHERE : 2u * ((unsigned)(c + (GATED && (r & 16) ? b_up_offset : 0)) * (unsigned)k)
                                             + 16 * ((lane & 7) ^ (GATED ? r >> 1 & 7 : (r >> 1 & 1) | (r >> 3 & 3) << 1));
    }
    const int slabs = k / SLAB;
    unsigned landing = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(lds_ptr_t)buffers) + 1024 * wave;
    int asked = 0;
    auto ask = [&]() __attribute__((always_inline)) {
        const unsigned from = min(asked, slabs - 1) * (2 * SLAB);  // (behind the last slab: that once more, into a buffer that nobody reads again)
        load_16_bytes_a_lane_to_lds(a_buffer, a_at, from, landing);
#pragma unroll
        for (int u = 0; u < 2; ++u) load_16_bytes_a_lane_to_lds(b_buffer, b_at[u], from, landing + 8192 * (1 + u));
        ++asked;
        landing += asked % STREAM_BUFFERS == 0 ? -(STREAM_BUFFERS - 1) * BUFFER : BUFFER;
    };
    f32x4 sums[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) sums[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int pieces[2] = {16 * (quad ^ (col >> 1)), 16 * ((quad + 4) ^ (col >> 1))};
    const unsigned char* a_rows = buffers + (32 * wave_m + col) * 128;
    const unsigned char* b_rows = buffers + (TILE_M + 32 * wave_n + (GATED ? col : 8 * (col >> 2) + (col & 3))) * 128;
    constexpr int B_STEP = (GATED ? 16 : 4) * 128;                 // (not GATED: a lane has eight neighbouring columns of the result)
    const int used = __builtin_amdgcn_readfirstlane((rows_of[32 * wave_m] >= 0) + (rows_of[32 * wave_m + 16] >= 0));      // rows of MFMA tiles that hold pairs
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (the count below starts from nothing under way)
#pragma unroll
    for (int i = 0; i < STREAM_BUFFERS - 1; ++i) ask();
    int buffer = 0;
    for (int slab = 0; slab < slabs; ++slab) {
        loads_landed_then_barrier<3 * (STREAM_BUFFERS - 2)>();     // and everybody is through with the slab before this one, whose buffer is asked for
        bf16x8 av[2][2], bv[2][2];
        if (used)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    if (i < used) av[s][i] = *reinterpret_cast<const bf16x8*>(a_rows + buffer + 2048 * i + pieces[s]);
#pragma unroll
                for (int j = 0; j < 2; ++j) bv[s][j] = *reinterpret_cast<const bf16x8*>(b_rows + buffer + B_STEP * j + pieces[s]);
            }
        __builtin_amdgcn_sched_barrier(0);
        ask();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (i < used)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int j = 0; j < 2; ++j) sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[s][j], av[s][i], sums[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        buffer = buffer == (STREAM_BUFFERS - 1) * BUFFER ? 0 : buffer + BUFFER;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (no load may land when this LDS is somebody else's)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int of = rows_of[32 * wave_m + 16 * i + col], n = n0 + (GATED ? 16 * wave_n + 4 * quad : 32 * wave_n + 8 * quad);
        if (of < 0 || n >= n_out) continue;                        // (n_out is a multiple of 32)
        O* o = out + (size_t)of * out_stride + n;
        if (GATED) {
            struct alignas(4 * sizeof(O)) Four { O v[4]; } four;
#pragma unroll
            for (int r = 0; r < 4; ++r) four.v[r] = (O)gated_activation(sums[i][0][r], sums[i][1][r], limit);
            *reinterpret_cast<Four*>(o) = four;
        } else {
            struct alignas(16) Eight { O v[8]; } eight;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const float z = sums[i][r >> 2][r & 3];
                eight.v[r] = (O)(FORM == 2 ? rectified_square(z) : z);
            }
            *reinterpret_cast<Eight*>(o) = eight;
        }
    }
}

// ---- many pairs an expert ---------------------------------------------------------------------------------------------------
// C = A . B^T as above for tiles of 256 sorted pairs and 256 rows of the expert's matrix (GATED: 128 gate rows and their up rows, 128 columns of the result).
//   What bounds it is what passes between the XCDs' L2 and the memory side: a workgroup's share of an expert's matrix is read once for each 256 of its pairs and
// half of that comes from the neighbour's read.  12,288 pairs of 64 gated experts of 1,408 at width 2,048, chosen unevenly, us a launch, first and second product, with sixteen
// wavefronts of 64 x 64 in step and now: 251 + 143, 224 + 138 (191 of them the matrices' loads alone); 32,760 pairs of 2,112 without gates, all launches 808, 710; with the same
// number of pairs everywhere and experts of 2,048 230 for the first product (1.19 PFLOP/s).  (Of few slabs it is the slower one, by its start: 16 experts of 352 at 512, 4,096 tokens, all
// launches 65.9, 68.1.)  No faster: one workgroup a compute unit that goes from tile to tile with its loads running on;
// shares of the XCDs by work; slabs in another order for each block of columns; the experts' pairs shared evenly by its tiles; three slabs of the matrix in LDS.
template <int FORM, typename O>
__global__ __launch_bounds__(WIDE_THREADS) void experts_wide_kernel(const bf16_t* __restrict__ a, int a_stride, int pair_div,
                                                           const bf16_t* __restrict__ b, long expert_stride, int b_up_offset,
                                                           const int* __restrict__ sorted, const Tile* __restrict__ tiles_of, int max_tiles,
                                                           O* __restrict__ out, int out_stride, int n_out, int k, float limit, int blocks) {
    constexpr bool GATED = FORM == 1;
    constexpr int COLUMNS = GATED ? WIDE_TILE / 2 : WIDE_TILE;     // output columns of a workgroup
    __shared__ __attribute__((aligned(1024))) unsigned char buffers[2 * WIDE_BUFFER];
    __shared__ int rows_of[WIDE_TILE];
    // Workgroups go to the eight XCDs in turn by their number: an XCD gets an eighth of the tiles and walks one expert's (at most
    // eight) through all blocks of columns, so that their rows stay in its L2 while the expert's matrix comes into it once.  What passes
    // between L2 and memory: 1.1 GB for 32,760 pairs of 64 experts of 2,112 at width 2,048, 1.5 with groups of four tiles whatever their experts.
    const int tiles = tiles_of[max_tiles].expert, share = (tiles + 7) / 8, begin = (int)(blockIdx.x % 8) * share, end = min(begin + share, tiles);
    const int index = blockIdx.x / 8, slot = begin + index / blocks;
    if (slot >= end) return;
    const Tile of = tiles_of[slot];
    const int within = (slot - of.first) & ~7;                     // (the expert's tiles eight at a time)
    const int group = max(begin, of.first + within), group_tiles = min(min(end, of.first + of.count), of.first + within + 8) - group;
    const int in_group = index - (group - begin) * blocks;
    const int block_n = in_group / group_tiles, tile = group + in_group % group_tiles;
    const int expert = of.expert;
    if (threadIdx.x < WIDE_TILE) rows_of[threadIdx.x] = sorted[tile * WIDE_TILE + threadIdx.x];
    __syncthreads();
    const int n0 = block_n * COLUMNS;
    auto a_offset = [&](int r) __attribute__((always_inline)) {
        const int pair = rows_of[r];                               // (padding stands behind the expert's last pair)
        return pair < 0 ? NOWHERE : 2u * ((unsigned)(pair / pair_div) * (unsigned)a_stride);
    };
    auto b_offset = [&](int r) __attribute__((always_inline)) {
        const int column = n0 + (GATED ? r & (WIDE_TILE / 2 - 1) : r);
        return column >= n_out ? NOWHERE : 2u * ((unsigned)(column + (GATED && r >= WIDE_TILE / 2 ? b_up_offset : 0)) * (unsigned)k);
    };
    const int row_blocks = 1 + (rows_of[64] >= 0) + (rows_of[128] >= 0) + (rows_of[192] >= 0);
    WideSums sums;
    wide_product(sums, buffers, a, a_offset, b + (size_t)expert * expert_stride, b_offset, k, __builtin_amdgcn_readfirstlane(row_blocks),
                 GATED || n0 + WIDE_TILE / 2 < n_out);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int pair = rows_of[wide_row(half, i, wave, lane)];
            if (pair < 0) continue;
            O* o = out + (size_t)pair * out_stride + n0;
#pragma unroll
            for (int other = 0; other < (GATED ? 1 : 2); ++other) {
                const int c = wide_column(other, wave, lane);
                if (n0 + c >= n_out) continue;                     // (n_out is a multiple of 32)
                struct alignas(16) Eight { O v[8]; } eight;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float z = sums[half][other][i][j][r];
                        eight.v[4 * j + r] = (O)(GATED ? gated_activation(z, sums[half][1][i][j][r], limit) : FORM == 2 ? rectified_square(z) : z);
                    }
                *reinterpret_cast<Eight*>(o + c) = eight;
            }
        }
}

// out[t][c] = sum_s weights[t][s] * y[t * top + s][c]; with `beside`: identity experts (choices from `experts` on) put the token's
// row in place of y, and the shared expert's output joins times the token's gate.  grid (tokens, blocks of 256 V columns), a
// thread has V neighbouring columns of one token.
template <int V>
__global__ __launch_bounds__(256) void experts_combine_kernel(const float* __restrict__ y, const float* __restrict__ weights,
                                                              float* __restrict__ out, int top, int width, const int* __restrict__ chosen,
                                                              int experts, BesideExperts<bf16_t> beside) {
    struct alignas(4 * V) Floats { float v[V]; };
    struct alignas(2 * V) Halves { bf16_t v[V]; };
    const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * V;
    if (c >= width) return;
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.f;
    if (beside.y) {
        const Halves h = *reinterpret_cast<const Halves*>(beside.y + (size_t)t * width + c);
        const float gate = beside.gate ? beside.gate[t] : 1.f;
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = gate * (float)h.v[v];
    }
    float identity_weight = 0.f;
#pragma unroll 4
    for (int s = 0; s < top; ++s) {                          // (choice and weight are the same for the whole workgroup)
        const float weight = weights[(size_t)t * top + s];
        if (beside.x && chosen[(size_t)t * top + s] >= experts) {
            identity_weight += weight;
            continue;
        }
        const Floats f = *reinterpret_cast<const Floats*>(y + ((size_t)t * top + s) * width + c);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += weight * f.v[v];
    }
    if (beside.x) {
        const Halves h = *reinterpret_cast<const Halves*>(beside.x + (size_t)t * width + c);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] += identity_weight * (float)h.v[v];
    }
    Floats result;
#pragma unroll
    for (int v = 0; v < V; ++v) result.v[v] = acc[v];
    *reinterpret_cast<Floats*>(out + (size_t)t * width + c) = result;
}

// Whether loads straight into LDS can multiply such a step (the wide kernel's and those of few pairs an expert): they are of 16 bytes at multiples of 16 (`aligned`: x, gate_up and down
// begin at such), from offsets of 32 bits.
static bool wide_fits(int pairs, int inter, int width, bool aligned) {
    return aligned && (size_t)pairs * (size_t)(inter > width ? inter : width) * 2 < BUFFER_BYTES && (size_t)2 * inter * width * 2 < BUFFER_BYTES;
}

// Pairs a tile that lsa_experts_tiled should take for a step with so many pairs: 256 (the wide kernel) or 64.  The line: some 40 pairs an
// expert, and the two products make 224 workgroups or more together, not quite one a compute unit for each: with fewer, tiles of 64 pairs spread the same work over units that
// would stand idle.  All launches of a step, us, narrow and wide, pairs chosen unevenly: 64 experts of 1,408 at width 2,048, 40 pairs an expert 254, 247; 64: 277, 280; 96: 323, 307;
// 128: 377, 343; 192: 477, 400; 128 of 768 at 2,048, 40 pairs 274, 267; 32 of 2,048 at 4,096 (1,024 workgroups) 356, 336; 16 of them (512) 196, 203, 128 pairs 285, 298, 192: 361, 320;
// 8 (256), 128 pairs 157, 154; 4 (128) 79, 131, with 192 pairs 93, 138; 8 of 1,408 at 2,048 (152) with 192 pairs 75, 97; 4 (76) 47, 90; 1 of 512 at 1,024 (8) with 256 pairs 26,
// 58.  (Behind the line there are steps that the narrow tiles, since their matrices go through LDS without registers, would make faster: 16 of 768 at 2,048 (224) with 128 pairs
// 64, 87; without gates, 16 of 1,024 at 4,096 (320) with 128 pairs 125, 155.)
//   Inner dimensions below 512 are so few slabs that a wide launch is mostly its start: 64 of 256 at 1,024, 40 pairs 43, 59; 128: 67, 76; 200: 87, 89; 256: 101, 95.
LSA_EXPORT int lsa_experts_tile_rows(int pairs, int experts, int inter, int width, int plain, int aligned) {
    if (pairs < (inter < 512 || width < 512 ? 200 : 40) * experts || !wide_fits(pairs, inter, width, aligned != 0)) return TILE_M;
    const long tiles = (long)experts * ((pairs / experts + WIDE_M - 1) / WIDE_M), columns = plain ? WIDE_TILE : WIDE_TILE / 2;
    return tiles * ((inter + columns - 1) / columns) + tiles * ((width + WIDE_TILE - 1) / WIDE_TILE) >= 224 ? WIDE_M : TILE_M;
}

// Whether the product of few pairs an expert goes to experts_stream_kernel.  Two of its workgroups a compute unit are 512, and where the experts that so many pairs can be
// expected to choose make little more than that, the second round is nearly empty; the tiles above, five a compute unit, are then as fast or faster: 32 experts of
// 2,048 at 4,096, first product, at 12, 16, 24 and 32 tokens (21, 25, 27 and 29 chosen, 32 blocks each) 152, 169, 183, 192 us and 169, 178, 189, 190; 96 of 512 at 1,024, 32
// tokens (69 chosen, 8 blocks) 31.2 and 32.9.  With shorter rows it pays earlier (64 of 1,408 at 2,048, 36 chosen, 22 blocks: 145, 135 for all launches).
static bool stream_pays(int pairs, int experts, int blocks, int k) {
    const double chosen = experts * (1.0 - exp(-(double)pairs / experts)), rounds = chosen * blocks / 512;
    return rounds <= 1.0 || rounds >= (k > 3072 ? 1.85 : 1.3);
}

// Ints of scratch memory that lsa_experts_tiled wants: the sorted pairs, then the tiles and their number.
LSA_EXPORT int lsa_experts_tiled_ints(int pairs, int experts, int tile_rows) { return ((pairs + tile_rows - 1) / tile_rows + experts) * (tile_rows + 3) + 3; }

// Sorted, tiled products for bfloat16: hidden = silu(G x) * (U x) and y = D hidden for all pairs, then the weighted sums.
// Scratch: lsa_experts_tiled_ints ints, y [pairs, width] floats.  tile_rows: 64 or, where the wide kernel can, 256.
LSA_EXPORT int lsa_experts_tiled(const void* x, const void* gate_up, const void* down, const int* chosen, const float* weights,
                                 void* hidden, float* y, float* out, int* scratch, int tile_rows, int n, int top,
                                 int inter, int width, int experts, float limit, int identity, const float* shared_gate, const void* shared_y,
                                 int plain, hipStream_t stream) {
    if (n <= 0) return 0;
    if (shared_gate != nullptr && shared_y == nullptr) return -1;
    const int pairs = n * top;
    if (width % 32 || inter % 32 || (size_t)experts * 8 > 60000) return -1;
    const bool wide = tile_rows == WIDE_M;
    if (!wide && tile_rows != TILE_M) return -1;
    const bool whole_pieces = wide_fits(pairs, inter, width, ((size_t)x | (size_t)gate_up | (size_t)down | (size_t)hidden) % 16 == 0);
    if (wide && !whole_pieces) return -1;
    const int max_tiles = (pairs + tile_rows - 1) / tile_rows + experts;
    int* sorted = scratch;
    Tile* tiles_of = reinterpret_cast<Tile*>(scratch + (size_t)max_tiles * tile_rows);
    experts_sort_kernel<<<1, 1024, (size_t)experts * 2 * sizeof(int), stream>>>(chosen, pairs, experts, tile_rows, sorted, tiles_of, max_tiles);
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* gu = (const bf16_t*)gate_up;
    const bf16_t* dn = (const bf16_t*)down;
    bf16_t* hb = (bf16_t*)hidden;
    if (wide) {
        const int gated_blocks = (inter + WIDE_TILE / 2 - 1) / (WIDE_TILE / 2), plain_blocks = (inter + WIDE_TILE - 1) / WIDE_TILE, down_blocks = (width + WIDE_TILE - 1) / WIDE_TILE;
        const int numbers = 8 * ((max_tiles + 7) / 8);
        if (plain)
            experts_wide_kernel<2, bf16_t><<<numbers * plain_blocks, WIDE_THREADS, 0, stream>>>(xb, width, top, gu, (long)inter * width, 0, sorted, tiles_of, max_tiles, hb,
                                                                                       inter, inter, width, 0.f, plain_blocks);
        else
            experts_wide_kernel<1, bf16_t><<<numbers * gated_blocks, WIDE_THREADS, 0, stream>>>(xb, width, top, gu, (long)2 * inter * width, inter, sorted, tiles_of,
                                                                                       max_tiles, hb, inter, inter, width, limit, gated_blocks);
        experts_wide_kernel<0, float><<<numbers * down_blocks, WIDE_THREADS, 0, stream>>>(hb, inter, 1, dn, (long)width * inter, 0, sorted, tiles_of, max_tiles, y, width,
                                                                                 width, inter, 0.f, down_blocks);
    } else {
        const bool many = pairs >= 16 * experts;                // pairs to an expert: wide tiles pay
#define LSA_TILES(BK, NT) do { \
        dim3 grid1(max_tiles, (inter + 16 * NT - 1) / (16 * NT)), gridp(max_tiles, (inter + 32 * NT - 1) / (32 * NT)), grid2(max_tiles, (width + 32 * NT - 1) / (32 * NT)); \
        if (!second && plain) experts_tile_kernel<BK, 2, bf16_t, NT><<<gridp, 256, 0, stream>>>(xb, width, top, gu, (long)inter * width, inter, 0, sorted, tiles_of, hb, inter, inter, width, 0.f); \
        else if (!second) experts_tile_kernel<BK, 1, bf16_t, NT><<<grid1, 256, 0, stream>>>(xb, width, top, gu, (long)2 * inter * width, 2 * inter, inter, sorted, tiles_of, hb, inter, inter, width, limit); \
        else experts_tile_kernel<BK, 0, float, NT><<<grid2, 256, 0, stream>>>(hb, inter, 1, dn, (long)width * inter, width, 0, sorted, tiles_of, y, width, width, inter, 0.f); \
    } while (0)
        for (int pass = 0; pass < 2; ++pass) {
            const bool second = pass == 1;
            const bool wide_slab = (second ? inter : width) % 64 == 0;
            const int k = second ? inter : width, columns = second ? width : inter, block = second || plain ? STREAM_ROWS : STREAM_ROWS / 2;
            const int blocks = (columns + block - 1) / block;
            const long grid = ((long)max_tiles * blocks + XCDS - 1) / XCDS * XCDS;
            if (whole_pieces && wide_slab && grid < (1 << 23) && stream_pays(pairs, experts, blocks, k)) {
                if (second) experts_stream_kernel<0, float><<<(int)grid, STREAM_THREADS, 0, stream>>>(hb, inter, 1, dn, (long)width * inter, 0, sorted, tiles_of, max_tiles, y, width, width, inter, 0.f, blocks);
                else if (plain) experts_stream_kernel<2, bf16_t><<<(int)grid, STREAM_THREADS, 0, stream>>>(xb, width, top, gu, (long)inter * width, 0, sorted, tiles_of, max_tiles, hb, inter, inter, width, 0.f, blocks);
                else experts_stream_kernel<1, bf16_t><<<(int)grid, STREAM_THREADS, 0, stream>>>(xb, width, top, gu, (long)2 * inter * width, inter, sorted, tiles_of, max_tiles, hb, inter, inter, width, limit, blocks);
            } else
            if (wide_slab && many) LSA_TILES(64, 8);
            else if (wide_slab) LSA_TILES(64, 4);
            else if (many) LSA_TILES(32, 8);
            else LSA_TILES(32, 4);
        }
#undef LSA_TILES
    }
    experts_combine_kernel<4><<<dim3(n, (width + 1023) / 1024), 256, 0, stream>>>(y, weights, out, top, width, chosen, experts,
                                                 BesideExperts<bf16_t>{identity ? xb : nullptr, shared_gate, (const bf16_t*)shared_y, nullptr, nullptr, 0});
    LSA_LAUNCH_CHECK();
}
