// Kernels of blocks and mixers that several designs can share: the gated delta rule with its short convolutions,
// the difference of two attention maps, and a block whose two sublayers join a 32-bit stream together under gates.
// Everything behind a projection is float32 here, whatever the type of the projections' results.
#include <type_traits>

#include "common.hpp"
#include "chunks.hpp"

using namespace lsa;

namespace {

__device__ inline float sigmoid_of(float z) { return 1.f / (1.f + expf(-z)); }
__device__ inline float softplus_of(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// ---- a block whose sublayers' results join the stream together ---------------------------------------------------------
// x[t] += s1 * sigmoid(gates[t][:W]) * y1[t] + s2 * sigmoid(gates[t][W:]) * y2[t] (y2 may be absent), in float32 where x
// lies; then, with next_weight, normed[t] = x[t] * rsqrt(mean(x[t]^2) + eps) * next_weight.  One workgroup a token.  Rows of
// up to 256 * COLS numbers (COLS > 0): a thread issues all its loads (the stream, gates, results, scales, the next norm's
// weights) before the first store and before the sum of squares, so a row of one token waits for memory once, and keeps its
// columns in registers between the sum and the norm.  Longer rows walk their columns and read the stored row again.
constexpr int UPDATE_COLS = 16;
template <typename G, typename Y1, typename Y2, typename N, int COLS>
__global__ __launch_bounds__(256) void gated_pair_update_kernel(float* __restrict__ x, const G* __restrict__ gates, int gate_width,
                                                                const Y1* __restrict__ y1, const float* __restrict__ s1,
                                                                const Y2* __restrict__ y2, const float* __restrict__ s2,
                                                                const float* __restrict__ next_weight, float eps, N* __restrict__ normed, int width) {
    __shared__ float scratch[16];
    const int t = blockIdx.x;
    float* row = x + (size_t)t * width;
    const G* g = gates + (size_t)t * gate_width;
    if constexpr (COLS > 0) {
        float xv[COLS > 0 ? COLS : 1], g1[COLS > 0 ? COLS : 1], a1[COLS > 0 ? COLS : 1], w1[COLS > 0 ? COLS : 1], g2[COLS > 0 ? COLS : 1],
            a2[COLS > 0 ? COLS : 1], w2[COLS > 0 ? COLS : 1], nw[COLS > 0 ? COLS : 1];
        // every load is of a place that is there (a column beyond the row reads the row's last one, an absent second
        // sublayer reads the first one's operands, an absent norm the first scale), so none stands under a condition
        // (the launcher makes Y2 float where there is no second sublayer, so the stream's own row can stand in)
        const Y2* second = y2 ? y2 + (size_t)t * width : reinterpret_cast<const Y2*>(row);
        const float* second_scale = y2 ? s2 : s1;
        const float* following = next_weight ? next_weight : s1;
        const int second_gate = y2 ? width : 0;
        const float counts = y2 ? 1.f : 0.f;
#pragma unroll
        for (int n = 0; n < COLS; ++n) {
            const int c = min((int)threadIdx.x + 256 * n, width - 1);
            xv[n] = row[c];
            g1[n] = (float)g[c];
            a1[n] = (float)y1[(size_t)t * width + c];
            w1[n] = s1[c];
            g2[n] = (float)g[second_gate + c];
            a2[n] = (float)second[c];
            w2[n] = second_scale[c] * counts;
            nw[n] = following[c];
        }
        float sq = 0.f;
#pragma unroll
        for (int n = 0; n < COLS; ++n) {
            xv[n] += w1[n] * sigmoid_of(g1[n]) * a1[n] + w2[n] * sigmoid_of(g2[n]) * a2[n];
            if ((int)threadIdx.x + 256 * n < width) sq += xv[n] * xv[n];
        }
#pragma unroll
        for (int n = 0; n < COLS; ++n) {
            const int c = threadIdx.x + 256 * n;
            if (c < width) row[c] = xv[n];
        }
        if (!next_weight) return;
        const float inv = rsqrtf(block_sum(sq, scratch) / (float)width + eps);
#pragma unroll
        for (int n = 0; n < COLS; ++n) {
            const int c = threadIdx.x + 256 * n;
            if (c < width) normed[(size_t)t * width + c] = (N)(xv[n] * inv * nw[n]);
        }
        return;
    }
    float sq = 0.f;
    for (int c = threadIdx.x; c < width; c += 256) {
        float v = row[c] + s1[c] * sigmoid_of((float)g[c]) * (float)y1[(size_t)t * width + c];
        if (y2) v += s2[c] * sigmoid_of((float)g[width + c]) * (float)y2[(size_t)t * width + c];
        row[c] = v;
        sq += v * v;
    }
    if (!next_weight) return;
    const float inv = rsqrtf(block_sum(sq, scratch) / (float)width + eps);
    for (int c = threadIdx.x; c < width; c += 256) normed[(size_t)t * width + c] = (N)(row[c] * inv * next_weight[c]);
}

// ---- differential attention: a1 - lambda a2 per head, divided by its root mean square, times a constant -------------------
// grid (tokens, heads), one wavefront.  attended [T][kv_heads][2][group][row]; out [T][kv_heads * group][value_dim].
template <typename T>
__global__ __launch_bounds__(64) void differential_heads_kernel(const T* __restrict__ attended, float lam, float keep, float eps,
                                                                T* __restrict__ out, int group, int value_dim, int row) {
    const int t = blockIdx.x, head = blockIdx.y, heads = gridDim.y, lane = threadIdx.x;
    const int g = head / group, r = head % group;
    const T* a1 = attended + (((size_t)t * (heads / group) + g) * 2 * group + r) * row;
    const T* a2 = a1 + (size_t)group * row;
    float sq = 0.f;
    for (int j = lane; j < value_dim; j += 64) {
        const float d = (float)a1[j] - lam * (float)a2[j];
        sq += d * d;
    }
    const float inv = rsqrtf(wave_sum(sq) / (float)value_dim + eps) * keep;
    T* o = out + ((size_t)t * heads + head) * value_dim;
    for (int j = lane; j < value_dim; j += 64) o[j] = (T)(((float)a1[j] - lam * (float)a2[j]) * inv);
}

template <int CTRL>
__device__ inline float add_across(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// the sum over the 16 lanes of a row of lanes; every lane gets it
__device__ inline float sum_of_16(float v) {
    v = add_across<0xB1>(v);        // quad_perm [1, 0, 3, 2]
    v = add_across<0x4E>(v);        // quad_perm [2, 3, 0, 1]
    v = add_across<0x141>(v);       // row_half_mirror
    v = add_across<0x140>(v);       // row_mirror
    return v;
}

// ---- the delta rule's inputs ----------------------------------------------------------------------------------------------
// grid (tokens, 2 kv_heads + 2 heads), one wavefront.  Blocks 0 .. 2 kv_heads - 1: a query or key head: causal convolution over
// the request's tokens per channel, silu, the head divided by sqrt(sum of squares + unit_eps), queries times q_scale.  The next
// `heads` blocks: a value head (convolution and silu).  The last `heads` blocks: the head's write strength sigmoid(b) and its
// decay exp(-exp(A) softplus(z + bias)), one number or one per key channel.  A token's predecessors come from the step's own
// rows where the step brings them and from state[slot][k][channel] (the request's last taps - 1 inputs, oldest first) where it
// does not; zeros before the sequence.  keep (steps of one token a row): the thread that has read a channel's state moves it on.
constexpr int MOST_DIM = 256;       // key channels of a head
template <typename T>
__global__ __launch_bounds__(64) void delta_prepare_kernel(const T* __restrict__ proj, long stride, const float* __restrict__ w, int taps,
                                                           float* state, long state_stride, const int* __restrict__ slots,
                                                           const int* __restrict__ token_row, const int* __restrict__ positions,
                                                           const int* __restrict__ row_start, float* __restrict__ out,
                                                           int kv_heads, int heads, int dim, int value_dim, float q_scale, float unit_eps, int keep,
                                                           const T* __restrict__ strength, long strength_stride, const void* __restrict__ decay,
                                                           long decay_stride, int per_channel, const float* __restrict__ decay_scale,
                                                           const float* __restrict__ decay_bias, float* __restrict__ out_strength,
                                                           float* __restrict__ out_decay) {
    const int t = blockIdx.x, block = blockIdx.y, lane = threadIdx.x;
    const int keys = kv_heads * dim, channels = 2 * keys + heads * value_dim;
    if (block >= 2 * kv_heads + heads) {
        const int head = block - 2 * kv_heads - heads;
        const float rate = expf(decay_scale[head]);
        if (per_channel) {
            const float* z = reinterpret_cast<const float*>(decay) + (size_t)t * decay_stride + (size_t)head * dim;
            for (int e = lane; e < dim; e += 64)
                out_decay[((size_t)t * heads + head) * dim + e] = expf(-rate * softplus_of(z[e] + decay_bias[head * dim + e]));
        } else if (lane == 0) {
            const float z = (float)reinterpret_cast<const T*>(decay)[(size_t)t * decay_stride + head];
            out_decay[(size_t)t * heads + head] = expf(-rate * softplus_of(z + decay_bias[head]));
        }
        if (lane == 0) out_strength[(size_t)t * heads + head] = sigmoid_of((float)strength[(size_t)t * strength_stride + head]);
        return;
    }
    const bool unit = block < 2 * kv_heads;
    const int size = unit ? dim : value_dim;
    const int base = unit ? block * dim : 2 * keys + (block - 2 * kv_heads) * value_dim;
    const int row = token_row[t], position = positions[t];
    const int first = position - (t - row_start[row]);
    const int kept = taps - 1;
    float* mine = kept ? state + (size_t)slots[row] * state_stride : nullptr;
    float held[MOST_DIM / 64];
    float sq = 0.f;
    int n = 0;
    for (int e = lane; e < size; e += 64, ++n) {
        const int c = base + e;
        float acc = 0.f;
        // both places a tap's input can come from are read, at rows that are there, and one is chosen: no load stands
        // under a condition, so a thread's loads are in flight together
        const float* kept_rows = mine ? mine : w;
#pragma unroll 4
        for (int j = 0; j < taps; ++j) {
            const int back = kept - j, place = position - back;
            const bool in_step = place >= first, from_state = !in_step && place >= 0;
            const float here = (float)proj[(size_t)(in_step ? t - back : t) * stride + c];
            const float before = kept_rows[(size_t)(from_state ? kept - (first - place) : 0) * channels + c];
            acc += w[(size_t)c * taps + j] * (in_step ? here : from_state ? before : 0.f);
        }
        acc *= sigmoid_of(acc);
        if (unit) {
            held[n] = acc;
            sq += acc * acc;
        } else {
            out[(size_t)t * channels + c] = acc;
        }
        if (keep && mine) {
            for (int k = 0; k + 1 < kept; ++k) mine[(size_t)k * channels + c] = mine[(size_t)(k + 1) * channels + c];
            mine[(size_t)(kept - 1) * channels + c] = (float)proj[(size_t)t * stride + c];
        }
    }
    if (!unit) return;
    const float inv = rsqrtf(wave_sum(sq) + unit_eps) * (block < kv_heads ? q_scale : 1.f);
    n = 0;
    for (int e = lane; e < size; e += 64, ++n) out[(size_t)t * channels + base + e] = held[n] * inv;
}

// The same for TAPS taps known when the kernel is compiled and heads of up to 128 channels whose rows lie at multiples of 16 bytes: sixteen lanes a (token, block),
// eight neighbouring channels a lane.  A token whose predecessors are all rows of the step asks for those alone; any other asks for both places that
// a tap's input can come from, all at once, and with `keep` puts the state's rows that it has read back one place on.  us, the kernel above and this one: 1,900
// tokens of 16 + 16 + 16 heads of 128 57, 32; one token 6.4, 4.3.
template <typename T>
__device__ __forceinline__ void load_eight(const T* p, float (&v)[8]) {
    constexpr int V = Elem<T>::kVec;
#pragma unroll
    for (int at = 0; at < 8; at += V) {
        const Vec16<T> piece = load_vec16(p + at);
#pragma unroll
        for (int k = 0; k < V; ++k) v[at + k] = (float)piece.v[k];
    }
}
__device__ __forceinline__ void store_eight(float* p, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
template <typename T, int TAPS>
__global__ __launch_bounds__(256) void delta_prepare_wide_kernel(const T* __restrict__ proj, long stride, const float* __restrict__ w,
                                                                 float* state, long state_stride, const int* __restrict__ slots,
                                                                 const int* __restrict__ token_row, const int* __restrict__ positions,
                                                                 const int* __restrict__ row_start, float* __restrict__ out,
                                                                 int kv_heads, int heads, int dim, int value_dim, float q_scale, float unit_eps, int keep,
                                                                 const T* __restrict__ strength, long strength_stride, const void* __restrict__ decay,
                                                                 long decay_stride, int per_channel, const float* __restrict__ decay_scale,
                                                                 const float* __restrict__ decay_bias, float* __restrict__ out_strength,
                                                                 float* __restrict__ out_decay, int n_tokens) {
    constexpr int KEPT = TAPS - 1;
    const int blocks = 2 * kv_heads + 2 * heads, index = (int)blockIdx.x * 16 + (threadIdx.x >> 4), e = 8 * (threadIdx.x & 15);
    const bool there = index < n_tokens * blocks;
    const int t = there ? index / blocks : 0, block = there ? index - t * blocks : 0;
    const int keys = kv_heads * dim, channels = 2 * keys + heads * value_dim;
    if (there && block >= 2 * kv_heads + heads) {
        const int head = block - 2 * kv_heads - heads;
        const float rate = expf(decay_scale[head]);
        if (per_channel) {
            if (e < dim) {
                float z[8], bias[8];
                load_eight(reinterpret_cast<const float*>(decay) + (size_t)t * decay_stride + (size_t)head * dim + e, z);
                load_eight(decay_bias + (size_t)head * dim + e, bias);
#pragma unroll
                for (int k = 0; k < 8; ++k) z[k] = expf(-rate * softplus_of(z[k] + bias[k]));
                store_eight(out_decay + ((size_t)t * heads + head) * dim + e, z);
            }
        } else if (e == 0) {
            const float z = (float)reinterpret_cast<const T*>(decay)[(size_t)t * decay_stride + head];
            out_decay[(size_t)t * heads + head] = expf(-rate * softplus_of(z + decay_bias[head]));
        }
        if (e == 0) out_strength[(size_t)t * heads + head] = sigmoid_of((float)strength[(size_t)t * strength_stride + head]);
    }
    const bool convolves = there && block < 2 * kv_heads + heads, unit = block < 2 * kv_heads;
    const int size = unit ? dim : value_dim;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int c = (unit ? block * dim : 2 * keys + (block - 2 * kv_heads) * value_dim) + e;
    if (convolves && e < size) {
        const int row = token_row[t], position = positions[t];
        const int first = position - (t - row_start[row]);
        const T* here = proj + (size_t)t * stride + c;
        float own[8], before[KEPT][8], taps[8 * TAPS];
        load_eight(here, own);
#pragma unroll
        for (int k = 0; k < TAPS; ++k) load_eight(w + (size_t)c * TAPS + 8 * k, *reinterpret_cast<float (*)[8]>(taps + 8 * k));
        if (position - KEPT >= first) {
#pragma unroll
            for (int j = 0; j < KEPT; ++j) load_eight(here - (size_t)(KEPT - j) * stride, before[j]);
        } else {
            float* mine = state + (size_t)slots[row] * state_stride + c;
            float of_step[KEPT][8];
#pragma unroll
            for (int j = 0; j < KEPT; ++j) {
                const int place = position - (KEPT - j);
                load_eight(place >= first ? here - (size_t)(KEPT - j) * stride : here, of_step[j]);
                load_eight(mine + (size_t)max(place >= first ? 0 : KEPT - (first - place), 0) * channels, before[j]);
            }
            if (keep) {                                    // (steps of one token a row: every tap in front of the token is the state's)
#pragma unroll
                for (int k = 0; k + 1 < KEPT; ++k) store_eight(mine + (size_t)k * channels, before[k + 1]);
                store_eight(mine + (size_t)(KEPT - 1) * channels, own);
            }
#pragma unroll
            for (int j = 0; j < KEPT; ++j) {
                const int place = position - (KEPT - j);
#pragma unroll
                for (int k = 0; k < 8; ++k) before[j][k] = place >= first ? of_step[j][k] : place >= 0 ? before[j][k] : 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
#pragma unroll
            for (int j = 0; j < KEPT; ++j) acc[k] += taps[k * TAPS + j] * before[j][k];
            acc[k] += taps[k * TAPS + KEPT] * own[k];
            acc[k] *= sigmoid_of(acc[k]);
        }
    }
    float sq = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) sq += acc[k] * acc[k];
    sq = sum_of_16(sq);                                    // (every lane takes part)
    if (!convolves || e >= size) return;
    if (unit) {
        const float inv = rsqrtf(sq + unit_eps) * (block < kv_heads ? q_scale : 1.f);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] *= inv;
    }
    store_eight(out + (size_t)t * channels + c, acc);
}

// After the step: state[slot][k] = input at position end - kept + k, from the step's rows where it brought that position, from
// the old state where it did not (k + count then indexes it), zero before the sequence.  A thread owns a channel of a row
// and goes through k upwards, so what it still has to read lies above what it has written.
template <typename T>
__global__ __launch_bounds__(256) void delta_conv_keep_kernel(const T* __restrict__ proj, long stride, float* __restrict__ state, long state_stride,
                                                              const int* __restrict__ slots, const int* __restrict__ row_start,
                                                              const int* __restrict__ row_len, const int* __restrict__ row_ctx, int kept, int channels) {
    const int row = blockIdx.x;
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= channels) return;
    const int count = row_len[row], end = row_ctx[row], start = row_start[row];
    if (count <= 0) return;
    const int first = end - count;
    float* mine = state + (size_t)slots[row] * state_stride;
    for (int k = 0; k < kept; ++k) {
        const int place = end - kept + k;
        float v = 0.f;
        if (place >= first) v = (float)proj[(size_t)(start + place - first) * stride + c];
        else if (place >= 0) v = mine[(size_t)(k + count) * channels + c];
        mine[(size_t)k * channels + c] = v;
    }
}

// ---- the delta rule ------------------------------------------------------------------------------------------------------------
// Per head S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q, token by token.  A column of S (one value channel)
// needs only its own v and the head's q, k, g, beta, so columns run side by side.  grid (rows, heads, blocks of 16 value
// columns), four wavefronts; a wavefront has four columns, and the 16 lanes of a column share its key channels: lane part p
// keeps the channels p, p + 16, ... (DP of them) of the column in registers for the whole row, so the state is read once
// before a row's first token and written once behind its last.  What the state returns for the key, and the read-out, are
// sums over a column's 16 lanes (four adds across lanes).  Tokens go through LDS in chunks of 16: queries, keys and decays of
// the head laid out by lane part, the chunk's values and write strengths.  Every sum is formed in one order whatever the
// cut and the batch.
constexpr int PARTS = 16;           // lanes that share a column's key channels
constexpr int CHUNK = 16;           // tokens staged at a time
constexpr int BLOCK_COLUMNS = 16;   // value columns a workgroup


// One token of a column's walk: `S` the lane's key channels of the column, `kp`, `qp`, `gp` the token's key, query and
// decays as the lane's part reads them, `g` the head's decay where there is one a head.
template <int DP, bool PER_CHANNEL>
__device__ inline float delta_token(float (&S)[DP], const float* __restrict__ kp, const float* __restrict__ qp, const float* __restrict__ gp,
                                    float g, float beta, float v) {
    float k[DP], seen[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < DP; ++i) {
        k[i] = kp[i];
        S[i] *= PER_CHANNEL ? gp[i] : g;
        seen[i & 1] += S[i] * k[i];
    }
    const float u = beta * (v - sum_of_16(seen[0] + seen[1]));
    float read[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < DP; ++i) {
        S[i] += k[i] * u;
        read[i & 1] += S[i] * qp[i];
    }
    return sum_of_16(read[0] + read[1]);
}

// state[slot]: per head and block of 16 value columns a tile [dim][16], so that a workgroup's share of the state is one
// contiguous piece, read and written 16 bytes a thread and turned into the lanes' order through LDS.
template <int DP, bool PER_CHANNEL>
__global__ __launch_bounds__(256) void delta_rule_kernel(const float* __restrict__ prepared, const float* __restrict__ strength,
                                                         const float* __restrict__ decay, float* state, long state_stride,
                                                         const int* __restrict__ slots, const int* __restrict__ row_start,
                                                         const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                                         float* __restrict__ out, int heads, int kv_heads, int dim, int value_dim) {
    constexpr int PADDED = DP * PARTS;
    static_assert(CHUNK == BLOCK_COLUMNS, "the staging buffer of the queries doubles as the state's tile");
    __shared__ __align__(16) float s_q[CHUNK][PADDED], s_k[CHUNK][PADDED], s_g[PER_CHANNEL ? CHUNK : 1][PER_CHANNEL ? PADDED : 1];
    __shared__ float s_v[CHUNK][BLOCK_COLUMNS], s_beta[CHUNK], s_decay[CHUNK];
    const int row = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int count = row_len[row];
    if (count <= 0) return;
    const int start = row_start[row];
    const bool fresh = row_ctx[row] - count == 0;
    const int p = lane & (PARTS - 1);
    const int local = wave * 4 + (lane >> 4);
    const int column = blockIdx.z * BLOCK_COLUMNS + local;
    const bool live = column < value_dim;
    const int kv_head = head / (heads / kv_heads);
    const int keys = kv_heads * dim, channels = 2 * keys + heads * value_dim;
    float* tile = state + (size_t)slots[row] * state_stride + ((size_t)head * gridDim.z + blockIdx.z) * dim * BLOCK_COLUMNS;
    float* turned = &s_q[0][0];                     // [PADDED][16], rows beyond dim unused
    float S[DP];
    if (fresh) {
#pragma unroll
        for (int i = 0; i < DP; ++i) S[i] = 0.f;
    } else {
        for (int piece = tid; piece < dim * (BLOCK_COLUMNS / 4); piece += 256)
            reinterpret_cast<float4*>(turned)[piece] = reinterpret_cast<const float4*>(tile)[piece];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < DP; ++i) {
            const int ch = i * PARTS + p;
            S[i] = (ch < dim && live) ? turned[ch * BLOCK_COLUMNS + local] : 0.f;      // (columns beyond the values stay zero)
        }
    }
    for (int begin = 0; begin < count; begin += CHUNK) {
        const int tokens = min(CHUNK, count - begin);
        __syncthreads();
        // stage the chunk: channel ch of a token goes to [ch % 16][ch / 16], where lane part ch % 16 reads it
        for (int index = tid; index < tokens * PADDED; index += 256) {
            const int j = index / PADDED, ch = index % PADDED;
            const size_t t = (size_t)(start + begin + j);
            const int at = (ch % PARTS) * DP + ch / PARTS;
            const bool there = ch < dim;
            s_q[j][at] = there ? prepared[t * channels + kv_head * dim + ch] : 0.f;
            s_k[j][at] = there ? prepared[t * channels + keys + kv_head * dim + ch] : 0.f;
            if (PER_CHANNEL) s_g[j][at] = there ? decay[(t * heads + head) * dim + ch] : 1.f;
        }
        for (int index = tid; index < tokens * BLOCK_COLUMNS; index += 256) {
            const int j = index / BLOCK_COLUMNS, c = index % BLOCK_COLUMNS;
            const int col = blockIdx.z * BLOCK_COLUMNS + c;
            s_v[j][c] = col < value_dim ? prepared[(size_t)(start + begin + j) * channels + 2 * keys + head * value_dim + col] : 0.f;
        }
        if (tid < tokens) {
            s_beta[tid] = strength[(size_t)(start + begin + tid) * heads + head];
            if (!PER_CHANNEL) s_decay[tid] = decay[(size_t)(start + begin + tid) * heads + head];
        }
        __syncthreads();
        float* o = out + (size_t)(start + begin) * heads * value_dim + (size_t)head * value_dim + column;
        const bool writes = p == 0 && live;
        if (tokens == CHUNK) {
            // a whole chunk runs unrolled: a token's LDS loads are issued ahead of the token before it, and its read-out's
            // sum across lanes overlaps the next token's walk
            // (the read-outs wait in registers for the chunk's end: a store under a condition between two tokens would end
            // the stretch of code that the loads can move within)
            float r[CHUNK];
#pragma unroll
            for (int j = 0; j < CHUNK; ++j)
                r[j] = delta_token<DP, PER_CHANNEL>(S, &s_k[j][p * DP], &s_q[j][p * DP], PER_CHANNEL ? &s_g[j][p * DP] : nullptr,
                                                    PER_CHANNEL ? 1.f : s_decay[j], s_beta[j], s_v[j][local]);
            if (writes) {
#pragma unroll
                for (int j = 0; j < CHUNK; ++j) o[(size_t)j * heads * value_dim] = r[j];
            }
        } else {
            for (int j = 0; j < tokens; ++j) {
                const float r = delta_token<DP, PER_CHANNEL>(S, &s_k[j][p * DP], &s_q[j][p * DP], PER_CHANNEL ? &s_g[j][p * DP] : nullptr,
                                                             PER_CHANNEL ? 1.f : s_decay[j], s_beta[j], s_v[j][local]);
                if (writes) o[(size_t)j * heads * value_dim] = r;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DP; ++i) {
        const int ch = i * PARTS + p;
        if (ch < dim) turned[ch * BLOCK_COLUMNS + local] = S[i];
    }
    __syncthreads();
    for (int piece = tid; piece < dim * (BLOCK_COLUMNS / 4); piece += 256)
        reinterpret_cast<float4*>(tile)[piece] = reinterpret_cast<const float4*>(turned)[piece];
}

// ---- the delta rule in chunks -----------------------------------------------------------------------------------------------------
// Walking a row's tokens one by one takes 0.36 us a token whatever the card could do beside it (680 us for 1,900 tokens of 16
// heads of 128 x 128).  In chunks of 64 tokens what a chunk writes is the solution of a triangular system: with W(t, j) the
// product of the decays behind token j up to token t,
//   u_t = beta_t (v_t - (W(t, start) k_t)^T S_0 - sum_{j < t} (sum_c k_t W(t, j) k_j) u_j),
// so with L = beta (sum_c k_t W(t, j) k_j), U = (I + L)^-1 beta v and K = (I + L)^-1 beta (W(t, start) k_t) the chunk's writes are
// U - K S_0, the state behind it M S_0 + C with M = diag(W(end, start)) - E^T K, C = E^T U, E_j = W(end, j) k_j, and the
// read-outs Q S_0 + B U with B_tj = sum_c q_t W(t, j) k_j (j <= t) and Q_t = W(t, start) q_t - B K.  M, C, Q and B U need no state:
// (1) forms them for all chunks at once, (2) walks S <- M S + C, one product of 128 x 128 x 16 a chunk and 16 columns, and leaves
// the state in front of each chunk where its C was, (3) adds Q S_0: 105, 57 and 27 us for the 1,900 tokens, 190 together.
// All operands are 32-bit.  The walk's and the keys' products are 32-bit too, four partial sums each, added up in 64-bit; what a token
// writes and reads (U, B, B U, Q S_0) is summed in 64-bit, because a rounding there goes into all of its channels, where the walk's fall
// on each channel by itself and average out.  With 32-bit sums a read-out's error against 64 bits was 1.4 times that of the token by
// token walk where the memory is short; as it stands it is 0.5 to 1.0 times that (decays around 0.999 to 0.5, 1,900 tokens).
// What lies in scratch memory lies as the matrix instructions hold it: pieces of 16 x 16, a lane's four numbers side by side, so
// every load and store of it moves 1 KB of a wavefront in a row.
constexpr int CHUNKED_MOST_DIM = 128;
constexpr int CHUNK_TILES = 16;          // blocks of 16 columns (of K or U) a workgroup: two a wavefront

template <int P>                         // P: key channels filled up to 64 or 128
struct DeltaChunkLds {
    static constexpr int A = P + 4;
    float q[MC * A];                     // queries; then W(t, start) q
    float k[MC * A];                     // keys; then E
    float d[MC * A];                     // decays; then W(t, start) k
    float kk[MC * MC_A];                 // L
    float qk[MC * MC_A];                 // B
    float inverse[MC / BC][BC * 20];     // of I + L's blocks on the diagonal
    float beta[MC];
    double total[MC / BC][P];
};

// (1) grid (items, heads, blocks of 256 columns of K | U), eight wavefronts; LDS leaves room for one workgroup a CU.  What it waits for
// are the products (7 MFLOP a workgroup of 16 column blocks) and, in front of them, the weights inside the blocks of 16.
template <int P, bool PER_CHANNEL>
__global__ __launch_bounds__(512) void delta_chunk_kernel(const float* __restrict__ prepared, const float* __restrict__ strength,
                                                          const float* __restrict__ decay, const int* __restrict__ row_start,
                                                          const int* __restrict__ row_len, const int* __restrict__ row_ctx, int rows,
                                                          mc_f4* __restrict__ sums, mc_f4* __restrict__ steps, mc_f4* __restrict__ queries,
                                                          float* __restrict__ out, int heads, int kv_heads, int dim, int value_dim) {
    extern __shared__ __align__(16) float lds[];
    typedef DeltaChunkLds<P> Lds;
    Lds& s = *reinterpret_cast<Lds*>(lds);
    constexpr int A = Lds::A, KT = P / 16;
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int count = row_len[row], n = min(MC, count - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const int keys = kv_heads * dim, channels = 2 * keys + heads * value_dim;
    const int key_column = head / (heads / kv_heads) * dim;
    const int value_tiles = (value_dim + 15) / 16;
    const int tile0 = blockIdx.z * CHUNK_TILES + 2 * wave;               // KT is even: a wavefront's two are both of K or both of U
    const bool of_keys = tile0 < KT;

    // The chunk's rows; tokens behind its last one and channels behind the head's last one read and write nothing and keep
    // everything.  (Every load is of a place that is there: none stands under a condition.)
    float values[2][MC / 4];                                             // [column block][(block of 16 tokens) * 4 + e]: token 16 block + 4 e + g
    {
        constexpr int PER = MC * P / 512;
        float raw_q[PER], raw_k[PER], raw_d[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + 512 * e, t = min(i / P, n - 1), c = min(i % P, dim - 1);
            const float* mine = prepared + (token0 + t) * channels + key_column + c;
            raw_q[e] = mine[0];
            raw_k[e] = mine[keys];
            raw_d[e] = PER_CHANNEL ? decay[((token0 + t) * heads + head) * dim + c] : decay[(token0 + t) * heads + head];
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int column = min(max((tile0 + m - KT) * 16 + r, 0), value_dim - 1);
#pragma unroll
            for (int e = 0; e < MC / 4; ++e)
                values[m][e] = prepared[(token0 + min(16 * (e / 4) + 4 * (e % 4) + g, n - 1)) * channels + 2 * keys + (size_t)head * value_dim + column];
        }
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + 512 * e, t = i / P, c = i % P;
            const bool there = t < n && c < dim;
            s.q[t * A + c] = there ? raw_q[e] : 0.f;
            s.k[t * A + c] = there ? raw_k[e] : 0.f;
            s.d[t * A + c] = there ? raw_d[e] : 1.f;
        }
        for (int i = tid; i < MC * MC_A; i += 512) s.kk[i] = s.qk[i] = 0.f;
        if (tid < MC) s.beta[tid] = tid < n ? strength[(token0 + min(tid, n - 1)) * heads + head] : 0.f;
    }
    __syncthreads();

    // Inside the blocks: wavefront = (block, half of the channels), lane = (token t of the block, a quarter of every 16 channels).  The
    // diagonals j = t - back one after another, W(t, j) in registers.
    {
        const int block = wave >> 1, half = wave & 1, t = r, c0 = half * (P / 2) + 4 * g;
        constexpr int U = P / 32;
        float weight[U][4], query[U][4], key[U][4];
        double by_query[BC], by_key[BC];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float4 x = *reinterpret_cast<const float4*>(&s.q[(block * BC + t) * A + c0 + 16 * u]);
            const float4 y = *reinterpret_cast<const float4*>(&s.k[(block * BC + t) * A + c0 + 16 * u]);
            query[u][0] = x.x; query[u][1] = x.y; query[u][2] = x.z; query[u][3] = x.w;
            key[u][0] = y.x; key[u][1] = y.y; key[u][2] = y.z; key[u][3] = y.w;
#pragma unroll
            for (int e = 0; e < 4; ++e) weight[u][e] = 1.f;
        }
#pragma unroll
        for (int back = 0; back < BC; ++back) {
            const int j = block * BC + max(t - back, 0);
            float part_q[4] = {}, part_k[4] = {};
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float4 x = *reinterpret_cast<const float4*>(&s.k[j * A + c0 + 16 * u]);
                const float4 f = *reinterpret_cast<const float4*>(&s.d[j * A + c0 + 16 * u]);
                const float ks[4] = {x.x, x.y, x.z, x.w}, ds[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float kept = weight[u][e] * ks[e];
                    part_q[e] = __builtin_fmaf(query[u][e], kept, part_q[e]);
                    part_k[e] = __builtin_fmaf(key[u][e], kept, part_k[e]);
                    weight[u][e] *= ds[e];                                         // (the next diagonal lies behind token j's decay)
                }
            }
            by_query[back] = ((double)part_q[0] + (double)part_q[1]) + ((double)part_q[2] + (double)part_q[3]);
            by_key[back] = ((double)part_k[0] + (double)part_k[1]) + ((double)part_k[2] + (double)part_k[3]);
        }
#pragma unroll
        for (int back = 0; back < BC; ++back) {
            by_query[back] += __shfl_xor(by_query[back], 16, 64);
            by_query[back] += __shfl_xor(by_query[back], 32, 64);
            by_key[back] += __shfl_xor(by_key[back], 16, 64);
            by_key[back] += __shfl_xor(by_key[back], 32, 64);
        }
        const int at = (block * BC + t) * MC_A + block * BC + t;
        for (int turn = 0; turn < 2; ++turn) {                                     // one half of the channels after the other
            if (half == turn && lane < 16) {
#pragma unroll
                for (int back = 0; back < BC; ++back) {
                    if (back > t) continue;
                    s.qk[at - back] += by_query[back];
                    if (back > 0) s.kk[at - back] += by_key[back];
                }
            }
            __syncthreads();
        }
    }

    // Queries and keys times the decays from their block's first token, keys times those up to its last one; a thread a (block,
    // channel).  The products are formed in 64-bit: sixteen factors then cost a weight one rounding, as they do the scan's state.
    for (int i = tid; i < (MC / BC) * P; i += 512) {
        const int block = i / P, c = i % P;
        float* qs = &s.q[block * BC * A + c];
        float* ks = &s.k[block * BC * A + c];
        float* ds = &s.d[block * BC * A + c];
        float d[BC], k[BC];
#pragma unroll
        for (int t = 0; t < BC; ++t) d[t] = ds[t * A], k[t] = ks[t * A];
        double product = 1.0;
#pragma unroll
        for (int t = 0; t < BC; ++t) {
            product *= (double)d[t];
            qs[t * A] = (float)((double)qs[t * A] * product);
            ds[t * A] = (float)((double)k[t] * product);
        }
        s.total[block][c] = product;
        product = 1.0;
#pragma unroll
        for (int t = BC - 1; t >= 0; --t) {
            ks[t * A] = (float)((double)k[t] * product);
            product *= (double)d[t];
        }
    }
    __syncthreads();

    // Between blocks: twelve tiles of 16 x 16 weights, two on wavefronts 4 to 7 and one on the others, which invert a block on the
    // diagonal each as well: lane = column, its rows one after another.
    for (int task = wave < 4 ? 8 + wave : wave - 4; task < (wave < 4 ? 12 : 8); task += 4) {
        const int pair = task >> 1, block = pair < 3 ? 3 : pair < 5 ? 2 : 1, other = pair < 3 ? pair : pair < 5 ? pair - 3 : 0;
        const float* a = (task & 1 ? s.d : s.q) + (block * BC + r) * A + g;
        const float* b = &s.k[(other * BC + r) * A + g];
        mc_d4 sum = {};
#pragma unroll 4
        for (int i = 0; i < P; i += 4) {
            double x = (double)a[i];
            if (block - other > 1) x *= s.total[other + 1][i + g];
            if (block - other > 2) x *= s.total[other + 2][i + g];
            sum = __builtin_amdgcn_mfma_f64_16x16x4f64(x, (double)b[i], sum, 0, 0, 0);
        }
        float* to = task & 1 ? s.kk : s.qk;
#pragma unroll
        for (int e = 0; e < 4; ++e) to[(block * BC + 4 * e + g) * MC_A + other * BC + r] = (float)sum[e];
    }
    if (wave < 4) {
        float x[BC];
#pragma unroll
        for (int t = 0; t < BC; ++t) {
            const float* line = &s.kk[(wave * BC + t) * MC_A + wave * BC];
            const float beta = s.beta[wave * BC + t];
            float acc[2] = {t == r ? 1.f : 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < t; ++j) acc[j & 1] -= beta * line[j] * x[j];
            x[t] = acc[0] + acc[1];
        }
        if (g == 0) {
#pragma unroll
            for (int t = 0; t < BC; ++t) s.inverse[wave][t * 20 + r] = x[t];
        }
    }
    __syncthreads();

    // Everything brought from its block to the chunk, whatever lies in front of or behind the block in one product, 64-bit as above.
    {
        constexpr int PER = MC * P / 512;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + 512 * e, t = i / P, c = i % P, block = t / BC;
            double before = 1.0, behind = 1.0;
#pragma unroll
            for (int o = 0; o < MC / BC; ++o) {
                const double total = s.total[o][c];
                before *= o < block ? total : 1.0;
                behind *= o > block ? total : 1.0;
            }
            s.q[t * A + c] = (float)((double)s.q[t * A + c] * before);
            s.d[t * A + c] = (float)((double)s.d[t * A + c] * before);
            s.k[t * A + c] = (float)((double)s.k[t * A + c] * behind);
        }
        for (int i = tid; i < MC * MC; i += 512) s.kk[(i / MC) * MC_A + i % MC] *= s.beta[i / MC];
    }
    __syncthreads();

    if (tile0 >= KT + value_tiles) return;
    if (of_keys && chunk == 0 && row_ctx[row] == count) return;          // nothing stands in front of a sequence's first chunk: no K is asked for
    // From here a wavefront goes on by itself with its 32 columns of the right side, beta (W(t, start) k) or beta v: the columns of the
    // solution stay in registers as the matrix instructions leave them, which is how these take them as an operand again.
    auto own_columns = [&](auto keys_side) {
        constexpr bool KEYS = decltype(keys_side)::value;
        auto token_of = [&](int e) { return KEYS ? 4 * g + e : 4 * e + g; };     // a block's row that a lane's number e belongs to
        // The matrix instructions multiply the zeros above a block's diagonal too.  Where a token's column is no number, the blocks on the
        // diagonal are multiplied without them, so that the tokens in front of it keep theirs: of a block's lower half `lower` (rows of
        // `pitch`) and its 16 x 16 numbers y (as x below), row `t`, column `column`.
        auto numbers = [&](const auto& of) {
            float zero = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) zero = __builtin_fmaf((float)of[e], 0.f, zero);
            return !__any(zero != 0.f);
        };
        auto row_of_lower = [&](const float* lower, int pitch, const auto& y, int t, int column) {
            double sum = 0.0;
#pragma unroll
            for (int j = 0; j < BC; ++j) {
                const double there = __shfl((double)y[KEYS ? j % 4 : j / 4], 16 * (KEYS ? j / 4 : j % 4) + column, 64);
                if (j <= t) sum += (double)lower[t * pitch + j] * there;
            }
            return sum;
        };
        mc_f4 x[2][MC / BC];
#pragma unroll
        for (int i = 0; i < MC / BC; ++i) {
            if constexpr (KEYS) {
                mc_f4 part[2][4] = {};
#pragma unroll
                for (int o = 0; o < i; ++o) {
                    const mc_f4 a = *reinterpret_cast<const mc_f4*>(&s.kk[(i * BC + r) * MC_A + o * BC + 4 * g]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int m = 0; m < 2; ++m) part[m][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], x[m][o][e], part[m][e], 0, 0, 0);
                }
                const mc_f4 beta = *reinterpret_cast<const mc_f4*>(&s.beta[i * BC + 4 * g]);
                const mc_f4 a = *reinterpret_cast<const mc_f4*>(&s.inverse[i][r * 20 + 4 * g]);
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    mc_f4 right = -together(part[m]), sum[4] = {};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        right[e] = __builtin_fmaf(beta[e], s.d[(i * BC + 4 * g + e) * A + (tile0 + m) * 16 + r], right[e]);
                        sum[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], right[e], sum[e], 0, 0, 0);
                    }
                    x[m][i] = together(sum);
                    if (!numbers(x[m][i])) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[m][i][e] = (float)row_of_lower(s.inverse[i], 20, right, 4 * g + e, r);
                    }
                }
            } else {
                mc_d4 right[2] = {};
#pragma unroll
                for (int o = 0; o < i; ++o)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double a = -(double)s.kk[(i * BC + r) * MC_A + o * BC + 4 * e + g];
#pragma unroll
                        for (int m = 0; m < 2; ++m) right[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)x[m][o][e], right[m], 0, 0, 0);
                    }
                mc_d4 sum[2] = {};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = i * BC + 4 * e + g;
                    const double a = (double)s.inverse[i][r * 20 + 4 * e + g], beta = (double)s.beta[t];
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        const bool there = t < n && (tile0 + m - KT) * 16 + r < value_dim;
                        right[m][e] = there ? right[m][e] + beta * (double)values[m][4 * i + e] : 0.0;
                        sum[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, right[m][e], sum[m], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int m = 0; m < 2; ++m) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[m][i][e] = (float)sum[m][e];
                    if (!numbers(x[m][i])) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[m][i][e] = (float)row_of_lower(s.inverse[i], 20, right[m], 4 * e + g, r);
                    }
                }
            }
        }
        const size_t cell = (size_t)blockIdx.x * heads + head;
#pragma unroll 2
        for (int tile = 0; tile < KT; ++tile) {
            mc_f4 part[2][4] = {};
#pragma unroll
            for (int i = 0; i < MC / BC; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float end = s.k[(i * BC + token_of(e)) * A + tile * 16 + r];
#pragma unroll
                    for (int m = 0; m < 2; ++m)
                        part[m][e] = KEYS ? __builtin_amdgcn_mfma_f32_16x16x4f32(x[m][i][e], end, part[m][e], 0, 0, 0)
                                          : __builtin_amdgcn_mfma_f32_16x16x4f32(end, x[m][i][e], part[m][e], 0, 0, 0);
                }
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                mc_f4 sum = together(part[m]);
                if (KEYS) {                                              // a row of M per lane, four of its columns
                    const int c = tile * 16 + r;
                    const float whole = (float)((s.total[0][c] * s.total[1][c]) * (s.total[2][c] * s.total[3][c]));
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] = ((tile0 + m) * 16 + 4 * g + e == c ? whole : 0.f) - sum[e];
                    steps[((cell * KT + tile) * KT + tile0 + m) * 64 + lane] = sum;
                } else if (tile0 + m < KT + value_tiles) {               // a column of C per lane, four of its rows
                    sums[((cell * value_tiles + tile0 + m - KT) * KT + tile) * 64 + lane] = sum;
                }
            }
        }
#pragma unroll
        for (int block = 0; block < MC / BC; ++block) {
            if constexpr (KEYS) {
                mc_f4 part[2][4] = {};
#pragma unroll
                for (int i = 0; i <= block; ++i) {
                    const mc_f4 a = *reinterpret_cast<const mc_f4*>(&s.qk[(block * BC + r) * MC_A + i * BC + 4 * g]);
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        if (i == block && !numbers(x[m][i])) continue;
#pragma unroll
                        for (int e = 0; e < 4; ++e) part[m][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[m][i][e], a[e], part[m][e], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int m = 0; m < 2; ++m) {                            // a token per lane, four of its channels
                    mc_f4 own = *reinterpret_cast<const mc_f4*>(&s.q[(block * BC + r) * A + (tile0 + m) * 16 + 4 * g]);
                    own -= together(part[m]);
                    if (!numbers(x[m][block])) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) own[e] -= (float)row_of_lower(&s.qk[block * BC * MC_A + block * BC], MC_A, x[m][block], r, 4 * g + e);
                    }
                    queries[((cell * (MC / BC) + block) * KT + tile0 + m) * 64 + lane] = own;
                }
            } else {
                mc_d4 sum[2] = {};
#pragma unroll
                for (int i = 0; i <= block; ++i)
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        if (i == block && !numbers(x[m][i])) continue;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const double a = (double)s.qk[(block * BC + r) * MC_A + i * BC + 4 * e + g];
                            sum[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)x[m][i][e], sum[m], 0, 0, 0);
                        }
                    }
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int column = (tile0 + m - KT) * 16 + r;
                    if (!numbers(x[m][block])) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum[m][e] += row_of_lower(&s.qk[block * BC * MC_A + block * BC], MC_A, x[m][block], 4 * e + g, r);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int t = block * BC + 4 * e + g;
                        if (t < n && column < value_dim) out[(token0 + t) * heads * value_dim + (size_t)head * value_dim + column] = (float)sum[m][e];
                    }
                }
            }
        }
    };
    if (of_keys) own_columns(std::true_type{});
    else own_columns(std::false_type{});
}

// (2) S <- M S + C over a row's chunks, the state in front of each left in C's place; grid (rows, heads, blocks of 16 value columns),
// four wavefronts, each P / 64 blocks of 16 of the state's rows.  M comes straight from memory into registers, a piece read again for
// the next chunk as soon as its products have been issued; the state goes round the wavefronts through LDS.
template <int P>
__global__ __launch_bounds__(256) void delta_chunk_walk_kernel(mc_f4* sums, const mc_f4* __restrict__ steps, float* state, long state_stride,
                                                               const int* __restrict__ slots, const int* __restrict__ row_len,
                                                               const int* __restrict__ row_ctx, int heads, int dim, int value_dim) {
    constexpr int KT = P / 16, TILES = P / 64, LINE = P + 4;
    __shared__ __align__(16) float shared_state[2][16 * LINE];           // [column][channel]
    const int row = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int count = row_len[row];
    if (count <= 0) return;
    const int chunks = (count + MC - 1) / MC;
    int item = 0;
    for (int before = 0; before < row; ++before) item += row_len[before] > 0 ? (row_len[before] + MC - 1) / MC : 0;
    const bool fresh = row_ctx[row] == count;
    const bool live = (int)blockIdx.z * 16 + r < value_dim;
    float* tile = state + (size_t)slots[row] * state_stride + ((size_t)head * gridDim.z + blockIdx.z) * dim * BLOCK_COLUMNS;
    const size_t sum_cell = (size_t)gridDim.z * KT * 64, step_cell = (size_t)KT * KT * 64;
    mc_f4* sum = sums + ((size_t)item * heads + head) * sum_cell + (size_t)blockIdx.z * KT * 64 + wave * TILES * 64 + lane;
    const mc_f4* step = steps + ((size_t)item * heads + head) * step_cell + (size_t)wave * TILES * KT * 64 + lane;
    mc_f4 S[TILES], C[TILES], M[TILES][KT];
    int chunk = 0;
    if (fresh) {
#pragma unroll
        for (int n = 0; n < TILES; ++n) S[n] = sum[n * 64];
        chunk = 1;
        sum += sum_cell * heads;
        step += step_cell * heads;
    } else {
#pragma unroll
        for (int n = 0; n < TILES; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = (wave * TILES + n) * 16 + 4 * g + e;
                const float there = tile[min(c, dim - 1) * BLOCK_COLUMNS + r];
                S[n][e] = c < dim && live ? there : 0.f;
            }
    }
    if (chunk < chunks) {
#pragma unroll
        for (int n = 0; n < TILES; ++n) {
            C[n] = sum[n * 64];
#pragma unroll
            for (int u = 0; u < KT; ++u) M[n][u] = step[(n * KT + u) * 64];
        }
    }
    for (; chunk < chunks; ++chunk) {
        float* turned = shared_state[chunk & 1];
#pragma unroll
        for (int n = 0; n < TILES; ++n) {
            *reinterpret_cast<mc_f4*>(&turned[r * LINE + (wave * TILES + n) * 16 + 4 * g]) = S[n];
            sum[n * 64] = S[n];
        }
        __syncthreads();
        const bool more = chunk + 1 < chunks;
        sum += more ? sum_cell * heads : 0;
        step += more ? step_cell * heads : 0;
        mc_f4 part[TILES][4] = {};
#pragma unroll
        for (int u = 0; u < KT; ++u) {
            const mc_f4 b = *reinterpret_cast<const mc_f4*>(&turned[r * LINE + u * 16 + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < TILES; ++n) part[n][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[n][u][e], b[e], part[n][e], 0, 0, 0);
#pragma unroll
            for (int n = 0; n < TILES; ++n) M[n][u] = step[(n * KT + u) * 64];
        }
#pragma unroll
        for (int n = 0; n < TILES; ++n) {
            S[n] = C[n] + together(part[n]);
            C[n] = sum[n * 64];
        }
    }
#pragma unroll
    for (int n = 0; n < TILES; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = (wave * TILES + n) * 16 + 4 * g + e;
            if (c < dim) tile[c * BLOCK_COLUMNS + r] = S[n][e];
        }
}

// (3) out += Q S_0; grid (items, heads, blocks of 64 value columns), a wavefront a block of 16 tokens.
template <int P>
__global__ __launch_bounds__(256) void delta_chunk_read_kernel(const mc_f4* __restrict__ sums, const mc_f4* __restrict__ queries,
                                                               const int* __restrict__ row_start, const int* __restrict__ row_len,
                                                               const int* __restrict__ row_ctx, int rows, float* __restrict__ out, int heads,
                                                               int value_dim) {
    constexpr int KT = P / 16;
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, lane = threadIdx.x & 63, block = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int count = row_len[row], n = min(MC, count - chunk * MC);
    if ((chunk == 0 && row_ctx[row] == count) || block * BC >= n) return;
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const int value_tiles = (value_dim + 15) / 16;
    const size_t cell = (size_t)blockIdx.x * heads + head;
    const mc_f4* mine = queries + (cell * (MC / BC) + block) * KT * 64 + lane;
    mc_d4 sum[4] = {};
#pragma unroll
    for (int u = 0; u < KT; ++u) {
        const mc_f4 a = mine[u * 64];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const mc_f4 b = sums[((cell * value_tiles + min((int)blockIdx.z * 4 + m, value_tiles - 1)) * KT + u) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[m] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[e], (double)b[e], sum[m], 0, 0, 0);
        }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int column = (blockIdx.z * 4 + m) * 16 + r;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = block * BC + 4 * e + g;
            if (t < n && column < value_dim) {
                float* o = out + (token0 + t) * heads * value_dim + (size_t)head * value_dim + column;
                *o = (float)((double)*o + sum[m][e]);
            }
        }
    }
}

}  // namespace

LSA_EXPORT int lsa_gated_pair_update(float* x, const void* gates, int gates_code, int gate_width, const void* y1, int y1_code, const float* s1,
                                     const void* y2, int y2_code, const float* s2, const float* next_weight, float eps, void* normed,
                                     int normed_code, int n, int width, hipStream_t stream) {
    if (n <= 0) return 0;
    if (gate_width != (y2 ? 2 * width : width) || (y2 && !s2) || (next_weight && !normed)) return -1;
    if (!y2) y2_code = 0;
#define LSA_LAUNCH_R(G, Y1, Y2, N, R) gated_pair_update_kernel<G, Y1, Y2, N, R><<<n, 256, 0, stream>>>(x, (const G*)gates, gate_width, (const Y1*)y1, s1, \
        (const Y2*)y2, s2, next_weight, eps, (N*)normed, width)
#define LSA_LAUNCH(G, Y1, Y2, N) do { if (width <= 1024) LSA_LAUNCH_R(G, Y1, Y2, N, 4); else if (width <= 2048) LSA_LAUNCH_R(G, Y1, Y2, N, 8); \
                                      else if (width <= 256 * UPDATE_COLS) LSA_LAUNCH_R(G, Y1, Y2, N, UPDATE_COLS); else LSA_LAUNCH_R(G, Y1, Y2, N, 0); } while (0)
#define LSA_BY_N(G, Y1, Y2) do { if (normed_code) LSA_LAUNCH(G, Y1, Y2, bf16_t); else LSA_LAUNCH(G, Y1, Y2, float); } while (0)
#define LSA_BY_Y2(G, Y1) do { if (y2_code) LSA_BY_N(G, Y1, bf16_t); else LSA_BY_N(G, Y1, float); } while (0)
#define LSA_BY_Y1(G) do { if (y1_code) LSA_BY_Y2(G, bf16_t); else LSA_BY_Y2(G, float); } while (0)
    if (gates_code) LSA_BY_Y1(bf16_t); else LSA_BY_Y1(float);
#undef LSA_BY_Y1
#undef LSA_BY_Y2
#undef LSA_BY_N
#undef LSA_LAUNCH
#undef LSA_LAUNCH_R
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_differential_heads(int code, const void* attended, float lam, float keep, float eps, void* out, int n, int kv_heads,
                                      int group, int value_dim, int row, hipStream_t stream) {
    if (n <= 0) return 0;
    if (value_dim > row || kv_heads < 1 || group < 1) return -1;
    dim3 grid(n, kv_heads * group);
    if (code) differential_heads_kernel<bf16_t><<<grid, 64, 0, stream>>>((const bf16_t*)attended, lam, keep, eps, (bf16_t*)out, group, value_dim, row);
    else differential_heads_kernel<float><<<grid, 64, 0, stream>>>((const float*)attended, lam, keep, eps, (float*)out, group, value_dim, row);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_delta_most_dim() { return MOST_DIM; }
LSA_EXPORT int lsa_delta_state_columns() { return BLOCK_COLUMNS; }

LSA_EXPORT int lsa_delta_prepare(int code, const void* proj, long stride, const float* w, int taps, float* state, long state_stride,
                                 const int* slots, const int* token_row, const int* positions, const int* row_start, float* out,
                                 int kv_heads, int heads, int dim, int value_dim, float q_scale, float unit_eps, int keep,
                                 const void* strength, long strength_stride, const void* decay, long decay_stride, int per_channel,
                                 const float* decay_scale, const float* decay_bias, float* out_strength, float* out_decay, int n,
                                 hipStream_t stream) {
    if (n <= 0) return 0;
    if (taps < 1 || dim < 1 || dim > MOST_DIM || heads < 1 || kv_heads < 1 || heads % kv_heads || (taps > 1 && (!state || !slots))) return -1;
    const int blocks = 2 * kv_heads + 2 * heads;
    const bool pieces = dim % 8 == 0 && value_dim % 8 == 0 && dim <= 128 && value_dim <= 128 && stride % 8 == 0 && state_stride % 4 == 0
        && (!per_channel || decay_stride % 4 == 0) && (long)n * blocks < 0x7fffffffL
        && ((size_t)proj | (size_t)w | (size_t)state | (size_t)out | (per_channel ? (size_t)decay | (size_t)decay_bias | (size_t)out_decay : 0)) % 16 == 0;
    if (pieces && taps >= 2 && taps <= 4) {
        const unsigned workgroups = (unsigned)(((long)n * blocks + 15) / 16);
#define LSA_LAUNCH(T, TAPS) delta_prepare_wide_kernel<T, TAPS><<<workgroups, 256, 0, stream>>>((const T*)proj, stride, w, state, state_stride, slots, token_row, \
        positions, row_start, out, kv_heads, heads, dim, value_dim, q_scale, unit_eps, keep, (const T*)strength, strength_stride, decay, decay_stride, per_channel, \
        decay_scale, decay_bias, out_strength, out_decay, n)
        if (taps == 2) { if (code) LSA_LAUNCH(bf16_t, 2); else LSA_LAUNCH(float, 2); }
        else if (taps == 3) { if (code) LSA_LAUNCH(bf16_t, 3); else LSA_LAUNCH(float, 3); }
        else { if (code) LSA_LAUNCH(bf16_t, 4); else LSA_LAUNCH(float, 4); }
#undef LSA_LAUNCH
        LSA_LAUNCH_CHECK();
    }
    dim3 grid(n, blocks);
#define LSA_LAUNCH(T) delta_prepare_kernel<T><<<grid, 64, 0, stream>>>((const T*)proj, stride, w, taps, state, state_stride, slots, token_row, positions, \
        row_start, out, kv_heads, heads, dim, value_dim, q_scale, unit_eps, keep, (const T*)strength, strength_stride, decay, decay_stride, \
        per_channel, decay_scale, decay_bias, out_strength, out_decay)
    if (code) LSA_LAUNCH(bf16_t); else LSA_LAUNCH(float);
#undef LSA_LAUNCH
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_delta_conv_keep(int code, const void* proj, long stride, float* state, long state_stride, const int* slots,
                                   const int* row_start, const int* row_len, const int* row_ctx, int kept, int channels, int rows,
                                   hipStream_t stream) {
    if (rows <= 0 || kept <= 0) return 0;
    dim3 grid(rows, (channels + 255) / 256);
    if (code) delta_conv_keep_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)proj, stride, state, state_stride, slots, row_start, row_len, row_ctx, kept, channels);
    else delta_conv_keep_kernel<float><<<grid, 256, 0, stream>>>((const float*)proj, stride, state, state_stride, slots, row_start, row_len, row_ctx, kept, channels);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_delta_rule(const float* prepared, const float* strength, const float* decay, int per_channel, float* state,
                              long state_stride, const int* slots, const int* row_start, const int* row_len, const int* row_ctx,
                              float* out, int rows, int heads, int kv_heads, int dim, int value_dim, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > MOST_DIM || heads < 1 || kv_heads < 1 || heads % kv_heads || value_dim < 1 || !state) return -1;
    dim3 grid(rows, heads, (value_dim + BLOCK_COLUMNS - 1) / BLOCK_COLUMNS);
    if (state_stride < (long)heads * grid.z * dim * BLOCK_COLUMNS || state_stride % 4 || ((size_t)state % 16)) return -1;
    const int parts = (dim + PARTS - 1) / PARTS;
#define LSA_LAUNCH(DP, PC) delta_rule_kernel<DP, PC><<<grid, 256, 0, stream>>>(prepared, strength, decay, state, state_stride, slots, row_start, \
        row_len, row_ctx, out, heads, kv_heads, dim, value_dim)
#define LSA_BY_DP(PC) do { if (parts <= 1) LSA_LAUNCH(1, PC); else if (parts <= 2) LSA_LAUNCH(2, PC); else if (parts <= 4) LSA_LAUNCH(4, PC); \
                           else if (parts <= 8) LSA_LAUNCH(8, PC); else LSA_LAUNCH(16, PC); } while (0)
    if (per_channel) LSA_BY_DP(true); else LSA_BY_DP(false);
#undef LSA_BY_DP
#undef LSA_LAUNCH
    LSA_LAUNCH_CHECK();
}

// The same in chunks.  items is no less than the number of chunks of 64 tokens that the rows have together; scratch is the caller's,
// [items][heads] times lsa_delta_chunk_floats.
LSA_EXPORT int lsa_delta_chunked_most_dim() { return CHUNKED_MOST_DIM; }

LSA_EXPORT int lsa_delta_chunk_floats(int dim, int value_dim) {
    const int P = dim <= 64 ? 64 : 128;
    return (value_dim + 15) / 16 * 16 * P + P * P + MC * P;
}

// Once, when the library has been loaded and before any launch (a launch may be recorded into a graph): lets the kernel ask for more
// dynamic LDS than the default limit.
LSA_EXPORT int lsa_delta_allow_lds() {
    hipError_t first = hipSuccess;
#define LSA_ALLOW(P, PC) do { \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&delta_chunk_kernel<P, PC>), hipFuncAttributeMaxDynamicSharedMemorySize, \
                                                 (int)sizeof(DeltaChunkLds<P>)); \
        if (e != hipSuccess && first == hipSuccess) first = e; \
    } while (0)
    LSA_ALLOW(64, false); LSA_ALLOW(64, true); LSA_ALLOW(128, false); LSA_ALLOW(128, true);
#undef LSA_ALLOW
    (void)hipGetLastError();
    return (int)first;
}

template <int P>
static void run_delta_chunks(const float* prepared, const float* strength, const float* decay, int per_channel, float* state, long state_stride,
                             const int* slots, const int* row_start, const int* row_len, const int* row_ctx, float* out, int rows, int heads,
                             int kv_heads, int dim, int value_dim, float* scratch, int items, hipStream_t stream) {
    static_assert(sizeof(DeltaChunkLds<P>) <= 160 * 1024, "a CU has 160 KB of LDS");
    const int blocks = (value_dim + 15) / 16;
    const size_t cells = (size_t)items * heads;
    mc_f4* sums = reinterpret_cast<mc_f4*>(scratch);
    mc_f4* steps = sums + cells * blocks * (16 * P / 4);
    mc_f4* queries = steps + cells * (P * P / 4);
    const dim3 grid(items, heads, (P / 16 + blocks + CHUNK_TILES - 1) / CHUNK_TILES);
#define LSA_LAUNCH(PC) delta_chunk_kernel<P, PC><<<grid, 512, sizeof(DeltaChunkLds<P>), stream>>>(prepared, strength, decay, row_start, row_len, row_ctx, rows, \
        sums, steps, queries, out, heads, kv_heads, dim, value_dim)
    if (per_channel) LSA_LAUNCH(true); else LSA_LAUNCH(false);
#undef LSA_LAUNCH
    delta_chunk_walk_kernel<P><<<dim3(rows, heads, blocks), 256, 0, stream>>>(sums, steps, state, state_stride, slots, row_len, row_ctx, heads, dim, value_dim);
    delta_chunk_read_kernel<P><<<dim3(items, heads, (blocks + 3) / 4), 256, 0, stream>>>(sums, queries, row_start, row_len, row_ctx, rows, out, heads, value_dim);
}

LSA_EXPORT int lsa_delta_rule_chunked(const float* prepared, const float* strength, const float* decay, int per_channel, float* state,
                                      long state_stride, const int* slots, const int* row_start, const int* row_len, const int* row_ctx,
                                      float* out, int rows, int heads, int kv_heads, int dim, int value_dim, float* scratch, int items,
                                      hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > CHUNKED_MOST_DIM || heads < 1 || kv_heads < 1 || heads % kv_heads || value_dim < 1 || !state) return -1;
    if (items <= 0 || !scratch || (size_t)scratch % 16 || (size_t)state % 16 || state_stride % 4) return -1;
    if (state_stride < (long)heads * ((value_dim + 15) / 16) * dim * BLOCK_COLUMNS) return -1;
    if (dim <= 64) run_delta_chunks<64>(prepared, strength, decay, per_channel, state, state_stride, slots, row_start, row_len, row_ctx, out, rows, heads,
                                        kv_heads, dim, value_dim, scratch, items, stream);
    else run_delta_chunks<128>(prepared, strength, decay, per_channel, state, state_stride, slots, row_start, row_len, row_ctx, out, rows, heads,
                               kv_heads, dim, value_dim, scratch, items, stream);
    LSA_LAUNCH_CHECK();
}
