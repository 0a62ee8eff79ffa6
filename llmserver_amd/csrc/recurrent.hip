// Kernels of the mixers that carry a state of fixed size from token to token: the mix of a token's row with the row
// before it, the linear recurrence S_t = diag(d_t) S_(t-1) + k_t v_t^T with its read-out, the recurrences with one decay
// per head (the matrix memory with exponential gates and a normaliser; the plain S_t = a_t S_(t-1) + b_t k_t v_t^T), and the
// per-head norm and gate behind them.  Decays, their exponentials and logarithms, the state, the sums and the norm are float32; projections
// arrive in the activations' type and are widened where they are read; a result for a 16-bit consumer is rounded once.
#include "common.hpp"
#include <type_traits>
#include "chunks.hpp"

using namespace lsa;

// out[m][t] = h[t] + (before[t] - h[t]) * mu[m], before[t] = the row of the token before t in its request: a row of this
// step, the request's state for a row's first token, zeros at position 0.  grid (tokens, blocks of 256 V columns): a thread
// has V neighbouring columns of one token (one where the width or an address is no multiple of 16 bytes), so its two loads are the only ones it waits for.  keep (only in steps of one token per
// row, where a column of a row's state is one thread's): the state becomes this token's row.  2,048 tokens of 2,048 columns in five mixes, us: a column a
// thread 28.9, eight 13.2.
template <typename T, int V>
__global__ __launch_bounds__(256) void token_shift_kernel(const T* __restrict__ h, const float* __restrict__ mu, int mixes,
                                                          float* state, long state_stride, const int* __restrict__ slots,
                                                          const int* __restrict__ token_row, const int* __restrict__ positions,
                                                          const int* __restrict__ row_start, T* __restrict__ out, int n_tokens, int width,
                                                          int keep) {
    const int t = blockIdx.x;
    const int row = token_row[t];
    const bool first_of_sequence = positions[t] == 0, first_of_row = t == row_start[row];
    float* mine = state + (size_t)slots[row] * state_stride;
    const int c = (blockIdx.y * blockDim.x + threadIdx.x) * V;
    if (c >= width) return;
    struct alignas(V * sizeof(T) >= 16 ? 16 : sizeof(T)) Few { T v[V]; };
    struct alignas(V * sizeof(float) >= 16 ? 16 : sizeof(float)) Floats { float v[V]; };
    const Few here = *reinterpret_cast<const Few*>(h + (size_t)t * width + c);
    float own[V], difference[V];
#pragma unroll
    for (int k = 0; k < V; ++k) own[k] = (float)here.v[k];
    if (first_of_sequence) {
#pragma unroll
        for (int k = 0; k < V; ++k) difference[k] = 0.f - own[k];
    } else if (first_of_row) {
#pragma unroll
        for (int k = 0; k < V; ++k) difference[k] = mine[c + k] - own[k];
    } else {
        const Few last = *reinterpret_cast<const Few*>(h + (size_t)(t - 1) * width + c);
#pragma unroll
        for (int k = 0; k < V; ++k) difference[k] = (float)last.v[k] - own[k];
    }
#pragma unroll 5
    for (int m = 0; m < mixes; ++m) {
        const Floats share = *reinterpret_cast<const Floats*>(mu + (size_t)m * width + c);
        Few mixed;
#pragma unroll
        for (int k = 0; k < V; ++k) mixed.v[k] = (T)(own[k] + difference[k] * share.v[k]);
        *reinterpret_cast<Few*>(out + ((size_t)m * n_tokens + t) * width + c) = mixed;
    }
    if (keep) {
#pragma unroll
        for (int k = 0; k < V; ++k) mine[c + k] = own[k];
    }
}

// state[slot] = the last row of every row of the step (rows without tokens keep theirs).
template <typename T>
__global__ __launch_bounds__(256) void token_shift_keep_kernel(const T* __restrict__ h, float* __restrict__ state, long state_stride,
                                                               const int* __restrict__ slots, const int* __restrict__ row_start,
                                                               const int* __restrict__ row_len, int width) {
    const int row = blockIdx.x;
    const int c = blockIdx.y * blockDim.x + threadIdx.x;
    const int count = row_len[row];
    if (c >= width || count <= 0) return;
    state[(size_t)slots[row] * state_stride + c] = (float)h[(size_t)(row_start[row] + count - 1) * width + c];
}

// The decay of a key channel from its 32-bit logit.  mode 0: sigmoid(z)^(1 / tau) = exp(log sigmoid(z) / tau);
// mode 1: exp(-exp(z)).
__device__ __forceinline__ float decay_of(float z, int mode, float inv_tau) {
    if (mode == 0) {
        const float log_sigmoid = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
        return expf(log_sigmoid * inv_tau);
    }
    return expf(-expf(z));
}

// One token of one wavefront's DK channels: the state's update and the channels' part of the read-out.  The channels come
// from LDS four at a time (16-byte broadcast reads: every row of a chunk and every wavefront's first channel lie at
// multiples of 32 bytes); four partial sums of the read-out make its chain of dependent multiply-adds a quarter as long.
template <int DK, bool BONUS>
__device__ __forceinline__ float recurrence_token(float (&S)[DK], const float (&u)[DK], const float* q_row, const float* k_row,
                                                  const float* d_row, float value) {
    const float4* tq = reinterpret_cast<const float4*>(q_row);
    const float4* tk = reinterpret_cast<const float4*>(k_row);
    const float4* td = reinterpret_cast<const float4*>(d_row);
    float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i4 = 0; i4 < DK / 4; ++i4) {
        const float4 q4 = tq[i4], k4 = tk[i4], d4 = td[i4];
        const float qs[4] = {q4.x, q4.y, q4.z, q4.w}, ks[4] = {k4.x, k4.y, k4.z, k4.w}, ds[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 4 * i4 + e;
            const float kv = ks[e] * value;
            if (BONUS) {
                o4[e] = __builtin_fmaf(__builtin_fmaf(u[i], kv, S[i]), qs[e], o4[e]);
                S[i] = __builtin_fmaf(ds[e], S[i], kv);
            } else {
                S[i] = __builtin_fmaf(ds[e], S[i], kv);
                o4[e] = __builtin_fmaf(S[i], qs[e], o4[e]);
            }
        }
    }
    return (o4[0] + o4[1]) + (o4[2] + o4[3]);
}

// grid (rows, heads, blocks of 64 value columns); a workgroup of NW wavefronts walks the row's tokens in order.
// Lane = value column; wavefront w (of up to eight) owns key channels [w * DK, (w + 1) * DK) and keeps its DK x 64 piece of the head's
// state in registers, so the state is read once before the row's first token and written once after its last one.
// The tokens go through LDS in chunks of CHUNK: queries (scaled), keys and decays of the head, widened and, for the
// decays, exponentiated once per (token, channel) by whichever thread loads them; the chunk's values of this block of
// columns; and, per wavefront, the partial read-outs of its channels, which are added up over the wavefronts when the
// chunk is through.  A wavefront reads its channels of a token from LDS as broadcasts; nothing crosses lanes.
//   BONUS false: S = d S + k v^T, then o = S^T q.      BONUS true: o = (S + (u k) v^T)^T q, then S = d S + k v^T.
// Every sum is formed in the same order whatever the step's other rows and however the sequence was cut into steps:
// the state after a token and the token's read-out are the same bits either way.
constexpr int CHUNK = 16;

template <typename T, int DK, bool BONUS>
__global__ __launch_bounds__(512) void linear_recurrence_kernel(const T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride,
                                         const T* __restrict__ v, long v_stride, const float* __restrict__ decay,
                                         const float* __restrict__ decay_bias, int mode, float inv_tau, const float* __restrict__ bonus,
                                         float q_scale, float* state, long state_stride, const int* __restrict__ slots,
                                         const int* __restrict__ row_start, const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                         float* __restrict__ out, int heads, int dim, int value_dim) {
    extern __shared__ __align__(16) float lds[];
    const int row = blockIdx.x, head = blockIdx.y, column0 = blockIdx.z * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int count = row_len[row];
    if (count <= 0) return;                              // (the whole workgroup: nobody waits at a barrier below)
    const int start = row_start[row], first_position = row_ctx[row] - count;
    const int padded = waves * DK;                       // channels as the wavefronts share them; those behind dim are zeros
    float* s_q = lds;                                    // [CHUNK][padded]
    float* s_k = s_q + CHUNK * padded;
    float* s_d = s_k + CHUNK * padded;
    float* s_v = s_d + CHUNK * padded;                   // [CHUNK][64]
    float* s_o = s_v + CHUNK * 64;                       // [waves][CHUNK][64]
    const int column = column0 + lane;
    const bool column_ok = column < value_dim;
    const int channel0 = wave * DK;
    float* mine = state + (size_t)slots[row] * state_stride + ((size_t)head * dim + channel0) * value_dim + column;
    float S[DK], u[DK];
#pragma unroll
    for (int i = 0; i < DK; ++i) {
        const bool ok = column_ok && channel0 + i < dim;
        S[i] = (ok && first_position > 0) ? mine[(size_t)i * value_dim] : 0.f;
        u[i] = (BONUS && channel0 + i < dim) ? bonus[(size_t)head * dim + channel0 + i] : 0.f;
    }
    const size_t key_column = (size_t)head * dim;
    for (int t0 = 0; t0 < count; t0 += CHUNK) {
        const int n = min(CHUNK, count - t0);
        __syncthreads();                                 // the chunk before has been read out of LDS
        // A thread stages PER numbers of each kind (CHUNK * padded = PER * blockDim.x): all their loads first, so that they are
        // in flight together, then the decays' exponentials and the stores.
        constexpr int PER = CHUNK * DK / 64;
        float raw_q[PER], raw_k[PER], raw_z[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = threadIdx.x + j * blockDim.x;
            const int t = i / padded, c = i - t * padded;
            raw_q[j] = 0.f; raw_k[j] = 0.f; raw_z[j] = 0.f;
            if (t < n && c < dim) {
                const size_t token = (size_t)(start + t0 + t);
                raw_q[j] = (float)q[token * q_stride + key_column + c];
                raw_k[j] = (float)k[token * k_stride + key_column + c];
                raw_z[j] = decay[token * (size_t)heads * dim + key_column + c] + (decay_bias ? decay_bias[key_column + c] : 0.f);
            }
        }
        for (int i = threadIdx.x; i < n * 64; i += blockDim.x) {
            const int t = i >> 6, c = column0 + (i & 63);
            s_v[i] = c < value_dim ? (float)v[(size_t)(start + t0 + t) * v_stride + (size_t)head * value_dim + c] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = threadIdx.x + j * blockDim.x;
            const int t = i / padded, c = i - t * padded;
            if (t >= n) continue;
            s_q[i] = raw_q[j] * q_scale;
            s_k[i] = raw_k[j];
            s_d[i] = c < dim ? decay_of(raw_z[j], mode, inv_tau) : 1.f;
        }
        __syncthreads();
        if (DK <= 16 && n == CHUNK) {
            // A whole chunk: the tokens' steps unrolled, their read-outs kept in registers and stored behind the last one, so
            // that no store to LDS stands between one token's loads and the next one's and the loads can run ahead.  (With
            // more channels a wavefront the state alone fills the registers, and running ahead would spill.)
            float kept[CHUNK];
#pragma unroll
            for (int t = 0; t < CHUNK; ++t)
                kept[t] = recurrence_token<DK, BONUS>(S, u, s_q + t * padded + channel0, s_k + t * padded + channel0,
                                                      s_d + t * padded + channel0, s_v[t * 64 + lane]);
#pragma unroll
            for (int t = 0; t < CHUNK; ++t) s_o[(wave * CHUNK + t) * 64 + lane] = kept[t];
        } else {
            for (int t = 0; t < n; ++t)
                s_o[(wave * CHUNK + t) * 64 + lane] = recurrence_token<DK, BONUS>(S, u, s_q + t * padded + channel0, s_k + t * padded + channel0,
                                                                                  s_d + t * padded + channel0, s_v[t * 64 + lane]);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n * 64; i += blockDim.x) {
            const int t = i >> 6, c = i & 63;
            if (column0 + c >= value_dim) continue;
            float total = 0.f;
            for (int w = 0; w < waves; ++w) total += s_o[(w * CHUNK + t) * 64 + c];
            out[(size_t)(start + t0 + t) * heads * value_dim + (size_t)head * value_dim + column0 + c] = total;
        }
    }
#pragma unroll
    for (int i = 0; i < DK; ++i)
        if (column_ok && channel0 + i < dim) mine[(size_t)i * value_dim] = S[i];
}

// grid (tokens, heads), one wavefront: out = x' / rms(x') * w * act(gate) over a head's value_dim numbers; x float32,
// w = weight[head * weight_stride + j] (weight_stride 0: one weight shared by the heads; no weight: 1), gate and out of type T;
// act: gate * sigmoid(gate) (gate_kind 0) or sigmoid(gate) (1).  x' = x, or, with below [tokens][heads][2]:
// x / (max(|below[0]|, below[1]) + floor), the read-out of a matrix memory under its normaliser.
template <typename T>
__global__ __launch_bounds__(64) void heads_norm_gate_kernel(const float* __restrict__ x, const float* __restrict__ weight, int weight_stride,
                                                             float eps, const T* __restrict__ gate, long gate_stride, T* __restrict__ out,
                                                             int heads, int value_dim, int gate_kind, const float* __restrict__ below,
                                                             float floor) {
    const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
    const float* row = x + ((size_t)t * heads + head) * value_dim;
    float under = 1.f;
    if (below) {
        const float* b = below + ((size_t)t * heads + head) * 2;
        under = fmaxf(fabsf(b[0]), b[1]) + floor;
    }
    float sq = 0.f;
    for (int j = lane; j < value_dim; j += 64) {
        const float xv = below ? row[j] / under : row[j];
        sq += xv * xv;
    }
    const float inv = rsqrtf(wave_sum(sq) / (float)value_dim + eps);
    const T* g = gate + (size_t)t * gate_stride + (size_t)head * value_dim;
    const float* w = weight ? weight + (size_t)head * weight_stride : nullptr;
    T* o = out + ((size_t)t * heads + head) * value_dim;
    for (int j = lane; j < value_dim; j += 64) {
        const float gv = (float)g[j];
        const float sigmoid = 1.f / (1.f + expf(-gv));
        const float xv = below ? row[j] / under : row[j];
        o[j] = (T)(xv * inv * (w ? w[j] : 1.f) * (gate_kind ? sigmoid : gv * sigmoid));
    }
}

// The same for rows at multiples of 16 bytes and heads of up to 128 C numbers: sixteen lanes a (token, head), eight neighbouring
// numbers a lane, sixteen heads a workgroup.  With two numbers a lane what is around them takes longer than they do: 2,048 tokens of 16 heads of
// 128 16.6 us, 10.3 so; with the read-out's denominators (2,001 tokens of 16 heads of 256) 29.7, 19.2; one token of 16 heads 2.9, 2.5; 32 tokens of 8 of 256 4.9, 4.0.
template <typename T, int C>
__global__ __launch_bounds__(256) void heads_norm_gate_eights_kernel(const float* __restrict__ x, const float* __restrict__ weight, int weight_stride,
                                                                   float eps, const T* __restrict__ gate, long gate_stride, T* __restrict__ out,
                                                                   int heads, int value_dim, int gate_kind, const float* __restrict__ below,
                                                                   float floor, int pairs) {
    const int index = (int)blockIdx.x * 16 + (threadIdx.x >> 4), first = 8 * (threadIdx.x & 15);
    const int pair = min(index, pairs - 1), t = pair / heads, head = pair - t * heads;
    struct alignas(16) Eight { float4 low, high; };
    struct alignas(16) Gates { T v[8]; };
    const float* row = x + (size_t)pair * value_dim;
    const T* g = gate + (size_t)t * gate_stride + (size_t)head * value_dim;
    float v[C][8];
    Gates gates[C];
    float sq = 0.f, under = 1.f;
    if (below) under = fmaxf(fabsf(below[(size_t)pair * 2]), below[(size_t)pair * 2 + 1]) + floor;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int j = first + 128 * c;
        if (j < value_dim) {
            const Eight here = *reinterpret_cast<const Eight*>(row + j);
            gates[c] = *reinterpret_cast<const Gates*>(g + j);
            const float eight[8] = {here.low.x, here.low.y, here.low.z, here.low.w, here.high.x, here.high.y, here.high.z, here.high.w};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[c][k] = below ? eight[k] / under : eight[k];
                sq += v[c][k] * v[c][k];
            }
        }
    }
    const auto across = [](float value, auto control) {
        return value + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(value), decltype(control)::value, 0xf, 0xf, true));
    };
    sq = across(sq, std::integral_constant<int, 0xB1>());          // quad_perm [1, 0, 3, 2]
    sq = across(sq, std::integral_constant<int, 0x4E>());          // quad_perm [2, 3, 0, 1]
    sq = across(sq, std::integral_constant<int, 0x141>());         // row_half_mirror
    sq = across(sq, std::integral_constant<int, 0x140>());         // row_mirror
    if (index >= pairs) return;
    const float inv = rsqrtf(sq / (float)value_dim + eps);
    const float* w = weight ? weight + (size_t)head * weight_stride : nullptr;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int j = first + 128 * c;
        if (j < value_dim) {
            float scale[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
            if (w) {
                const Eight here = *reinterpret_cast<const Eight*>(w + j);
                scale[0] = here.low.x; scale[1] = here.low.y; scale[2] = here.low.z; scale[3] = here.low.w;
                scale[4] = here.high.x; scale[5] = here.high.y; scale[6] = here.high.z; scale[7] = here.high.w;
            }
            Gates result;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float gv = (float)gates[c].v[k], sigmoid = 1.f / (1.f + expf(-gv));
                result.v[k] = (T)(v[c][k] * inv * scale[k] * (gate_kind ? sigmoid : gv * sigmoid));
            }
            *reinterpret_cast<Gates*>(out + (size_t)pair * value_dim + j) = result;
        }
    }
}

// ---- a matrix memory with exponential gates --------------------------------------------------------------------------
// Per head and token: log input gate i = cap tanh(z_i / cap), log forget gate f = logsigmoid(cap tanh(z_f / cap)), a running
// maximum m_t = max(f + m_(t-1), i) (0 in front of the first token), and from them what the memory's update needs: keep = exp(f + m_(t-1) -
// m_t), take = exp(i - m_t), and exp(-m_t) for the read-out's denominator.  grid (rows, heads), eight wavefronts: the row's
// tokens 448 at a time; seven wavefronts have a thread a token for the transcendental functions, one thread of the eighth
// walks the maximum through the tokens (two dependent instructions a token), and while it walks a group the others
// prepare the group behind it and finish the group before it.  gates [T][2 heads] (inputs, then forgets), coef [T][heads][2] (keep, take),
// below [T][heads][2] (its second number is written here), top[slot][head] the maximum between steps (0 at position 0).
// run (or nullptr) [T][heads]: the sum of log keep from the first token of a token's chunk of 64 (counted from the row's
// first token of this step) up to the token itself, in 64-bit: what the chunked form of the memory forms its weights from.
constexpr int GATES_WAVES = 8;            // the first walks, the others work: seven chunks of 64 tokens at a time
__global__ __launch_bounds__(64 * GATES_WAVES) void memory_gates_kernel(const float* __restrict__ gates, float cap, float* state, long state_stride,
                                                          long top_offset, const int* __restrict__ slots, const int* __restrict__ row_start,
                                                          const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                                          float* __restrict__ coef, float* __restrict__ below, int heads,
                                                          double* __restrict__ run) {
    constexpr int GROUP = 64 * (GATES_WAVES - 1);                      // tokens at a time: a working wavefront a chunk of 64
    // two of each: while one group's maxima are walked, the group behind it is prepared and the group before it finished
    __shared__ __align__(16) float s_in[2][GROUP], s_forget[2][GROUP], s_top[2][GROUP + 8];                 // (the maximum in front of a group's token t at [3 + t], behind it at [4 + t]: sixteen bytes at a time)
    const int row = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int count = row_len[row];
    if (count <= 0) return;
    const int start = row_start[row], first_position = row_ctx[row] - count;
    float* kept = state + (size_t)slots[row] * state_stride + top_offset + head;
    const float inv_cap = 1.f / cap;
    const int groups = (count + GROUP - 1) / GROUP;
    const bool walker = tid < 64;
    const int mine = tid - 64;                                         // a worker's token of a group
    float m = 0.f;                                                     // (the walker's: the maximum so far)
    if (tid == 0) m = first_position > 0 ? *kept : 0.f;
    // what a worker keeps of its token of the group that is being walked, until the maxima are there
    float log_in = 0.f, log_forget = 0.f;
    auto prepare = [&](int g) {                                        // caps and logarithms of group g's gates
        const int n = min(GROUP, count - g * GROUP);
        log_in = 0.f; log_forget = 0.f;
        if (mine < n) {
            const size_t token = (size_t)(start + g * GROUP + mine);
            log_in = cap * tanhf(gates[token * 2 * heads + head] * inv_cap);
            const float z = cap * tanhf(gates[token * 2 * heads + heads + head] * inv_cap);
            log_forget = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
        }
        s_in[g & 1][mine] = log_in;
        s_forget[g & 1][mine] = log_forget;
    };
    auto finish = [&](int g, float li, float lf) {                     // group g's coefficients, from its maxima
        const int n = min(GROUP, count - g * GROUP);
        const size_t token = (size_t)(start + g * GROUP + mine);
        float log_keep = 0.f;
        if (mine < n) {
            const float before = s_top[g & 1][3 + mine], now = s_top[g & 1][4 + mine];
            log_keep = (lf + before) - now;
            coef[(token * heads + head) * 2] = expf(log_keep);
            coef[(token * heads + head) * 2 + 1] = expf(li - now);
            below[(token * heads + head) * 2 + 1] = expf(-now);
        }
        if (run != nullptr) {                                          // the chunk's running sum of log keep, token by token
            double total = (double)log_keep;
#pragma unroll
            for (int step = 1; step < 64; step <<= 1) {
                const double other = __shfl_up(total, step, 64);
                if (lane >= step) total += other;
            }
            if (mine < n) run[token * heads + head] = total;
        }
    };
    if (!walker) prepare(0);
    __syncthreads();
    float walked_in = 0.f, walked_forget = 0.f;                        // a worker's token of the group that is being walked
    for (int g = 0; g < groups; ++g) {
        if (walker) {
            if (tid == 0) {                                            // the walk: one thread, two dependent instructions a token
                const int n = min(GROUP, count - g * GROUP);
                const float* fs_all = s_forget[g & 1];
                const float* is_all = s_in[g & 1];
                float* tops = s_top[g & 1];
                tops[3] = m;
                int t = 0;
                for (; t + 64 <= n; t += 64) {                         // a whole chunk: all loads first, then the chain alone
                    float fs[64], is[64], ms[64];
#pragma unroll
                    for (int t4 = 0; t4 < 16; ++t4) {
                        const float4 f4 = reinterpret_cast<const float4*>(fs_all + t)[t4], i4 = reinterpret_cast<const float4*>(is_all + t)[t4];
                        fs[4 * t4] = f4.x; fs[4 * t4 + 1] = f4.y; fs[4 * t4 + 2] = f4.z; fs[4 * t4 + 3] = f4.w;
                        is[4 * t4] = i4.x; is[4 * t4 + 1] = i4.y; is[4 * t4 + 2] = i4.z; is[4 * t4 + 3] = i4.w;
                    }
#pragma unroll
                    for (int u = 0; u < 64; ++u) {
                        m = fmaxf(fs[u] + m, is[u]);
                        ms[u] = m;
                    }
#pragma unroll
                    for (int u4 = 0; u4 < 16; ++u4)
                        reinterpret_cast<float4*>(tops + 4 + t)[u4] = make_float4(ms[4 * u4], ms[4 * u4 + 1], ms[4 * u4 + 2], ms[4 * u4 + 3]);
                }
                for (; t < n; ++t) {
                    m = fmaxf(fs_all[t] + m, is_all[t]);
                    tops[4 + t] = m;
                }
            }
        } else {
            const float li = walked_in, lf = walked_forget;            // (group g - 1's, whose maxima are there)
            walked_in = log_in; walked_forget = log_forget;            // (group g's, which is being walked)
            if (g + 1 < groups) prepare(g + 1);
            if (g > 0) finish(g - 1, li, lf);
        }
        __syncthreads();
    }
    if (!walker) finish(groups - 1, walked_in, walked_forget);
    if (tid == 0) *kept = m;
}

// ---- recurrences with one decay per head: S_t = keep_t S_(t-1) + take_t k_t v_t^T, o_t = S_t^T q_t -------------------------
// Where a token's two numbers of a head come from: pairs (keep, take) that another kernel has made (the matrix memory's
// gates), or the logarithm of keep, per token and head or (log_stride 0) per head, with take per token and head or 1.
struct DecayWeights {
    const float* coef;                   // [T][heads][2], or nullptr: the two below
    const float* log_keep;               // [T][heads] (log_stride = heads) or [heads] (log_stride = 0)
    long log_stride;
    const float* take;                   // [T][heads], or nullptr: 1
    __device__ __forceinline__ float keep_of(size_t token, int head, int heads) const {
        return coef ? coef[(token * heads + head) * 2] : expf(log_keep[token * log_stride + head]);
    }
    __device__ __forceinline__ float take_of(size_t token, int head, int heads) const {
        return coef ? coef[(token * heads + head) * 2 + 1] : (take ? take[token * heads + head] : 1.f);
    }
};

// One token of one wavefront's DK channels of such a recurrence: S = keep S + k value (value: the token's value column times its
// take), and the channels' part of the read-out S^T q; the channels come from LDS as in recurrence_token.
template <int DK>
__device__ __forceinline__ float memory_token(float (&S)[DK], const float* q_row, const float* k_row, float keep, float value) {
    const float4* tq = reinterpret_cast<const float4*>(q_row);
    const float4* tk = reinterpret_cast<const float4*>(k_row);
    float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i4 = 0; i4 < DK / 4; ++i4) {
        const float4 q4 = tq[i4], k4 = tk[i4];
        const float qs[4] = {q4.x, q4.y, q4.z, q4.w}, ks[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 4 * i4 + e;
            S[i] = __builtin_fmaf(keep, S[i], ks[e] * value);
            o4[e] = __builtin_fmaf(S[i], qs[e], o4[e]);
        }
    }
    return (o4[0] + o4[1]) + (o4[2] + o4[3]);
}

// The memory itself, laid out as linear_recurrence_kernel: grid (rows, heads, blocks of 64 columns), lane = column,
// wavefront w owns key channels [w * DK, (w + 1) * DK) and keeps its piece of the state in registers over the row's tokens.
// Groups of `group` heads share a query and key head.  The columns are the head's value_dim value columns and, with `ones`
// (the matrix memory), behind them one more whose "value" is 1: its piece of the state is the normaliser n, which obeys the same recurrence with k in place of k v^T, and its read-out is n . q.  So
// out [T][heads * value_dim] gets the numerators S^T q and below [T][heads][2] (first number) gets n . q; the division is
// left to the kernel that normalises the heads.  state[slot]: the matrices [heads][dim][value_dim], then the normalisers
// [heads][dim].  Every sum is formed in the same order however the sequence was cut into steps.
template <typename T, typename V, int DK>
__global__ __launch_bounds__(512) void matrix_memory_kernel(const T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride,
                                         const V* __restrict__ v, long v_stride, DecayWeights weights, float q_scale,
                                         float* state, long state_stride, const int* __restrict__ slots,
                                         const int* __restrict__ row_start, const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                         float* __restrict__ out, float* __restrict__ below, int heads, int dim, int value_dim, int group, int ones) {
    extern __shared__ __align__(16) float lds[];
    const int row = blockIdx.x, head = blockIdx.y, column0 = blockIdx.z * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int count = row_len[row];
    if (count <= 0) return;                              // (the whole workgroup: nobody waits at a barrier below)
    const int start = row_start[row], first_position = row_ctx[row] - count;
    const int padded = waves * DK;                       // channels as the wavefronts share them; those behind dim are zeros
    float* s_q = lds;                                    // [CHUNK][padded]
    float* s_k = s_q + CHUNK * padded;
    float* s_v = s_k + CHUNK * padded;                   // [CHUNK][64], each value times its token's take
    float* s_keep = s_v + CHUNK * 64;                    // [CHUNK]
    float* s_o = s_keep + CHUNK;                         // [waves][CHUNK][64]
    const int column = column0 + lane;
    const bool is_value = column < value_dim, is_normaliser = ones && column == value_dim;
    const int channel0 = wave * DK;
    float* slot = state + (size_t)slots[row] * state_stride;
    // a channel's number of this column: in the matrix, or in the normaliser behind the matrices
    float* mine = is_value ? slot + ((size_t)head * dim + channel0) * value_dim + column
                           : slot + (size_t)heads * dim * value_dim + (size_t)head * dim + channel0;
    const size_t channel_stride = is_value ? (size_t)value_dim : 1;
    float S[DK];
#pragma unroll
    for (int i = 0; i < DK; ++i) {
        const bool ok = (is_value || is_normaliser) && channel0 + i < dim;
        S[i] = (ok && first_position > 0) ? mine[(size_t)i * channel_stride] : 0.f;
    }
    const size_t key_column = (size_t)(head / group) * dim;
    for (int t0 = 0; t0 < count; t0 += CHUNK) {
        const int n = min(CHUNK, count - t0);
        __syncthreads();                                 // the chunk before has been read out of LDS
        constexpr int PER = CHUNK * DK / 64;
        float raw_q[PER], raw_k[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = threadIdx.x + j * blockDim.x;
            const int t = i / padded, c = i - t * padded;
            raw_q[j] = 0.f; raw_k[j] = 0.f;
            if (t < n && c < dim) {
                const size_t token = (size_t)(start + t0 + t);
                raw_q[j] = (float)q[token * q_stride + key_column + c];
                raw_k[j] = (float)k[token * k_stride + key_column + c];
            }
        }
        for (int i = threadIdx.x; i < n * 64; i += blockDim.x) {
            const int t = i >> 6, c = column0 + (i & 63);
            const size_t token = (size_t)(start + t0 + t);
            const float take = weights.take_of(token, head, heads);
            const float value = c < value_dim ? (float)v[token * v_stride + (size_t)head * value_dim + c] : (c == value_dim ? 1.f : 0.f);
            s_v[i] = take * value;
        }
        if (threadIdx.x < n) s_keep[threadIdx.x] = weights.keep_of((size_t)(start + t0 + threadIdx.x), head, heads);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = threadIdx.x + j * blockDim.x;
            if (i / padded >= n) continue;
            s_q[i] = raw_q[j] * q_scale;
            s_k[i] = raw_k[j];
        }
        __syncthreads();
        if (DK <= 16 && n == CHUNK) {
            float kept[CHUNK];
#pragma unroll
            for (int t = 0; t < CHUNK; ++t)
                kept[t] = memory_token<DK>(S, s_q + t * padded + channel0, s_k + t * padded + channel0, s_keep[t], s_v[t * 64 + lane]);
#pragma unroll
            for (int t = 0; t < CHUNK; ++t) s_o[(wave * CHUNK + t) * 64 + lane] = kept[t];
        } else {
            for (int t = 0; t < n; ++t)
                s_o[(wave * CHUNK + t) * 64 + lane] = memory_token<DK>(S, s_q + t * padded + channel0, s_k + t * padded + channel0,
                                                                       s_keep[t], s_v[t * 64 + lane]);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < n * 64; i += blockDim.x) {
            const int t = i >> 6, c = column0 + (i & 63);
            if (c >= value_dim + ones) continue;
            float total = 0.f;
            for (int w = 0; w < waves; ++w) total += s_o[(w * CHUNK + t) * 64 + (i & 63)];
            const size_t token = (size_t)(start + t0 + t);
            if (c < value_dim) out[token * heads * value_dim + (size_t)head * value_dim + c] = total;
            else below[(token * heads + head) * 2] = total;
        }
    }
#pragma unroll
    for (int i = 0; i < DK; ++i)
        if ((is_value || is_normaliser) && channel0 + i < dim) mine[(size_t)i * channel_stride] = S[i];
}

// The same for steps of about a token a row, where the state's way through the chip is what there is to do: sixteen lanes have 64 columns, four
// each (16-byte loads and stores of the state), and DK channels as a wavefront above has; a token's queries, keys and values come straight into
// registers behind the state's loads, and the read-outs' partial sums alone go through LDS.  The same sums in the same order as above.  It wants
// value columns in fours, channels in whole DKs and 16-byte pieces at multiples of 16 bytes.
//   us, the walk above and this, cold caches: 64 heads of 128 x 64 in bfloat16, 1 row 6.5, 5.7; 8 rows 12.2, 10.4; 32 rows (134 MB both ways) 37.1, 23.4 (5.7
// TB/s); 128 rows 140, 100; 8 heads of 128 x 256, 32 rows 21.4, 14.8; 32 heads of 64 x 64, 3 rows 5.8, 5.0, 32 rows 12.0, 9.4; 16 of 128 x 128 in
// float32 at 32 rows 21.6, 13.8.  The walk's workgroups hold 53 KB of LDS for tokens that are not there, three a compute unit.
template <typename T, typename V, int DK>
__global__ __launch_bounds__(128) void matrix_memory_single_kernel(const T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride,
                                         const V* __restrict__ v, long v_stride, DecayWeights weights, float q_scale,
                                         float* state, long state_stride, const int* __restrict__ slots,
                                         const int* __restrict__ row_start, const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                         float* __restrict__ out, float* __restrict__ below, int heads, int dim, int value_dim, int group, int ones) {
    struct alignas(sizeof(T) * 8 < 16 ? sizeof(T) * 8 : 16) Eight { T v[8]; };
    struct alignas(sizeof(V) * 4) Four { V v[4]; };
    __shared__ __align__(16) float s_o[8 * 64];
    const int row = blockIdx.x, head = blockIdx.y, column0 = blockIdx.z * 64;
    const int count = row_len[row], start = row_start[row], context = row_ctx[row];
    const size_t place = (size_t)slots[row] * state_stride;
    if (count <= 0) return;                              // (the whole workgroup)
    const int part = threadIdx.x >> 4, parts = dim / DK, channel0 = part * DK;
    const int column = column0 + 4 * (threadIdx.x & 15);
    const bool is_value = column < value_dim, is_normaliser = ones && column == value_dim;
    const bool active = part < parts && (is_value || is_normaliser);
    float* mine = is_value ? state + place + ((size_t)head * dim + channel0) * value_dim + column
                           : state + place + (size_t)heads * dim * value_dim + (size_t)head * dim + channel0;
    float S[DK][4];
#pragma unroll
    for (int i = 0; i < DK; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) S[i][c] = 0.f;
    if (active && context > count) {
        if (is_value) {
#pragma unroll
            for (int i = 0; i < DK; ++i) {
                const float4 s4 = *reinterpret_cast<const float4*>(mine + (size_t)i * value_dim);
                S[i][0] = s4.x; S[i][1] = s4.y; S[i][2] = s4.z; S[i][3] = s4.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < DK; ++i) S[i][0] = mine[i];
        }
    }
    const size_t key_column = (size_t)(head / group) * dim + channel0;
    for (int t = 0; t < count; ++t) {
        const size_t token = (size_t)(start + t);
        float sums[4] = {0.f, 0.f, 0.f, 0.f};
        if (active) {
            Eight q8[DK / 8], k8[DK / 8];
#pragma unroll
            for (int i = 0; i < DK / 8; ++i) {
                q8[i] = *reinterpret_cast<const Eight*>(q + token * q_stride + key_column + 8 * i);
                k8[i] = *reinterpret_cast<const Eight*>(k + token * k_stride + key_column + 8 * i);
            }
            const float take = weights.take_of(token, head, heads), keep = weights.keep_of(token, head, heads);
            float value[4] = {take, 0.f, 0.f, 0.f};      // (the column behind the values is one of ones)
            if (is_value) {
                const Four v4 = *reinterpret_cast<const Four*>(v + token * v_stride + (size_t)head * value_dim + column);
#pragma unroll
                for (int c = 0; c < 4; ++c) value[c] = take * (float)v4.v[c];
            }
            float o[4][4] = {};
#pragma unroll
            for (int i = 0; i < DK; ++i) {
                const float ki = (float)k8[i / 8].v[i % 8], qi = (float)q8[i / 8].v[i % 8] * q_scale;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[i][c] = __builtin_fmaf(keep, S[i][c], ki * value[c]);
                    o[i % 4][c] = __builtin_fmaf(S[i][c], qi, o[i % 4][c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) sums[c] = (o[0][c] + o[1][c]) + (o[2][c] + o[3][c]);
        }
        if (t > 0) __syncthreads();                      // the token before has been read out of LDS
        if (part < parts) *reinterpret_cast<float4*>(s_o + part * 64 + 4 * (threadIdx.x & 15)) = make_float4(sums[0], sums[1], sums[2], sums[3]);
        if (t + 1 == count && active) {
            if (is_value) {
#pragma unroll
                for (int i = 0; i < DK; ++i) *reinterpret_cast<float4*>(mine + (size_t)i * value_dim) = make_float4(S[i][0], S[i][1], S[i][2], S[i][3]);
            } else {
#pragma unroll
                for (int i = 0; i < DK; ++i) mine[i] = S[i][0];
            }
        }
        __syncthreads();
        const int c = column0 + (int)threadIdx.x;
        if (threadIdx.x < 64 && c < value_dim + ones) {
            float total = 0.f;
            for (int w = 0; w < parts; ++w) total += s_o[w * 64 + threadIdx.x];
            if (c < value_dim) out[token * heads * value_dim + (size_t)head * value_dim + c] = total;
            else below[(token * heads + head) * 2] = total;
        }
    }
}

// ---- the same recurrences in chunks -------------------------------------------------------------------------------------
// A row's tokens of a step in chunks of 64, counted from the row's first token of the step.  With L_t the sum of log keep
// from the chunk's first token to t, the state behind token t is e^(L_t) S_0 + sum_(j <= t) e^(L_t - L_j) take_j k_j v_j^T
// (S_0 the state in front of the chunk), and every weight is at most 1.  So (1) every chunk's own sum
// U = sum_j e^(L_last - L_j) take_j k_j v_j^T is a matrix product, all chunks at once; (2) a walk over a row's chunks,
// S <- e^(L_last) S + U, leaves the state in front of every chunk where U stood, and the row's last state in its slot; (3) a
// chunk's read-outs are two products, (scores q_t . k_j times their weights) x values and (e^(L_t) q_t) x S_0, again all
// chunks at once.  With `ones`, one more column behind the values, whose "value" is 1, carries the normaliser as in the scan.  All
// operands are float32 in LDS and the products run on v_mfma_f32_16x16x4_f32; a workgroup of four wavefronts forms 64 x 64
// results, a wavefront 32 x 32 of them.  An item is a (row, chunk): the grid has as many as the step could have at most,
// and a workgroup finds its row by walking the rows' lengths.
// acc += A B over inner indices [0, inner) (a multiple of 16; what lies behind an operand's end is zeros): A's (m, i) at
// a[m * MC_A + i], m counted from the wavefront's first row; B's (i, n) at b[i * b_inner + n * b_column], n counted from the
// wavefront's first column.  acc[mi][ni][e] is the result at row 16 mi + 4 (lane / 16) + e, column 16 ni + lane % 16.
// Sixteen inner indices at a time: their sixteen LDS loads are issued before the first of their sixteen products.
__device__ __forceinline__ void memory_product(mc_f4 (&acc)[2][2], const float* a, const float* b, int b_inner, int b_column, int inner, int lane) {
    const int r = lane & 15, g = lane >> 4;
    const float* a0 = a + r * MC_A + g;
    const float* a1 = a0 + 16 * MC_A;
    const float* b0 = b + g * b_inner + r * b_column;
    const float* b1 = b0 + 16 * b_column;
    for (int i = 0; i < inner; i += 16) {
        float x0[4], x1[4], y0[4], y1[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x0[u] = a0[i + 4 * u]; x1[u] = a1[i + 4 * u];
            y0[u] = b0[(i + 4 * u) * b_inner]; y1[u] = b1[(i + 4 * u) * b_inner];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x0[u], y0[u], acc[0][0], 0, 0, 0);
            acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x0[u], y1[u], acc[0][1], 0, 0, 0);
            acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[u], y0[u], acc[1][0], 0, 0, 0);
            acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x1[u], y1[u], acc[1][1], 0, 0, 0);
        }
    }
}

// L_t and take_t of a chunk's token `tid` (the first wavefront's lanes; lanes behind the chunk's n tokens: the last L, take 0):
// from `run` and the pairs of coefficients where another kernel has summed the logarithms up, or summed here, in 64-bit.
__device__ __forceinline__ void memory_chunk_weights(const DecayWeights& weights, const double* __restrict__ run, size_t token0, int n, int head,
                                                     int heads, int lane, double& total, float& take) {
    const size_t token = token0 + min(lane, n - 1);
    take = lane < n ? weights.take_of(token, head, heads) : 0.f;
    if (run != nullptr) {
        total = run[token * heads + head];
        return;
    }
    total = lane < n ? (double)weights.log_keep[token * weights.log_stride + head] : 0.0;
#pragma unroll
    for (int step = 1; step < 64; step <<= 1) {
        const double other = __shfl_up(total, step, 64);
        if (lane >= step) total += other;
    }
}

// A chunk's values of 64 columns from column0 on, [token][column] in LDS: zeros behind the chunk's last token and behind the
// column of ones that stands behind the values.  All of a thread's loads are issued before it stores.
template <typename T>
__device__ __forceinline__ void memory_stage_values(float* s_v, const T* __restrict__ v, long v_stride, size_t token0, int n, int head,
                                                    int value_dim, int column0, int tid) {
    T values[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        // (every load is of a place that is there, so that none stands under a condition and all are on their way together)
        const int t = min(4 * j + (tid >> 6), n - 1), c = min(column0 + (tid & 63), value_dim - 1);
        values[j] = v[(token0 + t) * v_stride + (size_t)head * value_dim + c];
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int t = 4 * j + (tid >> 6), c = column0 + (tid & 63);
        s_v[t * MC_B + (tid & 63)] = t < n ? (c < value_dim ? (float)values[j] : (c == value_dim ? 1.f : 0.f)) : 0.f;
    }
}

// (1) sums[item][head][channel][column] = sum_j e^(L_last - L_j) take_j k_j[channel] value_j[column]; grid (items, heads,
// blocks of 64 columns of value_dim + ones), 256 threads.  A = the weighted keys, read as [channel][token]; B = the values.
// totals (or nullptr) [item][head] = e^(L_last), for the walk.
template <typename T, typename V>
__global__ __launch_bounds__(256) void memory_chunk_sums_kernel(const T* __restrict__ k, long k_stride, const V* __restrict__ v, long v_stride,
                                                                DecayWeights weights, const double* __restrict__ run,
                                                                const int* __restrict__ row_start, const int* __restrict__ row_len, int rows,
                                                                float* __restrict__ sums, float* __restrict__ totals, int heads, int dim,
                                                                int value_dim, int group, int ones) {
    __shared__ float s_k[MC * MC_A];                     // [channel][token]
    __shared__ float s_v[MC * MC_B];                     // [token][column]
    __shared__ float s_w[MC];
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, column0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = min(MC, row_len[row] - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const int ld = value_dim + ones;
    const size_t key_column = (size_t)(head / group) * dim;
    if (tid < MC) {
        double total;
        float take;
        memory_chunk_weights(weights, run, token0, n, head, heads, tid, total, take);
        const double last = __shfl(total, n - 1, 64);
        s_w[tid] = expf((float)(last - total)) * take;
        if (totals != nullptr && tid == 0 && blockIdx.z == 0) totals[(size_t)blockIdx.x * heads + head] = expf((float)last);
    }
    memory_stage_values(s_v, v, v_stride, token0, n, head, value_dim, column0, tid);
    const int mt = wave >> 1, nt = wave & 1;
    const int inner = (n + 15) & ~15;
    for (int slab = 0; slab < dim; slab += 64) {
        T keys[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = min(4 * j + (tid >> 6), n - 1), c = min(slab + (tid & 63), dim - 1);    // (neighbouring threads read neighbouring channels of one token)
            keys[j] = k[(token0 + t) * k_stride + key_column + c];
        }
        __syncthreads();                                 // s_w is there; the slab before has been read
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = 4 * j + (tid >> 6), c = tid & 63;
            s_k[c * MC_A + t] = (t < n && slab + c < dim) ? (float)keys[j] * s_w[t] : 0.f;
        }
        __syncthreads();
        if (slab + mt * 32 >= dim || column0 + nt * 32 >= ld) continue;
        mc_f4 acc[2][2] = {};
        memory_product(acc, s_k + mt * 32 * MC_A, s_v + nt * 32, MC_B, 1, inner, lane);
        float* base = sums + (((size_t)blockIdx.x * heads + head) * dim) * ld;
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int channel = slab + mt * 32 + 16 * mi + 4 * (lane >> 4) + e, column = column0 + nt * 32 + 16 * ni + (lane & 15);
                    if (channel < dim && column < ld) base[(size_t)channel * ld + column] = acc[mi][ni][e];
                }
    }
}

// (2) grid (rows, heads, blocks of 256 numbers of a head's dim x (value_dim + ones)); a thread walks one number of the state
// through the row's chunks.  The next chunk's sum is loaded before this chunk's place is overwritten.  What a chunk keeps of
// the state is e^(run) at its last token, totals [item][head] or, by_channel, totals [item][head][dim].
__global__ __launch_bounds__(256) void memory_chunk_carry_kernel(float* __restrict__ sums, const double* __restrict__ run, const float* __restrict__ totals, float* state, long state_stride,
                                                                 const int* __restrict__ slots, const int* __restrict__ row_start,
                                                                 const int* __restrict__ row_len, const int* __restrict__ row_ctx,
                                                                 int heads, int dim, int value_dim, int ones, int by_channel) {
    const int row = blockIdx.x, head = blockIdx.y;
    const int count = row_len[row];
    if (count <= 0) return;
    const int ld = value_dim + ones;
    const long e = (long)blockIdx.z * 256 + threadIdx.x;
    if (e >= (long)dim * ld) return;
    const int channel = (int)(e / ld), column = (int)(e - (long)channel * ld);
    int base = 0;
    for (int r = 0; r < row; ++r) base += row_len[r] > 0 ? (row_len[r] + MC - 1) / MC : 0;
    const int chunks = (count + MC - 1) / MC, start = row_start[row];
    float* slot = state + (size_t)slots[row] * state_stride;
    float* mine = column < value_dim ? slot + ((size_t)head * dim + channel) * value_dim + column
                                     : slot + (size_t)heads * dim * value_dim + (size_t)head * dim + channel;
    float S = row_ctx[row] - count > 0 ? *mine : 0.f;
    const size_t step = (size_t)heads * dim * ld;
    float* place = sums + ((size_t)base * heads + head) * dim * ld + e;
    float sum = *place;
    for (int c = 0; c < chunks; ++c) {
        const float next = c + 1 < chunks ? place[step] : 0.f;
        const size_t last = (size_t)start + min(count, (c + 1) * MC) - 1;
        const size_t of_head = (size_t)(base + c) * heads + head;
        const float keep = totals ? totals[by_channel ? of_head * dim + channel : of_head] : expf((float)run[last * heads + head]);
        *place = S;
        S = __builtin_fmaf(keep, S, sum);
        sum = next;
        place += step;
    }
    *mine = S;
}

// The same with four numbers of a channel a thread, where value_dim, the state's place and its stride are multiples of four and there is
// no column of ones; the sums of two chunks are on their way while one is added.  It moves a state and a sum a chunk and nothing
// else: 32 rows of one chunk, 16 heads of 128 x 128, 102 us with a number a thread.
__global__ __launch_bounds__(256) void memory_chunk_carry4_kernel(float4* __restrict__ sums, const float* __restrict__ totals, float4* state,
                                                                  long state_stride, const int* __restrict__ slots,
                                                                  const int* __restrict__ row_len, const int* __restrict__ row_ctx, int heads, int dim,
                                                                  int value_dim, int by_channel) {
    const int row = blockIdx.x, head = blockIdx.y;
    const int count = row_len[row];
    const int quads = value_dim / 4, e = blockIdx.z * 256 + threadIdx.x;
    if (count <= 0 || e >= dim * quads) return;
    int base = 0;
    for (int r = 0; r < row; ++r) base += row_len[r] > 0 ? (row_len[r] + MC - 1) / MC : 0;
    const int chunks = (count + MC - 1) / MC;
    float4* mine = state + (size_t)slots[row] * state_stride + (size_t)head * dim * quads + e;
    float4 S = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row_ctx[row] - count > 0) S = *mine;
    const size_t step = (size_t)heads * dim * quads;
    float4* place = sums + ((size_t)base * heads + head) * dim * quads + e;
    const long keep_step = by_channel ? (long)heads * dim : heads;
    const float* keep = totals + (by_channel ? ((size_t)base * heads + head) * dim + e / quads : (size_t)base * heads + head);
    float4 sum = *place, next = place[chunks > 1 ? step : 0];
    float kept = *keep, next_kept = keep[chunks > 1 ? keep_step : 0];
    for (int c = 0; c < chunks; ++c) {
        const float4 ahead = place[c + 2 < chunks ? 2 * step : 0];
        const float ahead_kept = keep[c + 2 < chunks ? 2 * keep_step : 0];
        *place = S;
        S.x = __builtin_fmaf(kept, S.x, sum.x); S.y = __builtin_fmaf(kept, S.y, sum.y);
        S.z = __builtin_fmaf(kept, S.z, sum.z); S.w = __builtin_fmaf(kept, S.w, sum.w);
        sum = next; next = ahead;
        kept = next_kept; next_kept = ahead_kept;
        place += step;
        keep += keep_step;
    }
    *mine = S;
}

// (3) out[t][head][column] = sum_(j <= t) (q_t . k_j) e^(L_t - L_j) take_j value_j[column] + e^(L_t) sum_channel q_t[channel] S_0[channel][column],
// q scaled; with `ones` the column behind the values goes to below[t][head][0].  grid and workgroup as in (1).
template <typename T, typename V>
__global__ __launch_bounds__(256) void memory_chunk_read_kernel(const T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride,
                                                                const V* __restrict__ v, long v_stride, DecayWeights weights,
                                                                const double* __restrict__ run, float q_scale,
                                                                const int* __restrict__ row_start, const int* __restrict__ row_len,
                                                                const int* __restrict__ row_ctx, int rows, const float* __restrict__ sums,
                                                                float* __restrict__ out, float* __restrict__ below, int heads, int dim, int value_dim,
                                                                int group, int ones) {
    __shared__ float s_q[MC * MC_A];                     // [token][channel]
    __shared__ float s_k[MC * MC_A];                     // [token][channel]; then the weighted scores [token t][token j]
    __shared__ float s_v[MC * MC_B];                     // [token or channel][column]
    __shared__ double s_run[MC];
    __shared__ float s_take[MC], s_decay[MC];            // take_j; e^(L_t)
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, column0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int count = row_len[row];
    const int n = min(MC, count - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const int ld = value_dim + ones;
    const size_t key_column = (size_t)(head / group) * dim;
    const bool from_zero = chunk == 0 && row_ctx[row] - count == 0;      // nothing stands in front of the sequence's first chunk
    if (tid < MC) {
        double total;
        float take;
        memory_chunk_weights(weights, run, token0, n, head, heads, tid, total, take);
        s_run[tid] = total;
        s_take[tid] = take;
        s_decay[tid] = expf((float)total);
    }
    const int mt = wave >> 1, nt = wave & 1;
    // the scores of the wavefront's 32 tokens t against 32 tokens j (nothing to do where every j lies behind every t)
    mc_f4 scores[2][2] = {};
    for (int slab = 0; slab < dim; slab += 64) {
        T queries[16], keys[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = min(4 * j + (tid >> 6), n - 1), c = min(slab + (tid & 63), dim - 1);
            queries[j] = q[(token0 + t) * q_stride + key_column + c];
            keys[j] = k[(token0 + t) * k_stride + key_column + c];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int t = 4 * j + (tid >> 6), c = tid & 63;
            const bool there = t < n && slab + c < dim;
            s_q[t * MC_A + c] = there ? (float)queries[j] * q_scale : 0.f;
            s_k[t * MC_A + c] = there ? (float)keys[j] : 0.f;
        }
        __syncthreads();
        if (nt <= mt) memory_product(scores, s_q + mt * 32 * MC_A, s_k + nt * 32 * MC_A, 1, MC_A, min(64, (dim - slab + 15) & ~15), lane);
    }
    __syncthreads();                                     // everybody has read the keys: their place takes the weighted scores
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = mt * 32 + 16 * mi + 4 * (lane >> 4) + e, j = nt * 32 + 16 * ni + (lane & 15);
                float weight = 0.f;
                if (j <= t && t < n) weight = expf((float)(s_run[t] - s_run[j])) * s_take[j];
                s_k[t * MC_A + j] = scores[mi][ni][e] * weight;
            }
    memory_stage_values(s_v, v, v_stride, token0, n, head, value_dim, column0, tid);
    __syncthreads();
    const bool wanted = column0 + nt * 32 < ld;  // (uniform in a wavefront)
    mc_f4 acc[2][2] = {};
    if (wanted) memory_product(acc, s_k + mt * 32 * MC_A, s_v + nt * 32, MC_B, 1, (mt + 1) * 32, lane);
    if (!from_zero) {
        const float* before = sums + (((size_t)blockIdx.x * heads + head) * dim) * ld;
        for (int slab = 0; slab < dim; slab += 64) {
            T queries[16];
            float kept[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int t = 4 * j + (tid >> 6), c = tid & 63;          // queries [token][channel] times what the chunk's state has kept
                queries[j] = q[(token0 + min(t, n - 1)) * q_stride + key_column + min(slab + c, dim - 1)];
                const int channel = min(slab + t, dim - 1), column = min(column0 + c, ld - 1);      // the state's slab [channel][column]
                kept[j] = before[(size_t)channel * ld + column];
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int t = 4 * j + (tid >> 6), c = tid & 63;
                s_q[t * MC_A + c] = (t < n && slab + c < dim) ? (float)queries[j] * q_scale * s_decay[t] : 0.f;
                s_v[t * MC_B + c] = (slab + t < dim && column0 + c < ld) ? kept[j] : 0.f;
            }
            __syncthreads();
            if (wanted) memory_product(acc, s_q + mt * 32 * MC_A, s_v + nt * 32, MC_B, 1, min(64, (dim - slab + 15) & ~15), lane);
        }
    }
    if (!wanted) return;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = mt * 32 + 16 * mi + 4 * (lane >> 4) + e, column = column0 + nt * 32 + 16 * ni + (lane & 15);
                if (t >= n || column >= ld) continue;
                if (column < value_dim) out[(token0 + t) * heads * value_dim + (size_t)head * value_dim + column] = acc[mi][ni][e];
                else below[((token0 + t) * heads + head) * 2] = acc[mi][ni][e];
            }
}

// (3) where queries and keys are 16-bit and a head has a multiple of 32 channels: the same by wavefronts of 32 columns that need nothing of
// each other.  The kernel above makes the scores on 32-bit MFMA once per 64 columns and waits at barriers for every slab; 16-bit
// MFMA gives the same products of 16-bit numbers, summed in 32 bits, at an eighth of the time, so every wavefront makes them for
// itself, transposed: what an instruction leaves of them is then what the next one takes as its operand, and they never leave the
// registers.  The rest stays 32-bit: weighted scores x values, and decayed queries x the state, which comes straight from memory a
// step of 32 channels ahead.  Three workgroups a CU (153 registers) hide more of the state's way than two with all the registers they like
// (77 us).  Rows of 668, 667 and 667 tokens, 16 heads of 128 x 256 and a column of ones: 123 -> 66 us, of which the matrix cores are busy 21.
// Its error against 64 bits is half that of the kernel above, whose one sum takes up the scores' and the state's products alike.
// grid (items, heads, blocks of 128 columns).
typedef __bf16 mc_b8 __attribute__((ext_vector_type(8)));
constexpr int READ16_MOST = 128, READ16_PITCH = READ16_MOST + 8;       // channels of a head; numbers of a row in LDS

template <typename V>
__global__ __launch_bounds__(256, 3) void memory_chunk_read16_kernel(const bf16_t* __restrict__ q, long q_stride, const bf16_t* __restrict__ k, long k_stride,
                                                                  const V* __restrict__ v, long v_stride, DecayWeights weights,
                                                                  const double* __restrict__ run, float q_scale, const int* __restrict__ row_start,
                                                                  const int* __restrict__ row_len, const int* __restrict__ row_ctx, int rows,
                                                                  const float* __restrict__ sums, float* __restrict__ out,
                                                                  float* __restrict__ below, int heads, int dim, int value_dim, int group, int ones) {
    constexpr int TB = MC / 16;                          // blocks of 16 tokens
    __shared__ __align__(16) bf16_t s_q[MC * READ16_PITCH], s_k[MC * READ16_PITCH];
    __shared__ double s_run[MC];
    __shared__ float s_take[MC], s_decay[MC];            // take_j; e^(L_t)
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    const int count = row_len[row], n = min(MC, count - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const int ld = value_dim + ones, column0 = blockIdx.z * 128 + wave * 32;
    const size_t key_column = (size_t)(head / group) * dim;
    const bool from_zero = chunk == 0 && row_ctx[row] - count == 0;      // nothing stands in front of the sequence's first chunk
    // Every load is of a place that is there: a token behind the chunk's last one reads that one again, a column behind the last one the
    // last one; both count nothing.
    mc_b8 staged[2][READ16_MOST / 8 * MC / 256];
    const int pieces = MC * (dim / 8);
#pragma unroll
    for (int u = 0; u < READ16_MOST / 8 * MC / 256; ++u) {
        const int i = min(tid + 256 * u, pieces - 1), t = i / (dim / 8), c = 8 * (i % (dim / 8));
        const size_t token = token0 + min(t, n - 1);
        staged[0][u] = *reinterpret_cast<const mc_b8*>(q + token * q_stride + key_column + c);
        staged[1][u] = *reinterpret_cast<const mc_b8*>(k + token * k_stride + key_column + c);
    }
    if (tid < MC) {
        double total;
        float take;
        memory_chunk_weights(weights, run, token0, n, head, heads, tid, total, take);
        s_run[tid] = total;
        s_take[tid] = take;
        s_decay[tid] = expf((float)total);
    }
#pragma unroll
    for (int u = 0; u < READ16_MOST / 8 * MC / 256; ++u) {
        const int i = tid + 256 * u, t = i / (dim / 8), c = 8 * (i % (dim / 8));
        if (i >= pieces) break;
        *reinterpret_cast<mc_b8*>(&s_q[t * READ16_PITCH + c]) = staged[0][u];
        *reinterpret_cast<mc_b8*>(&s_k[t * READ16_PITCH + c]) = staged[1][u];
    }
    __syncthreads();
    if (column0 >= ld) return;
    float values[TB][4][2];
#pragma unroll
    for (int b = 0; b < TB; ++b) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const int j = 16 * b + 4 * g + e, column = column0 + 16 * m + r;
                const float there = (float)v[(token0 + min(j, n - 1)) * v_stride + (size_t)head * value_dim + min(column, value_dim - 1)];
                values[b][e][m] = j < n && column < ld ? (column < value_dim ? there : 1.f) : 0.f;
            }
    }

    // The state in front of the chunk, the first 32 channels of it asked for before anything else is waited for (no one reads what stands in
    // front of a sequence's first chunk: that place is there, and what it holds is not used).
    const float* before = sums + (((size_t)blockIdx.x * heads + head) * dim + 8 * g) * ld;
    struct Slab { float kept[2][8]; };
    auto load = [&](Slab& to, int slab) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int u = 0; u < 8; ++u) to.kept[m][u] = before[(size_t)(slab + u) * ld + min(column0 + 16 * m + r, ld - 1)];
    };
    auto query_of = [&](int block, int slab) { return *reinterpret_cast<const mc_b8*>(&s_q[(16 * block + r) * READ16_PITCH + slab + 8 * g]); };
    auto key_of = [&](int block, int slab) { return *reinterpret_cast<const mc_b8*>(&s_k[(16 * block + r) * READ16_PITCH + slab + 8 * g]); };
    Slab even;
    load(even, 0);

    // scores[t block][j block]: lane = token t = 16 tb + lane % 16, number e = token j = 16 jb + 4 (lane / 16) + e
    mc_f4 scores[TB][TB] = {};
    for (int slab = 0; slab < dim; slab += 32) {
        mc_b8 queries[TB], keys[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) queries[b] = query_of(b, slab), keys[b] = key_of(b, slab);
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int jb = 0; jb <= tb; ++jb) scores[tb][jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(keys[jb], queries[tb], scores[tb][jb], 0, 0, 0);
    }
    mc_f4 acc[TB][2] = {}, read[TB][2] = {};
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
        const int t = 16 * tb + r;
        const double total = s_run[t];
#pragma unroll
        for (int jb = 0; jb <= tb; ++jb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 16 * jb + 4 * g + e;
                const float weighted = j <= t && t < n ? scores[tb][jb][e] * q_scale * (expf((float)(total - s_run[j])) * s_take[j]) : 0.f;
#pragma unroll
                for (int m = 0; m < 2; ++m) acc[tb][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(weighted, values[jb][e][m], acc[tb][m], 0, 0, 0);
            }
    }

    if (!from_zero) {
        float decay[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) decay[b] = s_decay[16 * b + r];
        auto multiply = [&](const Slab& of, int slab) {
            mc_b8 queries[TB];
#pragma unroll
            for (int b = 0; b < TB; ++b) queries[b] = query_of(b, slab);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int b = 0; b < TB; ++b) {
                    const float query = (float)queries[b][u] * q_scale * decay[b];
#pragma unroll
                    for (int m = 0; m < 2; ++m) read[b][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(query, of.kept[m][u], read[b][m], 0, 0, 0);
                }
        };
        Slab odd;
        for (int slab = 0; slab < dim; slab += 64) {
            load(odd, min(slab + 32, dim - 32));
            multiply(even, slab);
            load(even, min(slab + 64, dim - 32));
            if (slab + 32 < dim) multiply(odd, slab + 32);
        }
    }
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * tb + 4 * g + e, column = column0 + 16 * m + r;
                if (t >= n || column >= ld) continue;
                const float sum = acc[tb][m][e] + read[tb][m][e];
                if (column < value_dim) out[(token0 + t) * heads * value_dim + (size_t)head * value_dim + column] = sum;
                else below[((token0 + t) * heads + head) * 2] = sum;
            }
}

// ---- the linear recurrence in chunks: a decay per key channel ---------------------------------------------------------
// S_t = diag(d_t) S_(t-1) + k_t v_t^T over a row's tokens of a step in chunks of 64 (items as above).  The weight of token j in
// what token t reads is, per channel, the product of the decays between them: a product of numbers of [0, 1], never a quotient of
// cumulative ones (exp(-exp(z)) reaches zero) and never a difference of their logarithms.  A chunk is cut into four blocks of
// 16 tokens: with P_t the product from t's block's first token to t, E_j the product behind j to its block's last token and T_I a
// block's whole product,
//   between blocks J < I   score[t][j] = sum_c (q_t P_t)[c] (T_(J+1) .. T_(I-1))[c] (k_j E_j)[c]       a matrix product,
//   inside a block         score[t][j] = sum_c q_t[c] k_j[c] (d_(j+1) .. d_t)[c]                       16 diagonals, on the vector units,
// and then, as with one decay a head, the chunk's read-outs are scores x values + (q_t P_t T_0 .. T_(I-1)) x S_0, its own sum is
// (k_j E_j T_(J+1) .. T_3)^T x values, and T_0 T_1 T_2 T_3 is what the chunk keeps of the state in front of it.  With a bonus the
// read-out is of the state before the token: the products end in front of d_t, and the token itself enters through its bonus.
//
// What bounds the scan is the chain of a row's tokens (0.45 us a token, on rows * heads * value_dim / 64 workgroups: 918 us for
// one row of 2,048 tokens, 16 heads of 128 x 128, 1,171 us for 8 heads of 128 x 256, most of the chip idle); here all chunks
// run at once and only the walk over the chunks (2) is serial.  A workgroup has one (chunk, head, 128 value columns): scores are formed once
// for all of them, operands stay in LDS (146 KB at 128 channels, so one workgroup a compute unit), products run on 32-bit MFMA but where said.
//   What bounds the first launch is what one compute unit gets through between its barriers, operands from memory and their decays, diagonals, 64-bit products, one
// after another; sixteen wavefronts hide more of it than eight did.  They share the work so that every sum is formed in the order that eight formed it in (diagonals between two wavefronts, not their
// channels; a tile's four sums between two), and the results are the same bits.  us with the walk and the read-out, eight wavefronts and sixteen: 2,048 tokens of 16 heads of
// 128 x 128 125, 110; of 8 heads of 128 x 256 123, 107; 1,024 tokens 102, 86 and 100, 85; 2,048 of 16 heads of 64 x 64 67, 60; six rows of 510 tokens of those 104, 91.  (3) is
// no faster with its loads a slab ahead, and with registers for four workgroups a compute unit faster behind 768 of them only (120, 114; 92, 96).
constexpr int CHANNEL_MOST = 128;        // widest head that fits LDS so
constexpr int CHANNEL_COLUMNS = 128;     // value columns a workgroup
constexpr int CHANNEL_THREADS = 1024;    // of a workgroup: sixteen wavefronts
constexpr int CHANNEL_DIAGONALS = 8;     // that a wavefront forms of a block of tokens: two share its sixteen, for each half of the channels

template <int DP>
struct ChannelChunkLds {                 // DP: key channels filled up to 64 or 128
    static constexpr int A = DP + 4;     // row length of an operand read down its rows
    static constexpr int B = DP + 16;    // ... read along its rows
    float q[MC * B];                     // queries; then (row length B) the keys as the chunk's sum wants them
    float k[MC * B];                     // (row length A) keys; then (row length B) what rounding took from the keys as the sum wants them
    float d[MC * (A > MC_B ? A : MC_B)]; // decays; then (row length A) what rounding took from the keys; then the values of the first 64 columns (row length MC_B)
    float score[MC * MC_A];
    double total[MC / BC][DP];
    union {
        double diagonal[2][BC][MC];                                                // sums of a half of the channels: [tokens back][token]
        double between[6][64][4];                                                  // ... of every second four of them, as a wavefront's lanes hold a tile
        float v[MC * MC_B];                                                        // the values of the second 64 columns
    };
    int no_number[2];                                                              // one once a value of the first or the second 64 columns is none
};

// (1) out = the chunks' own read-outs, sums [item][head][dim][value_dim] and totals [item][head][dim] as the walk wants them,
// and queries [T][heads][dim] as they read the state in front of their chunk.  grid (items, heads, blocks of 128 value columns).
template <typename T, int DP>
__global__ __launch_bounds__(CHANNEL_THREADS) void channel_chunk_kernel(const T* __restrict__ q, long q_stride, const T* __restrict__ k, long k_stride,
                                                            const T* __restrict__ v, long v_stride, const float* __restrict__ decay,
                                                            const float* __restrict__ decay_bias, int mode, float inv_tau,
                                                            const float* __restrict__ bonus, float q_scale, const int* __restrict__ row_start,
                                                            const int* __restrict__ row_len, int rows, float* __restrict__ sums,
                                                            float* __restrict__ totals, float* __restrict__ queries, float* __restrict__ out,
                                                            int heads, int dim, int value_dim) {
    extern __shared__ __align__(16) float lds[];
    typedef ChannelChunkLds<DP> Lds;
    Lds& s = *reinterpret_cast<Lds*>(lds);
    constexpr int A = Lds::A, B = Lds::B;
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = min(MC, row_len[row] - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const size_t key_column = (size_t)head * dim;
    const bool first_columns = blockIdx.z == 0;

    // Queries, keys and decays into LDS; tokens behind the chunk's last one and channels behind the head's last one read and write
    // nothing and keep everything.  (Every load is of a place that is there: none stands under a condition.)
    {
        constexpr int PER = MC * DP / CHANNEL_THREADS;
        T raw_q[PER], raw_k[PER];
        float raw_z[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + CHANNEL_THREADS * e, t = min(i / DP, n - 1), c = min(i % DP, dim - 1);
            const size_t token = token0 + t;
            raw_q[e] = q[token * q_stride + key_column + c];
            raw_k[e] = k[token * k_stride + key_column + c];
            raw_z[e] = decay[token * (size_t)heads * dim + key_column + c] + (decay_bias ? decay_bias[key_column + c] : 0.f);
        }
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + CHANNEL_THREADS * e, t = i / DP, c = i % DP;
            const bool there = t < n && c < dim;
            s.q[t * A + c] = there ? (float)raw_q[e] * q_scale : 0.f;
            s.k[t * A + c] = there ? (float)raw_k[e] : 0.f;
            s.d[t * A + c] = there ? decay_of(raw_z[e], mode, inv_tau) : 1.f;
        }
        for (int i = tid; i < MC * MC_A; i += CHANNEL_THREADS) s.score[i] = 0.f;
        if (tid < 2) s.no_number[tid] = 0;
    }
    __syncthreads();

    // Inside the blocks: wavefront = (block, half of the channels, half of the diagonals), lane = (token t of the block, a quarter of every 16 channels).
    // The diagonals j = t - back one after another, the query times its decays so far in registers (the later half of them begins behind the earlier one's decays).
    {
        const int block = wave >> 2, half = (wave >> 1) & 1, first = CHANNEL_DIAGONALS * (wave & 1), t = lane & 15, c0 = half * (DP / 2) + 4 * (lane >> 4);
        constexpr int U = DP / 32;
        float weighted[U][4];
        double sum[CHANNEL_DIAGONALS];                                             // (their last additions would be the score's largest roundings)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float4 x = *reinterpret_cast<const float4*>(&s.q[(block * BC + t) * A + c0 + 16 * u]);
            weighted[u][0] = x.x; weighted[u][1] = x.y; weighted[u][2] = x.z; weighted[u][3] = x.w;
        }
        for (int back = bonus == nullptr ? 0 : 1; back < first; ++back) {
            const int j = block * BC + max(t - back, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float4 f = *reinterpret_cast<const float4*>(&s.d[j * A + c0 + 16 * u]);
                weighted[u][0] *= f.x; weighted[u][1] *= f.y; weighted[u][2] *= f.z; weighted[u][3] *= f.w;
            }
        }
#pragma unroll
        for (int i = 0; i < CHANNEL_DIAGONALS; ++i) {
            const int back = first + i, j = block * BC + max(t - back, 0);
            float part[4] = {};
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float4 x = *reinterpret_cast<const float4*>(&s.k[j * A + c0 + 16 * u]);
                const float4 f = *reinterpret_cast<const float4*>(&s.d[j * A + c0 + 16 * u]);
                const float ks[4] = {x.x, x.y, x.z, x.w}, ds[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float own = weighted[u][e];
                    if (i == 0 && bonus != nullptr && back == 0) {
                        const int c = c0 + 16 * u + e;
                        own *= bonus[key_column + min(c, dim - 1)];               // (channels behind the head's last one: q is 0)
                    }
                    part[e] = __builtin_fmaf(own, ks[e], part[e]);
                    if (i > 0 || bonus == nullptr || back > 0) weighted[u][e] *= ds[e];     // (the next diagonal lies behind token j's decay)
                }
            }
            sum[i] = ((double)part[0] + (double)part[1]) + ((double)part[2] + (double)part[3]);
        }
        // (added up over the four lanes of a token, neighbours first, each of which ends with two of the diagonals)
        const bool upper = lane & 32, odd = lane & 16;
#pragma unroll
        for (int i = 0; i < CHANNEL_DIAGONALS / 2; ++i) {
            const double other = __shfl_xor(odd ? sum[i] : sum[CHANNEL_DIAGONALS / 2 + i], 16, 64);
            sum[i] = (odd ? sum[CHANNEL_DIAGONALS / 2 + i] : sum[i]) + other;
        }
#pragma unroll
        for (int i = 0; i < CHANNEL_DIAGONALS / 4; ++i) {
            const double other = __shfl_xor(upper ? sum[i] : sum[CHANNEL_DIAGONALS / 4 + i], 32, 64);
            s.diagonal[half][first + (odd ? CHANNEL_DIAGONALS / 2 : 0) + (upper ? CHANNEL_DIAGONALS / 4 : 0) + i][block * BC + t] = (upper ? sum[CHANNEL_DIAGONALS / 4 + i] : sum[i]) + other;
        }
    }
    __syncthreads();
    {                                                                              // (a thread one score: BC diagonals of MC tokens)
        const int t = tid % MC, back = tid / MC;
        if (back <= t % BC) s.score[t * MC_A + t - back] = (float)((double)(float)(0.0 + s.diagonal[0][back][t]) + s.diagonal[1][back][t]);
    }

    // Queries times the decays from their block's first token (one half of the threads), keys times those up to its last one (the other); a thread a (block, channel).
    // The products are formed in 64-bit: sixteen factors then cost a weight one rounding, as they do the scan's state.
    {
        const bool keys = tid >= (MC / BC) * DP;
        const int i = keys ? tid - (MC / BC) * DP : tid, block = i / DP, c = i % DP;
        const bool some = i < (MC / BC) * DP;
        float d[BC];
#pragma unroll
        for (int t = 0; t < BC; ++t) d[t] = some ? s.d[(block * BC + t) * A + c] : 1.f;
        __syncthreads();                                                           // (what the keys lose in rounding takes the decays' place)
        double product = 1.0;
        if (some && !keys) {
            float* qs = &s.q[block * BC * A + c];
#pragma unroll
            for (int t = 0; t < BC; ++t) {
                if (bonus == nullptr) product *= (double)d[t];
                qs[t * A] = (float)((double)qs[t * A] * product);
                if (bonus != nullptr) product *= (double)d[t];
            }
            s.total[block][c] = product;
        } else if (some) {
            float* ks = &s.k[block * BC * A + c];
#pragma unroll
            for (int t = BC - 1; t >= 0; --t) {
                const double key = (double)ks[t * A] * product;
                ks[t * A] = (float)key;
                s.d[(block * BC + t) * A + c] = (float)(key - (double)(float)key);
                product *= (double)d[t];
            }
        }
    }
    __syncthreads();

    // Between blocks: six tiles of 16 x 16 scores, two wavefronts a tile, each with two of the four sums of every fourth channel group that make one.
    {
        const int tile = wave >> 1, half = wave & 1, block = tile < 3 ? 3 : tile < 5 ? 2 : 1, other = tile < 3 ? tile : tile < 5 ? tile - 3 : 0;
        const int r = lane & 15, g = lane >> 4;
        double sum[4] = {};
        if (tile < 6) {
            const float* a = &s.q[(block * BC + r) * A + g + 8 * half];
            const float* b = &s.k[(other * BC + r) * A + g + 8 * half];
            mc_f4 part[2] = {};
            for (int i = 0; i < DP; i += 16) {
                float x[2], y[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int c = i + 8 * half + 4 * u + g;
                    y[u] = b[i + 4 * u];
                    const double next = s.total[other + 1][c], after = s.total[min(other + 2, MC / BC - 1)][c];
                    const double skipped = (block > other + 1 ? next : 1.0) * (block > other + 2 ? after : 1.0);
                    x[u] = (float)((double)a[i + 4 * u] * skipped);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) part[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], y[u], part[u], 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] = (double)part[0][e] + (double)part[1][e];
                if (half == 1) s.between[tile][lane][e] = sum[e];
            }
        }
        __syncthreads();
        if (tile < 6 && half == 0)
#pragma unroll
            for (int e = 0; e < 4; ++e) s.score[(block * BC + 4 * g + e) * MC_A + other * BC + r] = (float)(sum[e] + s.between[tile][lane][e]);
    }

    // The queries and the totals leave (whatever lies in front of or behind a block in one product, 64-bit as above); the keys are brought up to the chunk's end, into the queries' place behind them.
    {
        constexpr int PER = MC * DP / CHANNEL_THREADS;
        float kept[PER], rest[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + CHANNEL_THREADS * e, t = i / DP, c = i % DP, block = t / BC;
            double before = 1.0, behind = 1.0;
#pragma unroll
            for (int o = 0; o < MC / BC; ++o) {
                const double total = s.total[o][c];
                before *= o < block ? total : 1.0;
                behind *= o > block ? total : 1.0;
            }
            if (first_columns && t < n && c < dim) queries[(token0 + t) * (size_t)heads * dim + key_column + c] = (float)((double)s.q[t * A + c] * before);
            const double key = ((double)s.k[t * A + c] + (double)s.d[t * A + c]) * behind;
            kept[e] = (float)key;
            rest[e] = (float)(key - (double)kept[e]);
        }
        if (first_columns && tid < dim)
            totals[((size_t)blockIdx.x * heads + head) * dim + tid] = (float)((s.total[0][tid] * s.total[1][tid]) * (s.total[2][tid] * s.total[3][tid]));
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int i = tid + CHANNEL_THREADS * e;
            s.q[(i / DP) * B + i % DP] = kept[e];
            s.k[(i / DP) * B + i % DP] = rest[e];
        }
    }

    // Scores x values, and the keys' sum with the values: 64 columns for each eight wavefronts.
    const int of = wave / 8, column0 = blockIdx.z * CHANNEL_COLUMNS + 64 * of;
    float* s_v = of ? s.v : s.d;
    constexpr int VALUES = MC * 64 / 512;
    T values[VALUES];
#pragma unroll
    for (int e = 0; e < VALUES; ++e) {
        const int t = min(8 * e + (wave & 7), n - 1), c = min(column0 + lane, value_dim - 1);
        values[e] = v[(token0 + t) * v_stride + (size_t)head * value_dim + c];
    }
    __syncthreads();                                     // the keys are in place, and nobody reads what the values replace
    float no_number = 0.f;                               // NaN once a value is no number
#pragma unroll
    for (int e = 0; e < VALUES; ++e) {
        const int t = 8 * e + (wave & 7);
        const float value = t < n && column0 + lane < value_dim ? (float)values[e] : 0.f;
        s_v[t * MC_B + lane] = value;
        no_number = __builtin_fmaf(value, 0.f, no_number);
    }
    if (no_number != 0.f) s.no_number[of] = 1;
    __syncthreads();
    const bool all_finite = s.no_number[of] == 0;        // (of these 64 columns: what lies in the others does not change how theirs are formed)
    if (column0 < value_dim) {
        const int r = lane & 15, g = lane >> 4, half = wave & 1;
        {
            const int block = (wave & 7) >> 1;
            mc_f4 acc[2] = {};
            if (all_finite) {
                channel_product<2>(acc, &s.score[block * BC * MC_A], MC_A, 1, s_v + 32 * half, MC_B, 1, (block + 1) * BC, lane);
            } else {
                // (the products above the diagonal are of zeros: a later token's infinity or NaN must not meet them)
#pragma unroll 1
                for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int t = block * BC + 4 * g + e;
                        double sum = 0.0;
                        for (int j = 0; j <= t; ++j) sum += (double)s.score[t * MC_A + j] * (double)s_v[j * MC_B + 32 * half + 16 * ni + r];
                        if (ni == 0) acc[0][e] = (float)sum;
                        else acc[1][e] = (float)sum;
                    }
            }
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = block * BC + 4 * g + e, column = column0 + 32 * half + 16 * ni + r;
                    if (t < n && column < value_dim) out[(token0 + t) * heads * value_dim + (size_t)head * value_dim + column] = acc[ni][e];
                }
        }
        float* base = sums + (((size_t)blockIdx.x * heads + head) * dim) * value_dim;
        // The tokens of the chunk's last two blocks weigh most in what is left of it: their products are 64-bit, of keys that no rounding has
        // touched.  With 32-bit ones the state behind a short memory (decays around 0.6 a token) was off by 1.32 times what the walk's
        // is (bfloat16; 1.15 in float32); it is 1.06 and 0.90, 0.76 of it where memories are long.  11 us of 133 for 2,048 tokens of 16 heads.
        const int exact_from = BC * max(0, (n + BC - 1) / BC - 2);
        for (int tile = (wave & 7) >> 1; tile < DP / 16; tile += 4) {
            mc_f4 part[2][4] = {};
            const int turned = 4 * (r & 3) + (r >> 2);   // (in this order of rows the 32-bit instruction's results lie where the 64-bit one's do)
            for (int i = 0; i < exact_from; i += 16) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float key = s.q[(i + 4 * u + g) * B + tile * 16 + turned];
#pragma unroll
                    for (int ni = 0; ni < 2; ++ni)
                        part[ni][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(key, s_v[(i + 4 * u + g) * MC_B + 32 * half + 16 * ni + r], part[ni][u], 0, 0, 0);
                }
            }
            mc_d4 acc[2][2] = {};
            for (int i = exact_from; i < min(exact_from + 2 * BC, MC); i += 16)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int t = i + 4 * u + g;
                    const double key = (double)s.q[t * B + tile * 16 + r] + (double)s.k[t * B + tile * 16 + r];
#pragma unroll
                    for (int ni = 0; ni < 2; ++ni)
                        acc[ni][u & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(key, (double)s_v[t * MC_B + 32 * half + 16 * ni + r], acc[ni][u & 1], 0, 0, 0);
                }
#pragma unroll
            for (int ni = 0; ni < 2; ++ni)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int channel = tile * 16 + 4 * e + g, column = column0 + 32 * half + 16 * ni + r;
                    if (channel < dim && column < value_dim) {
                        const double early = ((double)part[ni][0][e] + (double)part[ni][1][e]) + ((double)part[ni][2][e] + (double)part[ni][3][e]);
                        base[(size_t)channel * value_dim + column] = (float)(acc[ni][0][e] + acc[ni][1][e] + early);
                    }
                }
        }
    }
}

// (3) out[t] += queries[t] x S_0, S_0 the state in front of the token's chunk, as the walk left it in sums; grid (items, heads, blocks of
// 64 value columns), four wavefronts of 16 tokens.  What stands in front of a sequence's first chunk is nothing.
__global__ __launch_bounds__(256) void channel_chunk_read_kernel(const float* __restrict__ queries, const float* __restrict__ sums,
                                                                 const int* __restrict__ row_start, const int* __restrict__ row_len,
                                                                 const int* __restrict__ row_ctx, int rows, float* __restrict__ out, int heads,
                                                                 int dim, int value_dim) {
    __shared__ float s_q[MC * MC_A];                     // [token][channel]
    __shared__ float s_s[64 * MC_B];                     // [channel][column]
    int row, chunk;
    if (!chunk_item(blockIdx.x, rows, row_len, row, chunk)) return;
    const int head = blockIdx.y, column0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int count = row_len[row];
    if (chunk == 0 && row_ctx[row] - count == 0) return;
    const int n = min(MC, count - chunk * MC);
    const size_t token0 = (size_t)row_start[row] + (size_t)chunk * MC;
    const float* before = sums + (((size_t)blockIdx.x * heads + head) * dim) * value_dim;
    const int r = lane & 15, g = lane >> 4;
    mc_f4 acc[4] = {};
    for (int slab = 0; slab < dim; slab += 64) {
        float read[16], kept[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int line = 4 * j + (tid >> 6), c = tid & 63;
            read[j] = queries[(token0 + min(line, n - 1)) * (size_t)heads * dim + (size_t)head * dim + min(slab + c, dim - 1)];
            kept[j] = before[(size_t)min(slab + line, dim - 1) * value_dim + min(column0 + c, value_dim - 1)];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int line = 4 * j + (tid >> 6), c = tid & 63;
            s_q[line * MC_A + c] = line < n && slab + c < dim ? read[j] : 0.f;
            s_s[line * MC_B + c] = slab + line < dim && column0 + c < value_dim ? kept[j] : 0.f;
        }
        __syncthreads();
        channel_product<4>(acc, s_q + wave * 16 * MC_A, MC_A, 1, s_s, MC_B, 1, min(64, (dim - slab + 15) & ~15), lane);
    }
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = wave * 16 + 4 * g + e, column = column0 + 16 * ni + r;
            if (t < n && column < value_dim) out[(token0 + t) * heads * value_dim + (size_t)head * value_dim + column] += acc[ni][e];
        }
}

template <typename T>
__global__ __launch_bounds__(256) void tanh_kernel(T* __restrict__ x, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = (T)tanhf((float)x[i]);
}

template <typename T>
__global__ __launch_bounds__(256) void scaled_sum_kernel(const T* __restrict__ x, float a, const T* __restrict__ y, float b,
                                                         T* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (T)(a * (float)x[i] + b * (float)y[i]);
}

LSA_EXPORT int lsa_token_shift(int code, const void* h, const float* mu, int mixes, float* state, long state_stride, const int* slots,
                               const int* token_row, const int* positions, const int* row_start, void* out, int n_tokens, int width,
                               int keep, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (mixes < 1 || state == nullptr || slots == nullptr) return -1;
    // (16 bytes a load leave too few threads where there are few numbers: five mixes of 2,048 columns in bfloat16, us, one number a load and eight, 32 tokens 3.5, 4.1, 96
    // tokens 4.1, 4.2, 128 tokens (2^18 numbers) 4.8, 4.3, 512 tokens 8.4, 5.8)
    const bool wide = width % 8 == 0 && ((size_t)h | (size_t)mu | (size_t)out) % 16 == 0 && (long)n_tokens * width >= 1 << 18;
    const int columns = 256 * (!wide ? 1 : code ? 8 : 4);
    const dim3 grid(n_tokens, (width + columns - 1) / columns);
#define LSA_LAUNCH(T) do { if (wide) LSA_LAUNCH_OF(T, Elem<T>::kVec); else LSA_LAUNCH_OF(T, 1); } while (0)
#define LSA_LAUNCH_OF(T, V) token_shift_kernel<T, V><<<grid, 256, 0, stream>>>((const T*)h, mu, mixes, state, state_stride, slots, token_row, positions, \
        row_start, (T*)out, n_tokens, width, keep)
    if (code) LSA_LAUNCH(bf16_t); else LSA_LAUNCH(float);
#undef LSA_LAUNCH_OF
#undef LSA_LAUNCH
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_token_shift_keep(int code, const void* h, float* state, long state_stride, const int* slots, const int* row_start,
                                    const int* row_len, int rows, int width, hipStream_t stream) {
    if (rows <= 0) return 0;
    dim3 grid(rows, (width + 255) / 256);
    if (code) token_shift_keep_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, state, state_stride, slots, row_start, row_len, width);
    else token_shift_keep_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, state, state_stride, slots, row_start, row_len, width);
    LSA_LAUNCH_CHECK();
}

// Key channels a wavefront takes: 8 for heads of up to 64 channels, 16 up to 128, 32 up to 256, 64 up to 512: at most eight
// wavefronts a workgroup, and what the tokens' chunk and the wavefronts' partial read-outs take of LDS stays below 160 KB.
constexpr int MOST_DIM = 512;
constexpr int MOST_LDS = 160 * 1024;

LSA_EXPORT int lsa_linear_recurrence_most_dim() { return MOST_DIM; }

static size_t recurrence_lds(int dim, int& dk, int& waves) {
    dk = dim <= 64 ? 8 : dim <= 128 ? 16 : dim <= 256 ? 32 : 64;
    waves = (dim + dk - 1) / dk;
    return sizeof(float) * ((size_t)3 * CHUNK * waves * dk + (size_t)CHUNK * 64 + (size_t)waves * CHUNK * 64);
}

// Once, when the library has been loaded and before any launch: lets every form of the recurrence kernel ask for more
// dynamic LDS than the default limit.  (Not part of a launch: a launch may be recorded into a graph, and a stream
// that is being captured must see launches only.)
LSA_EXPORT int lsa_recurrent_prepare() {
    hipError_t first = hipSuccess;
#define LSA_ALLOW(T, DK, B) do { \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_recurrence_kernel<T, DK, B>), \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS); \
        if (e != hipSuccess && first == hipSuccess) first = e; \
    } while (0)
#define LSA_ALLOW_ALL(T) do { LSA_ALLOW(T, 8, false); LSA_ALLOW(T, 8, true); LSA_ALLOW(T, 16, false); LSA_ALLOW(T, 16, true); \
                              LSA_ALLOW(T, 32, false); LSA_ALLOW(T, 32, true); LSA_ALLOW(T, 64, false); LSA_ALLOW(T, 64, true); } while (0)
    LSA_ALLOW_ALL(float);
    LSA_ALLOW_ALL(bf16_t);
#undef LSA_ALLOW_ALL
#undef LSA_ALLOW
#define LSA_ALLOW(T, V, DK) do { \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&matrix_memory_kernel<T, V, DK>), \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS); \
        if (e != hipSuccess && first == hipSuccess) first = e; \
    } while (0)
#define LSA_ALLOW_ALL(T, V) do { LSA_ALLOW(T, V, 8); LSA_ALLOW(T, V, 16); LSA_ALLOW(T, V, 32); LSA_ALLOW(T, V, 64); } while (0)
    LSA_ALLOW_ALL(float, float);
    LSA_ALLOW_ALL(bf16_t, bf16_t);
    LSA_ALLOW_ALL(float, bf16_t);
#undef LSA_ALLOW_ALL
#undef LSA_ALLOW
#define LSA_ALLOW(T, DP) do { \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&channel_chunk_kernel<T, DP>), \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, MOST_LDS); \
        if (e != hipSuccess && first == hipSuccess) first = e; \
    } while (0)
    LSA_ALLOW(float, 64); LSA_ALLOW(float, 128); LSA_ALLOW(bf16_t, 64); LSA_ALLOW(bf16_t, 128);
#undef LSA_ALLOW
    (void)hipGetLastError();
    return (int)first;
}

// The walk over the chunks, four numbers a thread where that is possible.
static void run_carry(float* sums, const double* run, const float* totals, float* state, long state_stride, const int* slots, const int* row_start,
                      const int* row_len, const int* row_ctx, int rows, int heads, int dim, int value_dim, int ones, int by_channel,
                      hipStream_t stream) {
    if (ones == 0 && totals != nullptr && value_dim % 4 == 0 && state_stride % 4 == 0 && reinterpret_cast<size_t>(state) % 16 == 0 &&
        reinterpret_cast<size_t>(sums) % 16 == 0) {
        const dim3 grid(rows, heads, (unsigned)(((long)dim * (value_dim / 4) + 255) / 256));
        memory_chunk_carry4_kernel<<<grid, 256, 0, stream>>>(reinterpret_cast<float4*>(sums), totals, reinterpret_cast<float4*>(state), state_stride / 4,
                                                             slots, row_len, row_ctx, heads, dim, value_dim, by_channel);
        return;
    }
    const dim3 grid(rows, heads, (unsigned)(((long)dim * (value_dim + ones) + 255) / 256));
    memory_chunk_carry_kernel<<<grid, 256, 0, stream>>>(sums, run, totals, state, state_stride, slots, row_start, row_len, row_ctx, heads, dim,
                                                        value_dim, ones, by_channel);
}

LSA_EXPORT int lsa_linear_recurrence(int code, const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                                     const float* decay, const float* decay_bias, int mode, float tau, const float* bonus, float q_scale,
                                     float* state, long state_stride, const int* slots, const int* row_start, const int* row_len,
                                     const int* row_ctx, float* out, int rows, int heads, int dim, int value_dim, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > MOST_DIM || value_dim < 1 || heads < 1 || (mode != 0 && mode != 1) || !(tau > 0.f) || state == nullptr) return -1;
    int dk, waves;
    const size_t lds = recurrence_lds(dim, dk, waves);
    if (lds > (size_t)MOST_LDS) return -1;
    dim3 grid(rows, heads, (value_dim + 63) / 64);
#define LSA_LAUNCH(T, DK, B) \
        linear_recurrence_kernel<T, DK, B><<<grid, waves * 64, lds, stream>>>((const T*)q, q_stride, (const T*)k, k_stride, (const T*)v, v_stride, \
            decay, decay_bias, mode, 1.f / tau, bonus, q_scale, state, state_stride, slots, row_start, row_len, row_ctx, out, heads, dim, value_dim)
#define LSA_BY_DK(T, B) do { if (dk == 8) LSA_LAUNCH(T, 8, B); else if (dk == 16) LSA_LAUNCH(T, 16, B); else if (dk == 32) LSA_LAUNCH(T, 32, B); \
                             else LSA_LAUNCH(T, 64, B); } while (0)
    if (code) { if (bonus) LSA_BY_DK(bf16_t, true); else LSA_BY_DK(bf16_t, false); }
    else { if (bonus) LSA_BY_DK(float, true); else LSA_BY_DK(float, false); }
#undef LSA_BY_DK
#undef LSA_LAUNCH
    LSA_LAUNCH_CHECK();
}

// The same in chunks.  items is no less than the number of chunks of 64 tokens that the rows have together; sums [items][heads][dim][value_dim],
// totals [items][heads][dim] and queries [T][heads][dim] are the caller's scratch memory.
LSA_EXPORT int lsa_linear_recurrence_chunked_most_dim() { return CHANNEL_MOST; }

LSA_EXPORT int lsa_linear_recurrence_chunked(int code, const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                                             const float* decay, const float* decay_bias, int mode, float tau, const float* bonus, float q_scale,
                                             float* state, long state_stride, const int* slots, const int* row_start, const int* row_len,
                                             const int* row_ctx, float* out, int rows, int heads, int dim, int value_dim, float* sums, float* totals,
                                             float* queries, int items, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > CHANNEL_MOST || value_dim < 1 || heads < 1 || (mode != 0 && mode != 1) || !(tau > 0.f) || state == nullptr) return -1;
    if (items <= 0 || sums == nullptr || totals == nullptr || queries == nullptr) return -1;
    const dim3 grid(items, heads, (value_dim + CHANNEL_COLUMNS - 1) / CHANNEL_COLUMNS);
#define LSA_LAUNCH(T, DP) \
        channel_chunk_kernel<T, DP><<<grid, CHANNEL_THREADS, sizeof(ChannelChunkLds<DP>), stream>>>((const T*)q, q_stride, (const T*)k, k_stride, (const T*)v, v_stride, \
            decay, decay_bias, mode, 1.f / tau, bonus, q_scale, row_start, row_len, rows, sums, totals, queries, out, heads, dim, value_dim)
    if (code) { if (dim <= 64) LSA_LAUNCH(bf16_t, 64); else LSA_LAUNCH(bf16_t, 128); }
    else { if (dim <= 64) LSA_LAUNCH(float, 64); else LSA_LAUNCH(float, 128); }
#undef LSA_LAUNCH
    run_carry(sums, nullptr, totals, state, state_stride, slots, row_start, row_len, row_ctx, rows, heads, dim, value_dim, 0, 1, stream);
    channel_chunk_read_kernel<<<dim3(items, heads, (value_dim + 63) / 64), 256, 0, stream>>>(queries, sums, row_start, row_len, row_ctx, rows, out, heads,
                                                                                             dim, value_dim);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_heads_norm_gate(int code, const float* x, const float* weight, int weight_per_channel, float eps, const void* gate,
                                   long gate_stride, void* out, int n_tokens, int heads, int value_dim, int gate_kind, const float* below,
                                   float floor, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (gate_kind != 0 && gate_kind != 1) return -1;
    dim3 grid(n_tokens, heads);
    const int weight_stride = weight_per_channel ? value_dim : 0;
    const long pairs = (long)n_tokens * heads;
    // (heads of up to 64 numbers leave half of its lanes idle, which pays for many of them only: 64 heads of 64, us, the kernel above and this one, 8 tokens 2.7, 3.0,
    // 32 tokens 2.9, 3.1, 64 tokens 3.3, 3.2, 512 tokens 10.2, 7.9; in float32 2.7, 3.2; 2.8, 3.3; 3.3, 3.2; 10.5, 9.0)
    if (pairs < 0x7fffffffL && value_dim % 8 == 0 && value_dim <= 256 && gate_stride % 8 == 0 && (value_dim > 64 || pairs >= 4096)
        && ((size_t)x | (size_t)weight | (size_t)gate | (size_t)out) % 16 == 0) {
        const unsigned blocks = (unsigned)((pairs + 15) / 16);
#define LSA_LONG(T, C) heads_norm_gate_eights_kernel<T, C><<<blocks, 256, 0, stream>>>(x, weight, weight_stride, eps, (const T*)gate, gate_stride, (T*)out, heads, \
        value_dim, gate_kind, below, floor, (int)pairs)
        if (value_dim <= 128) { if (code) LSA_LONG(bf16_t, 1); else LSA_LONG(float, 1); }
        else { if (code) LSA_LONG(bf16_t, 2); else LSA_LONG(float, 2); }
#undef LSA_LONG
        LSA_LAUNCH_CHECK();
    }
    if (code) heads_norm_gate_kernel<bf16_t><<<grid, 64, 0, stream>>>(x, weight, weight_stride, eps, (const bf16_t*)gate, gate_stride, (bf16_t*)out, heads, value_dim, gate_kind, below, floor);
    else heads_norm_gate_kernel<float><<<grid, 64, 0, stream>>>(x, weight, weight_stride, eps, (const float*)gate, gate_stride, (float*)out, heads, value_dim, gate_kind, below, floor);
    LSA_LAUNCH_CHECK();
}

// The recurrence itself, in either form; sums == nullptr: token by token.  In chunks, sums [items][heads][dim][value_dim + ones]
// and, without `run`, totals [items][heads] are the caller's scratch memory; items is no less than the number of chunks of 64
// tokens that the rows have together.
template <typename T, typename V>
static int run_decayed(const T* q, long q_stride, const T* k, long k_stride, const V* v, long v_stride, DecayWeights weights, const double* run,
                       float q_scale, float* state, long state_stride, const int* slots, const int* row_start, const int* row_len,
                       const int* row_ctx, float* out, float* below, int rows, int heads, int group, int dim, int value_dim, int ones,
                       float* sums, float* totals, int items, hipStream_t stream) {
    const int columns = value_dim + ones;
    if (sums != nullptr) {
        if (items <= 0 || (run == nullptr && totals == nullptr)) return -1;
        const dim3 chunk_grid(items, heads, (columns + 63) / 64);
        memory_chunk_sums_kernel<T, V><<<chunk_grid, 256, 0, stream>>>(k, k_stride, v, v_stride, weights, run, row_start, row_len, rows, sums, totals,
                                                                       heads, dim, value_dim, group, ones);
        run_carry(sums, run, totals, state, state_stride, slots, row_start, row_len, row_ctx, rows, heads, dim, value_dim, ones, 0, stream);
        if constexpr (sizeof(T) == 2) {
            // Its loads of queries and keys are of eight numbers, at multiples of 16 bytes.  A workgroup of it takes longer than one of the kernel
            // below and has 128 columns where that has 64, so it pays once those go more than one round over the compute units (256 of them;
            // two where half of its wavefronts would have no column).  All launches of a memory, us, the kernel below and this one: 16
            // heads of 128 x 128 and a column of ones, rows of 64 tokens (96 workgroups below) 36.3, 38.0; 256 (240) 43.1, 44.2; 320 (288) 52.4, 48.4; 1,024
            // 91, 84; three of 667 139, 110; 32 heads of 64 x 64, 512 tokens (288) 34.2, 36.2; eight rows of 64 (512) 32.1, 34.3; 16 of 16 (640) 42.3, 34.6.
            const long below_workgroups = (long)items * heads * ((columns + 63) / 64);
            const bool enough = below_workgroups > (columns > 64 ? 256 : 512);
            if (enough && dim % 32 == 0 && dim <= READ16_MOST && q_stride % 8 == 0 && k_stride % 8 == 0 && ((size_t)q | (size_t)k) % 16 == 0) {
                memory_chunk_read16_kernel<V><<<dim3(items, heads, (columns + 127) / 128), 256, 0, stream>>>(
                    q, q_stride, k, k_stride, v, v_stride, weights, run, q_scale, row_start, row_len, row_ctx, rows, sums, out, below, heads, dim, value_dim,
                    group, ones);
                LSA_LAUNCH_CHECK();
            }
        }
        memory_chunk_read_kernel<T, V><<<chunk_grid, 256, 0, stream>>>(q, q_stride, k, k_stride, v, v_stride, weights, run, q_scale, row_start, row_len,
                                                                       row_ctx, rows, sums, out, below, heads, dim, value_dim, group, ones);
        LSA_LAUNCH_CHECK();
    }
    int dk, waves;
    recurrence_lds(dim, dk, waves);
    const size_t lds = sizeof(float) * ((size_t)2 * CHUNK * waves * dk + (size_t)CHUNK * 64 + CHUNK + (size_t)waves * CHUNK * 64);
    if (lds > (size_t)MOST_LDS) return -1;
    dim3 grid(rows, heads, (columns + 63) / 64);
    // (items: without sums, how many tokens the step has; 0 if that is not known.)  About a token a row: see the kernel for both sides.  More
    // tokens are what the walk stages in LDS sixteen at a time.
    if (items > 0 && items <= rows && dk <= 16 && dim % dk == 0 && value_dim % 4 == 0 && state_stride % 4 == 0
        && q_stride * sizeof(T) % 16 == 0 && k_stride * sizeof(T) % 16 == 0 && v_stride % 4 == 0
        && ((size_t)state | (size_t)q | (size_t)k) % 16 == 0 && (size_t)v % (4 * sizeof(V)) == 0) {
        const int threads = (dim / dk * 16 + 63) / 64 * 64;
#define LSA_SINGLE(DK) \
        matrix_memory_single_kernel<T, V, DK><<<grid, threads, 0, stream>>>(q, q_stride, k, k_stride, v, v_stride, weights, q_scale, state, state_stride, \
            slots, row_start, row_len, row_ctx, out, below, heads, dim, value_dim, group, ones)
        if (dk == 8) LSA_SINGLE(8); else LSA_SINGLE(16);
#undef LSA_SINGLE
        LSA_LAUNCH_CHECK();
    }
#define LSA_LAUNCH(DK) \
        matrix_memory_kernel<T, V, DK><<<grid, waves * 64, lds, stream>>>(q, q_stride, k, k_stride, v, v_stride, weights, q_scale, state, state_stride, \
            slots, row_start, row_len, row_ctx, out, below, heads, dim, value_dim, group, ones)
    if (dk == 8) LSA_LAUNCH(8); else if (dk == 16) LSA_LAUNCH(16); else if (dk == 32) LSA_LAUNCH(32); else LSA_LAUNCH(64);
#undef LSA_LAUNCH
    LSA_LAUNCH_CHECK();
}

// state[slot]: the matrices [heads][dim][value_dim], the normalisers [heads][dim], the maxima [heads].
LSA_EXPORT int lsa_matrix_memory(int code, const void* q, long q_stride, const void* k, long k_stride, const void* v, long v_stride,
                                 const float* gates, float cap, float q_scale, float* state, long state_stride, const int* slots,
                                 const int* row_start, const int* row_len, const int* row_ctx, float* coef, float* out, float* below,
                                 int rows, int heads, int dim, int value_dim, double* run, float* sums, int items, hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > MOST_DIM || value_dim < 1 || heads < 1 || !(cap > 0.f) || state == nullptr || coef == nullptr || below == nullptr) return -1;
    if (state_stride < (long)heads * dim * value_dim + (long)heads * dim + heads || (run == nullptr) != (sums == nullptr)) return -1;
    memory_gates_kernel<<<dim3(rows, heads), 64 * GATES_WAVES, 0, stream>>>(gates, cap, state, state_stride, (long)heads * dim * value_dim + (long)heads * dim,
                                                              slots, row_start, row_len, row_ctx, coef, below, heads, run);
    const DecayWeights weights{coef, nullptr, 0, nullptr};
#define LSA_RUN(T) run_decayed<T, T>((const T*)q, q_stride, (const T*)k, k_stride, (const T*)v, v_stride, weights, run, q_scale, state, state_stride, \
                                     slots, row_start, row_len, row_ctx, out, below, rows, heads, 1, dim, value_dim, 1, sums, nullptr, items, stream)
    return code ? LSA_RUN(bf16_t) : LSA_RUN(float);
#undef LSA_RUN
}

// S_t = exp(log_keep) S_(t-1) + take k_t v_t^T, out_t = S_t^T (q_t q_scale) per head; groups of `group` heads share a query and a
// key head; queries and keys of one type, values of the same or, behind float32 queries and keys, bfloat16.
// state[slot]: the matrices [heads][dim][value_dim].
LSA_EXPORT int lsa_decayed_recurrence(int key_code, const void* q, long q_stride, const void* k, long k_stride, int value_code, const void* v,
                                      long v_stride, const float* log_keep, long log_stride, const float* take, float q_scale, float* state,
                                      long state_stride, const int* slots, const int* row_start, const int* row_len, const int* row_ctx, float* out,
                                      int rows, int heads, int group, int dim, int value_dim, float* sums, float* totals, int items,
                                      hipStream_t stream) {
    if (rows <= 0) return 0;
    if (dim < 1 || dim > MOST_DIM || value_dim < 1 || heads < 1 || group < 1 || heads % group || state == nullptr || log_keep == nullptr) return -1;
    if ((log_stride != 0 && log_stride != heads) || (key_code && !value_code)) return -1;
    const DecayWeights weights{nullptr, log_keep, log_stride, take};
#define LSA_RUN(T, V) run_decayed<T, V>((const T*)q, q_stride, (const T*)k, k_stride, (const V*)v, v_stride, weights, nullptr, q_scale, state, state_stride, \
                                        slots, row_start, row_len, row_ctx, out, nullptr, rows, heads, group, dim, value_dim, 0, sums, totals, items, stream)
    if (key_code) return LSA_RUN(bf16_t, bf16_t);
    return value_code ? LSA_RUN(float, bf16_t) : LSA_RUN(float, float);
#undef LSA_RUN
}

LSA_EXPORT int lsa_tanh(int code, void* x, long n, hipStream_t stream) {
    if (n <= 0) return 0;
    const int blocks = (int)((n + 255) / 256);
    if (code) tanh_kernel<bf16_t><<<blocks, 256, 0, stream>>>((bf16_t*)x, n);
    else tanh_kernel<float><<<blocks, 256, 0, stream>>>((float*)x, n);
    LSA_LAUNCH_CHECK();
}

LSA_EXPORT int lsa_scaled_sum(int code, const void* x, float a, const void* y, float b, void* out, long n, hipStream_t stream) {
    if (n <= 0) return 0;
    const int blocks = (int)((n + 255) / 256);
    if (code) scaled_sum_kernel<bf16_t><<<blocks, 256, 0, stream>>>((const bf16_t*)x, a, (const bf16_t*)y, b, (bf16_t*)out, n);
    else scaled_sum_kernel<float><<<blocks, 256, 0, stream>>>((const float*)x, a, (const float*)y, b, (float*)out, n);
    LSA_LAUNCH_CHECK();
}
