// Attention of steps in which every row brings one token, row i's at place i of the step, and contexts are short: a part of attention.hip.
//
// A workgroup has a row's keys of one KV head all to itself, its wavefronts take the key steps in turn (wavefront w steps w, w + WAVES, ...)
// and meet in LDS at the end.  What bounds such a step is no stream but one chain: so many trips to memory one behind the other, then the
// instructions of one wavefront, one every five cycles or so.  The kernel for all steps (paged_attention_kernel) makes three trips (the
// item; its row; queries and keys) and brings 30 KB of instructions for ranges that begin and end anywhere.  Here the workgroup's place in the
// grid says the row, so that the context's length, the table's entries, the query, the rotation and the norm weights are one trip and the
// keys and values the second; keys outside the context are masked where they are used (a step always lies in pages that exist) instead of
// by addresses; and pages are looked up by a scalar, which takes pages of a multiple of 16 keys.
// Beyond a few dozen keys the keys and values themselves count: one compute unit pulls about 40 GB/s of them (bfloat16, 512 keys: 0.26 MB in 6 us).
// us a launch behind 64 MB of other reads, that kernel (with lsa_qk_norm_rope_kv_write in front where it cannot fuse) against this one, at contexts of
// 16, 128 and 512 keys:
//   bfloat16, 16 heads on 8 of 128 dimensions, 1 row 8.5, 8.7, 13.3 against 6.3, 7.5, 12.2; 32 rows 8.4, 9.8, 17.3 against 6.3, 8.7, 15.6
//   bfloat16, 16 heads on 1 of 256, 8 rows 9.3, 9.2, 20.8 against 6.4, 8.4, 18.4
//   float32, 16 heads on 8 of 128, 1 row 9.6, 12.1, 21.9 against 6.4, 9.5, 19.8; 32 rows 10.4, 14.5, 30.0 against 6.9, 11.1, 26.1
// (The host takes this kernel as long as every workgroup has a compute unit of its own, and beyond that where it stays the faster one.  float32, 16 heads
// on 1 of 256, 16, 128, 256 and 512 keys: 11.7, 18.3, 27.2, 43.9 against 9.8, 17.0, 27.2, 48.4: the last of these contexts are a little slower.)
// (Figures of one workgroup to a row's keys of a KV head.)  Where there are few rows, four workgroups share them (PARTS): what one compute unit pulls is the bound, so each
// reads all keys, forms all scores and takes a quarter of the value's dimensions, five eighths of the bytes, and nothing has to meet afterwards; the sums, and so the
// bits, are the same.  us, one workgroup and four, norm and rotation folded in, at contexts of 16, 128, 333 and 512 keys:
//   float32, 16 heads on 8 of 128, 1 row 7.5, 11.4, 17.5, 23.4 and 7.2, 9.8, 14.0, 17.8; 4 rows 7.6, 11.9, 18.6, 25.2 and 7.3, 10.1, 14.7, 19.0; 16 on 1 of 256, 4 rows 11.3, 20.4,
//   38.0, 51.5 and 9.0, 14.3, 22.6, 28.4
//   bfloat16, 16 heads on 8 of 128, 1 row 7.0, 8.7, 11.5, 14.5 and 6.8, 8.1, 10.3, 12.6; 8 rows (256 workgroups) 7.4, 9.5, 12.9, 16.4 and 7.2, 8.9, 11.9, 14.4; 16 on 1 of 256,
//   16 rows 9.5, 13.4, 19.2, 25.1 and 8.0, 10.2, 13.8, 17.1
// Eight wavefronts where registers and LDS allow it (up to 256 keys in one round), else four.  A thread computes one head's outputs at the end, so
// that few of them work out the wavefronts' weights (all of them doing so: 6.9 us instead of 6.2 at 40 keys).
#pragma once

// Over the four quads of a column, and over the sixteen columns of a quad; every lane gets the result.  (Exchanges between lanes without LDS,
// whose latency a single wavefront would wait out every time.)
template <typename F> __device__ __forceinline__ float over_quads(float x, F f) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const unsigned a = __builtin_bit_cast(unsigned, x);
    const u32x2 halves = __builtin_amdgcn_permlane32_swap(a, a, false, false);
    const unsigned first = halves[0], second = halves[1];
    const float y = f(__builtin_bit_cast(float, first), __builtin_bit_cast(float, second));
    const unsigned b = __builtin_bit_cast(unsigned, y);
    const u32x2 rows = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const unsigned even = rows[0], odd = rows[1];
    return f(__builtin_bit_cast(float, even), __builtin_bit_cast(float, odd));
}
template <int N> __device__ __forceinline__ float turned_in_row(float x) {                // column c gets column c + N's (of sixteen, in a circle)
    const int bits = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(bits, bits, 0x120 + N, 0xf, 0xf, false));      // row_ror:N
}
template <typename F> __device__ __forceinline__ float over_columns(float x, F f) {
    x = f(x, turned_in_row<8>(x));
    x = f(x, turned_in_row<4>(x));
    x = f(x, turned_in_row<2>(x));
    return f(x, turned_in_row<1>(x));
}
__device__ __forceinline__ float larger(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ float added(float a, float b) { return a + b; }

template <int MODE, int WAVES, int HEADS, int PARTS>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void attention_single_kernel(
    const elem_t* __restrict__ q, long q_token_stride, elem_t* __restrict__ out, const elem_t* keys, const elem_t* values,
    const int* __restrict__ table, int table_stride, const int* __restrict__ row_ctx, Geometry g, DecodeFusion fusion) {
    constexpr bool FUSED = (MODE & 1) != 0, NEW_TOKEN = (MODE & 2) != 0;
    // HEADS > 0 (float32 only): that many query heads share the KV head, and the products are plain multiply-adds of a lane's own
    // numbers: the 32-bit matrix products would do sixteen columns' work for one or two of them (1,024 cycles against 128 a step and head).
    constexpr bool VECTOR = HEADS > 0;
    // PARTS workgroups share a row's keys of a KV head: each forms all scores and takes a part of the value's dimensions, first_value on.
    constexpr int NV = ND / PARTS;
    const int first_value = PARTS == 1 ? 0 : (int)blockIdx.z * 16 * NV;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int col = lane & 15, quad = lane >> 4;
    const int row = blockIdx.x, kv_head = blockIdx.y / g.gtiles, gtile = blockIdx.y % g.gtiles;
    const int ps = g.page_size;
    const size_t page_elems = (size_t)g.n_kv * ps * D;
    const int* row_table = table + (size_t)row * table_stride;
    const int ctx = row_ctx[row], q_pos = ctx - 1;
    // The column's query head; columns behind the last head repeat it (their results are dropped).
    const int heads = min(g.gheads, g.group - gtile * g.gheads), first_head = kv_head * g.group + gtile * g.gheads;
    const int head = first_head + min(col, heads - 1);
    const elem_t* token = q + (size_t)row * q_token_stride;
    const int lo = max(first_key_of(q_pos, g), 0), hi = NEW_TOKEN ? ctx - 1 : ctx;       // the keys that come from pages
    // Page ids: lane l holds the entry of block l, which is asked for before anybody knows how many there are; contexts of more than 64 blocks
    // look the others up one by one.  An entry that names no page stands for any page: its keys are masked.
    const int pages = row_table[min(lane, table_stride - 1)];
    auto page_of = [&](int key) {
        const int block = (int)__umulhi((unsigned)key, g.page_magic);
        const int page = block < 64 ? __builtin_amdgcn_readlane(pages, block) : row_table[min(block, table_stride - 1)];
        return (size_t)max(page, 0) * page_elems;
    };

#if LSA_BF16
    constexpr int PIECE = 8;                                       // neighbouring dimensions a lane holds of every 4 * PIECE
    typedef bf16x8 piece_t;
#else
    constexpr int PIECE = 4;
    typedef f32x4 piece_t;
#endif
    struct Step {
        piece_t k[KEY_STEP / 16][NS];
#if LSA_BF16
        bf16x4 v[NV][2];
#else
        f32x4 v[NV];
#endif
    };
    auto load_step = [&](Step& f, int kt) {
#pragma unroll
        for (int t = 0; t < KEY_STEP / 16; ++t) {
            const int first = kt + 16 * t;
            const size_t page = page_of(first);
            const int slot = first - (int)__umulhi((unsigned)first, g.page_magic) * ps;
            const elem_t* kp = keys + page + ((size_t)kv_head * ps + slot + col) * D + PIECE * quad;
#pragma unroll
            for (int s = 0; s < NS; ++s) f.k[t][s] = *reinterpret_cast<const piece_t*>(kp + 4 * PIECE * s);
            const elem_t* vp = values + page + ((size_t)kv_head * D + first_value + col) * ps + slot + 4 * quad;
#pragma unroll
            for (int c = 0; c < NV; ++c) {
#if LSA_BF16
                f.v[c][t] = *reinterpret_cast<const bf16x4*>(vp + (size_t)(16 * c) * ps);
#else
                f.v[c] = *reinterpret_cast<const f32x4*>(vp + (size_t)(16 * c) * ps);
#endif
            }
        }
    };

    // First trip: beside the context's length and the table, all that the queries need.
    piece_t qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = *reinterpret_cast<const piece_t*>(token + (size_t)head * D + 4 * PIECE * s + PIECE * quad);
    constexpr int F = FUSED ? NS : 1, H = FUSED ? NS / 2 : 1;
    f32x4 weights[F][PIECE / 4], cosines[H][PIECE / 4], sines[H][PIECE / 4];
    if constexpr (FUSED) {
        const float* cs = fusion.cos_sin + (size_t)row * D + PIECE * quad;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int p = 0; p < PIECE / 4; ++p) {
                weights[s][p] = *reinterpret_cast<const f32x4*>(fusion.q_weight + 4 * PIECE * s + PIECE * quad + 4 * p);
                if (s < NS / 2) {
                    cosines[s][p] = *reinterpret_cast<const f32x4*>(cs + 4 * PIECE * s + 4 * p);
                    sines[s][p] = *reinterpret_cast<const f32x4*>(cs + D / 2 + 4 * PIECE * s + 4 * p);
                }
            }
    }
    // Which outputs a thread writes at the very end, always of one head (VECTOR: one of its 16 * NV; else four neighbouring ones, every `places`th of
    // them), and that head's sink and gate (where there is none, any number will do).
    const int places = VECTOR ? 1 : 64 * WAVES / heads, my_head = VECTOR ? (int)threadIdx.x / (16 * NV) : (int)threadIdx.x % heads;
    const int my_place = VECTOR ? (int)threadIdx.x % (16 * NV) : (int)threadIdx.x / heads;
    const int last_head = first_head + min(my_head, heads - 1);
    const float sink = *(g.sinks != nullptr ? g.sinks + last_head : reinterpret_cast<const float*>(row_ctx));
    const float gate = (float)*(g.gates != nullptr ? g.gates + (size_t)row * g.gate_stride + last_head : token);
    float slope = 0.f;
    if constexpr (!FUSED && !VECTOR) if (g.slopes != nullptr) slope = g.slopes[head];
    // The new token is the last wavefront's, which has the fewest steps.
    piece_t kh[NEW_TOKEN ? NS : 1];
    const bool takes_new_token = NEW_TOKEN && wave == WAVES - 1;
    const int first_step = lo / KEY_STEP;
    int kt = (first_step + wave) * KEY_STEP;
    Step now;

    // A head in the operands' layout, normalised over the head and rotated as lsa_qk_norm_rope_kv_write does it; the four quads of a
    // column share a head.
    auto norm_rotate = [&](piece_t (&h)[NS]) {
        float x[NS][PIECE], sq = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < PIECE; ++e) {
                x[s][e] = (float)h[s][e];
                sq += x[s][e] * x[s][e];
            }
        sq = over_quads(sq, added);
        const float rstd = rsqrtf(sq / (float)D + fusion.eps);
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < PIECE; ++e) x[s][e] = x[s][e] * rstd * weights[FUSED ? s : 0][e / 4][e % 4];
#pragma unroll
        for (int s = 0; s < NS / 2; ++s)
#pragma unroll
            for (int e = 0; e < PIECE; ++e) {
                const float co = cosines[FUSED ? s : 0][e / 4][e % 4], si = sines[FUSED ? s : 0][e / 4][e % 4];
                const float x1 = x[s][e], x2 = x[s + NS / 2][e];
                x[s][e] = x1 * co - x2 * si;
                x[s + NS / 2][e] = x2 * co + x1 * si;
            }
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < PIECE; ++e) h[s][e] = (elem_t)x[s][e];
    };
    // Second trip: the first keys and values, under way while the queries are prepared; or the new token's.  (No branch joins another between
    // the loads and that work, or it would wait for all of them.)
    if (takes_new_token) {
#pragma unroll
        for (int s = 0; s < (NEW_TOKEN ? NS : 1); ++s) kh[s] = *reinterpret_cast<const piece_t*>(token + (size_t)(g.n_q + kv_head) * D + 4 * PIECE * s + PIECE * quad);
        if constexpr (FUSED) norm_rotate(qf);
    } else if (kt < hi) {
        load_step(now, kt);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (FUSED) norm_rotate(qf);
    }

    constexpr int R = VECTOR ? HEADS : 1;                          // running maxima and sums a lane keeps
    float run_max[R], run_sum[R];
#pragma unroll
    for (int h = 0; h < R; ++h) {
        run_max[h] = NEG_INF;
        run_sum[h] = 0.f;
    }
#if !LSA_BF16
    // (VECTOR) The heads' queries, in LDS for the whole step (a lane reads its quad's numbers of a head, the same for all columns: in
    // registers they would leave no room for the next step's keys), and a lane's share of the output: dimension 16 c + col, keys of its quad.
    __shared__ f32x4 queries[VECTOR ? WAVES : 1][VECTOR ? HEADS : 1][VECTOR ? NS * 4 : 1];
    float share[VECTOR ? HEADS : 1][VECTOR ? NV : 1];
    auto query = [&](int h, int s) { return queries[VECTOR ? wave : 0][h][VECTOR ? 4 * s + quad : 0]; };
    if constexpr (VECTOR) {
        if (col < HEADS) {
#pragma unroll
            for (int s = 0; s < NS; ++s) queries[wave][col][4 * s + quad] = qf[s];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < HEADS; ++h)
#pragma unroll
            for (int c = 0; c < NV; ++c) share[h][c] = 0.f;
    }
#endif
    f32x4 acc[VECTOR ? 1 : NV];
    if constexpr (!VECTOR) {
#pragma unroll
        for (int c = 0; c < NV; ++c) acc[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    if constexpr (NEW_TOKEN) if (takes_new_token) {
        // The softmax starts from the new token's key (maximum = its score, sum = 1, output = its value); its key and value go into the cache.
        const int slot = q_pos - (int)__umulhi((unsigned)q_pos, g.page_magic) * ps;
        const int entry = row_table[min((int)__umulhi((unsigned)q_pos, g.page_magic), table_stride - 1)];
        const elem_t* vh = token + (size_t)(g.n_q + g.n_kv + kv_head) * D + first_value;
#if LSA_BF16
        bf16x4 vnew[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) vnew[c] = *reinterpret_cast<const bf16x4*>(vh + 16 * c + 4 * quad);
#else
        f32x4 vnew[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) vnew[c] = *reinterpret_cast<const f32x4*>(vh + 16 * c + 4 * quad);
#endif
        if constexpr (FUSED) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int p = 0; p < PIECE / 4; ++p)
                    weights[s][p] = *reinterpret_cast<const f32x4*>(fusion.k_weight + 4 * PIECE * s + PIECE * quad + 4 * p);
            norm_rotate(kh);
        }
        if constexpr (VECTOR) {
#if !LSA_BF16
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                float dot = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const f32x4 mine = query(h, s);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dot += kh[s][e] * mine[e];
                }
                dot = over_quads(dot, added);
                run_max[h] = dot * g.scale;
                run_sum[h] = 1.f / 16.f;                           // (of the column's sixteenth: the sums of the columns are added up)
                // the value's dimension 16 c + col, in quad 0 alone
#pragma unroll
                for (int c = 0; c < NV; ++c) share[h][c] = quad == 0 ? vh[16 * c + col] : 0.f;
            }
#endif
        } else {
            float dot = 0.f;
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int e = 0; e < PIECE; ++e) dot += (float)kh[s][e] * (float)qf[s][e];
            dot = over_quads(dot, added);
            run_max[0] = capped(dot * g.scale, g);
            run_sum[0] = quad == 0 ? 1.f : 0.f;
#pragma unroll
            for (int c = 0; c < NV; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[c][r] = (float)vnew[c][r];
        }
        if (col == 0 && entry >= 0 && gtile == 0) {
            elem_t* kp = const_cast<elem_t*>(keys) + (size_t)entry * page_elems + ((size_t)kv_head * ps + slot) * D + PIECE * quad;
            if (first_value == 0) {
#pragma unroll
                for (int s = 0; s < NS; ++s) *reinterpret_cast<piece_t*>(kp + 4 * PIECE * s) = kh[s];
            }
            elem_t* vp = const_cast<elem_t*>(values) + (size_t)entry * page_elems + ((size_t)kv_head * D + first_value + 4 * quad) * ps + slot;
#pragma unroll
            for (int c = 0; c < NV; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) vp[(size_t)(16 * c + r) * ps] = vnew[c][r];
        }
        if (kt < hi) load_step(now, kt);
    }

    while (kt < hi) {
        const int following = kt + WAVES * KEY_STEP;
        Step next;                                                 // its loads are under way while this one is multiplied
        if (following < hi) load_step(next, following);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (VECTOR) {
#if !LSA_BF16
            const int key = kt + col;
            const bool seen = key >= lo && key < hi;
#pragma unroll
            for (int r = 0; r < 4; ++r) {                          // values of keys outside may hold anything: keep them out of the sum
                const bool there = kt + 4 * quad + r >= lo && kt + 4 * quad + r < hi;
#pragma unroll
                for (int c = 0; c < NV; ++c) now.v[c][r] = there ? now.v[c][r] : 0.f;
            }
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                float dot = 0.f;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const f32x4 mine = query(h, s);
#pragma unroll
                    for (int e = 0; e < 4; ++e) dot += now.k[0][s][e] * mine[e];
                }
                dot = over_quads(dot, added);
                const float score = seen ? dot * g.scale : NEG_INF;
                const float new_max = fmaxf(run_max[h], over_columns(score, larger)), use_max = new_max == NEG_INF ? 0.f : new_max;
                const float alpha = expf(run_max[h] - use_max), p = expf(score - use_max);
                run_max[h] = new_max;
                run_sum[h] = run_sum[h] * alpha + p;
                float weight[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) weight[r] = __shfl(p, 16 * quad + 4 * quad + r, 64);
#pragma unroll
                for (int c = 0; c < NV; ++c) {
                    float sum = share[h][c] * alpha;
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum += weight[r] * now.v[c][r];
                    share[h][c] = sum;
                }
            }
#endif
        } else {
            constexpr int T = KEY_STEP / 16;
            float score[T][4], top = NEG_INF;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < NS; ++s) {
#if LSA_BF16
                    s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now.k[t][s], qf[s], s4, 0, 0, 0);
#else
#pragma unroll
                    for (int e = 0; e < 4; ++e) s4 = __builtin_amdgcn_mfma_f32_16x16x4f32(now.k[t][s][e], qf[s][e], s4, 0, 0, 0);
#endif
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int key = kt + 16 * t + 4 * quad + r;
                    const float v = capped(s4[r] * g.scale, g) - slope * (float)(q_pos - key);
                    score[t][r] = key >= lo && key < hi ? v : NEG_INF;
                    top = fmaxf(top, score[t][r]);
                }
            }
            const float new_max = fmaxf(run_max[0], over_quads(top, larger)), use_max = new_max == NEG_INF ? 0.f : new_max;
#if LSA_BF16
            const float alpha = __expf(run_max[0] - use_max);
#else
            const float alpha = expf(run_max[0] - use_max);
#endif
            run_max[0] = new_max;
            run_sum[0] *= alpha;
#if LSA_BF16
            bf16x8 weight;
            unsigned keep[2][2];                                   // (pairs of bfloat16) values of keys outside may hold anything
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = __expf(score[t][r] - use_max);
                    run_sum[0] += p;
                    weight[4 * t + r] = (bf16_t)p;
                    const int key = kt + 16 * t + 4 * quad + r;
                    const unsigned there = key >= lo && key < hi ? 0xffffu << (16 * (r & 1)) : 0u;
                    keep[t][r / 2] = r & 1 ? keep[t][r / 2] | there : there;
                }
#pragma unroll
            for (int c = 0; c < NV; ++c) {
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
                const u32x2 a = __builtin_bit_cast(u32x2, now.v[c][0]), b = __builtin_bit_cast(u32x2, now.v[c][1]);
                const u32x4_t both = {a[0] & keep[0][0], a[1] & keep[0][1], b[0] & keep[1][0], b[1] & keep[1][1]};
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, both), weight, acc[c] * alpha, 0, 0, 0);
            }
#else
            float weight[4];
            bool there[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                weight[r] = expf(score[0][r] - use_max);
                run_sum[0] += weight[r];
                there[r] = kt + 4 * quad + r >= lo && kt + 4 * quad + r < hi;
            }
#pragma unroll
            for (int c = 0; c < NV; ++c) {
                acc[c] *= alpha;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(there[r] ? now.v[c][r] : 0.f, weight[r], acc[c], 0, 0, 0);
            }
#endif
        }
        if (following < hi) now = next;
        kt = following;
    }

    // The wavefronts' sums meet in LDS, CHUNK times 16 dimensions a round; every wavefront gets here, and the loop's trips are the workgroup's.
    constexpr int CHUNK = NV < 8 ? NV : 8;
    extern __shared__ f32x4 partial[];                             // [WAVES][CHUNK][4][heads], VECTOR: [WAVES][HEADS][CHUNK][16] of four quads' shares
    __shared__ float wave_max_of[WAVES][16], wave_sum_of[WAVES][16];
    if constexpr (VECTOR) {
#pragma unroll
        for (int h = 0; h < R; ++h) {
            const float sum = over_columns(run_sum[h], added);
            if (lane == 0) {
                wave_max_of[wave][h] = run_max[h];
                wave_sum_of[wave][h] = sum;
            }
        }
    } else {
        run_sum[0] = over_quads(run_sum[0], added);
        if (quad == 0) {
            wave_max_of[wave][col] = run_max[0];
            wave_sum_of[wave][col] = run_sum[0];
        }
    }
    // What a wavefront's sums of head h of the tile count at the very end (inverse_of_sum and gate_of, from what was asked for at the start).
    float scale_of[WAVES];
    auto find_scales = [&](int h) {
        float top = NEG_INF, total = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) top = fmaxf(top, wave_max_of[w][h]);
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float m = wave_max_of[w][h];
            scale_of[w] = m == NEG_INF ? 0.f : expf(m - top);
            total += scale_of[w] * wave_sum_of[w][h];
        }
        float inv = 0.f;
        if (total > 0.f && top != NEG_INF) {
            inv = 1.f / total;
            if (g.sinks != nullptr) {
                const float common = fmaxf(top, sink), kept = expf(top - common);
                inv = kept / (total * kept + expf(sink - common));
            }
            if (g.gates != nullptr) inv *= 1.f / (1.f + expf(-gate));
        }
#pragma unroll
        for (int w = 0; w < WAVES; ++w) scale_of[w] *= inv;
    };
    elem_t* row_out = out + ((size_t)row * g.n_q + first_head) * D + first_value;
#pragma unroll
    for (int c0 = 0; c0 < NV; c0 += CHUNK) {
        if (c0) __syncthreads();                                   // (the round before has been read)
        const int chunk = min(CHUNK, NV - c0);
        if constexpr (VECTOR) {
#if !LSA_BF16
#pragma unroll
            for (int h = 0; h < R; ++h)
#pragma unroll
                for (int c = 0; c < CHUNK; ++c)
                    if (c0 + c < NV) reinterpret_cast<float*>(partial)[(((wave * HEADS + h) * CHUNK + c) * 16 + col) * 4 + quad] = share[h][c0 + c];
            __syncthreads();
            static_assert(CHUNK == NV && CHUNK * 16 * HEADS <= 64 * WAVES, "an output a thread");
            if (my_head < HEADS) {
                find_scales(my_head);
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < WAVES; ++w) sum += partial[((w * HEADS + my_head) * CHUNK) * 16 + my_place] * scale_of[w];
                row_out[(size_t)my_head * D + my_place] = (elem_t)((sum[0] + sum[1]) + (sum[2] + sum[3]));
            }
#endif
        } else {
#pragma unroll
            for (int c = 0; c < CHUNK; ++c)
                if (c0 + c < NV && col < heads) partial[((wave * CHUNK + c) * 4 + quad) * heads + col] = acc[c0 + c];
            __syncthreads();
            if (my_place < chunk * 4 && my_place < places) {
                if (c0 == 0) find_scales(my_head);
                for (int place = my_place; place < chunk * 4; place += places) {
                    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int w = 0; w < WAVES; ++w) sum += partial[(w * CHUNK * 4 + place) * heads + my_head] * scale_of[w];
                    elem_t* o = row_out + (size_t)my_head * D + 16 * c0 + 4 * place;
#if LSA_BF16
                    bf16x4 four;
#pragma unroll
                    for (int r = 0; r < 4; ++r) four[r] = (bf16_t)sum[r];
                    *reinterpret_cast<bf16x4*>(o) = four;
#else
                    *reinterpret_cast<f32x4*>(o) = sum;
#endif
                }
            }
        }
    }
}
