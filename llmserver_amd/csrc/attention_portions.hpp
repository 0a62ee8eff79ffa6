// Portions of prompts, 32 (token, head) pairs a wavefront: the kernel for workgroups of eight tiles of 16 pairs.  Included by attention.hip
// (bfloat16 only).
//
// MFMA use (32x32x16, lane = 32 * h + col):
//   scores:  S^T[key][pair] = K . Q^T      A = K rows (lane: key of col, dims 16 s + 8 h .. + 8), B = Q^T (lane: pair col, same dims)
//            leaves lane (h, col) the rows 8 i + 4 h + j of pair col.  Row 16 n + 8 i + 4 h + j of a block of 32 is key
//            16 n + 8 h + 4 i + j, so that those are, register by register, keys 16 n + 8 h + 0 .. 7:
//   output:  O^T[dim][pair] += V^T . P^T   A = V^T rows (lane: dim of col, keys 16 n + 8 h .. + 8), B = P^T, the rounded weights as they lie.
//
// Keys go by in blocks of 32.  While a block's weights are computed (exponentials: the vector unit), the matrix cores multiply the next block's keys
// and the values of the block before: three blocks are under way in a wavefront, and none of the three waits for another.  A trip of the
// loop is two blocks; each of the four wavefronts that share the keys brings 16 of the 64 keys and 16 of the 64 values that the next trip
// multiplies, straight into LDS, into rings of four blocks.  One barrier a trip.
//
// What bounds it: a block is 18 products (576 cycles of a matrix core) beside some 400 cycles of the vector unit, of which the exponentials take 256; two wavefronts a
// SIMD (one beyond head size 128) fill three fifths of the matrix cores.  Where every compute unit has many workgroups that is 1.0 PFLOP/s at head size 128 (of the 1.44 of a
// large product, at a clock that the card lowers by then); a single prompt waits for the workgroup with the most keys, 1.3 us a trip.  us, 16x16 products of 16 pairs
// with two tiles a wavefront before, this: 32 heads on 8 of 128, 2,048 tokens 70, 56, 8,192 tokens 694, 548; 16 on 16, 1,900 tokens 67, 39; 32 on 8 of 64,
// 2,048 tokens 48, 38; 190 tokens of 16 on 8 behind 8,064, captured (four tiles a workgroup before) 51, 34.
constexpr int PORTION_TILES = 8;                             // tiles of 16 pairs of a workgroup
constexpr int PK = 64;                                       // keys of a trip
constexpr int P_PIECES = 2 * ND;                             // 16-byte pieces of a key's row
constexpr int P_CHUNKS = (ND + 1) / 2;                       // 1 KB loads that bring 16 keys, or their values
constexpr int P_QUARTER = 1024 * P_CHUNKS, P_BLOCK = 2 * P_QUARTER;      // bytes of 16 and of 32 keys, or their values
constexpr int P_KEYS = 0, P_VALUES = 4 * P_BLOCK, P_RING = 8 * P_BLOCK;      // where the two rings lie, and what both take
constexpr int P_DIMS = (ND + 1) / 2;                         // blocks of 32 output dimensions
// LDS places.  Rows of keys lie end to end without padding; a row's pieces change places with each other (XOR) so that 16 lanes that read the same
// piece of 16 rows meet all 64 banks: rows whose length is P_SPREAD * 16 bytes times an odd number come back to the same banks after 16 / P_SPREAD rows.
// The two pieces of a value row (keys 0 .. 7 and 8 .. 15 of the quarter) change places in every other eight rows, for the same reason.
// (Counted: no bank conflicts, four cycles a read.)
constexpr int P_SPREAD = (P_PIECES & -P_PIECES) < 16 ? (P_PIECES & -P_PIECES) : 16;
__device__ __forceinline__ int piece_turn(int key) { return (key / (16 / P_SPREAD)) & (P_SPREAD - 1); }

// The larger of what a pair's two lanes have.
__device__ __forceinline__ float max_of_pair(float x) {
    const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
    const unsigned low = both[0], high = both[1];
    return fmaxf(__builtin_bit_cast(float, low), __builtin_bit_cast(float, high));
}
typedef float f32x16 __attribute__((ext_vector_type(16)));

// PAGES_OF_16: pages hold a multiple of 16 keys, so that 16 keys from a multiple of 16 on lie in one; otherwise of eight keys.
template <int HALVES, bool BIAS, bool PAGES_OF_16>
__global__ __launch_bounds__(256 * HALVES, LSA_MIN_WAVES) void paged_attention_portion_kernel(
    const elem_t* __restrict__ q, long q_token_stride, elem_t* __restrict__ out,
    const elem_t* __restrict__ keys, const elem_t* __restrict__ values,
    const int* __restrict__ table, int table_stride,
    const int* __restrict__ row_start, const int* __restrict__ row_len, const int* __restrict__ row_ctx,
    const Item* __restrict__ tiles, const TileSlots* __restrict__ tile_slots, float* __restrict__ part_acc, float* __restrict__ part_ml,
    Geometry g) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds_all[HALVES * P_RING];
    const int half = HALVES > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 8)) : 0;     // (the same in all lanes, and known to be)
    unsigned char* const lds = lds_all + half * P_RING;                // this half's: four blocks of keys, then four of values
    const unsigned lds_begin = (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)(size_t)(lds_ptr_t)lds_all + (unsigned)(half * P_RING)));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) & 3);
    const int heads = g.n_kv * g.gtiles;                               // (the KV head runs fastest over the XCDs, see paged_attention_tile_kernel)
    const Item tile = tiles[blockIdx.x / heads];
    const int head_index = blockIdx.x % heads;
    const int kv_head = head_index / g.gtiles, gtile = head_index % g.gtiles;
    const int col = lane & 31, h = lane >> 5;
    const int row = tile.row;
    const int n = row_len[row], first_pos = row_ctx[row] - n, token0 = row_start[row];
    const int q0 = tile.q0 + wave * 2 * g.tokens_per_tile;             // first token of this wavefront's two tiles
    const int of_tile = col & 15, which = col >> 4;
    const int pair_token = of_tile / g.gheads, pair_head_in_group = gtile * g.gheads + of_tile % g.gheads;
    const int head = kv_head * g.group + pair_head_in_group;
    const int token_of_row = q0 + which * g.tokens_per_tile + pair_token;
    const bool pair_valid = pair_token < g.tokens_per_tile && token_of_row < n && pair_head_in_group < g.group;
    const int q_pos = pair_valid ? first_pos + token_of_row : -1, first_seen = first_key_of(q_pos, g);
    float slope = 0.f;                                                 // (scores stay in units of 1 / scale, and so does what they lose per position)
    if constexpr (BIAS) slope = g.slopes[min(head, g.n_q - 1)] * g.scale_inverse;
    const int* row_table = table + (size_t)row * table_stride;
    const int ps = g.page_size;
    const size_t page_elems = (size_t)g.n_kv * ps * D;
    const elem_t* const head_keys = keys + (size_t)kv_head * ps * D;
    const elem_t* const head_values = values + (size_t)kv_head * D * ps;
    // Keys this wavefront's pairs can see at all: [wave_lo, wave_hi).
    const int wave_tokens = max(0, min(2 * g.tokens_per_tile, n - q0));
    const int wave_hi = wave_tokens > 0 ? first_pos + q0 + wave_tokens : 0;
    const int wave_lo = max(0, first_key_of(first_pos + q0, g));
    const float scale_log2 = g.scale * 1.44269504088896340736f;

    bf16x8 qf[ND];
#pragma unroll
    for (int s = 0; s < ND; ++s) {
        bf16x8 x = {0, 0, 0, 0, 0, 0, 0, 0};
        if (pair_valid) x = *reinterpret_cast<const bf16x8*>(q + (size_t)(token0 + token_of_row) * q_token_stride + (size_t)head * D + 16 * s + 8 * h);
        qf[s] = x;
    }
    f32x16 acc[P_DIMS];
#pragma unroll
    for (int c = 0; c < P_DIMS; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][r] = 0.f;
    float run_max = NEG_INF;                                           // in units of ln 2, scale applied
    f32x16 weight_sum;                                                 // of a pair's rounded weights, in the first number of both its lanes
#pragma unroll
    for (int r = 0; r < 16; ++r) weight_sum[r] = 0.f;

    // The steps of 64 keys that cover the tile's keys, and this half's share of them: [k_begin, k_end).
    const int first_step = (tile.k_begin / PK) * PK;
    const int all_steps = tile.k_begin < tile.k_end ? (tile.k_end - 1 - first_step) / PK + 1 : 0;
    const int trips = (all_steps + HALVES - 1) / HALVES;              // of every wavefront through the loop below
    const int cut = min(tile.k_end, first_step + PK * trips);         // where the second half's keys begin
    const int k_begin = half ? cut : tile.k_begin, k_end = half ? tile.k_end : cut;
    const int my_steps = half ? all_steps - trips : trips;

    // -- loads: lane `lane` of load m brings 16 bytes to place 64 m + lane of its wavefront's quarter --
    int key_offset[P_CHUNKS];                                          // from where the first of the 16 keys lies, in bytes
#pragma unroll
    for (int m = 0; m < P_CHUNKS; ++m) {
        const int place = min(64 * m + lane, 16 * P_PIECES - 1), key = place / P_PIECES;
        key_offset[m] = (PAGES_OF_16 ? key * (2 * D) : 0) + 16 * ((place % P_PIECES) ^ piece_turn(key));
    }
    const int value_key = 8 * ((lane & 1) ^ ((lane >> 4) & 1));        // the first of the piece's eight keys; its dimension is 32 m + lane / 2
    auto value_dim = [&](int m) { return 32 * m + 32 <= D ? lane >> 1 : min(lane >> 1, D - 1 - 32 * m); };      // ... beyond 32 m
    // Pages outside the range are never read (they may not be the request's): for 16 (or eight) keys that lie outside, the nearest ones that do not
    // stand in.  Scores and values of keys outside are masked and cleared where they are used.
    constexpr int UNIT = PAGES_OF_16 ? 16 : 8;
    const int last_unit = max(k_end - 1, 0) & ~(UNIT - 1), first_unit = min(k_begin & ~(UNIT - 1), last_unit);
    auto inside = [&](int key) { return min(max(key, first_unit), last_unit); };
    // Page numbers, 64 blocks of the table at a time, one in each lane.  After the load of the next 64 the wavefront waits for every load
    // it has in flight, this one included, and says so to the compiler: a wait that the compiler places itself would stand in every trip.
    int chunk = -1, chunk_pages = 0;
    auto page_of = [&](int first) __attribute__((always_inline)) {     // (`first` is the same in all lanes)
        const int block = (int)__umulhi((unsigned)inside(first), g.page_magic);
        if ((block >> 6) != chunk) {
            chunk = block >> 6;
            chunk_pages = row_table[min(64 * chunk + lane, table_stride - 1)];
            __builtin_amdgcn_s_waitcnt(0x0F70);
        }
        return __builtin_amdgcn_readlane(chunk_pages, block & 63);
    };
    auto slot_of = [&](int key) { return key - (int)__umulhi((unsigned)key, g.page_magic) * ps; };
    // Sixteen keys or values from `first` on, of the page `page` (pages of 8 keys and their odd multiples: every lane looks its key's page up).
    struct Source { const char* base; int first; unsigned to; };
    auto keys_from = [&](int first, int slot_of_ring, int page) {
        const unsigned to = lds_begin + (unsigned)(P_KEYS + slot_of_ring * P_BLOCK + (wave & 1) * P_QUARTER);
        return Source{reinterpret_cast<const char*>(head_keys + (size_t)(unsigned)page * page_elems) + slot_of(inside(first)) * (2 * D), first, to};
    };
    auto values_from = [&](int first, int slot_of_ring, int page) {
        const unsigned to = lds_begin + (unsigned)(P_VALUES + slot_of_ring * P_BLOCK + (wave & 1) * P_QUARTER);
        return Source{reinterpret_cast<const char*>(head_values + (size_t)(unsigned)page * page_elems + slot_of(inside(first))), first, to};
    };
    auto issue_keys = [&](const Source& from, int m) __attribute__((always_inline)) {
        if constexpr (PAGES_OF_16) {
            load_16_bytes_a_lane_to_lds(from.base, (unsigned)key_offset[m], from.to + 1024u * m);
        } else {
            const int wanted = from.first + min(64 * m + lane, 16 * P_PIECES - 1) / P_PIECES, key = inside(wanted & ~7) + (wanted & 7);
            const int block = (int)__umulhi((unsigned)key, g.page_magic);
            const char* source = reinterpret_cast<const char*>(head_keys + (size_t)row_table[block] * page_elems + (size_t)(key - block * ps) * D);
            load_16_bytes_a_lane_to_lds(source + key_offset[m], from.to + 1024u * m);
        }
    };
    auto issue_values = [&](const Source& from, int m) __attribute__((always_inline)) {
        if constexpr (PAGES_OF_16) {
            load_16_bytes_a_lane_to_lds(from.base + m * (64 * ps), (unsigned)(2 * (value_dim(m) * ps + value_key)), from.to + 1024u * m);
        } else {
            const int key = inside(from.first + value_key), block = (int)__umulhi((unsigned)key, g.page_magic);
            const elem_t* source = head_values + (size_t)row_table[block] * page_elems + (key - block * ps);
            load_16_bytes_a_lane_to_lds(source + (size_t)(32 * m + value_dim(m)) * ps, from.to + 1024u * m);
        }
    };

    // -- operands: where this lane reads them in a buffer --
    const int key_of_row = (col & 16) | (col & 4) << 1 | (col & 8) >> 1 | (col & 3);      // the key of row `col` of a block of 32
    const int key_row_at = (key_of_row >> 4) * P_QUARTER + (key_of_row & 15) * (2 * D), key_turn = piece_turn(key_of_row & 15);
    int key_at[P_SPREAD == 16 ? 1 : ND];
#pragma unroll
    for (int s = 0; s < (P_SPREAD == 16 ? 1 : ND); ++s) key_at[s] = key_row_at + 16 * ((2 * s + h) ^ key_turn);
    const int value_at = 16 * (2 * col + (h ^ ((col >> 3) & 1)));

    struct KeyOperands { bf16x8 part[ND]; };
    struct ValueOperands { bf16x8 part[2][P_DIMS]; };
    auto read_keys = [&](KeyOperands& k, int slot_of_ring) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < ND; ++s) {
            const int at = P_SPREAD == 16 ? (key_at[0] + slot_of_ring * P_BLOCK) ^ (32 * s) : key_at[P_SPREAD == 16 ? 0 : s] + slot_of_ring * P_BLOCK;
            k.part[s] = *reinterpret_cast<const bf16x8*>(lds + P_KEYS + at);
        }
    };
    auto read_values = [&](ValueOperands& v, int slot_of_ring) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int c = 0; c < P_DIMS; ++c) v.part[n][c] = *reinterpret_cast<const bf16x8*>(lds + P_VALUES + slot_of_ring * P_BLOCK + value_at + n * P_QUARTER + 1024 * c);
    };
    auto multiply_keys = [&](f32x16& scores, const KeyOperands& k, int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < ND; ++s)
            if (s >= from && s < to) scores = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k.part[s], qf[s], scores, 0, 0, 0);
    };
    struct Weights { bf16x8 part[2]; };                                // of a block's keys, rounded
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (bf16_t)1.f;
    auto multiply_values = [&](const ValueOperands& v, const Weights& w, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < P_DIMS; ++c) acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v.part[n][c], w.part[n], acc[c], 0, 0, 0);
        weight_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ones, w.part[n], weight_sum, 0, 0, 0);
    };
    // The keys that every pair of the wavefront sees lie in [full_from, full_to): blocks of those need no mask (lanes without a pair multiply
    // zeros by whatever lies there, and nobody asks for their results).  Trips that have anything for its pairs begin in (wave_lo - PK, wave_hi).
    const int full_from = max(k_begin, first_key_of(first_pos + q0 + wave_tokens - 1, g));
    const int full_to = min(k_end, first_pos + q0 + 1);
    // The running maximum follows only when a score beats it by more than half a unit of ln 2: until then weights grow to at most 1.41, and the
    // exchange between the lanes of a pair and the rescaling of the accumulators (400 cycles) are skipped.  What that costs in roundings (the largest weight is no
    // longer one exactly), the sum of the weights as they were rounded more than pays back: errors against float32 of 32 heads on 8 of 128, 2,048 tokens, scores
    // of spread 0.3, 1 and 3: 0.002083, 0.002008, 0.001758; every maximum followed and the weights summed as they were before 0.002097, 0.002016, 0.001758; a slack
    // of 8 0.002088, 0.002080, 0.001914 (and 10 % less time).
    constexpr float SLACK = 0.5f;
    float slack = NEG_INF;                                             // (no maximum yet: any score beats it)

    // A block of 32 keys at `kb`, whose scores are there: the products of the block before it with its values, its weights, the next block's scores.
    // `asked_for`: the loads that go out between those products, of either half of the block.
    auto block_of_keys = [&](f32x16& scores, f32x16& next_scores, Weights& weights, const Weights& weights_before, const ValueOperands& v, int kb,
                             int next_slot, auto more, auto ask) __attribute__((always_inline)) {
        if (g.cap > 0.f) {
#pragma unroll
            for (int r = 0; r < 16; ++r) scores[r] = capped(scores[r] * g.scale, g) * g.scale_inverse;
        }
        if constexpr (BIAS) {
            const float nearest = slope * (float)(kb + 8 * h - q_pos);
#pragma unroll
            for (int r = 0; r < 16; ++r) scores[r] += __builtin_fmaf(slope, (float)(16 * (r >> 3) + (r & 7)), nearest);
        }
        if (kb < full_from || kb + 32 > full_to) {
            // (masks are rare: what they need of the lane is kept from being worked out once for all blocks, which would hold registers through all of them)
            int of_lane = 8 * h;
            asm volatile("" : "+v"(of_lane));
            const int from = max(k_begin, first_seen) - kb - of_lane, to = min(k_end - 1, q_pos) - kb - of_lane;      // places that the pair sees: [from, to]
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int place = 16 * (r >> 3) + (r & 7);
                scores[r] = place >= from && place <= to ? scores[r] : NEG_INF;
            }
        }
        KeyOperands k;
        float shift = run_max == NEG_INF ? 0.f : -run_max;
        float top = NEG_INF;
        auto highest = [&](int part) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 8 * part; r < 8 * part + 8; ++r) top = fmaxf(top, __builtin_fmaf(scores[r], scale_log2, shift));
        };
        __builtin_amdgcn_sched_barrier(0);
        ask(0);
        multiply_values(v, weights_before, 0);
        highest(0);
        __builtin_amdgcn_sched_barrier(0);
        ask(1);
        multiply_values(v, weights_before, 1);
        read_keys(k, next_slot);
        highest(1);
        if (__any(top > slack)) {
            top = max_of_pair(top);
            const float before = run_max;
            run_max = before == NEG_INF ? top : before + fmaxf(top, 0.f);
            const float alpha = before == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(before - run_max);
            slack = run_max == NEG_INF ? NEG_INF : SLACK;
            shift = run_max == NEG_INF ? 0.f : -run_max;
            weight_sum[0] *= alpha;
#pragma unroll
            for (int c = 0; c < P_DIMS; ++c) acc[c] *= alpha;
        }
        auto weigh = [&](int part) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 8 * part; r < 8 * part + 8; ++r) {
                weights.part[part][r & 7] = (bf16_t)__builtin_amdgcn_exp2f(__builtin_fmaf(scores[r], scale_log2, shift));
            }
            asm volatile("" : "+v"(weights.part[part]));       // (the weights are worked out here, beside the products, and not where they are used)
        };
        ask(2);
        more();
        f32x16 x;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = 0.f;
        multiply_keys(x, k, 0, ND / 2);
        weigh(0);
        __builtin_amdgcn_sched_barrier(0);
        ask(3);
        multiply_keys(x, k, ND / 2, ND);
        weigh(1);
        next_scores = x;
        __builtin_amdgcn_sched_barrier(0);
    };
    // Values of keys outside the range may be anything (a page's places behind the context were never written): their weights are zero, and so
    // that zero times anything stays zero, the lane that brought them clears them in LDS, once they have landed and before the others read them.
    auto clear_values_outside = [&](int first, int slot_of_ring) __attribute__((always_inline)) {
        const int key = first + value_key;
        u32x4 keep;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            keep[i] = ((key + 2 * i >= k_begin && key + 2 * i < k_end) ? 0x0000ffffu : 0u) | ((key + 2 * i + 1 >= k_begin && key + 2 * i + 1 < k_end) ? 0xffff0000u : 0u);
        unsigned char* mine = lds + P_VALUES + slot_of_ring * P_BLOCK + (wave & 1) * P_QUARTER + 16 * lane;
#pragma unroll
        for (int m = 0; m < P_CHUNKS; ++m) *reinterpret_cast<u32x4*>(mine + 1024 * m) &= keep;
    };

    if (all_steps > 0) {
        // Trip t takes the softmax of blocks 2 t and 2 t + 1; it multiplies the keys of blocks 2 t + 1 and 2 t + 2 and the values of blocks 2 t - 1
        // and 2 t, and asks for what the next trip multiplies: from the keys of block 2 t + 3 on, and from the values of block 2 t + 1 on, 64 each, of which 16 a
        // wavefront.  Block b lies in slot b & 3 of its ring.  Loads are issued unconditionally, past either end too (stand-ins).
        const int begin = half ? first_step + PK * trips : first_step;
        // (every load so far has landed before the first one into LDS is issued: the compiler, which does not see
        // those, then never waits for "all loads" inside the loop on behalf of the queries)
        __builtin_amdgcn_s_waitcnt(0x0F70);
        int page_values = 0, page_keys = 0;
        const int mine = begin + 16 * wave;
        if (PAGES_OF_16) page_values = page_of(mine - 32), page_keys = page_of(mine + 32);
        {
            const Source before = keys_from(mine - 32, wave < 2 ? 3 : 0, page_values), ahead = keys_from(mine + 32, wave < 2 ? 1 : 2, page_keys);
            const Source values_before = values_from(mine - 32, wave < 2 ? 3 : 0, page_values);
#pragma unroll
            for (int m = 0; m < P_CHUNKS; ++m) issue_keys(before, m), issue_keys(ahead, m), issue_values(values_before, m);
        }
        f32x16 even, odd;
        Weights even_weights, odd_weights;
#pragma unroll
        for (int e = 0; e < 8; ++e) odd_weights.part[0][e] = odd_weights.part[1][e] = (bf16_t)0.f;
        auto scores_of = [&](int slot_of_ring) __attribute__((always_inline)) {
            KeyOperands k;
            read_keys(k, slot_of_ring);
#pragma unroll
            for (int r = 0; r < 16; ++r) even[r] = 0.f;
            multiply_keys(even, k, 0, ND);
        };
        // What trip `trip` multiplies has landed, and everybody is through with the blocks that the next loads overwrite.
        auto meet = [&](int trip) __attribute__((always_inline)) {
            const int parity = 2 * (trip & 1), first = begin + PK * trip - 32 + 16 * wave;
            if (first < k_begin || first + 16 > k_end) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                clear_values_outside(first, wave < 2 ? 3 - parity : parity);
            }
            loads_landed_then_barrier<0>();
        };
        Source ask_values, ask_keys;
        auto ask_ahead = [&](int trip) __attribute__((always_inline)) {
            const int parity = 2 * (trip & 1), first = begin + PK * trip + 32 + 16 * wave;
            page_values = page_keys;
            if (PAGES_OF_16) page_keys = page_of(first + PK);
            ask_values = values_from(first, wave < 2 ? 1 + parity : 2 - parity, page_values);
            ask_keys = keys_from(first + PK, wave < 2 ? 3 - parity : parity, page_keys);
        };
        auto ask_for = [&](bool keys, int from, int to) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < P_CHUNKS; ++m)
                if (m >= from && m < to) {
                    if (keys) issue_keys(ask_keys, m);
                    else issue_values(ask_values, m);
                }
        };
        // This wavefront's pairs see something in the trips [from, to); in the others it only brings its quarters and meets the rest.
        const int last_trip = min(my_steps, (wave_hi - begin + PK - 1) / PK), first_trip = max(0, (wave_lo - begin) / PK);
        const int from = wave_hi > begin && first_trip < last_trip ? first_trip : trips, to = from < trips ? last_trip : trips;
        loads_landed_then_barrier<0>();
        if (from == 0) scores_of(0);
        for (int trip = 0; trip < from; ++trip) {
            meet(trip);
            ask_ahead(trip);
            ask_for(false, 0, P_CHUNKS);
            ask_for(true, 0, P_CHUNKS);
            if (trip + 1 == from && from < to) scores_of(2 - 2 * (trip & 1));
        }
        for (int trip = from; trip < to; ++trip) {
            const int kt = begin + PK * trip, parity = 2 * (trip & 1);
            meet(trip);
            ValueOperands v;
            read_values(v, 3 - parity);
            ask_ahead(trip);
            block_of_keys(even, odd, even_weights, odd_weights, v, kt, 1 + parity, [&] { read_values(v, parity); },
                          [&](int quarter) { ask_for(false, quarter * P_CHUNKS / 4, (quarter + 1) * P_CHUNKS / 4); });
            block_of_keys(odd, even, odd_weights, even_weights, v, kt + 32, 2 - parity, [] {},
                          [&](int quarter) { ask_for(true, quarter * P_CHUNKS / 4, (quarter + 1) * P_CHUNKS / 4); });
        }
        meet(to);
        if (from < to) {                                               // the values of the last block
            ValueOperands v;
            read_values(v, 3 - 2 * (to & 1));
            multiply_values(v, odd_weights, 0);
            multiply_values(v, odd_weights, 1);
        }
        for (int trip = to; trip < trips; ++trip) {
            ask_ahead(trip);
            ask_for(false, 0, P_CHUNKS);
            ask_for(true, 0, P_CHUNKS);
            meet(trip + 1);
        }
    }
    // Where this entry's results go: the output, or a slot per tile (asked for here, at the end, where it is needed).
    TileSlots slots = {-1, 0};
    if (tile_slots != nullptr) slots = tile_slots[blockIdx.x / heads];
    loads_landed_then_barrier<0>();                                   // (the loads issued past the end still write LDS)
    float run_sum = weight_sum[0];
    float weight = 1.f;
    if constexpr (HALVES > 1) {
        // The second half's wavefronts hand over what they have; the first half's add it to theirs.
        constexpr int PER_WAVE = P_DIMS * 1024 + 64;                // floats: accumulators, then max and sum of 32 pairs
        static_assert(4 * PER_WAVE * sizeof(float) <= sizeof(lds_all), "the buffers of keys and values hold what the second half hands over");
        float* mine = reinterpret_cast<float*>(lds_all) + wave * PER_WAVE;
        if (half) {
#pragma unroll
            for (int c = 0; c < P_DIMS; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<f32x4*>(mine + ((4 * c + i) * 64 + lane) * 4) = (f32x4){acc[c][4 * i], acc[c][4 * i + 1], acc[c][4 * i + 2], acc[c][4 * i + 3]};
            if (h == 0) {
                mine[P_DIMS * 1024 + col] = run_max;
                mine[P_DIMS * 1024 + 32 + col] = run_sum;
            }
        }
        __syncthreads();
        if (half) return;
        const float other_max = mine[P_DIMS * 1024 + col], other_sum = mine[P_DIMS * 1024 + 32 + col];
        const float top = fmaxf(run_max, other_max);
        weight = run_max == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(run_max - top);
        const float other_weight = other_max == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(other_max - top);
        run_sum = weight * run_sum + other_weight * other_sum;
        run_max = top;
#pragma unroll
        for (int c = 0; c < P_DIMS; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 other = *reinterpret_cast<const f32x4*>(mine + ((4 * c + i) * 64 + lane) * 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[c][4 * i + j] = acc[c][4 * i + j] * weight + other[j] * other_weight;
            }
    }
    if (!pair_valid) return;
    const float max_seen = run_max == NEG_INF ? NEG_INF : run_max * 0.69314718055994530942f;
    if (slots.first >= 0) {
        const size_t base = ((size_t)(slots.first + (wave * 2 + which) * slots.stride) * heads + head_index) * 16 + of_tile;
        float* pa = part_acc + base * D + 4 * h;
#pragma unroll
        for (int c = 0; c < P_DIMS; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (32 * c + 8 * i < D)
                    *reinterpret_cast<f32x4*>(pa + 32 * c + 8 * i) = (f32x4){acc[c][4 * i], acc[c][4 * i + 1], acc[c][4 * i + 2], acc[c][4 * i + 3]};
        if (h == 0) {
            part_ml[base * 2] = max_seen;
            part_ml[base * 2 + 1] = run_sum;
        }
        return;
    }
    const size_t token = (size_t)(token0 + token_of_row);
    const float inv = inverse_of_sum(run_sum, max_seen, g.sinks, head) * gate_of(g, token, head);
    elem_t* o = out + (token * g.n_q + head) * D + 4 * h;
#pragma unroll
    for (int c = 0; c < P_DIMS; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (32 * c + 8 * i < D) {
                bf16x4 r4;
#pragma unroll
                for (int j = 0; j < 4; ++j) r4[j] = (bf16_t)(acc[c][4 * i + j] * inv);
                *reinterpret_cast<bf16x4*>(o + 32 * c + 8 * i) = r4;
            }
}
