// Matrix products of many rows, Y[M, N] = X[M, K] . W[N, K]^T in bfloat16 with 32-bit sums, for prompts and portions of prompts: where the library's tiles leave
// compute units idle (some hundred rows, small weights), and where what follows the product can go into it:
//   plain       round(sum)
//   gated       W stacks a gate matrix on an up matrix ([2N, K], gate first): round(act(gate) * up), [M, N]
//   activated   round(act(sum))
//   sums        the sums themselves, of `parts` ranges of K, [parts, M, N] in 32-bit: whoever reads the product adds them up
//
// Two kernels.  The one below has small tiles, which a step of a few hundred rows has enough of to go round the compute units; the other one multiplies tiles
// of 256 x 256 (wide_product.hpp) for prompts of a thousand tokens and more.
#include "common.hpp"
#include "lds_loads.hpp"
#include "wide_product.hpp"

using namespace lsa;

enum Form { PLAIN, GATED, ACTIVATED, SUMS };
enum Activation { SILU, GELU_TANH, RELU2 };          // (the last one has no gated form)

__device__ __forceinline__ float activation_of(int activation, float z) {
    if (activation == SILU) return z / (1.f + expf(-z));
    if (activation == GELU_TANH) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    const float r = fmaxf(z, 0.f);
    return r * r;
}

constexpr int XCDS = 8;
// Workgroups go to the eight XCDs in turn by their number: an XCD gets neighbours of an order that walks eight rows of tiles through all columns, so that the
// rows of X stay in its L2 while every row of W comes into it once.
__device__ __forceinline__ bool tile_of_workgroup(int rows, int columns, int& row, int& column) {
    const int tiles = rows * columns, share = (tiles + XCDS - 1) / XCDS, index = blockIdx.x / XCDS, tile = (int)(blockIdx.x % XCDS) * share + index;
    if (index >= share || tile >= tiles) return false;
    const int group = tile / (8 * columns), within = tile - group * 8 * columns, group_rows = min(8, rows - 8 * group);
    row = 8 * group + within % group_rows;
    column = within / group_rows;
    return true;
}
static int workgroups(int M, int N, int tile_m, int tile_n) {
    const long tiles = (long)((M + tile_m - 1) / tile_m) * ((N + tile_n - 1) / tile_n);
    return tiles > (1 << 24) - XCDS ? -1 : (int)((tiles + XCDS - 1) / XCDS * XCDS);
}

constexpr int SLAB = 64;

// Tiles of 16 MI WAVES_M rows x 32 WAVES_N columns (GATED: half of them gate columns, half their up columns), a wavefront 16 MI x 32.  Slabs of 64 of K go
// through BUFFERS buffers of LDS that loads fill without registers, BUFFERS - 1 slabs ahead; one barrier a slab.  grid (tiles, parts), a part of K each.
//   What bounds it: with every tile on a compute unit of its own a slab takes 0.25 us (64 x 64 tiles, 4 wavefronts), 0.31 (128 x 64, 8) and 0.5 (128 x 128, 8), in
// turn waiting, reading LDS and multiplying, and a launch 3 to 4 us around them; the kernel is for products of one such round, whatever the chip could
// do with more.  us alone, library and here: 190 rows, 4,096 x 2,048 13.8, 11.9; 2,048 x 2,048 in four parts 12.0, 7.6; 12,288 x 2,048 26.3, 20.6; 2,048 x 6,144 in four
// parts 22.9, 13.6; 1,000 rows, 4,096 x 2,048 23.9, 20.7; 2,048 rows, 2,048 x 2,048 24.6, 21.9.  No faster: operands of half a slab read while the other half is
// multiplied; slabs shared by groups of wavefronts that add up in LDS; four wavefronts of 64 x 64.
template <int WAVES_M, int WAVES_N, int MI, int BUFFERS, int FORM>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void product_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out,
                                                                         int M, int N, int K, int activation) {
    constexpr int TILE_M = WAVES_M * MI * 16, TILE_B = WAVES_N * 32, COLUMNS = FORM == GATED ? TILE_B / 2 : TILE_B, WAVES = WAVES_M * WAVES_N;
    constexpr int BUFFER = (TILE_M + TILE_B) * SLAB * 2, A_LOADS = TILE_M / 8 / WAVES, B_LOADS = TILE_B / 8 / WAVES, LOADS = A_LOADS + B_LOADS;
    static_assert(TILE_M % (8 * WAVES) == 0 && TILE_B % (8 * WAVES) == 0 && BUFFERS * BUFFER <= 160 * 1024, "a load is 8 rows");
    __shared__ __attribute__((aligned(1024))) unsigned char buffers[BUFFERS * BUFFER];
    int tile_m, tile_n;
    if (!tile_of_workgroup((M + TILE_M - 1) / TILE_M, (N + COLUMNS - 1) / COLUMNS, tile_m, tile_n)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), col = lane & 15, quad = lane >> 4;
    const int wave_m = wave / WAVES_N, wave_n = wave % WAVES_N, m0 = tile_m * TILE_M, n0 = tile_n * COLUMNS;
    const int all = K / SLAB, first = (int)((long)all * blockIdx.y / gridDim.y), slabs = (int)((long)all * (blockIdx.y + 1) / gridDim.y) - first;
    const buffer_t a_buffer = buffer_at(x + (size_t)m0 * K), b_buffer = buffer_at(w + (FORM == GATED ? 0 : (size_t)n0 * K));
    // The eight 16-byte pieces of row r stand at places piece ^ f(r), so that sixteen lanes whose reads are served together meet all 64 banks.  Rows of W are read in
    // the order of the columns (GATED: sixteen gate rows and their up rows for each 32), or so that a lane has eight neighbouring columns of the result.
    unsigned a_at[A_LOADS], b_at[B_LOADS];
#pragma unroll
    for (int u = 0; u < A_LOADS; ++u) {
        const int r = 8 * (wave + WAVES * u) + (lane >> 3);
        a_at[u] = (unsigned)min(r, M - 1 - m0) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ (r >> 1 & 7));
    }
#pragma unroll
    for (int u = 0; u < B_LOADS; ++u) {
        const int r = 8 * (wave + WAVES * u) + (lane >> 3);
        if (FORM == GATED) {
            const int c = min(n0 + 16 * (r >> 5) + (r & 15), N - 1);
            b_at[u] = (unsigned)(c + (r & 16 ? N : 0)) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ (r >> 1 & 7));
        } else {
            b_at[u] = (unsigned)min(r, N - 1 - n0) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ ((r >> 1 & 1) | (r >> 3 & 3) << 1));
        }
    }
    unsigned place = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(lds_ptr_t)buffers) + 1024 * wave;
    int asked = 0, slot = 0;
    auto ask = [&]() __attribute__((always_inline)) {
        const unsigned from = (first + min(asked, slabs - 1)) * (2 * SLAB);       // (behind the last slab: that once more, into a buffer that nobody reads again)
#pragma unroll
        for (int u = 0; u < A_LOADS; ++u) load_16_bytes_a_lane_to_lds(a_buffer, a_at[u], from, place + 1024 * WAVES * u);
#pragma unroll
        for (int u = 0; u < B_LOADS; ++u) load_16_bytes_a_lane_to_lds(b_buffer, b_at[u], from, place + TILE_M * 128 + 1024 * WAVES * u);
        ++asked;
        slot = slot == BUFFERS - 1 ? 0 : slot + 1;
        place += slot == 0 ? -(BUFFERS - 1) * BUFFER : BUFFER;
    };
    f32x4 sums[MI][2];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) sums[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int pieces[2] = {16 * (quad ^ (col >> 1)), 16 * ((quad + 4) ^ (col >> 1))};
    const unsigned char* a_rows = buffers + (16 * MI * wave_m + col) * 128;
    const unsigned char* b_rows = buffers + (TILE_M + 32 * wave_n + (FORM == GATED ? col : 8 * (col >> 2) + (col & 3))) * 128;
    constexpr int B_STEP = (FORM == GATED ? 16 : 4) * 128;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (the count below starts from nothing under way)
#pragma unroll
    for (int b = 0; b < BUFFERS - 1; ++b) ask();
    int buffer = 0;
    for (int slab = 0; slab < slabs; ++slab) {
        loads_landed_then_barrier<LOADS * (BUFFERS - 2)>();        // and everybody is through with the slab before this one, whose buffer is asked for
        bf16x8 a[2][MI], b[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < MI; ++i) a[s][i] = *reinterpret_cast<const bf16x8*>(a_rows + buffer + 2048 * i + pieces[s]);
#pragma unroll
            for (int j = 0; j < 2; ++j) b[s][j] = *reinterpret_cast<const bf16x8*>(b_rows + buffer + B_STEP * j + pieces[s]);
        }
        __builtin_amdgcn_sched_barrier(0);
        ask();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) sums[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s][j], a[s][i], sums[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        buffer = buffer == (BUFFERS - 1) * BUFFER ? 0 : buffer + BUFFER;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // (no load may land when this LDS is somebody else's)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + 16 * (MI * wave_m + i) + col;
        if (m >= M) continue;
        if (FORM == GATED) {
            const int n = n0 + 16 * wave_n + 4 * quad;             // (N is a multiple of 8 in every form)
            if (n >= N) continue;
            struct alignas(8) Four { bf16_t v[4]; } four;
#pragma unroll
            for (int r = 0; r < 4; ++r) four.v[r] = (bf16_t)(activation_of(activation, sums[i][0][r]) * sums[i][1][r]);
            *reinterpret_cast<Four*>((bf16_t*)out + (size_t)m * N + n) = four;
            continue;
        }
        const int n = n0 + 32 * wave_n + 8 * quad;
        if (n >= N) continue;
        if (FORM == SUMS) {
            float* to = (float*)out + ((size_t)blockIdx.y * M + m) * N + n;
            *reinterpret_cast<f32x4*>(to) = sums[i][0];
            *reinterpret_cast<f32x4*>(to + 4) = sums[i][1];
            continue;
        }
        bf16x8 eight;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const float z = sums[i][r >> 2][r & 3];
            eight[r] = (bf16_t)(FORM == ACTIVATED ? activation_of(activation, z) : z);
        }
        *reinterpret_cast<bf16x8*>((bf16_t*)out + (size_t)m * N + n) = eight;
    }
}

// The gated form on tiles of 256 x 256: 256 rows, 128 columns of the result.
//   The library's products of such sizes run at what power allows, as this one does; what it saves is the activation's launch and the way of the gate's and the up
// projection's columns through memory.  us with the activation, library and here: 2,048 rows, 12,288 x 4,096 316, 304; 8,192 x 4,096 210, 203; 4,096 rows 593, 576 and 400, 390.
// Without a gate there is half as much to save (2,048 rows, 8,192 x 4,096 103, 107): that stays the library's.
__global__ __launch_bounds__(WIDE_THREADS) void wide_gated_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, bf16_t* __restrict__ out, int M, int N, int K,
                                                                  int activation) {
    constexpr int COLUMNS = WIDE_TILE / 2;
    __shared__ __attribute__((aligned(1024))) unsigned char buffers[2 * WIDE_BUFFER];
    int tile_m, tile_n;
    if (!tile_of_workgroup((M + WIDE_TILE - 1) / WIDE_TILE, (N + COLUMNS - 1) / COLUMNS, tile_m, tile_n)) return;
    const int m0 = tile_m * WIDE_TILE, n0 = tile_n * COLUMNS;
    auto a_offset = [&](int r) __attribute__((always_inline)) { return m0 + r < M ? (unsigned)r * (unsigned)(2 * K) : NOWHERE; };
    auto b_offset = [&](int r) __attribute__((always_inline)) {    // gate rows, then their up rows
        const int c = r & (COLUMNS - 1);
        return n0 + c >= N ? NOWHERE : (unsigned)(c + (r >= COLUMNS ? N : 0)) * (unsigned)(2 * K);
    };
    WideSums sums;
    wide_product(sums, buffers, x + (size_t)m0 * K, a_offset, w + (size_t)n0 * K, b_offset, K, min(4, (M - m0 + 63) / 64), true);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = n0 + wide_column(0, wave, lane);
    if (n >= N) return;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + wide_row(half, i, wave, lane);
            if (m >= M) continue;
            bf16x8 eight;
#pragma unroll
            for (int r = 0; r < 8; ++r) eight[r] = (bf16_t)(activation_of(activation, sums[half][0][i][r >> 2][r & 3]) * sums[half][1][i][r >> 2][r & 3]);
            *reinterpret_cast<bf16x8*>(out + (size_t)m * N + n) = eight;
        }
}

// What lsa_product can be asked for: a tile, and for SUMS the parts of K, as 16 parts + tile.  ADDED in a plan for PLAIN or GATED: the sums, and a kernel behind
// them that adds the parts up (lsa_sum_parts, lsa_gated_parts).
enum Tile { NONE, SMALL, TALL, LARGE, WIDE };
struct TileShape { int rows, columns; double start, slab, alone, among, last, rate; };
// Columns of W; us of a launch, of a slab, and what a slab takes more for each compute unit in use (its share of all) where one workgroup alone reads its lines of W and where many read
// them, and for a last block of rows that is full (times its share squared); TB/s of W's way.  Fitted to 1,000 to 2,000 sizes each, within 4 to 6 %.
static const TileShape SHAPES[] = {{0, 0, 0, 0, 0, 0, 0, 0}, {64, 64, 3.94, 0.2, 0.12, 0.02, 0.04, 4.7}, {128, 64, 4.22, 0.25, 0.13, 0.06, 0.105, 4.7},
                                   {128, 128, 4.41, 0.375, 0.28, 0.08, 0.06, 4.5}, {256, 256, 0, 0, 0, 0, 0, 0}};
constexpr int UNITS = 256;                                         // compute units
// SMALL's tiles are 64 x 32 where that many still go round the compute units once.  A slab takes as long as its bytes do on the way from L2 into a compute unit, some 30 a cycle, next to what
// the weights' way takes: half the columns are a quarter less, and twice as many units pull the weights.  us, 64 x 64 and 64 x 32, the weights from memory: 33 rows of 3,840 x 2,560 activated
// 16.2, 11.2, gated 15.9, 11.8; 128 of 4,096 x 2,048 activated 13.6, 10.8; 190 of 1,024 x 3,072 gated 16.5, 12.8; 190 of 1,408 x 2,048 9.5, 9.2; 17 of 2,048 x 1,024 in four parts 3.7, 3.8.  119 sizes
// of 17 to 250 rows that the plan has them for are 1.20 times as fast.  Beyond one round they lose: 33 rows of 10,240 x 5,120 (320) 31.0, 35.3; 96 rows of 6,144 x 2,048 (384) 11.4, 16.2.
//   Both add up the same products in the same order, so that their results are the same bits.  Those of parts and of the library need not be, and the plan, which decides between them, goes on
// pricing 64 x 64: what it takes ends sooner than it says, and what goes another way keeps its bits.  By a price of 64 x 32 it would take more from both: gated 32 rows of 2,816 x 4,096 15.4 in
// parts, 14.3 so; 33 rows of 6,144 x 4,096 within a step 17.2 by the library, 15.6 (33 requests decoding, eight steps: 9,050 to 9,230, by the library 9,090 to 9,150).
static int small_columns(int form, int M, int N, int parts) {
    const int slim = form == GATED ? 16 : 32;
    return (long)((M + 63) / 64) * ((N + slim - 1) / slim) * parts <= UNITS ? slim : 2 * slim;
}
constexpr int MOST_PARTS = 8, ADDED = 1 << 12;

constexpr int FEW_ROWS = 128;
static bool fits(int form, long M, long N, long K) {
    return M >= 1 && N >= 8 && K >= SLAB && K % SLAB == 0 && N % 8 == 0 && (form == GATED ? 2 * N : 256) * K * 2 + K * 2 < (long)BUFFER_BYTES && 256 * K * 2 < (long)BUFFER_BYTES;
}

// The tile (and parts) for a product of these sizes, or 0 where the other way is expected to be as fast: the library's product, with the kernel of the activation behind
// it, or up to 128 rows the few-row kernels.  Both times are lines through what was measured, every tile beside the other way, at 70 numbers of rows from 17 to 4,096 of 73 products of this
// package's models: for the tiles a launch's start and a slab's time, for the library (whose own choice of tiles nobody can foretell: with its tiles' rounds in the line its
// times are met no better, within an eighth) a start, K and the operations.  So where the library has just begun a round, or has one of its slow sizes (many whole multiples of 64 rows: 256
// rows of 6,144 x 2,048 24.8, 17.4 here), its price is too low, and sizes that the tiles would make faster stay with it.  At 70 other numbers of rows 1,923 of 4,094 sizes are taken, up to
// 128 rows and beyond: gated 1.18 and 1.20 times as fast as the other way, plain 1.24 and 1.20, activated 1.25 and 1.23, sums with the norm behind them 1.13 and 1.16, heads 1.08 and none.
// Seventeen of them are slower than 0.97 of it: 95 rows of 2,560 x 4,096 0.93, 63 of 4,096 x 3,072 0.94, 320 to 448 of 64 x 2,048 0.95, 30 of 2,112 x 2,048 activated 0.97; sums at 531
// and 545 rows of 2,048 x 2,048 0.93 and 0.95, 232 of 2,560 x 9,728 0.94, 127 of 5,120 x 17,408 0.96, 35 of 4,096 x 8,192 and 255 of 4,096 x 12,288 0.97 (counted with tiles of 64 x 64
// everywhere, before any of 64 x 32 ran).  A product whose tiles
// do not go round the compute units in one round stays the
// library's unless it is gated and large.  Up to 128 rows the parts may be added up by a launch of their own (64 rows, 2,816 x 2,048 library 12.1, one launch 12.2, so 9.7; 32
// rows of 4,096 x 4,096 13.9, 17.9, 12.0; gated 2,816 x 4,096 15.4, 18.4, 12.2).
LSA_EXPORT int lsa_product_plan(int form, int M, int N, int K) {
    if (form < PLAIN || form > SUMS || !fits(form, M, N, K)) return NONE;
    // (sums beyond 128 rows were measured from 1,024 columns on: fewer go the library's way, whole or in ranges; and in parts of few slabs they are slower from 257 rows on: 384 and 512 rows
    // of 2,048 x 1,408 with the norm 15.8 and 17.1, the library 14.8 and 15.3; and beyond 1,100 rows: 1,121, 1,223 and 1,338 of 1,024 x 2,048 19.3, 19.6 and 21.2, the library 19.1, 19.6 and
    // 19.2, 1,330 and 1,980 of 1,024 x 3,072 25.1 and 27.9, 24.0 and 28.3)
    if (form == SUMS && M > FEW_ROWS && (N < 1024 || M > 1100 || (M > 2 * FEW_ROWS && K < 2048))) return NONE;
    const double slabs = K / SLAB, weights = (form == GATED ? 2.0 : 1.0) * N, megabytes = weights * K * 2e-6, gigaflops = 2e-9 * M * weights * K;
    double best = 1e30;
    int plan = NONE;
    for (int tile = SMALL; tile <= LARGE; ++tile) {
        const TileShape& shape = SHAPES[tile];
        const int columns = form == GATED ? shape.columns / 2 : shape.columns;
        const long tiles = (long)((M + shape.rows - 1) / shape.rows) * ((N + columns - 1) / columns);
        const bool added = (form == PLAIN || form == GATED) && M <= FEW_ROWS;
        for (int parts = 1; parts <= (form == SUMS || added ? MOST_PARTS : 1); parts *= 2) {
            // (the sums take the tile's 64 or 128 rows of W whatever they are: gated, half as many tiles)
            // (two of the small tiles' workgroups fit a compute unit: where the weights' way bounds them, 33 rows of 32,768 x 4,096 63 us for the library, 55; gated products
            // beyond one round, and with less than 1,024 of K, stay with the kernel that shares the activations, or the library)
            if (tiles * parts > (tile == SMALL && parts == 1 && form != GATED ? 2 : 1) * UNITS || slabs < 4 * parts || (form == GATED && slabs < 16)) continue;
            // (rows behind the last one repeat it and cost no way of their own: tiles of 128 x 64, us for 2,048 x 2,048 at 257, 320 and 384 rows 13.9, 14.4 and 16.7; 513 and 512 rows 14.2
            // and 16.8, where tiles of 64 x 64 take 12.0 for 512, one a compute unit)
            const double load = tiles * parts < UNITS ? (double)(tiles * parts) / UNITS : 1.0, blocks = (M + shape.rows - 1) / shape.rows, last = (double)((M - 1) % shape.rows + 1) / shape.rows;
            const double slab = shape.slab + load * (shape.among + (shape.alone - shape.among) / blocks) + shape.last * last * last;
            double us = shape.start + slab * ((K / SLAB + parts - 1) / parts) * (tiles * parts > UNITS ? 1.9 : 1.0);
            // (the weights come as fast as many workgroups pull: with 160 of them 33 rows of 5,120 x 25,600 took 71 us, with 320 67)
            const double way = megabytes / (shape.rate * (0.5 + 0.5 * load)) + 3.0;
            us = us > way ? us : way;
            if (form == SUMS) us += parts * 1.7e-6 * M * N;        // written and read
            else if (parts > 1) us += 2.2 + parts * 2.0e-6 * M * weights;      // and a launch
            if (us < best) {
                best = us;
                plan = 16 * parts + tile + (form != SUMS && parts > 1 ? ADDED : 0);
            }
        }
    }
    double library = 9.9 + 0.0016 * K + (gigaflops < 40 ? 0.77 * gigaflops : 30.8 + 0.69 * (gigaflops - 40));
    // (it cuts K where few rows meet few columns: from 129 rows on, us at 156 and 191 rows of 2,048 x 4,096 16.1 and 16.4, in whole tiles here 17.7 and 19.8)
    if (form != GATED && M > FEW_ROWS && K >= 4096 && (double)M * N < 4.5e5 && library > 3.7 + 0.0033 * K + 0.77 * gigaflops) library = 3.7 + 0.0033 * K + 0.77 * gigaflops;
    if (M <= 64 && N <= 2048 && form != GATED) library = 4.0 + 0.0022 * K;        // (it cuts K there)
    library = library > megabytes / 4.5 ? library : megabytes / 4.5;
    if (form == GATED) library += 3.5 + 6e-6 * M * N / 5.0;
    if (form == ACTIVATED) library += 3.5 + 4e-6 * M * N / 5.0;
    if (form == GATED && slabs >= 16) {
        const long tiles = (long)((M + WIDE_TILE - 1) / WIDE_TILE) * ((N + WIDE_TILE / 2 - 1) / (WIDE_TILE / 2)), last = tiles % UNITS;
        // A launch takes 13 us around the slabs of its last round and 6 around those of a full one (1,024 rows of 3,072 x 1,024, 16 slabs on 96 compute units, 33 us, 26.6 for the
        // library's product and the activation), a slab 1.0 us where few compute units work, 1.5 where all do: power.  A tile of 64 rows and fewer leaves three tenths of that out,
        // and there the weights' way is what counts (17 rows, 25,600 x 5,120 on 200 compute units 101 us, 17,408 x 5,120 on 136 84).
        const double load = (double)last / UNITS, blocks = M > 192 ? 4 : (M + 63) / 64, pulled = tiles < UNITS ? load : 1.0;
        const double products = 7.0 + tiles / UNITS * (6.0 + 1.5 * slabs) + (last ? 6.0 + (1.0 + 0.5 * load) * (0.6 + 0.1 * blocks) * slabs : 0.0);
        const double way = megabytes / (5.4 * (0.5 + 0.5 * pulled)) + 3.0, us = products > way ? products : way;
        if (us < best && us < 0.99 * library) return 16 + WIDE;
    }
    // Up to 128 rows the other way for sums is the kernel that shares the rows in LDS (lsa_gemm_split): slower for weights of up to 50 MB throughout (33 rows, with the norm,
    // 2,048 x 6,144 13.7, 12.3; 4,096 x 4,096 15.3, 14.1; 100 rows 18.8, 15.2 and 21.3, 17.9); beyond that its time, again with the norm, is a line in the weights and the rows, and
    // where tiles leave compute units idle it is the faster one: 48 rows of 5,120 x 25,600 62.8, 79.0, of 5,120 x 17,408 49.6, 52.5, 29 rows of 5,120 x 5,120 20.6, 24.5, of
    // 4,096 x 8,192 21.5, 23.3; 128 rows of 4,096 x 12,288 41.4, 35.6.
    if (form == SUMS && M <= FEW_ROWS)
        return weights * K <= 2.6e7 || best + 4.0 < 0.93 * (7.1 + megabytes / 4.9 + 0.05 * M + 0.00066 * M * megabytes) ? plan : NONE;
    // (a weight of more than 50 MB in parts: the library cuts K up to 32 rows and not beyond: 18, 28, 34 and 44 rows of 4,096 x 8,192 17.6, 18.6, 22.9 and 23.0, here 19.9, 20.1, 20.2
    // and 20.6; 2,048 x 8,448, at 18 rows 27.2, here 11.5, and 4,096 x 4,096, 13.3 and 11.1, lie before that)
    if (form == PLAIN && (plan & ADDED) && M <= 32 && weights * K > 2.6e7) return NONE;
    // How far the lines are trusted: up to 128 rows the library takes longer than its line nearly everywhere, and a gated product's (with the activation) at any number of rows.
    static const double MARGINS[4][2] = {{1.22, 0.95}, {1.1, 1.1}, {0.87, 0.92}, {0, 0.94}};
    return best < (plan & ADDED ? 0.92 : MARGINS[form][M > FEW_ROWS]) * library ? plan : NONE;
}

template <int FORM>
static int launch(int tile, int parts, const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int activation, hipStream_t stream) {
    const int columns = tile == SMALL ? small_columns(FORM, M, N, parts) : FORM == GATED ? SHAPES[tile].columns / 2 : SHAPES[tile].columns;
    const int blocks = workgroups(M, N, SHAPES[tile].rows, columns);
    if (blocks < 0) return -1;
    const dim3 grid(blocks, parts);
    if (tile == SMALL && columns == (FORM == GATED ? 16 : 32)) product_kernel<4, 1, 1, 10, FORM><<<grid, 256, 0, stream>>>(x, w, out, M, N, K, activation);
    else if (tile == SMALL) product_kernel<2, 2, 2, 5, FORM><<<grid, 256, 0, stream>>>(x, w, out, M, N, K, activation);
    else if (tile == TALL) product_kernel<4, 2, 2, 6, FORM><<<grid, 512, 0, stream>>>(x, w, out, M, N, K, activation);
    else product_kernel<2, 4, 4, 4, FORM><<<grid, 512, 0, stream>>>(x, w, out, M, N, K, activation);
    LSA_LAUNCH_CHECK();
}

// plan: what lsa_product_plan gave, or any other tile (1 to 4; with 16 parts, 1 to 8, for SUMS).  x, w and out begin at multiples of 16 bytes.
LSA_EXPORT int lsa_product(int plan, int form, int activation, const void* x, const void* w, void* out, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const int tile = plan % 16, parts = plan / 16;
    if (form < PLAIN || form > SUMS || !fits(form, M, N, K) || tile < SMALL || tile > WIDE || parts < 1 || parts > MOST_PARTS || parts > K / SLAB
        || (parts > 1 && form != SUMS) || activation < SILU || activation > (form == GATED ? GELU_TANH : RELU2) || (((size_t)x | (size_t)w | (size_t)out) & 15)) return -1;
    const bf16_t *xb = (const bf16_t*)x, *wb = (const bf16_t*)w;
    if (tile != WIDE) {
        if (form == PLAIN) return launch<PLAIN>(tile, parts, xb, wb, out, M, N, K, activation, stream);
        if (form == GATED) return launch<GATED>(tile, parts, xb, wb, out, M, N, K, activation, stream);
        if (form == ACTIVATED) return launch<ACTIVATED>(tile, parts, xb, wb, out, M, N, K, activation, stream);
        return launch<SUMS>(tile, parts, xb, wb, out, M, N, K, activation, stream);
    }
    const int blocks = workgroups(M, N, WIDE_TILE, WIDE_TILE / 2);
    if (blocks < 0 || form != GATED) return -1;
    wide_gated_kernel<<<blocks, WIDE_THREADS, 0, stream>>>(xb, wb, (bf16_t*)out, M, N, K, activation);
    LSA_LAUNCH_CHECK();
}
