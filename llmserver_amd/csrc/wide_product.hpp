// A tile of C = A . B^T: 256 rows of A against 256 rows of B (K contiguous in both, bfloat16, 32-bit sums), by eight wavefronts that take turns at
// the matrix cores.
#pragma once
#include "common.hpp"
#include "lds_loads.hpp"

namespace lsa {

// load_16_bytes_a_lane_to_lds through a buffer descriptor of `base`: a byte offset per lane and one for all of them, so that a walk along rows costs no vector additions.  Their
// sum stays below BUFFER_BYTES; a lane whose own offset is NOWHERE or up to 127 beside it reads nothing from memory, and zeros land.
constexpr unsigned BUFFER_BYTES = 0xFFFFFE00u, NOWHERE = 0xFFFFFF00u;
typedef int buffer_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ buffer_t buffer_at(const void* base) {
    const unsigned long long address = (unsigned long long)base;
    buffer_t made;
    made[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)address);
    made[1] = __builtin_amdgcn_readfirstlane((int)(unsigned)(address >> 32)) & 0xFFFF;
    made[2] = (int)BUFFER_BYTES;
    made[3] = 0x00027000;                                         // 32-bit data, no swizzle
    return made;
}
__device__ __forceinline__ void load_16_bytes_a_lane_to_lds(buffer_t buffer, unsigned offset, unsigned common_offset, unsigned lds_address) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(offset), "s"(buffer), "s"(common_offset), "s"(lds_address) : "memory", "m0");
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int WIDE_TILE = 256, WIDE_SLAB = 64, WIDE_THREADS = 512;
constexpr int WIDE_BUFFER = 2 * WIDE_TILE * WIDE_SLAB * 2;            // bytes: a slab of 64 columns of both operands
constexpr int WIDE_HALF = WIDE_TILE / 2 * WIDE_SLAB * 2;              // bytes: half the rows of one of them

// Where in a wavefront's sums a number stands: sums[a][b][i][j][r] is row wide_row(a, i, wave, lane), column wide_column(b, wave, lane) + 4 j + r, so that
// a lane has eight neighbouring columns of a row.
typedef f32x4 WideSums[2][2][4][2];
__device__ __forceinline__ int wide_row(int a, int i, int wave, int lane) { return WIDE_TILE / 2 * a + 32 * i + 16 * (wave >> 2) + (lane & 15); }
__device__ __forceinline__ int wide_column(int b, int wave, int lane) { return WIDE_TILE / 2 * b + 32 * (wave & 3) + 8 * (lane >> 4); }

// Barriers of the workgroup: behind this wavefront's reads of LDS, and behind all but its newest PENDING loads too.
__device__ __forceinline__ void wide_barrier() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ void wide_barrier_behind_reads() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int N> struct WideLeft { static constexpr int value = N; };

// a_offset(r), b_offset(r): bytes from `a` (`b`) to the first number of the tile's row r, 0 <= r < 256, or NOWHERE for a row whose sums nobody wants.
// k: a multiple of 32.  row_blocks: how many of the four blocks of 64 rows of A are wanted (1 to 4), second_half: whether columns from 128 on are;
// sums of others are left undefined.  `buffers`: 2 * WIDE_BUFFER bytes at a multiple of 1,024.  All 512 threads come here; nothing is under way afterwards.
//
//   What bounds it is power: by counters a tile takes 2,290 cycles a slab, of which the matrix cores are busy 2,048, and 32,000 around its slabs, with half the compute units
// as with all of them; but the clock is 2.5 GHz with half, 2.0 with all and falls on in launches one behind the other (256 tiles of 128 slabs: 185 and 206 us, 128 tiles 140).  So
// what counts beside full matrix cores is what else takes energy: products of 16 x 16 x 32 and not of 32 x 32 x 16 (1.49 against 1.33 PFLOP/s: the
// clock falls to 1.52 GHz), and products of padding are left out.
//   A slab is four regions, the halves of A and of B (128 rows of 128 bytes, 16 KB), and four phases, of which each multiplies one half of A with
// one half of B, reads one region's operands from LDS for the phases behind it, and asks for one region of the slab after the next:
//     phase      reads                 multiplies        asks for (two slabs on)
//       0        A0                    A0 B0             B0
//       1        B1                    A0 B1             A0
//       2        A1                    A1 B1             B1
//       3        B0 of the next slab   A1 B0             A1
// Seven phases lie between a load and its use, and every phase waits for the loads of six phases ago, whatever its number.
//   The two wavefronts of a SIMD are half a phase apart (the second four go through one barrier more at the start, the first four at the end): between
// two barriers one of them reads and asks while the other one multiplies.  Without that, 3,090 cycles a slab.
//   A region's eight 16-byte pieces of row r stand at places piece ^ f(r), so that the sixteen lanes whose 16-byte reads are served together meet all 64 banks.  A lane
// that holds column c of an MFMA reads row 8 (c / 4) + c % 4 (+ 4) of B, so that two MFMAs give it eight neighbouring columns of the result.
// WHOLE: all rows and columns are wanted; their products go without a branch between them (32,760 pairs of 64 experts, all launches: 730 -> 710 us).
template <bool WHOLE, typename AOffset, typename BOffset>
__device__ __forceinline__ void wide_product_of(WideSums& sums, unsigned char* buffers, const void* a, AOffset a_offset, const void* b, BOffset b_offset, int k,
                                             int row_blocks, bool second_half) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), col = lane & 15, quad = lane >> 4;
    const unsigned lds_begin = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(lds_ptr_t)buffers);
    const int slabs = (k + WIDE_SLAB - 1) / WIDE_SLAB;
    const bool half_slab = k % WIDE_SLAB != 0;                        // then the last slab is half a slab: what lies behind the rows' end is not read
    // A load of a wavefront is 8 rows of a region; wavefront w has rows 8 w and 64 + 8 w on of every region.
    const buffer_t a_buffer = buffer_at(a), b_buffer = buffer_at(b);
    unsigned a_at[2][2], b_at[2][2];
    const int place = lane & 7, line = 8 * wave + (lane >> 3);
    const int a_piece = place ^ (line >> 1 & 7), b_piece = place ^ ((line >> 1 & 1) | (line >> 3 & 3) << 1);     // (64 rows on: the same)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            a_at[half][u] = a_offset(128 * half + 64 * u + line) + 16 * a_piece;
            b_at[half][u] = b_offset(128 * half + 64 * u + line) + 16 * b_piece;
        }
    auto last_slab_is_next = [&]() __attribute__((always_inline)) {
        if (!half_slab) return;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                a_at[half][u] -= a_piece >= 4 ? 64 : 0;
                b_at[half][u] -= b_piece >= 4 ? 64 : 0;
            }
    };
    const unsigned landing = lds_begin + 1024 * wave;
    auto ask_a = [&](int half, int slab, int buffer) __attribute__((always_inline)) {
        const unsigned to = landing + buffer + half * WIDE_HALF, from = slab * (2 * WIDE_SLAB);
        load_16_bytes_a_lane_to_lds(a_buffer, a_at[half][0], from, to);
        load_16_bytes_a_lane_to_lds(a_buffer, a_at[half][1], from, to + WIDE_HALF / 2);
    };
    auto ask_b = [&](int half, int slab, int buffer) __attribute__((always_inline)) {
        const unsigned to = landing + buffer + (2 + half) * WIDE_HALF, from = slab * (2 * WIDE_SLAB);
        load_16_bytes_a_lane_to_lds(b_buffer, b_at[half][0], from, to);
        load_16_bytes_a_lane_to_lds(b_buffer, b_at[half][1], from, to + WIDE_HALF / 2);
    };
    struct AOperands { bf16x8 v[4][2]; };
    struct BOperands { bf16x8 v[2][2]; };
    AOperands xa;
    BOperands xb[3];                                                  // B1, and B0 of this slab and of the next
    const int pieces[2] = {16 * (quad ^ (col >> 1)), 16 * ((quad + 4) ^ (col >> 1))};
    const unsigned char* a_rows = buffers + (16 * (wave >> 2) + col) * 128;
    const unsigned char* b_rows = buffers + 2 * WIDE_HALF + (32 * (wave & 3) + 8 * (col >> 2) + (col & 3)) * 128;
    const int blocks[2] = {min(row_blocks, 2), max(row_blocks - 2, 0)};
    auto read_a = [&](int half, int buffer) __attribute__((always_inline)) {
        const unsigned char* rows = a_rows + buffer + half * WIDE_HALF;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (WHOLE || i < 2 * blocks[half])
#pragma unroll
                for (int s = 0; s < 2; ++s) xa.v[i][s] = *reinterpret_cast<const bf16x8*>(rows + 4096 * i + pieces[s]);
    };
    auto read_b = [&](BOperands& x, int half, int buffer) __attribute__((always_inline)) {
        const unsigned char* rows = b_rows + buffer + half * WIDE_HALF;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int s = 0; s < 2; ++s) x.v[j][s] = *reinterpret_cast<const bf16x8*>(rows + 512 * j + pieces[s]);
    };
    // (a block of 64 rows is two rows of MFMA tiles of each of the two rows of wavefronts)
    auto multiply = [&](int half_a, int half_b, const BOperands& x, bool second_piece) __attribute__((always_inline)) {
        auto some = [&](int s, int first, int last) __attribute__((always_inline)) {
#pragma unroll
            for (int i = first; i < last; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    sums[half_a][half_b][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v[j][s], xa.v[i][s], sums[half_a][half_b][i][j], 0, 0, 0);
        };
        __builtin_amdgcn_sched_barrier(0);
        if (WHOLE) {
            some(0, 0, 4);
            if (second_piece) some(1, 0, 4);
        } else if (half_b == 0 || second_half) {
#pragma unroll
            for (int block = 0; block < 2; ++block)
                if (block < blocks[half_a]) {
                    some(0, 2 * block, 2 * block + 2);
                    if (second_piece) some(1, 2 * block, 2 * block + 2);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // LEFT: slabs behind this one (2: two or more), of which `asked` is the one to ask for.  `buffer` is this slab's, and that one's.
    auto step = [&](int buffer, int asked, auto left, bool whole, BOperands& now, BOperands& next) __attribute__((always_inline)) {
        constexpr int LEFT = decltype(left)::value;
        read_a(0, buffer);
        __builtin_amdgcn_sched_barrier(0);
        if (LEFT == 2) ask_b(0, asked, buffer);
        loads_landed_then_barrier<LEFT == 2 ? 12 : LEFT == 1 ? 10 : 2>();
        multiply(0, 0, now, whole);
        wide_barrier();
        if (WHOLE || second_half) read_b(xb[2], 1, buffer);
        __builtin_amdgcn_sched_barrier(0);
        if (LEFT == 2) ask_a(0, asked, buffer);
        loads_landed_then_barrier<LEFT == 2 ? 12 : LEFT == 1 ? 8 : 0>();
        multiply(0, 1, xb[2], whole);
        wide_barrier();
        read_a(1, buffer);
        __builtin_amdgcn_sched_barrier(0);
        if (LEFT == 2) ask_b(1, asked, buffer);
        loads_landed_then_barrier<LEFT == 2 ? 12 : LEFT == 1 ? 6 : 0>();
        multiply(1, 1, xb[2], whole);
        wide_barrier();
        if (LEFT > 0) read_b(next, 0, buffer ^ WIDE_BUFFER);
        __builtin_amdgcn_sched_barrier(0);
        if (LEFT == 2) ask_a(1, asked, buffer);
        loads_landed_then_barrier<LEFT == 2 ? 12 : LEFT == 1 ? 4 : 0>();
        multiply(1, 0, now, whole);
        wide_barrier();
    };
#pragma unroll
    for (int e = 0; e < 32; ++e) sums[e >> 4][e >> 3 & 1][e >> 1 & 3][e & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // (the counts below start from nothing under way)
    if (slabs == 1) last_slab_is_next();
    ask_b(0, 0, 0); ask_a(0, 0, 0); ask_b(1, 0, 0); ask_a(1, 0, 0);
    if (slabs == 2) last_slab_is_next();
    const int second = min(1, slabs - 1);                             // (a single slab once more)
    ask_b(0, second, WIDE_BUFFER); ask_a(0, second, WIDE_BUFFER); ask_b(1, second, WIDE_BUFFER); ask_a(1, second, WIDE_BUFFER);
    loads_landed_then_barrier<12>();
    read_b(xb[0], 0, 0);
    wide_barrier_behind_reads();
    if (wave >= 4) wide_barrier();
    int slab = 0, buffer = 0;
    for (; slab + 3 < slabs; slab += 2) {
        step(0, slab + 2, WideLeft<2>{}, true, xb[0], xb[1]);
        if (slab + 4 == slabs) last_slab_is_next();
        step(WIDE_BUFFER, slab + 3, WideLeft<2>{}, true, xb[1], xb[0]);
    }
    if (slab + 2 < slabs) {
        last_slab_is_next();
        step(0, slab + 2, WideLeft<2>{}, true, xb[0], xb[1]);
        buffer = WIDE_BUFFER;
        xb[0] = xb[1];
    }
    if (slabs > 1) {
        step(buffer, 0, WideLeft<1>{}, true, xb[0], xb[1]);
        buffer ^= WIDE_BUFFER;
        xb[0] = xb[1];
    }
    step(buffer, 0, WideLeft<0>{}, !half_slab, xb[0], xb[1]);
    if (wave < 4) wide_barrier();
}

template <typename AOffset, typename BOffset>
__device__ __forceinline__ void wide_product(WideSums& sums, unsigned char* buffers, const void* a, AOffset a_offset, const void* b, BOffset b_offset, int k,
                                             int row_blocks, bool second_half) {
    if (row_blocks == 4 && second_half) wide_product_of<true>(sums, buffers, a, a_offset, b, b_offset, k, row_blocks, second_half);
    else wide_product_of<false>(sums, buffers, a, a_offset, b, b_offset, k, row_blocks, second_half);
}

}  // namespace lsa
