// What the chunked forms of the recurrences share: a row's tokens of a step in chunks of 64, counted from the row's first token, an
// item being a (row, chunk); and 32-bit matrix products of operands in LDS.
#pragma once
#include "common.hpp"

namespace lsa {

constexpr int MC = 64;                   // tokens a chunk
constexpr int MC_A = 68;                 // row length in LDS of an operand read down its rows (a lane a row)
constexpr int MC_B = 80;                 // ... of an operand read along its rows (a lane a column)

// Item number `item` of a step's rows; false behind the last one (a grid has as many as the step could have at most).
__device__ __forceinline__ bool chunk_item(int item, int rows, const int* __restrict__ row_len, int& row, int& chunk) {
    int base = 0;
    for (int r = 0; r < rows; ++r) {
        const int count = row_len[r];
        const int chunks = count > 0 ? (count + MC - 1) / MC : 0;
        if (item < base + chunks) { row = r; chunk = item - base; return true; }
        base += chunks;
    }
    return false;
}

constexpr int BC = 16;                   // tokens a block, where chunks are cut further

typedef float mc_f4 __attribute__((ext_vector_type(4)));
typedef double mc_d4 __attribute__((ext_vector_type(4)));

// What the four partial sums of a product make together, rounded once.
__device__ __forceinline__ mc_f4 together(const mc_f4 (&part)[4]) {
    mc_f4 sum;
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[e] = (float)(((double)part[0][e] + (double)part[1][e]) + ((double)part[2][e] + (double)part[3][e]));
    return sum;
}

// acc[ni] += A B for 16 rows and NN times 16 columns over inner indices [0, inner), a multiple of 16; A's (m, i) at a[m * a_row + i * a_inner],
// B's (i, n) at b[i * b_inner + n * b_column].  Every fourth product goes to the same partial sum: four short chains round less than
// one long one.
template <int NN>
__device__ __forceinline__ void channel_product(mc_f4 (&acc)[NN], const float* a, int a_row, int a_inner, const float* b, int b_inner, int b_column,
                                                int inner, int lane) {
    const int r = lane & 15, g = lane >> 4;
    a += r * a_row + g * a_inner;
    b += g * b_inner + r * b_column;
    mc_f4 part[NN][4] = {};
    for (int i = 0; i < inner; i += 16) {
        float x[4], y[NN][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = a[(i + 4 * u) * a_inner];
#pragma unroll
            for (int ni = 0; ni < NN; ++ni) y[ni][u] = b[(i + 4 * u) * b_inner + 16 * ni * b_column];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int ni = 0; ni < NN; ++ni) part[ni][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], y[ni][u], part[ni][u], 0, 0, 0);
    }
#pragma unroll
    for (int ni = 0; ni < NN; ++ni) acc[ni] += together(part[ni]);
}

}  // namespace lsa
