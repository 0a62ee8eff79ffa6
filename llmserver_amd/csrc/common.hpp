// Shared helpers of the gfx950 kernels: element types, conversions, wavefront reductions.
// Wavefronts are 64 lanes wide; every reduction below is written for that width.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lsa {

typedef __bf16 bf16_t;

template <typename T> struct Elem;
template <> struct Elem<float> {
    static constexpr int kVec = 4;                       // elements per 16-byte vector
    __device__ static inline float load(const float* p) { return *p; }
    __device__ static inline void store(float* p, float v) { *p = v; }
    __device__ static inline float round(float v) { return v; }
};
template <> struct Elem<bf16_t> {
    static constexpr int kVec = 8;
    __device__ static inline float load(const bf16_t* p) { return (float)(*p); }
    __device__ static inline void store(bf16_t* p, float v) { *p = (bf16_t)v; }
    __device__ static inline float round(float v) { return (float)((bf16_t)v); }
};

// A 16-byte vector of T, loaded and stored as one transaction.
template <typename T> struct alignas(16) Vec16 {
    T v[Elem<T>::kVec];
};

template <typename T>
__device__ inline Vec16<T> load_vec16(const T* p) {
    return *reinterpret_cast<const Vec16<T>*>(p);
}
template <typename T>
__device__ inline void store_vec16(T* p, const Vec16<T>& x) {
    *reinterpret_cast<Vec16<T>*>(p) = x;
}

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, 64);
    return v;
}
__device__ inline float wave_max(float v) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, 64));
    return v;
}

// Sum over a block of up to 1024 threads; every thread gets the result. `scratch` holds 16 floats.
__device__ inline float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = (blockDim.x + 63) >> 6;
    v = wave_sum(v);
    __syncthreads();                      // scratch may still be read from an earlier call
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < waves; ++w) total += scratch[w];   // same order in every thread
    return total;
}

// Puts 64 consecutive tokens of one KV head, staged in LDS as [VT_TOKENS][pitch] with `filled` numbers a token, into their
// pages values[page][kv_head][0 .. dims)[slot] (of d dimensions), zeros for the dimensions from `filled` to `dims`.  Four slots of one dimension go out at
// a time (8 or 16 bytes) wherever four tokens are neighbours in one page from a slot that is a multiple of four on, which is the rule inside a portion; a page's
// [d][page_size] block is contiguous, so these stores coalesce.  At least 64 threads; whoever wrote the tile need not have waited.
// Every token's place is found once, by a thread of its own, and only then are the tokens sorted into fours and singles: a tile in which portions meet
// has up to sixty singles, and looking each of their numbers' places up (row, position, table: three trips to memory behind one another) took the
// whole launch 24 us for 512 tokens of three float32 portions instead of 9.5 (one portion 11.3 and 9.1; bfloat16, 2,048 tokens 16.9 and 14.4).
constexpr int VT_TOKENS = 64;
template <typename T>
__device__ __forceinline__ void store_value_tile(const T* tile, int pitch, int token0, int kv_head, int filled, T* __restrict__ values,
                                                 const int* __restrict__ table, int table_stride, const int* __restrict__ token_row,
                                                 const int* __restrict__ positions, int page_size, int n_kv, int d, int n_tokens, int dims) {
    __shared__ long place_of[VT_TOKENS];                   // element offset of the token's slot in `values`, or -1
    __shared__ unsigned char fours[VT_TOKENS / 4], singles[VT_TOKENS];       // first tokens of fours; tokens that go alone
    __shared__ int n_fours, n_singles;
    if (threadIdx.x < VT_TOKENS) {                         // (the first wavefront)
        const int t = threadIdx.x, token = token0 + t;
        long place = -1;
        if (token < n_tokens) {
            const int pos = positions[token], block = pos / page_size;
            const int p = table[(size_t)token_row[token] * table_stride + block];
            if (p >= 0) place = (((long)p * n_kv + kv_head) * d) * page_size + (pos - block * page_size);
        }
        place_of[t] = place;                               // (read behind the barrier)
        // The token behind this one lies behind it in its page: told from lane to lane, not through LDS, where nothing would order another lane's
        // write in front of the read.  (A slot's number modulo four is its offset's: pages are a multiple of four slots.)
        const unsigned long long next_behind = __ballot(__shfl_down((long long)place, 1) == place + 1 && t + 1 < VT_TOKENS);
        const bool first = place >= 0 && (place & 3) == 0 && (next_behind >> t & 7) == 7;
        const unsigned long long firsts = __ballot(first), together = firsts | firsts << 1 | firsts << 2 | firsts << 3;
        const unsigned long long alone = __ballot(place >= 0) & ~together, below = (1ull << t) - 1;
        if (first) fours[__popcll(firsts & below)] = (unsigned char)t;
        if (alone >> t & 1) singles[__popcll(alone & below)] = (unsigned char)t;
        if (t == 0) {
            n_fours = __popcll(firsts);
            n_singles = __popcll(alone);
        }
    }
    __syncthreads();
    const int groups = n_fours, rest = n_singles;
    for (int e = threadIdx.x; e < (VT_TOKENS / 4) * dims; e += blockDim.x) {
        const int g = e & (VT_TOKENS / 4 - 1), i = e / (VT_TOKENS / 4);      // neighbouring threads: neighbouring groups of slots
        if (g >= groups) continue;
        const int first = fours[g];
        T four[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) four[r] = i < filled ? tile[(first + r) * pitch + i] : (T)0.f;
        T* dst = values + place_of[first] + (size_t)i * page_size;
        if (sizeof(T) == 2) *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(four);
        else *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(four);
    }
    for (int e = threadIdx.x; e < rest * dims; e += blockDim.x) {        // (a handful where portions meet, all of them where a page's slots are in no order)
        const int g = e / dims, i = e - g * dims, t = singles[g];
        values[place_of[t] + (long)i * page_size] = i < filled ? tile[t * pitch + i] : (T)0.f;
    }
}

}  // namespace lsa

#define LSA_EXPORT extern "C" __attribute__((visibility("default")))
#define LSA_LAUNCH_CHECK() return (int)hipGetLastError()
