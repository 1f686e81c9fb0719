// Softmax attention in plain FP32 arithmetic: what a matrix kernel goes back to for a workgroup's rows where its products have met
// numbers that they cannot carry (infinities and NaNs, which zero weights do not silence, scores far outside the range of its
// reference maxima).  Only what a row sees enters its maximum, its sum and its output, each number once and as it is.
#pragma once

#include <hip/hip_runtime.h>

namespace sd {

// A key or value row on a 16-byte boundary: FP32, or BF16; null: there is none.
struct PlainRow {
    const void* at;
    bool bf16;
    __device__ __forceinline__ float4 four(int c) const {
        if (!bf16) return *reinterpret_cast<const float4*>(static_cast<const float*>(at) + c);
        const uint2 x = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(at) + c);
        return float4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u)};
    }
    __device__ __forceinline__ float operator[](int c) const {
        return bf16 ? __uint_as_float(uint32_t(static_cast<const uint16_t*>(at)[c]) << 16) : static_cast<const float*>(at)[c];
    }
};

constexpr int PLAIN_TILE = 32;                    // keys at a time
constexpr size_t plain_attention_bytes(int rows, int dim) { return size_t(rows) * (dim + PLAIN_TILE + 3) * 4; }

// ROWS query rows over the keys begin .. end - 1, by a whole workgroup; lds: plain_attention_bytes.  query(row, column); key(index) and
// value(index) are rows, asked for only where sees(row, index); done(row, column, unnormalised output, maximum, sum).
template<int ROWS, int DIM, int THREADS, class Query, class Key, class Value, class Sees, class Done>
__device__ void plain_attention(uint8_t* lds, unsigned begin, unsigned end, float scale, Query query, Key key, Value value, Sees sees, Done done) {
    constexpr int PARTS = THREADS > DIM ? THREADS / DIM : 1, MINE = ROWS / PARTS, COLUMNS = THREADS > DIM ? 1 : DIM / THREADS;     // a thread's rows and columns
    const int t = threadIdx.x, row0 = t / (THREADS / PARTS) * MINE, column0 = t % (THREADS / PARTS);
    float* const queries = reinterpret_cast<float*>(lds);       // [ROWS][DIM]
    float* const weights = queries + ROWS * DIM;                // [ROWS][TILE]
    float* const top = weights + ROWS * PLAIN_TILE;             // [ROWS] each
    float* const total = top + ROWS;
    float* const keep = total + ROWS;
    __syncthreads();
    for (int i = t; i < ROWS * DIM; i += THREADS) queries[i] = query(i / DIM, i % DIM);
    if (t < ROWS) { top[t] = -INFINITY; total[t] = 0.0f; }
    float acc[COLUMNS][MINE];
    #pragma unroll
    for (int c = 0; c < COLUMNS; ++c)
        #pragma unroll
        for (int r = 0; r < MINE; ++r) acc[c][r] = 0.0f;
    for (unsigned first = begin; first < end; first += PLAIN_TILE) {
        const unsigned count = min(end - first, unsigned(PLAIN_TILE));
        __syncthreads();
        for (int i = t; i < ROWS * PLAIN_TILE; i += THREADS) {
            const int row = i / PLAIN_TILE;
            const unsigned index = first + i % PLAIN_TILE;
            float score = -INFINITY;
            if (index < end && sees(row, index)) {
                const PlainRow k = key(index);
                float dot = 0.0f;
                if (k.at) {
                    const float* const q = queries + row * DIM;
                    #pragma unroll 1
                    for (int c = 0; c < DIM; c += 4) {
                        const float4 x = k.four(c);
                        dot = fmaf(q[c], x.x, dot); dot = fmaf(q[c + 1], x.y, dot); dot = fmaf(q[c + 2], x.z, dot); dot = fmaf(q[c + 3], x.w, dot);
                    }
                    score = dot * scale;
                }
            }
            weights[i] = score;
        }
        __syncthreads();
        if (t < ROWS) {
            float* const mine = weights + t * PLAIN_TILE;
            const float before = top[t];
            float now = before, sum = 0.0f;
            for (int i = 0; i < PLAIN_TILE; ++i) now = fmaxf(now, mine[i]);
            for (int i = 0; i < PLAIN_TILE; ++i) {
                mine[i] = mine[i] == -INFINITY ? 0.0f : expf(mine[i] - now);
                sum += mine[i];
            }
            keep[t] = before == -INFINITY ? 0.0f : expf(before - now);
            top[t] = now;
            total[t] = fmaf(total[t], keep[t], sum);
        }
        __syncthreads();
        #pragma unroll
        for (int c = 0; c < COLUMNS; ++c)
            #pragma unroll
            for (int r = 0; r < MINE; ++r) acc[c][r] *= keep[row0 + r];
        #pragma unroll 1
        for (unsigned i = 0; i < count; ++i) {
            const PlainRow v = value(first + i);
            if (!v.at) continue;
            #pragma unroll
            for (int c = 0; c < COLUMNS; ++c) {
                const float x = v[column0 + c * THREADS];
                #pragma unroll
                for (int r = 0; r < MINE; ++r)
                    if (sees(row0 + r, first + i)) acc[c][r] = fmaf(weights[(row0 + r) * PLAIN_TILE + i], x, acc[c][r]);
            }
        }
    }
    __syncthreads();
    #pragma unroll
    for (int c = 0; c < COLUMNS; ++c)
        #pragma unroll
        for (int r = 0; r < MINE; ++r) done(row0 + r, column0 + c * THREADS, acc[c][r], top[row0 + r], total[row0 + r]);
    __syncthreads();
}

}  // namespace sd
