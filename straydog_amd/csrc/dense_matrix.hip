// sd_op_attention on the FP32 matrix instruction, 128 or 256 columns a head (reference gpu/token_mixing.hpp:356-520, 652-693): causal
// grouped-query attention over FP32 caches [context][kv_heads][dim], every product and sum in FP32.
//
// A workgroup of four waves owns TQ x 32 query rows of one K/V head (a query row = a token and one of the group's heads) and a run
// of steps of 32 keys.  The waves share the columns: S^T = K . Q^T by v_mfma_f32_32x32x2_f32 over a wave's quarter of them, the four
// partial scores added through LDS, the weights formed by every wave for itself, O^T += V^T . P^T for its quarter of the value columns.
// The quarter keeps queries and accumulators at 64 registers each for 64 query rows, so two workgroups fit a compute unit and the
// one multiplies while the other is between its products; and it makes one decode token (8 query rows) a step of 4 x 4096 cycles
// where a wave with all columns would take 16384.
//   * A step's K and V rows go from memory to LDS by themselves, 16-byte pieces turned by the row number so that the 32 rows of an
//     operand lie in different banks; one buffer each: the next K is asked for when the scores have been exchanged, the next V when the
//     products with this one are done (at 256 columns the exchange lies over K's buffer).
//   * A read of four columns of a key feeds four products a query tile; the C layout of S^T (lane = query row; keys 8 (r / 4) +
//     4 (lane / 32) + r % 4) is the B operand of O^T, register r for the two keys of the lane halves.
//   * Few query rows: the keys are cut into runs until every compute unit has two workgroups; dense_merge_kernel joins them.
//   * Values that are no finite numbers: found in the finished sums, which they always reach (a weight of zero does not silence
//     them), and the workgroup's run is worked again in plain arithmetic (plain_attention.hpp).  Kept out of the products in the loop
//     instead, and counted beside them by sign, they cost the loop registers: 120 us for the 115 below.
// Measured, 128 rows x 16 heads over 2 K/V heads of 256 columns at position 4096 (8.7 GFLOP): 115 us (76 TFLOP/s; 107 the kernel, 8 the merge; in the
// first milliseconds of load 118-122 the kernel) where the general kernel
// (LDS-fed vector FMAs, a workgroup a row and K/V head) took 5360; one row at 4096: 17 us where it took 295, at 60: 10 where it took 31.
#include "kernels.hpp"
#include "paged_rows.hpp"
#include "plain_attention.hpp"
#include "../../include/straydog_gpu.h"

#include <algorithm>
#include <type_traits>

using namespace sd;
using namespace sd::paged;

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

struct DenseArgs {
    const float *q, *keys, *values;
    const int32_t* positions;
    const float* gate;
    float* out;
    float* partial;                 // splits > 1: [pair][split][dim], then [pair][split] (maximum, sum); a pair = (row, head)
    unsigned context, rows, heads, kv_heads, group, splits;
    float scale;
};

// the lane's keys seen by a row at `position`, clipped to the cache
__device__ __forceinline__ int seen_keys(int position, unsigned context) { return position < 0 ? 0 : int(min(unsigned(position) + 1u, context)); }

template<int DIM, int TQ>
__global__ void __launch_bounds__(256, 2) dense_matrix_kernel(DenseArgs a) {
    constexpr int COLS = DIM / 4, ROW = DIM * 4, PIECES = DIM / 4, CT = COLS / 32, SIDE = 32 * ROW;      // a wave's columns; bytes and 16-byte pieces of a row; column tiles
    constexpr int PER_LOAD = 1024 / ROW, MINE = 32 / PER_LOAD / 4;                                     // rows a load, loads a wave and side
    const int thread = threadIdx.x, lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread >> 6), i = lane & 31, half = lane >> 5;
    const unsigned tile = blockIdx.x, split = blockIdx.y, kvh = blockIdx.z;
    extern __shared__ uint8_t lds[];
    uint8_t *kside = lds, *vside = lds + SIDE;
    floatx4* exchange = reinterpret_cast<floatx4*>(DIM == 256 ? kside : lds + 2 * SIDE);               // [wave][TQ][4][64]

    const unsigned last_row = a.rows * a.group - 1;
    int limit[TQ], most = 0, least = 0x7fffffff;          // the keys a row sees; the most and the fewest of the tile's rows
    float q[TQ][COLS / 2];
    #pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const unsigned at = tile * 32 * TQ + 32 * t + i, here = min(at, last_row);
        const unsigned row = here / a.group, head = kvh * a.group + here % a.group;
        const int seen = seen_keys(a.positions[row], a.context);
        limit[t] = at <= last_row ? seen : 0;
        most = max(most, limit[t]);
        if (at <= last_row) least = min(least, seen);
        const float* from = a.q + (size_t(row) * a.heads + head) * DIM + wave * COLS + 4 * half;
        #pragma unroll
        for (int c = 0; c < COLS / 8; ++c) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(from + 8 * c);
            #pragma unroll
            for (int j = 0; j < 4; ++j) q[t][4 * c + j] = x[j];
        }
    }
    #pragma unroll
    for (int offset = 16; offset; offset /= 2) { most = max(most, __shfl_xor(most, offset)); least = min(least, __shfl_xor(least, offset)); }
    most = __builtin_amdgcn_readfirstlane(most); least = __builtin_amdgcn_readfirstlane(least);
    const unsigned steps = unsigned(most + 31) / 32;
    const unsigned begin = unsigned(uint64_t(steps) * split / a.splits), end = unsigned(uint64_t(steps) * (split + 1) / a.splits);

    // A side's rows of a step, a quarter of them a wave: a piece of row r at place piece ^ (r % 16).  Rows past the last key any
    // query row sees are read from that one.
    const auto ask = [&](const float* from, uint8_t* side, unsigned step) {
        const int lane = fresh(thread) & 63;
        #pragma unroll
        for (int n = 0; n < MINE; ++n) {
            const int r = PER_LOAD * (MINE * wave + n) + lane / PIECES, piece = (lane % PIECES) ^ (r & 15);
            const unsigned key = min(step * 32 + r, unsigned(most - 1));
            load_to_lds<false>(from + (size_t(key) * a.kv_heads + kvh) * DIM + 4 * piece, side + 1024 * (MINE * wave + n));
        }
    };
    floatx16 acc[TQ][CT];
    float m[TQ], l[TQ];
    #pragma unroll
    for (int t = 0; t < TQ; ++t) {
        m[t] = NEG_BIG; l[t] = 0.0f;
        #pragma unroll
        for (int c = 0; c < CT; ++c)
            #pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][c][r] = 0.0f;
    }
    settle_loads();
    if (begin < end) { ask(a.keys, kside, begin); ask(a.values, vside, begin); }
    const auto advance = [&](auto every_row_sees, unsigned step) {
        constexpr bool WHOLE = decltype(every_row_sees)::value;
        // (loads finish in the order they were asked for: K's before V's)
        wait_loads<MINE>();
        ring_barrier();
        floatx16 s[TQ];
        #pragma unroll
        for (int t = 0; t < TQ; ++t)
            #pragma unroll
            for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
        const int here = fresh(thread) & 63, i = here & 31, half = here >> 5;
        const uint8_t* krow = kside + i * ROW;
        #pragma unroll
        for (int c = 0; c < COLS / 8; ++c) {
            const floatx4 k = *reinterpret_cast<const floatx4*>(krow + 16 * ((wave * (COLS / 4) + 2 * c + half) ^ (i & 15)));
            #pragma unroll
            for (int j = 0; j < 4; ++j)
                #pragma unroll
                for (int t = 0; t < TQ; ++t) s[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[j], q[t][4 * c + j], s[t], 0, 0, 0);
        }
        if (DIM == 256) ring_barrier();                    // K's buffer is free: the exchange lies over it
        #pragma unroll
        for (int t = 0; t < TQ; ++t)
            #pragma unroll
            for (int n = 0; n < 4; ++n)
                exchange[((wave * TQ + t) * 4 + n) * 64 + lane] = floatx4{s[t][4 * n], s[t][4 * n + 1], s[t][4 * n + 2], s[t][4 * n + 3]};
        ring_barrier();
        #pragma unroll
        for (int t = 0; t < TQ; ++t)
            #pragma unroll
            for (int n = 0; n < 4; ++n) {
                const floatx4* from = exchange + (t * 4 + n) * 64 + lane;
                const floatx4 sum = (from[0] + from[TQ * 256]) + (from[2 * TQ * 256] + from[3 * TQ * 256]);
                #pragma unroll
                for (int j = 0; j < 4; ++j) s[t][4 * n + j] = sum[j] * a.scale;
                if (n & 1) __builtin_amdgcn_sched_barrier(0);          // (eight reads in flight: with all thirty-two the registers spill)
            }
        wait_loads<0>();                                   // V's rows
        ring_barrier();
        if (step + 1 < end) ask(a.keys, kside, step + 1);
        #pragma unroll
        for (int t = 0; t < TQ; ++t) {
            float top = NEG_BIG;
            [[maybe_unused]] const int keys_left = limit[t] - int(step * 32) - 4 * half;
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (!WHOLE) s[t][r] = 8 * (r / 4) + r % 4 < keys_left ? s[t][r] : -INFINITY;
                top = fmaxf(top, s[t][r]);
            }
            float other = top;
            swap_halves(top, other);
            top = fmaxf(top, other);
            // the reference maximum moves only when some row's has outgrown it by more than 2^8 (weights stay below 2^8)
            if (step == begin) m[t] = top;
            else if (__any((top - m[t]) * LOG2E > 8.0f)) {
                asm volatile("; new reference maxima" ::: "memory");
                const float higher = fmaxf(m[t], top), alpha = __builtin_amdgcn_exp2f((m[t] - higher) * LOG2E);
                m[t] = higher;
                l[t] *= alpha;
                #pragma unroll
                for (int c = 0; c < CT; ++c) acc[t][c] *= alpha;
            }
            const float offset = -m[t] * LOG2E;
            float sum = 0.0f;
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[t][r] = __builtin_amdgcn_exp2f(fmaf(s[t][r], LOG2E, offset));
                sum += s[t][r];
            }
            l[t] += sum;
        }
        const auto key_of = [&](int r) { return 8 * (r / 4) + 4 * half + r % 4; };
        const auto value_place = [&](int r) {
            return reinterpret_cast<const float*>(vside + key_of(r) * ROW + 16 * ((wave * (COLS / 4) + (CT * i) / 4) ^ (key_of(r) & 15)) + 4 * ((CT * i) % 4));
        };
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
            float v[CT];
            if (CT == 2) { const float2 pair = *reinterpret_cast<const float2*>(value_place(r)); v[0] = pair.x; v[CT - 1] = pair.y; }
            else v[0] = value_place(r)[0];
            #pragma unroll
            for (int t = 0; t < TQ; ++t)
                #pragma unroll
                for (int c = 0; c < CT; ++c) acc[t][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[c], s[t][r], acc[t][c], 0, 0, 0);
        }
        ring_barrier();
        if (step + 1 < end) ask(a.values, vside, step + 1);
    };
    // the steps whose keys every row sees, then those that some rows see the end of
    unsigned step = begin;
    for (; step < end && int(step * 32 + 32) <= least; ++step) advance(std::true_type{}, step);
    for (; step < end; ++step) advance(std::false_type{}, step);
    // Sums that are no finite numbers: a value is none (zero times it is not zero, so it has reached rows that do not see its key too), or a
    // score.  A sum of weights that is not positive, of a row that sees keys of the run: its scores all lie below the reference
    // maximum that stands for nothing seen.  The run is then worked again in plain arithmetic.
    bool odd = false;
    #pragma unroll
    for (int t = 0; t < TQ; ++t) {
        float sum = l[t], other = sum;
        swap_halves(sum, other);
        l[t] = sum + other;
        odd |= begin < end && limit[t] > int(begin * 32) && !(l[t] > 0.0f && l[t] < INFINITY);
        #pragma unroll
        for (int c = 0; c < CT; ++c) {
            float probe = 0.0f;
            #pragma unroll
            for (int r = 0; r < 16; ++r) probe = fmaf(acc[t][c][r], 0.0f, probe);
            odd |= probe != 0.0f;
        }
    }
    uint32_t* const odd_waves = reinterpret_cast<uint32_t*>(lds + 2 * SIDE - 16);       // (past the stretches that outputs leave through)
    const bool odd_wave = __any(odd);
    if (lane == 0) odd_waves[wave] = odd_wave;
    ring_barrier();
    const uint4 odds = *reinterpret_cast<const uint4*>(odd_waves);
    const bool whole = a.splits == 1;
    const size_t pairs = size_t(a.rows) * a.heads;
    const auto pair_of = [&](unsigned at) { return size_t(at / a.group) * a.heads + kvh * a.group + at % a.group; };
    if (__builtin_expect(odds.x | odds.y | odds.z | odds.w, 0)) {
        constexpr int ROWS = 8;
        static_assert(plain_attention_bytes(ROWS, DIM) <= 2 * SIDE, "over the keys' and values' buffers");
        #pragma unroll 1
        for (unsigned first = tile * 32 * TQ; first < min(tile * 32 * TQ + 32 * TQ, last_row + 1); first += ROWS) {
            const auto row_of = [&](int row) { return min(first + row, last_row); };
            const auto sees = [&](int row, unsigned key) { return int(key) < seen_keys(a.positions[row_of(row) / a.group], a.context); };
            const auto row_at = [&](const float* from, unsigned key) { return PlainRow{from + (size_t(key) * a.kv_heads + kvh) * DIM, false}; };
            plain_attention<ROWS, DIM, 256>(
                lds, begin * 32, min(end * 32, unsigned(most)), a.scale, [&](int row, int column) { return a.q[pair_of(row_of(row)) * DIM + column]; },
                [&](unsigned key) { return row_at(a.keys, key); }, [&](unsigned key) { return row_at(a.values, key); }, sees,
                [&](int row, int column, float value, float top, float sum) {
                    if (first + row > last_row) return;
                    const size_t pair = pair_of(first + row);
                    if (whole) {
                        value /= sum;
                        if (a.gate) value *= 1.0f / (1.0f + expf(-a.gate[pair * DIM + column]));
                        a.out[pair * DIM + column] = value;
                        return;
                    }
                    a.partial[(pair * a.splits + split) * DIM + column] = value;
                    float* stats = a.partial + pairs * a.splits * DIM + (pair * a.splits + split) * 2;
                    if (column == 0) { stats[0] = top; stats[1] = sum; }
                });
        }
        return;
    }
    // Out through LDS, a stretch of its own for every wave: [32 query rows][COLS + 4]; then 16-byte pieces of rows.
    float* mine = reinterpret_cast<float*>(lds) + wave * 32 * (COLS + 4);
    constexpr int LANES = COLS / 4, ROWS_AT_ONCE = 64 / LANES;
    static_assert(4 * 32 * (COLS + 4) * 4 <= 2 * SIDE - 16, "the stretches");
    #pragma unroll
    for (int t = 0; t < TQ; ++t) {
        const float inverse = whole ? 1.0f / l[t] : 1.0f;
        #pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int x = 8 * (r / 4) + 4 * half + r % 4;
            #pragma unroll
            for (int c = 0; c < CT; ++c) mine[i * (COLS + 4) + CT * x + c] = acc[t][c][r] * inverse;
        }
        const unsigned first = tile * 32 * TQ + 32 * t;
        if (!whole && wave == 0 && half == 0 && first + i <= last_row) {
            const size_t pair = pair_of(first + i);
            float* stats = a.partial + pairs * a.splits * DIM + (pair * a.splits + split) * 2;
            stats[0] = l[t] > 0.0f ? m[t] : -INFINITY; stats[1] = l[t];
        }
        #pragma unroll 4
        for (int n = 0; n < 32; n += ROWS_AT_ONCE) {
            const unsigned at = first + n + lane / LANES;
            floatx4 x = *reinterpret_cast<const floatx4*>(mine + (n + lane / LANES) * (COLS + 4) + 4 * (lane % LANES));
            if (at > last_row) continue;
            const size_t pair = pair_of(at), column = wave * COLS + 4 * (lane % LANES);
            if (whole) {
                if (a.gate) {
                    const floatx4 gate = *reinterpret_cast<const floatx4*>(a.gate + pair * DIM + column);
                    #pragma unroll
                    for (int j = 0; j < 4; ++j) x[j] *= 1.0f / (1.0f + expf(-gate[j]));
                }
                *reinterpret_cast<floatx4*>(a.out + pair * DIM + column) = x;
            } else *reinterpret_cast<floatx4*>(a.partial + (pair * a.splits + split) * DIM + column) = x;
        }
    }
}

// (row, head): the runs under their common maximum, normalised and gated.  256 threads: a lane group has four columns each, the
// groups take the runs in turn, eight loads in flight, and are added through LDS.
template<int DIM>
__global__ void __launch_bounds__(256) dense_merge_kernel(DenseArgs a) {
    constexpr int LANES = DIM / 4, GROUPS = 256 / LANES, AT_ONCE = 8;
    const size_t pair = blockIdx.x, pairs = size_t(a.rows) * a.heads;
    const int lane = threadIdx.x & 63, column = 4 * (threadIdx.x % LANES);
    const unsigned part = threadIdx.x / LANES;
    const float* values = a.partial + pair * a.splits * DIM + column;
    const float* stats = a.partial + pairs * a.splits * DIM + pair * a.splits * 2;
    __shared__ floatx4 sums[GROUPS][LANES];
    __shared__ float totals[GROUPS];
    float top = -INFINITY;                    // (a run without a weight has that one)
    for (unsigned s = lane; s < a.splits; s += 64) top = fmaxf(top, stats[2 * s]);
    #pragma unroll
    for (int offset = 32; offset; offset /= 2) top = fmaxf(top, __shfl_xor(top, offset));
    floatx4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    float total = 0.0f;
    for (unsigned s0 = part; s0 < a.splits; s0 += GROUPS * AT_ONCE) {
        floatx4 x[AT_ONCE];
        float tops[AT_ONCE], parts[AT_ONCE];
        #pragma unroll
        for (int n = 0; n < AT_ONCE; ++n) {
            const unsigned s = min(s0 + GROUPS * n, a.splits - 1);
            x[n] = *reinterpret_cast<const floatx4*>(values + size_t(s) * DIM);
            tops[n] = stats[2 * s]; parts[n] = stats[2 * s + 1];
        }
        #pragma unroll
        for (int n = 0; n < AT_ONCE; ++n) {
            // (past the last run: its numbers again; they, and those of a run without a weight, may be none that zero silences)
            const bool real = s0 + GROUPS * n < a.splits && tops[n] != -INFINITY;
            const float weight = __builtin_amdgcn_exp2f((tops[n] - top) * LOG2E);
            total = real ? fmaf(parts[n], weight, total) : total;
            #pragma unroll
            for (int j = 0; j < 4; ++j) sum[j] = real ? fmaf(x[n][j], weight, sum[j]) : sum[j];
        }
    }
    sums[part][threadIdx.x % LANES] = sum;
    if (threadIdx.x % LANES == 0) totals[part] = total;
    __syncthreads();
    if (part) return;
    #pragma unroll
    for (int g = 1; g < GROUPS; ++g) { sum += sums[g][threadIdx.x]; total += totals[g]; }
    sum *= 1.0f / total;
    if (a.gate) {
        const floatx4 gate = *reinterpret_cast<const floatx4*>(a.gate + pair * DIM + column);
        #pragma unroll
        for (int j = 0; j < 4; ++j) sum[j] *= 1.0f / (1.0f + expf(-gate[j]));
    }
    *reinterpret_cast<floatx4*>(a.out + pair * DIM + column) = sum;
}

template<int DIM, int TQ>
void launch(Device& d, const DenseArgs& args, unsigned tiles) {
    constexpr size_t shared = 2 * 32 * size_t(DIM) * 4 + (DIM == 256 ? 0 : TQ * 4 * 4096);
    raise_shared_limit(d, reinterpret_cast<const void*>(&dense_matrix_kernel<DIM, TQ>), shared);
    timed_launch(d, &dense_matrix_kernel<DIM, TQ>, dim3(tiles, args.splits, args.kv_heads), dim3(256), shared, args);
    SD_CHECK(hipGetLastError());
    if (args.splits > 1) {
        dense_merge_kernel<DIM><<<unsigned(size_t(args.rows) * args.heads), 256, 0, d.stream>>>(args);
        SD_CHECK(hipGetLastError());
    }
}

}  // namespace

namespace sd {

bool dense_matrix_supported(uint64_t context, uint64_t rows, uint64_t heads, uint64_t kv_heads, uint64_t dim, const float* q, const float* keys, const float* values,
                            const float* gate, const float* out) {
    return (dim == 128 || dim == 256) && context < (uint64_t(1) << 31) && rows * (heads / kv_heads) < (uint64_t(1) << 31) && kv_heads < 65536 &&
           (uintptr_t(q) | uintptr_t(keys) | uintptr_t(values) | uintptr_t(gate) | uintptr_t(out)) % 16 == 0;
}

// scratch: room for `scratch_splits` runs of every (row, head), the caller's (the reference's contract)
void dense_matrix(Device& d, const float* q, const float* keys, const float* values, uint64_t context, const int32_t* positions, uint64_t rows, uint64_t heads,
                  uint64_t kv_heads, uint64_t dim, float scale, const float* gate, float* scratch, uint64_t scratch_splits, float* out) {
    DenseArgs args{};
    args.q = q; args.keys = keys; args.values = values; args.positions = positions; args.gate = gate; args.out = out; args.partial = scratch;
    args.context = unsigned(context); args.rows = unsigned(rows); args.heads = unsigned(heads); args.kv_heads = unsigned(kv_heads); args.group = unsigned(heads / kv_heads);
    args.scale = scale;
    const uint64_t query_rows = rows * args.group;
    const int tq = query_rows > 32 ? 2 : 1;
    const unsigned tiles = unsigned((query_rows + 32 * tq - 1) / (32 * tq));
    // runs of keys until every compute unit has two workgroups, a step of 32 keys each at least; where the caller's scratch does not
    // hold them they go to the handle's workspace
    const uint64_t steps = (context + 31) / 32, items = uint64_t(tiles) * kv_heads;
    args.splits = unsigned(std::min<uint64_t>({std::max<uint64_t>(1, 2 * uint64_t(d.compute_units) / items), steps, 128}));
    OptionalSpace space;
    if (args.splits > scratch_splits || uintptr_t(scratch) % 16) {
        if (args.splits > 1) space = optional_space(d, size_t(rows * heads) * args.splits * (dim + 2) * 4);
        args.partial = static_cast<float*>(space.at);
        if (!args.partial) {                              // (a graph is being recorded and the workspace is smaller)
            args.splits = uintptr_t(scratch) % 16 ? 1 : unsigned(std::min<uint64_t>(args.splits, scratch_splits));
            args.partial = scratch;
        }
    }
    if (dim == 128) { if (tq == 2) launch<128, 2>(d, args, tiles); else launch<128, 1>(d, args, tiles); }
    else { if (tq == 2) launch<256, 2>(d, args, tiles); else launch<256, 1>(d, args, tiles); }
}

}  // namespace sd
