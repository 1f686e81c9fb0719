// sd_op_sparse_attention on the matrix cores, rows of 512 columns: each query row attends the window rows of a ring and the
// compressed rows its selection lists, keys = values, a per-head sink in the maximum and the denominator only, rope on the last
// columns of the queries and (turned back) of the outputs (reference gpu/ops.hpp:1240-1297, rope :1318-1328, entry
// gpu/kernels.cpp:5311-5476).
//
// FP32 in, FP32 out: the products run on v_mfma_f32_16x16x32_bf16, sixteen times the FP32 matrix rate, with every FP32 operand as
// three BF16 terms (value, what its rounding left, what that one's left: 24 bits, exact).  A BF16 row has one term, so a score is
// three products a column and a value sum three (the weights' terms); a row in FP32 (the window's, or compressed rows in FP32)
// takes the six pairs of terms above 2^-24; the three smallest pairs, below the last place of an FP32 product, are left out.  A score
// has an accumulator for each order of magnitude, added smallest first; a value sum has one, which takes a step's planes of terms
// smallest first.  An FP32 row whose values fit BF16 gives the bits of the tagged BF16 row: the extra products add zeros.  Infinities, NaNs and numbers past BF16's
// largest make NaNs of the sums they reach: the workgroup's run is then worked again in plain arithmetic (plain_attention.hpp); the
// test for it, once a run, is 0.5 us of one row's 54 and nothing that shows of 256 rows' 418.
//
// Shape of the work (wave64, one workgroup a compute unit):
//   * a workgroup owns one query row, HT x 16 of its heads (64: a gathered row serves all heads at once) and a run of steps of 32
//     keys; two waves share 16 heads, each with half of the 512 columns: it multiplies its half of the queries (96 registers of terms)
//     with its half of the keys, the two add their partial scores through LDS, both form the weights, and each sums its half of the
//     value columns (64 registers).  That fits two waves a SIMD, which a wave with all 512 columns (320 registers) does not;
//   * a wave brings in whole rows (32 / waves of them a step, the row's address the wave's): BF16 rows go from memory to a padded tile
//     in LDS by themselves, a step ahead, their numbers in the selection read another step ahead (fetched through registers they left
//     51 registers to spill, and each number waited for the row before it: 128 us, then 109, then 97); FP32 rows are split into three
//     planes of terms on their way;
//   * the scores S^T = K . Q^T leave the weights in the B-operand layout of O^T += V^T . P^T; a lane's place in a value operand
//     stands for eight neighbouring columns in eight products, so nothing is transposed (as in latent_gather.hip).
// Many rows (a prompt) give every compute unit a workgroup that finishes its outputs; few rows are cut into runs of steps whose
// (maximum, sum, unnormalised outputs) latent_rows_merge_kernel puts together.
// Measured at 64 heads, a window of 128 and 512 selected BF16 rows: 256 rows in 89 us (93-97 in the first milliseconds of load, as the figures above) where the general kernel (FP32 on the vector
// units, a key row read once for eight heads) took 1400; one row in 15.4 + 4.6 us where it took 447.  Of the 97 us the
// queries and outputs take 13 (67 MB); a step of BF16 rows takes 3.3 us, of which its products are 1.4 and its LDS reads, in phase with them, 0.9.  The differences from 64-bit
// arithmetic are as large as before, 1e-6 at outputs of order one.
#include "kernels.hpp"
#include "paged_rows.hpp"
#include "plain_attention.hpp"

#include <algorithm>

using namespace sd;
using namespace sd::paged;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int DIM = 512, HALF = DIM / 2, PITCH = 2 * DIM + 16, PLANE = STEP * PITCH, PAIRS_MAX = 64;

struct RowsArgs {
    const float* q;                    // [rows][heads][512]
    const float* raw;                  // [raw_rows][512], position p in row p % raw_rows
    unsigned raw_rows;
    const int32_t* positions;
    long long window;
    const void* compressed;            // [compressed_rows][512] BF16 or FP32
    unsigned compressed_rows;
    const int32_t* selected;           // [rows][selections], an entry that names no row is skipped
    unsigned selections;
    const float* sinks;
    unsigned heads, chunks;
    float scale;
    unsigned pairs; const float* frequencies;
    const double2* turns;              // the pass's table of (cosine, sine), pairs a row, or null: formed here
    float* out;                        // [rows][heads][512]
    float* partial;                    // chunks > 1: [row][chunk][head][512], then [row][chunk][head] (maximum, sum)
};

// (v_cvt_pk_bf16_f32: two values to BF16, nearest even)
__device__ __forceinline__ uint32_t to_bf16_pair(float low, float high) {
    uint32_t pair;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(pair) : "v"(low), "v"(high));
    return pair;
}
// Two values as three pairs of BF16 terms.
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& high, uint32_t& middle, uint32_t& low) {
    high = to_bf16_pair(x, y);
    x -= __uint_as_float(high << 16); y -= __uint_as_float(high & 0xffff0000u);
    middle = to_bf16_pair(x, y);
    x -= __uint_as_float(middle << 16); y -= __uint_as_float(middle & 0xffff0000u);
    low = to_bf16_pair(x, y);
}
struct Terms { uint4 high, middle, low; };       // eight values
__device__ __forceinline__ Terms split_eight(const float (&x)[8]) {
    Terms t;
    split_pair(x[0], x[1], t.high.x, t.middle.x, t.low.x);
    split_pair(x[2], x[3], t.high.y, t.middle.y, t.low.y);
    split_pair(x[4], x[5], t.high.z, t.middle.z, t.low.z);
    split_pair(x[6], x[7], t.high.w, t.middle.w, t.low.w);
    return t;
}
__device__ __forceinline__ bf16x8 operand(const uint4& bits) { return __builtin_bit_cast(bf16x8, bits); }
__device__ __forceinline__ floatx4 product(const bf16x8& a, const bf16x8& b, const floatx4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// (x, y) turned by the table's angle
__device__ __forceinline__ void turn(float& x, float& y, double2 t) {
    const double a = x, b = y;
    x = float(a * t.x - b * t.y);
    y = float(a * t.y + b * t.x);
}

// O^T += V^T . P^T for eight products: place li of product c's operand is value column c of the lane's eight from `from` on, its k-slots
// the tile's rows {4g..4g+3, 16+4g..16+4g+3}; the N weight operands follow one another, two columns in turn.
template<int N>
__device__ __forceinline__ void value_products(const uint8_t* from, const bf16x8 (&weights)[N], floatx4* acc) {
    uint4 rows8[8];
    #pragma unroll
    for (int e = 0; e < 8; ++e) rows8[e] = *reinterpret_cast<const uint4*>(from + (e < 4 ? e : 12 + e) * PITCH);
    #pragma unroll
    for (int c = 0; c < 8; c += 2) {
        bf16x8 v[2];
        #pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t words[4];
            #pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint4 &low = rows8[2 * w], &high = rows8[2 * w + 1];
                const uint32_t lo = c == 0 ? low.x : c == 2 ? low.y : c == 4 ? low.z : low.w, hi = c == 0 ? high.x : c == 2 ? high.y : c == 4 ? high.z : high.w;
                words[w] = byte_perm(hi, lo, i ? 0x07060302u : 0x05040100u);
            }
            v[i] = operand(uint4{words[0], words[1], words[2], words[3]});
        }
        #pragma unroll
        for (int n = 0; n < N; ++n)
            #pragma unroll
            for (int i = 0; i < 2; ++i) acc[c + i] = product(v[i], weights[n], acc[c + i]);
    }
}

constexpr size_t shared_bytes(int ht) {
    const size_t loop = 3 * size_t(PLANE) + 2 * 2 * ht * 64 * 8 * 4, leave = size_t(2 * ht) * 16 * (HALF + 4) * 4;
    return (loop > leave ? loop : leave) + PAIRS_MAX * 16 + 2 * STEP * 4;
}

template<int HT, bool BF16>
__global__ void __launch_bounds__(128 * HT, HT == 4 ? 2 : 1) latent_rows_kernel(RowsArgs a) {
    constexpr int WAVES_HERE = 2 * HT, MINE = STEP / WAVES_HERE, KSTEPS = HALF / 32, TILES = HALF / 16;
    const unsigned row = blockIdx.x / a.chunks, chunk = blockIdx.x % a.chunks;
    const int thread = threadIdx.x, lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread >> 6), li = lane & 15, g = lane >> 4;
    const int half = wave & 1, head0 = int(blockIdx.y) * 16 * HT + 16 * (wave >> 1), head = head0 + li;
    extern __shared__ uint8_t lds[];
    double2* turns = reinterpret_cast<double2*>(lds);                                   // [pairs]
    uint32_t* seen = reinterpret_cast<uint32_t*>(lds + PAIRS_MAX * 16);                 // two of [32]: whether the step's row exists
    uint8_t* tiles = lds + PAIRS_MAX * 16 + 2 * STEP * 4;                               // [3][32][PITCH]
    floatx4* exchange = reinterpret_cast<floatx4*>(tiles + 3 * PLANE);                  // two of [wave][2][64]

    const long long p = a.positions[row], first = max(0ll, p - a.window + 1);
    const unsigned raw_count = p < 0 ? 0u : unsigned(p - first + 1), raw_steps = (raw_count + STEP - 1) / STEP;
    const unsigned steps = raw_steps + (a.selections + STEP - 1) / STEP;
    const unsigned begin = unsigned(uint64_t(steps) * chunk / a.chunks), end = unsigned(uint64_t(steps) * (chunk + 1) / a.chunks);
    const int32_t* selected = a.selected + size_t(row) * a.selections;

    if (thread < int(a.pairs)) {
        double2 t;
        if (a.turns) t = a.turns[size_t(row) * a.pairs + thread];
        else sincos(double(p) * double(a.frequencies[thread]), &t.y, &t.x);
        turns[thread] = t;
    }
    // A step's rows.  BF16 rows go straight to their plane of the tile, a row an instruction, asked for a step ahead; FP32 rows come
    // through registers, where they are split.  A row that does not exist is read from the ring's first and zeroed afterwards.  The
    // selection's entries are read another step ahead, the wave's MINE rows in as many lanes: asked for where they are needed, each
    // would wait for the row before it.
    int32_t names = -1;
    const auto read_names = [&](unsigned step) {
        const unsigned index = (step - raw_steps) * STEP + wave + WAVES_HERE * (lane % MINE);
        const int32_t entry = selected[min(index, a.selections - 1)];
        names = index < a.selections ? entry : -1;
    };
    const auto named_row = [&](int j, bool& exists) -> const uint8_t* {
        const uint32_t at = uint32_t(__builtin_amdgcn_readlane(names, j));
        exists = at < a.compressed_rows;                                                    // (a negative entry is a large unsigned one)
        return exists ? static_cast<const uint8_t*>(a.compressed) + size_t(at) * DIM * (BF16 ? 2 : 4) : reinterpret_cast<const uint8_t*>(a.raw);
    };
    uint32_t present = 0, any_row = 0;       // bit j: the wave's j-th row of the step asked for ahead, or of any step, exists
    const auto ask = [&](unsigned step) {
        present = 0;
        #pragma unroll
        for (int j = 0; j < MINE; ++j) {
            bool exists;
            const uint8_t* from = named_row(j, exists);
            load_run_to_lds<false, 1>(from, lds_address(tiles + (step & 1) * PLANE + (wave + WAVES_HERE * j) * PITCH), 16 * lane);
            present |= exists ? 1u << j : 0u;
        }
        any_row |= present;
        if (step + 1 < end) read_names(step + 1);
    };
    if (end > raw_steps) read_names(max(begin, raw_steps));

    // queries: the wave's half of its heads' columns as three terms
    uint4 qh[KSTEPS], qm[KSTEPS], ql[KSTEPS];
    ring_barrier();
    {
        const float* from = a.q + (size_t(row) * a.heads + min(head, int(a.heads) - 1)) * DIM + HALF * half + 8 * g;
        const int rotated = DIM - 2 * int(a.pairs);
        #pragma unroll
        for (int b = 0; b < KSTEPS; ++b) {
            const float4 x0 = *reinterpret_cast<const float4*>(from + 32 * b), x1 = *reinterpret_cast<const float4*>(from + 32 * b + 4);
            float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            if (b >= KSTEPS / 2 && half && HALF + 32 * b + 32 > rotated) {             // (at most 128 columns are turned)
                #pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    const int column = HALF + 32 * b + 8 * g + i;
                    float u = x[i], v = x[i + 1];
                    turn(u, v, turns[max(column - rotated, 0) / 2]);
                    x[i] = column >= rotated ? u : x[i]; x[i + 1] = column >= rotated ? v : x[i + 1];
                }
            }
            const Terms t = split_eight(x);
            qh[b] = t.high; qm[b] = t.middle; ql[b] = t.low;
        }
    }
    floatx4 acc[TILES];
    #pragma unroll
    for (int j = 0; j < TILES; ++j) acc[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = NEG_BIG, l = 0.0f;

    for (unsigned step = begin; step < end; ++step) {
        const bool wide = !BF16 || step < raw_steps;                     // rows of three terms: all three planes; else planes 0 and 1 in turn
        const unsigned turn_of = step & 1;
        uint8_t* tile = tiles + (wide ? 0u : turn_of * PLANE);
        uint32_t* here = seen + turn_of * STEP;
        if (wide) {
            float4 pieces[MINE][2];
            present = 0;
            #pragma unroll
            for (int j = 0; j < MINE; ++j) {
                bool exists;
                const uint8_t* from;
                if (BF16 || step < raw_steps) {
                    const unsigned index = step * STEP + wave + WAVES_HERE * j;
                    exists = index < raw_count;
                    from = reinterpret_cast<const uint8_t*>(a.raw + size_t(exists ? unsigned(first + index) % a.raw_rows : 0u) * DIM);
                } else from = named_row(j, exists);
                pieces[j][0] = reinterpret_cast<const float4*>(from)[2 * lane]; pieces[j][1] = reinterpret_cast<const float4*>(from)[2 * lane + 1];
                present |= exists ? 1u << j : 0u;
            }
            any_row |= present;
            if (!BF16 && step >= raw_steps && step + 1 < end) read_names(step + 1);
            #pragma unroll
            for (int j = 0; j < MINE; ++j) {
                const float4 u = pieces[j][0], v = pieces[j][1];
                const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
                Terms t = split_eight(x);
                if (!((present >> j) & 1u)) t.high = t.middle = t.low = uint4{0u, 0u, 0u, 0u};             // (its weights are zero, and zero times anything finite adds nothing)
                uint8_t* to = tile + (wave + WAVES_HERE * j) * PITCH + 16 * lane;
                *reinterpret_cast<uint4*>(to) = t.high;
                *reinterpret_cast<uint4*>(to + PLANE) = t.middle;
                *reinterpret_cast<uint4*>(to + 2 * PLANE) = t.low;
                if (lane == 0) here[wave + WAVES_HERE * j] = (present >> j) & 1u;
            }
        } else {
            if (step == begin || step == raw_steps) ask(step);
            wait_loads_here<0>();
            #pragma unroll
            for (int j = 0; j < MINE; ++j) {
                const int r = wave + WAVES_HERE * j;
                if (!((present >> j) & 1u)) *reinterpret_cast<uint4*>(tile + r * PITCH + 16 * lane) = uint4{0u, 0u, 0u, 0u};
                if (lane == 0) here[r] = (present >> j) & 1u;
            }
        }
        ring_barrier();
        if (!wide && step + 1 < end) ask(step + 1);
        // S^T over the wave's columns: keys (4 a lane group) x heads (lane li), one accumulator an order of magnitude
        floatx4 s[2];
        {
            floatx4 s0[2], s1[2], s2[2];
            #pragma unroll
            for (int t = 0; t < 2; ++t) s0[t] = s1[t] = s2[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            const uint8_t* rows_at = tile + li * PITCH + 2 * HALF * half + 16 * g;
            #pragma unroll
            for (int b = 0; b < KSTEPS; ++b)
                #pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const bf16x8 k = *reinterpret_cast<const bf16x8*>(rows_at + 16 * t * PITCH + 64 * b);
                    s0[t] = product(k, operand(qh[b]), s0[t]);
                    s1[t] = product(k, operand(qm[b]), s1[t]);
                    s2[t] = product(k, operand(ql[b]), s2[t]);
                }
            if (wide) {
                #pragma unroll
                for (int b = 0; b < KSTEPS; ++b)
                    #pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const bf16x8 km = *reinterpret_cast<const bf16x8*>(rows_at + PLANE + 16 * t * PITCH + 64 * b);
                        const bf16x8 kl = *reinterpret_cast<const bf16x8*>(rows_at + 2 * PLANE + 16 * t * PITCH + 64 * b);
                        s1[t] = product(km, operand(qh[b]), s1[t]);
                        s2[t] = product(km, operand(qm[b]), s2[t]);
                        s2[t] = product(kl, operand(qh[b]), s2[t]);
                    }
            }
            #pragma unroll
            for (int t = 0; t < 2; ++t) s[t] = (s2[t] + s1[t]) + s0[t];
        }
        floatx4* given = exchange + (turn_of * WAVES_HERE + wave) * 128;
        const floatx4* taken = exchange + (turn_of * WAVES_HERE + (wave ^ 1)) * 128;
        given[lane] = s[0]; given[64 + lane] = s[1];
        ring_barrier();
        s[0] += taken[lane]; s[1] += taken[64 + lane];
        float w[8], top = NEG_BIG;
        #pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint4 flags = *reinterpret_cast<const uint4*>(here + 16 * t + 4 * g);
            const uint32_t flag[4] = {flags.x, flags.y, flags.z, flags.w};
            #pragma unroll
            for (int r = 0; r < 4; ++r) {
                w[4 * t + r] = flag[r] ? s[t][r] * a.scale : -INFINITY;
                top = fmaxf(top, w[4 * t + r]);
            }
        }
        top = row_max(top);
        // the reference maximum moves only when some head's has outgrown it by more than 2^8 (weights stay below 2^8)
        if (step == begin) m = top;
        else if (__any((top - m) * LOG2E > 8.0f)) {
            asm volatile("; new reference maxima" ::: "memory");
            const float m_new = fmaxf(m, top), alpha = __builtin_amdgcn_exp2f((m - m_new) * LOG2E);
            m = m_new;
            l *= alpha;
            #pragma unroll
            for (int j = 0; j < TILES; ++j) acc[j] *= alpha;
        }
        const float offset = -m * LOG2E;
        #pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = __builtin_amdgcn_exp2f(fmaf(w[i], LOG2E, offset));
        l += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
        const Terms wt = split_eight(w);
        const bf16x8 wh = operand(wt.high), wm = operand(wt.middle), wl = operand(wt.low);
        // O^T: place li of a value operand stands for column HALF * half + 128 q + 8 li + c in tile 8 q + c
        #pragma unroll
        for (int q = 0; q < TILES / 8; ++q) {
            const uint8_t* from = tile + 4 * g * PITCH + 2 * (HALF * half + 128 * q + 8 * li);
            if (wide) {
                value_products<1>(from + 2 * PLANE, {wh}, acc + 8 * q);
                value_products<2>(from + PLANE, {wm, wh}, acc + 8 * q);
            }
            value_products<3>(from, {wl, wm, wh}, acc + 8 * q);
        }
        if (wide) ring_barrier();          // the planes are written again by the next step
    }
    l = row_sum(l);
    // Sums that are no finite numbers: an operand is none, or lies beyond BF16's largest (its terms, and zero weights, then make NaNs of what
    // has nothing to do with it), or a score.  A head's sum of weights that is zero though there are rows: its scores lie below the reference maximum that stands for
    // nothing seen.  The run is worked again in plain arithmetic.
    bool odd = !(l < INFINITY);
    #pragma unroll
    for (int j = 0; j < TILES; j += 4) {
        float probe = 0.0f;
        #pragma unroll
        for (int i = 0; i < 16; ++i) probe = fmaf(acc[j + i / 4][i % 4], 0.0f, probe);
        odd |= probe != 0.0f;
    }
    const uint32_t found = (__any(odd) ? 1u : 0u) | (__any(l == 0.0f) ? 2u : 0u) | (any_row ? 4u : 0u);
    uint32_t* const found_by = seen + (end & 1) * STEP;        // (the half that the last step did not use)
    if (lane == 0) found_by[wave] = found;
    ring_barrier();
    uint32_t odds = 0;
    #pragma unroll
    for (int w = 0; w < WAVES_HERE; ++w) odds |= found_by[w];
    const int back = DIM - 2 * int(a.pairs);
    float* const to = a.chunks == 1 ? a.out + size_t(row) * a.heads * DIM : a.partial + size_t(blockIdx.x) * a.heads * DIM;
    float* const stats = a.partial + size_t(gridDim.x) * a.heads * DIM + size_t(blockIdx.x) * a.heads * 2;      // (chunks > 1)
    if (__builtin_expect((odds & 1) || odds >= 6, 0)) {
        constexpr int ROWS = 16;
        static_assert(plain_attention_bytes(ROWS, DIM) <= 3 * PLANE, "over the tiles");
        const auto key_row = [&](unsigned index) {
            if (index < raw_steps * STEP) return PlainRow{index < raw_count ? a.raw + size_t(unsigned(first + index) % a.raw_rows) * DIM : nullptr, false};
            const unsigned place = index - raw_steps * STEP;
            const uint32_t at = place < a.selections ? uint32_t(selected[place]) : 0xffffffffu;
            return PlainRow{at < a.compressed_rows ? static_cast<const uint8_t*>(a.compressed) + size_t(at) * DIM * (BF16 ? 2 : 4) : nullptr, BF16};
        };
        float* const results = reinterpret_cast<float*>(tiles);              // [ROWS][DIM]
        #pragma unroll 1
        for (int head_first = int(blockIdx.y) * 16 * HT; head_first < min(int(blockIdx.y + 1) * 16 * HT, int(a.heads)); head_first += ROWS) {
            plain_attention<ROWS, DIM, 128 * HT>(
                tiles, begin * STEP, end * STEP, a.scale,
                [&](int r, int column) {
                    const float* from = a.q + (size_t(row) * a.heads + min(head_first + r, int(a.heads) - 1)) * DIM;
                    if (column < back) return from[column];
                    float u = from[column & ~1], v = from[column | 1];
                    turn(u, v, turns[(column - back) / 2]);
                    return column & 1 ? v : u;
                },
                key_row, key_row, [](int, unsigned) { return true; },
                [&](int r, int column, float value, float top, float sum) {
                    const int h = head_first + r;
                    if (h >= int(a.heads)) return;
                    if (a.chunks == 1) {
                        const float sink = a.sinks[h], higher = fmaxf(top, sink), keep = top == -INFINITY ? 0.0f : expf(top - higher);
                        value = value * keep / (sum * keep + expf(sink - higher));
                    } else if (column == 0) { stats[2 * h] = top; stats[2 * h + 1] = sum; }
                    results[r * DIM + column] = value;
                });
            for (int i = thread; i < ROWS * DIM; i += 128 * HT) {
                const int h = head_first + i / DIM, column = i % DIM;
                if (h >= int(a.heads)) break;
                float value = results[i];
                if (a.chunks == 1 && column >= back) {
                    double2 t = turns[(column - back) / 2];
                    t.y = -t.y;
                    float u = results[i & ~1], v = results[i | 1];
                    turn(u, v, t);
                    value = column & 1 ? v : u;
                }
                to[size_t(h) * DIM + column] = value;
            }
        }
        return;
    }
    // out through LDS (an accumulator's four values are columns 8 apart), a stretch of its own for every wave
    constexpr int ROW_WORDS = HALF + 4;
    float* mine = reinterpret_cast<float*>(tiles) + wave * 16 * ROW_WORDS;
    float inverse = 1.0f;
    if (a.chunks == 1) {
        const float sink = a.sinks[min(head, int(a.heads) - 1)], top = fmaxf(l > 0.0f ? m : -INFINITY, sink), keep = l > 0.0f ? __builtin_amdgcn_exp2f((m - top) * LOG2E) : 0.0f;
        inverse = keep / (l * keep + __builtin_amdgcn_exp2f((sink - top) * LOG2E));
    }
    #pragma unroll
    for (int j = 0; j < TILES; ++j)
        #pragma unroll
        for (int r = 0; r < 4; ++r) mine[li * ROW_WORDS + 128 * (j / 8) + 8 * (4 * g + r) + j % 8] = acc[j][r] * inverse;
    const int column = HALF * half + 4 * lane;
    #pragma unroll 4
    for (int h = 0; h < 16; ++h) {
        if (head0 + h >= int(a.heads)) break;
        floatx4 x = *reinterpret_cast<const floatx4*>(mine + h * ROW_WORDS + 4 * lane);
        if (a.chunks == 1 && column + 2 >= back) {
            #pragma unroll
            for (int i = 0; i < 4; i += 2)
                if (column + i >= back) {
                    double2 t = turns[(column + i - back) / 2];
                    t.y = -t.y;
                    float u = x[i], v = x[i + 1];
                    turn(u, v, t);
                    x[i] = u; x[i + 1] = v;
                }
        }
        *reinterpret_cast<floatx4*>(to + size_t(head0 + h) * DIM + column) = x;
    }
    if (a.chunks > 1 && half == 0 && g == 0 && head < int(a.heads)) { stats[2 * head] = l > 0.0f ? m : -INFINITY; stats[2 * head + 1] = l; }
}

// (row, head): the runs merged under their common maximum with the head's sink, normalised, turned back.  The runs' pieces are
// asked for eight at a time.
__global__ void __launch_bounds__(DIM / 4) latent_rows_merge_kernel(RowsArgs a) {
    const size_t row = blockIdx.x / a.heads, head = blockIdx.x % a.heads;
    const int t = threadIdx.x;
    const float* base = a.partial + (row * a.chunks * a.heads + head) * DIM;
    const float* stats = a.partial + size_t(gridDim.x) * a.chunks * DIM + (row * a.chunks * a.heads + head) * 2;
    const size_t step = size_t(a.heads) * DIM, stats_step = size_t(a.heads) * 2;
    __shared__ double2 turns[PAIRS_MAX];
    if (t < int(a.pairs)) {
        double2 at;
        if (a.turns) at = a.turns[row * a.pairs + t];
        else sincos(double(a.positions[row]) * double(a.frequencies[t]), &at.y, &at.x);
        turns[t] = at;
    }
    constexpr unsigned AT_ONCE = 8;
    const float sink = a.sinks[head];
    float top = sink;                                  // (a run without a weight has minus infinity for its maximum)
    for (unsigned c0 = 0; c0 < a.chunks; c0 += AT_ONCE) {
        float tops[AT_ONCE];
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) tops[i] = stats[min(c0 + i, a.chunks - 1) * stats_step];
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) top = fmaxf(top, tops[i]);
    }
    floatx4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    float sum = __builtin_amdgcn_exp2f((sink - top) * LOG2E);
    for (unsigned c0 = 0; c0 < a.chunks; c0 += AT_ONCE) {
        floatx4 values[AT_ONCE];
        float tops[AT_ONCE], sums[AT_ONCE];
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) {
            const size_t chunk = min(c0 + i, a.chunks - 1);
            values[i] = *reinterpret_cast<const floatx4*>(base + chunk * step + 4 * t);
            tops[i] = stats[chunk * stats_step];
            sums[i] = stats[chunk * stats_step + 1];
        }
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) {
            // (past the last run: its numbers again, which may be none that zero silences)
            const bool real = c0 + i < a.chunks;
            const float weight = __builtin_amdgcn_exp2f((tops[i] - top) * LOG2E);
            sum = real ? fmaf(sums[i], weight, sum) : sum;
            #pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = real ? fmaf(values[i][j], weight, x[j]) : x[j];
        }
    }
    x *= 1.0f / sum;
    __syncthreads();
    const int column = 4 * t, back = DIM - 2 * int(a.pairs);
    #pragma unroll
    for (int i = 0; i < 4; i += 2)
        if (column + i >= back) {
            double2 at = turns[(column + i - back) / 2];
            at.y = -at.y;
            float u = x[i], v = x[i + 1];
            turn(u, v, at);
            x[i] = u; x[i + 1] = v;
        }
    *reinterpret_cast<floatx4*>(a.out + size_t(blockIdx.x) * DIM + column) = x;
}

template<int HT, bool BF16>
void launch(Device& d, const RowsArgs& args, size_t rows, unsigned blocks) {
    raise_shared_limit(d, reinterpret_cast<const void*>(&latent_rows_kernel<HT, BF16>), shared_bytes(HT));
    timed_launch(d, &latent_rows_kernel<HT, BF16>, dim3(unsigned(rows * args.chunks), blocks), dim3(128 * HT), shared_bytes(HT), args);
}

}  // namespace

namespace sd {

bool latent_rows_supported(uint64_t dim, uint64_t raw_rows, uint64_t window, uint64_t compressed_rows, uint64_t selections, const void* q, const void* raw,
                           const void* compressed, const void* out) {
    constexpr uint64_t most = uint64_t(1) << 31;       // (counts the kernel keeps in 32 bits)
    return dim == DIM && raw_rows < most && window < most && compressed_rows < most && selections < most &&
           (uintptr_t(q) | uintptr_t(raw) | uintptr_t(compressed) | uintptr_t(out)) % 16 == 0;
}

void latent_rows(Device& d, const float* q, const float* raw, uint64_t raw_rows, const int32_t* positions, uint64_t window, const void* compressed, bool bf16,
                 uint64_t compressed_rows, const int32_t* selected, uint64_t selections, const float* sinks, uint64_t rows, uint64_t heads, float scale,
                 uint64_t pairs, const float* frequencies, const double2* turns, float* out) {
    RowsArgs args{};
    args.q = q; args.raw = raw; args.raw_rows = unsigned(raw_rows); args.positions = positions; args.window = (long long)(window); args.compressed = compressed;
    args.compressed_rows = unsigned(compressed_rows); args.selected = selected; args.selections = unsigned(selections); args.sinks = sinks;
    args.heads = unsigned(heads); args.scale = scale; args.pairs = unsigned(pairs); args.frequencies = frequencies; args.turns = turns; args.out = out;
    const int ht = heads > 32 ? 4 : 2;
    const unsigned blocks = unsigned((heads + 16 * ht - 1) / (16 * ht));
    // few rows: their steps of 32 keys in as many runs as give every compute unit a workgroup, the runs merged by a second launch
    const uint64_t steps = (window + STEP - 1) / STEP + (selections + STEP - 1) / STEP, room = d.compute_units / (rows * blocks);
    args.chunks = unsigned(std::min<uint64_t>(std::min<uint64_t>(steps, 64), std::max<uint64_t>(1, room)));
    OptionalSpace space;
    if (args.chunks > 1) {
        space = optional_space(d, size_t(rows) * args.chunks * heads * (DIM + 2) * 4);
        args.partial = static_cast<float*>(space.at);
        if (!args.partial) args.chunks = 1;            // (a graph is being recorded and the workspace is smaller: one run a row needs none)
    }
    if (ht == 4) { if (bf16) launch<4, true>(d, args, rows, blocks); else launch<4, false>(d, args, rows, blocks); }
    else { if (bf16) launch<2, true>(d, args, rows, blocks); else launch<2, false>(d, args, rows, blocks); }
    SD_CHECK(hipGetLastError());
    if (args.chunks > 1) {
        latent_rows_merge_kernel<<<unsigned(rows * heads), DIM / 4, 0, d.stream>>>(args);
        SD_CHECK(hipGetLastError());
    }
}

}  // namespace sd
