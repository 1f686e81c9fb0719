// Qwen's block indexer: the index inputs' normalisation and rotation, the pooled keys of four-position blocks, the exact block
// scores and the choice of the 512 best blocks per row.
//
// The arithmetic is the reference's (gpu/sparse_attention.hpp:2-23 qsa_rope/qsa_normalize, :87-139 qsa_pool/qsa_save_history,
// :141-155 qsa_block_scores, :172-241 qsa_select, :314-400 qsa_select_rows, :403-414 qsa_index_exact):
//   score(block) = sum over the 4 index heads, in order, of max(dot_h, 0), dot_h a chain of fused multiply-adds over the 128
//   columns in order (the bits do not depend on the tiling); a row with more than 512 complete blocks keeps the 512 whose raw
//   score bits are highest, ties to the earliest blocks, listed in block order with their four positions each, then the
//   positions of the incomplete block; a row with at most 512 complete blocks keeps every causal position.  Positions and the
//   count are stored as floats.
// The layout is the reference's too: pooled keys column-major blocks[column * pool + block], pool = context / 4 + 1, so a wave
// reading 64 neighbouring blocks of one column reads 256 contiguous bytes.
//
// Wave64 forms: one lane per block and all of a span's rows per lane while the span is short (decode, verification: the keys
// are read once from HBM, 512 bytes a block); a 32-row x 256-block tile per workgroup with operands staged through LDS for a
// prefill chunk (FP32 FMA-bound); a 1024-thread workgroup per row for the selection, the row's scores read once and held in LDS (and registers,
// beyond 32768 blocks), four 8-bit radix passes over per-wave LDS histograms (the first, where nearly all values share a digit, counted by ballots), and
// one ordered pass whose slots come from 64-wide ballots and a scan over (run, wave) counts.
#include "kernels.hpp"
#include "kv_codec.hpp"
#include "bound_choice.hpp"
#include "tree_sum.hpp"

using namespace sd;

namespace {

constexpr int HEADS = 4, COLUMNS = 128, KEEP = 512, RING = 16;

__device__ __forceinline__ float turn_angle(unsigned column, size_t position) { return float(position) / powf(1e7f, float(column % 32) / 32.0f); }
__device__ __forceinline__ float turned(float own, float partner, unsigned column, float cosine, float sine) { return own * cosine + (column < 32 ? -partner : partner) * sine; }
__device__ __forceinline__ float turn(float own, float partner, unsigned column, size_t position) {
    if (column >= 64) return own;
    const float angle = turn_angle(column, position);
    return turned(own, partner, column, cosf(angle), sinf(angle));
}

// A vector of `width` values (128 or 256), one per thread c < width: x * norm / sqrt(mean(x^2) + 1e-6), the first 64 columns turned
// for `position`.  Every thread of the workgroup calls it (the sum has barriers); values and sums are 256 floats of LDS each.
__device__ __forceinline__ float normalized(float x, const float* norm, unsigned width, size_t position, float* values, float* sums) {
    const unsigned c = threadIdx.x;
    if (c < width) values[c] = x * norm[c];
    const float denominator = sqrtf(tree_sum(c < width ? x * x : 0.0f, sums, width) / float(width) + 1e-6f);
    const float own = c < width ? values[c] / denominator : 0.0f;
    const float partner = c < 64 ? values[(c + 32) % 64] / denominator : 0.0f;
    const float value = turn(own, partner, c, position);
    __syncthreads();        // (values may be written again at once)
    return value;
}

// One workgroup of `width` threads per (row, head).
__global__ void __launch_bounds__(256) normalize_kernel(const float* source, const float* norm, unsigned heads, unsigned width, size_t stride,
                                                        size_t position, float* target) {
    __shared__ float values[256], sums[256];
    const size_t head = blockIdx.x, token = head / heads;
    const unsigned c = threadIdx.x;
    target[head * width + c] = normalized(source[head * stride + c], norm, width, position + token, values, sums);
}

// The mean of a block's four index-key inputs as a thread's column: taps in position order, earlier ones from the ring.
__device__ __forceinline__ float pooled_mean(const float* incoming, size_t incoming_stride, const float* history, size_t begin, size_t base, unsigned c) {
    float x = 0.0f;
    #pragma unroll
    for (size_t tap = 0; tap < 4; ++tap) {
        const size_t pos = begin + tap;
        x += pos < base ? history[(pos % RING) * COLUMNS + c] : incoming[(pos - base) * incoming_stride + c];
    }
    return x / 4.0f;
}

// One workgroup of 128 threads per block completed by the span.
__global__ void __launch_bounds__(COLUMNS) pool_kernel(const float* incoming, size_t incoming_stride, const float* history, const float* norm, size_t pool,
                                                       size_t base, float* blocks) {
    __shared__ float values[256], sums[256];
    const size_t block = base / 4 + blockIdx.x, begin = block * 4;
    const unsigned c = threadIdx.x;
    blocks[c * pool + block] = normalized(pooled_mean(incoming, incoming_stride, history, begin, base, c), norm, COLUMNS, begin, values, sums);
}

__global__ void __launch_bounds__(256) save_history_kernel(const float* incoming, size_t incoming_stride, size_t base, size_t steps, float* history) {
    const size_t i = threadIdx.x + size_t(blockIdx.x) * 256, kept = steps < 4 ? steps : 4;
    if (i >= kept * COLUMNS) return;
    const size_t token = steps - kept + i / COLUMNS;
    history[((base + token) % RING) * COLUMNS + i % COLUMNS] = incoming[token * incoming_stride + i % COLUMNS];
}

__device__ __forceinline__ float positive_sum(const float (&dot)[HEADS]) {
    float total = fmaxf(dot[0], 0.0f) + fmaxf(dot[1], 0.0f);
    total += fmaxf(dot[2], 0.0f);
    total += fmaxf(dot[3], 0.0f);
    return total;
}

// ---- scores of a short span: a lane per block, a wave per head, T rows per lane ----------------------------------------------
// The chains of a block's four heads run in four waves of the workgroup (the same 64 blocks, the keys read by each: the second
// to fourth find them in the cache), so a compute unit holds four times the waves to hide the loads behind; the four sums meet
// in LDS and are added in head order.  The queries sit in LDS as [row][head][column]: a wave-uniform read a column.
// maxima (may be null): of every row the highest score of each sixteen neighbouring blocks, for the selection to begin with.
constexpr int SIXTEENS = 16, MAXIMA_ROW = 65536 / SIXTEENS + 64, MAXIMA_ROWS = 8;
template<int T>
__global__ void __launch_bounds__(64 * HEADS) scores_rows_kernel(const float* __restrict__ queries, size_t query_stride, const float* __restrict__ blocks,
                                                                size_t pool, size_t base, const uint32_t* dynamic, unsigned steps, float* __restrict__ scores,
                                                                uint32_t* __restrict__ maxima) {
    __shared__ float q[T][HEADS][COLUMNS];
    __shared__ float sums[HEADS][T][64];
    if (dynamic) base = *dynamic;
    const size_t most = min((base + steps) / 4, pool), first = size_t(blockIdx.x) * 64;   // the last row's complete blocks
    const unsigned lane = threadIdx.x % 64, head = threadIdx.x / 64;
    if (most <= KEEP || first >= most) return;
    for (unsigned i = threadIdx.x; i < T * HEADS * COLUMNS; i += 64 * HEADS) {
        const unsigned row = i / (HEADS * COLUMNS);
        q[row][i / COLUMNS % HEADS][i % COLUMNS] = row < steps ? queries[row * query_stride + i % (HEADS * COLUMNS)] : 0.0f;
    }
    __syncthreads();
    const float* column = blocks + min(first + lane, pool - 1);
    float dot[T] = {};
    #pragma unroll 1
    for (unsigned c0 = 0; c0 < COLUMNS; c0 += 16) {
        float key[16];
        #pragma unroll
        for (unsigned j = 0; j < 16; ++j) key[j] = column[size_t(c0 + j) * pool];
        #pragma unroll
        for (unsigned j = 0; j < 16; ++j)
            #pragma unroll
            for (int row = 0; row < T; ++row) dot[row] = fmaf(key[j], q[row][head][c0 + j], dot[row]);
    }
    #pragma unroll
    for (int row = 0; row < T; ++row) sums[head][row][lane] = dot[row];
    __syncthreads();
    for (unsigned row = head; row < unsigned(T); row += HEADS) {
        const size_t complete = (base + row + 1) / 4;
        const float four[HEADS] = {sums[0][row][lane], sums[1][row][lane], sums[2][row][lane], sums[3][row][lane]};
        const bool counts = row < steps && complete > KEEP && first + lane < min(complete, pool);
        const float score = positive_sum(four);
        if (counts) scores[row * pool + first + lane] = score;
        if (maxima && row < steps) {
            uint32_t top = counts ? __float_as_uint(score) : 0u;       // (sums of max(., 0): their bits order as they do)
            top = max(top, from_lane<0x111>(0u, top)); top = max(top, from_lane<0x112>(0u, top));
            top = max(top, from_lane<0x114>(0u, top)); top = max(top, from_lane<0x118>(0u, top));          // (lane 15 of every sixteen: all of them)
            if (lane % SIXTEENS == SIXTEENS - 1) maxima[row * MAXIMA_ROW + (first + lane) / SIXTEENS] = top;
        }
    }
}

// ---- scores of a prefill chunk: 32 rows x 256 blocks per workgroup ---------------------------------------------------------
// Eight waves; a lane owns 4 neighbouring blocks, a wave 4 rows, so a thread carries 4 x 4 x 4 chains.  Sixteen columns of
// keys [column][block] and queries [column][row * 4 + head] are staged at a time: the key read is 16 bytes a lane without
// bank conflicts, the query read is wave-uniform.  The next sixteen columns travel from global memory into registers while
// the current ones are multiplied.
constexpr int TILE_ROWS = 32, TILE_BLOCKS = 256, TILE_COLUMNS = 16, TILE_THREADS = 512, QUERY_PITCH = TILE_ROWS * HEADS + 4;
// One tile of 32 rows x 256 blocks (every thread of the workgroup calls it; `most`: the complete blocks of the tile's last row).
__device__ __forceinline__ void scores_tile(const float* __restrict__ queries, size_t query_stride, const float* __restrict__ blocks, size_t pool,
                                            size_t base, size_t steps, float* __restrict__ scores, size_t first_row, size_t first_block,
                                            float (&keys)[2][TILE_COLUMNS][TILE_BLOCKS], float (&query)[2][TILE_COLUMNS][QUERY_PITCH]) {
    const unsigned t = threadIdx.x, lane = t % 64, wave = t / 64;
    constexpr int KEY_LOADS = TILE_COLUMNS * TILE_BLOCKS / TILE_THREADS, QUERY_LOADS = TILE_COLUMNS * TILE_ROWS * HEADS / TILE_THREADS;
    float key_next[KEY_LOADS], query_next[QUERY_LOADS];
    const size_t key_block = min(first_block + t % TILE_BLOCKS, pool - 1);
    const auto fetch = [&](unsigned k) {
        #pragma unroll
        for (int j = 0; j < KEY_LOADS; ++j) key_next[j] = blocks[size_t(k + t / TILE_BLOCKS + j * (TILE_THREADS / TILE_BLOCKS)) * pool + key_block];
        #pragma unroll
        for (int j = 0; j < QUERY_LOADS; ++j) {
            const unsigned i = t + j * TILE_THREADS, c = i % TILE_COLUMNS, slot = i / TILE_COLUMNS;      // slot = row * 4 + head
            const size_t row = first_row + slot / HEADS;
            query_next[j] = row < steps ? queries[row * query_stride + (slot % HEADS) * COLUMNS + k + c] : 0.0f;
        }
    };
    const auto place = [&](int buffer) {
        #pragma unroll
        for (int j = 0; j < KEY_LOADS; ++j) keys[buffer][t / TILE_BLOCKS + j * (TILE_THREADS / TILE_BLOCKS)][t % TILE_BLOCKS] = key_next[j];
        #pragma unroll
        for (int j = 0; j < QUERY_LOADS; ++j) {
            const unsigned i = t + j * TILE_THREADS;
            query[buffer][i % TILE_COLUMNS][i / TILE_COLUMNS] = query_next[j];
        }
    };
    float sums[4][HEADS][4] = {};   // row, head, block
    fetch(0);
    place(0);
    __syncthreads();
    #pragma unroll 1
    for (unsigned k = 0; k < COLUMNS; k += TILE_COLUMNS) {
        const int buffer = (k / TILE_COLUMNS) & 1;
        if (k + TILE_COLUMNS < COLUMNS) fetch(k + TILE_COLUMNS);
        #pragma unroll 2
        for (unsigned c = 0; c < TILE_COLUMNS; ++c) {
            const float4 four = *reinterpret_cast<const float4*>(&keys[buffer][c][lane * 4]);
            const float key[4] = {four.x, four.y, four.z, four.w};
            #pragma unroll
            for (unsigned i = 0; i < 4; ++i) {
                const float4 heads = *reinterpret_cast<const float4*>(&query[buffer][c][(wave * 4 + i) * HEADS]);
                const float qh[HEADS] = {heads.x, heads.y, heads.z, heads.w};
                #pragma unroll
                for (unsigned h = 0; h < HEADS; ++h) {
                    #pragma unroll
                    for (unsigned b = 0; b < 4; ++b) sums[i][h][b] = fmaf(key[b], qh[h], sums[i][h][b]);
                }
            }
        }
        if (k + TILE_COLUMNS < COLUMNS) place(buffer ^ 1);      // the other buffer was last read before the barrier below, an iteration ago
        __syncthreads();
    }
    #pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
        const size_t row = first_row + wave * 4 + i, complete = min((base + row + 1) / 4, pool);
        if (row >= steps || complete <= KEEP) continue;
        #pragma unroll
        for (unsigned b = 0; b < 4; ++b) {
            const size_t block = first_block + lane * 4 + b;
            const float dot[HEADS] = {sums[i][0][b], sums[i][1][b], sums[i][2][b], sums[i][3][b]};
            if (block < complete) scores[row * pool + block] = positive_sum(dot);
        }
    }
}

// ONLY = false: a workgroup per tile.  ONLY = true (behind the interval selection): the tiles of the rows it left undecided, which
// only[row] marks and only[gate] counts; a launch has fewer workgroups than tiles of blocks, each takes every gridDim.x-th, and
// every workgroup leaves at once when no row is marked.
template<bool ONLY>
__global__ void __launch_bounds__(TILE_THREADS) scores_tiled_kernel(const float* __restrict__ queries, size_t query_stride,
                                                                    const float* __restrict__ blocks, size_t pool, size_t base, size_t steps,
                                                                    float* __restrict__ scores, const uint32_t* __restrict__ only, unsigned gate) {
    __shared__ __align__(16) float keys[2][TILE_COLUMNS][TILE_BLOCKS];
    __shared__ __align__(16) float query[2][TILE_COLUMNS][QUERY_PITCH];
    const size_t first_row = size_t(blockIdx.y) * TILE_ROWS;
    const size_t most = min((base + min(steps, first_row + TILE_ROWS)) / 4, pool);        // complete blocks of the tile's last row
    if (most <= KEEP) return;
    if (ONLY) {
        if (!only[gate]) return;
        bool any = false;
        for (size_t r = first_row; r < min(steps, first_row + TILE_ROWS); ++r) any |= only[r] != 0;
        if (!any) return;
        for (size_t first_block = size_t(blockIdx.x) * TILE_BLOCKS; first_block < most; first_block += size_t(gridDim.x) * TILE_BLOCKS)
            scores_tile(queries, query_stride, blocks, pool, base, steps, scores, first_row, first_block, keys, query);
    } else {
        const size_t first_block = size_t(blockIdx.x) * TILE_BLOCKS;
        if (first_block < most) scores_tile(queries, query_stride, blocks, pool, base, steps, scores, first_row, first_block, keys, query);
    }
}

// ---- the selection ----------------------------------------------------------------------------------------------------------
constexpr int SELECT_THREADS = CHOICE_THREADS, SELECT_WAVES = CHOICE_WAVES, LDS_RUNS = 31, LIST_RUNS = 2, LIST = LIST_RUNS * SELECT_THREADS, SIXTEENS_MOST = 1024;

// Exclusive prefix of `value` over the workgroup in thread order, and the workgroup's sum.
__device__ __forceinline__ uint32_t group_scan(uint32_t value, uint32_t* wave_sums, uint32_t& total) {
    const unsigned lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const uint32_t inclusive = wave_prefix(value);
    __syncthreads();
    if (lane == 63) wave_sums[wave] = inclusive;
    __syncthreads();
    uint32_t before = 0, sum = 0;
    #pragma unroll
    for (int w = 0; w < SELECT_WAVES; ++w) {
        const uint32_t c = wave_sums[w];
        before += unsigned(w) < wave ? c : 0u;
        sum += c;
    }
    total = sum;
    return before + inclusive - value;
}

// What the selection keeps between its steps, in LDS.
struct SelectShared {
    union {
        struct {
            uint32_t bins[SELECT_WAVES * 256];              // a histogram per wave; at other times the (run, wave) counts or the sample's histogram
            uint2 list[LIST_RUNS * SELECT_THREADS];         // (score bits, block) of the values that reach the guess
        };
        struct {
            ChoiceShared choice;
            uint32_t names[SIXTEENS_MOST];                  // of the sixteens that reach the bound
        };
    };
    uint32_t wave_sums[SELECT_WAVES], threshold, remaining;
};

// The choice itself over values a thread holds as (run i, thread t) in ascending block order: each_run(body) calls
// body(i, bits, valid) for the thread's value of every run, block_of(i) names its block.  Values below `guess` are known
// not to be among the 512 highest; should fewer than 512 be left, the guess is dropped.  Four 8-bit radix passes find the 512th
// highest value (a per-wave histogram; the first pass, where nearly all values share the digit, adds once per digit by a
// ballot), then one ordered pass gives every kept value its slot: ballots rank the lanes of a wave, a scan over the (run, wave)
// counts ranks the waves, and the values equal to the 512th are taken from the earliest blocks on.
template<class Each, class BlockOf>
__device__ __forceinline__ void choose_blocks(SelectShared& sh, Each each_run, BlockOf block_of, unsigned runs, unsigned most_runs, uint32_t guess,
                                              float* out) {
    const unsigned t = threadIdx.x, lane = t % 64, wave = t / 64;
    uint32_t prefix = 0, wanted = KEEP, mask = 0;
    uint32_t* own = sh.bins + wave * 256;
    #pragma unroll 1
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (unsigned i = t; i < SELECT_WAVES * 256; i += SELECT_THREADS) sh.bins[i] = 0;
        __syncthreads();
        each_run([&](unsigned, uint32_t bits, bool valid) {
            const bool live = valid && bits >= guess && (bits & mask) == prefix;
            const uint32_t digit = (bits >> shift) & 255u;
            if (shift == 24) {
                uint64_t todo = __ballot(live);
                while (todo) {
                    const int leader = __ffsll(static_cast<long long>(todo)) - 1;
                    const uint32_t d = uint32_t(__builtin_amdgcn_readlane(int(digit), leader));
                    const uint64_t same = __ballot(live && digit == d);
                    if (int(lane) == leader) atomicAdd(own + d, uint32_t(__popcll(same)));
                    todo &= ~same;
                }
            } else if (live) {
                atomicAdd(own + digit, 1u);
            }
        });
        __syncthreads();
        // thread i < 256 holds bin 255 - i: the scan counts the values in higher bins
        const uint32_t bucket = 255u - (t & 255u);
        uint32_t count = 0, every;
        if (t < 256)
            for (int w = 0; w < SELECT_WAVES; ++w) count += sh.bins[w * 256 + bucket];
        const uint32_t above = group_scan(count, sh.wave_sums, every);
        if (shift == 24 && every < KEEP) {                   // the guess was too high: once more, over every value
            guess = 0;
            shift += 8;
            continue;
        }
        if (t < 256 && above < wanted && above + count >= wanted) { sh.threshold = prefix | (bucket << shift); sh.remaining = wanted - above; }
        __syncthreads();
        prefix = sh.threshold; wanted = sh.remaining;
        mask |= 255u << shift;
    }
    // Kept: every value above `prefix` and the first `wanted` equal to it, in block order.
    uint32_t* greater = sh.bins;
    uint32_t* equal = sh.bins + most_runs * SELECT_WAVES;
    each_run([&](unsigned i, uint32_t bits, bool valid) {
        const uint64_t above = __ballot(valid && bits > prefix), same = __ballot(valid && bits == prefix);
        if (lane == 0) { greater[i * SELECT_WAVES + wave] = uint32_t(__popcll(above)); equal[i * SELECT_WAVES + wave] = uint32_t(__popcll(same)); }
    });
    __syncthreads();
    const unsigned entries = runs * SELECT_WAVES;           // at most 1024: one per thread
    const uint32_t g = t < entries ? greater[t] : 0u, e = t < entries ? equal[t] : 0u;
    uint32_t every;
    const uint32_t greater_before = group_scan(g, sh.wave_sums, every);
    const uint32_t equal_before = group_scan(e, sh.wave_sums, every);
    if (t < entries) { greater[t] = greater_before; equal[t] = equal_before; }
    __syncthreads();
    const uint64_t below = (uint64_t(1) << lane) - 1;
    each_run([&](unsigned i, uint32_t bits, bool valid) {
        const bool above = valid && bits > prefix, same = valid && bits == prefix;
        const uint64_t above_mask = __ballot(above), same_mask = __ballot(same);
        if (!above && !same) return;
        const uint32_t equal_seen = equal[i * SELECT_WAVES + wave] + uint32_t(__popcll(same_mask & below));
        if (same && equal_seen >= wanted) return;
        const size_t at = size_t(greater[i * SELECT_WAVES + wave] + uint32_t(__popcll(above_mask & below)) + min(equal_seen, wanted)) * 4;
        const size_t block = block_of(i);
        #pragma unroll
        for (size_t tap = 0; tap < 4; ++tap) out[at + tap] = float(block * 4 + tap);
    });
}

// A short span's rows (a decode step, a verification span) would leave all but a few compute units idle while one workgroup a row
// sweeps 60K values.  Their scores' kernel leaves the highest score of each sixteen neighbouring blocks: the 512th highest of those is reached by 512
// scores, and little more (some 550 of 60K in no order), so it is a bound that only its own sixteens have to be read for.  Where neighbours are alike whole sixteens reach it, up to 16K scores: more
// than the list holds, they are read again for each step of the choice (a row of 32768 blocks alike over sixteen 17.5 us; swept, with the attempt, 38; not alike 12.9).
// Writes the row's entries; false, and nothing written: many scores are equal, the row's workgroup sweeps the row itself, as it does below 8192 blocks, whose sixteens are
// fewer than the bound is asked of (a decode row's whole stage at 20K tokens 40.0 us, at 33K 34.4).  (Thirty-two workgroups a row that each found
// a bound from the same sample of it and listed their stretch took a launch of 10 us; a decode row's whole stage at 242K tokens 52.4 us with them, 38.7 now.)
constexpr int MAXIMA_EACH = (65536 / SIXTEENS + SELECT_THREADS) / SELECT_THREADS;
__device__ __forceinline__ bool select_by_maxima(SelectShared& sh, const uint32_t (&top)[MAXIMA_EACH], const float* row, uint32_t complete, float* out) {
    const unsigned t = threadIdx.x, count = (complete + SIXTEENS - 1) / SIXTEENS;
    constexpr uint32_t NONE = 0xffffffffu;                  // (no score's bits)
    uint32_t valid[MAXIMA_EACH];
    #pragma unroll
    for (int i = 0; i < MAXIMA_EACH; ++i) valid[i] = i * SELECT_THREADS + t < count ? top[i] : NONE;
    uint32_t high;
    const uint32_t bound = bound_by_maxima(sh.choice, valid, NONE, KEEP, SIXTEENS_MOST, high);
    if (!bound) return false;
    // the sixteens that reach it are named, then their scores that do are listed
    #pragma unroll
    for (int i = 0; i < MAXIMA_EACH; ++i)
        if (valid[i] != NONE && valid[i] >= bound) sh.names[atomicAdd(&sh.choice.named, 1u)] = i * SELECT_THREADS + t;
    __syncthreads();
    const unsigned named = sh.choice.named;
    const auto read = [&](auto enough, auto use) {
        constexpr int AT_ONCE = 4;                          // reads in flight
        #pragma unroll 1
        for (unsigned base = 0; base < named && !enough(); base += AT_ONCE * (SELECT_THREADS / SIXTEENS)) {
            uint32_t block[AT_ONCE], bits[AT_ONCE];
            #pragma unroll
            for (int i = 0; i < AT_ONCE; ++i) {
                const unsigned name = base + i * (SELECT_THREADS / SIXTEENS) + t / SIXTEENS;
                block[i] = name < named ? sh.names[name] * SIXTEENS + t % SIXTEENS : complete;
                bits[i] = __float_as_uint(row[min(block[i], complete - 1)]);
            }
            #pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                if (block[i] < complete && bits[i] >= bound) use(bits[i], block[i]);
        }
    };
    // (neighbours that are alike: most of what was named, which the list does not hold; a wave that sees it full adds no more)
    read([&] { return *const_cast<volatile uint32_t*>(&sh.choice.listed) > unsigned(CHOICE_LIST); }, [&](uint32_t value, uint32_t name) {
        const uint32_t at = atomicAdd(&sh.choice.listed, 1u);
        if (at < unsigned(CHOICE_LIST)) sh.choice.list[at] = make_uint2(value, name);
    });
    __syncthreads();
    const auto emit = [&](size_t slot, uint32_t block) {
        #pragma unroll
        for (size_t tap = 0; tap < 4; ++tap) out[slot * 4 + tap] = float(size_t(block) * 4 + tap);
    };
    const unsigned n = sh.choice.listed;
    if (n > unsigned(CHOICE_LIST)) {
        choose(sh.choice, KEEP, bound, high, [&](auto use) { read([] { return false; }, use); }, emit);
        return true;
    }
    const uint2 own = sh.choice.list[t];
    choose(sh.choice, KEEP, bound, high, [&](auto use) { if (t < n) use(own.x, own.y); }, emit);
    return true;
}

// One workgroup per row; block i * 1024 + t is thread t's value i.  The row is read once and stays on the chip: its first
// LDS_RUNS runs of 1024 values in LDS (as many as the row has: the launch sizes the array), the runs beyond, for the longest
// rows, in REGS registers a thread.
//
// A long row is thinned first, since every sweep over 64 values a thread costs about as much as all the rest: the R-th
// highest of a sample of four values a thread (spread over the runs in LDS; R: one and a half times the sample's share of 512, and
// a margin), found to 24 bits by two 4096-bin histograms, is a guess below the 512th highest value of the row.  Two light sweeps count and list, in block order, the values that reach the guess; when they are
// at least 512 and fit the list, the choice runs over the list alone, otherwise over the whole row.
static_assert(sizeof(SelectShared) + LDS_RUNS * SELECT_THREADS * 4 <= 160 * 1024, "a compute unit's LDS");
template<int REGS>
__global__ void __launch_bounds__(SELECT_THREADS) select_kernel(const float* __restrict__ scores, size_t pool, size_t base, const uint32_t* dynamic,
                                                                size_t selected, unsigned held_runs, float* __restrict__ indices,
                                                                float* __restrict__ counts, const uint32_t* __restrict__ maxima,
                                                                const uint32_t* __restrict__ only) {
    extern __shared__ uint32_t held[];                       // [run][1024]
    if (only && !only[blockIdx.x]) return;
    __shared__ SelectShared sh;
    // (the maxima are asked for beside the position; those past the row's are not used)
    uint32_t tops[MAXIMA_EACH];
    if (maxima)
        #pragma unroll
        for (int i = 0; i < MAXIMA_EACH; ++i) tops[i] = maxima[size_t(blockIdx.x) * MAXIMA_ROW + min(i * SELECT_THREADS + threadIdx.x, unsigned(MAXIMA_ROW) - 1)];
    if (dynamic) base = *dynamic;
    const size_t token = blockIdx.x, position = base + token, complete = (position + 1) / 4;
    const unsigned t = threadIdx.x, lane = t % 64, wave = t / 64;
    float* out = indices + token * selected;
    if (position + 1 > 4 * pool || complete > size_t(held_runs + REGS) * SELECT_THREADS) {   // a position this key pool (or this launch) cannot hold
        if (t == 0) counts[token] = 0.0f;
        return;
    }
    if (complete <= KEEP) {
        for (size_t i = t; i <= position; i += SELECT_THREADS) out[i] = float(i);
        if (t == 0) counts[token] = float(position + 1);
        return;
    }
    const float* row = scores + token * pool;
    const unsigned runs = unsigned((complete + SELECT_THREADS - 1) / SELECT_THREADS), lds_runs = min(runs, held_runs);
    uint32_t values[REGS ? REGS : 1];
    uint32_t guess = 0;
    bool listed = false;
    uint32_t list_count = 0;
    bool done = false;
    if (maxima && complete >= size_t(KEEP) * SIXTEENS) {
        done = select_by_maxima(sh, tops, row, uint32_t(complete), out);
        __syncthreads();
    }
    if (!done) {
    #pragma unroll 8
    for (unsigned i = 0; i < lds_runs; ++i) {
        const size_t block = size_t(i) * SELECT_THREADS + t;
        held[i * SELECT_THREADS + t] = block < complete ? __float_as_uint(row[block]) : 0u;
    }
    if constexpr (REGS > 0) {
        #pragma unroll
        for (int j = 0; j < REGS; ++j) {
            const size_t block = size_t(LDS_RUNS + j) * SELECT_THREADS + t;
            values[j] = block < complete ? __float_as_uint(row[block]) : 0u;
        }
    }
    // body(run, bits, valid) for every run of the row, in run order (every thread reads back only what it wrote)
    const auto each_run = [&](auto body) {
        unsigned i = 0;
        for (; i + 4 <= lds_runs; i += 4) {                  // four reads in flight at a time
            uint32_t four[4];
            #pragma unroll
            for (unsigned j = 0; j < 4; ++j) four[j] = held[(i + j) * SELECT_THREADS + t];
            #pragma unroll
            for (unsigned j = 0; j < 4; ++j) body(i + j, four[j], size_t(i + j) * SELECT_THREADS + t < complete);
        }
        for (; i < lds_runs; ++i) body(i, held[i * SELECT_THREADS + t], size_t(i) * SELECT_THREADS + t < complete);
        if constexpr (REGS > 0) {
            unsigned again = t;
            asm volatile("" : "+v"(again));                  // (the runs' places are formed again: kept from the loads on they are more registers than there are)
            #pragma unroll
            for (int j = 0; j < REGS; ++j)
                if (unsigned(LDS_RUNS + j) < runs) body(unsigned(LDS_RUNS + j), values[j], size_t(LDS_RUNS + j) * SELECT_THREADS + again < complete);
        }
    };
    if (runs >= 8) {
        constexpr unsigned SAMPLES = 4;                      // values a thread gives to the sample
        uint32_t sample[SAMPLES];
        bool sampled[SAMPLES];
        #pragma unroll
        for (unsigned k = 0; k < SAMPLES; ++k) {
            const unsigned run = (t + 7 * k) % lds_runs;
            sampled[k] = size_t(run) * SELECT_THREADS + t < complete;
            sample[k] = held[run * SELECT_THREADS + t];
        }
        uint32_t rank = uint32_t(3 * size_t(KEEP) * SAMPLES * SELECT_THREADS / (2 * complete)) + 16;
        #pragma unroll 1
        for (int shift = 20; shift >= 8; shift -= 12) {     // the sample's rank-th highest value to 24 bits: 12 bits a level
            for (unsigned i = t; i < SELECT_WAVES * 256; i += SELECT_THREADS) sh.bins[i] = 0;
            if (t == 0) { sh.threshold = guess; sh.remaining = rank; }
            __syncthreads();
            #pragma unroll
            for (unsigned k = 0; k < SAMPLES; ++k)
                if (sampled[k] && (shift == 20 || (sample[k] >> 20) == (guess >> 20))) atomicAdd(sh.bins + ((sample[k] >> shift) & 4095u), 1u);
            __syncthreads();
            uint32_t four[4], sum = 0, every;
            #pragma unroll
            for (unsigned j = 0; j < 4; ++j) { four[j] = sh.bins[4095 - 4 * t - j]; sum += four[j]; }
            uint32_t above = group_scan(sum, sh.wave_sums, every);
            #pragma unroll
            for (unsigned j = 0; j < 4; ++j) {
                if (above < rank && above + four[j] >= rank) { sh.threshold = guess | ((4095 - 4 * t - j) << shift); sh.remaining = rank - above; }
                above += four[j];
            }
            __syncthreads();
            guess = sh.threshold; rank = sh.remaining;
            __syncthreads();
        }
        // how many values reach the guess, per (run, wave) in block order
        uint32_t* reach = sh.bins;
        each_run([&](unsigned i, uint32_t bits, bool valid) {
            const uint64_t reaching = __ballot(valid && bits >= guess);
            if (lane == 0) reach[i * SELECT_WAVES + wave] = uint32_t(__popcll(reaching));
        });
        __syncthreads();
        const unsigned entries = runs * SELECT_WAVES;
        const uint32_t mine = t < entries ? reach[t] : 0u;
        const uint32_t before = group_scan(mine, sh.wave_sums, list_count);
        if (t < entries) reach[t] = before;
        __syncthreads();
        if (list_count < KEEP) guess = 0;                    // too high a guess: the whole row, every value
        listed = list_count >= KEEP && list_count <= LIST;
        if (listed) {
            const uint64_t below = (uint64_t(1) << lane) - 1;
            each_run([&](unsigned i, uint32_t bits, bool valid) {
                const bool reaches = valid && bits >= guess;
                const uint64_t reaching = __ballot(reaches);
                unsigned again = t;
                asm volatile("" : "+v"(again));
                if (reaches) sh.list[reach[i * SELECT_WAVES + wave] + uint32_t(__popcll(reaching & below))] = make_uint2(bits, i * SELECT_THREADS + again);
            });
        }
        __syncthreads();
    }
    if (listed) {
        uint2 mine[LIST_RUNS];
        #pragma unroll
        for (int j = 0; j < LIST_RUNS; ++j) mine[j] = unsigned(j) * SELECT_THREADS + t < list_count ? sh.list[j * SELECT_THREADS + t] : make_uint2(0u, 0u);
        const unsigned list_runs = (list_count + SELECT_THREADS - 1) / SELECT_THREADS;
        choose_blocks(sh, [&](auto body) {
            #pragma unroll
            for (int j = 0; j < LIST_RUNS; ++j)
                if (unsigned(j) < list_runs) body(unsigned(j), mine[j].x, unsigned(j) * SELECT_THREADS + t < list_count);
        }, [&](unsigned j) { return size_t(j == 0 ? mine[0].y : mine[1].y); }, list_runs, LIST_RUNS, 0u, out);
    } else {
        choose_blocks(sh, each_run, [&](unsigned i) {
            unsigned again = t;
            asm volatile("" : "+v"(again));
            return size_t(i) * SELECT_THREADS + again;
        }, runs, LDS_RUNS + REGS, guess, out);
    }
    }
    const size_t head = size_t(KEEP) * 4;
    for (size_t i = t; complete * 4 + i <= position; i += SELECT_THREADS) out[head + i] = float(complete * 4 + i);
    if (t == 0) counts[token] = float(head + position + 1 - complete * 4);
}

template<int REGS>
void launch_select(Device& d, const float* scores, size_t pool, size_t base, const uint32_t* dynamic, size_t selected, size_t most, unsigned rows,
                   float* indices, float* counts, const uint32_t* maxima, const uint32_t* only = nullptr) {
    const unsigned held_runs = unsigned(std::min<size_t>((most + SELECT_THREADS - 1) / SELECT_THREADS, LDS_RUNS));
    const size_t shared = size_t(std::max(held_runs, 1u)) * SELECT_THREADS * 4;
    if (shared > 48 * 1024) raise_shared_limit(d, reinterpret_cast<const void*>(&select_kernel<REGS>), LDS_RUNS * SELECT_THREADS * 4);
    select_kernel<REGS><<<rows, SELECT_THREADS, shared, d.stream>>>(scores, pool, base, dynamic, selected, held_runs, indices, counts, maxima, only);
}

// ---- a decode or verification pass's inputs in one launch --------------------------------------------------------------
// The reference's qsa_normalize_rows (gpu/qsa_decode.hpp:86-111): blockIdx.y = row; blockIdx.x = a query head (normalised and turned
// into `queries`), then a K/V head (the key normalised and turned, key and value rows encoded into the cache at the row's
// position), then the four index-query heads (in place), then one workgroup that pools the index keys of all rows in turn
// (a row completes a block from the ring the rows before it wrote).  Positions and rope positions are read on the device.
struct StageArgs {
    float* projections;            // row r at r * stride: heads x [query 256 | gate 256], kv x key 256, kv x value 256, 4 x index query 128, index key 128
    size_t stride;
    const float *q_norm, *k_norm, *index_q_norm, *index_k_norm;
    unsigned heads, kv_heads, steps;
    const uint32_t *positions, *ropes;   // device-resident positions of the rows (stage_prepare_kernel)
    size_t base;
    uint8_t* pages;
    unsigned page_tokens, row_bytes;
    const int32_t* page_table;
    size_t page_count;
    size_t context;
    float* queries;                // [steps][heads][256]
    float *blocks, *history;
    size_t pool;
};
__global__ void __launch_bounds__(256) stage_prepare_kernel(StageArgs a) {
    __shared__ float values[256], sums[256];
    __shared__ __align__(16) float key[256];
    const unsigned block = blockIdx.x, c = threadIdx.x;
    const size_t row = blockIdx.y, pos = a.positions[row], rope = a.ropes[row];
    float* own = a.projections + row * a.stride;
    const size_t keys_at = size_t(a.heads) * 512, values_at = keys_at + size_t(a.kv_heads) * 256, index_at = keys_at + size_t(a.kv_heads) * 512;
    if (block < a.heads) {
        a.queries[(row * a.heads + block) * 256 + c] = normalized(own[size_t(block) * 512 + c], a.q_norm, 256, rope, values, sums);
    } else if (block < a.heads + a.kv_heads) {
        const unsigned head = block - a.heads;
        key[c] = normalized(own[keys_at + head * 256 + c], a.k_norm, 256, rope, values, sums);
        __syncthreads();
        if (pos >= a.context || c >= 128) return;           // a position outside the cache writes no row; two waves encode
        const long long entry = a.page_table ? a.page_table[pos / a.page_tokens] : 0;
        if (entry < 0 || size_t(entry) >= a.page_count) return;   // nor does a table entry that names no page of the pool
        const size_t page = size_t(entry), in_page = a.page_table ? pos % a.page_tokens : pos;
        const bool is_value = c >= 64;
        const unsigned quad = c % 64;                       // four columns a thread: a wave holds the row, 8 lanes a 32-column block
        uint8_t* target = a.pages + ((page * 2 * a.kv_heads + (is_value ? a.kv_heads : 0) + head) * a.page_tokens + in_page) * a.row_bytes;
        const float* from = is_value ? own + values_at + head * 256 + 4 * quad : key + 4 * quad;
        const float x[4] = {from[0], from[1], from[2], from[3]};
        kv_store_quad(target, quad, 256, a.row_bytes != 512, x, true);
    } else if (block < a.heads + a.kv_heads + HEADS) {
        const unsigned head = block - a.heads - a.kv_heads;
        float* vector = own + index_at + head * COLUMNS;
        const float value = normalized(c < COLUMNS ? vector[c] : 0.0f, a.index_q_norm, COLUMNS, rope, values, sums);
        if (c < COLUMNS) vector[c] = value;
    } else if (row == 0) {
        for (size_t r = 0; r < a.steps; ++r) {
            const size_t at = a.positions[r];
            if (c < COLUMNS) a.history[(at % RING) * COLUMNS + c] = a.projections[r * a.stride + index_at + HEADS * COLUMNS + c];
            if ((at + 1) % 4 == 0 && at / 4 < a.pool) {
                float x = 0.0f;
                if (c < COLUMNS) {
                    #pragma unroll
                    for (size_t tap = 0; tap < 4; ++tap) x += a.history[((at - 3 + tap) % RING) * COLUMNS + c];
                    x /= 4.0f;
                }
                const float value = normalized(x, a.index_k_norm, COLUMNS, size_t(a.ropes[r]) - 3, values, sums);
                if (c < COLUMNS) a.blocks[c * a.pool + at / 4] = value;
            }
        }
    }
}

// The same vectors of a prompt chunk's rows (row r is at base + r), a wave a vector at a time: the sum of squares is formed lane by lane
// in the halving tree's order, so there is no barrier, and a row's angles are formed once for the vectors a wave has, which
// are all asked for before the first is summed.  Measured, 1024 rows of 24 + 2 + 4 vectors, eight a wave: 22 us (57 MB read, 29 written) where a workgroup a
// vector takes 43 (an angle's power, cosine and sine are a third of a vector's instructions, its barriers most of its time).
constexpr int STAGE_WAVES = 4;
__device__ __forceinline__ float tree_of_four(const float (&x)[4], bool wide) {
    #pragma clang fp contract(off)
    const float first = x[0] * x[0], second = x[1] * x[1];
    float sum = wide ? (first + x[2] * x[2]) + (second + x[3] * x[3]) : first + second;
    #pragma unroll
    for (unsigned offset = 32; offset; offset /= 2) sum += __shfl_down(sum, offset);
    return __shfl(sum, 0);
}
template<int STAGE_EACH>
__global__ void __launch_bounds__(64 * STAGE_WAVES) stage_rows_kernel(StageArgs a) {
    __shared__ __align__(16) float keys[STAGE_WAVES][256];
    const unsigned lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), vectors = a.heads + a.kv_heads + HEADS;
    const size_t row = blockIdx.y, pos = a.base + row;
    float* own = a.projections + row * a.stride;
    const size_t keys_at = size_t(a.heads) * 512, values_at = keys_at + size_t(a.kv_heads) * 256, index_at = keys_at + size_t(a.kv_heads) * 512;
    const auto vector_of = [&](int i) { return (blockIdx.x * STAGE_EACH + i) * STAGE_WAVES + wave; };
    const auto place_of = [&](unsigned v) {
        return v < a.heads ? size_t(v) * 512 : v < a.heads + a.kv_heads ? keys_at + size_t(v - a.heads) * 256 : index_at + size_t(v - a.heads - a.kv_heads) * COLUMNS;
    };
    float x[STAGE_EACH][4];
    #pragma unroll
    for (int i = 0; i < STAGE_EACH; ++i) {
        const unsigned v = min(vector_of(i), vectors - 1);
        const float* from = own + place_of(v) + lane;
        x[i][0] = from[0]; x[i][1] = from[64];
        x[i][2] = x[i][3] = 0.0f;
        if (v < a.heads + a.kv_heads) { x[i][2] = from[128]; x[i][3] = from[192]; }
    }
    const float angle = turn_angle(lane, pos), cosine = cosf(angle), sine = sinf(angle);
    #pragma unroll
    for (int i = 0; i < STAGE_EACH; ++i) {
        const unsigned v = vector_of(i);
        if (v >= vectors) return;
        const bool wide = v < a.heads + a.kv_heads;
        const float* norm = (v < a.heads ? a.q_norm : wide ? a.k_norm : a.index_q_norm) + lane;
        const float denominator = sqrtf(tree_of_four(x[i], wide) / float(wide ? 256 : COLUMNS) + 1e-6f);
        float value[4];
        value[0] = x[i][0] * norm[0] / denominator; value[1] = x[i][1] * norm[64] / denominator;
        if (wide) { value[2] = x[i][2] * norm[128] / denominator; value[3] = x[i][3] * norm[192] / denominator; }
        value[0] = turned(value[0], __shfl_xor(value[0], 32), lane, cosine, sine);
        if (v < a.heads) {
            float* to = a.queries + (row * a.heads + v) * 256 + lane;
            to[0] = value[0]; to[64] = value[1]; to[128] = value[2]; to[192] = value[3];
        } else if (!wide) {
            float* to = own + place_of(v) + lane;
            to[0] = value[0]; to[64] = value[1];
        } else {
            const unsigned head = v - a.heads;
            const long long entry = pos >= a.context ? -1 : a.page_table ? a.page_table[pos / a.page_tokens] : 0;
            if (entry < 0 || size_t(entry) >= a.page_count) continue;      // a position outside the cache, or an entry that names no page of the pool, writes no row
            const size_t page = size_t(entry), in_page = a.page_table ? pos % a.page_tokens : pos;
            #pragma unroll
            for (int j = 0; j < 4; ++j) keys[wave][lane + 64 * j] = value[j];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // (the wave's own stretch)
            uint8_t* target = a.pages + ((page * 2 * a.kv_heads + head) * a.page_tokens + in_page) * a.row_bytes;
            const float4 k = *reinterpret_cast<const float4*>(&keys[wave][4 * lane]);
            const float* from = own + values_at + size_t(head) * 256 + 4 * lane;
            const float key4[4] = {k.x, k.y, k.z, k.w}, value4[4] = {from[0], from[1], from[2], from[3]};
            kv_store_quad(target, lane, 256, a.row_bytes != 512, key4, true);
            kv_store_quad(target + size_t(a.kv_heads) * a.page_tokens * a.row_bytes, lane, 256, a.row_bytes != 512, value4, true);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // (read before the next key head's are written)
        }
    }
}

template<int T>
void launch_rows(Device& d, const float* queries, size_t stride, const float* blocks, size_t pool, size_t base, const uint32_t* dynamic, size_t steps,
                 size_t most, float* scores, uint32_t* maxima) {
    timed_launch(d, &scores_rows_kernel<T>, dim3(checked_blocks(most, 64)), dim3(64 * HEADS), 0, queries, stride, blocks, pool, base, dynamic, unsigned(steps), scores, maxima);
}

}  // namespace

namespace sd {
// The maxima of a short span's rows: allocated once per handle, never while a graph is being recorded (sd_graph_begin
// calls this first, so that a recorded pass takes the same path as an eager one).
void select_maxima_reserve(Device& d) {
    if (d.select_maxima) return;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    SD_CHECK(hipStreamIsCapturing(d.stream, &capturing));
    if (capturing == hipStreamCaptureStatusNone) d.select_maxima = static_cast<uint32_t*>(allocate(d, size_t(MAXIMA_ROWS) * MAXIMA_ROW * 4, true));
}
}  // namespace sd

extern "C" {

int sdx_qsa_normalize(void* handle, const float* source, const float* norm, uint64_t rows, uint64_t heads, uint64_t width, uint64_t stride,
                      uint64_t position, float* target) {
    SD_OP_BEGIN
    if (!rows || !heads || (width != 128 && width != 256) || stride < width) throw std::runtime_error("sdx_qsa_normalize: rows and heads >= 1, width 128 or 256, stride >= width");
    const size_t vectors = checked_product({rows, heads});
    op_span(value, source, checked_floats({uint64_t(vectors - 1), stride}) + width * 4, "sdx_qsa_normalize source");
    op_span(value, norm, width * 4, "sdx_qsa_normalize norm");
    op_span(value, target, checked_floats({uint64_t(vectors), width}), "sdx_qsa_normalize target");
    if (position + rows > (uint64_t(1) << 24)) throw std::runtime_error("sdx_qsa_normalize: positions beyond 2^24");
    normalize_kernel<<<checked_blocks(vectors, 1), unsigned(width), 0, value.stream>>>(source, norm, unsigned(heads), unsigned(width), stride, position, target);
    SD_OP_END
}

int sdx_qsa_pool(void* handle, const float* incoming, float* history, const float* norm, uint64_t pool, uint64_t base, uint64_t steps, float* blocks) {
    SD_OP_BEGIN
    if (!steps || !pool || (base + steps) / 4 > pool || base + steps > (uint64_t(1) << 24)) throw std::runtime_error("sdx_qsa_pool: steps >= 1 and (base + steps) / 4 blocks must fit the pool");
    op_span(value, incoming, checked_floats({steps, uint64_t(COLUMNS)}), "sdx_qsa_pool incoming");
    op_span(value, history, size_t(RING) * COLUMNS * 4, "sdx_qsa_pool history");
    op_span(value, norm, COLUMNS * 4, "sdx_qsa_pool norm");
    op_span(value, blocks, checked_floats({pool, uint64_t(COLUMNS)}), "sdx_qsa_pool blocks");
    const size_t completed = (base + steps) / 4 - base / 4;
    if (completed) pool_kernel<<<checked_blocks(completed, 1), COLUMNS, 0, value.stream>>>(incoming, COLUMNS, history, norm, pool, base, blocks);
    save_history_kernel<<<checked_blocks(std::min<size_t>(steps, 4) * COLUMNS), 256, 0, value.stream>>>(incoming, COLUMNS, base, steps, history);
    SD_OP_END
}

int sdx_qsa_index(void* handle, const float* queries, uint64_t query_stride, const float* blocks, uint64_t pool, uint64_t base,
                  const uint32_t* dynamic_base, uint64_t steps, uint64_t selected, float* scores, float* indices, float* counts) {
    SD_OP_BEGIN
    constexpr size_t widest = size_t(64) * SELECT_THREADS;      // complete blocks a row's selection can hold in registers
    if (!steps || !pool || query_stride < HEADS * COLUMNS) throw std::runtime_error("sdx_qsa_index: steps and pool >= 1, query stride >= 512");
    if (pool > widest + 1) throw std::runtime_error("sdx_qsa_index: a pool of more than 65537 blocks (a context beyond 262144)");
    if (!dynamic_base && ((base + steps) / 4 > pool || base + steps > 4 * pool)) throw std::runtime_error("sdx_qsa_index: the span's blocks must fit the pool");
    const size_t needed = dynamic_base ? std::min<size_t>(4 * pool, 2052) : std::min<size_t>(base + steps, 2052);
    if (selected < needed) throw std::runtime_error("sdx_qsa_index: `selected` is smaller than a row's selection can be");
    op_span(value, queries, checked_floats({steps - 1, query_stride}) + HEADS * COLUMNS * 4, "sdx_qsa_index queries");
    op_span(value, blocks, checked_floats({pool, uint64_t(COLUMNS)}), "sdx_qsa_index blocks");
    op_span(value, scores, checked_floats({steps, pool}), "sdx_qsa_index scores");
    op_span(value, indices, checked_floats({steps, selected}), "sdx_qsa_index indices");
    op_span(value, counts, checked_floats({steps}), "sdx_qsa_index counts");
    if (dynamic_base) op_span(value, dynamic_base, 4, "sdx_qsa_index position");
    const size_t most = dynamic_base ? size_t(pool) : size_t((base + steps) / 4);       // complete blocks of the last row, at most
    // a few long rows: their selection begins with the maxima that the scores' kernel leaves (in a small buffer that the handle keeps from the first
    // such call, or from the first sd_graph_begin, on: a call recorded into a graph finds it there)
    uint32_t* maxima = nullptr;
    if (steps <= MAXIMA_ROWS && most >= size_t(KEEP) * SIXTEENS) {
        select_maxima_reserve(value);
        maxima = value.select_maxima;
    }
    if (most > KEEP) {
        if (steps <= 1) launch_rows<1>(value, queries, query_stride, blocks, pool, base, dynamic_base, steps, most, scores, maxima);
        else if (steps <= 2) launch_rows<2>(value, queries, query_stride, blocks, pool, base, dynamic_base, steps, most, scores, maxima);
        else if (steps <= 4) launch_rows<4>(value, queries, query_stride, blocks, pool, base, dynamic_base, steps, most, scores, maxima);
        else if (steps <= 8) launch_rows<8>(value, queries, query_stride, blocks, pool, base, dynamic_base, steps, most, scores, maxima);
        else {
            if (dynamic_base) throw std::runtime_error("sdx_qsa_index: a device-resident position serves spans of up to 8 rows");
            timed_launch(value, &scores_tiled_kernel<false>, dim3(checked_blocks(most, TILE_BLOCKS), checked_blocks(steps, TILE_ROWS)), dim3(TILE_THREADS), 0,
                         queries, query_stride, blocks, pool, base, steps, scores, static_cast<const uint32_t*>(nullptr), 0u);
        }
    }
    const unsigned rows = checked_blocks(steps, 1);
    if (most <= size_t(LDS_RUNS) * SELECT_THREADS) launch_select<0>(value, scores, pool, base, dynamic_base, selected, most, rows, indices, counts, maxima);
    else launch_select<33>(value, scores, pool, base, dynamic_base, selected, most, rows, indices, counts, maxima);
    SD_OP_END
}

uint64_t sdx_qsa_index_interval_scratch(uint64_t steps, uint64_t pool) {
    try { return interval_scratch_bytes(size_t(checked_product({steps, 1})), size_t(checked_product({pool, 1}))); } catch (const std::exception&) { return 0; }
}

int sdx_qsa_index_interval(void* handle, const float* queries, uint64_t query_stride, const float* blocks, uint64_t pool, uint64_t base, uint64_t steps,
                           uint64_t selected, float* scores, float* indices, float* counts, void* scratch, uint64_t scratch_bytes, uint64_t* valid) {
    if (handle && !interval_serves(size_t(base))) {
        // a short context: the exact kernels' time is small, and a sample of it says little
        if (valid) *valid = 0;
        return sdx_qsa_index(handle, queries, query_stride, blocks, pool, base, nullptr, steps, selected, scores, indices, counts);
    }
    SD_OP_BEGIN
    if (!steps || steps > 4096 || !pool || query_stride < HEADS * COLUMNS) throw std::runtime_error("sdx_qsa_index_interval: 1 to 4096 steps, pool >= 1, query stride >= 512");
    if (pool > size_t(64) * SELECT_THREADS + 1) throw std::runtime_error("sdx_qsa_index_interval: a pool of more than 65537 blocks (a context beyond 262144)");
    if ((base + steps) / 4 > pool || base + steps > 4 * pool) throw std::runtime_error("sdx_qsa_index_interval: the span's blocks must fit the pool");
    if (selected < 2052) throw std::runtime_error("sdx_qsa_index_interval: `selected` is smaller than a row's selection can be");
    op_span(value, queries, checked_floats({steps - 1, query_stride}) + HEADS * COLUMNS * 4, "sdx_qsa_index_interval queries");
    op_span(value, blocks, checked_floats({pool, uint64_t(COLUMNS)}), "sdx_qsa_index_interval blocks");
    op_span(value, scores, checked_floats({steps, pool}), "sdx_qsa_index_interval scores");
    op_span(value, indices, checked_floats({steps, selected}), "sdx_qsa_index_interval indices");
    op_span(value, counts, checked_floats({steps}), "sdx_qsa_index_interval counts");
    const size_t need = interval_scratch_bytes(steps, pool);
    if (scratch_bytes < need) throw std::runtime_error("sdx_qsa_index_interval: scratch too small (see sdx_qsa_index_interval_scratch)");
    op_span(value, scratch, need, "sdx_qsa_index_interval scratch");
    unsigned gate = 0;
    const uint32_t* undecided = interval_select(value, queries, query_stride, blocks, pool, base, steps, selected, scores, indices, counts, scratch, valid, &gate);
    // the rows the intervals left undecided, by the exact kernels (workgroups of other rows leave at once)
    const size_t most = size_t((base + steps) / 4);
    scores_tiled_kernel<true><<<dim3(std::min(checked_blocks(most, TILE_BLOCKS), 64u), checked_blocks(steps, TILE_ROWS)), TILE_THREADS, 0, value.stream>>>(
        queries, query_stride, blocks, pool, base, steps, scores, undecided, gate);
    const unsigned rows = checked_blocks(steps, 1);
    if (most <= size_t(LDS_RUNS) * SELECT_THREADS) launch_select<0>(value, scores, pool, base, nullptr, selected, most, rows, indices, counts, nullptr, undecided);
    else launch_select<33>(value, scores, pool, base, nullptr, selected, most, rows, indices, counts, nullptr, undecided);
    SD_OP_END
}

int sdx_qsa_index_interval_undecided(void* handle, const void* scratch, uint64_t steps, uint64_t pool, uint64_t* rows) {
    SD_OP_BEGIN
    if (!rows || !steps || steps > 4096 || !pool) throw std::runtime_error("sdx_qsa_index_interval_undecided: steps, pool, rows");
    op_span(value, scratch, interval_scratch_bytes(steps, pool), "sdx_qsa_index_interval scratch");
    *rows = interval_undecided(value, scratch, steps, pool);
    SD_OP_END
}

uint64_t sdx_qsa_decode_attend_scratch(uint64_t steps, uint64_t heads, uint64_t kv_heads, uint64_t context) {
    try {
        const uint64_t pool = context / 4 + 1;
        return checked_floats({steps, heads * 256 + pool + 2052 + 1}) + 256 + sdx_selected_attention_scratch(steps, kv_heads, 2052);
    } catch (const std::exception&) { return 0; }
}

int sdx_qsa_decode_attend(void* handle, const sdx_qsa_state* state, float* projections, uint64_t stride, uint64_t steps, const uint32_t* positions,
                          const uint32_t* ropes, void* scratch, uint64_t scratch_bytes, float* attended) {
    {
        SD_OP_BEGIN
        if (!state || !state->kv) throw std::runtime_error("sdx_qsa_decode_attend: no state");
        const sdx_kv_pool& kv = *state->kv;
        const uint64_t heads = state->heads, context = state->context, pool = context / 4 + 1;
        if (kv.dim != 256 || !heads || heads % kv.kv_heads || heads / kv.kv_heads > 16 || !steps || steps > 8 || !context || context > (uint64_t(1) << 24) ||
            stride < heads * 512 + uint64_t(kv.kv_heads) * 512 + HEADS * COLUMNS + COLUMNS)
            throw std::runtime_error("sdx_qsa_decode_attend: 1..8 rows of heads x 512 + K/V heads x 512 + 640 projections, K/V rows of 256 columns");
        if (!state->page_table && kv.page_tokens < context) throw std::runtime_error("sdx_qsa_decode_attend: without a page table one page must hold the context");
        if (state->page_table) op_span(value, state->page_table, checked_floats({(context + kv.page_tokens - 1) / kv.page_tokens}), "a page table");
        validate_pool(value, state->kv);        // (the rows are written below: page moves queued so far come first)
        op_span(value, state->blocks, checked_floats({pool, uint64_t(COLUMNS)}), "pooled index keys");
        op_span(value, state->history, size_t(RING) * COLUMNS * 4, "the index history");
        op_span(value, state->q_norm, 256 * 4, "a query norm weight");
        op_span(value, state->k_norm, 256 * 4, "a key norm weight");
        op_span(value, state->index_q_norm, COLUMNS * 4, "an index query norm weight");
        op_span(value, state->index_k_norm, COLUMNS * 4, "an index key norm weight");
        op_span(value, projections, checked_floats({steps - 1, stride}) + (heads * 512 + uint64_t(kv.kv_heads) * 512 + 640) * 4, "projections");
        op_span(value, positions, checked_floats({steps}), "positions");
        op_span(value, ropes, checked_floats({steps}), "rope positions");
        op_span(value, attended, checked_floats({steps, heads, 256}), "an attention output");
        const uint64_t need = sdx_qsa_decode_attend_scratch(steps, heads, kv.kv_heads, context);
        if (!need || scratch_bytes < need) throw std::runtime_error("sdx_qsa_decode_attend: scratch too small (see sdx_qsa_decode_attend_scratch)");
        op_span(value, scratch, need, "stage scratch");
        StageArgs args{};
        args.projections = projections; args.stride = stride;
        args.q_norm = state->q_norm; args.k_norm = state->k_norm; args.index_q_norm = state->index_q_norm; args.index_k_norm = state->index_k_norm;
        args.heads = unsigned(heads); args.kv_heads = kv.kv_heads; args.steps = unsigned(steps); args.positions = positions; args.ropes = ropes;
        args.pages = static_cast<uint8_t*>(kv.pages); args.page_tokens = kv.page_tokens; args.row_bytes = kv.row_bytes; args.page_table = state->page_table; args.page_count = size_t(kv.page_count);
        args.context = context; args.queries = static_cast<float*>(scratch); args.blocks = state->blocks; args.history = state->history; args.pool = pool;
        stage_prepare_kernel<<<dim3(unsigned(heads + kv.kv_heads + HEADS + 1), unsigned(steps)), 256, 0, value.stream>>>(args);
        SD_CHECK(hipGetLastError());
    } catch (const std::exception& e) { ::sd::last_error = e.what(); return -1; }
    }
    // the two stages behind it, on the position the device holds
    const uint64_t heads = state->heads, pool = state->context / 4 + 1;
    float* queries = static_cast<float*>(scratch);
    float* scores = queries + steps * heads * 256;
    float* indices = scores + steps * pool;
    float* counts = indices + steps * 2052;
    uint8_t* partial = reinterpret_cast<uint8_t*>((reinterpret_cast<uintptr_t>(counts + steps) + 255) & ~uintptr_t(255));
    const size_t index_at = heads * 512 + size_t(state->kv->kv_heads) * 512;
    if (sdx_qsa_index(handle, projections + index_at, stride, state->blocks, pool, 0, positions, steps, 2052, scores, indices, counts) < 0) return -1;
    return sdx_selected_attention(handle, state->kv, state->page_table, state->context, 0, positions, indices, 2052, counts, queries, 0, steps, heads, 0.0625f,
                                  projections + 256, 512, stride, attended, 0, partial, sdx_selected_attention_scratch(steps, state->kv->kv_heads, 2052));
}

uint64_t sdx_qsa_prefill_attend_scratch(uint64_t steps, uint64_t heads, uint64_t kv_heads, uint64_t context) {
    try {
        const uint64_t pool = context / 4 + 1;
        const uint64_t first = (checked_floats({steps, heads * 256 + pool + 2052 + 1}) + 255) & ~uint64_t(255);
        const uint64_t partial = (sdx_selected_attention_scratch(steps, kv_heads, 2052) + 255) & ~uint64_t(255);
        return first + partial + sdx_qsa_index_interval_scratch(steps, pool);
    } catch (const std::exception&) { return 0; }
}

int sdx_qsa_prefill_attend(void* handle, const sdx_qsa_state* state, float* projections, uint64_t stride, uint64_t steps, uint64_t base, void* scratch,
                           uint64_t scratch_bytes, uint64_t* valid, float* attended) {
    size_t index_at = 0;
    uint64_t pool = 0;
    {
        SD_OP_BEGIN
        if (!state || !state->kv) throw std::runtime_error("sdx_qsa_prefill_attend: no state");
        const sdx_kv_pool& kv = *state->kv;
        const uint64_t heads = state->heads, context = state->context;
        pool = context / 4 + 1;
        if (kv.dim != 256 || !heads || heads % kv.kv_heads || heads / kv.kv_heads > 16 || !steps || steps > 4096 || !context || context > (uint64_t(1) << 24) ||
            base + steps > context || stride < heads * 512 + uint64_t(kv.kv_heads) * 512 + HEADS * COLUMNS + COLUMNS)
            throw std::runtime_error("sdx_qsa_prefill_attend: 1..4096 rows of heads x 512 + K/V heads x 512 + 640 projections inside the context, K/V rows of 256 columns");
        if (!state->page_table && kv.page_tokens < context) throw std::runtime_error("sdx_qsa_prefill_attend: without a page table one page must hold the context");
        if (state->page_table) op_span(value, state->page_table, checked_floats({(context + kv.page_tokens - 1) / kv.page_tokens}), "a page table");
        validate_pool(value, state->kv);
        op_span(value, state->blocks, checked_floats({pool, uint64_t(COLUMNS)}), "pooled index keys");
        op_span(value, state->history, size_t(RING) * COLUMNS * 4, "the index history");
        op_span(value, state->q_norm, 256 * 4, "a query norm weight");
        op_span(value, state->k_norm, 256 * 4, "a key norm weight");
        op_span(value, state->index_q_norm, COLUMNS * 4, "an index query norm weight");
        op_span(value, state->index_k_norm, COLUMNS * 4, "an index key norm weight");
        op_span(value, projections, checked_floats({steps - 1, stride}) + (heads * 512 + uint64_t(kv.kv_heads) * 512 + 640) * 4, "projections");
        op_span(value, attended, checked_floats({steps, heads, 256}), "an attention output");
        const uint64_t need = sdx_qsa_prefill_attend_scratch(steps, heads, kv.kv_heads, context);
        if (!need || scratch_bytes < need) throw std::runtime_error("sdx_qsa_prefill_attend: scratch too small (see sdx_qsa_prefill_attend_scratch)");
        if (uintptr_t(scratch) % 256) throw std::runtime_error("sdx_qsa_prefill_attend: the scratch must lie on a 256-byte boundary");
        op_span(value, scratch, need, "stage scratch");
        StageArgs args{};
        args.projections = projections; args.stride = stride;
        args.q_norm = state->q_norm; args.k_norm = state->k_norm; args.index_q_norm = state->index_q_norm; args.index_k_norm = state->index_k_norm;
        args.heads = unsigned(heads); args.kv_heads = kv.kv_heads; args.steps = unsigned(steps); args.positions = nullptr; args.ropes = nullptr; args.base = size_t(base);
        args.pages = static_cast<uint8_t*>(kv.pages); args.page_tokens = kv.page_tokens; args.row_bytes = kv.row_bytes; args.page_table = state->page_table; args.page_count = size_t(kv.page_count);
        args.context = context; args.queries = static_cast<float*>(scratch); args.blocks = state->blocks; args.history = state->history; args.pool = pool;
        // 1. rows normalised and turned, K/V rows appended
        // vectors a wave: as many as leave the card waves enough (the whole stage: 9 rows one 83 us, eight 92; 256 rows two 167, eight 176)
        const auto launch_stage = [&](auto kernel, unsigned each) {
            kernel<<<dim3(unsigned((heads + kv.kv_heads + HEADS + STAGE_WAVES * each - 1) / (STAGE_WAVES * each)), unsigned(steps)), 64 * STAGE_WAVES, 0, value.stream>>>(args);
        };
        if (steps >= 512) launch_stage(stage_rows_kernel<8>, 8); else if (steps >= 128) launch_stage(stage_rows_kernel<2>, 2); else launch_stage(stage_rows_kernel<1>, 1);
        SD_CHECK(hipGetLastError());
        // 2. the blocks the span completes, and the ring's newest rows
        index_at = heads * 512 + size_t(kv.kv_heads) * 512;
        const float* incoming = projections + index_at + HEADS * COLUMNS;
        const size_t completed = size_t((base + steps) / 4 - base / 4);
        if (completed) pool_kernel<<<checked_blocks(completed, 1), COLUMNS, 0, value.stream>>>(incoming, size_t(stride), state->history, state->index_k_norm, size_t(pool), size_t(base), state->blocks);
        save_history_kernel<<<checked_blocks(std::min<size_t>(steps, 4) * COLUMNS), 256, 0, value.stream>>>(incoming, size_t(stride), size_t(base), size_t(steps), state->history);
        SD_CHECK(hipGetLastError());
    } catch (const std::exception& e) { ::sd::last_error = e.what(); return -1; }
    }
    // 3. the rows' selections (by intervals past 32768 positions, the packed keys carried from chunk to chunk in the scratch);
    // 4. each row over its selection, gated
    const uint64_t heads = state->heads, kv_heads = state->kv->kv_heads;
    float* queries = static_cast<float*>(scratch);
    float* scores = queries + steps * heads * 256;
    float* indices = scores + steps * pool;
    float* counts = indices + steps * 2052;
    uint8_t* partial = reinterpret_cast<uint8_t*>((reinterpret_cast<uintptr_t>(counts + steps) + 255) & ~uintptr_t(255));
    const uint64_t partial_bytes = sdx_selected_attention_scratch(steps, kv_heads, 2052);
    uint8_t* interval = partial + ((partial_bytes + 255) & ~uint64_t(255));
    if (sdx_qsa_index_interval(handle, projections + index_at, stride, state->blocks, pool, base, steps, 2052, scores, indices, counts, interval,
                               sdx_qsa_index_interval_scratch(steps, pool), valid) < 0) return -1;
    return sdx_selected_attention(handle, state->kv, state->page_table, state->context, base, nullptr, indices, 2052, counts, queries, 0, steps, heads, 0.0625f,
                                  projections + 256, 512, stride, attended, 0, partial, partial_bytes);
}

}  // extern "C"
