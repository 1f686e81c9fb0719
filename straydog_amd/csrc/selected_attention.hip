// Selection-list attention over Q8_0 / FP16 K/V rows of 256 columns: every query row attends the positions its own list
// names.  Stands in for the reference's qsa_attention / qsa_attention_rows (gpu/sparse_attention_compute.hpp:609-647:
// qsa_decode_parts :41-135, block = 32 selected keys x 1 K/V head x all grouped query heads, and qsa_decode_merge :139-170),
// with the validity rule of attention_scores (gpu/kernels.cpp:100-165: an entry counts iff 0 <= raw <= position and
// raw < context) and the output gate qsa_gate (gpu/sparse_attention.hpp:439-442, sigmoid as gpu/core.hpp:1108-1111).
//
// Two forms on gfx950, with the same bits: the chunks of a list on workgroups of their own, described here, and for many rows a workgroup
// for a row's whole list (selected_list_kernel; lists_pay says where).
//
// Chunks: a workgroup of 4 waves owns (row, K/V head, 128 entries of the row's list); a wave takes 32
// entries, one per lane for the address arithmetic (list entry -> position -> page -> row address), and gathers the 32 K rows
// and 32 V rows into its LDS stage by 16-byte global->LDS loads whose lanes each name their own piece of a row (a row is 17 or
// 32 such pieces), so a gathered step lands in the stage exactly as a contiguous step of the paged decode kernel does and the
// operand code (paged_rows.hpp) is shared: S^T = K . Q^T and O^T += V^T . P^T on v_mfma_f32_16x16x32_f16 with the group's
// query heads (up to 16) as one tile.  The four waves merge through LDS; the workgroups' partial results (maximum, sum,
// unnormalised output) are merged, normalised and gated by a second kernel, a block per (row, head).
#include "kernels.hpp"
#include "paged_rows.hpp"

#include <type_traits>

using namespace sd;
using namespace sd::paged;

namespace {

constexpr int DIM = 256, CHUNK = WAVES * STEP;       // list entries per workgroup

struct SelectedArgs {
    const uint8_t* pages;
    unsigned page_tokens, kv_heads, heads, group;
    const int32_t* page_table;     // null: one page holds the context
    unsigned page_last;            // the pool's last page (table entries outside the pool are taken as the nearest page of it)
    size_t context, base;
    const uint32_t* dynamic_base;
    const float* indices;
    size_t selected;
    const float* counts;
    const void* q;
    int q_f16;
    float scale_log2;
    float* partial;                // [row][kv head][chunk][16][DIM + 2]
    unsigned chunks;
    const float* gate;             // null: none
    size_t gate_stride, gate_row_stride;
    void* out;
};

__device__ __forceinline__ unsigned list_length(const SelectedArgs& a, size_t row) {
    const float c = a.counts[row];
    return c > 0.0f ? unsigned(min(size_t(c), a.selected)) : 0u;
}

// The group's query heads as B operands: lane li holds head li (zeros past the group).
__device__ __forceinline__ void load_queries(const SelectedArgs& a, size_t row, unsigned kvh, int li, int g, half8 (&qf)[DIM / 32]) {
    const bool real = li < int(a.group);
    const size_t at = (row * a.heads + kvh * a.group + (real ? li : 0)) * DIM;
    #pragma unroll
    for (int b = 0; b < DIM / 32; ++b) {
        half8 value = {};
        if (real) {
            if (a.q_f16) value = *reinterpret_cast<const half8*>(static_cast<const _Float16*>(a.q) + at + 32 * b + 8 * g);
            else {
                const float* from = static_cast<const float*>(a.q) + at + 32 * b + 8 * g;
                #pragma unroll
                for (int i = 0; i < 8; ++i) value[i] = (_Float16)from[i];
            }
        }
        qf[b] = value;
    }
}

// A list entry's row, counted in rows of the pool from plane 0 of page 0 on, and whether the entry counts.  An entry that does not
// is read from the row's own position (a written row: its score is masked, its weight is zero).
__device__ __forceinline__ size_t entry_row(const SelectedArgs& a, float raw, size_t position, unsigned kvh, bool& counts_in) {
    counts_in = raw >= 0.0f && raw <= float(position) && raw < float(a.context);
    const size_t token = counts_in ? size_t(raw) : min(position, a.context - 1);
    const size_t page = a.page_table ? size_t(pool_page(a.page_table[token / a.page_tokens], a.page_last)) : 0, in_page = a.page_table ? token % a.page_tokens : token;
    return (page * 2 * a.kv_heads + kvh) * a.page_tokens + in_page;
}

// 32 entries' weights for the group's heads under their own maximum m; l: the lane's share of their sum.
template<bool Q8>
__device__ __forceinline__ half8 unit_weights(const SelectedArgs& a, const RowLoad<DIM, Q8>& current, const half8 (&qf)[DIM / 32], uint32_t usable, int g, float& m, float& l) {
    floatx4 s[2];
    #pragma unroll
    for (int t = 0; t < 2; ++t) {
        s[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        #pragma unroll
        for (int b = 0; b < DIM / 32; ++b) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(key_operand<DIM>(current, t, b), qf[b], s[t], 0, 0, 0);
        #pragma unroll
        for (int r = 0; r < 4; ++r)
            if (!((usable >> (16 * t + 4 * g + r)) & 1)) s[t][r] = -INFINITY;
    }
    const float top = row_max(fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])), fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3]))));
    m = fmaxf(NEG_BIG, top);
    const float offset = -m * a.scale_log2;
    half8 p;
    l = 0.0f;
    #pragma unroll
    for (int t = 0; t < 2; ++t)
        #pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float w = __builtin_amdgcn_exp2f(fmaf(s[t][r], a.scale_log2, offset));
            l += w;
            p[4 * t + r] = (_Float16)w;
        }
    return p;
}
// The weighted sum of the unit's values for output tile jj, from nothing.
template<bool Q8>
__device__ __forceinline__ floatx4 unit_values(const RowLoad<DIM, Q8>& current, const ValueScales<DIM>& vs, const half8& p, int jj) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(value_operand<DIM>(current, vs, jj), p, floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// The order in which a row's entries are put together is the same however its chunks are spread over waves and workgroups, so a row
// has the same bits alone and among the rows of a prompt: a chunk's four units under their common maximum, in order; the chunks of
// each quarter of the list in order, the sums so far scaled down where a chunk raises the maximum; the quarters in order likewise.
constexpr unsigned QUARTERS = 4;
// a unit's maximum in exponent units, rounded (not contracted with a difference that follows)
__device__ __forceinline__ float exponent_of(float m, float scale_log2) {
    #pragma clang fp contract(off)
    return m * scale_log2;
}
__device__ __forceinline__ unsigned quarter_begin(unsigned chunks, unsigned quarter) { return chunks * quarter / QUARTERS; }
struct Running { float top, sum; };
__device__ __forceinline__ void chunk_factors(Running& so_far, float top, float sum, float& keep, float& take) {
    const float higher = fmaxf(so_far.top, top);
    keep = __builtin_amdgcn_exp2f(so_far.top - higher); take = __builtin_amdgcn_exp2f(top - higher);
    so_far.top = higher;
    so_far.sum = fmaf(sum, take, so_far.sum * keep);
}
__device__ __forceinline__ float chunk_added(float so_far, float value, float keep, float take) { return fmaf(value, take, so_far * keep); }
__device__ __forceinline__ float finished(float value, float sum) { return sum > 0.0f ? value / sum : 0.0f; }
__device__ __forceinline__ float gated(float value, float x) {
    const float e = expf(-fabsf(x));
    return value * (x >= 0.0f ? 1.0f / (1.0f + e) : e / (1.0f + e));
}

template<bool Q8>
__global__ void __launch_bounds__(WAVES * 64) selected_attention_kernel(SelectedArgs a) {
    constexpr int ROW = Q8 ? DIM + DIM / 16 : 2 * DIM, W = DIM / 16, TILES = DIM / 16;
    constexpr int SLAB = STEP * ROW, PIECES = ROW / 16, UNITS = (STEP * PIECES + 63) / 64, STRIDE = DIM + 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, g = lane >> 4;
    const unsigned chunk = blockIdx.x, kvh = blockIdx.y;
    const size_t row = blockIdx.z, position = (a.dynamic_base ? size_t(*a.dynamic_base) : a.base) + row;
    const unsigned count = list_length(a, row);
    if (chunk * CHUNK >= count) return;                 // (the merge knows how many chunks a row has)
    extern __shared__ float lds[];
    uint8_t* const stage = reinterpret_cast<uint8_t*>(lds) + wave * (2 * SLAB);
    const unsigned first = chunk * CHUNK + wave * STEP;  // the wave's entries: first + (0..31)

    floatx4 acc[TILES];
    #pragma unroll
    for (int jj = 0; jj < TILES; ++jj) acc[jj] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = NEG_BIG, l = 0.0f;
    if (first < count) {
        half8 qf[DIM / 32];
        load_queries(a, row, kvh, li, g, qf);
        // lane e < 32: entry first + e
        float raw = -1.0f;
        if (lane < STEP && first + lane < count) raw = a.indices[row * a.selected + first + lane];
        bool counts_in;
        const size_t plane_bytes = size_t(a.page_tokens) * ROW;
        const uint8_t* const krow = a.pages + entry_row(a, raw, position, kvh, counts_in) * ROW;
        const uint64_t usable = __ballot(counts_in);
        settle_loads();
        #pragma unroll
        for (int part = 0; part < 2; ++part) {
            #pragma unroll
            for (int j = 0; j < UNITS; ++j) {
                const int piece = 64 * j + lane, entry = piece / PIECES, within = piece % PIECES;
                const uint64_t from = __shfl(uint64_t(reinterpret_cast<uintptr_t>(krow)), entry & 31);
                if (64 * j + 64 <= STEP * PIECES || piece < STEP * PIECES)
                    load_to_lds<false>(reinterpret_cast<const uint8_t*>(from) + size_t(part ? a.kv_heads : 0) * plane_bytes + 16 * within,
                                       stage + part * SLAB + 1024 * j);
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);             // vmcnt(0): the gathered rows have landed
        RowLoad<DIM, Q8> current;
        load_step<DIM>(current, stage, stage + SLAB, li, g);
        const half8 p = unit_weights<Q8>(a, current, qf, uint32_t(usable), g, m, l);
        ValueScales<DIM> vs;
        value_scales<DIM>(current, vs);
        #pragma unroll
        for (int jj = 0; jj < TILES; ++jj) acc[jj] = unit_values<Q8>(current, vs, p, jj);
    }

    // Merge the waves through LDS: per wave and query head the maximum, the sum and the unnormalised output.
    __syncthreads();    // the merge area overlays the stages
    {
        const float sum = row_sum(l);
        float* mine = lds + (size_t(wave) * 16 + li) * STRIDE;
        if (g == 0) { mine[DIM] = exponent_of(m, a.scale_log2); mine[DIM + 1] = sum; }      // maxima leave in exponent units
        #pragma unroll
        for (int jj = 0; jj < TILES; ++jj)
            #pragma unroll
            for (int r = 0; r < 4; ++r) mine[W * (4 * g + r) + jj] = acc[jj][r];
    }
    __syncthreads();
    float* out = a.partial + ((row * a.kv_heads + kvh) * a.chunks + chunk) * 16 * STRIDE;
    for (unsigned i = threadIdx.x; i < a.group * STRIDE; i += WAVES * 64) {
        const unsigned head = i / STRIDE, col = i % STRIDE;
        float top = NEG_BIG;
        #pragma unroll
        for (int w = 0; w < WAVES; ++w) top = fmaxf(top, lds[(size_t(w) * 16 + head) * STRIDE + DIM]);
        float value;
        if (col == DIM) value = top;
        else {
            value = 0.0f;
            #pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const float* other = lds + (size_t(w) * 16 + head) * STRIDE;
                value = fmaf(other[col], __builtin_amdgcn_exp2f(other[DIM] - top), value);
            }
        }
        out[i] = value;
    }
}

// A block per (row, head), a thread per column: the row's chunks merged, normalised, gated.
template<bool F16_OUT>
__global__ void __launch_bounds__(DIM) selected_merge_kernel(SelectedArgs a) {
    constexpr int STRIDE = DIM + 2;
    const size_t row = blockIdx.x / a.heads;
    const unsigned head = blockIdx.x % a.heads, kvh = head / a.group, col = threadIdx.x;
    const unsigned used = __builtin_amdgcn_readfirstlane((list_length(a, row) + CHUNK - 1) / CHUNK);
    const float* base = a.partial + ((row * a.kv_heads + kvh) * a.chunks) * 16 * STRIDE + size_t(head % a.group) * STRIDE;
    Running so_far{NEG_BIG, 0.0f}, quarter{NEG_BIG, 0.0f};
    float value = 0.0f, quarter_value = 0.0f, keep, take;
    unsigned quarters = 0;                             // those closed
    const auto close = [&] {
        chunk_factors(so_far, quarter.top, quarter.sum, keep, take);
        value = chunk_added(value, quarter_value, keep, take);
        quarter = Running{NEG_BIG, 0.0f};
        quarter_value = 0.0f;
        ++quarters;
    };
    // the chunks' pieces are asked for twenty at a time (a list of 2052 has 17): as many loads in flight, not one after the other; four or
    // eight where there are no more (32 rows of 128 entries, the call 14.2 us with twenty, 12.1; 2048 of 1024 364, 335)
    const auto add = [&](auto at_once) {
        constexpr unsigned AT_ONCE = decltype(at_once)::value;
        for (unsigned c0 = 0; c0 < used; c0 += AT_ONCE) {
            float tops[AT_ONCE], sums[AT_ONCE], values[AT_ONCE];
            #pragma unroll
            for (unsigned i = 0; i < AT_ONCE; ++i) {
                const float* part = base + size_t(min(c0 + i, used - 1)) * 16 * STRIDE;
                tops[i] = part[DIM]; sums[i] = part[DIM + 1]; values[i] = part[col];
            }
            #pragma unroll
            for (unsigned i = 0; i < AT_ONCE; ++i) asm volatile("" : "+v"(values[i]), "+v"(tops[i]), "+v"(sums[i]));      // (here, not one by one behind the branches below)
            #pragma unroll
            for (unsigned i = 0; i < AT_ONCE; ++i) {
                if (c0 + i >= used) break;
                while (c0 + i >= quarter_begin(used, quarters + 1)) close();
                chunk_factors(quarter, tops[i], sums[i], keep, take);
                quarter_value = chunk_added(quarter_value, values[i], keep, take);
            }
        }
    };
    if (used <= 4) add(std::integral_constant<unsigned, 4>{});
    else if (used <= 8) add(std::integral_constant<unsigned, 8>{});
    else add(std::integral_constant<unsigned, 20>{});
    while (quarters < QUARTERS) close();
    value = finished(value, so_far.sum);
    if (a.gate) value = gated(value, a.gate[row * a.gate_row_stride + head * a.gate_stride + col]);
    const size_t at = (row * a.heads + head) * DIM + col;
    if (F16_OUT) static_cast<_Float16*>(a.out)[at] = (_Float16)value;
    else static_cast<float*>(a.out)[at] = value;
}

// The rows of a prompt chunk: a workgroup works a row's whole list for one K/V head, a wave a quarter of it, and stores the finished
// outputs.
//   * The list is turned into places of the pool once, in LDS.  From there on the waves are on their own: each gathers slabs of 32
//     rows (K or V) into a ring of two, asks for the next but one as soon as a slab's operands are in registers, and meets the others
//     only when its quarter is done.
//   * A chunk's four units give their weights first and are then summed, in the order that chunks as workgroups have.
//   * Q8_0 rows lie in a slab as 256 bytes of values and, behind all of them, 16 of scales; the 16-byte piece a lane brings is the one that
//     belongs at its place turned by the row's number, so operands are read without bank conflicts and a row's address costs a lane
//     two instructions (an LDS word, shifted and added).
//   * 77 KB of LDS (Q8_0, a list of 2052) and 256 registers: two workgroups a compute unit, so each SIMD has a second wave while one waits or multiplies.
//     (Units exchanged through LDS chunk by chunk, with 142 KB and one wave a SIMD, took 552 us below.)
//   * Workgroups that run together on one die have neighbouring rows and the same K/V head: their selections overlap, and the die's
//     L2 serves a row to all of them.
// Bound by vector instructions (turning Q8_0 bytes into FP16 operands is 384 of a unit's ~700).  Measured, 1024 rows of 2052 Q8_0
// entries, 24 heads over 2: 276 us where chunks as workgroups and their merge take 741 + 112; FP16 rows, the whole stage: 626 us for 1943.
constexpr unsigned LIST_MAX = 4096;
template<bool Q8> struct ListShape {
    static constexpr int ROW = Q8 ? DIM + DIM / 16 : 2 * DIM, PIECES = ROW / 16, SLAB = STEP * ROW, STAGES = WAVES * 2 * SLAB, LOADS = Q8 ? 9 : 16;
    static constexpr int BYTES = STAGES + WAVES * 16 * 8 + LIST_MAX / 8;      // the list follows
    static_assert(STAGES >= WAVES * WAVES * 4 * 1024, "the waves' sums meet over the stages");
};
// Four global->LDS loads to `to` and the three KiB after it, from four addresses a lane.
__device__ __forceinline__ void load_four_to_lds(const uint8_t* const (&from)[4], uint32_t to) {
    uint32_t keep;
#define SD_NEXT_LOAD "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\t" SD_NEXT_LOAD "global_load_lds_dwordx4 %3, off\n\t"
                 SD_NEXT_LOAD "global_load_lds_dwordx4 %4, off\n\t" SD_NEXT_LOAD "global_load_lds_dwordx4 %5, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(to), "v"(from[0]), "v"(from[1]), "v"(from[2]), "v"(from[3]) : "memory", "scc");
#undef SD_NEXT_LOAD
}
// A slab's rows, asked for; list: the places (in 16-byte pieces of the plane) of its 32 rows.
template<bool Q8>
__device__ __forceinline__ void gather_slab(const uint8_t* plane, const uint32_t* list, uint8_t* slab, int thread) {
    const int lane = fresh(thread) & 63;
    const uint32_t to = __builtin_amdgcn_readfirstlane(lds_address(slab));
    const auto place = [&](uint32_t row_at, uint32_t piece) { return plane + (uint64_t(row_at + piece) << 4); };
    constexpr int SPAN = Q8 ? 16 : 32, ROWS = 64 / SPAN;                 // a lane's piece is one of SPAN; rows a load
    const uint32_t* from = list + lane / SPAN;
    const uint32_t turned = (lane % SPAN) ^ (lane / SPAN);               // (row % 16 = (ROWS * j) % 16 + lane / SPAN, the two without a common bit)
    #pragma unroll
    for (int j = 0; j < SPAN / 2; j += 4) {
        const uint8_t* at[4];
        #pragma unroll
        for (int i = 0; i < 4; ++i) at[i] = place(from[ROWS * (j + i)], turned ^ ((ROWS * (j + i)) % 16));
        load_four_to_lds(at, to + 1024 * j);
    }
    if (Q8 && lane < STEP) load_to_lds<false>(place(list[lane], 16), slab + STEP * DIM);
}
// A slab's operands as paged_rows.hpp takes them: the K side, the V side.
__device__ __forceinline__ void slab_keys(RowLoad<DIM, true>& r, const uint8_t* slab, int thread) {
    const int lane = fresh(thread), li = lane & 15, g = lane >> 4 & 3;
    #pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t row = (16 * t + li) * DIM + 16 * (g / 2 ^ li) + 8 * (g & 1);
        #pragma unroll
        for (int b = 0; b < DIM / 32; ++b) r.k[t][b] = *reinterpret_cast<const uint2*>(slab + (row ^ 32 * b));
        const uint4 scales = *reinterpret_cast<const uint4*>(slab + STEP * DIM + 16 * (16 * t + li));
        r.kscale[t][0] = scales.x; r.kscale[t][1] = scales.y; r.kscale[t][2] = scales.z; r.kscale[t][3] = scales.w;
    }
}
__device__ __forceinline__ void slab_values(RowLoad<DIM, true>& r, const uint8_t* slab, int thread) {
    const int lane = fresh(thread), li = lane & 15, g = lane >> 4 & 3;
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int token = 4 * g + (e < 4 ? e : 12 + e);
        const uint4 words = *reinterpret_cast<const uint4*>(slab + token * DIM + 16 * (li ^ (token & 15)));
        r.v[e][0] = words.x; r.v[e][1] = words.y; r.v[e][2] = words.z; r.v[e][3] = words.w;
        r.vscale[e] = *reinterpret_cast<const uint16_t*>(slab + STEP * DIM + 16 * token + 2 * (li / 2));
    }
}
__device__ __forceinline__ void slab_keys(RowLoad<DIM, false>& r, const uint8_t* slab, int thread) {
    const int lane = fresh(thread), li = lane & 15, g = lane >> 4 & 3;
    #pragma unroll
    for (int t = 0; t < 2; ++t)
        #pragma unroll
        for (int b = 0; b < DIM / 32; ++b) r.k[t][b] = *reinterpret_cast<const half8*>(slab + (16 * t + li) * 2 * DIM + 16 * ((4 * b + g) ^ li));
}
__device__ __forceinline__ void slab_values(RowLoad<DIM, false>& r, const uint8_t* slab, int thread) {
    const int lane = fresh(thread), li = lane & 15, g = lane >> 4 & 3;
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int token = 4 * g + (e < 4 ? e : 12 + e);
        #pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint4 words = *reinterpret_cast<const uint4*>(slab + token * 2 * DIM + 16 * ((2 * li + h) ^ (token & 15)));
            r.v[e][4 * h] = words.x; r.v[e][4 * h + 1] = words.y; r.v[e][4 * h + 2] = words.z; r.v[e][4 * h + 3] = words.w;
        }
    }
}
template<bool Q8, bool F16_OUT>
__global__ void __launch_bounds__(WAVES * 64, Q8 ? 2 : 1) selected_list_kernel(SelectedArgs a, unsigned rows) {
    using Shape = ListShape<Q8>;
    constexpr int TILES = DIM / 16, UNITS = CHUNK / STEP;
    const unsigned items = rows * a.kv_heads, per_die = (items + 7) / 8, item = blockIdx.x % 8 * per_die + blockIdx.x / 8;
    if (item >= items || blockIdx.x / 8 >= per_die) return;
    const unsigned kvh = item / rows;
    const size_t row = item % rows, position = (a.dynamic_base ? size_t(*a.dynamic_base) : a.base) + row;
    const int thread = threadIdx.x, lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread >> 6), li = lane & 15, g = lane >> 4;
    const unsigned count = __builtin_amdgcn_readfirstlane(list_length(a, row)), units = (count + STEP - 1) / STEP, chunks = (count + CHUNK - 1) / CHUNK;
    extern __shared__ uint8_t bytes[];
    uint8_t* const ring = bytes + wave * 2 * Shape::SLAB;
    float2* const stats = reinterpret_cast<float2*>(bytes + Shape::STAGES);                                  // [wave][16]: (maximum, sum)
    uint32_t* const usable = reinterpret_cast<uint32_t*>(stats + WAVES * 16);                                // [unit]
    uint32_t* const list = usable + LIST_MAX / 32;

    for (unsigned e = thread; e < chunks * CHUNK; e += WAVES * 64) {
        bool counts_in;
        list[e] = uint32_t(entry_row(a, e < count ? a.indices[row * a.selected + e] : -1.0f, position, kvh, counts_in)) * Shape::PIECES;
        const uint64_t these = __ballot(counts_in);
        if (lane == 0) { usable[e / STEP] = uint32_t(these); usable[e / STEP + 1] = uint32_t(these >> 32); }
    }
    half8 qf[DIM / 32];
    load_queries(a, row, kvh, li, g, qf);
    settle_loads();
    ring_barrier();
    // The wave's slabs in order: of every chunk of its quarter the units' keys, then their values.
    const uint8_t* const value_plane = a.pages + size_t(a.kv_heads) * a.page_tokens * Shape::ROW;
    const unsigned begin = quarter_begin(chunks, wave), end = quarter_begin(chunks, wave + 1);
    unsigned ahead_chunk = begin, ahead_slab = 0, asked = 0, taken = 0;
    const auto units_of = [&](unsigned chunk) { return min(units - chunk * UNITS, unsigned(UNITS)); };
    const auto ask = [&] {
        if (ahead_chunk >= end) return;
        const unsigned n = units_of(ahead_chunk), unit = ahead_chunk * UNITS + (ahead_slab < n ? ahead_slab : ahead_slab - n);
        gather_slab<Q8>(ahead_slab < n ? a.pages : value_plane, list + unit * STEP, ring + (asked & 1) * Shape::SLAB, thread);
        ++asked;
        if (++ahead_slab == 2 * n) { ahead_slab = 0; ++ahead_chunk; }
    };
    const auto landed = [&] {                               // the next slab, complete
        if (asked - taken > 1) wait_loads_here<Shape::LOADS>(); else wait_loads_here<0>();
        return ring + (taken++ & 1) * Shape::SLAB;
    };
    const auto read = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };       // its operands are in registers: it may be overwritten
    ask();
    ask();
    Running so_far{NEG_BIG, 0.0f};
    floatx4 total[TILES];
    #pragma unroll
    for (int jj = 0; jj < TILES; ++jj) total[jj] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (unsigned chunk = begin; chunk < end; ++chunk) {
        const unsigned n = units_of(chunk);
        half8 p[UNITS];
        float tops[UNITS], weight[UNITS], top = NEG_BIG, chunk_sum = 0.0f;
        #pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            float m = NEG_BIG, l = 0.0f;
            if (u < int(n)) {
                const uint8_t* slab = landed();
                RowLoad<DIM, Q8> current;
                slab_keys(current, slab, thread);
                const uint32_t mask = usable[chunk * UNITS + u];
                read();
                ask();
                p[u] = unit_weights<Q8>(a, current, qf, mask, g, m, l);
            }
            tops[u] = exponent_of(m, a.scale_log2);
            top = fmaxf(top, tops[u]);
            weight[u] = row_sum(l);
        }
        #pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const float sum = weight[u];
            weight[u] = __builtin_amdgcn_exp2f(tops[u] - top);
            chunk_sum = fmaf(sum, weight[u], chunk_sum);
        }
        floatx4 value[TILES];
        #pragma unroll
        for (int jj = 0; jj < TILES; ++jj) value[jj] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        #pragma unroll
        for (int u = 0; u < UNITS; ++u)
            if (u < int(n)) {
                const uint8_t* slab = landed();
                RowLoad<DIM, Q8> current;
                slab_values(current, slab, thread);
                read();
                ask();
                ValueScales<DIM> vs;
                value_scales<DIM>(current, vs);
                #pragma unroll
                for (int jj = 0; jj < TILES; jj += 2) {
                    const floatx4 part[2] = {unit_values<Q8>(current, vs, p[u], jj), unit_values<Q8>(current, vs, p[u], jj + 1)};
                    #pragma unroll
                    for (int i = 0; i < 2; ++i)
                        #pragma unroll
                        for (int r = 0; r < 4; ++r) value[jj + i][r] = fmaf(part[i][r], weight[u], value[jj + i][r]);
                    __builtin_amdgcn_sched_barrier(0);      // (more tiles in flight and the registers spill)
                }
            }
        float keep, take;
        chunk_factors(so_far, top, chunk_sum, keep, take);
        #pragma unroll
        for (int jj = 0; jj < TILES; ++jj)
            #pragma unroll
            for (int r = 0; r < 4; ++r) total[jj][r] = chunk_added(total[jj][r], value[jj][r], keep, take);
    }
    // The quarters meet over the stages, lane to lane: wave w takes the value tiles 4 w .. 4 w + 3 of all four.
    ring_barrier();
    floatx4* const exchange = reinterpret_cast<floatx4*>(bytes);                                             // [to][from][4][64]
    if (g == 0) stats[wave * 16 + li] = float2{so_far.top, so_far.sum};
    #pragma unroll
    for (int jj = 0; jj < TILES; ++jj) exchange[((jj / 4 * WAVES + wave) * 4 + jj % 4) * 64 + lane] = total[jj];
    ring_barrier();
    so_far = Running{NEG_BIG, 0.0f};
    floatx4 sums[4];
    #pragma unroll
    for (int t = 0; t < 4; ++t) sums[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    #pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const float2 quarter = stats[w * 16 + li];
        float keep, take;
        chunk_factors(so_far, quarter.x, quarter.y, keep, take);
        #pragma unroll
        for (int t = 0; t < 4; ++t) {
            const floatx4 part = exchange[((wave * WAVES + w) * 4 + t) * 64 + lane];
            #pragma unroll
            for (int r = 0; r < 4; ++r) sums[t][r] = chunk_added(sums[t][r], part[r], keep, take);
        }
    }
    if (li >= int(a.group)) return;
    // a lane's sums: head li, columns 16 (4 g + r) + 4 wave + t
    const unsigned head = kvh * a.group + li;
    #pragma unroll
    for (int r = 0; r < 4; ++r) {
        const unsigned column = 16 * (4 * g + r) + 4 * wave;
        float value[4];
        #pragma unroll
        for (int t = 0; t < 4; ++t) value[t] = finished(sums[t][r], so_far.sum);
        if (a.gate) {
            const float4 x = *reinterpret_cast<const float4*>(a.gate + row * a.gate_row_stride + head * a.gate_stride + column);
            value[0] = gated(value[0], x.x); value[1] = gated(value[1], x.y); value[2] = gated(value[2], x.z); value[3] = gated(value[3], x.w);
        }
        const size_t at = (row * a.heads + head) * DIM + column;
        if (F16_OUT) {
            typedef _Float16 half4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<half4*>(static_cast<_Float16*>(a.out) + at) = half4{(_Float16)value[0], (_Float16)value[1], (_Float16)value[2], (_Float16)value[3]};
        } else *reinterpret_cast<float4*>(static_cast<float*>(a.out) + at) = float4{value[0], value[1], value[2], value[3]};
    }
}
static_assert(WAVES == QUARTERS, "a wave a quarter");

// Whether rows are better worked a workgroup a row and K/V head (an item) than their chunks of 128 entries a workgroup each: once there are enough
// items for the card, and the lists long enough for a workgroup's four waves, each of which has whole chunks of the list, and for the
// merge that chunks need, which grows with the query heads of a K/V head (the group).  Measured in us, chunks / lists:
//   2052 entries, the stage of a prompt chunk over two K/V heads: Q8_0 32 rows 108 / 127, 48 123 / 132, 64 138 / 134, 256 304 / 175; FP16, whose chunks
//     fill a compute unit's LDS, 16 rows 106 / 115, 24 122 / 118, 64 185 / 125.  Q8_0 over four K/V heads of four: 32 rows 48 / 55 (the call).
//   1024 and 512: Q8_0, 128 items of 12 heads 31 / 31 and 20 / 20, of 4 heads 24 / 30 and 15 / 19, 192 of 8 41 / 31 and 26 / 20.
//   256: Q8_0, 128 items 15 / 17, 256 of 8 heads 19 / 18, of 4 15 / 17, 512 of one 24 / 22; FP16, 128 items of 12 heads 17 / 16, of 4 14 / 15.
//   128, one chunk: Q8_0, 256 items of 8 heads 15 / 17, 512 of 12 26 / 20, 1024 of 4 30 / 35, 2048 of one 43 / 67; FP16, 128 of 12 15 / 14, 1024 of one 47 / 56.
//   64 and 32: Q8_0, 128 items of 12 heads 13 / 12, 512 of 4 16 / 13, of one 12 / 13; FP16, 96 of 4 heads 11 / 10, 512 of one 19 / 22.
bool lists_pay(uint64_t units, bool q8, unsigned group, uint64_t entries, uint64_t items) {
    if (entries <= 128 && group < 4) return false;
    if (entries <= 64 || (entries > 1024 && (group >= 8 || !q8))) return items * (q8 ? 2 : 6) >= units;
    if (entries <= 128) return group >= 8 && (q8 ? items >= 2 * units : items * 4 >= units);
    if (entries <= 256) return q8 ? items >= (group >= 8 ? units : 2 * units) : items * 2 >= units;
    return q8 ? items * 4 >= 3 * units : items * (entries <= 512 ? 4 : 6) >= units;       // (and Q8_0 lists of more under few heads)
}

uint64_t scratch_bytes_for(uint64_t rows, uint64_t kv_heads, uint64_t selected) {
    return checked_floats({rows, kv_heads, (selected + CHUNK - 1) / CHUNK, 16, uint64_t(DIM) + 2});
}

template<bool Q8, bool F16_OUT>
void launch(Device& d, const SelectedArgs& args, size_t rows, bool lists) {
    using Shape = ListShape<Q8>;
    if (lists) {
        const size_t shared = Shape::BYTES + size_t(args.chunks) * CHUNK * 4;
        raise_shared_limit(d, reinterpret_cast<const void*>(&selected_list_kernel<Q8, F16_OUT>), Shape::BYTES + LIST_MAX * 4);
        timed_launch(d, &selected_list_kernel<Q8, F16_OUT>, dim3(unsigned((rows * args.kv_heads + 7) / 8 * 8)), dim3(WAVES * 64), shared, args, unsigned(rows));
        return;
    }
    const size_t shared = std::max<size_t>(size_t(Shape::STAGES), size_t(WAVES) * 16 * (DIM + 2) * 4);
    raise_shared_limit(d, reinterpret_cast<const void*>(&selected_attention_kernel<Q8>), shared);
    timed_launch(d, &selected_attention_kernel<Q8>, dim3(args.chunks, args.kv_heads, unsigned(rows)), dim3(WAVES * 64), shared, args);
    SD_CHECK(hipGetLastError());
    selected_merge_kernel<F16_OUT><<<unsigned(rows * args.heads), DIM, 0, d.stream>>>(args);
}

}  // namespace

extern "C" {

uint64_t sdx_selected_attention_scratch(uint64_t rows, uint64_t kv_heads, uint64_t selected) {
    try { return scratch_bytes_for(rows, kv_heads, selected); } catch (const std::exception&) { return 0; }
}

int sdx_selected_attention(void* handle, const sdx_kv_pool* pool, const int32_t* page_table, uint64_t context, uint64_t base,
                           const uint32_t* dynamic_base, const float* indices, uint64_t selected, const float* counts, const void* q, int q_f16,
                           uint64_t rows, uint64_t heads, float scale, const float* gate, uint64_t gate_stride, uint64_t gate_row_stride, void* out, int out_f16,
                           void* scratch, uint64_t scratch_bytes) {
    SD_OP_BEGIN
    validate_pool(value, pool);
    if (pool->dim != DIM) throw std::runtime_error("sdx_selected_attention: rows of 256 columns");
    if (!(scale > 0.0f) || !rows || rows > 65535 || !heads || heads % pool->kv_heads || heads / pool->kv_heads > 16 || !selected || !context ||
        context > (uint64_t(1) << 24) || pool->kv_heads > 65535)
        throw std::runtime_error("sdx_selected_attention: rows, heads (a multiple of the K/V heads, at most 16 each), selected and context >= 1, scale > 0");
    const uint64_t pages = (context + pool->page_tokens - 1) / pool->page_tokens;
    if (page_table) op_span(value, page_table, checked_floats({pages}), "a page table");
    else if (pool->page_tokens < context) throw std::runtime_error("sdx_selected_attention: without a page table one page must hold the context");
    if (!dynamic_base && base + rows > context) throw std::runtime_error("sdx_selected_attention: rows past the context");
    if (dynamic_base) op_span(value, dynamic_base, 4, "a position");
    op_span(value, indices, checked_floats({rows, selected}), "selection lists");
    op_span(value, counts, checked_floats({rows}), "selection counts");
    op_span(value, q, checked_product({rows, heads, uint64_t(DIM), q_f16 ? 2u : 4u}), "attention queries");
    op_span(value, out, checked_product({rows, heads, uint64_t(DIM), out_f16 ? 2u : 4u}), "an attention output");
    if (gate) {
        if (!gate_row_stride) gate_row_stride = heads * gate_stride;
        if (gate_stride < DIM || gate_row_stride < (heads - 1) * gate_stride + DIM) throw std::runtime_error("sdx_selected_attention: gate strides below a head's 256 values or a row's heads");
        op_span(value, gate, checked_floats({rows - 1, gate_row_stride}) + ((heads - 1) * gate_stride + DIM) * 4, "an attention gate");
    }
    const size_t need = scratch_bytes_for(rows, pool->kv_heads, selected);
    if (scratch_bytes < need) throw std::runtime_error("sdx_selected_attention: scratch too small (see sdx_selected_attention_scratch)");
    op_span(value, scratch, need, "attention scratch");
    SelectedArgs args{};
    args.pages = static_cast<const uint8_t*>(pool->pages);
    args.page_tokens = pool->page_tokens; args.kv_heads = pool->kv_heads; args.heads = unsigned(heads); args.group = unsigned(heads / pool->kv_heads);
    args.page_table = page_table; args.page_last = unsigned(std::min<uint64_t>(pool->page_count - 1, 0x7fffffffu)); args.context = context; args.base = base; args.dynamic_base = dynamic_base;
    args.indices = indices; args.selected = selected; args.counts = counts; args.q = q; args.q_f16 = q_f16;
    args.scale_log2 = scale * 1.4426950408889634f;
    args.partial = static_cast<float*>(scratch);
    args.chunks = unsigned((selected + CHUNK - 1) / CHUNK);
    args.gate = gate; args.gate_stride = size_t(gate_stride); args.gate_row_stride = size_t(gate_row_stride); args.out = out;
    const bool q8 = pool->row_bytes != 2 * pool->dim;
    const bool lists = lists_pay(value.compute_units, q8, args.group, selected, rows * pool->kv_heads) && args.chunks * CHUNK <= LIST_MAX &&
                       checked_product({pool->page_count, 2, pool->kv_heads, pool->page_tokens, pool->row_bytes / 16}) <= (uint64_t(1) << 32) && rows * pool->kv_heads < (uint64_t(1) << 31) &&
                       (uintptr_t(out) | uintptr_t(gate)) % 16 == 0 && (gate_stride | gate_row_stride) % 4 == 0;
    if (q8) { if (out_f16) launch<true, true>(value, args, rows, lists); else launch<true, false>(value, args, rows, lists); }
    else { if (out_f16) launch<false, true>(value, args, rows, lists); else launch<false, false>(value, args, rows, lists); }
    SD_OP_END
}

}  // extern "C"
