// Selection-list attention over Q8_0 / FP16 K/V rows of 256 columns: every query row attends the positions its own list
// names.  Stands in for the reference's qsa_attention / qsa_attention_rows (gpu/sparse_attention_compute.hpp:609-647:
// qsa_decode_parts :41-135, block = 32 selected keys x 1 K/V head x all grouped query heads, and qsa_decode_merge :139-170),
// with the validity rule of attention_scores (gpu/kernels.cpp:100-165: an entry counts iff 0 <= raw <= position and
// raw < context) and the output gate qsa_gate (gpu/sparse_attention.hpp:439-442, sigmoid as gpu/core.hpp:1108-1111).
//
// Shape of the work on gfx950: a workgroup of 4 waves owns (row, K/V head, 128 entries of the row's list); a wave takes 32
// entries, one per lane for the address arithmetic (list entry -> position -> page -> row address), and gathers the 32 K rows
// and 32 V rows into its LDS stage by 16-byte global->LDS loads whose lanes each name their own piece of a row (a row is 17 or
// 32 such pieces), so a gathered step lands in the stage exactly as a contiguous step of the paged decode kernel does and the
// operand code (paged_rows.hpp) is shared: S^T = K . Q^T and O^T += V^T . P^T on v_mfma_f32_16x16x32_f16 with the group's
// query heads (up to 16) as one tile.  The four waves merge through LDS; the workgroups' partial results (maximum, sum,
// unnormalised output) are merged, normalised and gated by a second kernel, a block per (row, head).
#include "paged_rows.hpp"

using namespace sd;
using namespace sd::paged;

namespace sd {
void validate_pool(Device& d, const sdx_kv_pool* pool);
}

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

// 32 entries' scores, weights and value sums, from nothing.
template<bool Q8>
__device__ __forceinline__ void unit_attention(const SelectedArgs& a, const RowLoad<DIM, Q8>& current, const half8 (&qf)[DIM / 32], uint32_t usable, int g, float& m, float& l,
                                               floatx4 (&acc)[DIM / 16]) {
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
    ValueScales<DIM> vs;
    value_scales<DIM>(current, vs);
    #pragma unroll
    for (int jj = 0; jj < DIM / 16; ++jj)
        acc[jj] = __builtin_amdgcn_mfma_f32_16x16x32_f16(value_operand<DIM>(current, vs, jj), p, floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// The order in which a row's entries are put together is the same however its chunks are spread over workgroups, so a row has the
// same bits alone and among the rows of a prompt: a chunk's four units under their common maximum, in order; then the chunks in
// order, the sums so far scaled down where a chunk raises the maximum.
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
        unit_attention<Q8>(a, current, qf, uint32_t(usable), g, m, l, acc);
    }

    // Merge the waves through LDS: per wave and query head the maximum, the sum and the unnormalised output.
    __syncthreads();    // the merge area overlays the stages
    {
        const float sum = row_sum(l);
        float* mine = lds + (size_t(wave) * 16 + li) * STRIDE;
        if (g == 0) { mine[DIM] = m * a.scale_log2; mine[DIM + 1] = sum; }      // maxima leave in exponent units
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
    const unsigned used = (list_length(a, row) + CHUNK - 1) / CHUNK;
    const float* base = a.partial + ((row * a.kv_heads + kvh) * a.chunks) * 16 * STRIDE + size_t(head % a.group) * STRIDE;
    // the chunks' pieces are asked for eight at a time: eight loads in flight, not one after the other
    constexpr unsigned AT_ONCE = 8;
    Running so_far{NEG_BIG, 0.0f};
    float value = 0.0f;
    for (unsigned c0 = 0; c0 < used; c0 += AT_ONCE) {
        float tops[AT_ONCE], sums[AT_ONCE], values[AT_ONCE];
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) {
            const float* part = base + size_t(min(c0 + i, used - 1)) * 16 * STRIDE;
            tops[i] = part[DIM]; sums[i] = part[DIM + 1]; values[i] = part[col];
        }
        #pragma unroll
        for (unsigned i = 0; i < AT_ONCE; ++i) {
            // (a place past the last chunk: nothing is taken and everything kept)
            float keep, take;
            chunk_factors(so_far, c0 + i < used ? tops[i] : NEG_BIG, c0 + i < used ? sums[i] : 0.0f, keep, take);
            value = chunk_added(value, c0 + i < used ? values[i] : 0.0f, keep, take);
        }
    }
    value = finished(value, so_far.sum);
    if (a.gate) value = gated(value, a.gate[row * a.gate_row_stride + head * a.gate_stride + col]);
    const size_t at = (row * a.heads + head) * DIM + col;
    if (F16_OUT) static_cast<_Float16*>(a.out)[at] = (_Float16)value;
    else static_cast<float*>(a.out)[at] = value;
}

// The rows of a prompt chunk: a workgroup works a row's whole list for one K/V head, chunk after chunk, and stores the finished
// outputs -- no partial results, which for 1024 rows were 0.43 GB written and read again.
//   * The list is turned into pool rows once, in LDS.  A unit's rows are gathered into the wave's stage while the unit before is
//     multiplied: its operands are in registers by then.
//   * A chunk's four units meet through LDS lane to lane: wave w takes the value tiles 4 w .. 4 w + 3 of all four (16 registers of
//     running sums a wave), with FP16 rows over the value slabs, whose next rows are then asked for afterwards.
//   * Workgroups that run together on one die have neighbouring rows and the same K/V head: their selections overlap, and the die's
//     L2 serves a row to all of them.
// Bound by vector instructions (turning Q8_0 bytes into FP16 operands is 384 of a unit's ~600).  Measured, 1024 rows of 2052 entries, 24
// heads over 2: PROMPT_AFTER us where chunks as workgroups and their merge took 741 + 112.
constexpr unsigned LIST_MAX = 4096;
template<bool Q8> struct ListShape {
    static constexpr int ROW = Q8 ? DIM + DIM / 16 : 2 * DIM, SLAB = STEP * ROW, STAGES = WAVES * 2 * SLAB, EXCHANGE = WAVES * WAVES * 4 * 1024;
    static constexpr int BYTES = STAGES + (Q8 ? EXCHANGE : 0) + WAVES * 16 * 8 + LIST_MAX / 8;      // the list follows
};
template<bool Q8, bool F16_OUT>
__global__ void __launch_bounds__(WAVES * 64) selected_list_kernel(SelectedArgs a, unsigned rows) {
    using Shape = ListShape<Q8>;
    constexpr int ROW = Shape::ROW, SLAB = Shape::SLAB, PIECES = ROW / 16, UNITS = (STEP * PIECES + 63) / 64, TILES = DIM / 16;
    const unsigned items = rows * a.kv_heads, per_die = (items + 7) / 8, item = blockIdx.x % 8 * per_die + blockIdx.x / 8;
    if (item >= items || blockIdx.x / 8 >= per_die) return;
    const unsigned kvh = item / rows;
    const size_t row = item % rows, position = (a.dynamic_base ? size_t(*a.dynamic_base) : a.base) + row;
    const int thread = threadIdx.x, lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread >> 6), li = lane & 15, g = lane >> 4;
    const unsigned count = list_length(a, row), chunks = (count + CHUNK - 1) / CHUNK;
    extern __shared__ uint8_t bytes[];
    uint8_t *const kstage = bytes + wave * SLAB, *const vstage = bytes + (WAVES + wave) * SLAB;
    floatx4* const exchange = reinterpret_cast<floatx4*>(bytes + (Q8 ? Shape::STAGES : WAVES * SLAB));       // [to][from][4][64]
    float2* const stats = reinterpret_cast<float2*>(bytes + Shape::STAGES + (Q8 ? Shape::EXCHANGE : 0));     // [wave][16]: (maximum, sum)
    uint32_t* const usable = reinterpret_cast<uint32_t*>(stats + WAVES * 16);                                // [unit]
    uint32_t* const list = usable + LIST_MAX / 32;

    for (unsigned e = thread; e < chunks * CHUNK; e += WAVES * 64) {
        bool counts_in;
        list[e] = uint32_t(entry_row(a, e < count ? a.indices[row * a.selected + e] : -1.0f, position, kvh, counts_in));
        const uint64_t these = __ballot(counts_in);
        if (lane == 0) { usable[e / STEP] = uint32_t(these); usable[e / STEP + 1] = uint32_t(these >> 32); }
    }
    half8 qf[DIM / 32];
    load_queries(a, row, kvh, li, g, qf);
    const size_t value_plane = size_t(a.kv_heads) * a.page_tokens * ROW;
    const auto gather = [&](unsigned unit, uint8_t* to, size_t plane) {
        #pragma unroll
        for (int j = 0; j < UNITS; ++j) {
            const int piece = 64 * j + lane, entry = piece / PIECES, within = piece % PIECES;
            if (64 * j + 64 <= STEP * PIECES || piece < STEP * PIECES)
                load_to_lds<false>(a.pages + plane + size_t(list[unit * STEP + entry]) * ROW + 16 * within, to + 1024 * j);
        }
    };
    settle_loads();
    ring_barrier();
    if (wave * STEP < count) { gather(wave, kstage, 0); gather(wave, vstage, value_plane); }
    Running so_far{NEG_BIG, 0.0f};
    floatx4 total[4];
    #pragma unroll
    for (int t = 0; t < 4; ++t) total[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (unsigned chunk = 0; chunk < chunks; ++chunk) {
        const unsigned unit = chunk * WAVES + wave;
        const bool more = (unit + WAVES) * STEP < count;
        floatx4 acc[TILES];
        float m = NEG_BIG, l = 0.0f;
        if (unit * STEP < count) {
            __builtin_amdgcn_s_waitcnt(0x0f70);             // the gathered rows have landed
            RowLoad<DIM, Q8> current;
            load_step<DIM>(current, kstage, vstage, li, g);
            const uint32_t mask = usable[unit];
            __builtin_amdgcn_s_waitcnt(0xc07f);             // the operands are in registers: the stage is free
            asm volatile("" ::: "memory");
            if (more) { gather(unit + WAVES, kstage, 0); if (Q8) gather(unit + WAVES, vstage, value_plane); }
            unit_attention<Q8>(a, current, qf, mask, g, m, l, acc);
        } else {
            #pragma unroll
            for (int jj = 0; jj < TILES; ++jj) acc[jj] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        const float sum = row_sum(l);
        ring_barrier();                                     // the units of the chunk before have been taken (and, with FP16 rows, every wave has its values)
        if (g == 0) stats[wave * 16 + li] = float2{m * a.scale_log2, sum};
        #pragma unroll
        for (int jj = 0; jj < TILES; ++jj) exchange[((jj / 4 * WAVES + wave) * 4 + jj % 4) * 64 + lane] = acc[jj];
        ring_barrier();
        float2 unit_stats[WAVES];
        float top = NEG_BIG;
        #pragma unroll
        for (int w = 0; w < WAVES; ++w) { unit_stats[w] = stats[w * 16 + li]; top = fmaxf(top, unit_stats[w].x); }
        float weight[WAVES], chunk_sum = 0.0f;
        #pragma unroll
        for (int w = 0; w < WAVES; ++w) { weight[w] = __builtin_amdgcn_exp2f(unit_stats[w].x - top); chunk_sum = fmaf(unit_stats[w].y, weight[w], chunk_sum); }
        float keep, take;
        chunk_factors(so_far, top, chunk_sum, keep, take);
        #pragma unroll
        for (int t = 0; t < 4; ++t) {
            floatx4 part[WAVES];
            #pragma unroll
            for (int w = 0; w < WAVES; ++w) part[w] = exchange[((wave * WAVES + w) * 4 + t) * 64 + lane];
            #pragma unroll
            for (int r = 0; r < 4; ++r) {
                float value = 0.0f;
                #pragma unroll
                for (int w = 0; w < WAVES; ++w) value = fmaf(part[w][r], weight[w], value);
                total[t][r] = chunk_added(total[t][r], value, keep, take);
            }
        }
        if (!Q8 && chunk + 1 < chunks) {
            ring_barrier();                                 // the exchange lay over the value slabs
            if (more) gather(unit + WAVES, vstage, value_plane);
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
        for (int t = 0; t < 4; ++t) value[t] = finished(total[t][r], so_far.sum);
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
    // A workgroup a row and K/V head once there are enough of them: LISTS_RULE
    const bool lists = rows * pool->kv_heads * 4 >= value.compute_units && args.chunks * CHUNK <= LIST_MAX &&
                       checked_product({pool->page_count, 2, pool->kv_heads, pool->page_tokens}) <= (uint64_t(1) << 32) && rows * pool->kv_heads < (uint64_t(1) << 31) &&
                       (uintptr_t(out) | uintptr_t(gate)) % 16 == 0 && (gate_stride | gate_row_stride) % 4 == 0;
    if (q8) { if (out_f16) launch<true, true>(value, args, rows, lists); else launch<true, false>(value, args, rows, lists); }
    else { if (out_f16) launch<false, true>(value, args, rows, lists); else launch<false, false>(value, args, rows, lists); }
    SD_OP_END
}

}  // extern "C"
