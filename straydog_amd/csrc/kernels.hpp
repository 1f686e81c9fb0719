// What the files of kernels have for one another and for the entry points (each is explained where it is defined).
#pragma once
#include "device.hpp"
#include "../../include/straydog_gpu_ext.h"

namespace sd {

// kv_write.hip
void validate_pool(Device& d, const sdx_kv_pool* pool);

// Called by sd_create (the first two) and sd_graph_begin: paged_attention.hip, harness.hip, block_index.hip
void paged_attention_setup(Device& d);
void harness_setup(Device& d);
void select_thin_reserve(Device& d);

// prefill_attention.hip
void prefill_attention(Device& d, const sdx_kv_pool* pool, const int32_t* page_table, uint64_t table_stride, const int32_t* positions,
                       uint64_t max_context, const void* q, int q_f16, uint64_t seqs, uint64_t span, uint64_t heads, float scale, void* out,
                       int out_f16);
void prefill_chunk(Device& d, const sdx_kv_pool* pool, const int32_t* page_table, uint64_t table_stride, const int32_t* positions,
                   uint64_t max_context, const void* keys, const void* values, int kv_f16, const void* q, int q_f16, uint64_t seqs, uint64_t span,
                   uint64_t heads, float scale, void* out, int out_f16, void* tiles, const int32_t* valid);
uint64_t prefill_tiles_bytes(uint64_t seqs, uint64_t kv_heads, uint64_t max_context);
unsigned union_tile_rows();
void prefill_union(Device& d, const sdx_kv_pool* pool, const int32_t* page_table, uint64_t base, const void* q, int q_f16, uint64_t tokens,
                   uint64_t heads, float scale, const float* gate, uint64_t gate_stride, uint64_t gate_row_stride, void* out, int out_f16,
                   const int32_t* union_pos, const uint32_t* union_mask, const uint32_t* union_count, unsigned union_cap);

// dense_matrix.hip
bool dense_matrix_supported(uint64_t context, uint64_t rows, uint64_t heads, uint64_t kv_heads, uint64_t dim, const float* q, const float* keys, const float* values,
                            const float* gate, const float* out);
void dense_matrix(Device& d, const float* q, const float* keys, const float* values, uint64_t context, const int32_t* positions, uint64_t rows, uint64_t heads,
                  uint64_t kv_heads, uint64_t dim, float scale, const float* gate, float* scratch, uint64_t scratch_splits, float* out);

// latent_gather.hip, latent_rows.hip
bool latent_gather_supported(uint64_t kdim, uint64_t vdim);
uint64_t latent_gather_scratch(uint64_t batch, uint64_t k, uint64_t heads, uint64_t vdim);
void latent_gather(Device& d, const void* q, const void* latents, const int32_t* selected, uint64_t batch, uint64_t groups, uint64_t k,
                   uint64_t heads, float scale, float* out, float* partial);
bool latent_rows_supported(uint64_t dim, uint64_t raw_rows, uint64_t window, uint64_t compressed_rows, uint64_t selections, const void* q, const void* raw,
                           const void* compressed, const void* out);
void latent_rows(Device& d, const float* q, const float* raw, uint64_t raw_rows, const int32_t* positions, uint64_t window, const void* compressed, bool bf16,
                 uint64_t compressed_rows, const int32_t* selected, uint64_t selections, const float* sinks, uint64_t rows, uint64_t heads, float scale,
                 uint64_t pairs, const float* frequencies, const double2* turns, float* out);

// block_interval.hip
size_t interval_scratch_bytes(size_t steps, size_t pool);
bool interval_serves(size_t base);
const uint32_t* interval_select(Device& d, const float* queries, size_t stride, const float* blocks, size_t pool, size_t base, size_t steps,
                                size_t selected, float* scores, float* indices, float* counts, void* scratch, uint64_t* valid, unsigned* gate);
size_t interval_undecided(Device& d, const void* scratch, size_t steps, size_t pool);

}  // namespace sd
