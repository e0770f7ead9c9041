// kernels.hpp — host-side launchers shared between translation units. Each
// launcher validates its shape arguments, enqueues on `s` and allocates nothing.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/objeta_hip.h"

struct objeta_hip_context;

namespace objeta {

int32_t launch_qgemv(objeta_hip_context* ctx, int32_t format, hipStream_t s, const void* d_q,
                     const float* d_x, float* d_y, uint64_t rows, uint64_t cols, uint64_t batch);

int32_t launch_fp4_split(objeta_hip_context* ctx, hipStream_t s, const void* d_w, const void* d_s,
                         const float* d_x, float* d_y, uint64_t rows, uint64_t cols, uint64_t batch);

int32_t launch_zero(hipStream_t s, void* d, uint64_t bytes);

// The device address of pinned host bytes [h, h + n) when a kernel can copy them
// (host memory from hipHostMalloc, h and n 16-byte multiples), else nullptr.
const void* pinned_device_ptr(const void* h, size_t n);
// dst[0, n) = the pinned host bytes at device address src_dev, by a kernel on `s`
// (n, dst and src_dev 16-byte multiples).
int32_t launch_h2d_copy(hipStream_t s, void* dst, const void* src_dev, size_t n);
// One copy of a batch: n bytes from a pinned source's device address to dst.
struct H2dCopy {
    void* dst;
    const void* src_dev;
    size_t n;
};
constexpr int kH2dBatch = 32;  // copies per launch (kernel arguments of 768 bytes)
// The n copies of c[] in ceil(n / kH2dBatch) launches on s (pointers and sizes 16-byte
// multiples, as for launch_h2d_copy).
int32_t launch_h2d_copy_batch(hipStream_t s, const H2dCopy* c, size_t n);

// GEMV over an FP8 E4M3 matrix with 128 x 128 E8M0 scale tiles (cols % 128 == 0).
int32_t launch_fp8_rows(objeta_hip_context* ctx, hipStream_t s, const void* d_w, const void* d_s,
                        const float* d_x, float* d_y, uint64_t rows, uint64_t cols, uint64_t batch);

// act_quant (deepseek.rs:1484-1525) of `rows` vectors of `cols` floats (cols % 128
// == 0): F8_E4M3 bytes to d_values, one E8M0 scale per 128 to d_scales, and when
// d_deq is set the dequantized values act_v * act_s (the factors of the reference's
// FP8 GEMVs) as floats. d_deq may alias d_x.
int32_t launch_act_quant(hipStream_t s, const float* d_x, uint64_t rows, uint64_t cols, uint8_t* d_values,
                         uint8_t* d_scales, float* d_deq);
// act_v * act_s as floats for FP8 activations and their 128-element scales.
int32_t launch_fp8_dequant(hipStream_t s, const uint8_t* d_values, const uint8_t* d_scales, uint64_t rows,
                           uint64_t cols, float* d_out);

// The router launch behind objeta_hip_router_topk_device (its epoch words and
// counters are the scratch of stream `s`). With table and sel_tab given and *sel_tab non-null, the router also
// writes the selected experts' table entries to (*sel_tab)[t * k + r] when it can
// (up to kSelTabMaxExperts experts, hidden a multiple of 1024); *sel_tab is set to
// nullptr when it does not.
constexpr uint64_t kSelTabMaxExperts = 256;
constexpr uint64_t kMaxRouterExperts = 1024;  // router workspace: 2 words per expert and token
int32_t launch_router(objeta_hip_context* ctx, hipStream_t s, const float* w_r, const float* bias,
                      const float* x, uint64_t n_tokens, uint64_t n_experts, uint64_t hidden, uint64_t k,
                      int32_t renormalize, uint32_t* ids, float* weights,
                      const objeta_hip_expert_ptrs* table, objeta_hip_expert_ptrs** sel_tab);

int32_t launch_moe_gate_up(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                           uint64_t n_table, const uint32_t* ids, uint64_t n_tokens, uint64_t k, const float* x,
                           float* act, uint64_t hidden, uint64_t inter, float limit,
                           const objeta_hip_expert_ptrs* sel = nullptr, const objeta_hip_expert_ptrs* shared = nullptr,
                           bool official = false);

// sel (optional): the assignments' table entries as the router resolved them; the
// kernels then skip the id and table lookups. shared (optional, a device pointer to
// one table entry): the shared expert, an extra slot per token with weight 1 added
// after the routed sum; act then holds k + 1 slots per token.
// Events recorded after the phases of launch_moe_official_fp4 (each nullable).
struct OfficialMarks {
    hipEvent_t gate_up_end, shared_gate_up_end, act_quant_end, down_end;
};
// The official-arithmetic FP4 MoE layer (FP8 activations, FP4 split routed experts,
// optional FP8 shared expert with 128 x 128 scale tiles).
int32_t launch_moe_official_fp4(objeta_hip_context* ctx, hipStream_t s, const objeta_hip_expert_ptrs* table,
                                uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids,
                                const float* wts, uint64_t n_tokens, uint64_t k, const float* x, float* out,
                                uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit,
                                uint8_t* inter_values, uint8_t* inter_scales, const OfficialMarks* marks);

// The same layer on the grouped-token products (wide.hip), for batches of at
// least kOfficialGroupedMinTokens tokens, or 3 (2) where the per-token kernels would read
// kOfficialGroupedReadBytes (kOfficialGroupedReadBytes2: two tokens share few experts), in
// the grouped path's limits. us, per-token / grouped: hidden 7168, intermediate 2048 at 2
// tokens, top-4, 262 MiB, 106 / 117, top-8, 441 MiB, 172 / 151, at 4 317 / 167; 4608 x 1664
// top-4 at 4 tokens, 274 MiB, 128 / 91; 2048 x 768 top-8 at 5 tokens, 118 MiB, 41 / 45.
constexpr uint64_t kOfficialGroupedMinTokens = 6;
constexpr uint64_t kOfficialGroupedReadBytes = uint64_t(256) << 20;
constexpr uint64_t kOfficialGroupedReadBytes2 = uint64_t(288) << 20;
bool official_grouped_supported(uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                                uint64_t out_dim);
// Whether launch_moe_official_grouped runs the batch on the sets of eight of grouped.hip.
bool official_few(uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter, uint64_t out_dim);
int32_t launch_moe_official_sets(objeta_hip_context* ctx, hipStream_t s, const objeta_hip_expert_ptrs* table,
                                 uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids,
                                 const float* wts, uint64_t n_tokens, uint64_t k, const float* x, float* out,
                                 uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit,
                                 uint8_t* inter_values, uint8_t* inter_scales);
int32_t launch_moe_official_grouped(objeta_hip_context* ctx, hipStream_t s, const objeta_hip_expert_ptrs* table,
                                    uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids,
                                    const float* wts, uint64_t n_tokens, uint64_t k, const float* x, float* out,
                                    uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit,
                                    uint8_t* inter_values, uint8_t* inter_scales);

int32_t launch_moe_down(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                        uint64_t n_table, const uint32_t* ids, const float* wts, uint64_t n_tokens, uint64_t k,
                        const float* act, const float* resid, float* out, uint64_t inter, uint64_t out_dim,
                        const objeta_hip_expert_ptrs* sel = nullptr, const objeta_hip_expert_ptrs* shared = nullptr);

// Looks up (once per device, with the context's device current) the device address
// of the static activation scratch of objeta_hip_moe_selected_device_noalloc and
// keeps it in ctx->static_act.
constexpr uint64_t kStaticActFloats = uint64_t(1) << 20;
int32_t bind_static_scratch(objeta_hip_context* ctx);

int32_t moe_act_scratch(objeta_hip_context* ctx, hipStream_t s, uint64_t n_tokens, uint64_t k, uint64_t inter,
                        float** out);

// Batched GEMV on the matrix cores (every weight decoded once for up to 8 vectors):
// Q4_0 / Q5_0 / IQ3_0 (cols % 64 == 0) or the split FP4 layout (cols % 128 == 0),
// weights 4-byte and x 16-byte aligned, from kGemvMfmaMinBatch vectors. Results
// within the fp32 tolerance of the per-vector kernels (activations split into two
// fp16 parts, 22 significant bits).
constexpr uint64_t kGemvMfmaMinBatch = 5;
bool gemv_mfma_supported(int32_t format, uint64_t rows, uint64_t cols, uint64_t batch, const void* w,
                         const float* x);
int32_t launch_gemv_mfma(objeta_hip_context* ctx, hipStream_t s, int32_t format, const void* w, const void* ws,
                         const float* x, float* y, uint64_t rows, uint64_t cols, uint64_t batch);
// Batches from this many tokens run the grouped-token products in the layer entry
// points (measured on MI355X over 48 Qwen3-A3B-shaped layers, hidden 2048, 128
// experts, top-8, us per layer per-assignment / grouped: 10 tokens 63.7 / 66.7, 12
// tokens 73.3 / 72.0, 16 tokens 85.1 / 76.4, 32 tokens 146.8 / 104.4).
constexpr uint64_t kGroupedMinTokens = 12;
// From 2 tokens when one expert's three matrices take at least this many bytes: at
// hidden 7168 / intermediate 2048 (23 MB FP4 experts, a shared expert, top-8) the grouped
// path takes 123 / 165 / 185 us at 2 / 3 / 4 tokens against 214 / 313 / 406 on the
// per-assignment kernels, top-2 65 / 73 / 81 against 72 / 99 / 130. Only at 2 to 4
// assignments in all are the per-assignment kernels ahead (top-1 without a shared expert
// 42 / 52 / 62 against 50 / 57 / 59). The Qwen3-A3B shape's 2.6 MB experts keep the
// 12-token switch.
constexpr uint64_t kGroupedLargeExpertBytes = uint64_t(8) << 20;
// And from 2 tokens when the per-assignment kernels would read this many bytes (us,
// per-assignment / grouped: Q5_0 2048 x 1408 top-4 at 6 tokens, 136 MiB, 63 / 46; Q4_0 2560
// x 1024 top-4 at 8, 135 MiB, 51 / 42; split FP4 3072 x 1408 top-4 at 5, 132 MiB, 63 / 51).
constexpr uint64_t kGroupedReadBytes = uint64_t(128) << 20;
// Later where the per-assignment kernels run best, with rows whose 64-column groups fill
// whole waves (hidden 2048, 4096, 8192) and an intermediate of at most 1024, while the
// grouped products walk such a row in one chain that grows with hidden: at 8192 not at all
// below 12 tokens. A shared expert is read once per token by the per-assignment kernels;
// at 4096 its bytes count. us, per-assignment / grouped:
//   2048 (cheap formats) Q4_0 2048 x 768 top-8, 8 tokens, 162 MiB, 44 / 46, 10, 203, 53 / 50
//   4096                 Q4_0 4096 x 1024 top-8, 4, 216 MiB, 59 / 70, top-4, 10, 270, 73 / 70
//   4096, shared expert  FP4 4096 x 768 top-4, 9, 215 MiB with it, 59 / 62, 11, 263, 67 / 65
//   4096, Q5_0 and IQ3_0 IQ3_0 4096 x 1024 top-8, 4, 168 MiB, 71 / 82, top-6, 6, 189, 80 / 79
//   8192                 Q4_0 8192 x 384 top-8, 8, 324 MiB, 85 / 108
constexpr uint64_t kGroupedReadBytes2048 = uint64_t(168) << 20;
constexpr uint64_t kGroupedReadBytes4096 = uint64_t(256) << 20;
constexpr uint64_t kGroupedReadBytesShared4096 = uint64_t(216) << 20;
constexpr uint64_t kGroupedReadBytesDear4096 = uint64_t(176) << 20;
// The workspace of a grouped launch, one layout for every form (sets of eight, wide
// products, official layer): a call prepares what any smaller batch of the shape needs under
// capture, whichever form that one takes.
struct GroupedWs {
    uint32_t* hdr;             // 4 words
    void *sets, *shared_sets;  // set records; those of a shared expert apart
    float *xd, *xmult, *amult, *act, *part;
    _Float16 *xh, *xl, *ah, *al;
};
constexpr size_t kWideSetBytes = 128;  // a set record of the wide products
int32_t grouped_workspace(objeta_hip_context* ctx, hipStream_t s, uint64_t n_tokens, uint64_t k, uint64_t n_table,
                          bool shared, uint64_t hidden, uint64_t inter, uint64_t out_dim, bool official, GroupedWs& w);
// Whether launch_moe_grouped (launch_moe_official_grouped) has its workspace or may make it.
bool grouped_ready(objeta_hip_context* ctx, hipStream_t s, int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k,
                   bool shared, uint64_t hidden, uint64_t inter, uint64_t out_dim, bool official);
// Whether an expert's matrices lie below 2^31 bytes, as every grouped form's 32-bit offsets need
// (`official`: with an FP8 shared expert's).
bool matrices_fit(int32_t format, bool official, uint64_t hidden, uint64_t inter, uint64_t out_dim);
// Tokens of one launch of the wide products.
uint64_t wide_tokens(uint64_t k, uint64_t hidden, uint64_t inter);
// Whether a layer of several such launches would write rows of x that a later launch reads:
// out overlaps x and its rows run ahead of x's (out == x with out_dim <= hidden does not).
bool wide_overwrites_x(const float* x, const float* out, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                       uint64_t out_dim);
// Whether the layer entry points run a batch of n_tokens on the grouped path.
bool grouped_preferred(int32_t format, uint64_t n_tokens, uint64_t k, bool shared, uint64_t hidden, uint64_t inter,
                       uint64_t out_dim);
// Whether launch_moe_grouped takes this shape.
bool grouped_supported(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden,
                       uint64_t inter, uint64_t out_dim);
int32_t launch_moe_grouped(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                           uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids, const float* wts,
                           uint64_t n_tokens, uint64_t k, const float* x, const float* resid, float* out,
                           uint64_t hidden, uint64_t inter, uint64_t out_dim, float limit);

// Whether launch_moe_grouped takes the sets of eight for the batch where the wide products
// take it too (measured at the definition).
bool few_assignments(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, bool shared, uint64_t hidden,
                     uint64_t inter, uint64_t out_dim);
// The same layer on the wide products (wide.hip): work items of up to 16 or 32 tokens of
// an expert, any number of tokens. Split FP4 takes them at any batch, the block formats
// from 9 tokens (below, sets of 8 hold every expert's tokens: Q5_0 3072 x 2048 at 3 tokens
// 57 us on them, 66 here), all but few_assignments.
constexpr uint64_t kWideMinTokens = 9;
bool wide_supported(int32_t format, uint64_t n_table, uint64_t n_tokens, uint64_t k, uint64_t hidden, uint64_t inter,
                    uint64_t out_dim);
int32_t launch_moe_wide(objeta_hip_context* ctx, int32_t format, hipStream_t s, const objeta_hip_expert_ptrs* table,
                        uint64_t n_table, const objeta_hip_expert_ptrs* shared, const uint32_t* ids, const float* wts,
                        uint64_t n_tokens, uint64_t k, const float* x, const float* resid, float* out, uint64_t hidden,
                        uint64_t inter, uint64_t out_dim, float limit);
// The batched GEMV from kGemvWideMinBatch vectors (wide.hip; where gemv_mfma_kernel
// would take a second pass); shapes and alignment as gemv_mfma_supported. Q4_0, us
// against the passes: 9 vectors by 2048 x 2048 14.2 / 15.2, 16 by 14336 x 4096 26.5 /
// 35.4, 128 84 / 275.
constexpr uint64_t kGemvWideMinBatch = 9;
bool gemv_wide_supported(int32_t format, uint64_t rows, uint64_t cols, uint64_t batch);
// Bytes of its workspace, and of launch_gemv_mfma's passes of 8 vectors.
size_t gemv_passes_bytes(uint64_t rows, uint64_t cols, uint64_t batch);
size_t gemv_wide_bytes(objeta_hip_context* ctx, int32_t format, uint64_t rows, uint64_t cols, uint64_t batch);
int32_t launch_gemv_wide(objeta_hip_context* ctx, hipStream_t s, int32_t format, const void* w, const void* ws,
                         const float* x, float* y, uint64_t rows, uint64_t cols, uint64_t batch);
// out = resid + sum_j w_j part_j (+ shared part), and the sum of a GEMV's column ranges.
void launch_moe_combine(hipStream_t s, const uint32_t* ids, const float* wts, const float* part,
                        const float* shared_part, const float* resid, float* out, uint32_t n_tokens, uint32_t k,
                        uint32_t out_dim, uint32_t n_table);
void launch_gemv_reduce(hipStream_t s, const float* part, float* y, uint32_t rows, uint32_t n_vec, uint32_t n_ranges);


}  // namespace objeta
