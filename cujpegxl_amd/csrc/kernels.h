// Host-callable launchers for the device kernels (device.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "common.h"

namespace cjx {

struct Constants;
struct CodeSet;
struct Layout;

std::size_t sizeof_constants();
std::size_t sizeof_codeset();
std::size_t sizeof_layout();
// Chunks of a frame's largest DC group (the stride of its chunk tables), and
// words of one chunk's staging slot.
std::uint32_t dc_chunks_per_group(const Geometry& geo);
std::size_t dc_chunk_slot_words();
// Host view of Constants to fill before upload.
void fill_constants(void* dst, const std::uint32_t* head, std::uint32_t head_bits,
                    const std::uint32_t* dc_global, std::uint32_t dc_global_bits,
                    const std::uint32_t* ac_prefix, std::uint32_t ac_prefix_bits,
                    const std::uint32_t* dc_pre, std::uint32_t dc_pre_bits,
                    const std::uint32_t* dc_mid, std::uint32_t dc_mid_bits);
bool constants_fit(std::uint32_t head_bits, std::uint32_t ac_prefix_bits, std::uint32_t dc_pre_bits,
                   std::uint32_t dc_mid_bits);

// A launcher's `start`/`stop`/`done` events, when given, are bound to the
// kernel itself (its start or completion), with no marker packet on the
// stream between it and its neighbours.
void launch_region(hipStream_t s, const Geometry& geo, const FrameParams& prm, const std::uint8_t* luma,
                   std::size_t luma_pitch, const std::uint8_t* chroma, std::size_t chroma_pitch,
                   std::uint16_t* coeffs, std::int8_t* acs, std::int32_t* qf, float* cfl_part,
                   std::uint32_t* list_count, const Clears& clr, hipEvent_t start = nullptr,
                   hipEvent_t stop = nullptr, float* features = nullptr);
// The selection network's weights for the region kernel (FP16 W1 [64][96]
// and W2 [7][64] bit patterns, FP32 biases, the confidence threshold as a
// logit magnitude).
bool set_mlp_weights(const std::uint16_t* w1, const float* b1, const std::uint16_t* w2, const float* b2,
                     float threshold);
// The weights the library was built with (csrc/mlp_weights.inc).
bool set_default_mlp_weights();
// Training: partial-gradient floats for a batch of n regions; one step
// (gradient of the batch's mean loss into `grad`, the loss into `loss[0]`,
// and with lr > 0 an Adam step on params / m / v); forward outputs [n][7].
std::size_t mlp_partial_floats(std::uint32_t n);
void launch_mlp_step(hipStream_t s, const float* x, const float* labels, std::uint32_t n, float lambda,
                     float* partial, float* grad, float* loss, float* params, float* m, float* v, std::uint32_t step,
                     float lr);
void launch_mlp_forward(hipStream_t s, const float* params, const float* x, std::uint32_t n, float* z);
// Config-1 semantics: DCT8 everywhere, uniform quant field, no CfL maps.
void launch_dct8_uniform(hipStream_t s, const Geometry& geo, const FrameParams& prm, const std::uint8_t* luma,
                         std::size_t luma_pitch, const std::uint8_t* chroma, std::size_t chroma_pitch,
                         std::int16_t* ac, std::int32_t* dc, std::int8_t* acs, std::int32_t* qf, std::int8_t* ytox,
                         std::int8_t* ytob);
void launch_tile_quantize(hipStream_t s, const Geometry& geo, const FrameParams& prm,
                          const std::uint16_t* coeffs, const std::int8_t* acs, const std::int32_t* qf,
                          const float* cfl_part, std::int16_t* ac, std::uint8_t* nz_grid,
                          std::uint16_t* nz_count, const ItemList& list, std::int32_t* dc, std::int8_t* ytox,
                          std::int8_t* ytob);
void launch_nz(hipStream_t s, const Geometry& geo, const std::int16_t* ac, const std::int8_t* acs,
               std::uint8_t* nz_grid, std::uint16_t* nz_count, const Clears& clr);
void launch_fill_u32(hipStream_t s, std::uint32_t* p, std::size_t n, std::uint32_t v);
// Mismatching results of the AQ terms' moderate-operand division and square
// root against the compiler's correctly rounded forms, over every float
// input of their domains (check_aq_math_kernel); false on a HIP error.
bool check_aq_math(unsigned long long* mismatches);
// The AC tokens, then the histograms of every AC cluster and DC group.
void launch_ac_tokens(hipStream_t s, const Geometry& geo, const std::int16_t* ac, const std::int8_t* acs,
                      const std::uint8_t* nz_grid, const std::uint16_t* nz_count, std::uint32_t* tokens,
                      std::uint16_t* item_tokens, std::uint32_t* partial, std::uint32_t* hists,
                      const ItemList& list, const std::int32_t* dc, const std::int32_t* qf, const std::int8_t* ytox,
                      const std::int8_t* ytob, std::uint32_t* fb_count);
std::size_t ac_partial_words();
// Builds the codes of `count` host histograms on the current device and copies
// the results back (stage harness; allocates).
bool build_codes_host(const std::uint32_t* hists, std::uint32_t count, std::uint32_t* alpha, std::uint8_t* depth,
                      std::uint16_t* bits, std::uint32_t* hdr_words, std::uint32_t* hdr_bits);
void launch_huffman(hipStream_t s, int count, const std::uint32_t* hists, CodeSet* cs);
// Words of one AC group's staging slot (bound on its token stream).
std::size_t ac_group_slot_words();
// Workgroups the emission gives each of `bands` bands in one launch.
std::uint32_t emit_band_wgs(std::uint32_t bands);
// Runs of one AC group (see entropy.inl's emission).
std::size_t ac_group_runs();
std::uint32_t ac_group_bands();
// The AC groups' runs and the DC groups' chunks into their staging slots,
// with their bit counts.
void launch_emit(hipStream_t s, const Geometry& geo, const std::int8_t* acs, const std::uint16_t* item_tokens,
                 const std::uint32_t* tokens, const CodeSet* cs, const Constants* k, const std::uint32_t* fb_count,
                 const std::int32_t* dc, const std::int32_t* qf, const std::int8_t* ytox, const std::int8_t* ytob,
                 std::uint32_t* ac_staging, std::uint16_t* ac_run_bits, std::uint32_t* dc_staging,
                 std::uint32_t* chunk_bits);
// `chunk_bits` becomes the chunks' bit offsets in their groups.
void launch_layout(hipStream_t s, const Geometry& geo, const Constants* k, const CodeSet* cs,
                   const std::uint16_t* ac_run_bits, std::uint32_t* chunk_bits, std::uint32_t* dc_group_bytes,
                   std::uint64_t* dc_group_bits, std::uint32_t* ac_group_bytes, std::uint64_t* ac_group_bits,
                   Layout* lay, std::uint64_t* ac_base, std::uint64_t* dc_base, std::uint64_t* total_out,
                   hipEvent_t done = nullptr);
void launch_assemble(hipStream_t s, const Geometry& geo, const Constants* k, const Layout* lay,
                     const std::uint32_t* dc_staging, const std::uint32_t* ac_staging, const std::uint64_t* dc_bits,
                     const std::uint16_t* ac_run_bits, const std::uint32_t* chunk_off, const std::uint64_t* dc_base,
                     const std::uint64_t* ac_base, std::uint8_t* out, std::uint64_t cap_bytes,
                     const FileHead& head = FileHead{nullptr, 0}, hipEvent_t done = nullptr);
// `bytes` (a multiple of 8, at 8-byte addresses) of mapped host memory to the
// device; `done` is bound to the copy's completion.
void launch_copy_in(hipStream_t s, std::uint8_t* dst, const std::uint8_t* src, std::size_t bytes, hipEvent_t done);

}  // namespace cjx
