// The encoder's device code in one translation unit (the kernels share the
// __constant__ tables), plus the host-callable launchers.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstring>

#include "common.h"
#include "kernels.h"
#include "prefix.h"

namespace cjx {
__constant__ __align__(16) DeviceTables g_tables;
}  // namespace cjx

#include "frontend.inl"
#include "entropy.inl"
#include "huffman.inl"
#include "assemble.inl"
#include "mlp.inl"
#include "batch.h"
#include "batch.inl"

namespace cjx {

namespace {
#include "mlp_weights.inc"
}  // namespace

bool init_device_tables() {
    const DeviceTables& t{host_tables()};
    return hipMemcpyToSymbol(HIP_SYMBOL(g_tables), &t, sizeof(t)) == hipSuccess && set_default_mlp_weights();
}

bool set_default_mlp_weights() {
    return set_mlp_weights(kTrainedW1, kTrainedB1, kTrainedW2, kTrainedB2, kTrainedThreshold);
}

bool set_mlp_weights(const std::uint16_t* w1, const float* b1, const std::uint16_t* w2, const float* b2,
                     float threshold) {
    MlpWeights m{};
    std::memcpy(m.w1, w1, sizeof(m.w1));
    std::memcpy(m.w2, w2, sizeof(m.w2));
    std::memcpy(m.b1, b1, sizeof(m.b1));
    std::memcpy(m.b2, b2, 7 * sizeof(float));
    m.threshold = threshold;
    return hipMemcpyToSymbol(HIP_SYMBOL(g_mlp), &m, sizeof(m)) == hipSuccess;
}

// Workgroups of the network's passes over n regions.
static std::uint32_t mlp_wgs(std::uint32_t n) {
    const std::uint32_t tiles{n / kMlpTiles + (n % kMlpTiles != 0 ? 1u : 0u)};
    return tiles < kMlpMaxWgs ? tiles : kMlpMaxWgs;
}

std::size_t mlp_partial_floats(std::uint32_t n) {
    return static_cast<std::size_t>(mlp_wgs(n)) * (kMlpParams + 1);  // a row per workgroup
}

void launch_mlp_step(hipStream_t s, const float* x, const float* labels, std::uint32_t n, float lambda,
                     float* partial, float* grad, float* loss, float* params, float* m, float* v, std::uint32_t step,
                     float lr) {
    const std::uint32_t rows{mlp_wgs(n)};
    mlp_grad_kernel<<<rows, kMlpThreads, 0, s>>>(params, x, labels, n, lambda, partial);
    mlp_reduce_kernel<<<(kMlpParams + 1 + 63) / 64, 64 * kMlpSlices, 0, s>>>(partial, rows, n, grad, loss, params, m, v,
                                                                             step, lr);
}

void launch_mlp_forward(hipStream_t s, const float* params, const float* x, std::uint32_t n, float* z) {
    mlp_forward_kernel<<<mlp_wgs(n), kMlpThreads, 0, s>>>(params, x, n, z);
}

// One thread per (block position, channel): non-zero AC counts of a
// first-block and the normalized grid over its covered positions, for frames
// whose coefficients are supplied directly.
__global__ void nz_kernel(Geometry geo, const std::int16_t* __restrict__ ac, const std::int8_t* __restrict__ acs,
                          std::uint8_t* __restrict__ nz_grid, std::uint16_t* __restrict__ nz_count, Clears clr) {
    clear_words(clr, Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y});
    const std::size_t i{blockIdx.x * 256ull + threadIdx.x};
    const std::size_t nblk{geo.nblocks};
    if (i >= 3 * nblk) {
        return;
    }
    const int c{static_cast<int>(i / nblk)};
    const std::size_t pos{i % nblk};
    const int n{acs[pos]};
    if (n == 0) {
        return;
    }
    const int bx{static_cast<int>(pos % geo.bw)}, by{static_cast<int>(pos / geo.bw)};
    const int m{n / 8};
    const std::int16_t* plane{ac + c * nblk * 64};
    std::uint32_t cnt{0};
    for (int e{0}; e < n * n; ++e) {
        if (e / n < m && e % n < m) {
            continue;
        }
        const int q{e >> 6};
        cnt += plane[(static_cast<std::size_t>(by + q / m) * geo.bw + bx + q % m) * 64 + (e & 63)] != 0;
    }
    nz_count[c * nblk + pos] = static_cast<std::uint16_t>(cnt);
    const std::uint32_t l2{n == 16 ? 2u : (n == 32 ? 4u : 0u)};
    for (int dy{0}; dy < m; ++dy) {
        for (int dx{0}; dx < m; ++dx) {
            nz_grid[c * nblk + static_cast<std::size_t>(by + dy) * geo.bw + bx + dx] =
                static_cast<std::uint8_t>((cnt + m * m - 1) >> l2);
        }
    }
}

__global__ void fill_u32_kernel(std::uint32_t* p, std::size_t n, std::uint32_t v) {
    for (std::size_t i{blockIdx.x * 256ull + threadIdx.x}; i < n; i += gridDim.x * 256ull) {
        p[i] = v;
    }
}

bool check_aq_math(unsigned long long* mismatches) {
    unsigned long long* dev{nullptr};
    if (hipMalloc(reinterpret_cast<void**>(&dev), sizeof(unsigned long long)) != hipSuccess) {
        return false;
    }
    bool ok{hipMemset(dev, 0, sizeof(unsigned long long)) == hipSuccess};
    if (ok) {
        // v in [0, 4): bit patterns 0 .. 0x40800000; masking_sqrt below 0.25.
        check_aq_math_kernel<<<8192, 256>>>(0u, 0x40800000u, 0x3e800000u, dev);
        ok = hipGetLastError() == hipSuccess &&
             hipMemcpy(mismatches, dev, sizeof(unsigned long long), hipMemcpyDeviceToHost) == hipSuccess;
    }
    (void)hipFree(dev);
    return ok;
}

std::size_t sizeof_constants() { return sizeof(Constants); }
std::size_t sizeof_codeset() { return sizeof(CodeSet); }
std::size_t sizeof_layout() { return sizeof(Layout); }
std::uint32_t dc_chunks_per_group(const Geometry& geo) {
    // Group 0 is the largest (dc_group_geo).
    const std::uint32_t w{geo.bw < 256 ? geo.bw : 256}, h{geo.bh < 256 ? geo.bh : 256};
    const std::uint32_t items{2 + 6 * w * h + 2 * ((w + 7) / 8) * ((h + 7) / 8)};
    return (items + kDcChunk - 1) / kDcChunk;
}
std::size_t dc_chunk_slot_words() { return kDcSlotWords; }

bool constants_fit(std::uint32_t head_bits, std::uint32_t ac_prefix_bits, std::uint32_t dc_pre_bits,
                   std::uint32_t dc_mid_bits) {
    // A DC header blob: at most 16 + 20 bits of values and one code header
    // beside the constant bits.
    constexpr std::uint32_t blob{32u * kBlobWords - 36u - 32u * kHdrWords};
    return head_bits <= 32u * kHeadConstWords && ac_prefix_bits <= 32u * (kAcGlobalWords / 2) &&
           dc_pre_bits <= blob && dc_mid_bits <= blob;
}

void fill_constants(void* dst, const std::uint32_t* head, std::uint32_t head_bits,
                    const std::uint32_t* dc_global, std::uint32_t dc_global_bits,
                    const std::uint32_t* ac_prefix, std::uint32_t ac_prefix_bits,
                    const std::uint32_t* dc_pre, std::uint32_t dc_pre_bits, const std::uint32_t* dc_mid,
                    std::uint32_t dc_mid_bits) {
    Constants* k{static_cast<Constants*>(dst)};
    std::memset(k, 0, sizeof(Constants));
    k->head_bits = head_bits;
    k->dc_global_bits = dc_global_bits;
    k->ac_prefix_bits = ac_prefix_bits;
    k->dc_pre_bits = dc_pre_bits;
    k->dc_mid_bits = dc_mid_bits;
    std::memcpy(k->head_words, head, (head_bits + 31) / 32 * 4);
    std::memcpy(k->dc_global_words, dc_global, (dc_global_bits + 31) / 32 * 4);
    std::memcpy(k->ac_prefix_words, ac_prefix, (ac_prefix_bits + 31) / 32 * 4);
    std::memcpy(k->dc_pre_words, dc_pre, (dc_pre_bits + 31) / 32 * 4);
    std::memcpy(k->dc_mid_words, dc_mid, (dc_mid_bits + 31) / 32 * 4);
}

static unsigned int grid_for(std::size_t n, std::size_t per) {
    return static_cast<unsigned int>((n + per - 1) / per);
}

void launch_region(hipStream_t s, const Geometry& geo, const FrameParams& prm, const std::uint8_t* luma,
                   std::size_t luma_pitch, const std::uint8_t* chroma, std::size_t chroma_pitch,
                   std::uint16_t* coeffs, std::int8_t* acs, std::int32_t* qf, float* cfl_part,
                   std::uint32_t* list_count, const Clears& clr, hipEvent_t start, hipEvent_t stop,
                   float* features) {
    // Eight equal runs of regions, one per XCD (the kernel maps workgroup i to
    // run i mod 8); workgroups past the last region exit at once.  The events,
    // when given, take the kernel's own start and end times (no marker
    // packets between it and its neighbours).
    const unsigned int per_xcd{(geo.rw * geo.rh + 7) / 8};
    const bool mf{(prm.mode & kModeMfma16) != 0}, learned{(prm.mode & kModeLearned) != 0};
    auto* const kernel{mf ? (learned ? region_kernel<true, true> : region_kernel<true, false>)
                          : (learned ? region_kernel<false, true> : region_kernel<false, false>)};
    hipExtLaunchKernelGGL(kernel, dim3(8 * per_xcd), dim3(256), 0, s, start, stop, 0, geo, prm, luma, luma_pitch,
                          chroma, chroma_pitch, coeffs, acs, qf, cfl_part, list_count, clr, features);
}

void launch_dct8_uniform(hipStream_t s, const Geometry& geo, const FrameParams& prm, const std::uint8_t* luma,
                         std::size_t luma_pitch, const std::uint8_t* chroma, std::size_t chroma_pitch,
                         std::int16_t* ac, std::int32_t* dc, std::int8_t* acs, std::int32_t* qf, std::int8_t* ytox,
                         std::int8_t* ytob) {
    const unsigned int per_xcd{(geo.rw * geo.rh + 7) / 8};
    dct8_uniform_kernel<<<8 * per_xcd, 256, 0, s>>>(geo, prm, luma, luma_pitch, chroma, chroma_pitch, ac, dc, acs,
                                                    qf, ytox, ytob);
}

void launch_tile_quantize(hipStream_t s, const Geometry& geo, const FrameParams& prm,
                          const std::uint16_t* coeffs, const std::int8_t* acs, const std::int32_t* qf,
                          const float* cfl_part, std::int16_t* ac, std::uint8_t* nz_grid,
                          std::uint16_t* nz_count, const ItemList& list, std::int32_t* dc, std::int8_t* ytox,
                          std::int8_t* ytob) {
    tile_quantize_kernel<<<geo.cmw * geo.cmh, 256, 0, s>>>(geo, prm, coeffs, acs, qf, cfl_part, ac, nz_grid,
                                                           nz_count, list, dc, ytox, ytob);
}

void launch_nz(hipStream_t s, const Geometry& geo, const std::int16_t* ac, const std::int8_t* acs,
               std::uint8_t* nz_grid, std::uint16_t* nz_count, const Clears& clr) {
    nz_kernel<<<grid_for(3ull * geo.nblocks, 256), 256, 0, s>>>(geo, ac, acs, nz_grid, nz_count, clr);
}

void launch_fill_u32(hipStream_t s, std::uint32_t* p, std::size_t n, std::uint32_t v) {
    const unsigned int g{grid_for(n, 256) < 1024 ? grid_for(n, 256) : 1024};
    fill_u32_kernel<<<g > 0 ? g : 1, 256, 0, s>>>(p, n, v);
}


void launch_ac_tokens(hipStream_t s, const Geometry& geo, const std::int16_t* ac, const std::int8_t* acs,
                      const std::uint8_t* nz_grid, const std::uint16_t* nz_count, std::uint32_t* tokens,
                      std::uint16_t* item_tokens, std::uint32_t* partial, std::uint32_t* hists,
                      const ItemList& list, const std::int32_t* dc, const std::int32_t* qf, const std::int8_t* ytox,
                      const std::int8_t* ytob, std::uint32_t* fb_count) {
    // One resident round of workgroups (occupancy x CUs of the current
    // device, at most kTokenGrid): a second partial round would double the
    // kernel's time for a few waves.
    static const unsigned int resident{[] {
        int per_cu{0}, dev{0}, cus{0};
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, ac_tokens_kernel, kTokenThreads, 0) != hipSuccess ||
            hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            per_cu <= 0 || cus <= 0) {
            return static_cast<unsigned int>(kTokenGrid);
        }
        const int n{per_cu * cus};
        return static_cast<unsigned int>(n < kTokenGrid ? n : kTokenGrid);
    }()};
    const unsigned int pairs{token_workgroups(geo)};
    const unsigned int grid{pairs < resident ? pairs : resident};
    ac_tokens_kernel<<<grid, kTokenThreads, 0, s>>>(geo, ac, acs, nz_grid, nz_count, tokens, item_tokens, partial,
                                                    list.items, list.count);
    const std::uint32_t chunks{dc_chunks_per_group(geo)};
    histograms_kernel<<<kReduceWgs + chunks * geo.num_dc, 256, 0, s>>>(geo, chunks, partial, static_cast<int>(grid),
                                                                       hists, dc, acs, qf, ytox, ytob, fb_count);
}

std::size_t ac_partial_words() {
    return static_cast<std::size_t>(kTokenGrid) * kNumClusters * kAcSymbols;
}

void launch_huffman(hipStream_t s, int count, const std::uint32_t* hists, CodeSet* cs) {
    huffman_kernel<<<count, 64 * kTrials, 0, s>>>(hists, cs);
}

bool build_codes_host(const std::uint32_t* hists, std::uint32_t count, std::uint32_t* alpha, std::uint8_t* depth,
                      std::uint16_t* bits, std::uint32_t* hdr_words, std::uint32_t* hdr_bits) {
    if (count == 0 || count > 96) {
        return false;
    }
    std::uint32_t* dh{nullptr};
    CodeSet* dcs{nullptr};
    const std::size_t hbytes{static_cast<std::size_t>(count) * kHistStride * sizeof(std::uint32_t)};
    bool ok{hipMalloc(&dh, hbytes) == hipSuccess && hipMalloc(&dcs, sizeof(CodeSet)) == hipSuccess &&
            hipMemcpy(dh, hists, hbytes, hipMemcpyHostToDevice) == hipSuccess};
    auto* host{new CodeSet};
    if (ok) {
        huffman_kernel<<<count, 64 * kTrials, 0, nullptr>>>(dh, dcs);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(host, dcs, sizeof(CodeSet), hipMemcpyDeviceToHost) == hipSuccess;
    }
    if (ok) {
        for (std::uint32_t h{0}; h < count; ++h) {
            alpha[h] = host->alpha[h];
            hdr_bits[h] = host->hdr_bits[h];
            std::memcpy(depth + h * kHistStride, host->depth[h], kHistStride);
            std::memcpy(bits + h * kHistStride, host->code[h], kHistStride * sizeof(std::uint16_t));
            std::memcpy(hdr_words + h * kHdrWords, host->hdr[h], kHdrWords * sizeof(std::uint32_t));
        }
    }
    delete host;
    (void)hipFree(dh);
    (void)hipFree(dcs);
    return ok;
}


std::size_t ac_group_slot_words() {
    return static_cast<std::size_t>(kGroupRuns) * kRunWords;
}

std::size_t ac_group_runs() {
    return kGroupRuns;
}

std::uint32_t ac_group_bands() {
    return kGroupBands;
}

// Workgroups per band of four block rows: enough to give every band's runs
// to different workgroups while the chip has idle slots (256 CUs x 8), one
// where the bands alone fill it (each workgroup numbers the band's tokens
// again).  Measured: 320x240 8.4 us with four, 27 us with one that keeps all
// items; 3840x2160 (1,080 bands) 25.3 us with one, 27.2 with two, 35 with
// four; 7680x4320 75 us with one, 80 with two.
std::uint32_t emit_band_wgs(std::uint32_t bands) {
    const std::uint32_t n{2048 / (bands > 0 ? bands : 1)};
    return n < 1 ? 1 : (n > 4 ? 4 : n);
}

void launch_emit(hipStream_t s, const Geometry& geo, const std::int8_t* acs, const std::uint16_t* item_tokens,
                 const std::uint32_t* tokens, const CodeSet* cs, const Constants* k, const std::uint32_t* fb_count,
                 const std::int32_t* dc, const std::int32_t* qf, const std::int8_t* ytox, const std::int8_t* ytob,
                 std::uint32_t* ac_staging, std::uint16_t* ac_run_bits, std::uint32_t* dc_staging,
                 std::uint32_t* chunk_bits) {
    const std::uint32_t chunks{dc_chunks_per_group(geo)};
    const std::uint32_t bands{geo.num_ac * kGroupBands};
    const std::uint32_t ac_wgs{bands * emit_band_wgs(bands)};
    const std::uint32_t wgs{ac_wgs + chunks * geo.num_dc};
    constexpr std::uint32_t kResident{8 * 256};  // eight workgroups on each of 256 CUs
    emit_kernel<<<wgs, kEmitThreads, 0, s>>>(
        geo, EmitArgs{acs, item_tokens, tokens, cs, k, fb_count, dc, qf, ytox, ytob, ac_staging, ac_run_bits,
                      dc_staging, chunk_bits, chunks, ac_wgs, wgs <= kResident});
}

void launch_layout(hipStream_t s, const Geometry& geo, const Constants* k, const CodeSet* cs,
                   const std::uint16_t* ac_run_bits, std::uint32_t* chunk_bits, std::uint32_t* dc_group_bytes,
                   std::uint64_t* dc_group_bits, std::uint32_t* ac_group_bytes, std::uint64_t* ac_group_bits,
                   Layout* lay, std::uint64_t* ac_base, std::uint64_t* dc_base, std::uint64_t* total_out,
                   hipEvent_t done) {
    hipExtLaunchKernelGGL(layout_kernel, dim3(1), dim3(kLayoutThreads), 0, s, nullptr, done, 0, geo, k, cs, ac_run_bits,
                          chunk_bits, dc_chunks_per_group(geo), dc_group_bytes, dc_group_bits, ac_group_bytes,
                          ac_group_bits, lay, ac_base, dc_base, total_out);
}

void launch_assemble(hipStream_t s, const Geometry& geo, const Constants* k, const Layout* lay,
                     const std::uint32_t* dc_staging, const std::uint32_t* ac_staging, const std::uint64_t* dc_bits,
                     const std::uint16_t* ac_run_bits, const std::uint32_t* chunk_off, const std::uint64_t* dc_base,
                     const std::uint64_t* ac_base, std::uint8_t* out, std::uint64_t cap_bytes, const FileHead& head,
                     hipEvent_t done) {
    const std::uint32_t chunks{dc_chunks_per_group(geo)};
    const Sources P{dc_staging, chunk_off, chunks, ac_staging, ac_run_bits, dc_bits, dc_base, ac_base};
    hipExtLaunchKernelGGL(assemble_kernel, dim3((frame_runs(geo, chunks) + 3) / 4), dim3(256), 0, s, nullptr, done, 0,
                          geo, k, lay, P, reinterpret_cast<std::uint32_t*>(out), cap_bytes, head);
}

// Host memory to the device by the shader: a 512 KB chunk takes 11 us, and 19
// from chunk to chunk with the completion bound to the launch; the runtime's
// copy takes 13 and, its event being a packet of its own, 23.
__global__ __launch_bounds__(256) void copy_in_kernel(uint2* __restrict__ dst, const uint2* __restrict__ src,
                                                      std::uint32_t count) {
    for (std::uint32_t i{blockIdx.x * 256u + threadIdx.x}; i < count; i += gridDim.x * 256u) {
        dst[i] = src[i];
    }
}

void launch_copy_in(hipStream_t s, std::uint8_t* dst, const std::uint8_t* src, std::size_t bytes, hipEvent_t done) {
    const std::uint32_t count{static_cast<std::uint32_t>(bytes / 8)};
    const std::uint32_t wgs{count < 256u * 256u ? (count + 255u) / 256u : 256u};
    hipExtLaunchKernelGGL(copy_in_kernel, dim3(wgs > 0 ? wgs : 1), dim3(256), 0, s, nullptr, done, 0,
                          reinterpret_cast<uint2*>(dst), reinterpret_cast<const uint2*>(src), count);
}

}  // namespace cjx

#ifdef CJX_REGION_CUT
// Profiling builds: the region kernel's cut step (0 = none).
extern "C" int cjx_set_region_cut(int k) {
    return hipMemcpyToSymbol(HIP_SYMBOL(cjx::g_region_cut), &k, sizeof(int)) == hipSuccess ? 0 : 1;
}
#endif
