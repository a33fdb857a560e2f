// Batched launches: one kernel per stage over every frame of a batch
// (included into device.hip after the stage bodies).  A workgroup finds its
// frame by a binary search over the frames' first workgroups of the stage
// (blockIdx.x is uniform, so the search runs on scalar loads) and runs the
// stage's body with the frame's own workgroup coordinates.

namespace cjx {

// The frame of batched workgroup `b` of a stage and the workgroup's
// coordinates in that frame's own grid.
__device__ __forceinline__ const FrameJob& batch_job_at(const FrameJob* __restrict__ jobs, int count, int stage,
                                                        std::uint32_t b, Wg& wg) {
    int lo{0}, hi{count - 1};
    while (lo < hi) {
        const int mid{(lo + hi + 1) >> 1};
        if (jobs[mid].grid[stage].first <= b) {
            lo = mid;
        } else {
            hi = mid - 1;
        }
    }
    const FrameJob& j{jobs[lo]};
    const StageGrid& g{j.grid[stage]};
    const std::uint32_t local{b - g.first};
    wg = Wg{local % g.nx, local / g.nx, g.nx, g.ny};
    return j;
}

__device__ __forceinline__ const FrameJob& batch_job(const FrameJob* __restrict__ jobs, int count, int stage,
                                                     Wg& wg) {
    return batch_job_at(jobs, count, stage, blockIdx.x, wg);
}

template <bool kMf16, bool kLearned>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void region_batch_kernel(
    const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBRegion, wg)};
    region_kernel_body<kMf16, kLearned>(wg, j.geo, j.prm, j.luma, j.luma_pitch, j.chroma, j.chroma_pitch, j.coeffs,
                                        j.acs, j.qf, j.cfl_part, j.item_count, j.clr, nullptr);
}

// The region stage as a persistent grid: workgroup i stays on XCD i mod 8
// and claims, through that XCD's counter, the batched region workgroups
// b = 8 t + (i mod 8) in turn (t = 0, 1, ...), which are the ones the
// one-workgroup-per-region launch would place on the same XCD: the same
// contiguous runs of regions per XCD.  Every workgroup leaves once its
// XCD's share is claimed; no workgroup waits for another.
template <bool kMf16, bool kLearned>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void region_persistent_batch_kernel(
    const FrameJob* __restrict__ jobs, int count, std::uint32_t total, std::uint32_t* __restrict__ counters) {
    __shared__ std::uint32_t claimed;
    const std::uint32_t x{blockIdx.x & 7u};
    for (;;) {
        __syncthreads();  // every thread is done with the previous region and with `claimed`
        if (threadIdx.x == 0) {
            claimed = atomicAdd(&counters[x], 1u);
        }
        __syncthreads();
        const std::uint32_t b{8u * claimed + x};
        if (b >= total) {
            break;
        }
        Wg wg;
        const FrameJob& j{batch_job_at(jobs, count, kBRegion, b, wg)};
        region_kernel_body<kMf16, kLearned>(wg, j.geo, j.prm, j.luma, j.luma_pitch, j.chroma, j.chroma_pitch,
                                            j.coeffs, j.acs, j.qf, j.cfl_part, j.item_count, j.clr, nullptr);
    }
}

__global__ void clear_counters_kernel(std::uint32_t* __restrict__ counters) {
    if (threadIdx.x < 8) {
        counters[threadIdx.x] = 0;
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void quantize_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBQuantize, wg)};
    tile_quantize_kernel_body(wg, j.geo, j.prm, j.coeffs, j.acs, j.qf, j.cfl_part, j.ac, j.nz_grid, j.nz_count,
                              ItemList{j.item_list, j.item_count}, j.dc, j.ytox, j.ytob);
}

__global__ __launch_bounds__(kTokenThreads) void tokens_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBTokens, wg)};
    ac_tokens_kernel_body(wg, j.geo, j.ac, j.acs, j.nz_grid, j.nz_count, j.tokens, j.item_tokens, j.hist_partial,
                          j.item_list, j.item_count);
}

__global__ __launch_bounds__(256) void histograms_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBHistograms, wg)};
    histograms_kernel_body(wg, j.geo, j.dc_chunks, j.hist_partial,
                           static_cast<int>(j.grid[kBTokens].nx), j.hists, j.dc, j.acs, j.qf, j.ytox, j.ytob,
                           j.fb_count);
}

__global__ __launch_bounds__(64 * kTrials) void huffman_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBHuffman, wg)};
    huffman_kernel_body(wg, j.hists, j.codes);
}

__global__ __launch_bounds__(kEmitThreads) void emit_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBEmit, wg)};
    emit_kernel_body(wg, j.geo, EmitArgs{j.acs, j.item_tokens, j.tokens, j.codes, j.k, j.fb_count, j.dc, j.qf, j.ytox,
                                         j.ytob, j.ac_staging, j.ac_run_bits, j.dc_staging, j.chunk_bits,
                                         j.dc_chunks, wg.nx - j.dc_chunks * j.geo.num_dc, false});
}

__global__ __launch_bounds__(kLayoutThreads) void layout_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBLayout, wg)};
    layout_kernel_body(wg, j.geo, j.k, j.codes, j.ac_run_bits, j.chunk_bits,
                       j.dc_chunks, j.dc_group_bytes,
                       j.dc_group_bits, j.ac_group_bytes, j.ac_group_bits, j.lay, j.ac_base, j.dc_base, j.size_out);
}

__global__ __launch_bounds__(256) void assemble_batch_kernel(const FrameJob* __restrict__ jobs, int count) {
    Wg wg;
    const FrameJob& j{batch_job(jobs, count, kBAssemble, wg)};
    const Sources P{j.dc_staging, j.chunk_bits, j.dc_chunks,
                    j.ac_staging, j.ac_run_bits, j.dc_group_bits, j.dc_base, j.ac_base};
    assemble_kernel_body(wg, j.geo, j.k, j.lay, P, j.out, j.cap, FileHead{nullptr, 0});
}

// Tokenizer workgroups of a batch, about: four times the 1,024 that are
// resident (four workgroups on each of 256 CUs), shared out by the frames'
// blocks.  A workgroup pays a prologue and writes an 8 KB histogram row that
// the next stage sums, so a small frame of a large batch gets few: 16 frames of
// 640x360 to 3840x2160 1253 -> 1175 us against up to 1,024 workgroups for each
// frame, eight frames of 3840x2160 1804 -> 1778.  (A branch of the batch
// launches its frames' part, which is no whole number of resident rounds: 1,536
// for three of the eight.)
constexpr std::uint64_t kBatchTokenWgs = 4096;

void batch_stage_grids(const Geometry& geo, const BatchShape& shape, std::uint64_t blocks, std::uint32_t band_wgs,
                       StageGrid (&g)[kBStages]) {
    const auto set = [&](BatchStage s, std::uint32_t nx, std::uint32_t ny) {
        g[s] = StageGrid{0, nx > 0 ? nx : 1, ny > 0 ? ny : 1, 0};
    };
    const std::uint32_t dc_wgs{dc_chunks_per_group(geo) * geo.num_dc};
    set(kBRegion, 8 * ((geo.rw * geo.rh + 7) / 8), 1);
    set(kBQuantize, geo.cmw * geo.cmh, 1);
    // A frame's share of the tokenizer's workgroups.
    const std::uint64_t share{(kBatchTokenWgs * static_cast<std::uint64_t>(geo.nblocks) + blocks - 1) / blocks};
    const std::uint32_t cap{std::min<std::uint32_t>(shape.token_cap, kTokenGrid)};
    set(kBTokens, std::min({token_workgroups(geo), cap, static_cast<std::uint32_t>(share)}), 1);
    set(kBHistograms, kReduceWgs + dc_wgs, 1);
    set(kBHuffman, kNumClusters + 2 * geo.num_dc, 1);
    set(kBEmit, geo.num_ac * kGroupBands * band_wgs + dc_wgs, 1);
    set(kBLayout, 1, 1);
    const std::uint64_t nb{geo.nblocks};
    const std::uint64_t words{(3 * nb * 384 + 48 * nb + (geo.num_ac + geo.num_dc) * 2048ull + 16384 + 3) / 4};
    const std::uint64_t per_wg{256ull * (shape.assemble_words > 0 ? shape.assemble_words : 1)};
    const std::uint64_t ag{(words + per_wg - 1) / per_wg};
    const std::uint32_t run_wgs{(frame_runs(geo, dc_chunks_per_group(geo)) + 3) / 4};
    set(kBAssemble, ag < run_wgs ? static_cast<std::uint32_t>(ag) : run_wgs, 1);
}

void launch_batch_regions(hipStream_t s, const FrameJob* jobs, int count, const std::uint32_t (&total)[kBStages],
                          std::uint32_t mode, const BatchShape& shape, std::uint32_t* counters) {
    const bool mf{(mode & kModeMfma16) != 0}, learned{(mode & kModeLearned) != 0};
    if (shape.region_wgs == 0) {
        auto* const region{mf ? (learned ? region_batch_kernel<true, true> : region_batch_kernel<true, false>)
                              : (learned ? region_batch_kernel<false, true> : region_batch_kernel<false, false>)};
        region<<<total[kBRegion], 256, 0, s>>>(jobs, count);
    } else {
        auto* const region{mf ? (learned ? region_persistent_batch_kernel<true, true>
                                         : region_persistent_batch_kernel<true, false>)
                              : (learned ? region_persistent_batch_kernel<false, true>
                                         : region_persistent_batch_kernel<false, false>)};
        clear_counters_kernel<<<1, 64, 0, s>>>(counters);
        region<<<shape.region_wgs, 256, 0, s>>>(jobs, count, total[kBRegion], counters);
    }
}

void launch_batch_files(hipStream_t s, const FrameJob* jobs, int count, const std::uint32_t (&total)[kBStages]) {
    quantize_batch_kernel<<<total[kBQuantize], 256, 0, s>>>(jobs, count);
    tokens_batch_kernel<<<total[kBTokens], kTokenThreads, 0, s>>>(jobs, count);
    histograms_batch_kernel<<<total[kBHistograms], 256, 0, s>>>(jobs, count);
    huffman_batch_kernel<<<total[kBHuffman], 64 * kTrials, 0, s>>>(jobs, count);
    emit_batch_kernel<<<total[kBEmit], kEmitThreads, 0, s>>>(jobs, count);
    layout_batch_kernel<<<total[kBLayout], kLayoutThreads, 0, s>>>(jobs, count);
    assemble_batch_kernel<<<total[kBAssemble], 256, 0, s>>>(jobs, count);
}

}  // namespace cjx
