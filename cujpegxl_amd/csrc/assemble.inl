// Codestream assembly kernels (included into device.hip).
//
// After the histograms, everything up to the final bytes stays on the device:
// one workgroup per histogram builds its prefix code and header; small
// single-workgroup kernels stitch the variable parts (alphabet sizes, code
// headers, first-block counts, TOC) onto constant bit strings the host built
// once per configuration, lay out the sections, and write the codestream head.

namespace cjx {

constexpr int kHdrWords = 64;      // 2048 bits: bound on one code header
constexpr int kAcGlobalWords = 8192;
constexpr int kMaxAcGroups = 32 * 64;  // at most 32 DC groups of 64 AC groups
// Codestream head: the constant headers (under 32 words) and the TOC, whose
// 2 + 32 + 2048 entries take at most 32 bits each at the largest accepted
// frame (2 + 30 for sections of 4,211,712 bytes or more).
constexpr int kHeadConstWords = 256;
constexpr int kHeadWords = ((kHeadConstWords * 32 + (2 + 32 + kMaxAcGroups) * 32 + 8 + 8191) / 8192) * 256;
static_assert(kHeadWords % 256 == 0 && kHeadWords * 32 >= kHeadConstWords * 32 + (2 + 32 + kMaxAcGroups) * 32 + 8,
              "the head holds the worst-case TOC");

struct Constants {
    // Bit strings precomputed on the host (see encoder.cc).
    std::uint32_t head_bits, dc_global_bits, ac_prefix_bits, dc_pre_bits, dc_mid_bits;
    std::uint32_t head_words[kHeadConstWords];
    std::uint32_t dc_global_words[4];
    std::uint32_t ac_prefix_words[kAcGlobalWords / 2];
    std::uint32_t dc_pre_words[64];
    std::uint32_t dc_mid_words[64];
};

struct CodeSet {
    // Per histogram (32 AC clusters, then DC of each group, then AcMetadata of
    // each group).
    std::uint8_t depth[96][kHistStride];
    std::uint16_t code[96][kHistStride];
    std::uint32_t hdr[96][kHdrWords];
    std::uint32_t hdr_bits[96];
    std::uint32_t alpha[96];
    // The AC codes as the emission reads them: depth | code << 16.
    alignas(16) std::uint32_t lut[kNumClusters * kAcSymbols];
};

struct Layout {
    std::uint64_t total_bytes;
    std::uint64_t codestream_bytes;
    std::uint32_t framing_bytes;
    std::uint32_t head_bytes;
    std::uint64_t dc_global_bit;   // absolute bit positions in the file
    std::uint64_t ac_global_bit;
    std::uint32_t ac_global_bits;
    std::uint32_t overflow;
    std::uint32_t ac_global_words[kAcGlobalWords];
    std::uint32_t head_words[kHeadWords];
    std::uint32_t head_total_bits;
    std::uint32_t framing_words[12];  // container framing, 40 or 48 bytes
};

// One 8-wave workgroup per histogram (the AC clusters', then the DC groups'):
// create_huffman_tree's count floors 1, 2, 4, ... are independent trials, so
// in round r wave w tries floor 2^(8r + w), and the smallest floor whose tree
// fits 15 bits wins (the serial builder stops at that same floor); floors up
// to 2^7 take one round.  Floors above 2^15 continue on wave 0.  Wave 0 then
// builds the codes and the header.
constexpr int kTrials = 8;
constexpr int kTrialRounds = 2;

struct HuffmanShared {
    WaveHuffScratch trial[kTrials];
    std::uint8_t trial_depth[kTrials][kHistStride];
    std::uint32_t trial_max[kTrials];
    WaveCodeScratch code_scratch;
    std::uint32_t hist[kHistStride];
    std::uint8_t depth[kHistStride];
    std::uint16_t code[kHistStride];
    std::uint32_t hdr[kHdrWords];
};

template <int R>
__device__ void huffman_depths(HuffmanShared& S, int alpha) {
    const int w{static_cast<int>(threadIdx.x) >> 6};
    const int lane{static_cast<int>(threadIdx.x) & 63};
    const Leaves<R> L{wave_leaves<R>(S.hist, alpha)};
    if (L.n < 2) {
        return;  // one symbol or none: the simple header, all depths stay 0
    }
    int win{-1};
    for (int round{0}; round < kTrialRounds && win < 0; ++round) {
        if (round > 0) {
            for (int i{lane}; i < kHistStride; i += 64) {
                S.trial_depth[w][i] = 0;
            }
            wave_sync();
        }
        const std::uint32_t maxd{tree_trial<R>(L, 1u << (round * kTrials + w), S.trial_depth[w], S.trial[w])};
        if (lane == 0) {
            S.trial_max[w] = maxd;
        }
        __syncthreads();
        for (int i{0}; i < kTrials; ++i) {
            if (S.trial_max[i] <= 15u) {
                win = i;
                break;
            }
        }
        __syncthreads();
    }
    if (win < 0 && w == 0) {
        for (std::uint32_t count_limit{1u << (kTrials * kTrialRounds)};; count_limit *= 2) {
            for (int i{static_cast<int>(threadIdx.x)}; i < kHistStride; i += 64) {
                S.trial_depth[0][i] = 0;
            }
            wave_sync();
            if (tree_trial<R>(L, count_limit, S.trial_depth[0], S.trial[0]) <= 15u) {
                break;
            }
        }
    }
    __syncthreads();
    const int src{win < 0 ? 0 : win};
    for (int i{static_cast<int>(threadIdx.x)}; i < kHistStride; i += 64 * kTrials) {
        S.depth[i] = S.trial_depth[src][i];
    }
}

__device__ __attribute__((always_inline)) inline void huffman_kernel_body(const Wg& wg, const std::uint32_t* __restrict__ hists,
                                                               CodeSet* __restrict__ cs) {
    __shared__ HuffmanShared S;
    const int h{static_cast<int>(wg.x)};
    const int t{static_cast<int>(threadIdx.x)};
    const int w{t >> 6};
    for (int i{t}; i < kHistStride; i += 64 * kTrials) {
        S.hist[i] = hists[h * kHistStride + i];
        S.depth[i] = 0;
        S.code[i] = 0;
    }
    for (int i{t}; i < kTrials * kHistStride; i += 64 * kTrials) {
        S.trial_depth[i / kHistStride][i % kHistStride] = 0;
    }
    if (t < kHdrWords) {
        S.hdr[t] = 0;
    }
    __syncthreads();
    std::uint32_t top{0};
    for (int i{t & 63}; i < kHistStride; i += 64) {
        if (S.hist[i] != 0) {
            top = static_cast<std::uint32_t>(i) + 1u;
        }
    }
    const int alpha{static_cast<int>(wave_max_u32(top > 1u ? top : 1u))};
    if (alpha > 1) {
        if (alpha <= 64) {
            huffman_depths<1>(S, alpha);
        } else {
            huffman_depths<4>(S, alpha);
        }
    }
    __syncthreads();
    std::uint32_t nbits{0};
    if (w == 0 && alpha > 1) {
        nbits = alpha <= 64 ? wave_finish_code<1>(S.hist, alpha, S.depth, S.code, S.hdr, kHdrWords, S.code_scratch)
                            : wave_finish_code<4>(S.hist, alpha, S.depth, S.code, S.hdr, kHdrWords, S.code_scratch);
    }
    __syncthreads();
    for (int i{t}; i < kHistStride; i += 64 * kTrials) {
        cs->depth[h][i] = S.depth[i];
        cs->code[h][i] = S.code[i];
    }
    if (h < kNumClusters && t < kAcSymbols) {
        cs->lut[h * kAcSymbols + t] =
            static_cast<std::uint32_t>(S.depth[t]) | (static_cast<std::uint32_t>(S.code[t]) << 16);
    }
    if (t < kHdrWords) {
        cs->hdr[h][t] = S.hdr[t];
    }
    if (t == 0) {
        cs->hdr_bits[h] = nbits;
        cs->alpha[h] = static_cast<std::uint32_t>(alpha);
    }
}

__global__ __launch_bounds__(64 * kTrials) void huffman_kernel(const std::uint32_t* __restrict__ hists,
                                                               CodeSet* __restrict__ cs) {
    huffman_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, hists, cs);
}

// Emission of a frame's tokens, one launch: workgroups below ac_wgs write
// runs of an AC group's band, the others one chunk of a DC group.  The DC chunks need no more time than a run and fit beside the
// runs, so they cost no launch of their own.
struct EmitArgs {
    const std::int8_t* acs;
    const std::uint16_t* item_tokens;
    const std::uint32_t* tokens;
    const CodeSet* cs;
    const Constants* k;
    const std::uint32_t* fb_count;
    const std::int32_t* dc;
    const std::int32_t* qf;
    const std::int8_t* ytox;
    const std::int8_t* ytob;
    std::uint32_t* ac_staging;
    std::uint16_t* ac_run_bits;
    std::uint32_t* dc_staging;
    std::uint32_t* chunk_bits;
    std::uint32_t dc_chunks;  // per DC group (the largest group's)
    std::uint32_t ac_wgs;     // workgroups of the AC groups
};

union EmitShared {
    GroupShared ac;
    DcEmitShared dc;
};

__device__ __attribute__((always_inline)) inline void emit_kernel_body(const Wg& wg, const Geometry& geo,
                                                                       const EmitArgs& a) {
    __shared__ EmitShared S;
    if (wg.x < a.ac_wgs) {
        ac_group_emit_body(S.ac, wg, geo, a.acs, a.item_tokens, a.tokens, a.cs->lut, a.ac_staging, a.ac_run_bits,
                           static_cast<int>(a.ac_wgs / (geo.num_ac * kGroupBands)));
        return;
    }
    const std::uint32_t i{wg.x - a.ac_wgs};
    const Wg dwg{i % a.dc_chunks, i / a.dc_chunks, a.dc_chunks, geo.num_dc};
    const int hd{kNumClusters + static_cast<int>(dwg.y)}, hm{hd + static_cast<int>(geo.num_dc)};
    const DcGroupGeo d{dc_group_geo(geo, static_cast<int>(dwg.y))};
    // blob_pre: constant prefix, data alphabet, code header; blob_mid:
    // (first blocks - 1), constant prefix, alphabet, header.
    DcBlob pre, mid;
    pre.lead_bits = 0;
    pre.lead = 0;
    pre.words = a.k->dc_pre_words;
    pre.word_bits = a.k->dc_pre_bits;
    pre.alpha_bits = var_len_u16(a.cs->alpha[hd] - 1, pre.alpha);
    pre.hdr = a.cs->hdr[hd];
    pre.hdr_bits = a.cs->hdr_bits[hd];
    mid.lead_bits = ceil_log2(static_cast<std::uint32_t>(d.n));
    mid.lead = a.fb_count[dwg.y] - 1;
    mid.words = a.k->dc_mid_words;
    mid.word_bits = a.k->dc_mid_bits;
    mid.alpha_bits = var_len_u16(a.cs->alpha[hm] - 1, mid.alpha);
    mid.hdr = a.cs->hdr[hm];
    mid.hdr_bits = a.cs->hdr_bits[hm];
    dc_emit_body(S.dc, dwg, geo, pre, mid, a.dc, a.acs, a.qf, a.ytox, a.ytob, a.cs->depth[hd], a.cs->code[hd],
                 a.cs->depth[hm], a.cs->code[hm], a.dc_staging, a.chunk_bits);
}

__global__ __launch_bounds__(kEmitThreads) void emit_kernel(Geometry geo, EmitArgs a) {
    emit_kernel_body(Wg{blockIdx.x, 0, gridDim.x, 1}, geo, a);
}

// U32 field coder choice (field_coder.h:46-107) as one code word: selector
// in the low 2 bits, then the offset bits.
__device__ __forceinline__ void u32_code(const Distr* d, std::uint32_t value, std::uint32_t& code,
                                         std::uint32_t& len) {
    std::uint32_t best{0}, best_bits{64};
    for (std::uint32_t s{0}; s < 4; ++s) {
        if (d[s].direct) {
            if (d[s].v == value) {
                best = s;
                best_bits = 2;
                break;
            }
            continue;
        }
        if (value < d[s].v ||
            static_cast<std::uint64_t>(value) >= static_cast<std::uint64_t>(d[s].v) + (1ull << d[s].bits)) {
            continue;
        }
        if (2 + d[s].bits < best_bits) {
            best = s;
            best_bits = 2 + d[s].bits;
        }
    }
    if (d[best].direct) {
        code = best;
        len = 2;
        return;
    }
    const std::uint32_t nb{d[best].bits};
    const std::uint32_t off{nb < 32 ? (value - d[best].v) & ((1u << nb) - 1u) : value - d[best].v};
    code = best | (off << 2);
    len = 2 + nb;
}

// AcGlobal, section sizes, TOC, head, framing and every section's position,
// by one 256-thread workgroup.  AcGlobal (constant prefix, 32 alphabet sizes,
// 32 code headers) and the head (constant bits, TOC) are assembled in LDS:
// every piece's bit offset comes from a block scan of the piece lengths, and
// the section bases from scans of the section sizes.  `single` frames (one AC
// group) concatenate DcGlobal, the DC group, AcGlobal and the AC tokens into
// one section without padding in between.
__device__ __attribute__((always_inline)) inline void layout_kernel_body(const Wg& wg, Geometry geo, const Constants* __restrict__ k,
                                                     const CodeSet* __restrict__ cs,
                                                     const std::uint16_t* __restrict__ ac_run_bits,
                                                     std::uint32_t* __restrict__ chunk_bits, std::uint32_t dc_chunks,
                                                     std::uint32_t* __restrict__ dc_group_bytes,
                                                     std::uint64_t* __restrict__ dc_group_bits,
                                                     std::uint32_t* __restrict__ ac_group_bytes,
                                                     std::uint64_t* __restrict__ ac_group_bits,
                                                     Layout* __restrict__ lay, std::uint64_t* __restrict__ ac_base,
                                                     std::uint64_t* __restrict__ dc_base,
                                                     std::uint64_t* __restrict__ total_out) {
    __shared__ std::uint32_t agw[kAcGlobalWords];
    __shared__ std::uint32_t hw[kHeadWords];
    __shared__ std::uint64_t agbits[kMaxAcGroups];
    __shared__ std::uint64_t sh[17];
    const int t{static_cast<int>(threadIdx.x)};
    // The reads that depend on nothing computed here, issued together before
    // the first wait: each thread's first word of the AcGlobal prefix and of
    // the head (the head's constant words are one per thread), its code
    // header's alphabet size or bit count, and its wave's first DC group's
    // chunk sizes.
    static_assert(kHeadConstWords == 256, "one head word per thread");
    __shared__ std::uint32_t dc_bits_s[32];
    const std::uint32_t pre_bits{k->ac_prefix_bits};
    const std::uint32_t hb{k->head_bits};
    const std::uint32_t dc_global_bits{k->dc_global_bits};
    const std::uint32_t prefix_w0{k->ac_prefix_words[t]};
    const std::uint32_t head_w0{k->head_words[t]};
    const std::uint32_t alpha_t{t < kNumClusters ? cs->alpha[t] : 0u};
    const std::uint32_t hdr_bits_t{t >= kNumClusters && t < 2 * kNumClusters ? cs->hdr_bits[t - kNumClusters] : 0u};
    // DC groups: wave w takes groups w, w + 4, ...; the group's chunk sizes
    // become their exclusive prefix sums (the assembly's chunk offsets).  All
    // of a group's sizes (at most kDcRounds per lane) are read at once.
    constexpr int kDcRounds{(kDcMaxChunks + 63) / 64};
    for (int g{t >> 6}; g < static_cast<int>(geo.num_dc); g += 4) {
        const int lane{t & 63};
        const DcGroupGeo d{dc_group_geo(geo, g)};
        const int used{static_cast<int>((d.items + kDcChunk - 1) / kDcChunk)};
        std::uint32_t* const cb{chunk_bits + static_cast<std::size_t>(g) * dc_chunks};
        std::uint32_t v[kDcRounds];
#pragma unroll
        for (int r{0}; r < kDcRounds; ++r) {
            v[r] = 64 * r + lane < used ? cb[64 * r + lane] : 0u;
        }
        std::uint32_t sum{0};
#pragma unroll
        for (int r{0}; r < kDcRounds; ++r) {
            const std::uint32_t incl{wave_incl_scan_u32(v[r])};
            if (64 * r + lane < static_cast<int>(dc_chunks)) {
                cb[64 * r + lane] = sum + incl - v[r];  // chunks past the group's end: empty, at its end
            }
            sum += static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
        }
        if (lane == 0) {
            dc_bits_s[g] = sum;
            dc_group_bits[g] = sum;
            dc_group_bytes[g] = (sum + 7) / 8;
        }
    }
    // AC group sizes: the sums of their runs' bits, eight to a 16-byte read.
    for (int g{t}; g < static_cast<int>(geo.num_ac); g += 256) {
        const uint4* const rb{reinterpret_cast<const uint4*>(ac_run_bits + static_cast<std::size_t>(g) * kGroupRuns)};
        constexpr int kVecs{kGroupRuns / 8};
        uint4 v[kVecs];
#pragma unroll
        for (int i{0}; i < kVecs; ++i) {
            v[i] = rb[i];
        }
        std::uint32_t sum{0};
#pragma unroll
        for (int i{0}; i < kVecs; ++i) {
            for (const std::uint32_t w : {v[i].x, v[i].y, v[i].z, v[i].w}) {
                sum += (w & 0xffffu) + (w >> 16);
            }
        }
        agbits[g] = sum;
        ac_group_bits[g] = sum;
        ac_group_bytes[g] = (sum + 7) / 8;
    }
    for (int i{t}; i < kAcGlobalWords; i += 256) {
        agw[i] = 0;
    }
    for (int i{t}; i < kHeadWords; i += 256) {
        hw[i] = 0;
    }
    __syncthreads();
    std::uint32_t overflow{0};
    const auto dc_bytes = [&](std::uint32_t g) { return (dc_bits_s[g] + 7) / 8; };

    // AcGlobal.
    for (std::uint32_t i{static_cast<std::uint32_t>(t)}; i < (pre_bits + 31) / 32; i += 256) {
        const std::uint32_t rem{pre_bits - 32 * i};
        const std::uint32_t w{i == static_cast<std::uint32_t>(t) ? prefix_w0 : k->ac_prefix_words[i]};
        agw[i] = rem >= 32 ? w : (w & ((1u << rem) - 1u));
    }
    std::uint32_t len{0}, val{0};
    if (t < kNumClusters) {
        len = var_len_u16(alpha_t - 1, val);
    } else if (t < 2 * kNumClusters) {
        len = hdr_bits_t;
    }
    std::uint64_t pieces{0};
    const std::uint64_t off{pre_bits + block_excl_scan(len, sh, pieces)};
    const std::uint64_t abits{pre_bits + pieces};
    if (abits > static_cast<std::uint64_t>(kAcGlobalWords) * 32) {
        overflow = 1;
    } else if (t < kNumClusters) {
        lds_or_bits(agw, kAcGlobalWords, static_cast<std::uint32_t>(off), val, len);
    } else if (t < 2 * kNumClusters) {
        const std::uint32_t* src{cs->hdr[t - kNumClusters]};
        for (std::uint32_t i{0}; i < len; i += 32) {
            lds_or_bits(agw, kAcGlobalWords, static_cast<std::uint32_t>(off) + i, src[i >> 5],
                        len - i < 32 ? len - i : 32u);
        }
    }

    // Head: constant bits, no permutation (one 0 bit), byte-aligned TOC.
    for (std::uint32_t i{static_cast<std::uint32_t>(t)}; i < (hb + 31) / 32; i += 256) {
        const std::uint32_t rem{hb - 32 * i};
        const std::uint32_t w{head_w0};  // i == t: the head has at most 256 words
        hw[i] = rem >= 32 ? w : (w & ((1u << rem) - 1u));
    }
    const Distr toc[4]{{false, 0, 10}, {false, 1024, 14}, {false, 17408, 22}, {false, 4211712, 30}};
    const bool single{geo.num_ac == 1};
    const std::uint32_t dcg{(dc_global_bits + 7) / 8};
    const std::uint32_t acg{static_cast<std::uint32_t>((abits + 7) / 8)};
    const std::uint32_t entries{single ? 1u : 2u + geo.num_dc + geo.num_ac};
    std::uint64_t at{(hb + 1u + 7u) & ~7u};
    std::uint64_t body{0};
    for (std::uint32_t e0{0}; e0 < entries; e0 += 256) {
        const std::uint32_t e{e0 + static_cast<std::uint32_t>(t)};
        std::uint32_t size{0}, code{0}, clen{0};
        if (e < entries) {
            if (single) {
                const std::uint64_t bits{dc_global_bits + dc_bits_s[0] + abits + agbits[0]};
                size = static_cast<std::uint32_t>((bits + 7) / 8);
            } else if (e == 0) {
                size = dcg;
            } else if (e <= geo.num_dc) {
                size = dc_bytes(e - 1);
            } else if (e == geo.num_dc + 1) {
                size = acg;
            } else {
                size = static_cast<std::uint32_t>((agbits[e - geo.num_dc - 2] + 7) / 8);
            }
            u32_code(toc, size, code, clen);
        }
        std::uint64_t chunk_bits{0}, chunk_bytes{0};
        const std::uint64_t p{at + block_excl_scan(clen, sh, chunk_bits)};
        (void)block_excl_scan(size, sh, chunk_bytes);
        if (clen != 0 && p + clen <= static_cast<std::uint64_t>(kHeadWords) * 32) {
            lds_or_bits(hw, kHeadWords, static_cast<std::uint32_t>(p), code, clen);
        }
        at += chunk_bits;
        body += chunk_bytes;
    }
    at = (at + 7) & ~7ull;
    if (at > static_cast<std::uint64_t>(kHeadWords) * 32) {
        overflow = 1;
    }
    const std::uint32_t head_bytes{static_cast<std::uint32_t>(at / 8)};
    const std::uint64_t cs_bytes{head_bytes + body};
    const std::uint32_t framing{cs_bytes >= 0x100000000ull - 8 ? 48u : 40u};

    // Section positions (absolute bits in the file).
    const std::uint64_t dcg_bit{(static_cast<std::uint64_t>(framing) + head_bytes) * 8};
    std::uint64_t ac_global_bit{0};
    if (single) {
        if (t == 0) {
            dc_base[0] = dcg_bit + dc_global_bits;
            ac_global_bit = dcg_bit + dc_global_bits + dc_bits_s[0];
            ac_base[0] = ac_global_bit + abits;
        }
    } else {
        const std::uint64_t first{dcg_bit + static_cast<std::uint64_t>(dcg) * 8};
        std::uint64_t dc_total{0};
        const std::uint32_t g{static_cast<std::uint32_t>(t)};
        const std::uint64_t dsz{g < geo.num_dc ? static_cast<std::uint64_t>(dc_bytes(g)) * 8 : 0ull};
        const std::uint64_t dpre{block_excl_scan(dsz, sh, dc_total)};
        if (g < geo.num_dc) {
            dc_base[g] = first + dpre;
        }
        ac_global_bit = first + dc_total;
        std::uint64_t run{ac_global_bit + static_cast<std::uint64_t>(acg) * 8};
        for (std::uint32_t g0{0}; g0 < geo.num_ac; g0 += 256) {
            const std::uint32_t ga{g0 + static_cast<std::uint32_t>(t)};
            const std::uint64_t asz{ga < geo.num_ac ? (agbits[ga] + 7) / 8 * 8 : 0ull};
            std::uint64_t chunk{0};
            const std::uint64_t apre{block_excl_scan(asz, sh, chunk)};
            if (ga < geo.num_ac) {
                ac_base[ga] = run + apre;
            }
            run += chunk;
        }
    }
    // Container framing (container.cc:35-54): the 32-byte signature and ftyp
    // box, then the jxlc box header (8 bytes, or 16 with a 64-bit size).
    // Lane i forms bytes 4i..4i+3.
    if (t < static_cast<int>(framing / 4)) {
        constexpr std::uint8_t sig[32]{0,   0,   0, 0x0c, 'J', 'X', 'L', ' ', 0x0d, 0x0a, 0x87,
                                       0x0a, 0,  0, 0,    0x14, 'f', 't', 'y', 'p', 'j',  'x',
                                       'l', ' ', 0, 0,    0,    0,   'j', 'x', 'l', ' '};
        const bool large{framing == 48};
        const std::uint64_t box{cs_bytes + (large ? 16 : 8)};
        const std::uint32_t field{large ? 1u : static_cast<std::uint32_t>(box)};
        std::uint32_t word{0};
        for (int j{0}; j < 4; ++j) {
            const int i{4 * t + j};
            std::uint8_t b;
            if (i < 32) {
                b = sig[i];
            } else if (i < 36) {
                b = static_cast<std::uint8_t>(field >> (8 * (35 - i)));
            } else if (i < 40) {
                b = static_cast<std::uint8_t>("jxlc"[i - 36]);
            } else {
                b = static_cast<std::uint8_t>(box >> (8 * (47 - i)));
            }
            word |= static_cast<std::uint32_t>(b) << (8 * j);
        }
        lay->framing_words[t] = word;
    }
    __syncthreads();
    for (int i{t}; i < kAcGlobalWords; i += 256) {
        lay->ac_global_words[i] = agw[i];
    }
    for (int i{t}; i < kHeadWords; i += 256) {
        lay->head_words[i] = hw[i];
    }
    if (t == 0) {
        lay->ac_global_bits = static_cast<std::uint32_t>(abits);
        lay->head_total_bits = static_cast<std::uint32_t>(at);
        lay->head_bytes = head_bytes;
        lay->framing_bytes = framing;
        lay->codestream_bytes = cs_bytes;
        lay->total_bytes = overflow ? ~0ull : framing + cs_bytes;
        *total_out = lay->total_bytes;
        lay->overflow = overflow;
        lay->dc_global_bit = dcg_bit;
        lay->ac_global_bit = ac_global_bit;
    }
}

__global__ __launch_bounds__(256) void layout_kernel(Geometry geo, const Constants* __restrict__ k,
                                                     const CodeSet* __restrict__ cs,
                                                     const std::uint16_t* __restrict__ ac_run_bits,
                                                     std::uint32_t* __restrict__ chunk_bits, std::uint32_t dc_chunks,
                                                     std::uint32_t* __restrict__ dc_group_bytes,
                                                     std::uint64_t* __restrict__ dc_group_bits,
                                                     std::uint32_t* __restrict__ ac_group_bytes,
                                                     std::uint64_t* __restrict__ ac_group_bits,
                                                     Layout* __restrict__ lay, std::uint64_t* __restrict__ ac_base,
                                                     std::uint64_t* __restrict__ dc_base,
                                                     std::uint64_t* __restrict__ total_out) {
    layout_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, k, cs, ac_run_bits, chunk_bits,
                       dc_chunks, dc_group_bytes, dc_group_bits, ac_group_bytes, ac_group_bits, lay, ac_base, dc_base,
                       total_out);
}

// The file is a sequence of bit strings ("runs") laid end to end, each at the
// position the layout gave it or that follows from it: framing, head (headers
// and TOC), DcGlobal, the chunks of the DC groups, AcGlobal, the runs of the
// AC groups.  Gaps between runs (section padding, under 8 bits) are zero bits.
// One wave takes a run and stores the 64-byte lines whose first bit lies
// between its start and the next run's, so that every output word is built
// and stored once (no clearing, no atomics, full lines over the host link);
// only the last of them takes bits of the runs that follow.
struct Sources {
    const std::uint32_t* dc_staging;  // dc_chunks slots of kDcSlotWords per group
    const std::uint32_t* chunk_off;   // the chunks' bit offsets in their group
    std::uint32_t dc_chunks;
    const std::uint32_t* ac_staging;   // kGroupRuns slots of kRunWords per group
    const std::uint16_t* ac_run_bits;  // the runs' bit counts
    const std::uint64_t* dc_bits;
    const std::uint64_t* dc_base;
    const std::uint64_t* ac_base;
};

// Runs of a frame: framing, head, DcGlobal, AcGlobal and the groups'.
__host__ __device__ __forceinline__ std::uint32_t frame_runs(const Geometry& geo, std::uint32_t dc_chunks) {
    return 4 + geo.num_dc * dc_chunks + geo.num_ac * kGroupRuns;
}

struct Run {
    std::uint64_t dst;
    std::uint32_t nbits;
    const std::uint32_t* src;
};

// Run i < 4 + num_dc * dc_chunks: every run but the AC groups'.
__device__ __forceinline__ Run front_run(const Geometry& geo, const Constants* k, const Layout* lay, const Sources& P,
                                         std::uint32_t i) {
    if (i == 0) {
        return {0, lay->framing_bytes * 8, lay->framing_words};
    }
    if (i == 1) {
        return {static_cast<std::uint64_t>(lay->framing_bytes) * 8, lay->head_total_bits, lay->head_words};
    }
    if (i == 2) {
        return {lay->dc_global_bit, k->dc_global_bits, k->dc_global_words};
    }
    if (i == 3 + geo.num_dc * P.dc_chunks) {
        return {lay->ac_global_bit, lay->ac_global_bits, lay->ac_global_words};
    }
    const std::uint32_t c{i - 3}, g{c / P.dc_chunks};
    const std::uint32_t off{P.chunk_off[c]};
    const std::uint32_t end{(c + 1) % P.dc_chunks != 0 ? P.chunk_off[c + 1] : static_cast<std::uint32_t>(P.dc_bits[g])};
    return {P.dc_base[g] + off, end - off, P.dc_staging + static_cast<std::size_t>(c) * kDcSlotWords};
}

// The runs of one AC group, in a wave: lane l holds the sizes of runs 2 l and
// 2 l + 1 and where they end, so that a run's place takes no memory access.
struct AcRuns {
    std::uint32_t g, pair, incl;
    std::uint64_t base;
};

__device__ __forceinline__ AcRuns ac_runs(const Sources& P, std::uint32_t g) {
    static_assert(kGroupRuns % 2 == 0 && kGroupRuns <= 128, "two run sizes per lane");
    const std::uint32_t lane{threadIdx.x & 63u};
    AcRuns a;
    a.g = g;
    a.base = P.ac_base[g];
    a.pair = 2 * lane < kGroupRuns
                 ? reinterpret_cast<const std::uint32_t*>(P.ac_run_bits)[g * (kGroupRuns / 2) + lane]
                 : 0u;
    a.incl = wave_incl_scan_u32((a.pair & 0xffffu) + (a.pair >> 16));
    return a;
}

__device__ __forceinline__ Run ac_run(const AcRuns& a, const Sources& P, std::uint32_t r) {
    const int at{static_cast<int>(r >> 1)};
    const std::uint32_t end{static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(a.incl), at))};
    const std::uint32_t pair{static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(a.pair), at))};
    const std::uint32_t lo{pair & 0xffffu}, hi{pair >> 16};
    const std::uint32_t nbits{(r & 1) != 0 ? hi : lo};
    return {a.base + (end - hi - ((r & 1) != 0 ? 0u : lo)), nbits,
            P.ac_staging + (static_cast<std::size_t>(a.g) * kGroupRuns + r) * kRunWords};
}

// First run at or after r with bits; kGroupRuns when there is none.
__device__ __forceinline__ std::uint32_t next_ac_run(const AcRuns& a, std::uint32_t r) {
    const std::uint64_t even{__ballot((a.pair & 0xffffu) != 0)}, odd{__ballot((a.pair >> 16) != 0)};
    const std::uint32_t e0{(r + 1) >> 1}, o0{r >> 1};  // first even / odd run at or after r, by lane
    const std::uint64_t e{e0 < 64 ? even >> e0 << e0 : 0ull}, o{o0 < 64 ? odd >> o0 << o0 : 0ull};
    const std::uint32_t er{e != 0 ? 2 * static_cast<std::uint32_t>(__builtin_ctzll(e)) : kGroupRuns};
    const std::uint32_t orr{o != 0 ? 2 * static_cast<std::uint32_t>(__builtin_ctzll(o)) + 1 : kGroupRuns};
    return er < orr ? er : orr;
}

// The bits of `r` that fall into the 32-bit word at bit b0 of the file.
__device__ __forceinline__ std::uint32_t run_word(const Run& r, std::uint64_t b0) {
    const std::uint64_t end{r.dst + r.nbits};
    const std::uint64_t s{r.dst > b0 ? r.dst : b0};
    const std::uint64_t e{end < b0 + 32 ? end : b0 + 32};
    if (s >= e) {
        return 0;
    }
    const std::uint32_t o{static_cast<std::uint32_t>(s - r.dst)}, len{static_cast<std::uint32_t>(e - s)};
    const std::uint32_t sh{o & 31u};
    std::uint32_t x{r.src[o >> 5] >> sh};
    if (sh != 0 && len > 32 - sh) {
        x |= r.src[(o >> 5) + 1] << (32 - sh);
    }
    if (len < 32) {
        x &= (1u << len) - 1u;
    }
    return x << static_cast<std::uint32_t>(s - b0);
}

__device__ __attribute__((always_inline)) inline void assemble_kernel_body(const Wg& wg, const Geometry& geo,
                                                                           const Constants* __restrict__ k,
                                                                           const Layout* __restrict__ lay,
                                                                           const Sources& P,
                                                                           std::uint32_t* __restrict__ out_words,
                                                                           std::uint64_t cap_bytes) {
    if (lay->overflow != 0) {
        return;
    }
    const std::uint32_t runs{frame_runs(geo, P.dc_chunks)};
    // Whole words up to the capacity, then the bytes of a partial last word
    // that still fit (the output may be the caller's mapped host buffer).
    std::uint64_t words{(lay->total_bytes + 3) / 4};
    const std::uint64_t cap_words{(cap_bytes + 3) / 4};
    words = words < cap_words ? words : cap_words;
    const std::uint32_t lane{threadIdx.x & 63u};
    const std::uint32_t wave{static_cast<std::uint32_t>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(wg.x * 4 + (threadIdx.x >> 6))))};
    const std::uint32_t front{4 + geo.num_dc * P.dc_chunks};
    for (std::uint32_t i{wave}; i < runs; i += wg.nx * 4) {
        AcRuns group{};
        Run own;
        if (i < front) {
            own = front_run(geo, k, lay, P, i);
        } else {
            group = ac_runs(P, (i - front) / kGroupRuns);
            own = ac_run(group, P, (i - front) % kGroupRuns);
        }
        // Padding never crosses a line: the next run's first line is the
        // first line at or after this run's end.
        const std::uint64_t own_end{own.dst + own.nbits};
        const std::uint64_t w0{(own.dst + 511) / 512 * 16};
        std::uint64_t w1{(own_end + 511) / 512 * 16};
        w1 = w1 < words ? w1 : words;
        for (std::uint64_t base{w0}; base < w1; base += 64) {
            const std::uint64_t w{base + lane};
            std::uint32_t v{w < w1 ? run_word(own, w * 32) : 0u};
            const std::uint64_t last{(base + 64 < w1 ? base + 64 : w1) * 32};  // bits this step stores end here
            if (own_end < last) {
                for (std::uint32_t j{i + 1}; j < runs; ++j) {
                    Run r;
                    if (j < front) {
                        if (j >= 3 && j + 1 < front) {
                            const std::uint32_t g{(j - 3) / P.dc_chunks};
                            const DcGroupGeo d{dc_group_geo(geo, static_cast<int>(g))};
                            if ((j - 3) % P.dc_chunks * kDcChunk >= d.items) {
                                j = 3 + (g + 1) * P.dc_chunks - 1;  // past a smaller group's last chunk
                                continue;
                            }
                        }
                        r = front_run(geo, k, lay, P, j);
                    } else {
                        const std::uint32_t g{(j - front) / kGroupRuns};
                        if (j == front || g != group.g) {
                            group = ac_runs(P, g);
                        }
                        const std::uint32_t n{next_ac_run(group, (j - front) % kGroupRuns)};
                        if (n == kGroupRuns) {
                            j = front + (g + 1) * kGroupRuns - 1;
                            continue;
                        }
                        j = front + g * kGroupRuns + n;
                        r = ac_run(group, P, n);
                    }
                    if (r.dst >= last) {
                        break;
                    }
                    if (w < w1) {
                        v |= run_word(r, w * 32);
                    }
                }
            }
            if (w >= w1) {
                continue;
            }
            if ((w + 1) * 4 <= cap_bytes) {
                out_words[w] = v;
            } else {
                auto* ob{reinterpret_cast<std::uint8_t*>(out_words)};
                for (std::uint64_t b{w * 4}; b < cap_bytes; ++b) {
                    ob[b] = static_cast<std::uint8_t>(v >> (8 * (b - w * 4)));
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void assemble_kernel(Geometry geo, const Constants* __restrict__ k,
                                                       const Layout* __restrict__ lay, Sources P,
                                                       std::uint32_t* __restrict__ out_words,
                                                       std::uint64_t cap_bytes) {
    assemble_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, k, lay, P, out_words, cap_bytes);
}

}  // namespace cjx
