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
// to 2^7 take one round.  Wave 0 then builds the codes and the header.
constexpr int kTrials = 8;

struct HuffmanShared {
    WaveHuffScratch trial[kTrials];
    std::uint8_t trial_depth[kTrials][kHistStride];
    std::uint32_t trial_fits[kTrials];
    alignas(16) std::uint32_t leaf[kHistStride];  // counts in input order
    std::uint32_t rank[kHistStride];              // by symbol
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
    // Ranks in the stable order of the counts, every wave against its share of
    // the leaves.
    constexpr int kShare{64 * R / kTrials};
    static_assert(kShare % 4 == 0, "four leaves per read");
    if (w == 0) {
#pragma unroll
        for (int r{0}; r < R; ++r) {
            if (L.cnt[r] != 0) {
                S.leaf[L.pos[r]] = L.cnt[r];
            }
        }
    }
    __syncthreads();
    std::uint32_t rank[R]{};
    if (kShare * w < L.n) {
#pragma unroll
        for (int b{0}; b < kShare; b += 4) {
            const uint4 x{*reinterpret_cast<const uint4*>(&S.leaf[kShare * w + b])};
            rank_after<R>(L, x.x, kShare * w + b, rank);
            rank_after<R>(L, x.y, kShare * w + b + 1, rank);
            rank_after<R>(L, x.z, kShare * w + b + 2, rank);
            rank_after<R>(L, x.w, kShare * w + b + 3, rank);
        }
#pragma unroll
        for (int r{0}; r < R; ++r) {
            if (L.cnt[r] != 0) {
                atomicAdd(&S.rank[64 * r + lane], rank[r]);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r{0}; r < R; ++r) {
        rank[r] = S.rank[64 * r + lane];
    }
    int win{-1};
    for (int round{0}; win < 0; ++round) {
        if (round > 0) {
            for (int i{lane}; i < kHistStride; i += 64) {
                S.trial_depth[w][i] = 0;
            }
            wave_sync();
        }
        // A floor of 2^31 makes every count equal: no tree is higher than 8.
        const bool fits{tree_trial<R, 64 * R>(L, rank, 1u << min(round * kTrials + w, 31), 15, S.trial_depth[w], S.trial[w])};
        if (lane == 0) {
            S.trial_fits[w] = fits ? 1u : 0u;
        }
        __syncthreads();
        const std::uint64_t all{__ballot(lane < kTrials && S.trial_fits[lane % kTrials] != 0)};
        win = all != 0 ? static_cast<int>(__builtin_ctzll(all)) : -1;
        __syncthreads();
    }
    for (int i{static_cast<int>(threadIdx.x)}; i < kHistStride; i += 64 * kTrials) {
        S.depth[i] = S.trial_depth[win][i];
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
        S.leaf[i] = kQueueEnd;  // where no leaf is: after every leaf
        S.rank[i] = 0;
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
    int alpha{1};
#pragma unroll
    for (int r{0}; r < kHistStride / 64; ++r) {
        const std::uint64_t m{__ballot(S.hist[64 * r + (t & 63)] != 0)};
        if (m != 0) {
            alpha = 64 * r + 64 - static_cast<int>(__builtin_clzll(m));
        }
    }
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
        nbits = alpha <= 64 ? wave_store_code<1>(S.hist, alpha, S.depth, S.hdr, kHdrWords, S.code_scratch)
                            : wave_store_code<4>(S.hist, alpha, S.depth, S.hdr, kHdrWords, S.code_scratch);
    }
    if (w == 1 && alpha > 1) {  // all depths 0 (one symbol or none): no code
        if (alpha <= 64) {
            wave_depths_to_codes<1>(S.depth, alpha, S.code);
        } else {
            wave_depths_to_codes<4>(S.depth, alpha, S.code);
        }
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

// Emission of a frame's tokens, one launch: ac_wgs workgroups
// write runs of an AC group's band, the others one chunk of a DC group each,
// which fit beside the runs and cost no launch of their own.
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
    // The DC groups' workgroups first: a DC chunk's chain is the longer one
    // where an AC workgroup has one run or none, so in a grid that is resident
    // as a whole it should not be dispatched last (1920x1080 12.4 -> 11.1 us,
    // 1368x776 10.3 -> 8.9); in a larger one the AC workgroups, with several
    // runs in a row, come first (3840x2160 25.0 us, 28.2 the other way round).
    bool dc_first;
};

union EmitShared {
    GroupShared ac;
    DcEmitShared dc;
};

__device__ __attribute__((always_inline)) inline void emit_kernel_body(const Wg& wg, const Geometry& geo,
                                                                       const EmitArgs& a) {
    __shared__ EmitShared S;
    const std::uint32_t dc_wgs{wg.nx - a.ac_wgs};
    // This workgroup's number with the AC groups' first.
    const std::uint32_t b{!a.dc_first ? wg.x : (wg.x < dc_wgs ? a.ac_wgs + wg.x : wg.x - dc_wgs)};
    if (b < a.ac_wgs) {
        ac_group_emit_body(S.ac, Wg{b, wg.y, wg.nx, wg.ny}, geo, a.acs, a.item_tokens, a.tokens, a.cs->lut, a.ac_staging, a.ac_run_bits,
                           static_cast<int>(a.ac_wgs / (geo.num_ac * kGroupBands)));
        return;
    }
    const std::uint32_t i{b - a.ac_wgs};
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

// Exclusive scans of two values per thread at once (one barrier), over
// kWaves waves; `sh` holds 2 kWaves words and must not be in use.
template <int kWaves>
__device__ __forceinline__ void block_excl_scan2(std::uint32_t& a, std::uint32_t& b, std::uint32_t* sh,
                                                 std::uint32_t& total_a, std::uint32_t& total_b) {
    const int lane{static_cast<int>(threadIdx.x) & 63}, wv{static_cast<int>(threadIdx.x) >> 6};
    const std::uint32_t xa{wave_incl_scan_u32(a)}, xb{wave_incl_scan_u32(b)};
    if (lane == 63) {
        sh[wv] = xa;
        sh[kWaves + wv] = xb;
    }
    __syncthreads();
    std::uint32_t base_a{0}, base_b{0};
    total_a = total_b = 0;
#pragma unroll
    for (int i{0}; i < kWaves; ++i) {
        const std::uint32_t ta{sh[i]}, tb{sh[kWaves + i]};
        base_a += i < wv ? ta : 0u;
        base_b += i < wv ? tb : 0u;
        total_a += ta;
        total_b += tb;
    }
    a = base_a + xa - a;
    b = base_b + xb - b;
}

// AcGlobal, section sizes, TOC, head, framing and every section's position,
// by one workgroup.  AcGlobal (constant prefix, 32 alphabet sizes, 32 code
// headers) and the head (constant bits, TOC) are assembled in LDS: the pieces'
// bit offsets come from one wave scan (64 pieces), the TOC's and the
// sections' from one scan over the TOC entries, which are in section order.
// `single` frames (one AC group) concatenate DcGlobal, the DC group, AcGlobal
// and the AC tokens into one section without padding in between.
//
// One workgroup's chain of latencies bounds it, so every global read is
// issued before the first wait (the code headers whole: 8 KB), 16 waves share
// the loops, and only the words in use are cleared and stored.  With 256
// threads, serial scans and the 66 KB worst case cleared and stored it took
// 11.3 us at 320x240, 12.3 at 3840x2160 and 19.0 at 7680x4320; this form 5.3,
// 6.5 and 9.0.
constexpr int kLayoutThreads = 1024;
constexpr int kLayoutWaves = kLayoutThreads / 64;
constexpr int kMaxSections = 2 + 32 + kMaxAcGroups;

struct LayoutShared {
    std::uint32_t agw[kAcGlobalWords];
    std::uint32_t hw[kHeadWords];
    std::uint32_t ac_bits[kMaxAcGroups];
    std::uint32_t dc_bits[32];
    std::uint32_t piece_off[2 * kNumClusters];
    std::uint32_t pos[kMaxSections];  // section starts, bytes after the head
    std::uint32_t sh[2][2 * kLayoutWaves];
    std::uint32_t ac_global_bits;
};

__device__ __attribute__((always_inline)) inline void layout_kernel_body(
    const Wg& wg, const Geometry& geo, const Constants* __restrict__ k, const CodeSet* __restrict__ cs,
    const std::uint16_t* __restrict__ ac_run_bits, std::uint32_t* __restrict__ chunk_bits, std::uint32_t dc_chunks,
    std::uint32_t* __restrict__ dc_group_bytes, std::uint64_t* __restrict__ dc_group_bits,
    std::uint32_t* __restrict__ ac_group_bytes, std::uint64_t* __restrict__ ac_group_bits, Layout* __restrict__ lay,
    std::uint64_t* __restrict__ ac_base, std::uint64_t* __restrict__ dc_base, std::uint64_t* __restrict__ total_out) {
    __shared__ LayoutShared S;
    const int t{static_cast<int>(threadIdx.x)};
    const int lane{t & 63}, wv{t >> 6};
    // The reads that depend on nothing computed here.
    static_assert(kHeadConstWords <= kLayoutThreads, "one head word per thread");
    static_assert(kNumClusters * kHdrWords == 2 * kLayoutThreads, "two code header words per thread");
    static_assert(2 * kNumClusters == 64, "AcGlobal's pieces fill one wave");
    const std::uint32_t pre_bits{k->ac_prefix_bits};
    const std::uint32_t hb{k->head_bits};
    const std::uint32_t dc_global_bits{k->dc_global_bits};
    const std::uint32_t prefix_w0{k->ac_prefix_words[t]};
    const std::uint32_t head_w0{t < kHeadConstWords ? k->head_words[t] : 0u};
    const std::uint32_t hdr_w[2]{(&cs->hdr[0][0])[t], (&cs->hdr[0][0])[kLayoutThreads + t]};
    const std::uint32_t hdr_len[2]{cs->hdr_bits[t / kHdrWords], cs->hdr_bits[(kLayoutThreads + t) / kHdrWords]};
    const std::uint32_t piece{wv == 0 ? (t < kNumClusters ? cs->alpha[t] : cs->hdr_bits[t - kNumClusters]) : 0u};
    // AC group sizes: the sums of their runs' bits, eight to a 16-byte read.
    for (int g{t}; g < static_cast<int>(geo.num_ac); g += kLayoutThreads) {
        const uint4* const rb{reinterpret_cast<const uint4*>(ac_run_bits + static_cast<std::size_t>(g) * kGroupRuns)};
        std::uint32_t sum{0};
#pragma unroll
        for (int i{0}; i < kGroupRuns / 8; ++i) {
            const uint4 v{rb[i]};
            sum += (v.x & 0xffffu) + (v.x >> 16) + (v.y & 0xffffu) + (v.y >> 16) + (v.z & 0xffffu) + (v.z >> 16) +
                   (v.w & 0xffffu) + (v.w >> 16);
        }
        S.ac_bits[g] = sum;
        ac_group_bits[g] = sum;
        ac_group_bytes[g] = (sum + 7) / 8;
    }
    // DC groups: wave w takes groups 15 - w, 31 - w; the group's chunk sizes
    // become their exclusive prefix sums (the assembly's chunk offsets).  All
    // of a group's sizes (at most kDcRounds per lane) are read at once.
    constexpr int kDcRounds{(kDcMaxChunks + 63) / 64};
    for (int g{kLayoutWaves - 1 - wv}; g < static_cast<int>(geo.num_dc); g += kLayoutWaves) {
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
            S.dc_bits[g] = sum;
            dc_group_bits[g] = sum;
            dc_group_bytes[g] = (sum + 7) / 8;
        }
    }
    // AcGlobal's pieces: alphabet sizes (lanes 0-31), headers (lanes 32-63).
    std::uint32_t alpha_code{0}, alpha_len{0};
    if (wv == 0) {
        if (t < kNumClusters) {
            alpha_len = var_len_u16(piece - 1, alpha_code);
        }
        const std::uint32_t len{t < kNumClusters ? alpha_len : piece};
        const std::uint32_t incl{wave_incl_scan_u32(len)};
        S.piece_off[t] = pre_bits + incl - len;
        if (t == 63) {
            S.ac_global_bits = pre_bits + incl;
        }
    }
    // The head's words in use at most: the constant bits, one bit, padding
    // and 32 bits per TOC entry.
    const bool single{geo.num_ac == 1};
    const std::uint32_t entries{single ? 1u : 2u + geo.num_dc + geo.num_ac};
    const int head_words{min(kHeadWords, static_cast<int>((hb + 8 + 32 * entries + 31) / 32))};
    for (int i{t}; i < head_words; i += kLayoutThreads) {
        const std::uint32_t at{32u * static_cast<std::uint32_t>(i)};
        const std::uint32_t rem{at < hb ? hb - at : 0u};
        S.hw[i] = rem >= 32 ? head_w0 : (head_w0 & ((1u << rem) - 1u));  // constant words: i == t
    }
    __syncthreads();

    // AcGlobal: cleared past the prefix, then the alphabets and headers.
    const std::uint32_t abits{S.ac_global_bits};
    std::uint32_t overflow{abits > static_cast<std::uint32_t>(kAcGlobalWords) * 32 ? 1u : 0u};
    const int ac_words{min(kAcGlobalWords, static_cast<int>((abits + 31) / 32))};
    for (int i{t}; i < ac_words; i += kLayoutThreads) {
        const std::uint32_t at{32u * static_cast<std::uint32_t>(i)};
        const std::uint32_t rem{at < pre_bits ? pre_bits - at : 0u};
        const std::uint32_t w{rem == 0 ? 0u : (i == t ? prefix_w0 : k->ac_prefix_words[i])};
        S.agw[i] = rem >= 32 ? w : (w & ((1u << rem) - 1u));
    }
    // TOC entries, in section order.  Sizes sum below 2^32 (a frame has at
    // most 32 DC groups).
    const Distr toc[4]{{false, 0, 10}, {false, 1024, 14}, {false, 17408, 22}, {false, 4211712, 30}};
    const std::uint32_t dcg{(dc_global_bits + 7) / 8};
    const std::uint32_t acg{(abits + 7) / 8};
    std::uint32_t at{(hb + 1u + 7u) & ~7u};
    std::uint32_t body{0};
    int buf{0};
    for (std::uint32_t e0{0}; e0 < entries; e0 += kLayoutThreads, buf ^= 1) {
        const std::uint32_t e{e0 + static_cast<std::uint32_t>(t)};
        std::uint32_t size{0}, code{0}, clen{0};
        if (e < entries) {
            if (single) {
                size = (dc_global_bits + S.dc_bits[0] + abits + S.ac_bits[0] + 7) / 8;
            } else if (e == 0) {
                size = dcg;
            } else if (e <= geo.num_dc) {
                size = (S.dc_bits[e - 1] + 7) / 8;
            } else if (e == geo.num_dc + 1) {
                size = acg;
            } else {
                size = (S.ac_bits[e - geo.num_dc - 2] + 7) / 8;
            }
            u32_code(toc, size, code, clen);
        }
        std::uint32_t p{clen}, q{size}, chunk_bits_sum{0}, chunk_bytes{0};
        // The barrier inside also orders the clearing above before the ORs.
        block_excl_scan2<kLayoutWaves>(p, q, S.sh[buf], chunk_bits_sum, chunk_bytes);
        if (clen != 0) {
            if (at + p + clen <= static_cast<std::uint32_t>(kHeadWords) * 32) {
                lds_or_bits(S.hw, kHeadWords, at + p, code, clen);
            }
            S.pos[e] = body + q;
        }
        at += chunk_bits_sum;
        body += chunk_bytes;
    }
    if (overflow == 0) {
        if (t < kNumClusters) {
            lds_or_bits(S.agw, kAcGlobalWords, S.piece_off[t], alpha_code, alpha_len);
        }
#pragma unroll
        for (int j{0}; j < 2; ++j) {
            const int idx{j * kLayoutThreads + t};
            const std::uint32_t bit{32u * static_cast<std::uint32_t>(idx % kHdrWords)};
            if (bit < hdr_len[j]) {
                lds_or_bits(S.agw, kAcGlobalWords, S.piece_off[kNumClusters + idx / kHdrWords] + bit, hdr_w[j],
                            hdr_len[j] - bit < 32 ? hdr_len[j] - bit : 32u);
            }
        }
    }
    at = (at + 7) & ~7u;
    if (at > static_cast<std::uint32_t>(kHeadWords) * 32) {
        overflow = 1;
    }
    const std::uint32_t head_bytes{at / 8};
    const std::uint64_t cs_bytes{static_cast<std::uint64_t>(head_bytes) + body};
    const std::uint32_t framing{cs_bytes >= 0x100000000ull - 8 ? 48u : 40u};

    // Section positions (absolute bits in the file).
    const std::uint64_t dcg_bit{(static_cast<std::uint64_t>(framing) + head_bytes) * 8};
    __syncthreads();
    const auto section = [&](std::uint32_t e) { return dcg_bit + static_cast<std::uint64_t>(S.pos[e]) * 8; };
    std::uint64_t ac_global_bit{0};
    if (single) {
        ac_global_bit = dcg_bit + dc_global_bits + S.dc_bits[0];
        if (t == 0) {
            dc_base[0] = dcg_bit + dc_global_bits;
            ac_base[0] = ac_global_bit + abits;
        }
    } else {
        ac_global_bit = section(geo.num_dc + 1);
        if (t < static_cast<int>(geo.num_dc)) {
            dc_base[t] = section(1 + static_cast<std::uint32_t>(t));
        }
        for (std::uint32_t g{static_cast<std::uint32_t>(t)}; g < geo.num_ac; g += kLayoutThreads) {
            ac_base[g] = section(geo.num_dc + 2 + g);
        }
    }
    // Container framing (container.cc:35-54): the 32-byte signature and ftyp
    // box, then the jxlc box header (8 bytes, or 16 with a 64-bit size).
    // Lane i of the last wave forms bytes 4i..4i+3.
    const int fl{t - (kLayoutThreads - 64)};
    if (fl >= 0 && fl < static_cast<int>(framing / 4)) {
        constexpr std::uint32_t sig[8]{0x0c000000u, 0x204c584au, 0x0a870a0du, 0x14000000u,
                                       0x70797466u, 0x206c786au, 0x00000000u, 0x206c786au};
        const bool large{framing == 48};
        const std::uint64_t box{cs_bytes + (large ? 16 : 8)};
        std::uint32_t word{fl < 8 ? sig[fl & 7] : 0u};
        if (fl == 8) {
            word = __builtin_bswap32(large ? 1u : static_cast<std::uint32_t>(box));
        } else if (fl == 9) {
            word = 0x636c786au;  // "jxlc"
        } else if (fl >= 10) {
            word = __builtin_bswap32(static_cast<std::uint32_t>(fl == 10 ? box >> 32 : box));
        }
        lay->framing_words[fl] = word;
    }
    for (int i{t}; i < ac_words; i += kLayoutThreads) {
        lay->ac_global_words[i] = S.agw[i];
    }
    for (int i{t}; i < static_cast<int>((at + 31) / 32) && i < kHeadWords; i += kLayoutThreads) {
        lay->head_words[i] = S.hw[i];
    }
    if (t == 0) {
        lay->ac_global_bits = abits;
        lay->head_total_bits = at;
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

__global__ __launch_bounds__(kLayoutThreads) void layout_kernel(Geometry geo, const Constants* __restrict__ k,
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
                                                                           std::uint64_t cap_bytes,
                                                                           const FileHead& head) {
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
            if (w < head.words) {
                head.to[w] = v;
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
                                                       std::uint64_t cap_bytes, FileHead head) {
    assemble_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, k, lay, P, out_words, cap_bytes, head);
}

}  // namespace cjx
