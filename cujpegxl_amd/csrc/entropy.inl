// Entropy-coding kernels (included into device.hip).
//
// AC: half a wave tokenizes one block-channel (an "item": first-block x
// channel in decoder order Y, X, B), 64 coefficients of the block's scan order
// at a time, classified with ballots: a lane's remaining-non-zero count, the
// serial dependency of the AC context model (entropy.cu:648-681,
// ac_context.h:78-84), comes from popcounts of the ballots below it, so every
// lane forms its tokens in parallel.  One pass writes the token records, their
// counts and the cluster histograms; the emission reads the records.
//
// DC: a DcGroup section is a list of items (header blobs, DC residual tokens,
// AcMetadata tokens), each with a known bit length once the codes exist.  A
// workgroup writes a chunk of 1,024 items at chunk-relative bits into a slot of
// its own, with its bit count; the layout scans the counts and the assembly
// joins the chunks.

namespace cjx {

// Block contexts by (channel in order Y, X, B; coefficient order).
constexpr std::uint8_t kCtxMap[39]{0, 1, 2, 2, 3,  3,  4,  5,  6,  6,  6,  6,  6,
                                   7, 8, 9, 9, 10, 11, 12, 13, 14, 14, 14, 14, 14,
                                   7, 8, 9, 9, 10, 11, 12, 13, 14, 14, 14, 14, 14};

// The clusters (ac_context.h:108-131) put the block contexts below 7 into one
// group and the others into a second: with the transforms in use, the Y items
// are the first group, whatever their transform.
constexpr bool groups_by_channel() {
    for (int row{0}; row < 3; ++row) {
        for (const int ord : {0, 2, 3}) {
            if ((kCtxMap[row * 13 + ord] < 7) != (row == 0)) {
                return false;
            }
        }
    }
    return true;
}
static_assert(groups_by_channel(), "an item's cluster group follows from its channel");

// Cluster of an item's zero-count token: the group's band of the predicted
// count (contexts of 15 blocks per bucket, buckets 8 and up for two counts).
__device__ __forceinline__ std::uint32_t count_cluster(int c, std::uint32_t pred) {
    const std::uint32_t bucket{pred < 8 ? pred : 4 + pred / 2};
    return (c == 1 ? 0u : 4u) + (bucket < 4 ? 0u : (bucket < 12 ? 1u : (bucket < 24 ? 2u : 3u)));
}

// Inclusive prefix sums over the wave by DPP moves (no LDS crossbar): within
// each row of 16 lanes by shifts of 1, 2, 4 and 8 (lanes shifted in from
// outside the row read 0), then the last lane of rows 0 and 2 into rows 1
// and 3 and the last lane of row 1 into rows 2 and 3 (row broadcasts; rows
// the mask leaves out add 0).
template <int kCtrl, int kRowMask>
__device__ __forceinline__ std::uint32_t dpp_u32(std::uint32_t x) {
    return static_cast<std::uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(x), kCtrl, kRowMask, 0xf, kCtrl < 0x140));
}

__device__ __forceinline__ std::uint32_t wave_incl_scan_u32(std::uint32_t x) {
    x += dpp_u32<0x111, 0xf>(x);
    x += dpp_u32<0x112, 0xf>(x);
    x += dpp_u32<0x114, 0xf>(x);
    x += dpp_u32<0x118, 0xf>(x);
    x += dpp_u32<0x142, 0xa>(x);
    return x + dpp_u32<0x143, 0xc>(x);
}

// Sum over the wave, in every lane (the scan's last lane, read as a scalar).
__device__ __forceinline__ int wave_sum_int(int v) {
    return __builtin_amdgcn_readlane(static_cast<int>(wave_incl_scan_u32(static_cast<std::uint32_t>(v))), 63);
}

// Exclusive prefix over the wave.
__device__ __forceinline__ int wave_excl_scan(int v, int lane) {
    (void)lane;
    return static_cast<int>(wave_incl_scan_u32(static_cast<std::uint32_t>(v)) - static_cast<std::uint32_t>(v));
}

// ORs `len` (<= 32) bits at bit `pos` of an LDS word buffer of `cap` words.
__device__ __forceinline__ void lds_or_bits(std::uint32_t* words, std::uint32_t cap, std::uint32_t pos,
                                            std::uint32_t value, std::uint32_t len) {
    if (len == 0) {
        return;
    }
    if (len < 32) {
        value &= (1u << len) - 1u;
    }
    const std::uint32_t wi{pos >> 5}, b{pos & 31u};
    if (wi < cap) {
        atomicOr(&words[wi], value << b);
    }
    if (b + len > 32 && wi + 1 < cap) {
        atomicOr(&words[wi + 1], value >> (32 - b));
    }
}

struct AcItem {
    std::uint32_t head;  // transform side (0: covered) | XYB channel << 6 | count token's cluster << 8 | AC non-zeros << 16
    std::uint32_t at;    // block column | block row << 16

    __device__ __forceinline__ int side() const { return static_cast<int>(head & 63u); }
    __device__ __forceinline__ int channel() const { return static_cast<int>((head >> 6) & 3u); }
    __device__ __forceinline__ std::uint32_t cluster() const { return (head >> 8) & 7u; }
    __device__ __forceinline__ std::uint32_t nonzeros() const { return head >> 16; }
    __device__ __forceinline__ int bx() const { return static_cast<int>(at & 0xffffu); }
    __device__ __forceinline__ int by() const { return static_cast<int>(at >> 16); }
};

// What an item's descriptor is made from, as read: all reads are issued
// before the first is used.
struct ItemReads {
    std::uint32_t pos;
    int c, n;
    std::uint32_t nz, top, left;
    int bx, by;
};

__device__ __forceinline__ ItemReads read_item(const Geometry& geo, const std::int8_t* acs,
                                               const std::uint8_t* nz_grid, const std::uint16_t* nz_count,
                                               std::uint32_t item) {
    ItemReads r;
    r.pos = item / 3u;
    const std::uint32_t ci{item - 3u * r.pos};
    r.c = ci == 0 ? 1 : (ci == 1 ? 0 : 2);
    r.by = static_cast<int>(r.pos / geo.bw);
    r.bx = static_cast<int>(r.pos - static_cast<std::uint32_t>(r.by) * geo.bw);
    const std::uint32_t at{static_cast<std::uint32_t>(r.c) * geo.nblocks + r.pos};
    r.n = acs[r.pos];
    r.nz = nz_count[at];
    r.top = nz_grid[r.by > 0 ? at - geo.bw : at];
    r.left = nz_grid[r.bx > 0 ? at - 1 : at];
    return r;
}

__device__ __forceinline__ AcItem make_item(const ItemReads& r) {
    const bool hl{(r.bx % kAcGroupBlocks) > 0}, ht{(r.by % kAcGroupBlocks) > 0};
    std::uint32_t pred{!hl ? (ht ? r.top : 32u) : (!ht ? r.left : (r.top + r.left + 1) / 2)};
    pred = pred >= 64 ? 64 : pred;
    AcItem it;
    it.head = static_cast<std::uint32_t>(r.n) | (static_cast<std::uint32_t>(r.c) << 6) |
              (count_cluster(r.c, pred) << 8) | (r.nz << 16);
    it.at = static_cast<std::uint32_t>(r.bx) | (static_cast<std::uint32_t>(r.by) << 16);
    return it;
}

// The tokenizer's tables into LDS, 16 bytes a thread.
__device__ __forceinline__ void load_token_tables(TokenTables& T) {
    static_assert(sizeof(TokenTables) % 16 == 0, "whole vectors");
    for (std::uint32_t i{threadIdx.x}; i < sizeof(TokenTables) / 16; i += blockDim.x) {
        reinterpret_cast<uint4*>(&T)[i] = reinterpret_cast<const uint4*>(&g_tables.tokens)[i];
    }
}

// Tokenizes two items per wave, one per 32-lane half (item `it` of this
// lane's half, its coefficients staged in `coef` block after block, so that
// a scan entry's raw index is their index; side 0 for a half without an
// item).  `emit(valid, k, cluster, sym, nbits, extra)` is called once per lane
// per chunk, k being the token's index in the item: 0 for the
// non-zero-count token (lane 0 of the half, first call), then one token per
// scan position from the first non-LLF position up to the last non-zero
// coefficient, so the valid lanes of a chunk are a prefix of the half.  A
// lane's remaining-non-zero count (entropy.cu:648-681, ac_context.h:78-84)
// comes from popcounts of the half's ballot bits below it; the context's
// previous-coefficient flag never changes the cluster.  Two chunks of 32
// positions go side by side: an 8x8 item is one step, and the lookups of a
// longer item's two chunks wait together.
template <typename Emit>
__device__ __forceinline__ void tokenize_item_pair(const TokenTables& T, const std::int16_t* coef, const AcItem& it,
                                                   int lane, Emit&& emit) {
    const int half{lane >> 5}, sub{lane & 31};
    const int n{it.side()};
    const std::uint32_t nz{it.nonzeros()};
    {
        std::uint32_t sym{0}, nb{0}, bits{0};
        hybrid420(nz, sym, nb, bits);
        emit(n != 0 && sub == 0, 0u, it.cluster(), sym, nb, bits);
    }
    const std::uint32_t l2{n == 16 ? 2u : (n == 32 ? 4u : 0u)};
    const std::uint32_t cb{1u << l2};
    const std::uint32_t size{64u << l2};
    const std::uint32_t group{8u + 12u * (it.cluster() >> 2)};
    const std::uint16_t* const scan{n == 32 ? T.scan32 : (n == 16 ? T.scan16 : T.scan8)};
    const std::uint32_t below{(1u << sub) - 1u};
    const auto half_of{[&](std::uint64_t m) {
        return half == 0 ? static_cast<std::uint32_t>(m) : static_cast<std::uint32_t>(m >> 32);
    }};
    std::uint32_t left{n != 0 ? nz : 0u};  // non-zeros not seen yet
    for (std::uint32_t base{cb}; __ballot(left != 0 && base < size) != 0; base += 64) {
        const std::uint32_t k0{base + static_cast<std::uint32_t>(sub)}, k1{k0 + 32};
        const bool on{left != 0}, on0{on && k0 < size}, on1{on && k1 < size};
        const std::uint32_t e0{scan[on0 ? k0 : 0]}, e1{scan[on1 ? k1 : 0]};
        const int c0{coef[e0 & 1023u]}, c1{coef[e1 & 1023u]};
        const int v0{on0 ? c0 : 0}, v1{on1 ? c1 : 0};
        const std::uint32_t m0{half_of(__ballot(v0 != 0))}, m1{half_of(__ballot(v1 != 0))};
        // Non-zeros left at each lane's position.
        const int left0{static_cast<int>(left) - static_cast<int>(__popc(m0 & below))};
        const int left1{static_cast<int>(left) - static_cast<int>(__popc(m0) + __popc(m1 & below))};
        const bool valid0{on0 && left0 > 0}, valid1{on1 && left1 > 0};
        const std::uint32_t r0{valid0 ? (static_cast<std::uint32_t>(left0) + cb - 1) >> l2 : 0u};
        const std::uint32_t r1{valid1 ? (static_cast<std::uint32_t>(left1) + cb - 1) >> l2 : 0u};
        const std::uint32_t band0{T.zero_band[r0 * 32 + (e0 >> 10)]}, band1{T.zero_band[r1 * 32 + (e1 >> 10)]};
        std::uint32_t sym{0}, nb{0}, bits{0};
        hybrid420(pack_signed(v0), sym, nb, bits);
        emit(valid0, 1u + (k0 - cb), group + band0, sym, nb, bits);
        hybrid420(pack_signed(v1), sym, nb, bits);
        emit(valid1, 1u + (k1 - cb), group + band1, sym, nb, bits);
        const std::uint32_t seen{static_cast<std::uint32_t>(__popc(m0) + __popc(m1))};
        left = seen < left ? left - seen : 0u;
    }
}

// Token records: cluster | symbol << 5 | extra-bit count << 13 | extra << 18
// (hybrid-uint extra bits of 16-bit magnitudes fit in 14 bits).  Token k of
// an item lives in the k-th coefficient slot of the item's covered blocks
// (an item has at most 1 + n*n - (n/8)^2 <= n*n tokens).
__device__ __forceinline__ std::uint32_t token_record(std::uint32_t cl, std::uint32_t sym, std::uint32_t nb,
                                                      std::uint32_t extra) {
    return cl | (sym << 5) | (nb << 13) | (extra << 18);
}

__device__ __forceinline__ std::size_t token_slot(const Geometry& geo, int c, int bx, int by, int m,
                                                  std::uint32_t k) {
    const int q{static_cast<int>(k >> 6)};
    const int l2m{m >> 1};  // m in {1, 2, 4}
    return static_cast<std::size_t>(c) * geo.nblocks * 64 +
           (static_cast<std::size_t>(by + (q >> l2m)) * geo.bw + static_cast<std::size_t>(bx + (q & (m - 1)))) * 64 +
           (k & 63u);
}

// Pass 1: tokenize every item once: token records, tokens per item and the
// per-cluster histograms.  AC symbols are below 64 (hybrid-uint tokens of
// 16-bit magnitudes and of counts <= 1024), so each workgroup counts into a
// 32 x 64 LDS histogram and writes it out whole as one partial; a second
// kernel sums the partials.  Grid-stride over item pairs, one wave per pair:
// the descriptors of 32 pairs are loaded at once (one item per lane), and
// each pair's coefficient blocks are read as 16-byte vectors while the
// previous pair is tokenized from its LDS copy.
// What bounds it: the latency of each wave's chain (descriptor, coefficients,
// then per 64 positions two LDS lookups, a ballot, another lookup and the LDS
// atomics), with the four workgroups per CU that 37 KB of LDS leave room for:
// three take 7 % longer at 7680x4320, two 32 %; one histogram copy (five
// workgroups) 15 %, more copies of the low symbols only 6 %.  So the first
// descriptors and coefficients are read while the tables are set up, the
// context lookups are one byte per (non-zeros left, frequency), an item's
// descriptor is two words to pass between lanes, and a step takes 64
// positions.  320x240 16.0 -> 11.0 us, 3840x2160 36.5 -> 28.5, 7680x4320 132
// -> 80.
constexpr int kAcSymbols = 64;
// LDS row stride of a cluster's histogram: one word more than the symbols,
// so equal symbols of different clusters fall in different banks.
constexpr int kHistRow = kAcSymbols + 1;
// Two copies of the histogram, taken by even and odd lanes (neighbouring
// lanes often carry the same cluster and symbol); the second starts 16
// banks after the first, so one key's two words sit in different banks.
constexpr int kHistCopy = kNumClusters * kHistRow + 16;
constexpr int kTokenGrid = 2048;
constexpr int kTokenBatch = 32;
constexpr std::uint32_t kTokenThreads = 256;

// Workgroups that leave every wave a pair of items.
inline std::uint32_t token_workgroups(const Geometry& geo) {
    constexpr std::uint32_t kItems{2 * kTokenThreads / 64};
    return (3 * geo.nblocks + kItems - 1) / kItems;
}

__device__ __forceinline__ AcItem shfl_item(const AcItem& d, int src) {
    return AcItem{static_cast<std::uint32_t>(__shfl(static_cast<int>(d.head), src, 64)),
                  static_cast<std::uint32_t>(__shfl(static_cast<int>(d.at), src, 64))};
}

// The m x m coefficient blocks of an item (m = n / 8; 8 to 128 vectors of
// 16 bytes), lane `sub` of the half taking vectors sub, sub + 32, sub + 64
// and sub + 96 (four named registers, so the set never goes to scratch).
struct ItemVecs {
    uint4 r0, r1, r2, r3;
};

__device__ __forceinline__ int item_vecs(int n) {
    return n == 32 ? 128 : (n == 16 ? 32 : (n == 8 ? 8 : 0));
}

__device__ __forceinline__ uint4 load_item_vec(const std::int16_t* plane, const Geometry& geo, const AcItem& it,
                                               int l2s, int u) {
    const int q{u >> 3};
    const std::size_t blk{static_cast<std::size_t>(it.by() + (q >> l2s)) * geo.bw +
                          static_cast<std::size_t>(it.bx() + (q & ((1 << l2s) - 1)))};
    return *reinterpret_cast<const uint4*>(plane + blk * 64 + (u & 7) * 8);
}

__device__ __forceinline__ void load_item_coefs(const Geometry& geo, const std::int16_t* ac, const AcItem& it,
                                                int sub, ItemVecs& v) {
    const int l2s{it.side() == 32 ? 2 : (it.side() == 16 ? 1 : 0)};
    const int vecs{item_vecs(it.side())};
    const std::int16_t* plane{ac + static_cast<std::size_t>(it.channel()) * geo.nblocks * 64};
    if (sub < vecs) {
        v.r0 = load_item_vec(plane, geo, it, l2s, sub);
    }
    if (sub + 32 < vecs) {
        v.r1 = load_item_vec(plane, geo, it, l2s, sub + 32);
        v.r2 = load_item_vec(plane, geo, it, l2s, sub + 64);
        v.r3 = load_item_vec(plane, geo, it, l2s, sub + 96);
    }
}

__device__ __forceinline__ void store_item_coefs(std::int16_t* coef, const AcItem& it, int sub, const ItemVecs& v) {
    const int vecs{item_vecs(it.side())};
    if (sub < vecs) {
        *reinterpret_cast<uint4*>(coef + sub * 8) = v.r0;
    }
    if (sub + 32 < vecs) {
        *reinterpret_cast<uint4*>(coef + (sub + 32) * 8) = v.r1;
        *reinterpret_cast<uint4*>(coef + (sub + 64) * 8) = v.r2;
        *reinterpret_cast<uint4*>(coef + (sub + 96) * 8) = v.r3;
    }
}

// An item's own index: block * 3 + (0: Y, 1: X, 2: B).
__device__ __forceinline__ std::uint32_t item_index(const Geometry& geo, const AcItem& it) {
    return (static_cast<std::uint32_t>(it.by()) * geo.bw + static_cast<std::uint32_t>(it.bx())) * 3u +
           (it.channel() == 1 ? 0u : (it.channel() == 0 ? 1u : 2u));
}

__device__ __attribute__((always_inline)) inline void ac_tokens_kernel_body(const Wg& wg, Geometry geo, const std::int16_t* __restrict__ ac,
                                                        const std::int8_t* __restrict__ acs,
                                                        const std::uint8_t* __restrict__ nz_grid,
                                                        const std::uint16_t* __restrict__ nz_count,
                                                        std::uint32_t* __restrict__ tokens,
                                                        std::uint16_t* __restrict__ item_tokens,
                                                        std::uint32_t* __restrict__ partial,
                                                        const std::uint32_t* __restrict__ list,
                                                        const std::uint32_t* __restrict__ list_count) {
    __shared__ __align__(16) std::uint32_t h2[2 * kHistCopy];
    __shared__ TokenTables T;
    __shared__ __align__(16) std::int16_t stage[kTokenThreads / 64][2][1024];
    const int lane{static_cast<int>(threadIdx.x) & 63};
    const int half{lane >> 5}, sub{lane & 31};
    std::uint32_t* const h{h2 + (lane & 1) * kHistCopy};
    std::int16_t* const coef{stage[threadIdx.x >> 6][half]};
    const std::uint32_t wave{wg.x * (kTokenThreads / 64) + (threadIdx.x >> 6)};
    const std::uint32_t stride{2 * wg.nx * (kTokenThreads / 64)};
    // The list of items with non-zeros from the quantizer when there is one
    // (covered blocks' items already have 0 tokens), else every item; at the
    // list's end the first blocks' items without non-zeros.  The wave's first
    // items and the thread's first item without non-zeros are read while the
    // tables are set up: entries past the list's ends are read too (they are
    // in the buffer), but not used.
    const std::uint32_t all{3u * geo.nblocks}, last{all - 1u};
    const auto item_at{[&](std::uint32_t base) {
        return base + stride * static_cast<std::uint32_t>(lane >> 1) + static_cast<std::uint32_t>(lane & 1);
    }};
    const std::uint32_t li{item_at(2 * wave)};
    const std::uint32_t zi{wg.x * kTokenThreads + threadIdx.x};
    std::uint32_t first{li}, zero{0};
    std::uint32_t items{all}, zeros{0};
    if (list != nullptr) {
        items = list_count[0];
        zeros = list_count[1];
        first = list[li < all ? li : 0u];
        zero = list[zi < all ? last - zi : 0u];
    }
    for (std::uint32_t i{threadIdx.x}; i < 2 * kHistCopy / 4; i += kTokenThreads) {
        reinterpret_cast<uint4*>(h2)[i] = uint4{0, 0, 0, 0};
    }
    static_assert(2 * kHistCopy % 4 == 0, "whole vectors");
    const ItemReads first_reads{read_item(geo, acs, nz_grid, nz_count, li < items ? first : 0u)};
    const ItemReads zero_reads{read_item(geo, acs, nz_grid, nz_count, zi < zeros ? zero : 0u)};
    load_token_tables(T);
    AcItem d{make_item(first_reads)};
    d.head = li < items ? d.head : 0u;
    AcItem cur{shfl_item(d, half)};
    ItemVecs v{};
    load_item_coefs(geo, ac, cur, sub, v);
    __syncthreads();
    // First blocks without non-zero coefficients, one per thread: their one
    // token is the zero count, in the count's context.
    {
        AcItem it{make_item(zero_reads)};
        for (std::uint32_t i{zi}; i < zeros; i += wg.nx * kTokenThreads) {
            if (i != zi) {
                it = make_item(read_item(geo, acs, nz_grid, nz_count, list[last - i]));
            }
            std::uint32_t sym{0}, nb{0}, bits{0};
            hybrid420(0u, sym, nb, bits);
            atomicAdd(&h[it.cluster() * kHistRow + (sym & (kAcSymbols - 1))], 1u);
            tokens[token_slot(geo, it.channel(), it.bx(), it.by(), 1, 0)] = token_record(it.cluster(), sym, nb, bits);
            item_tokens[item_index(geo, it)] = 1;
        }
    }
    for (std::uint32_t base{2 * wave}; base < items; base += stride * kTokenBatch) {
        if (base != 2 * wave) {
            const std::uint32_t i{item_at(base)};
            const ItemReads r{read_item(geo, acs, nz_grid, nz_count, i < items ? (list != nullptr ? list[i] : i) : 0u)};
            d = make_item(r);
            d.head = i < items ? d.head : 0u;
            cur = shfl_item(d, half);
            load_item_coefs(geo, ac, cur, sub, v);
        }
        const int npairs{static_cast<int>(min(static_cast<std::uint32_t>(kTokenBatch),
                                              (items - base + stride - 1) / stride))};
        for (int t{0}; t < npairs; ++t) {
            const std::uint32_t item{base + stride * static_cast<std::uint32_t>(t) + static_cast<std::uint32_t>(half)};
            wave_sync();
            store_item_coefs(coef, cur, sub, v);
            wave_sync();
            AcItem nx{};
            if (t + 1 < npairs) {
                nx = shfl_item(d, 2 * (t + 1) + half);
                load_item_coefs(geo, ac, nx, sub, v);
            }
            std::uint32_t count{0};
            if (__ballot(cur.side() != 0) != 0) {
                const AcItem it{cur};
                const std::uint32_t l2m{it.side() == 32 ? 2u : (it.side() == 16 ? 1u : 0u)};
                const std::uint32_t m{1u << l2m};
                // token_slot in 32 bits (3 * blocks * 64 < 2^32 for the
                // at most 32 DC groups a frame may have).
                const std::uint32_t slot0{static_cast<std::uint32_t>(
                    token_slot(geo, it.channel(), it.bx(), it.by(), 1, 0))};
                const std::uint32_t row{geo.bw * 64};
                tokenize_item_pair(T, coef, it, lane,
                                   [&](bool valid, std::uint32_t k, std::uint32_t cl, std::uint32_t sym,
                                       std::uint32_t nb, std::uint32_t extra) {
                                       if (valid) {
                                           atomicAdd(&h[cl * kHistRow + (sym & (kAcSymbols - 1))], 1u);
                                           const std::uint32_t q{k >> 6};
                                           tokens[slot0 + (q >> l2m) * row + ((q & (m - 1)) << 6) + (k & 63u)] =
                                               token_record(cl, sym, nb, extra);
                                       }
                                       const std::uint64_t ballot{__ballot(valid)};
                                       count += static_cast<std::uint32_t>(
                                           __popc(half == 0 ? static_cast<std::uint32_t>(ballot)
                                                            : static_cast<std::uint32_t>(ballot >> 32)));
                                   });
            }
            if (sub == 0 && item < items) {
                item_tokens[item_index(geo, cur)] = static_cast<std::uint16_t>(count);
            }
            cur = nx;
        }
    }
    __syncthreads();
    std::uint32_t* mine{partial + static_cast<std::size_t>(wg.x) * kNumClusters * kAcSymbols};
    for (int i{static_cast<int>(threadIdx.x)}; i < kNumClusters * kAcSymbols; i += kTokenThreads) {
        const int r{(i >> 6) * kHistRow + (i & (kAcSymbols - 1))};
        mine[i] = h2[r] + h2[kHistCopy + r];
    }
}

__global__ __launch_bounds__(kTokenThreads) void ac_tokens_kernel(Geometry geo, const std::int16_t* __restrict__ ac,
                                                        const std::int8_t* __restrict__ acs,
                                                        const std::uint8_t* __restrict__ nz_grid,
                                                        const std::uint16_t* __restrict__ nz_count,
                                                        std::uint32_t* __restrict__ tokens,
                                                        std::uint16_t* __restrict__ item_tokens,
                                                        std::uint32_t* __restrict__ partial,
                                                        const std::uint32_t* __restrict__ list,
                                                        const std::uint32_t* __restrict__ list_count) {
    ac_tokens_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, ac, acs, nz_grid, nz_count, tokens, item_tokens, partial, list, list_count);
}

// Sums `parts` partial histograms of 32 x 64 bins into the 32 x 256 cluster
// histograms: grid (bins / 256, slices); each thread adds its slice.
__device__ __forceinline__ void ac_hist_reduce_body(const Wg& wg, const std::uint32_t* __restrict__ partial, int parts,
                                                    std::uint32_t* __restrict__ hist) {
    const int bin{static_cast<int>(wg.x) * 256 + static_cast<int>(threadIdx.x)};
    const int per{(parts + static_cast<int>(wg.ny) - 1) / static_cast<int>(wg.ny)};
    const int p0{static_cast<int>(wg.y) * per};
    const int p1{min(parts, p0 + per)};
    std::uint32_t sum{0};
    for (int p{p0}; p < p1; ++p) {
        sum += partial[static_cast<std::size_t>(p) * kNumClusters * kAcSymbols + bin];
    }
    if (sum != 0) {
        atomicAdd(&hist[(bin / kAcSymbols) * kHistStride + bin % kAcSymbols], sum);
    }
}

// Exclusive scan of one value per thread over a workgroup of kWaves waves:
// the waves' totals go through `sh` (kWaves words), every thread adds those of
// the waves below its own.  `sh` must not be in use by a scan that a thread
// may still read (callers alternate two buffers, or have a barrier between).
template <int kWaves>
__device__ __forceinline__ std::uint32_t block_excl_scan_u32(std::uint32_t v, std::uint32_t* sh,
                                                             std::uint32_t& total) {
    const int lane{static_cast<int>(threadIdx.x) & 63}, wv{static_cast<int>(threadIdx.x) >> 6};
    const std::uint32_t x{wave_incl_scan_u32(v)};
    if (lane == 63) {
        sh[wv] = x;
    }
    __syncthreads();
    std::uint32_t base{0};
    total = 0;
#pragma unroll
    for (int i{0}; i < kWaves; ++i) {
        const std::uint32_t t{sh[i]};
        base += i < wv ? t : 0u;
        total += t;
    }
    return base + x - v;
}

// ---- AC groups emitted in runs ------------------------------------------------
//
// An AC group is cut into eight bands of four block rows (which the
// transforms never cross), and a band's tokens, in decoder order (block rows,
// blocks left to right, channels Y, X, B), into runs of kRunTokens.  Each run
// is written at run-relative bit positions into a staging slot of its own,
// with its bit count; the assembly reads the runs back to back.  `band_wgs`
// workgroups of 256 threads share a band: each numbers the band's tokens (a
// scan over its items' counts, items without tokens dropped) and takes runs
// j, j + band_wgs, ...: a thread finds its first token's item by a binary
// search, reads eight consecutive tokens and their codes, a block scan of
// the lengths gives the positions, and the stream is assembled in LDS.
//
// The work is a chain of latencies (counts, scan, search, token reads, scan,
// LDS atomics: about 12,000 clocks a run), so the runs of a band go to
// different workgroups instead of one after another, and the walk over a
// thread's tokens meets no item without tokens (up to 96 in a row where
// every transform is larger than 8x8).  One workgroup per band with all items
// kept took 27 us at 320x240 and 35 us at 3840x2160; this form 8.4 and 25 us.
constexpr int kGroupBands = 8;
constexpr int kBandRows = kAcGroupBlocks / kGroupBands;
constexpr int kBandItems = 3 * kAcGroupBlocks * kBandRows;
constexpr int kEmitThreads = 256;
constexpr int kPerThread = 8;
constexpr int kRunTokens = kEmitThreads * kPerThread;
// A band has at most one token per coefficient slot.
constexpr int kBandRuns = (kBandItems * 64 + kRunTokens - 1) / kRunTokens;
constexpr int kGroupRuns = kGroupBands * kBandRuns;
// A token is at most 28 bits (15-bit code, 13 extra bits).
constexpr int kRunWords = kRunTokens * 28 / 32;
static_assert(kRunWords * 32 < 65536, "a run's bit count fits 16 bits");
static_assert(kBandItems * 64 < 65536, "a band's token count fits 16 bits");
static_assert(kBandItems <= 2 * kEmitThreads, "two items per thread");
static_assert(kGroupRuns * sizeof(std::uint16_t) % 16 == 0, "16-byte reads of a group's run sizes");

struct GroupShared {
    std::uint32_t lut[kNumClusters * kAcSymbols];  // depth | code << 16
    // Items with tokens: {first token's number, token slot | log2(side / 8)
    // (a slot is a multiple of 64)}; one more entry ends the numbering.
    uint2 item[kBandItems + 1];
    std::uint32_t buf[kRunWords];
    std::uint32_t sh[2][kEmitThreads / 64];
};

__device__ __forceinline__ void ac_group_emit_body(
    GroupShared& S, const Wg& wg, const Geometry& geo, const std::int8_t* __restrict__ acs,
    const std::uint16_t* __restrict__ item_tokens, const std::uint32_t* __restrict__ tokens,
    const std::uint32_t* __restrict__ lut, std::uint32_t* __restrict__ staging,
    std::uint16_t* __restrict__ run_bits_out, int band_wgs) {
    const int tid{static_cast<int>(threadIdx.x)};
    const int g{static_cast<int>(wg.x) / (kGroupBands * band_wgs)};
    const int band{static_cast<int>(wg.x) / band_wgs % kGroupBands};
    const int first{static_cast<int>(wg.x) % band_wgs};
    const int bx0{(g % static_cast<int>(geo.xg)) * kAcGroupBlocks};
    const int by0{(g / static_cast<int>(geo.xg)) * kAcGroupBlocks + band * kBandRows};
    const int gbw{min(kAcGroupBlocks, static_cast<int>(geo.bw) - bx0)};
    const int gbh{min(kBandRows, static_cast<int>(geo.bh) - by0)};
    const int items{gbh > 0 ? 3 * gbw * gbh : 0};
    const std::size_t run0{(static_cast<std::size_t>(g) * kGroupBands + band) * kBandRuns};

    // 1. The band's items with tokens, and their token numbers.  Every read
    //    (the items' transforms and token counts, the code table) is issued
    //    before the first wait; a covered block's count is read too and then
    //    taken as 0.
    int item_n[2]{0, 0};
    std::uint32_t item_cnt[2]{0u, 0u}, item_slot[2]{0u, 0u};
#pragma unroll
    for (int k{0}; k < 2; ++k) {
        const int i{2 * tid + k};
        if (i < items) {
            const int row{i / (3 * gbw)}, rem{i % (3 * gbw)};
            const int ci{rem % 3};
            const std::size_t pos{static_cast<std::size_t>(by0 + row) * geo.bw + bx0 + rem / 3};
            item_n[k] = acs[pos];
            item_cnt[k] = item_tokens[pos * 3 + ci];
            item_slot[k] = static_cast<std::uint32_t>(
                token_slot(geo, ci == 0 ? 1 : (ci == 1 ? 0 : 2), bx0 + rem / 3, by0 + row, 1, 0));
        }
    }
    static_assert(kNumClusters * kAcSymbols == 2 * 4 * kEmitThreads, "two 16-byte reads of the code table");
    const uint4 code0{reinterpret_cast<const uint4*>(lut)[tid]};
    const uint4 code1{reinterpret_cast<const uint4*>(lut)[kEmitThreads + tid]};
    std::uint32_t packed{0};  // tokens | items with tokens << 16
#pragma unroll
    for (int k{0}; k < 2; ++k) {
        item_cnt[k] = item_n[k] != 0 ? item_cnt[k] : 0u;
        packed += item_cnt[k] + (item_cnt[k] != 0 ? 0x10000u : 0u);
    }
    std::uint32_t total{0};
    std::uint32_t at{block_excl_scan_u32<kEmitThreads / 64>(packed, S.sh[0], total)};
#pragma unroll
    for (int k{0}; k < 2; ++k) {
        if (item_cnt[k] != 0) {
            S.item[at >> 16] = uint2{at & 0xffffu, item_slot[k] | static_cast<std::uint32_t>(item_n[k] >> 4)};
            at += item_cnt[k] + 0x10000u;
        }
    }
    const std::uint32_t ntok{total & 0xffffu};
    const int nitems{static_cast<int>(total >> 16)};
    if (tid == 0) {
        S.item[nitems] = uint2{ntok, 0u};
    }
    reinterpret_cast<uint4*>(S.lut)[tid] = code0;
    reinterpret_cast<uint4*>(S.lut)[kEmitThreads + tid] = code1;

    // 2. The runs.
    for (int r{first}; r < kBandRuns; r += band_wgs) {
        const std::uint32_t f0{static_cast<std::uint32_t>(r) * kRunTokens};
        if (f0 >= ntok) {
            if (tid == 0) {
                run_bits_out[run0 + r] = 0;
            }
            continue;
        }
        __syncthreads();  // the items are in LDS; the last run's words have been stored
        for (int i{tid}; i < kRunWords; i += kEmitThreads) {
            S.buf[i] = 0;
        }
        const std::uint32_t fb{f0 + static_cast<std::uint32_t>(tid) * kPerThread};
        std::uint32_t rec[kPerThread];
        int lo{0};
        if (fb < ntok) {
            int hi{nitems - 1};
            while (lo < hi) {
                const int mid{(lo + hi + 1) >> 1};
                if (S.item[mid].x <= fb) {
                    lo = mid;
                } else {
                    hi = mid - 1;
                }
            }
        }
        uint2 cur{S.item[lo]};
        std::uint32_t next{S.item[lo + 1].x};
#pragma unroll
        for (int j{0}; j < kPerThread; ++j) {
            const std::uint32_t f{fb + static_cast<std::uint32_t>(j)};
            rec[j] = 0xffffffffu;
            if (f < ntok) {
                if (f >= next) {  // every item has a token: at most one step
                    ++lo;
                    cur = S.item[lo];
                    next = S.item[lo + 1].x;
                }
                const std::uint32_t k{f - cur.x};
                const std::uint32_t l2m{cur.y & 63u};
                const std::uint32_t q{k >> 6};
                rec[j] = tokens[(cur.y & ~63u) + (q >> l2m) * (geo.bw * 64) + ((q & ((1u << l2m) - 1u)) << 6) +
                                (k & 63u)];
            }
        }
        std::uint32_t len[kPerThread], val[kPerThread];
        std::uint32_t sum{0};
#pragma unroll
        for (int j{0}; j < kPerThread; ++j) {
            len[j] = 0;
            val[j] = 0;
            const std::uint32_t rc{rec[j]};
            if (rc != 0xffffffffu) {
                const std::uint32_t e{S.lut[(rc & 31u) * kAcSymbols + ((rc >> 5) & (kAcSymbols - 1))]};
                const std::uint32_t d{e & 0xffffu};
                len[j] = d + ((rc >> 13) & 31u);
                val[j] = ((e >> 16) | ((rc >> 18) << d)) & ((1u << len[j]) - 1u);
            }
            sum += len[j];
        }
        std::uint32_t bits{0};
        // The barrier inside also orders the clearing of S.buf before the ORs.
        std::uint32_t pos{block_excl_scan_u32<kEmitThreads / 64>(sum, S.sh[1], bits)};
#pragma unroll
        for (int j{0}; j < kPerThread; ++j) {
            if (len[j] != 0) {
                const std::uint32_t wi{pos >> 5}, b{pos & 31u};
                atomicOr(&S.buf[wi], val[j] << b);
                if (b + len[j] > 32) {
                    atomicOr(&S.buf[wi + 1], val[j] >> (32 - b));
                }
            }
            pos += len[j];
        }
        __syncthreads();
        std::uint32_t* const slot{staging + (run0 + r) * kRunWords};
        const int nw{static_cast<int>((bits + 31) / 32)};
        for (int i{tid}; i < nw; i += kEmitThreads) {
            slot[i] = S.buf[i];
        }
        if (tid == 0) {
            run_bits_out[run0 + r] = static_cast<std::uint16_t>(bits);
        }
    }
}

// ---- DC groups -------------------------------------------------------------

// Item kinds of a DcGroup section, in order (vardct_frame.cc:543-554):
//   0: blob_pre | [0,3n): DC residuals, channels Y, X, B, group raster |
//   blob_mid | meta: YtoX (cw*ch), YtoB (cw*ch), strategy per block (first
//   blocks only), quant field per block (first blocks only), EPF zeros (n).
struct DcGroupGeo {
    int bx0, by0, dgw, dgh, n, cw, ch;
    std::uint32_t items;
};

__device__ __forceinline__ DcGroupGeo dc_group_geo(const Geometry& geo, int g) {
    DcGroupGeo d{};
    d.bx0 = (g % static_cast<int>(geo.xdg)) * 256;
    d.by0 = (g / static_cast<int>(geo.xdg)) * 256;
    d.dgw = min(256, static_cast<int>(geo.bw) - d.bx0);
    d.dgh = min(256, static_cast<int>(geo.bh) - d.by0);
    d.n = d.dgw * d.dgh;
    d.cw = (d.dgw + 7) / 8;
    d.ch = (d.dgh + 7) / 8;
    d.items = static_cast<std::uint32_t>(2 + 6 * d.n + 2 * d.cw * d.ch);
    return d;
}

// dc_predict.h:22-49
__device__ __forceinline__ std::int32_t gradient_predict(bool hl, bool ht, std::int32_t wv,
                                                         std::int32_t nv, std::int32_t nwv) {
    const std::int32_t left{hl ? wv : (ht ? nv : 0)};
    const std::int32_t top{ht ? nv : left};
    const std::int32_t tl{(hl && ht) ? nwv : left};
    const std::int32_t lo{left < top ? left : top}, hi{left < top ? top : left};
    if (tl < lo) {
        return hi;
    }
    if (tl > hi) {
        return lo;
    }
    return static_cast<std::int32_t>(static_cast<std::int64_t>(left) + top - tl);
}

// Walks the items of a DcGroup section in order.  Sections: 0 blob_pre,
// 1 DC residuals (channel ci, block x, y), 2 blob_mid, 3 YtoX and 4 YtoB
// (tile x, y), 5 strategy and 6 quant field (block x, y), 7 EPF zeros.
// Positioning at item k divides once; advancing is incremental.
struct DcCursor {
    int sec, ci, x, y;
};

__device__ __forceinline__ DcCursor dc_cursor_at(const DcGroupGeo& d, std::uint32_t k) {
    DcCursor c{};
    const std::uint32_t n{static_cast<std::uint32_t>(d.n)};
    const std::uint32_t cwch{static_cast<std::uint32_t>(d.cw * d.ch)};
    if (k == 0) {
        c.sec = 0;
    } else if (k < 1 + 3 * n) {
        const std::uint32_t i{k - 1};
        const std::uint32_t p{i % n};
        c.sec = 1;
        c.ci = static_cast<int>(i / n);
        c.x = static_cast<int>(p % static_cast<std::uint32_t>(d.dgw));
        c.y = static_cast<int>(p / static_cast<std::uint32_t>(d.dgw));
    } else if (k == 1 + 3 * n) {
        c.sec = 2;
    } else {
        const std::uint32_t j{k - (2 + 3 * n)};
        if (j < 2 * cwch) {
            const std::uint32_t jj{j < cwch ? j : j - cwch};
            c.sec = j < cwch ? 3 : 4;
            c.x = static_cast<int>(jj % static_cast<std::uint32_t>(d.cw));
            c.y = static_cast<int>(jj / static_cast<std::uint32_t>(d.cw));
        } else if (j < 2 * cwch + 2 * n) {
            const std::uint32_t jj{(j - 2 * cwch) % n};
            c.sec = j < 2 * cwch + n ? 5 : 6;
            c.x = static_cast<int>(jj % static_cast<std::uint32_t>(d.dgw));
            c.y = static_cast<int>(jj / static_cast<std::uint32_t>(d.dgw));
        } else {
            c.sec = 7;
        }
    }
    return c;
}

__device__ __forceinline__ void dc_cursor_next(const DcGroupGeo& d, DcCursor& c) {
    switch (c.sec) {
        case 0:
        case 2:
            ++c.sec;
            c.ci = 0;
            c.x = 0;
            c.y = 0;
            break;
        case 1:
            if (++c.x == d.dgw) {
                c.x = 0;
                if (++c.y == d.dgh) {
                    c.y = 0;
                    if (++c.ci == 3) {
                        c.sec = 2;
                    }
                }
            }
            break;
        case 3:
        case 4:
            if (++c.x == d.cw) {
                c.x = 0;
                if (++c.y == d.ch) {
                    c.y = 0;
                    ++c.sec;
                }
            }
            break;
        case 5:
        case 6:
            if (++c.x == d.dgw) {
                c.x = 0;
                if (++c.y == d.dgh) {
                    c.y = 0;
                    ++c.sec;
                }
            }
            break;
        default:
            break;
    }
}

// Token of the cursor's item (sections 1 and 3-7).  Returns 0 for a DC code,
// 1 for an AcMetadata code, 2 for an absent item (a covered block's
// strategy / quant-field slot).
__device__ __forceinline__ int dc_cursor_token(const Geometry& geo, const DcGroupGeo& d, const DcCursor& c,
                                               const std::int32_t* dc, const std::int8_t* acs,
                                               const std::int32_t* qf, const std::int8_t* ytox,
                                               const std::int8_t* ytob, std::uint32_t& sym, std::uint32_t& nb,
                                               std::uint32_t& bits) {
    if (c.sec == 1) {
        const int ch{c.ci == 0 ? 1 : (c.ci == 1 ? 0 : 2)};
        const std::int32_t* pl{dc + static_cast<std::size_t>(ch) * geo.nblocks};
        const std::size_t b{static_cast<std::size_t>(d.by0 + c.y) * geo.bw + d.bx0 + c.x};
        const bool hl{c.x > 0}, ht{c.y > 0};
        const std::int32_t pred{gradient_predict(hl, ht, hl ? pl[b - 1] : 0, ht ? pl[b - geo.bw] : 0,
                                                 (hl && ht) ? pl[b - geo.bw - 1] : 0)};
        hybrid420(pack_signed(pl[b] - pred), sym, nb, bits);
        return 0;
    }
    std::int32_t v{0};
    if (c.sec == 3 || c.sec == 4) {
        const std::size_t t{static_cast<std::size_t>(d.by0 / 8 + c.y) * geo.cmw + d.bx0 / 8 + c.x};
        v = c.sec == 3 ? ytox[t] : ytob[t];
    } else if (c.sec == 5 || c.sec == 6) {
        const std::size_t b{static_cast<std::size_t>(d.by0 + c.y) * geo.bw + d.bx0 + c.x};
        const int side{acs[b]};
        if (side == 0) {
            return 2;
        }
        v = c.sec == 5 ? (side == 16 ? 4 : (side == 32 ? 5 : 0)) : qf[b] - 1;
    }
    hybrid420(pack_signed(v), sym, nb, bits);
    return 1;
}

constexpr int kDcChunk = 1024;               // items per workgroup in the DC passes
constexpr int kDcPerThread = kDcChunk / 256;  // consecutive items per thread
// Chunks of the largest DC group (256 x 256 blocks).
constexpr int kDcMaxChunks = (2 + 6 * 65536 + 2 * 1024 + kDcChunk - 1) / kDcChunk;
// Staging slot of one chunk: every item's token is at most 32 bits, plus the
// two header blobs.
constexpr int kBlobWords = 128;
constexpr int kDcSlotWords = kDcChunk + 2 * kBlobWords;

// DC and AcMetadata token histograms per group, plus the first-block count.
__device__ __forceinline__ void dc_hist_body(const Wg& wg, const Geometry& geo, const std::int32_t* __restrict__ dc,
                                             const std::int8_t* __restrict__ acs, const std::int32_t* __restrict__ qf,
                                             const std::int8_t* __restrict__ ytox,
                                             const std::int8_t* __restrict__ ytob,
                                             std::uint32_t* __restrict__ dc_hist, std::uint32_t* __restrict__ meta_hist,
                                             std::uint32_t* __restrict__ fb_count) {
    __shared__ std::uint32_t h[2 * kHistStride];
    __shared__ std::uint32_t cnt;
    const int g{static_cast<int>(wg.y)};
    const DcGroupGeo d{dc_group_geo(geo, g)};
    for (int i{static_cast<int>(threadIdx.x)}; i < 2 * kHistStride; i += 256) {
        h[i] = 0;
    }
    if (threadIdx.x == 0) {
        cnt = 0;
    }
    __syncthreads();
    // Lane-strided items (neighbouring lanes read neighbouring blocks); the
    // histogram does not depend on the order.
    const std::uint32_t k0{wg.x * kDcChunk};
    const std::uint32_t k1{min(k0 + static_cast<std::uint32_t>(kDcChunk), d.items)};
    std::uint32_t fb{0};
    for (std::uint32_t k{k0 + threadIdx.x}; k < k1; k += 256) {
        const DcCursor c{dc_cursor_at(d, k)};
        if (c.sec == 0 || c.sec == 2) {
            continue;
        }
        std::uint32_t sym, nb, bits;
        const int kind{dc_cursor_token(geo, d, c, dc, acs, qf, ytox, ytob, sym, nb, bits)};
        if (kind != 2) {
            atomicAdd(&h[(kind == 0 ? 0 : kHistStride) + static_cast<int>(sym)], 1u);
            fb += (kind == 1 && c.sec == 5) ? 1u : 0u;
        }
    }
    if (fb != 0) {
        atomicAdd(&cnt, fb);
    }
    __syncthreads();
    for (int i{static_cast<int>(threadIdx.x)}; i < kHistStride; i += 256) {
        if (h[i]) {
            atomicAdd(&dc_hist[g * kHistStride + i], h[i]);
        }
        if (h[kHistStride + i]) {
            atomicAdd(&meta_hist[g * kHistStride + i], h[kHistStride + i]);
        }
    }
    if (threadIdx.x == 0 && cnt) {
        atomicAdd(&fb_count[g], cnt);
    }
}

// The partial AC histograms' sum and the DC groups' histograms in one launch
// (independent work, a few microseconds each): workgroups below
// kReduceWgs reduce, the others take one chunk of one DC group each.
constexpr std::uint32_t kReduceBins = kNumClusters * kAcSymbols / 256;
constexpr std::uint32_t kReduceSlices = 80;
constexpr std::uint32_t kReduceWgs = kReduceBins * kReduceSlices;

__device__ __forceinline__ void histograms_kernel_body(const Wg& wg, const Geometry& geo, std::uint32_t dc_chunks,
                                                       const std::uint32_t* __restrict__ partial, int parts,
                                                       std::uint32_t* __restrict__ hists,
                                                       const std::int32_t* __restrict__ dc,
                                                       const std::int8_t* __restrict__ acs,
                                                       const std::int32_t* __restrict__ qf,
                                                       const std::int8_t* __restrict__ ytox,
                                                       const std::int8_t* __restrict__ ytob,
                                                       std::uint32_t* __restrict__ fb_count) {
    if (wg.x < kReduceWgs) {
        ac_hist_reduce_body(Wg{wg.x % kReduceBins, wg.x / kReduceBins, kReduceBins, kReduceSlices}, partial, parts,
                            hists);
    } else {
        const std::uint32_t i{wg.x - kReduceWgs};
        dc_hist_body(Wg{i % dc_chunks, i / dc_chunks, dc_chunks, geo.num_dc}, geo, dc, acs, qf, ytox, ytob,
                     hists + kNumClusters * kHistStride, hists + (kNumClusters + geo.num_dc) * kHistStride, fb_count);
    }
}

__global__ __launch_bounds__(256) void histograms_kernel(Geometry geo, std::uint32_t dc_chunks,
                                                         const std::uint32_t* __restrict__ partial, int parts,
                                                         std::uint32_t* __restrict__ hists,
                                                         const std::int32_t* __restrict__ dc,
                                                         const std::int8_t* __restrict__ acs,
                                                         const std::int32_t* __restrict__ qf,
                                                         const std::int8_t* __restrict__ ytox,
                                                         const std::int8_t* __restrict__ ytob,
                                                         std::uint32_t* __restrict__ fb_count) {
    histograms_kernel_body(Wg{blockIdx.x, 0, gridDim.x, 1}, geo, dc_chunks, partial, parts, hists, dc, acs, qf, ytox,
                           ytob, fb_count);
}

// The file's variable-length code of a 16-bit count (alphabet sizes).
__device__ __forceinline__ std::uint32_t var_len_u16(std::uint32_t n, std::uint32_t& val) {
    if (n == 0) {
        val = 0;
        return 1;
    }
    const std::uint32_t nb{31u - static_cast<std::uint32_t>(__builtin_clz(n))};
    val = 1u | (nb << 1) | ((n - (1u << nb)) << 5);
    return 5 + nb;
}

struct DcEmitShared {
    std::uint32_t lut[2 * kHistStride];  // DC, then AcMetadata: depth | code << 16
    std::uint32_t buf[kDcSlotWords];
    std::uint32_t sh[kEmitThreads / 64];
    std::uint32_t blob_at[2];  // chunk-relative bit positions of the header blobs
};

// A header blob's pieces: a value (none in the first blob), constant bits, a
// code's alphabet size and its header.
struct DcBlob {
    std::uint32_t lead_bits, lead;
    const std::uint32_t* words;
    std::uint32_t word_bits;
    std::uint32_t alpha_bits, alpha;
    const std::uint32_t* hdr;
    std::uint32_t hdr_bits;
};

__device__ __forceinline__ std::uint32_t blob_bits(DcBlob b) {
    return b.lead_bits + b.word_bits + b.alpha_bits + b.hdr_bits;
}

__device__ __forceinline__ void put_blob(std::uint32_t* buf, DcBlob b, std::uint32_t at) {
    const std::uint32_t t{threadIdx.x};
    if (t == 0) {
        lds_or_bits(buf, kDcSlotWords, at, b.lead, b.lead_bits);
        lds_or_bits(buf, kDcSlotWords, at + b.lead_bits + b.word_bits, b.alpha, b.alpha_bits);
    }
    const std::uint32_t w0{at + b.lead_bits}, h0{w0 + b.word_bits + b.alpha_bits};
    for (std::uint32_t i{32 * t}; i < b.word_bits; i += 32 * 256) {
        lds_or_bits(buf, kDcSlotWords, w0 + i, b.words[i >> 5], b.word_bits - i < 32 ? b.word_bits - i : 32u);
    }
    for (std::uint32_t i{32 * t}; i < b.hdr_bits; i += 32 * 256) {
        lds_or_bits(buf, kDcSlotWords, h0 + i, b.hdr[i >> 5], b.hdr_bits - i < 32 ? b.hdr_bits - i : 32u);
    }
}

// Emission of one chunk of a DC group's items at chunk-relative bit positions
// into the chunk's own staging slot, with its bit count (the layout scans the
// counts, the assembly reads the chunks back to back): one pass, since no
// chunk's place has to be known.  The two header blobs of a group are items
// of its chunks (the first item, and the one after the DC residuals).  The
// group's two codes are read into LDS first; an item is tokenized once.
__device__ __forceinline__ void dc_emit_body(DcEmitShared& S, const Wg& wg, const Geometry& geo,
                                             DcBlob pre, DcBlob mid, const std::int32_t* __restrict__ dc,
                                             const std::int8_t* __restrict__ acs, const std::int32_t* __restrict__ qf,
                                             const std::int8_t* __restrict__ ytox,
                                             const std::int8_t* __restrict__ ytob,
                                             const std::uint8_t* __restrict__ dc_depth,
                                             const std::uint16_t* __restrict__ dc_codes,
                                             const std::uint8_t* __restrict__ meta_depth,
                                             const std::uint16_t* __restrict__ meta_codes,
                                             std::uint32_t* __restrict__ staging,
                                             std::uint32_t* __restrict__ chunk_bits) {
    const int g{static_cast<int>(wg.y)};
    const int tid{static_cast<int>(threadIdx.x)};
    const DcGroupGeo d{dc_group_geo(geo, g)};
    if (wg.x * kDcChunk >= d.items) {
        return;  // the layout counts a group's own chunks
    }
    static_assert(kHistStride == 256, "one code of each per thread");
    S.lut[tid] = static_cast<std::uint32_t>(dc_depth[tid]) | (static_cast<std::uint32_t>(dc_codes[tid]) << 16);
    S.lut[256 + tid] =
        static_cast<std::uint32_t>(meta_depth[tid]) | (static_cast<std::uint32_t>(meta_codes[tid]) << 16);
    for (int i{tid}; i < kDcSlotWords; i += 256) {
        S.buf[i] = 0;
    }
    const std::uint32_t k0{wg.x * kDcChunk + threadIdx.x * kDcPerThread};
    int kind[kDcPerThread];  // 0 DC, 1 AcMetadata, 2 absent, 3 first blob, 4 second blob
    std::uint32_t sym[kDcPerThread]{}, nb[kDcPerThread]{}, ext[kDcPerThread]{};
    {
        DcCursor c{dc_cursor_at(d, k0 < d.items ? k0 : 0u)};
#pragma unroll
        for (int j{0}; j < kDcPerThread; ++j) {
            kind[j] = 2;
            if (k0 + static_cast<std::uint32_t>(j) < d.items) {
                if (c.sec == 0 || c.sec == 2) {
                    kind[j] = c.sec == 0 ? 3 : 4;
                } else {
                    kind[j] = dc_cursor_token(geo, d, c, dc, acs, qf, ytox, ytob, sym[j], nb[j], ext[j]);
                }
                dc_cursor_next(d, c);
            }
        }
    }
    __syncthreads();
    const std::uint32_t pre_bits{blob_bits(pre)}, mid_bits{blob_bits(mid)};
    std::uint32_t len[kDcPerThread], val[kDcPerThread];
    std::uint32_t run{0};
#pragma unroll
    for (int j{0}; j < kDcPerThread; ++j) {
        len[j] = 0;
        val[j] = 0;
        if (kind[j] < 2) {
            const std::uint32_t e{S.lut[kind[j] * kHistStride + static_cast<int>(sym[j])]};
            const std::uint32_t dd{e & 0xffffu};
            len[j] = dd + nb[j];
            val[j] = (e >> 16) | (ext[j] << dd);
        } else if (kind[j] > 2) {
            len[j] = kind[j] == 3 ? pre_bits : mid_bits;
        }
        run += len[j];
    }
    std::uint32_t total{0};
    std::uint32_t at{block_excl_scan_u32<kEmitThreads / 64>(run, S.sh, total)};
#pragma unroll
    for (int j{0}; j < kDcPerThread; ++j) {
        if (kind[j] < 2) {
            lds_or_bits(S.buf, kDcSlotWords, at, val[j], len[j]);
        } else if (kind[j] > 2) {
            S.blob_at[kind[j] - 3] = at;
        }
        at += len[j];
    }
    __syncthreads();
    const std::uint32_t mid_chunk{(1u + 3u * static_cast<std::uint32_t>(d.n)) / kDcChunk};
#pragma unroll
    for (int i{0}; i < 2; ++i) {
        if (wg.x == (i == 0 ? 0u : mid_chunk)) {
            put_blob(S.buf, i == 0 ? pre : mid, S.blob_at[i]);
        }
    }
    __syncthreads();
    const std::size_t chunk{static_cast<std::size_t>(g) * wg.nx + wg.x};
    std::uint32_t* const slot{staging + chunk * kDcSlotWords};
    const int nw{static_cast<int>((total + 31) / 32)};
    for (int i{tid}; i < nw && i < kDcSlotWords; i += 256) {
        slot[i] = S.buf[i];
    }
    if (tid == 0) {
        chunk_bits[chunk] = total;
    }
}

}  // namespace cjx
