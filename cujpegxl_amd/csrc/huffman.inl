// Length-limited prefix codes built by one wave (included into device.hip).
//
// Same results as the serial builder in prefix.h (prefix_code.cc:36-397):
// leaves in descending symbol order, stable sort by count, two-queue merge,
// count floor doubled until the depth limit holds, canonical LSB-first codes,
// simple / code-length-code headers.  The parallel parts:
//   - leaf positions from ballots, the stable sort as a rank computation over
//     (count, leaf position), every wave of a workgroup against its share of
//     the leaves; a count floor only regroups the ranks;
//   - the two-queue merge stays sequential, but its queues live in VGPRs (one
//     value per lane, read and written at a wave-uniform lane), so no step
//     waits on memory; the depths of up to 64 leaves by pointer jumping, of
//     more by a top-down walk;
//   - canonical codes from per-depth ballot ranks;
//   - the code-length-coded header as a wave scan of per-symbol bit lengths.
// Every lane runs the same control flow; loop bounds and queue indices are
// wave-uniform.
//
// What bounds it: one wave's chain of instructions (the merge of up to 64
// leaves, then the header), issued at six to eight cycles each, and the first
// fetch of its code.  All histograms of a frame run side by side: 9.4 us at
// 320x240 and 11.2 us at 3840x2160 (15.7 and 19.7 with a merge step of 345
// cycles, the sort in every wave and the codes before the header).

namespace cjx {

constexpr std::uint32_t kQueueEnd = 0xffffffffu;

// R values per lane: element idx lives in register idx / 64 of lane idx % 64.
template <int R>
struct LaneArray {
    std::uint32_t v[R];

    __device__ __forceinline__ std::uint32_t get(int idx) const {
        const int l{idx & 63};
        if constexpr (R == 1) {
            return static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v[0]), l));
        } else {
            const int r{idx >> 6};
            const int x{r == 0   ? __builtin_amdgcn_readlane(static_cast<int>(v[0]), l)
                        : r == 1 ? __builtin_amdgcn_readlane(static_cast<int>(v[1]), l)
                        : r == 2 ? __builtin_amdgcn_readlane(static_cast<int>(v[2]), l)
                                 : __builtin_amdgcn_readlane(static_cast<int>(v[3]), l)};
            return static_cast<std::uint32_t>(x);
        }
    }

    // Lane idx % 64 of register idx / 64 takes x (a compare and a select).
    __device__ __forceinline__ void set(int idx, std::uint32_t x) {
        const bool mine{(static_cast<int>(threadIdx.x) & 63) == (idx & 63)};
        if constexpr (R == 1) {
            v[0] = mine ? x : v[0];
        } else {
            const int r{idx >> 6};
#pragma unroll
            for (int k{0}; k < R; ++k) {
                v[k] = (mine && r == k) ? x : v[k];
            }
        }
    }
};

// LDS scratch of one wave's build.
struct WaveHuffScratch {
    std::uint32_t sorted_total[256 + 1];
    std::uint32_t sorted_symbol[256];
    std::uint32_t parent[128];  // of leaf i; of internal node k at 64 + k
};

// Value of x in lane `src` (wave-uniform) of the wave.
__device__ __forceinline__ std::uint32_t lane_value(std::uint32_t x, int src) {
    return static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(x), src));
}

// old with lane `lane` (wave-uniform) replaced by x (wave-uniform).
extern "C" __device__ int cjx_write_lane(int x, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// The merge and depths below for n <= 64 leaves.  Each queue is one VGPR
// (lane = queue index); entries that are not there are kQueueEnd.  A merge
// step takes the two smallest of the two queues' first two (both leaves, both
// internal nodes, or one of each; leaves first on ties).  One wave issues an
// instruction every six to eight cycles here, whatever it is, so the step is
// kept short and has no branch: minima of the four entries give the new node's
// total, two compares move the leaf queue, the other queue follows from the
// count of taken entries, and only the leaf queue's position is kept of the
// picks.  From those each step's lane writes the parent links of the entries
// it took, and the depths come from the links by pointer jumping: every node
// holds (distance d, ancestor p), initially (1, parent) and (0, root) at the
// root, packed as p | d << 8, and six rounds of d += d[p], p = p[p] leave each
// node's depth in d (depths are below 64).  Ancestors are internal nodes, so
// every lookup reads the internal nodes' register.
// (Picks by two selects with child links stored per step: 345 cycles a step;
// with branches 400; this form: 170.)  kFull: lane numbers may run
// past the last lane.
template <bool kFull>
__device__ std::uint32_t merge_depths_small(WaveHuffScratch& s, int n, std::uint8_t* depth) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    const std::uint32_t leaf{lane < n ? s.sorted_total[lane] : kQueueEnd};
    const std::uint32_t leaf1{lane + 1 < n ? s.sorted_total[lane + 1] : kQueueEnd};
    const std::uint32_t sym{lane < n ? s.sorted_symbol[lane] : 0u};
    std::uint32_t inner{kQueueEnd}, taken{0};
    // In scalar registers from the start (a constant may be shared with a
    // vector's, and the loop moved to vector instructions with it).
    int i, j, k, both;
    asm("s_mov_b32 %0, 0" : "=s"(i));
    asm("s_mov_b32 %0, 0" : "=s"(j));
    asm("s_mov_b32 %0, 0" : "=s"(k));
    asm("s_mov_b32 %0, 2" : "=s"(both));  // entries taken after the step
    for (; k < n - 1; ++k, both += 2) {
        std::uint32_t a0{lane_value(leaf, i)}, a1{lane_value(leaf1, i)};
        if constexpr (kFull) {
            asm("s_cmp_gt_i32 %[i], 63\n\t"
                "s_cselect_b32 %[a0], -1, %[a0]\n\t"
                "s_cselect_b32 %[a1], -1, %[a1]"
                : [a0] "+s"(a0), [a1] "+s"(a1)
                : [i] "s"(i)
                : "scc");
        }
        const std::uint32_t b0{lane_value(inner, j)}, b1{lane_value(inner, j + 1)};
        std::uint32_t sum, t, u;
        asm("s_min_u32 %[sum], %[a0], %[b0]\n\t"
            "s_max_u32 %[t], %[a0], %[b0]\n\t"
            "s_min_u32 %[u], %[a1], %[b1]\n\t"
            "s_min_u32 %[t], %[t], %[u]\n\t"
            "s_add_u32 %[sum], %[sum], %[t]\n\t"
            "s_cmp_le_u32 %[a1], %[b0]\n\t"   // two leaves
            "s_addc_u32 %[i], %[i], 1\n\t"
            "s_cmp_lt_u32 %[b1], %[a0]\n\t"   // no leaf
            "s_subb_u32 %[i], %[i], 0\n\t"
            "s_sub_i32 %[j], %[both], %[i]"
            : [i] "+s"(i), [j] "=&s"(j), [sum] "=&s"(sum), [t] "=&s"(t), [u] "=&s"(u)
            : [a0] "s"(a0), [a1] "s"(a1), [b0] "s"(b0), [b1] "s"(b1), [both] "s"(both)
            : "scc");
        inner = static_cast<std::uint32_t>(cjx_write_lane(static_cast<int>(sum), k, static_cast<int>(inner)));
        taken = static_cast<std::uint32_t>(cjx_write_lane(i, k, static_cast<int>(taken)));
    }
    // Step k took leaves [i0, i1) and internal nodes [2k - i0, 2k + 2 - i1).
    {
        const int i1{static_cast<int>(taken)};
        const int i0{__builtin_amdgcn_update_dpp(0, i1, 0x138, 0xf, 0xf, false)};  // the lane below's; 0 in lane 0
        const std::uint32_t me{static_cast<std::uint32_t>(lane)};
        if (lane < n - 1) {
            if (i1 > i0) {
                s.parent[i0] = me;
            }
            if (i1 > i0 + 1) {
                s.parent[i0 + 1] = me;
            }
            const int j0{2 * lane - i0};
            if (i1 < i0 + 2) {
                s.parent[64 + j0] = me;
            }
            if (i1 == i0) {
                s.parent[64 + j0 + 1] = me;
            }
        }
        wave_sync();
    }
    const std::uint32_t up_leaf{s.parent[lane]}, up_inner{s.parent[64 + lane]};
    const std::uint32_t root{static_cast<std::uint32_t>(n - 2)};
    std::uint32_t a{lane < n ? (up_leaf | 256u) : root};
    std::uint32_t b{lane < n - 2 ? (up_inner | 256u) : root};
#pragma unroll
    for (int r{0}; r < 6; ++r) {
        const std::uint32_t xa{static_cast<std::uint32_t>(__shfl(static_cast<int>(b), static_cast<int>(a & 255u), 64))};
        const std::uint32_t xb{static_cast<std::uint32_t>(__shfl(static_cast<int>(b), static_cast<int>(b & 255u), 64))};
        a = (a & ~255u) + xa;
        b = (b & ~255u) + xb;
    }
    if (lane < n) {
        depth[sym] = static_cast<std::uint8_t>(a >> 8);
    }
    return lane < n ? a >> 8 : 0u;
}

// Two-queue merge and top-down depths of the n (>= 2) sorted leaves in
// s.sorted_total / s.sorted_symbol; writes depth[symbol] and returns this
// lane's largest leaf depth.  Q * 64 >= n.
template <int Q>
__device__ std::uint32_t merge_depths_large(WaveHuffScratch& s, int n, std::uint8_t* depth) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    LaneArray<Q> leaf{}, sym{};
#pragma unroll
    for (int r{0}; r < Q; ++r) {
        const int t{64 * r + lane};
        leaf.v[r] = t < n ? s.sorted_total[t] : kQueueEnd;
        sym.v[r] = t < n ? s.sorted_symbol[t] : 0u;
    }
    // Two-queue merge: leaves (tree index i < n) and internal nodes
    // (internal k = tree index n + 1 + k), smaller total first, leaf on ties.
    LaneArray<Q> inner{}, kid_l{}, kid_r{};
    int i{0}, j{0};
    for (int k{0}; k < n - 1; ++k) {
        std::uint32_t a{i < n ? leaf.get(i) : kQueueEnd};
        std::uint32_t b{j < k ? inner.get(j) : kQueueEnd};
        int left, right;
        std::uint32_t lt, rt;
        if (a <= b) {
            left = i;
            lt = a;
            ++i;
            a = i < n ? leaf.get(i) : kQueueEnd;
        } else {
            left = n + 1 + j;
            lt = b;
            ++j;
            b = j < k ? inner.get(j) : kQueueEnd;
        }
        if (a <= b) {
            right = i;
            rt = a;
            ++i;
        } else {
            right = n + 1 + j;
            rt = b;
            ++j;
        }
        inner.set(k, lt + rt);
        kid_l.set(k, static_cast<std::uint32_t>(left));
        kid_r.set(k, static_cast<std::uint32_t>(right));
    }
    // Depths top-down from the root (internal n - 2): every child was
    // created before its parent.
    LaneArray<Q> node_depth{}, leaf_depth{};
    node_depth.set(n - 2, 0u);
    for (int k{n - 2}; k >= 0; --k) {
        const std::uint32_t d{node_depth.get(k) + 1u};
        const int cl{static_cast<int>(kid_l.get(k))}, cr{static_cast<int>(kid_r.get(k))};
        if (cl > n) {
            node_depth.set(cl - n - 1, d);
        } else {
            leaf_depth.set(cl, d);
        }
        if (cr > n) {
            node_depth.set(cr - n - 1, d);
        } else {
            leaf_depth.set(cr, d);
        }
    }
    std::uint32_t maxd{0};
#pragma unroll
    for (int r{0}; r < Q; ++r) {
        if (64 * r + lane < n) {
            depth[sym.v[r]] = static_cast<std::uint8_t>(leaf_depth.v[r]);
            maxd = leaf_depth.v[r] > maxd ? leaf_depth.v[r] : maxd;
        }
    }
    return maxd;
}

// Leaves of data[0..length) in create_huffman_tree's input order (descending
// symbol): per lane, the counts of symbols 64 r + lane, whether present, and
// the input position of each present one.
template <int R>
struct Leaves {
    std::uint32_t cnt[R];
    int pos[R];
    int n;
};

template <int R>
__device__ __forceinline__ Leaves<R> wave_leaves(const std::uint32_t* data, int length) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    Leaves<R> L{};
    std::uint64_t present[R];
#pragma unroll
    for (int r{0}; r < R; ++r) {
        const int sym{64 * r + lane};
        L.cnt[r] = sym < length ? data[sym] : 0u;
        present[r] = __ballot(L.cnt[r] != 0);
        L.n += __popcll(present[r]);
    }
    const std::uint64_t above{lane == 63 ? 0ull : (~0ull << (lane + 1))};
    int higher{0};
#pragma unroll
    for (int r{R - 1}; r >= 0; --r) {
        L.pos[r] = higher + __popcll(present[r] & above);
        higher += __popcll(present[r]);
    }
    return L;
}

// Whether each present leaf comes after a leaf of count x at input position
// `at` in the stable ascending order of the counts, added to its rank.
template <int R>
__device__ __forceinline__ void rank_after(const Leaves<R>& L, std::uint32_t x, int at, std::uint32_t (&rank)[R]) {
#pragma unroll
    for (int r{0}; r < R; ++r) {
        rank[r] += x < L.cnt[r] + (at < L.pos[r] ? 1u : 0u) ? 1u : 0u;
    }
}

// One pass of create_huffman_tree's loop (prefix_code.cc:36-96) with count
// floor `count_limit` for n >= 2 leaves (at most kMost) of the given ranks by
// (count, input position): writes depth[symbol] of every present symbol and
// returns whether no depth is above `limit`.
// (kMost keeps merges that cannot be needed out of the code: the kernel runs
// once over most of it, so what it is long it also waits to fetch.)
template <int R, int kMost>
__device__ bool tree_trial(const Leaves<R>& L, const std::uint32_t (&rank)[R], std::uint32_t count_limit, int limit,
                           std::uint8_t* depth, WaveHuffScratch& s) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    const int n{L.n};
    // The floor makes the counts below it equal: those leaves come first, in
    // input order (descending symbol), the others keep their ranks.
    const std::uint32_t least{count_limit - 1};
    const std::uint64_t above{lane == 63 ? 0ull : (~0ull << (lane + 1))};
    int higher{0};
#pragma unroll
    for (int r{R - 1}; r >= 0; --r) {
        const bool low{L.cnt[r] != 0 && L.cnt[r] <= least};
        const std::uint64_t lows{__ballot(low)};
        if (L.cnt[r] != 0) {
            const std::uint32_t at{low ? static_cast<std::uint32_t>(higher + __popcll(lows & above)) : rank[r]};
            s.sorted_total[at] = low ? least : L.cnt[r];
            s.sorted_symbol[at] = static_cast<std::uint32_t>(64 * r + lane);
        }
        higher += __popcll(lows);
    }
    wave_sync();
    std::uint32_t maxd{0};
    if (kMost <= 62 || n <= 62) {
        maxd = merge_depths_small<false>(s, n, depth);
    } else if (kMost <= 64 || n <= 64) {
        maxd = merge_depths_small<true>(s, n, depth);
    } else {
        maxd = merge_depths_large<4>(s, n, depth);
    }
    wave_sync();
    return __ballot(maxd > static_cast<std::uint32_t>(limit)) == 0;
}

// create_huffman_tree (prefix_code.cc:36-96) of at most kMost <= 64 symbols by
// one wave, floors tried in order.  data[0..length) and depth[0..length) are
// in LDS; depth is zero on entry for absent symbols.
template <int kMost>
__device__ void wave_create_tree(const std::uint32_t* data, int length, int limit, std::uint8_t* depth,
                                 WaveHuffScratch& s) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    const Leaves<1> L{wave_leaves<1>(data, length)};
    if (L.n == 0) {
        return;
    }
    if (L.n == 1) {
        if (L.cnt[0] != 0) {
            depth[lane] = 1;
        }
        return;
    }
    std::uint32_t rank[1]{0};
#pragma unroll
    for (int sym{0}; sym < kMost; ++sym) {
        const std::uint32_t x{lane_value(L.cnt[0], sym)};
        // Equal counts: the higher symbol first.
        rank[0] += x - 1u < L.cnt[0] - 1u + (lane < sym ? 1u : 0u) ? 1u : 0u;  // x = 0 is no leaf
    }
    for (std::uint32_t count_limit{1};; count_limit *= 2) {
        if (tree_trial<1, kMost>(L, rank, count_limit, limit, depth, s)) {
            return;
        }
    }
}

// Canonical codes (prefix_code.cc:111-130): bits[s] for depth[s] > 0.
template <int R>
__device__ void wave_depths_to_codes(const std::uint8_t* depth, int len, std::uint16_t* bits) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    int dep[R];
    std::uint32_t mine[R];
#pragma unroll
    for (int r{0}; r < R; ++r) {
        const int sym{64 * r + lane};
        dep[r] = sym < len ? depth[sym] : 0;
        mine[r] = 0;
    }
    std::uint32_t next{0};  // the next code of the depth
#pragma unroll
    for (int d{1}; d < 16; ++d) {
#pragma unroll
        for (int r{0}; r < R; ++r) {
            const std::uint64_t m{__ballot(dep[r] == d)};
            const std::uint32_t code{__builtin_amdgcn_mbcnt_hi(
                static_cast<std::uint32_t>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<std::uint32_t>(m), next))};
            mine[r] = dep[r] == d ? code : mine[r];
            next += static_cast<std::uint32_t>(__popcll(m));
        }
        next <<= 1;
    }
#pragma unroll
    for (int r{0}; r < R; ++r) {
        if (dep[r] != 0) {
            bits[64 * r + lane] = static_cast<std::uint16_t>(__builtin_bitreverse32(mine[r]) >> (32 - dep[r]));
        }
    }
}

struct WaveCodeScratch {
    WaveHuffScratch tree;
    std::uint32_t cl_hist[32];
    std::uint8_t cl_depth[32];
    std::uint16_t cl_bits[32];
    std::uint32_t pos;
};

// store_huffman_tree (prefix_code.cc:211-354) for depth[0..num): returns the
// header length in bits written into hdr (cap words, zeroed).
template <int R>
__device__ std::uint32_t wave_store_tree(const std::uint8_t* depth, int num, std::uint32_t* hdr,
                                         std::uint32_t cap, WaveCodeScratch& s) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    int dep[R];
    int new_len{0};
#pragma unroll
    for (int r{0}; r < R; ++r) {
        const int sym{64 * r + lane};
        dep[r] = sym < num ? depth[sym] : 0;
        const std::uint64_t m{__ballot(dep[r] != 0)};
        if (m != 0) {
            new_len = 64 * r + 64 - static_cast<int>(__builtin_clzll(m));
        }
    }
    // Histogram of depth values over [0, new_len).
    if (lane < 18) {
        s.cl_hist[lane] = 0;
        s.cl_depth[lane] = 0;
        s.cl_bits[lane] = 0;
    }
    wave_sync();
#pragma unroll
    for (int r{0}; r < R; ++r) {
        if (64 * r + lane < new_len) {
            atomicAdd(&s.cl_hist[dep[r]], 1u);
        }
    }
    wave_sync();
    const std::uint32_t uses{lane < 18 ? s.cl_hist[lane] : 0u};
    const std::uint64_t used{__ballot(uses != 0)};
    const int num_codes{used == 0 ? 0 : ((used & (used - 1)) == 0 ? 1 : 2)};  // 2: two or more
    const int code{used == 0 ? 0 : static_cast<int>(__builtin_ctzll(used))};
    wave_create_tree<18>(s.cl_hist, 18, 5, s.cl_depth, s.tree);
    wave_sync();
    wave_depths_to_codes<1>(s.cl_depth, 18, s.cl_bits);
    wave_sync();
    {
        // The code-length code's depths in the format's order (1, 2, 3, 4,
        // 0, 5, 17, 6, 16, 7, ..., 15), lane i taking entry i: the stored run
        // [skip, to_store) goes out as one prefix scan of the entries'
        // lengths (the fixed code of depths 0..5: lengths 2,4,3,2,2,4,
        // values 0,7,3,2,1,15, packed in nibbles).
        const int ord{lane < 4    ? lane + 1
                      : lane == 4 ? 0
                      : lane == 5 ? 5
                      : lane == 6 ? 17
                      : lane == 7 ? 6
                      : lane == 8 ? 16
                                  : lane - 2};
        const std::uint32_t l{lane < 18 ? static_cast<std::uint32_t>(s.cl_depth[ord]) : 0u};
        const std::uint64_t nonzero{__ballot(lane < 18 && l != 0)};
        const int to_store{num_codes > 1 ? (nonzero != 0 ? 64 - static_cast<int>(__builtin_clzll(nonzero)) : 0) : 18};
        const int skip{(nonzero & 3ull) != 0 ? 0 : ((nonzero & 4ull) != 0 ? 2 : 3)};
        const bool stored{lane >= skip && lane < to_store};
        const std::uint32_t nb{stored ? (0x422342u >> (4 * l)) & 15u : 0u};
        const std::uint32_t val{stored ? (0xf12370u >> (4 * l)) & 15u : 0u};
        const std::uint32_t pre{static_cast<std::uint32_t>(wave_excl_scan(static_cast<int>(nb), lane))};
        const std::uint32_t total{2u + static_cast<std::uint32_t>(wave_sum_int(static_cast<int>(nb)))};
        wave_sync();  // every lane has read cl_depth
        if (total <= cap * 32) {
            if (lane == 0) {
                lds_or_bits(hdr, cap, 0, static_cast<std::uint32_t>(skip), 2);
            }
            lds_or_bits(hdr, cap, 2 + pre, val, nb);
        }
        if (lane == 0) {
            if (num_codes == 1) {
                s.cl_depth[code] = 0;
            }
            s.pos = total <= cap * 32 ? total : cap * 32 + 1;
        }
    }
    wave_sync();
    std::uint32_t at{s.pos};
#pragma unroll
    for (int r{0}; r < R; ++r) {
        const bool in{64 * r + lane < new_len};
        const std::uint32_t l{in ? static_cast<std::uint32_t>(s.cl_depth[dep[r]]) : 0u};
        const std::uint32_t v{in ? static_cast<std::uint32_t>(s.cl_bits[dep[r]]) : 0u};
        const std::uint32_t pre{static_cast<std::uint32_t>(wave_excl_scan(static_cast<int>(l), lane))};
        if (at + pre + l <= cap * 32) {
            lds_or_bits(hdr, cap, at + pre, v, l);
        }
        at += static_cast<std::uint32_t>(wave_sum_int(static_cast<int>(l)));
    }
    return at;
}

// build_and_store_huffman_tree (prefix_code.cc:358-397) for hist[0..alpha),
// alpha >= 2, with depth[] already holding create_huffman_tree's result when
// more than one symbol is present (all zero otherwise): the header, by one
// wave.  (The codes are wave_depths_to_codes' from the same depths.)  Returns
// the header length in bits, or 0 if it would not fit `cap` words.
template <int R>
__device__ std::uint32_t wave_store_code(const std::uint32_t* hist, int alpha, const std::uint8_t* depth,
                                         std::uint32_t* hdr, std::uint32_t cap, WaveCodeScratch& s) {
    const int lane{static_cast<int>(threadIdx.x) & 63};
    std::uint64_t present[R];
    int count{0};
#pragma unroll
    for (int r{0}; r < R; ++r) {
        const int sym{64 * r + lane};
        present[r] = __ballot(sym < alpha && hist[sym] != 0);
        count += __popcll(present[r]);
    }
    if (count > 4) {
        const std::uint32_t nb{wave_store_tree<R>(depth, alpha, hdr, cap, s)};
        return nb <= cap * 32 ? nb : 0u;
    }
    // The present symbols, ascending.
    int s4[4]{0, 0, 0, 0};
    {
        int got{0};
#pragma unroll
        for (int r{0}; r < R; ++r) {
            std::uint64_t m{present[r]};
            while (m != 0 && got < 4) {
                s4[got++] = 64 * r + static_cast<int>(__builtin_ctzll(m));
                m &= m - 1;
            }
        }
    }
    int max_bits{0};
    for (int c{alpha - 1}; c; c >>= 1) {
        ++max_bits;
    }
    std::uint32_t pos{0};
    if (lane == 0) {
        BitSink w{hdr, 0, cap * 32};
        if (count <= 1) {
            w.write(4, 1);
            w.write(static_cast<std::uint32_t>(max_bits), static_cast<std::uint32_t>(s4[0]));
        } else {
            w.write(2, 1);
            w.write(2, static_cast<std::uint32_t>(count - 1));
            for (int i{0}; i < count; ++i) {
                for (int j{i + 1}; j < count; ++j) {
                    if (depth[s4[j]] < depth[s4[i]]) {
                        const int t{s4[j]};
                        s4[j] = s4[i];
                        s4[i] = t;
                    }
                }
            }
            for (int i{0}; i < count; ++i) {
                w.write(static_cast<std::uint32_t>(max_bits), static_cast<std::uint32_t>(s4[i]));
            }
            if (count == 4) {
                w.write(1, depth[s4[0]] == 1 ? 1u : 0u);
            }
        }
        pos = w.ok() ? w.pos : 0u;
    }
    return static_cast<std::uint32_t>(__shfl(static_cast<int>(pos), 0, 64));
}

}  // namespace cjx
