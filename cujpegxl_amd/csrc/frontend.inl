// Front-end kernels (included into device.hip).
//
// region_kernel: one 256-thread workgroup per 32x32-pixel selection region.
// The region's NV12 pixels plus a 2-pixel clamped halo are converted to XYB
// once into LDS; everything downstream reads LDS: inverse gaborish, the
// adaptive-quantization field, the RD transform selection over the 21 DCT8/16/32
// candidates of the sharpened Y, the chosen DCTs of all three channels and the
// CfL regression partials.  Only the FP16 coefficients, the transform map,
// the quant field and three floats per region reach HBM.
//
// tile_quantize_kernel: one workgroup per 64x64 CfL tile: the tile's colour
// maps, quantization of every coefficient with the CfL residual, the
// per-block non-zero counts the entropy coder predicts from, and the DC of
// every block (from the LLF coefficients it reads anyway).
//
// Element layout used throughout a region: thread (wave w, lane L) at
// iteration k owns element i = 256k + 64w + L of [0, 1024).  Element ids nest:
// a DCT32 owns [0,1024), the DCT16 on quad q owns [256q, 256q+256), the DCT8 on
// block j of quad q owns [256q + 64j, +64).  Position (quad k, block w) slot L
// holds raw coefficient e = 64 q + L of its first-block (q = covered ordinal).

namespace cjx {

constexpr int kHalo = 2;
constexpr int kTileW = 32 + 2 * kHalo;  // 36
// Chroma rows a tile's bilinear taps can reach: (32 + 2 halo) / 2 + 1 on each
// side.
constexpr int kChromaRows = kTileW / 2 + 2;  // 20

// Orders one wave's LDS accesses: writes before the barrier are seen by
// every lane's reads after it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Grid-strided zeroing of the Clears buffers by every thread of a launch
// (of the frame's workgroups, in a batched launch).
__device__ __forceinline__ void clear_words(const Clears& c, const Wg& wg) {
    const std::uint32_t stride{wg.nx * wg.ny * blockDim.x};
    const std::uint32_t first{(wg.y * wg.nx + wg.x) * blockDim.x};
#pragma unroll
    for (int k{0}; k < 4; ++k) {
        if (first < c.words[k]) {  // a scalar test: most workgroups have nothing to clear
            for (std::uint32_t i{first + threadIdx.x}; i < c.words[k]; i += stride) {
                c.ptr[k][i] = 0;
            }
        }
    }
}

// Cross-lane sums without the LDS crossbar.  add_down_row<n>: lane i adds
// lane i + n of its row of 16 lanes (a DPP row shift; n = 1, 2, 4, 8);
// add_down_16: lanes of rows 0 and 2 add rows 1 and 3 (v_permlane16_swap);
// add_down_32: lanes 0-31 add lanes 32-63 (v_permlane32_swap).  Callers read
// only lanes whose partners lie in the same row (or the upper row / half),
// where the result equals a shfl_down (or shfl_xor) tree's term for term.
template <int kN>
__device__ __forceinline__ float add_down_row(float v) {
    static_assert(kN == 1 || kN == 2 || kN == 4 || kN == 8, "row shift");
    return v + u2f(static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(f2u(v)), 0x100 + kN,
                                                                          0xf, 0xf, true)));
}

__device__ __forceinline__ float add_down_16(float v) {
    const auto r{__builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false)};
    return v + u2f(r[1]);
}

__device__ __forceinline__ float add_down_32(float v) {
    const auto r{__builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false)};
    return v + u2f(r[1]);
}

// Lane i - 1 of the same row of 16 lanes (DPP row shift right).
__device__ __forceinline__ float from_lane_below(float v) {
    return u2f(static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(f2u(v)), 0x111, 0xf, 0xf,
                                                                      true)));
}

// Four wave sums at once, each the shfl_down tree of its 64 values (offsets
// 32, 16, ..., 1; lane i adds lane i + offset) with the same operands in the
// same order: one permlane32 swap and add carry out offset 32 for two
// values (a in lanes 0-31, b in lanes 32-63; c and d likewise), one
// permlane16 swap and add offset 16 for all four (rows: a, c, b, d), then
// the row shifts 8..1 for all four.  The result holds sum(a) in lane 0,
// sum(c) in lane 16, sum(b) in lane 32 and sum(d) in lane 48.
__device__ __forceinline__ float wave_sum4(float a, float b, float c, float d) {
    const auto ab{__builtin_amdgcn_permlane32_swap(f2u(a), f2u(b), false, false)};
    const float x{u2f(ab[0]) + u2f(ab[1])};
    const auto cd{__builtin_amdgcn_permlane32_swap(f2u(c), f2u(d), false, false)};
    const float y{u2f(cd[0]) + u2f(cd[1])};
    const auto xy{__builtin_amdgcn_permlane16_swap(f2u(x), f2u(y), false, false)};
    float v{u2f(xy[0]) + u2f(xy[1])};
    v = add_down_row<8>(v);
    v = add_down_row<4>(v);
    v = add_down_row<2>(v);
    return add_down_row<1>(v);
}

// Lane l's value of v (a wave-uniform read).
__device__ __forceinline__ float lane_value(float v, int l) {
    return u2f(static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(f2u(v)), l)));
}

__device__ __forceinline__ float clamp01(float v) {
    return fminf(fmaxf(v, 0.0f), 1.0f);
}

// The table-driven powers with the series argument's two constants held in
// registers, so that placing the mantissa bits is one v_and_or_b32.
struct XybPowers {
    const float2* tab;
    std::uint32_t mask, one;

    __device__ __forceinline__ explicit XybPowers(const float2* t) : tab{t}, mask{0x0007ffffu}, one{0x4b000000u} {
        asm volatile("" : "+s"(mask), "+v"(one));
    }
    __device__ __forceinline__ float arg(std::uint32_t u, float r_scaled) const {
        return (u2f((u & mask) | one) - 8650752.0f) * r_scaled;
    }
    __device__ __forceinline__ float pow24(float x) const {
        const std::uint32_t u{f2u(x)};
        const float2 e{tab[kXybPow + ((u >> 19) - (122u << 4))]};
        return pow24_series(e.x, arg(u, e.y));
    }
    __device__ __forceinline__ float cbrt(float x) const {
        const std::uint32_t u{f2u(x)};
        const float2 e{tab[kXybCbrt + ((u >> 19) - (118u << 4))]};
        return cbrt_series(e.x, arg(u, e.y));
    }
};

// xyb_impl.cuh:37-70 on the shared numeric primitives, clamped to [0, 1] (the
// line lies there for e in [0, 1]).  Both branches are evaluated: a pixel's
// three curves then overlap instead of waiting for their table reads one
// after another in divergent branches (region kernel 159 -> 156 us at
// 3840x2160).
__device__ __forceinline__ float srgb_to_linear(float e, const XybPowers& pw) {
    const float line{e * (1.0f / 12.92f)};
    const float curve{clamp01(pw.pow24((e + 0.055f) * (1.0f / 1.055f)))};
    return e <= 0.04045f ? line : curve;
}

// Opsin absorbance bias of the XYB transform.
constexpr float kOpsinBias{0.0037930732552754493f};

// `neg_cbrt_bias` is -cbrt(kOpsinBias), evaluated once by the caller.
__device__ __forceinline__ void pixel_to_xyb(float yv, float cb, float cr, float& ox, float& oy, float& ob,
                                             const XybPowers& pw, float neg_cbrt_bias) {
    constexpr float m00{0.30f}, m02{0.078f}, m01{1.0f - 0.078f - 0.30f};
    constexpr float m10{0.23f}, m12{0.078f}, m11{1.0f - 0.078f - 0.23f};
    constexpr float m20{0.24342268924547819f}, m21{0.20476744424496821f};
    constexpr float m22{1.0f - 0.24342268924547819f - 0.20476744424496821f};
    constexpr float bias{kOpsinBias};
    const float r{srgb_to_linear(clamp01(yv + 1.5748f * cr), pw)};
    const float g{srgb_to_linear(clamp01(yv - 0.1873242729f * cb - 0.4681242729f * cr), pw)};
    const float b{srgb_to_linear(clamp01(yv + 1.8556f * cb), pw)};
    float q0{m00 * r + m01 * g + m02 * b + bias};  // positive: nothing to clamp
    float q1{m10 * r + m11 * g + m12 * b + bias};
    float q2{m20 * r + m21 * g + m22 * b + bias};
    q0 = pw.cbrt(q0) + neg_cbrt_bias;
    q1 = pw.cbrt(q1) + neg_cbrt_bias;
    q2 = pw.cbrt(q2) + neg_cbrt_bias;
    ox = 0.5f * (q0 - q1);
    oy = 0.5f * (q0 + q1);
    ob = q2;
}

// a / b and sqrt(x), correctly rounded, for normal operands of moderate
// size with normal results (the AQ terms: 0.01 <= a, b <= 2e4, 27 <= x <=
// 5e5): the compiler's correctly rounded sequences (a reciprocal, one
// Newton step and two Markstein corrections; a square root and its
// one-ulp neighbour tests) without their operand scaling and special-case
// steps, which are identities for such operands.  check_aq_math_kernel
// compares both against the compiler's forms over every reachable input.
__device__ __forceinline__ float div_moderate(float a, float b) {
    float r{__builtin_amdgcn_rcpf(b)};
    r = __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
    float q{a * r};
    q = __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), r, q);
}

__device__ __forceinline__ float sqrt_moderate(float x) {
    const float s{__builtin_amdgcn_sqrtf(x)};
    const float below{__builtin_bit_cast(float, __builtin_bit_cast(std::int32_t, s) - 1)};
    const float above{__builtin_bit_cast(float, __builtin_bit_cast(std::int32_t, s) + 1)};
    const float r{__builtin_fmaf(-below, s, x) <= 0.0f ? below : s};
    return __builtin_fmaf(-above, s, x) > 0.0f ? above : r;
}

// adaptive_quant_impl.cuh:29-61
template <bool kModerate = true>
__device__ __forceinline__ float ratio_cbrt_gamma(float v, bool invert) {
    constexpr float k_sg_mul{226.77216153508914f};
    constexpr float k_sg_log2{0.693147181f};
    constexpr float k_sg_mul2{1.0f / 73.377132366608819f};
    constexpr float k_sg_ret_mul{k_sg_mul2 * 18.6580932135f * k_sg_log2};
    constexpr float eps{1e-2f};
    constexpr float num_mul{k_sg_ret_mul * 3.0f * k_sg_mul};
    constexpr float v_offset{7.7825991679894591f * k_sg_log2 + eps};
    constexpr float den_mul{k_sg_log2 * k_sg_mul};
    v = v < 0.0f ? 0.0f : v;
    const float v2{v * v};
    const float num{num_mul * v2 + eps};
    const float den{den_mul * v * v2 + v_offset};
    if constexpr (kModerate) {
        return invert ? div_moderate(num, den) : div_moderate(den, num);
    } else {
        return invert ? num / den : den / num;
    }
}

template <bool kModerate = true>
__device__ __forceinline__ float masking_sqrt(float v) {
    constexpr float mul{211.66567973503678f * 1e8f};
    const float x{v * __builtin_sqrtf(mul) + 27.505837037000106f};
    if constexpr (kModerate) {
        return 0.25f * sqrt_moderate(x);
    } else {
        return 0.25f * __builtin_sqrtf(x);
    }
}

// The AQ terms' division and square root in both forms over every float
// input of their domains (ratio_cbrt_gamma: v in [0, 4), both directions;
// masking_sqrt: v in [0, 0.25)): mismatching bit patterns are counted.
__global__ void check_aq_math_kernel(std::uint32_t first, std::uint32_t count, std::uint32_t sqrt_limit,
                                     unsigned long long* mismatches) {
    unsigned int bad{0};
    for (std::uint32_t i{blockIdx.x * blockDim.x + threadIdx.x}; i < count; i += gridDim.x * blockDim.x) {
        const std::uint32_t bits{first + i};
        const float v{__builtin_bit_cast(float, bits)};
        bad += __builtin_bit_cast(std::uint32_t, ratio_cbrt_gamma<true>(v, true)) !=
               __builtin_bit_cast(std::uint32_t, ratio_cbrt_gamma<false>(v, true));
        bad += __builtin_bit_cast(std::uint32_t, ratio_cbrt_gamma<true>(v, false)) !=
               __builtin_bit_cast(std::uint32_t, ratio_cbrt_gamma<false>(v, false));
        if (bits < sqrt_limit) {
            bad += __builtin_bit_cast(std::uint32_t, masking_sqrt<true>(v)) !=
                   __builtin_bit_cast(std::uint32_t, masking_sqrt<false>(v));
        }
    }
    if (bad != 0) {
        atomicAdd(mismatches, static_cast<unsigned long long>(bad));
    }
}

__device__ __forceinline__ float compute_mask(float out_val) {
    const float v1{fmaxf(out_val * 0.80061762862741759f, 1e-3f)};
    const float v2{1.0f / (v1 + 302.59587815579727f)};
    const float v3{1.0f / (v1 * v1 + 3.7179635626140772f)};
    const float v4{1.0f / (v1 * v1 + 0.25f * 3.7179635626140772f)};
    return -0.7647f + 9.4708735624378946f * v4 + 17.35036561631863f * v2 + 6.7943250517376494f * v3;
}

__device__ __forceinline__ void cswap(float& a, float& b) {
    if (a > b) {
        const float t{a};
        a = b;
        b = t;
    }
}

// frontend_fused.cu:35-52 with adaptive_quant_impl.cuh:63-121: weighted sum
// of the four smallest cells of the clamped 3x3 neighbourhood.
__device__ float erosion_cell(const float* pre, int cx, int cy, const FrameParams& p) {
    const int xm1{cx > 0 ? cx - 1 : cx}, xp1{cx + 1 < 8 ? cx + 1 : cx};
    const int ym1{cy > 0 ? cy - 1 : cy}, yp1{cy + 1 < 8 ? cy + 1 : cy};
    float m0{pre[cy * 8 + cx]}, m1{pre[cy * 8 + xm1]}, m2{pre[cy * 8 + xp1]}, m3{pre[ym1 * 8 + xm1]};
    cswap(m0, m1);
    cswap(m0, m2);
    cswap(m0, m3);
    cswap(m1, m2);
    cswap(m1, m3);
    cswap(m2, m3);
    const float extra[5]{pre[ym1 * 8 + cx], pre[ym1 * 8 + xp1], pre[yp1 * 8 + xm1],
                         pre[yp1 * 8 + cx], pre[yp1 * 8 + xp1]};
#pragma unroll
    for (int i{0}; i < 5; ++i) {
        const float v{extra[i]};
        if (v < m3) {
            if (v < m0) {
                m3 = m2;
                m2 = m1;
                m1 = m0;
                m0 = v;
            } else if (v < m1) {
                m3 = m2;
                m2 = m1;
                m1 = v;
            } else if (v < m2) {
                m3 = m2;
                m2 = v;
            } else {
                m3 = v;
            }
        }
    }
    return p.km[0] * m0 + p.km[1] * m1 + p.km[2] * m2 + p.km[3] * m3;
}

// Separable DCT building block.  One lane owns one line of N inputs (a pixel
// row for the row pass, a row-pass output line for the column pass) and
// produces F consecutive frequencies k0..k0+F-1 of it:
//   out[f] = sum_{c = 0..N-1} A[k0 + f][c] * in[c]   (fmaf chain in c order).
// k0 is wave-uniform, so every basis value is a scalar operand; the line is
// read with 16-byte LDS loads.
template <int N>
__device__ __forceinline__ const float* basis_n() {
    if constexpr (N == 8) {
        return g_tables.basis8;
    } else if constexpr (N == 16) {
        return g_tables.basis16;
    } else {
        return g_tables.basis32;
    }
}

// Columns col0..col0 + N - 1 of the row at `src`, whose 16-byte groups are
// permuted by `swz` (group g stored at g ^ swz; 0 for the unpermuted row-pass
// lines).
template <int N, int F>
__device__ __forceinline__ void dct_line(const float* __restrict__ src, int k0, float (&out)[F], int col0 = 0,
                                         int swz = 0) {
    float p[N];
#pragma unroll
    for (int c{0}; c < N; c += 4) {
        const float4 v{*reinterpret_cast<const float4*>(src + ((((col0 + c) >> 2) ^ swz) << 2))};
        p[c] = v.x;
        p[c + 1] = v.y;
        p[c + 2] = v.z;
        p[c + 3] = v.w;
    }
    const float* A{basis_n<N>() + k0 * N};
#pragma unroll
    for (int f{0}; f < F; ++f) {
        float s{0.0f};
#pragma unroll
        for (int c{0}; c < N; ++c) {
            s = __builtin_fmaf(A[f * N + c], p[c], s);
        }
        out[f] = s;
    }
}

// Row-pass lines of the DCT8s (dct8_uniform_kernel): line (block b, frequency
// k) starts at b * BS + k * RS; RS a multiple of 4 (16-byte loads) such that
// eight consecutive lines start in eight different 4-bank groups.
struct RowBuf8 {
    static constexpr int RS = 12, BS = 104;
};

// Sharpened planes: rows of 32 floats without padding, the row's eight
// 16-byte groups permuted by (row / 2) mod 8, so that the 16 consecutive rows
// a matrix-core row pass reads at one column fall into 16 different 4-bank
// groups.  Planes are stored in the order X, B, Y.
constexpr int kSP = 32;
__device__ __forceinline__ int sp_swz(int row) {
    return (row >> 1) & 7;
}
__device__ __forceinline__ int sp_index(int row, int col) {
    return row * kSP + (((col >> 2) ^ sp_swz(row)) << 2) + (col & 3);
}
// Coefficient arrays are written four elements at a time in transposed
// (column) order by the transforms and read in element order: four pad halfs
// per 32 elements keep the 8-byte accesses aligned and spread the columns.
constexpr int kCoefPadded = 1024 + 4 * 32;
__device__ __forceinline__ int cpad(int e) {
    return e + 4 * (e >> 5);
}

// Arrays whose lifetimes do not overlap share storage, which keeps the
// workgroup at 23.5 KB of LDS: six resident workgroups per CU (80 VGPRs, no
// spill).  With a space of their own for the sharpened planes it was 31.7 KB
// and five per CU, and the kernel took 164 us at 3840x2160 (138 learned +
// FP16) instead of 159 (134):
// - `a`: the XYB tile until every thread has read it (its sharpened pixels
//   wait in registers), then the sharpened planes X, B, Y; Y's space and the
//   rest past it take the DCT32's selection terms once Y has been
//   transformed, then X's and B's coefficients of the chosen transforms.
// - `b`: the chroma rows and the powers' table of step 1, then the AQ terms
//   (steps 2-3), then Y's coefficients of the three candidate sizes, the
//   features and the network's hidden units.
struct AqTerms {
    float cells[64];
    float ero[64];     // fuzzy erosion of each cell
    float blk[16][3];  // per block: HF sum, gamma, blue sum
};

struct RegionShared {
    union {
        alignas(16) float xyb[3][kTileW * kTileW];  // NV12 -> XYB tile with halo
        float sharp[3][32 * kSP];
        struct {
            float planes[2][32 * kSP];  // X and B
            union {
                float t32[2][3][64][4];  // DCT32 terms (errors, rates) of waves 1-3's quadrants
                _Float16 xb[2][kCoefPadded];
            } y;
        } after;
    } a;
    union {
        struct {
            std::uint32_t h[kChromaRows * kTileW];
            float2 tab[kXybTabPairs];
        } in;
        AqTerms aq;
        struct {
            _Float16 y[3][kCoefPadded];  // DCT8, DCT16 and DCT32 candidates
            float feat[112];             // network features (block sums first; learned mode and export)
            float hid[72];               // the network's hidden units and outputs
        } s;
    } b;
    float cost8[16];       // quad-major
    float cost16[4];
    float cost32;
    float cost32p[4];      // matrix-core form: the DCT32 cost's part from each wave
    float cfl[4][3];
    int acs[16];           // region-local raster
    int blkqf[16];         // quant field of the region's blocks (export)
    int choice[4];         // the heuristic's choice per quad (export)
    int learned_ok;        // the network's decision was confident
};
// LDS is allocated in 1,280-byte blocks: six workgroups per CU (160 KB) need
// at most 21 blocks each.
static_assert(sizeof(RegionShared) <= 21 * 1280, "six workgroups per CU");
static_assert(offsetof(RegionShared, b) == sizeof(float) * 3 * kTileW * kTileW, "the XYB tile is the largest use of a");

// Sharpened plane of channel c (0 X, 1 Y, 2 B).
__device__ __forceinline__ float* plane_of(RegionShared& S, int c) {
    return S.a.sharp[c == 0 ? 0 : (c == 1 ? 2 : 1)];
}

// Y coefficients of candidate size 8 << sz, element order (cpad).
__device__ __forceinline__ _Float16* coefy_of(RegionShared& S, int sz) {
    return S.b.s.y[sz];
}

// Selection terms of M Y coefficients of one lane (transform_select_impl.cuh:
// 49-108): squared quantization error and rate proxy; LLF coefficients
// (llf[i], from the callers' closed forms for their lane layouts)
// contribute 0, which the terms of a zero coefficient are exactly (q = 0,
// err = 0, rate[0] = 0).  The two quotients are the correctly rounded ones,
// by reciprocals.  The weights come in as arguments (read four at a time by
// the callers, the frequencies of a lane run in fours); the rate entries of
// all M quotients are read together.
template <int M>
__device__ __forceinline__ void selection_terms(const float (&s)[M], const bool (&llf)[M], const float (&wq)[M],
                                                const float (&wi)[M], const FrameParams& prm, float (&d)[M],
                                                float (&rt)[M]) {
    float aq[M], r[M];
    float top{0.0f};
#pragma unroll
    for (int i{0}; i < M; ++i) {
        const float sv{llf[i] ? 0.0f : s[i]};
        const float q{__builtin_rintf(div_by_recip(sv * prm.qgsf_select, wq[i], wi[i]))};
        const float err{div_by_recip(q * wq[i], prm.qgsf_select, prm.inv_qgsf_select) - sv};
        d[i] = err * err;
        aq[i] = fabsf(q);
        top = fmaxf(top, aq[i]);
        r[i] = g_tables.rate[static_cast<std::uint32_t>(fminf(aq[i], 255.0f))];
    }
    // Past the table (one test for all M).
    if (__builtin_amdgcn_ballot_w64(top >= 256.0f) != 0) {
#pragma unroll
        for (int i{0}; i < M; ++i) {
            r[i] = aq[i] >= 256.0f ? 1.0f + log2_det(1.0f + aq[i]) : r[i];
        }
    }
#pragma unroll
    for (int i{0}; i < M; ++i) {
        rt[i] = r[i];
    }
}

// Weights and reciprocals of frequencies e0 .. e0 + 3 (e0 a multiple of 4)
// into wq[i0 ..], wi[i0 ..].
template <int M>
__device__ __forceinline__ void selection_weights4(const float* w, const float* w_inv, int e0, int i0,
                                                   float (&wq)[M], float (&wi)[M]) {
    const float4 a{*reinterpret_cast<const float4*>(w + e0)};
    const float4 b{*reinterpret_cast<const float4*>(w_inv + e0)};
    wq[i0] = a.x;
    wq[i0 + 1] = a.y;
    wq[i0 + 2] = a.z;
    wq[i0 + 3] = a.w;
    wi[i0] = b.x;
    wi[i0 + 1] = b.y;
    wi[i0 + 2] = b.z;
    wi[i0 + 3] = b.w;
}

// Colour maps of a 64x64 tile from its regions' partial sums (cfl.h:58-64 on
// (R00 + R10) + (R01 + R11); absent regions contribute zeros).
__device__ __forceinline__ void cfl_tile_maps(const float (&r)[4][3], int& mx, int& mb) {
    float s[3];
    for (int c{0}; c < 3; ++c) {
        s[c] = (r[0][c] + r[1][c]) + (r[2][c] + r[3][c]);
    }
    const double sxy{s[0]}, syy{s[1]}, sby{s[2]};
    const float fx{syy > 0.0 ? static_cast<float>(sxy / syy) : 0.0f};
    const float db{syy > 0.0 ? static_cast<float>(sby / syy) : 0.0f};
    mx = static_cast<int>(__builtin_rintf(fx * 84));
    mb = static_cast<int>(__builtin_rintf(db * 84));
    mx = mx < -128 ? -128 : (mx > 127 ? 127 : mx);
    mb = mb < -128 ? -128 : (mb > 127 ? 127 : mb);
}

// Partial sums of tile (tx, ty)'s regions, zeros for regions past the frame.
__device__ __forceinline__ void tile_partials(const Geometry& geo, const float* cfl_part, int tx, int ty,
                                              float (&r)[4][3]) {
    for (int i{0}; i < 4; ++i) {
        const int rx{tx * 2 + (i & 1)}, ry{ty * 2 + (i >> 1)};
        const bool ok{rx < static_cast<int>(geo.rw) && ry < static_cast<int>(geo.rh)};
        for (int c{0}; c < 3; ++c) {
            r[i][c] = ok ? cfl_part[(static_cast<std::size_t>(ry) * geo.rw + rx) * 3 + c] : 0.0f;
        }
    }
}

// Profiling builds only (CJX_REGION_CUT, never the shipped libraries): the
// region kernel returns, uniformly, at the start of step k + 1 when the
// device word says k (k = 6, 7, 8 cut the transform selection after its
// opening barrier, its transforms and its rate-distortion terms), so that the time
// and instruction counts of each step are differences of two cut builds.
#ifdef CJX_REGION_CUT
__device__ int g_region_cut;
#define CJX_REGION_CUT_AT(k)                                        \
    if (__builtin_amdgcn_readfirstlane(g_region_cut) == (k)) { \
        return;                                                     \
    }
#else
#define CJX_REGION_CUT_AT(k)
#endif

// Step 1 of a region: NV12 -> XYB over the 36x36 tile (2-pixel halo,
// clamped coordinates), exact 4:2:0 bilinear chroma (centred taps clamped
// to the plane, tests/reference.py:23-46).
//
// The bilinear's weights are 3/4 on the sample of the pixel's own chroma
// cell (coordinate x >> 1) and 1/4 on its neighbour towards the pixel
// (clamped to the plane), in each direction.  Every partial sum of the
// float form (products of samples and weights, then their sums) is exact,
// so the interpolated value is exactly (3 h_k + h_n) / 16 with the horizontal
// sums h = 3 s_k + s_n of the rows k and n: the tile computes these as
// integers, for Cb and Cr at once in the two halves of one word (at most
// 16 * 255 each), and scales by 1/16, which gives the float form's bits.
//
// Thread t takes column t % 36 of the tile, for the chroma rows (t / 36 + 7 j)
// and for the pixels (rows t / 36 + 7 k): the column's taps are computed
// once, and a row's horizontal sums once for the pixels above and below.  The
// kernel is bound by VALU issue, so away from the frame's top and bottom,
// where no row is clamped, every row's address is one of the thread's base
// registers plus a constant (LDS) or a scalar (planes), and the six luma reads
// are issued at once.  Other regions, and planes with a pitch that 32-bit
// offsets do not cover, compute each row's address.
// Region kernel at 3840x2160, one address computed per row and tap before:
// 156 -> 149 us (130.7 -> 124.5 learned + FP16); VALU instructions -9.6%.
__device__ __forceinline__ void xyb_tile(RegionShared& S, const std::uint8_t* luma, std::size_t luma_pitch,
                                         const std::uint8_t* chroma, std::size_t chroma_pitch, int px0, int py0,
                                         int W, int H, int tid) {
    float2* const tab{S.b.in.tab};
    std::uint32_t* const h{S.b.in.h};
    const int cw{W / 2}, ch{H / 2};
    const int cy0{(py0 >> 1) - 2};
    static_assert(kXybTabPairs == 256, "one table entry per thread");
    tab[tid] = g_tables.xyb_tab[tid];
    const int lx{tid % kTileW}, r0{tid / kTileW};
    const bool active{tid < 7 * kTileW};
    constexpr std::size_t kMaxPitch{std::size_t{1} << 28};
    const bool interior{py0 >= kHalo && py0 + 36 <= H && luma_pitch <= kMaxPitch && chroma_pitch <= kMaxPitch};
    int gx{px0 + lx - kHalo};
    gx = gx < 0 ? 0 : (gx >= W ? W - 1 : gx);
    constexpr int kPix{(kTileW + 6) / 7};  // pixel rows of a thread (the last one for r0 = 0 only)
    std::uint32_t lu[kPix]{};
    if (active) {
        const int kx{gx >> 1};
        const int nx{(gx & 1) != 0 ? (kx + 1 < cw ? kx + 1 : cw - 1) : (kx > 0 ? kx - 1 : 0)};
        // Chroma pairs (Cb | Cr << 8) at the two taps of up to three rows.
        constexpr int kRows{(kChromaRows + 6) / 7};
        std::uint16_t sk[kRows]{}, sn[kRows]{};
        if (interior) {
            const std::uint8_t* const lrow{luma + static_cast<std::size_t>(py0 - kHalo) * luma_pitch};
            const std::uint32_t lo{static_cast<std::uint32_t>(r0) * static_cast<std::uint32_t>(luma_pitch) +
                                   static_cast<std::uint32_t>(gx)};
#pragma unroll
            for (int k{0}; k < kPix; ++k) {
                if (7 * k + 6 < kTileW || r0 + 7 * k < kTileW) {
                    lu[k] = (lrow + static_cast<std::size_t>(7 * k) * luma_pitch)[lo];
                }
            }
            const std::uint8_t* const crow{chroma + static_cast<std::size_t>(cy0) * chroma_pitch};
            const std::uint32_t co{static_cast<std::uint32_t>(r0) * static_cast<std::uint32_t>(chroma_pitch)};
#pragma unroll
            for (int j{0}; j < kRows; ++j) {
                if (7 * j + 6 < kChromaRows || r0 + 7 * j < kChromaRows) {
                    const std::uint8_t* const row{crow + static_cast<std::size_t>(7 * j) * chroma_pitch};
                    __builtin_memcpy(&sk[j], row + (co + 2u * static_cast<std::uint32_t>(kx)), 2);
                    __builtin_memcpy(&sn[j], row + (co + 2u * static_cast<std::uint32_t>(nx)), 2);
                }
            }
        } else {
#pragma unroll 1
            for (int j{0}; j < kRows; ++j) {
                if (r0 + 7 * j < kChromaRows) {
                    int y{cy0 + r0 + 7 * j};
                    y = y < 0 ? 0 : (y >= ch ? ch - 1 : y);
                    const std::uint8_t* const row{chroma + static_cast<std::size_t>(static_cast<std::uint32_t>(y)) *
                                                               chroma_pitch};
                    std::uint16_t k, n;
                    __builtin_memcpy(&k, row + 2u * static_cast<std::uint32_t>(kx), 2);
                    __builtin_memcpy(&n, row + 2u * static_cast<std::uint32_t>(nx), 2);
                    const auto pair = [](std::uint32_t v) { return (v & 0xffu) | ((v & 0xff00u) << 8); };
                    h[(r0 + 7 * j) * kTileW + lx] = 3u * pair(k) + pair(n);
                }
            }
        }
        if (interior) {
#pragma unroll
            for (int j{0}; j < kRows; ++j) {
                if (7 * j + 6 < kChromaRows || r0 + 7 * j < kChromaRows) {
                    const auto pair = [](std::uint32_t v) { return (v & 0xffu) | ((v & 0xff00u) << 8); };
                    const std::uint32_t k{pair(sk[j])};
                    h[(r0 + 7 * j) * kTileW + lx] = (k << 1) + k + pair(sn[j]);
                }
            }
        }
    }
    __syncthreads();
    if (!active) {
        return;
    }
    const XybPowers pw{tab};
    const float neg_cbrt_bias{-pw.cbrt(kOpsinBias)};
    // (1/255) / 16, exact: the 1/16 of the sum folded into the scale.
    constexpr float kScale{(1.0f / 255.0f) * 0.0625f};
    const auto pixel = [&](std::uint32_t l, std::uint32_t hk, std::uint32_t hn, int i) {
        std::uint32_t kn{hk + hn};
        asm("" : "+v"(kn));  // two adds, not one quarter-rate v_mad_u64_u32
        const std::uint32_t v{(hk << 1) + kn};
        const float yv{static_cast<float>(l) * (1.0f / 255.0f)};
        const float cb{static_cast<float>(v & 0xffffu) * kScale - 128.0f / 255.0f};
        const float cr{static_cast<float>(v >> 16) * kScale - 128.0f / 255.0f};
        pixel_to_xyb(yv, cb, cr, S.a.xyb[0][i], S.a.xyb[1][i], S.a.xyb[2][i], pw, neg_cbrt_bias);
    };
    if (interior) {
        // Tile row ly lies in chroma row (ly + 2) / 2 of the tile's; its
        // neighbour is the next row for odd ly, the one before for even ly.
        // Rows r0 + 7 k alternate in parity: two base rows, 7 rows further
        // every second step.
        const int ke{((r0 + 2) >> 1) * kTileW + lx}, ko{((r0 + 9) >> 1) * kTileW + lx};
        const int de{(r0 & 1) != 0 ? kTileW : -kTileW};
        const int ne{ke + de}, no{ko - de};
#pragma unroll
        for (int k{0}; k < kPix; ++k) {
            if (7 * k + 6 < kTileW || r0 + 7 * k < kTileW) {
                const int at{(k >> 1) * 7 * kTileW};
                pixel(lu[k], h[((k & 1) != 0 ? ko : ke) + at], h[((k & 1) != 0 ? no : ne) + at],
                      r0 * kTileW + lx + 7 * k * kTileW);
            }
        }
        return;
    }
#pragma unroll 1
    for (int ly{r0}; ly < kTileW; ly += 7) {
        int gy{py0 + ly - kHalo};
        gy = gy < 0 ? 0 : (gy >= H ? H - 1 : gy);
        const std::uint32_t l{luma[static_cast<std::size_t>(static_cast<std::uint32_t>(gy)) * luma_pitch +
                                   static_cast<std::uint32_t>(gx)]};
        const int ky{gy >> 1};
        const int ny{(gy & 1) != 0 ? (ky + 1 < ch ? ky + 1 : ch - 1) : (ky > 0 ? ky - 1 : 0)};
        pixel(l, h[(ky - cy0) * kTileW + lx], h[(ny - cy0) * kTileW + lx], ly * kTileW + lx);
    }
}

// Step 2: inverse gaborish of the three channels (gaborish.h:16-28; tap order
// frontend_transform.cu:30-48).  Thread (gy, gx) = (tid / 8, tid % 8) returns
// the four outputs of row gy, columns 4 gx .. 4 gx + 3 of each channel.
__device__ __forceinline__ void gaborish_tile(const RegionShared& S, int tid, float4 (&out)[3]) {
    constexpr float k0{-0.09495815671340026f}, k1{-0.041031725066768575f};
    constexpr float k2{0.013710004822696948f}, k3{0.006510206083837737f};
    constexpr float k4{-0.0014789063378272242f};
    constexpr float nm{1.0f / (1.0f + 4.0f * (k0 + k1 + k2 + k4 + 2.0f * k3))};
    constexpr float wc{nm}, wr{nm * k0}, wr2{nm * k2}, wd{nm * k1}, wl{nm * k3}, wd2{nm * k4};
    // From the five input rows gy - 2 .. gy + 2, columns 4 gx - 2 .. 4 gx + 5
    // (two aligned 16-byte reads per row; the tile's row pitch is 36 floats).
    const int gx{tid & 7}, gy{tid >> 3};
#pragma unroll
    for (int c{0}; c < 3; ++c) {
        const float* const base{&S.a.xyb[c][gy * kTileW + 4 * gx]};
        float r[5][8];
#pragma unroll
        for (int dy{0}; dy < 5; ++dy) {
            const float4 a{*reinterpret_cast<const float4*>(base + dy * kTileW)};
            const float4 b{*reinterpret_cast<const float4*>(base + dy * kTileW + 4)};
            r[dy][0] = a.x;
            r[dy][1] = a.y;
            r[dy][2] = a.z;
            r[dy][3] = a.w;
            r[dy][4] = b.x;
            r[dy][5] = b.y;
            r[dy][6] = b.z;
            r[dy][7] = b.w;
        }
        float o[4];
#pragma unroll
        for (int k{0}; k < 4; ++k) {
#define AT(dx, dy) r[(dy) + 2][k + 2 + (dx)]
            const float e{AT(-1, 0) + AT(1, 0) + AT(0, -1) + AT(0, 1)};
            const float r2{AT(-2, 0) + AT(2, 0) + AT(0, -2) + AT(0, 2)};
            const float dg{AT(-1, -1) + AT(1, -1) + AT(-1, 1) + AT(1, 1)};
            const float l8{AT(-2, -1) + AT(2, -1) + AT(-2, 1) + AT(2, 1) + AT(-1, -2) + AT(1, -2) +
                           AT(-1, 2) + AT(1, 2)};
            const float d4{AT(-2, -2) + AT(2, -2) + AT(-2, 2) + AT(2, 2)};
            o[k] = wc * AT(0, 0) + wr * e + wr2 * r2 + wd * dg + wl * l8 + wd2 * d4;
#undef AT
        }
        out[c] = float4{o[0], o[1], o[2], o[3]};
        // Computed here: sunk to their use, they would keep all three
        // channels' inputs (120 registers) alive.
        asm volatile("" : "+v"(out[c].x), "+v"(out[c].y), "+v"(out[c].z), "+v"(out[c].w));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The outputs into the sharpened planes (every thread has read the XYB tile,
// whose space they take).
__device__ __forceinline__ void store_sharp(RegionShared& S, int tid, const float4 (&out)[3]) {
    const int gx{tid & 7}, gy{tid >> 3};
#pragma unroll
    for (int c{0}; c < 3; ++c) {
        *reinterpret_cast<float4*>(&plane_of(S, c)[sp_index(gy, 4 * gx)]) = out[c];
    }
}

// ---------------------------------------------------------------------------
// The plain form's DCTs on the matrix cores, exact.  v_mfma_f32_16x16x4_f32
// adds A[i][k] B[k][j], k = 0..3, to D[i][j] as the fmaf chain in k order (the
// hardware's result equals the chain bit for bit: 100 M results of 4 to 64
// steps, denormal products and exact cancellations among them), so a sequence
// of steps over c gives dct_line's chain.  Lane l supplies A[l % 16][l / 16]
// and B[l / 16][l % 16] and holds D[4 (l / 16) + u][l % 16], u = 0..3.
//
// A row pass T = P A^T takes the pixels as the first operand and the basis
// row of the lane's frequency as the second, the column pass C = A T the same
// basis values as the first operand.  Between them T moves from "row 4 g + u
// in register u of lane group g" to "row 4 u + g" (the natural order of the
// chain): a 4 x 4 transpose of registers and lane groups, four permlane
// swaps, no LDS.  A 16 x 16 quad is one tile per pass: a DCT16, or four DCT8s
// with a block-diagonal basis (a chain's zero steps add +0 to a sum that is
// never -0).  A DCT32 quadrant takes two row-pass tiles.  Every wave works on
// one quad and one quadrant.  With K = 1 steps, the DCT32 in wave 0 alone
// (1,024 clocks a pass), the DCT8s on the VALU and the row passes through LDS
// lines the region kernel took 179 us at 3840x2160, in this form 164.
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4v ex_step(float a, float b, f4v acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

__device__ __forceinline__ void ex_swap32(float& a, float& b) {
    const auto r{__builtin_amdgcn_permlane32_swap(f2u(a), f2u(b), false, false)};
    a = u2f(r[0]);
    b = u2f(r[1]);
}

__device__ __forceinline__ void ex_swap16(float& a, float& b) {
    const auto r{__builtin_amdgcn_permlane16_swap(f2u(a), f2u(b), false, false)};
    a = u2f(r[0]);
    b = u2f(r[1]);
}

// Register u of lane group g <-> register g of lane group u.
__device__ __forceinline__ void ex_turn(float (&t)[4]) {
    ex_swap32(t[0], t[2]);
    ex_swap32(t[1], t[3]);
    ex_swap16(t[0], t[1]);
    ex_swap16(t[2], t[3]);
}

// Pixels (row, col0 + 4 s + l / 16), s = 0 .. kSteps - 1 (col0 0 or 16, 0
// only with eight steps): the 16-byte group index of step s is step 0's with
// s XORed in.
template <int kSteps>
__device__ __forceinline__ void ex_pixels(const float* plane, int row, int col0, int lane, float (&p)[kSteps]) {
    const int base{row * kSP + (((col0 >> 2) ^ sp_swz(row)) << 2) + (lane >> 4)};
#pragma unroll
    for (int s{0}; s < kSteps; ++s) {
        p[s] = plane[base ^ (4 * s)];
    }
}

__device__ __forceinline__ f4v ex_rows(const float (&p)[4], const float4& b) {
    f4v t{0.0f, 0.0f, 0.0f, 0.0f};
    t = ex_step(p[0], b.x, t);
    t = ex_step(p[1], b.y, t);
    t = ex_step(p[2], b.z, t);
    return ex_step(p[3], b.w, t);
}

__device__ __forceinline__ f4v ex_cols(const float4& a, const f4v& rows, f4v acc) {
    float t[4]{rows[0], rows[1], rows[2], rows[3]};
    ex_turn(t);
    acc = ex_step(a.x, t[0], acc);
    acc = ex_step(a.y, t[1], acc);
    acc = ex_step(a.z, t[2], acc);
    return ex_step(a.w, t[3], acc);
}

// The 16x16 quad at (row0, col0) of `plane` through the lane's basis values:
// lane l returns C[4 (l / 16) + u][l % 16] (row = vertical frequency).
__device__ __forceinline__ f4v ex_quad(const float* plane, int row0, int col0, const float4& b, int lane) {
    float p[4];
    ex_pixels<4>(plane, row0 + (lane & 15), col0, lane, p);
    return ex_cols(b, ex_rows(p, b), f4v{0.0f, 0.0f, 0.0f, 0.0f});
}

// Lane values of the 32-point basis for frequencies 16 f .. 16 f + 15.
struct Ex32 {
    float4 lo, hi;
};
__device__ __forceinline__ Ex32 ex_basis32(int f, int lane) {
    const float4* const b{reinterpret_cast<const float4*>(&g_tables.ex32[f][lane][0])};
    return {b[0], b[1]};
}

// DCT32 of the region's plane: the row-pass tiles of horizontal frequencies
// 16 fxb .. (rows 0..15 and 16..31), the two chains side by side.
__device__ __forceinline__ void ex_rows32(const float* plane, const Ex32& b, int lane, f4v (&t)[2]) {
    float p[2][8];
    ex_pixels<8>(plane, lane & 15, 0, lane, p[0]);
    ex_pixels<8>(plane, 16 + (lane & 15), 0, lane, p[1]);
    const float bv[8]{b.lo.x, b.lo.y, b.lo.z, b.lo.w, b.hi.x, b.hi.y, b.hi.z, b.hi.w};
    t[0] = t[1] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s{0}; s < 8; ++s) {
        t[0] = ex_step(p[0][s], bv[s], t[0]);
        t[1] = ex_step(p[1][s], bv[s], t[1]);
    }
}

__device__ __forceinline__ f4v ex_cols32(const Ex32& a, const f4v (&t)[2]) {
    return ex_cols(a.hi, t[1], ex_cols(a.lo, t[0], f4v{0.0f, 0.0f, 0.0f, 0.0f}));
}

// Output tiles (0, 16 fxb) and (16, 16 fxb) (vertical, horizontal frequency
// origins) into c[0], c[1].
__device__ __forceinline__ void ex_dct32(const float* plane, int fxb, int lane, f4v (&c)[2]) {
    f4v t[2];
    ex_rows32(plane, ex_basis32(fxb, lane), lane, t);
    c[0] = ex_cols32(ex_basis32(0, lane), t);
    c[1] = ex_cols32(ex_basis32(1, lane), t);
}

// Lane l - 16's value, for lanes of the odd rows of 16.
__device__ __forceinline__ float from_row_above(float v) {
    const auto r{__builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false)};
    return u2f(r[0]);
}

// ---------------------------------------------------------------------------
// Matrix-core DCT form with FP16 operands (kModeMfma16).  Every transform is
// built from v_mfma_f32_16x16x16_f16 steps: D[i][j] += sum_k A[i][k] B[k][j]
// over a 16x16x16 tile, lane l supplying A[l % 16][4 (l / 16) + 0..3] and
// B[4 (l / 16) + 0..3][l % 16] and holding D[4 (l / 16) + u][l % 16], u =
// 0..3.  A row pass T = P B^T takes the pixels as A and the basis as B; the
// column pass C = B T takes the basis as A and T, exactly as the row pass
// leaves it in the lanes, as B: no data moves between the passes.  A 16x16
// quad is one tile per pass (basis A16, or blockdiag(A8, A8) for its four
// DCT8s); a DCT32 output tile is two K = 16 steps per pass.  Every operand is
// split into FP16 hi + lo (x = hi + lo to about 2^-22 relative) and each
// product is lo*hi + hi*lo + hi*hi in FP32 (lo*lo dropped), so the DC and
// the low frequencies keep about FP32 accuracy.  Pixels are scaled by 1/4
// (exact) into |x| <= 1 (sharpened XYB stays within 2.97 * 0.9) and the
// results by 4.
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
constexpr float kMfScale = 0.25f;

struct MfOp {
    h4v hi, lo;
};

__device__ __forceinline__ MfOp mf_split(float a, float b, float c, float d) {
    MfOp o;
    const float v[4]{a, b, c, d};
#pragma unroll
    for (int i{0}; i < 4; ++i) {
        const _Float16 h{static_cast<_Float16>(v[i])};
        o.hi[i] = h;
        o.lo[i] = static_cast<_Float16>(v[i] - static_cast<float>(h));
    }
    return o;
}

// Row r of an FP16 basis table pair (n columns), columns c0 .. c0 + 3.
__device__ __forceinline__ MfOp mf_basis(const std::uint16_t* hi, const std::uint16_t* lo, int n, int r, int c0) {
    MfOp o;
    o.hi = *reinterpret_cast<const h4v*>(hi + r * n + c0);
    o.lo = *reinterpret_cast<const h4v*>(lo + r * n + c0);
    return o;
}

// acc + A B with A = a.hi + a.lo, B = b.hi + b.lo; the small products first.
__device__ __forceinline__ f4v mf_mma(const MfOp& a, const MfOp& b, f4v acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a.lo, b.hi, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a.hi, b.lo, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a.hi, b.hi, acc, 0, 0, 0);
}

// Pixels (row, c0 .. c0 + 3) of a sharpened plane, scaled and split.
__device__ __forceinline__ MfOp mf_pixels(const float* plane, int row, int c0) {
    const float4 p{*reinterpret_cast<const float4*>(plane + sp_index(row, c0))};
    return mf_split(p.x * kMfScale, p.y * kMfScale, p.z * kMfScale, p.w * kMfScale);
}

// The 16x16 quad at (row0, col0) of `plane` through basis tables (hi, lo):
// lane l returns C[4 (l / 16) + u][l % 16] (row = vertical frequency).
__device__ __forceinline__ f4v mf_quad(const float* plane, int row0, int col0, const std::uint16_t* hi,
                                       const std::uint16_t* lo, int lane) {
    const int m{lane & 15}, g{lane >> 4};
    const MfOp b{mf_basis(hi, lo, 16, m, 4 * g)};
    const f4v zero{0.0f, 0.0f, 0.0f, 0.0f};
    const f4v t{mf_mma(mf_pixels(plane, row0 + m, col0 + 4 * g), b, zero)};
    const f4v c{mf_mma(b, mf_split(t[0], t[1], t[2], t[3]), zero)};
    return c * (1.0f / kMfScale);
}

// DCT32 of the region's plane: output tiles (0, fx0) and (16, fx0) (vertical,
// horizontal frequency origins) into c[0], c[1]; with `both` false only
// (fy0, fx0) into c[0].
__device__ __forceinline__ void mf_dct32(const float* plane, int fx0, int fy0, bool both, int lane, f4v (&c)[2]) {
    const int m{lane & 15}, g{lane >> 4};
    const std::uint16_t* hi{g_tables.mf32[0]};
    const std::uint16_t* lo{g_tables.mf32[1]};
    const f4v zero{0.0f, 0.0f, 0.0f, 0.0f};
    MfOp t[2];
#pragma unroll
    for (int h{0}; h < 2; ++h) {  // row-pass tiles at rows 16 h, frequencies fx0..
        f4v acc{zero};
#pragma unroll
        for (int k{0}; k < 2; ++k) {
            acc = mf_mma(mf_pixels(plane, 16 * h + m, 16 * k + 4 * g), mf_basis(hi, lo, 32, fx0 + m, 16 * k + 4 * g),
                         acc);
        }
        t[h] = mf_split(acc[0], acc[1], acc[2], acc[3]);
    }
#pragma unroll
    for (int o{0}; o < 2; ++o) {
        if (o == 1 && !both) {
            break;
        }
        const int f0{both ? 16 * o : fy0};
        f4v acc{zero};
#pragma unroll
        for (int h{0}; h < 2; ++h) {
            acc = mf_mma(mf_basis(hi, lo, 32, f0 + m, 16 * h + 4 * g), t[h], acc);
        }
        c[o] = acc * (1.0f / kMfScale);
    }
}

// Lane l's four elements of a quad result, as (block j of the quad, element
// e of the block's transform): DCT16 (n = 16) e = fx * 16 + fy, j = 0; four
// DCT8s (n = 8) j = 2 (fy / 8) + fx / 8, e = (fx % 8) * 8 + fy % 8.
__device__ __forceinline__ void mf_quad_element(int lane, int u, int n, int& j, int& e) {
    const int fx{lane & 15}, fy{4 * (lane >> 4) + u};
    if (n == 16) {
        j = 0;
        e = fx * 16 + fy;
    } else {
        j = 2 * (fy >> 3) + (fx >> 3);
        e = (fx & 7) * 8 + (fy & 7);
    }
}

// ---------------------------------------------------------------------------
// The learned transform selection (kModeLearned) and the feature export of
// the plain path that trains it.  Features of a region, 6 per 8x8 block b
// (region raster, 16 blocks), all from the block's DCT8 of the sharpened Y
// (the selection's DCT8 candidate, C[e] with e = fx * 8 + fy) and its
// selection terms:
//   f[6b + 0] = log2(1 + 4096 var)     var  = sum over AC of C^2
//   f[6b + 1] = log2(1 + 1024 grad)    grad = (64 / 112) sum (l[fx] + l[fy]) C^2
//   f[6b + 2] = log2(1 + 64 cost8)     the block's DCT8 RD cost
//   f[6b + 3] = log2(1 + 262144 dist)  dist = sum of squared quantization errors
//   f[6b + 4] = log2(1 + rate)         rate = sum of the rate terms
//   f[6b + 5] = 4 C[0]                 the block's mean
// With the basis' normalization (C = O P O^T / 8, O orthonormal) var is the
// pixels' variance and grad the mean squared difference of horizontally and
// vertically adjacent pixels inside the block (112 pairs): the DCT-II
// diagonalizes the path's difference operator with eigenvalues
// l[k] = 4 sin^2(pi k / 16).  Blocks past the frame's edge have all six at 0.
struct MlpWeights {
    std::uint16_t w1[64 * 96];  // FP16 bit patterns, row-major [hidden][input]
    std::uint16_t w2[7 * 64];   // [output][hidden]
    float b1[64];
    float b2[8];
    float threshold;  // |logit| below which a decision is not confident
};

__device__ __align__(16) MlpWeights g_mlp;

__device__ __forceinline__ float h2f(std::uint16_t h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, h));
}

// One thread's share of the network's weights, read at the kernel's start
// (the learned forms), so that no read waits inside the decision: layer 1's
// 24 weights of hidden unit tid / 4 (inputs 24 (tid % 4) ..) and its bias,
// and layer 2's 8 weights of output tid / 8 (hidden 8 (tid % 8) ..; threads
// below 56) and its bias.
struct MlpRegs {
    uint4 w1[3];
    uint4 w2;
    float b1, b2;
};

__device__ __forceinline__ MlpRegs mlp_load(int tid) {
    MlpRegs r;
    const int j{tid >> 2}, k{tid & 3};
    const std::uint16_t* const w{g_mlp.w1 + j * 96 + 24 * k};
#pragma unroll
    for (int i{0}; i < 3; ++i) {
        r.w1[i] = *reinterpret_cast<const uint4*>(w + 8 * i);
    }
    const int o{tid < 56 ? tid >> 3 : 0}, p{tid & 7};
    r.w2 = *reinterpret_cast<const uint4*>(g_mlp.w2 + o * 64 + 8 * p);
    r.b1 = g_mlp.b1[j];
    r.b2 = g_mlp.b2[o];
    return r;
}

// (64 / 112) l[k] of the gradient feature, k = 0..7.
__device__ __forceinline__ float grad_weight(int k) {
    constexpr float w[8]{0.0f, 0.08699481934309006f, 0.33473509550094604f, 0.7055046558380127f,
                         1.1428571939468384f, 1.5802096128463745f, 1.950979232788086f, 2.1987195014953613f};
    return w[k];
}

// Block b's raw sums (var, grad, dist, rate, mean) into S.b.s.feat[6 b ..]; the
// cost sits in S.cost8.
__device__ __forceinline__ void feature_store(RegionShared& S, int b, float var, float grad, float dist, float rate,
                                              float mean) {
    S.b.s.feat[6 * b + 0] = var;
    S.b.s.feat[6 * b + 1] = grad;
    S.b.s.feat[6 * b + 3] = dist;
    S.b.s.feat[6 * b + 4] = rate;
    S.b.s.feat[6 * b + 5] = mean;
}

// The raw sums -> the 96 features in S.b.s.feat (every thread calls this;
// barriers inside).
__device__ __forceinline__ void feature_finish(RegionShared& S, int tid, int bx0, int by0, int bw, int bh) {
    float f[6]{};
    if (tid < 16) {
        const int bx{tid & 3}, by{tid >> 2};
        if (bx0 + bx < bw && by0 + by < bh) {
            const float* s{&S.b.s.feat[6 * tid]};
            const float c8{S.cost8[((by >> 1) * 2 + (bx >> 1)) * 4 + (by & 1) * 2 + (bx & 1)]};
            f[0] = log2_det(1.0f + 4096.0f * fmaxf(s[0], 0.0f));
            f[1] = log2_det(1.0f + 1024.0f * fmaxf(s[1], 0.0f));
            f[2] = log2_det(1.0f + 64.0f * fmaxf(c8, 0.0f));
            f[3] = log2_det(1.0f + 262144.0f * fmaxf(s[3], 0.0f));
            f[4] = log2_det(1.0f + fmaxf(s[4], 0.0f));
            f[5] = 4.0f * s[5];
        }
    }
    __syncthreads();
    if (tid < 16) {
#pragma unroll
        for (int k{0}; k < 6; ++k) {
            S.b.s.feat[6 * tid + k] = f[k];
        }
    }
    __syncthreads();
}

// The network on the region's features and, when every decision it takes is
// confident (|logit| >= threshold for the root where a DCT32 fits and for
// each quad where a DCT16 fits), the transform map in S.acs.  Returns that
// confidence (the same value in every thread).  `hid` is LDS scratch of 72
// floats.  Every thread calls this; barriers inside.
__device__ __forceinline__ bool mlp_decide(RegionShared& S, const FrameParams& prm, const MlpRegs& mr, float* hid,
                                           int tid, int bx0, int by0, int bw, int bh) {
    {
        const int j{tid >> 2}, k{tid & 3};
        const float* const x{&S.b.s.feat[24 * k]};
        float s{0.0f};
#pragma unroll
        for (int i{0}; i < 24; i += 8) {
            const uint4 pw{mr.w1[i / 8]};
            const std::uint32_t word[4]{pw.x, pw.y, pw.z, pw.w};
#pragma unroll
            for (int h{0}; h < 4; ++h) {
                s = __builtin_fmaf(h2f(static_cast<std::uint16_t>(word[h] & 0xffffu)), x[i + 2 * h], s);
                s = __builtin_fmaf(h2f(static_cast<std::uint16_t>(word[h] >> 16)), x[i + 2 * h + 1], s);
            }
        }
        s = add_down_row<2>(s);
        s = add_down_row<1>(s);
        if (k == 0) {
            hid[j] = fmaxf(s + mr.b1, 0.0f);
        }
    }
    __syncthreads();
    if (tid < 56) {
        const int o{tid >> 3}, p{tid & 7};
        const std::uint32_t word[4]{mr.w2.x, mr.w2.y, mr.w2.z, mr.w2.w};
        float s{0.0f};
#pragma unroll
        for (int q{0}; q < 8; ++q) {
            const std::uint32_t w{word[q >> 1]};
            s = __builtin_fmaf(h2f(static_cast<std::uint16_t>((q & 1) != 0 ? w >> 16 : w & 0xffffu)), hid[8 * p + q], s);
        }
        s = add_down_row<4>(s);
        s = add_down_row<2>(s);
        s = add_down_row<1>(s);
        if (p == 0) {
            hid[64 + o] = s + mr.b2;
        }
    }
    __syncthreads();
    if (tid == 0) {
        const float* z{hid + 64};
        const float th{g_mlp.threshold};
        const std::uint32_t force{(prm.mode & kModeForceMask) >> kModeForceShift};
        const bool fit32{bx0 + 4 <= bw && by0 + 4 <= bh};
        bool ok{force == 0};
        const float root{z[1] - z[0]};
        ok = ok && (!fit32 || fabsf(root) >= th);
        const bool use32{fit32 && root > 0.0f};
        int choice[4];
        for (int q{0}; q < 4; ++q) {
            const int qx{q & 1}, qy{q >> 1};
            const bool fit16{bx0 + 2 * qx + 2 <= bw && by0 + 2 * qy + 2 <= bh};
            choice[q] = fit16 && z[2 + q] > 0.0f ? 16 : 8;
            if (!use32) {
                ok = ok && (!fit16 || fabsf(z[2 + q]) >= th);
            }
        }
        if (ok) {
            if (use32) {
                for (int b{0}; b < 16; ++b) {
                    S.acs[b] = b == 0 ? 32 : 0;
                }
            } else {
                for (int q{0}; q < 4; ++q) {
                    const int ox{2 * (q & 1)}, oy{2 * (q >> 1)};
                    if (choice[q] == 16) {
                        S.acs[oy * 4 + ox] = 16;
                        S.acs[oy * 4 + ox + 1] = 0;
                        S.acs[(oy + 1) * 4 + ox] = 0;
                        S.acs[(oy + 1) * 4 + ox + 1] = 0;
                    }
                }
            }
        }
        S.learned_ok = ok ? 1 : 0;
    }
    __syncthreads();
    return S.learned_ok != 0;
}

// Training rows of the plain path: the region's 96 features, then its labels
// (12 floats: DCT32 at the root, DCT16 per quad as the heuristic chose it,
// the mean log2 quant field of the region's blocks, the root mask (a DCT32
// fits), the quad masks (a DCT16 fits), 0).
constexpr int kFeatRow = 96 + 12;

__device__ __forceinline__ void export_features(const RegionShared& S, float* out, int region, int tid, int bx0,
                                                int by0, int bw, int bh) {
    float* const row{out + static_cast<std::size_t>(region) * kFeatRow};
    if (tid < 96) {
        row[tid] = S.b.s.feat[tid];
    } else if (tid < 108) {
        const int k{tid - 96};
        float v{0.0f};
        if (k == 0) {
            v = S.acs[0] == 32 ? 1.0f : 0.0f;
        } else if (k <= 4) {
            v = S.choice[k - 1] == 16 ? 1.0f : 0.0f;
        } else if (k == 5) {
            float s{0.0f};
            int n{0};
            for (int b{0}; b < 16; ++b) {
                if (bx0 + (b & 3) < bw && by0 + (b >> 2) < bh) {
                    s += log2_det(static_cast<float>(S.blkqf[b]));
                    ++n;
                }
            }
            v = s / static_cast<float>(n);
        } else if (k == 6) {
            v = bx0 + 4 <= bw && by0 + 4 <= bh ? 1.0f : 0.0f;
        } else if (k <= 10) {
            const int q{k - 7};
            v = bx0 + 2 * (q & 1) + 2 <= bw && by0 + 2 * (q >> 1) + 2 <= bh ? 1.0f : 0.0f;
        }
        row[96 + k] = v;
    }
}

template <bool kMf16, bool kLearned>
__device__ __attribute__((always_inline)) inline void region_kernel_body(const Wg& wg, 
    Geometry geo, FrameParams prm, const std::uint8_t* __restrict__ luma, std::size_t luma_pitch,
    const std::uint8_t* __restrict__ chroma, std::size_t chroma_pitch,
    std::uint16_t* __restrict__ coeffs, std::int8_t* __restrict__ acs_out,
    std::int32_t* __restrict__ qf_out, float* __restrict__ cfl_part, std::uint32_t* __restrict__ list_count,
    Clears clr, float* __restrict__ feat_out) {
    __shared__ RegionShared S;
    clear_words(clr, wg);  // every workgroup of the grid takes part
    const int tid{static_cast<int>(threadIdx.x)};
    if (wg.x == 0 && tid < 2 && list_count != nullptr) {
        list_count[tid] = 0;  // the quantizer's item lists, appended after this kernel
    }
    const int wu{__builtin_amdgcn_readfirstlane(tid >> 6)};  // the wave (uniform)
    [[maybe_unused]] MlpRegs mlp_regs;
    if constexpr (kLearned) {
        mlp_regs = mlp_load(tid);
    }
    const int lane{tid & 63};
    // Workgroup i runs on XCD i mod 8: give each XCD a contiguous run of
    // regions so that rows shared by neighbouring regions stay in one L2.
    const int nreg{static_cast<int>(geo.rw * geo.rh)};
    const int per_xcd{(nreg + 7) / 8};
    const int region{static_cast<int>(wg.x & 7u) * per_xcd + static_cast<int>(wg.x >> 3)};
    if (region >= nreg) {
        return;
    }
    const int rx{region % static_cast<int>(geo.rw)};
    const int ry{region / static_cast<int>(geo.rw)};
    const int px0{rx * 32}, py0{ry * 32};
    const int W{static_cast<int>(geo.width)}, H{static_cast<int>(geo.height)};
    const int bw{static_cast<int>(geo.bw)}, bh{static_cast<int>(geo.bh)};
    const int bx0{rx * 4}, by0{ry * 4};

    // 1. NV12 -> XYB over the 36x36 tile (2-pixel halo, clamped coordinates).
    xyb_tile(S, luma, luma_pitch, chroma, chroma_pitch, px0, py0, W, H, tid);
    if (tid < 16) {
        S.acs[tid] = 8;
    }
    __syncthreads();

    CJX_REGION_CUT_AT(1)
    // 2. Inverse gaborish (gaborish.h:16-28; tap order frontend_transform.cu:30-48),
    //    its results kept in registers while the XYB tile is still read.
    float4 sharp[3];
    gaborish_tile(S, tid, sharp);
    {
        // 3a. AQ pre-erosion terms per interior pixel (frontend_fused.cu:118-137)
        //     and their 4x4 cell sums in row order: four lanes per cell, one
        //     per row; row dy continues the running sum of row dy - 1.
        const int cell{tid >> 2}, dy{tid & 3};
        const int row{(cell >> 3) * 4 + dy}, col0{(cell & 7) * 4};
        float m[4];
#pragma unroll
        for (int dx{0}; dx < 4; ++dx) {
            const float* s{&S.a.xyb[1][(row + kHalo) * kTileW + col0 + dx + kHalo]};
            const float yv{s[0]};
            const float base{0.25f * (s[kTileW] + s[-kTileW] + s[-1] + s[1])};
            float diff{ratio_cbrt_gamma(yv + 0.019f, false) * (yv - base)};
            diff *= diff;
            diff = fminf(diff, 0.2f);
            m[dx] = masking_sqrt(diff);
        }
        float sum{0.0f};
#pragma unroll
        for (int k{0}; k < 4; ++k) {
            const float prev{from_lane_below(sum)};
            if (dy == k) {
                float acc{k == 0 ? 0.0f : prev};
                acc += m[0];
                acc += m[1];
                acc += m[2];
                acc += m[3];
                sum = acc;
            }
        }
        if (dy == 3) {
            S.b.aq.cells[cell] = 0.25f * sum;
        }
    }

    CJX_REGION_CUT_AT(2)
    // 3b. Per-block modulation and the quant integer (frontend_fused.cu:117-203):
    //     the per-pixel sums as wave sums, then (wave 0, after the barrier)
    //     the 64 cells' fuzzy erosion and the 16 blocks' final step in
    //     parallel lanes (a block's four erosion terms sum as
    //     (e0 + e2) + (e1 + e3), which is the wave tree over four non-zero
    //     lanes).
    {
        // Wave w takes blocks (w, j), j = 0..3, one pixel per lane.
        const int fx{lane & 7}, fy{lane >> 3};
        const int idx0{(fy + kHalo) * kTileW + wu * 8 + fx + kHalo};
        float hf[4], gm[4], bl[4];
#pragma unroll
        for (int j{0}; j < 4; ++j) {
            const int idx{idx0 + j * 8 * kTileW};
            const float yv{S.a.xyb[1][idx]}, xv{S.a.xyb[0][idx]}, bv{S.a.xyb[2][idx]};
            // Differences inside the block; the tile's halo makes the reads
            // past its edge valid.
            const float right{fminf(0.0206f, fabsf(yv - S.a.xyb[1][idx + 1]))};
            const float down{fminf(0.0206f, fabsf(yv - S.a.xyb[1][idx + kTileW]))};
            hf[j] = (fx < 7 ? right : 0.0f) + (fy < 7 ? down : 0.0f);
            const float iny{yv + 0.16f};
            gm[j] = ratio_cbrt_gamma(iny - xv, true) + ratio_cbrt_gamma(iny + xv, true);
            const float pye{yv + 0.084381641171960495f + fabsf(xv)};
            bl[j] = bv > pye ? fminf(bv - pye, 0.027121074570634722f) : 0.0f;
        }
        // Sums of blocks j = 0, 2, 1, 3 in lanes 0, 16, 32, 48.
        const float hs{wave_sum4(hf[0], hf[1], hf[2], hf[3])};
        const float gs{wave_sum4(gm[0], gm[1], gm[2], gm[3])};
        const float bs{wave_sum4(bl[0], bl[1], bl[2], bl[3])};
        if ((lane & 15) == 0) {
            const int j{((lane >> 3) & 2) | (lane >> 5)};
            S.b.aq.blk[4 * j + wu][0] = hs;
            S.b.aq.blk[4 * j + wu][1] = gs * (0.5f / 64.0f);
            S.b.aq.blk[4 * j + wu][2] = bs;
        }
    }
    __syncthreads();  // the XYB tile is dead from here on
    store_sharp(S, tid, sharp);
    if (tid < 64) {
        S.b.aq.ero[tid] = erosion_cell(S.b.aq.cells, tid & 7, tid >> 3, prm);
        wave_sync();
    }
    if (tid < 16) {
        const int lb{tid};
        const int lbx{lb & 3}, lby{lb >> 2};
        if (bx0 + lbx < bw && by0 + lby < bh) {
            const float e0{S.b.aq.ero[(2 * lby) * 8 + 2 * lbx]}, e1{S.b.aq.ero[(2 * lby) * 8 + 2 * lbx + 1]};
            const float e2{S.b.aq.ero[(2 * lby + 1) * 8 + 2 * lbx]}, e3{S.b.aq.ero[(2 * lby + 1) * 8 + 2 * lbx + 1]};
            const float aq{(e0 + e2) + (e1 + e3)};
            float blue_sum{S.b.aq.blk[lb][2]};
            constexpr float k_limit{0.027121074570634722f};
            if (blue_sum >= 32.0f * k_limit) {
                blue_sum = 64.0f * k_limit - blue_sum;
            }
            constexpr float k_max_limit{15.398788439047934f};
            if (blue_sum >= k_max_limit * k_limit) {
                blue_sum = k_max_limit * k_limit;
            }
            float ov{compute_mask(aq)};
            ov += S.b.aq.blk[lb][0] * -0.38f + 0.42f;
            ov += 0.1005613337192697f * log2_det(S.b.aq.blk[lb][1]);
            ov += blue_sum * 0.14207000358439159f;
            const float qval{exp_det(ov) * prm.mul_pb + prm.add_pb};
            int qi{static_cast<int>(qval * prm.inv_global_scale + 0.5f)};
            qi = qi < 1 ? 1 : (qi > 256 ? 256 : qi);
            qf_out[static_cast<std::size_t>(by0 + lby) * bw + bx0 + lbx] = qi;
            S.blkqf[lb] = qi;
        }
    }

    CJX_REGION_CUT_AT(3)
    // 4. Transform selection on the sharpened Y (transform_select_impl.cuh:49-201).
    //    Wave w transforms quad w as four DCT8s and as one DCT16, and quadrant
    //    w of the DCT32 (vertical frequencies 16 (w / 2).., horizontal ones
    //    16 (w % 2)..), on the matrix cores; the terms stay in registers and
    //    are summed there.  Learned: the DCT8s and their costs, the region's
    //    features and the network first; the DCT16 and DCT32 candidates only
    //    where the network is not confident (the heuristic decides there).
    __syncthreads();  // the sharpened planes are complete, the AQ terms dead
    CJX_REGION_CUT_AT(6)
    const int grp{lane >> 4}, t16{lane & 15};
    const float* const yp{plane_of(S, 1)};
    const int qrow{(wu >> 1) * 16}, qcol{(wu & 1) * 16};  // the wave's quad
    const bool want_features{kLearned || feat_out != nullptr};
    // Four consecutive elements e0 .. e0 + 3 (e0 a multiple of 4) of an array.
    const auto store4 = [](_Float16* dst, int e0, const f4v& c) {
        const h4v h{static_cast<_Float16>(c[0]), static_cast<_Float16>(c[1]), static_cast<_Float16>(c[2]),
                    static_cast<_Float16>(c[3])};
        *reinterpret_cast<h4v*>(dst + cpad(e0)) = h;
    };
    // Plain pieces.  The costs' summation orders are fixed: a DCT8 column's
    // eight terms in order, then its block's eight columns as a lane tree; a
    // DCT16 lane's four terms (one column, fy = 4 g ..), then the wave tree;
    // for the DCT32 the four quadrants' terms of a lane (16 in order, wave 0's
    // quadrant first), then the wave tree.
    const auto ex_dct8_costs = [&](const f4v& c8) {
        // Lane group g holds rows 4 g + u of the quad: rows 0-3 of a block's
        // column in the even group, 4-7 in the odd one, which takes the even
        // one's running sums over.
        float v[4], wq[4], wi[4], d[4], rt[4];
        bool llf[4];
        int j, e0;
        mf_quad_element(lane, 0, 8, j, e0);
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            v[u] = c8[u];
            llf[u] = u == 0 && (lane & 7) == 0 && (grp & 1) == 0;  // the DC
        }
        selection_weights4(g_tables.wsel8, g_tables.wsel_inv8, e0, 0, wq, wi);
        selection_terms(v, llf, wq, wi, prm, d, rt);
        store4(coefy_of(S, 0), 256 * wu + 64 * j + e0, c8);
        const auto column = [&](const float (&x)[4]) {
            const float top{((x[0] + x[1]) + x[2]) + x[3]};
            return (((from_row_above(top) + x[0]) + x[1]) + x[2]) + x[3];  // in the odd groups
        };
        const auto sum8 = [](float x) { return add_down_row<1>(add_down_row<2>(add_down_row<4>(x))); };
        const float ad{sum8(column(d))}, ar{sum8(column(rt))};
        float fv{0.0f}, fg{0.0f}, dc{0.0f};
        if (want_features) {
            float c2[4];
#pragma unroll
            for (int u{0}; u < 4; ++u) {
                c2[u] = v[u] * v[u];
            }
            const int fx{lane & 7};
            const auto run = [&](float sv, float sg, float& ov, float& og) {
#pragma unroll
                for (int u{0}; u < 4; ++u) {
                    sv += llf[u] ? 0.0f : c2[u];
                    sg = __builtin_fmaf(grad_weight(fx) + grad_weight(4 * (grp & 1) + u), c2[u], sg);
                }
                ov = sv;
                og = sg;
            };
            float tv, tg;
            run(0.0f, 0.0f, tv, tg);
            run(from_row_above(tv), from_row_above(tg), fv, fg);
            fv = sum8(fv);
            fg = sum8(fg);
            dc = from_row_above(v[0]);
        }
        if ((lane & 7) == 0 && (grp & 1) != 0) {
            S.cost8[wu * 4 + j] = 64.0f * ad + 6.0e-4f * ar;
            if (want_features) {
                feature_store(S, (2 * (wu >> 1) + (j >> 1)) * 4 + 2 * (wu & 1) + (j & 1), fv, fg, ad, ar, dc);
            }
        }
    };
    const auto ex_dct16_costs = [&](const f4v& c16) {
        const int e0{t16 * 16 + 4 * grp};
        float v[4], wq[4], wi[4], d[4], rt[4];
        bool llf[4];
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            v[u] = c16[u];
            llf[u] = u < 2 && lane < 2;  // fx, fy < 2
        }
        selection_weights4(g_tables.wsel16, g_tables.wsel_inv16, e0, 0, wq, wi);
        selection_terms(v, llf, wq, wi, prm, d, rt);
        const float ad{((d[0] + d[1]) + d[2]) + d[3]}, ar{((rt[0] + rt[1]) + rt[2]) + rt[3]};
        const float sums{wave_sum4(ad, ar, 0.0f, 0.0f)};  // lanes 0, 32
        const float rs{lane_value(sums, 32)};
        if (lane == 0) {
            S.cost16[wu] = 256.0f * sums + 6.0e-4f * rs;
        }
    };
    const int e32{(qcol + t16) * 32 + qrow + 4 * grp};
    [[maybe_unused]] float own32[2]{0.0f, 0.0f};  // wave 0's terms, summed
    const auto ex_dct32_terms = [&](const f4v& c32) {
        float v[4], wq[4], wi[4], d[4], rt[4];
        bool llf[4];
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            v[u] = c32[u];
            llf[u] = wu == 0 && lane < 4;  // fx, fy < 4
        }
        selection_weights4(g_tables.wsel32, g_tables.wsel_inv32, e32, 0, wq, wi);
        selection_terms(v, llf, wq, wi, prm, d, rt);
        if (wu == 0) {
            own32[0] = ((d[0] + d[1]) + d[2]) + d[3];
            own32[1] = ((rt[0] + rt[1]) + rt[2]) + rt[3];
        } else {
            *reinterpret_cast<float4*>(S.a.after.y.t32[0][wu - 1][lane]) = float4{d[0], d[1], d[2], d[3]};
            *reinterpret_cast<float4*>(S.a.after.y.t32[1][wu - 1][lane]) = float4{rt[0], rt[1], rt[2], rt[3]};
        }
    };
    // Wave 0, after a barrier: the DCT32's cost from the four waves' terms.
    const auto ex_dct32_cost = [&]() {
        float s[2]{own32[0], own32[1]};
#pragma unroll
        for (int k{0}; k < 2; ++k) {
#pragma unroll
            for (int b{0}; b < 3; ++b) {
                const float4 x{*reinterpret_cast<const float4*>(S.a.after.y.t32[k][b][lane])};
                s[k] += x.x;
                s[k] += x.y;
                s[k] += x.z;
                s[k] += x.w;
            }
        }
        const float sums{wave_sum4(s[0], s[1], 0.0f, 0.0f)};  // lanes 0, 32
        const float rs{lane_value(sums, 32)};
        if (lane == 0) {
            S.cost32 = 1024.0f * sums + 6.0e-4f * rs;
        }
        wave_sync();
    };
    // The larger candidates' coefficients and costs, after every wave has
    // transformed Y (whose space takes the DCT32's terms).
    const auto ex_big = [&](const f4v& c16, const f4v& c32) {
        store4(coefy_of(S, 1), 256 * wu + t16 * 16 + 4 * grp, c16);
        store4(coefy_of(S, 2), e32, c32);
        ex_dct16_costs(c16);
        ex_dct32_terms(c32);
        __syncthreads();
        if (wu == 0) {
            ex_dct32_cost();
        }
    };
    // Matrix-core FP16 pieces: wave w transforms quad w as four DCT8s (with
    // their costs, from registers) and as one DCT16, and output tile w of the
    // DCT32 (vertical origin 16 (w / 2), horizontal 16 (w % 2)).
    const auto mf_dct8_costs = [&]() {
        const int q{wu};
        const f4v c8{mf_quad(yp, (q >> 1) * 16, (q & 1) * 16, g_tables.mf8[0], g_tables.mf8[1], lane)};
        float d8{0.0f}, r8{0.0f}, fv{0.0f}, fg{0.0f};
        float v[4], wq[4], wi[4], d[4], rt[4];
        int e[4], j[4];
        bool llf[4];
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            mf_quad_element(lane, u, 8, j[u], e[u]);
            v[u] = c8[u];
            llf[u] = u == 0 && (lane & 7) == 0 && (grp & 1) == 0;  // the DC
        }
        selection_weights4(g_tables.wsel8, g_tables.wsel_inv8, e[0], 0, wq, wi);
        selection_terms(v, llf, wq, wi, prm, d, rt);
        store4(coefy_of(S, 0), 256 * q + 64 * j[0] + e[0], c8);
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            d8 += d[u];
            r8 += rt[u];
            if (want_features) {
                const float c2{c8[u] * c8[u]};
                fv += e[u] != 0 ? c2 : 0.0f;
                fg = __builtin_fmaf(grad_weight(e[u] >> 3) + grad_weight(e[u] & 7), c2, fg);
            }
        }
        // The DC of block (grp / 2, column / 8) sits in lane 16 grp + 8 k,
        // element u = 0, for even grp.
        const float dc{c8[0]};
        // A DCT8 block's 64 terms sit in 16 lanes: bits 0-2 of the column and
        // bit 0 of the lane group vary within it.
        const auto sum16 = [](float x) { return add_down_16(add_down_row<4>(add_down_row<2>(add_down_row<1>(x)))); };
        d8 = sum16(d8);
        r8 = sum16(r8);
        if (want_features) {
            fv = sum16(fv);
            fg = sum16(fg);
        }
        if ((lane & 7) == 0 && (grp & 1) == 0) {
            const int j{2 * (grp >> 1) + ((lane & 15) >> 3)};
            S.cost8[q * 4 + j] = 64.0f * d8 + 6.0e-4f * r8;
            if (want_features) {
                const int b{(2 * (q >> 1) + (j >> 1)) * 4 + 2 * (q & 1) + (j & 1)};
                feature_store(S, b, fv, fg, d8, r8, dc);
            }
        }
    };
    const auto mf_big = [&]() {  // every wave; barriers inside
        const int q{wu};
        const f4v c16{mf_quad(yp, (q >> 1) * 16, (q & 1) * 16, g_tables.mf16[0], g_tables.mf16[1], lane)};
        f4v c32[2];
        mf_dct32(yp, 16 * (wu & 1), 16 * (wu >> 1), false, lane, c32);
        float d16{0.0f}, r16{0.0f}, d32{0.0f}, r32{0.0f};
        float v16[4], w16[4], wi16[4], v32[4], w32[4], wi32[4], d[2][4], rt[2][4];
        int e16[4];
        bool llf16[4], llf32[4];
        const int e32_0{(16 * (wu & 1) + t16) * 32 + 16 * (wu >> 1) + 4 * grp};
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            int j;
            mf_quad_element(lane, u, 16, j, e16[u]);
            v16[u] = c16[u];
            v32[u] = c32[0][u];
            llf16[u] = u < 2 && lane < 2;   // fx, fy < 2
            llf32[u] = wu == 0 && lane < 4;  // fx, fy < 4
        }
        selection_weights4(g_tables.wsel16, g_tables.wsel_inv16, e16[0], 0, w16, wi16);
        selection_weights4(g_tables.wsel32, g_tables.wsel_inv32, e32_0, 0, w32, wi32);
        selection_terms(v16, llf16, w16, wi16, prm, d[0], rt[0]);
        selection_terms(v32, llf32, w32, wi32, prm, d[1], rt[1]);
        store4(coefy_of(S, 1), 256 * q + e16[0], c16);
        store4(coefy_of(S, 2), e32_0, c32[0]);
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            d16 += d[0][u];
            r16 += rt[0][u];
            d32 += d[1][u];
            r32 += rt[1][u];
        }
        const float sums{wave_sum4(d16, r16, d32, r32)};  // lanes 0, 32, 16, 48
        const float ds16{sums}, rs16{lane_value(sums, 32)}, ds32{lane_value(sums, 16)}, rs32{lane_value(sums, 48)};
        if (lane == 0) {
            S.cost16[q] = 256.0f * ds16 + 6.0e-4f * rs16;
            S.cost32p[q] = 1024.0f * ds32 + 6.0e-4f * rs32;
        }
        __syncthreads();
        if (wu == 0) {
            if (lane == 0) {
                S.cost32 = (S.cost32p[0] + S.cost32p[1]) + (S.cost32p[2] + S.cost32p[3]);
            }
            wave_sync();
        }
    };
    // The heuristic's decision from the costs, by wave 0: lane b < 16 decides
    // the quad of block b (region raster).
    const auto decide = [&]() {
        constexpr float inf{1.0e30f}, eps{1.0e-6f};
        // A forced size (test modes): 1 DCT8, 2 DCT16, 3 DCT32 wherever it fits.
        const std::uint32_t force{(prm.mode & kModeForceMask) >> kModeForceShift};
        const bool fit32{bx0 + 4 <= bw && by0 + 4 <= bh};
        const float c32{fit32 ? S.cost32 : inf};
        const int qx{(lane >> 1) & 1}, qy{(lane >> 3) & 1}, q{2 * qy + qx};
        float sum8{0.0f};
        bool any8{false};
#pragma unroll
        for (int k{0}; k < 4; ++k) {
            if (bx0 + 2 * qx + (k & 1) < bw && by0 + 2 * qy + (k >> 1) < bh) {
                sum8 += S.cost8[q * 4 + k];
                any8 = true;
            }
        }
        const bool fit16{bx0 + 2 * qx + 2 <= bw && by0 + 2 * qy + 2 <= bh};
        const float c16{fit16 ? S.cost16[q] : inf};
        const bool use16{any8 && (force != 0 ? (force >= 2 && fit16) : (fit16 && c16 <= sum8 + eps))};
        const float cost{any8 ? (use16 ? c16 : sum8) : 0.0f};
        // The quads' costs in order (an absent quad adds 0).
        const float split{((lane_value(cost, 0) + lane_value(cost, 2)) + lane_value(cost, 8)) + lane_value(cost, 10)};
        const bool root32{force != 0 ? (force == 3 && fit32) : (fit32 && c32 <= split + eps)};
        if (lane < 16) {
            const bool first{(lane & 5) == 0};  // the quad's first block
            if (first) {
                S.choice[q] = any8 ? (use16 ? 16 : 8) : -1;
            }
            S.acs[lane] = root32 ? (lane == 0 ? 32 : 0) : (use16 ? (first ? 16 : 0) : 8);
        }
    };

    [[maybe_unused]] f4v c16{}, c32{};
    if constexpr (!kMf16) {
        const float4 b8{*reinterpret_cast<const float4*>(g_tables.ex8[lane])};
        float p[4];
        ex_pixels<4>(yp, qrow + t16, qcol, lane, p);
        if constexpr (kLearned) {
            ex_dct8_costs(ex_cols(b8, ex_rows(p, b8), f4v{0.0f, 0.0f, 0.0f, 0.0f}));
        } else {
            const float4 b16{*reinterpret_cast<const float4*>(g_tables.ex16[lane])};
            const Ex32 a32{ex_basis32(wu >> 1, lane)};
            f4v t32[2];
            ex_rows32(yp, ex_basis32(wu & 1, lane), lane, t32);
            const f4v t8{ex_rows(p, b8)}, r16{ex_rows(p, b16)};
            const f4v zero{0.0f, 0.0f, 0.0f, 0.0f};
            c32 = ex_cols32(a32, t32);
            const f4v c8{ex_cols(b8, t8, zero)};
            c16 = ex_cols(b16, r16, zero);
            __syncthreads();  // Y is dead from here on
            CJX_REGION_CUT_AT(7)
            ex_dct8_costs(c8);
            ex_big(c16, c32);
        }
    } else {
        mf_dct8_costs();
        if constexpr (!kLearned) {
            mf_big();
        }
    }
    CJX_REGION_CUT_AT(8)
    bool fallback{!kLearned};
    if (want_features) {
        __syncthreads();
        feature_finish(S, tid, bx0, by0, bw, bh);
    }
    if constexpr (kLearned) {
        fallback = !mlp_decide(S, prm, mlp_regs, S.b.s.hid, tid, bx0, by0, bw, bh);
        if (fallback) {
            // The heuristic for this region: the larger candidates and the
            // decision from the costs.
            if constexpr (!kMf16) {
                const float4 b16{*reinterpret_cast<const float4*>(g_tables.ex16[lane])};
                c16 = ex_quad(yp, qrow, qcol, b16, lane);
                f4v t32[2];
                ex_rows32(yp, ex_basis32(wu & 1, lane), lane, t32);
                c32 = ex_cols32(ex_basis32(wu >> 1, lane), t32);
                __syncthreads();  // Y is dead from here on
                ex_big(c16, c32);
            } else {
                mf_big();
            }
        }
    }
    if (fallback && wu == 0) {
        decide();
    }
    __syncthreads();
    if (feat_out != nullptr) {
        export_features(S, feat_out, region, tid, bx0, by0, bw, bh);
    }
    if (tid < 16) {
        const int bx{bx0 + (tid & 3)}, by{by0 + (tid >> 2)};
        if (bx < bw && by < bh) {
            acs_out[static_cast<std::size_t>(by) * bw + bx] = static_cast<std::int8_t>(S.acs[tid]);
        }
    }

    CJX_REGION_CUT_AT(4)
    // 5. Chosen DCTs of X and B (Y reuses the selection coefficients; a region
    //    the network decided transforms Y here too when it chose a DCT16 or
    //    DCT32) into the coefficient arrays in element order, then FP16 out
    //    and the CfL partials (frontend_quantize.cu:49-117 on this region).
    const bool need_y{kLearned && !fallback};
    // The coefficients of X and B go to Y's space (and past it): Y is dead
    // unless a region that the network decided transforms it here.
    const auto cxb = [&](int ch) { return S.a.after.y.xb[ch]; };
    const int acs0{__builtin_amdgcn_readfirstlane(S.acs[0])};
    const auto dct32 = [&](const float* plane, int fxb, f4v (&c)[2]) {
        if constexpr (kMf16) {
            mf_dct32(plane, 16 * fxb, 0, true, lane, c);
        } else {
            ex_dct32(plane, fxb, lane, c);
        }
    };
    if (acs0 == 32) {
        // Wave w: channel w % 2 (X, B), horizontal frequencies 16 (w / 2)..;
        // waves 0-1 also Y's half w when it has no coefficients yet.
        const int ch{wu & 1}, fxb{wu >> 1};
        f4v c[2], cy[2];
        dct32(plane_of(S, 2 * ch), fxb, c);
        if (need_y && wu < 2) {
            dct32(plane_of(S, 1), wu, cy);
        }
        if (need_y) {
            __syncthreads();
        }
#pragma unroll
        for (int o{0}; o < 2; ++o) {
            store4(cxb(ch), (16 * fxb + t16) * 32 + 16 * o + 4 * grp, c[o]);
            if (need_y && wu < 2) {
                store4(coefy_of(S, 2), (16 * wu + t16) * 32 + 16 * o + 4 * grp, cy[o]);
            }
        }
    } else {
        // Wave w transforms quad w of X and B (and of Y, when it has no
        // coefficients yet and takes a DCT16): one DCT16 or four DCT8s.
        const int q{wu};
        const int n{__builtin_amdgcn_readfirstlane(S.acs[(q >> 1) * 8 + (q & 1) * 2]) == 16 ? 16 : 8};
        const bool y16{need_y && n == 16};
        f4v cx, cb, cy{};
        if constexpr (kMf16) {
            const std::uint16_t* hi{n == 16 ? g_tables.mf16[0] : g_tables.mf8[0]};
            const std::uint16_t* lo{n == 16 ? g_tables.mf16[1] : g_tables.mf8[1]};
            cx = mf_quad(plane_of(S, 0), qrow, qcol, hi, lo, lane);
            cb = mf_quad(plane_of(S, 2), qrow, qcol, hi, lo, lane);
            if (y16) {
                cy = mf_quad(plane_of(S, 1), qrow, qcol, hi, lo, lane);
            }
        } else {
            const float4 b{*reinterpret_cast<const float4*>(n == 16 ? g_tables.ex16[lane] : g_tables.ex8[lane])};
            cx = ex_quad(plane_of(S, 0), qrow, qcol, b, lane);
            cb = ex_quad(plane_of(S, 2), qrow, qcol, b, lane);
            if (y16) {
                cy = ex_quad(plane_of(S, 1), qrow, qcol, b, lane);
            }
        }
        if (need_y) {
            __syncthreads();
        }
        int j, e;
        mf_quad_element(lane, 0, n, j, e);
        store4(cxb(0), 256 * q + 64 * j + e, cx);
        store4(cxb(1), 256 * q + 64 * j + e, cb);
        if (y16) {
            store4(coefy_of(S, 1), 256 * q + e, cy);
        }
    }
    __syncthreads();

    CJX_REGION_CUT_AT(5)
    // Lane l takes coefficients 4 (l % 16) .. + 3 of block k = l / 16 of the
    // wave's four blocks, (2 (k % 2) + w % 2, 2 (k / 2) + w / 2): one 8-byte
    // LDS read and one 8-byte store per plane.
    const std::size_t cplane{static_cast<std::size_t>(geo.nblocks) * 64};
    float v[3][4];
    {
        const int k{grp}, s4{4 * t16};
        const int bxl{2 * (k & 1) + (wu & 1)}, byl{2 * (k >> 1) + (wu >> 1)};
        const bool is32{acs0 == 32};
        const int n{is32 ? 32 : (S.acs[(byl & ~1) * 4 + (bxl & ~1)] == 16 ? 16 : 8)};
        const int qc{is32 ? byl * 4 + bxl : (n == 16 ? wu : 0)};
        const int e{qc * 64 + s4};
        const int idx{cpad(is32 ? e : 256 * k + 64 * wu + s4)};
        const h4v hx{*reinterpret_cast<const h4v*>(cxb(0) + idx)};
        const h4v hy{*reinterpret_cast<const h4v*>(coefy_of(S, n >> 4) + idx)};
        const h4v hb{*reinterpret_cast<const h4v*>(cxb(1) + idx)};
        const bool in{bx0 + bxl < bw && by0 + byl < bh};
        if (in) {
            std::uint16_t* const out{coeffs + (static_cast<std::size_t>(by0 + byl) * bw + bx0 + bxl) * 64 + s4};
            *reinterpret_cast<h4v*>(out) = hx;
            *reinterpret_cast<h4v*>(out + cplane) = hy;
            *reinterpret_cast<h4v*>(out + 2 * cplane) = hb;
        }
        // CfL terms; 0 for the LLF coefficients (the first m of the four
        // where a row fx < m of the transform starts) and outside the frame.
        const int m{n >> 3};
        const int nllf{in ? ((e & (n - 1)) == 0 && e < m * n ? m : 0) : 4};
#pragma unroll
        for (int i{0}; i < 4; ++i) {
            const float xr{static_cast<float>(hx[i])}, yr{static_cast<float>(hy[i])}, br{static_cast<float>(hb[i])};
            const bool use{i >= nllf};
            v[0][i] = use ? xr * yr : 0.0f;
            v[1][i] = use ? yr * yr : 0.0f;
            v[2][i] = use ? (br - yr) * yr : 0.0f;
        }
    }
    // Slot by slot the four blocks in order, then the tree over the 64 slots
    // (offsets 32 .. 1): after the turn, register k of lane group g holds
    // slot 4 (l % 16) + g of block k.
    {
        float sum[3];
#pragma unroll
        for (int c{0}; c < 3; ++c) {
            ex_turn(v[c]);
            float x{((v[c][0] + v[c][1]) + v[c][2]) + v[c][3]};
            x = add_down_row<8>(x);
            x = add_down_row<4>(x);
            x = add_down_row<2>(x);
            x = add_down_row<1>(x);
            sum[c] = add_down_16(add_down_32(x));
        }
        if (lane == 0) {
            S.cfl[wu][0] = sum[0];
            S.cfl[wu][1] = sum[1];
            S.cfl[wu][2] = sum[2];
        }
    }
    __syncthreads();
    if (tid < 3) {
        cfl_part[static_cast<std::size_t>(region) * 3 + tid] =
            (S.cfl[0][tid] + S.cfl[1][tid]) + (S.cfl[2][tid] + S.cfl[3][tid]);
    }
}

template <bool kMf16, bool kLearned>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void region_kernel(
    Geometry geo, FrameParams prm, const std::uint8_t* __restrict__ luma, std::size_t luma_pitch,
    const std::uint8_t* __restrict__ chroma, std::size_t chroma_pitch,
    std::uint16_t* __restrict__ coeffs, std::int8_t* __restrict__ acs_out,
    std::int32_t* __restrict__ qf_out, float* __restrict__ cfl_part, std::uint32_t* __restrict__ list_count,
    Clears clr, float* __restrict__ feat_out) {
    region_kernel_body<kMf16, kLearned>(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, prm, luma, luma_pitch, chroma, chroma_pitch, coeffs, acs_out, qf_out, cfl_part, list_count, clr, feat_out);
}

// ---------------------------------------------------------------------------

struct TileShared {
    unsigned int nz[64][3];
    int own[64];              // packed owner: local position | (n << 8)
    float2 scale[64];         // the block's quantizer q and RN(1 / q)
    float maps[2];
    // LLF coefficients: (fx, fy) of the transform at local position op in
    // slot op + 8 fx + fy (the blocks it covers, so no two transforms meet).
    float llf[3][64];
    double resample[4 + 16];  // g_tables.llf2, llf4
};

// DC coefficient of channel c of the block at local position p of a tile
// (frontend_quantize.cu:181-199, dc_from_llf_strided): the owner transform's
// (n/8)^2 lowest frequencies, resampled to the block, from the FP16
// coefficients.
__device__ __forceinline__ float block_dc(const TileShared& S, int p, int c) {
    const int own{S.own[p]};
    const int n{own >> 8}, op{own & 255};
    const int m{n >> 3}, dx{(p & 7) - (op & 7)}, dy{(p >> 3) - (op >> 3)};
    if (m == 1) {
        return S.llf[c][op];
    }
    const double* const t{S.resample + (m == 2 ? 0 : 4)};
    double sum{0.0};
#pragma unroll 1
    for (int fx{0}; fx < m; ++fx) {
#pragma unroll 2
        for (int fy{0}; fy < m; ++fy) {
            sum += t[fx * m + dx] * t[fy * m + dy] * static_cast<double>(S.llf[c][op + 8 * fx + fy]);
        }
    }
    return static_cast<float>(static_cast<double>(m) * sum);
}

// What bounds it: at 3840x2160 vector instructions (10.3 M, 21 us of issue) and
// 100 MB in and out (19 us at a copy's rate), in one resident round of eight
// waves per SIMD, 36.4 us.  Owners, quantizers and reciprocals are set up once
// per block, one 32-bit offset serves a step's reads and writes, the LLF
// coefficients are masked after packing and non-zeros are counted in packed
// halves (12.4 M instructions, 40.4 us with a quotient, a test and a 64-bit
// address for each of those; 320x240 10.1 -> 8.7 us, 7680x4320 150 -> 113).
// The next step's coefficients read ahead gain nothing (36.8).
__device__ __attribute__((always_inline)) inline void tile_quantize_kernel_body(const Wg& wg, 
    Geometry geo, FrameParams prm, const std::uint16_t* __restrict__ coeffs,
    const std::int8_t* __restrict__ acs, const std::int32_t* __restrict__ qf,
    const float* __restrict__ cfl_part, std::int16_t* __restrict__ ac,
    std::uint8_t* __restrict__ nz_grid, std::uint16_t* __restrict__ nz_count, ItemList list,
    std::int32_t* __restrict__ dc, std::int8_t* __restrict__ ytox, std::int8_t* __restrict__ ytob) {
    __shared__ TileShared S;
    const int tid{static_cast<int>(threadIdx.x)};
    const int w{tid >> 6};
    const int lane{tid & 63};
    const int tile{static_cast<int>(wg.x)};
    const int tx{tile % static_cast<int>(geo.cmw)}, ty{tile / static_cast<int>(geo.cmw)};
    const int bw{static_cast<int>(geo.bw)}, bh{static_cast<int>(geo.bh)};
    const std::size_t nblk{geo.nblocks};
    const std::size_t cplane{nblk * 64};

    if (tid < 64) {
        S.nz[tid][0] = S.nz[tid][1] = S.nz[tid][2] = 0u;
        const int bx{tx * 8 + (tid & 7)}, by{ty * 8 + (tid >> 3)};
        // The transform that covers the block: the 32x32 or 16x16 one whose
        // first block its aligned square starts with, else its own.  Every
        // candidate is read before any is looked at.
        int op{tid}, n{8};
        float quant{1.0f};  // of blocks past the frame, which no lane uses
        if (bx < bw && by < bh) {
            const std::uint32_t row{static_cast<std::uint32_t>(bw)};
            const std::uint32_t at8{static_cast<std::uint32_t>(by) * row + static_cast<std::uint32_t>(bx)};
            const std::uint32_t at16{static_cast<std::uint32_t>(by & ~1) * row + static_cast<std::uint32_t>(bx & ~1)};
            const std::uint32_t at32{static_cast<std::uint32_t>(by & ~3) * row + static_cast<std::uint32_t>(bx & ~3)};
            const int n32{acs[at32]}, n16{acs[at16]};
            const std::int32_t f8{qf[at8]}, f16{qf[at16]}, f32{qf[at32]};
            n = n32 == 32 ? 32 : (n16 == 16 ? 16 : 8);
            op = n == 32 ? tid & 0x24 : (n == 16 ? tid & 0x36 : tid);
            quant = static_cast<float>(n == 32 ? f32 : (n == 16 ? f16 : f8));
        }
        S.own[tid] = op | (n << 8);
        const float qgsf{quant * prm.global_scale_float};
        S.scale[tid] = float2{qgsf, 1.0f / qgsf};
    }
    if (tid >= 128 && tid < 148) {
        const int i{tid - 128};
        S.resample[i] = i < 4 ? g_tables.llf2[i] : g_tables.llf4[i - 4];
    }
    if (tid == 64) {  // wave 1, beside wave 0's owners
        float r[4][3];
        tile_partials(geo, cfl_part, tx, ty, r);
        int mx, mb;
        cfl_tile_maps(r, mx, mb);
        S.maps[0] = 0.0f + static_cast<float>(mx) * (1.0f / 84);
        S.maps[1] = 1.0f + static_cast<float>(mb) * (1.0f / 84);
        ytox[tile] = static_cast<std::int8_t>(mx);
        ytob[tile] = static_cast<std::int8_t>(mb);
    }
    __syncthreads();

    const float yx{S.maps[0]}, yb{S.maps[1]};
    // Lane l quantizes coefficients 4 (l % 16) .. 4 (l % 16) + 3 of block
    // p = 16 j + 4 (l / 16) + w: a wave takes four blocks per step, one
    // 8-byte read per plane and lane, the weights and their reciprocals as
    // 16-byte reads.  y_round = qy wy / qgsf is the correctly rounded
    // quotient, by the block's RN(1 / qgsf).
    const int grp{lane >> 4}, e4{4 * (lane & 15)};
    // Weights and reciprocals of a transform size at one distance, so that
    // one offset serves both; 32-bit offsets (an accepted frame's plane has
    // at most 2^28 bytes).
    constexpr std::uint32_t kInverse{offsetof(DeviceTables, dequant_inv8) - offsetof(DeviceTables, dequant8)};
    static_assert(offsetof(DeviceTables, dequant8) % 16 == 0 && offsetof(DeviceTables, dequant16) % 16 == 0 &&
                      offsetof(DeviceTables, dequant32) % 16 == 0 && kInverse % 16 == 0 &&
                      offsetof(DeviceTables, dequant_inv16) == offsetof(DeviceTables, dequant16) + kInverse &&
                      offsetof(DeviceTables, dequant_inv32) == offsetof(DeviceTables, dequant32) + kInverse,
                  "16-byte weight reads");
    const auto* const weights{reinterpret_cast<const std::uint8_t*>(&g_tables.dequant8[0][0])};
    const auto* const inverses{reinterpret_cast<const std::uint8_t*>(&g_tables.dequant_inv8[0][0])};
    const auto* const in0{reinterpret_cast<const std::uint8_t*>(coeffs)};
    const auto* const in1{reinterpret_cast<const std::uint8_t*>(coeffs + cplane)};
    const auto* const in2{reinterpret_cast<const std::uint8_t*>(coeffs + 2 * cplane)};
    auto* const out0{reinterpret_cast<std::uint8_t*>(ac)};
    auto* const out1{reinterpret_cast<std::uint8_t*>(ac + cplane)};
    auto* const out2{reinterpret_cast<std::uint8_t*>(ac + 2 * cplane)};
    const auto f16_at = [](uint2 h, int i) {
        const std::uint32_t wd{i < 2 ? h.x : h.y};
        return static_cast<float>(
            __builtin_bit_cast(_Float16, static_cast<std::uint16_t>((i & 1) != 0 ? wd >> 16 : wd & 0xffffu)));
    };
    const auto f4_at = [](const float4& v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w)); };
    // The low halves of two integers in one word.
    const auto pair = [](int lo, int hi) {
        return __builtin_amdgcn_perm(static_cast<std::uint32_t>(hi), static_cast<std::uint32_t>(lo), 0x05040100u);
    };
    // Non-zeros among four 16-bit values.
    const auto nonzeros = [](std::uint32_t a, std::uint32_t b) {
        using u16x2 = std::uint16_t __attribute__((ext_vector_type(2)));
        const u16x2 one{1, 1};
        const u16x2 n{__builtin_elementwise_min(__builtin_bit_cast(u16x2, a), one) +
                      __builtin_elementwise_min(__builtin_bit_cast(u16x2, b), one)};
        const std::uint32_t both{__builtin_bit_cast(std::uint32_t, n)};
        return (both & 0xffffu) + (both >> 16);
    };
#pragma unroll 1
    for (int j{0}; j < 4; ++j) {
        const int p{16 * j + 4 * grp + w};
        const int bx{tx * 8 + (p & 7)}, by{ty * 8 + (p >> 3)};
        const bool in{bx < bw && by < bh};
        const int own{S.own[p]};
        const int n{own >> 8}, op{own & 255};
        // Non-zeros among the lane's four: X | Y << 8 | B << 16.
        std::uint32_t cnt{0};
        if (in) {
            const int m{n >> 3};
            const int e0{(((p >> 3) - (op >> 3)) * m + ((p & 7) - (op & 7))) * 64 + e4};
            const std::uint32_t at{2u * ((static_cast<std::uint32_t>(by) * static_cast<std::uint32_t>(bw) +
                                          static_cast<std::uint32_t>(bx)) * 64u + static_cast<std::uint32_t>(e4))};
            const uint2 hx{*reinterpret_cast<const uint2*>(in0 + at)};
            const uint2 hy{*reinterpret_cast<const uint2*>(in1 + at)};
            const uint2 hb{*reinterpret_cast<const uint2*>(in2 + at)};
            const std::uint32_t next{4u * static_cast<std::uint32_t>(n * n)};
            const std::uint32_t wx_at{
                (n == 32 ? static_cast<std::uint32_t>(offsetof(DeviceTables, dequant32) - offsetof(DeviceTables, dequant8))
                         : (n == 16 ? static_cast<std::uint32_t>(offsetof(DeviceTables, dequant16) -
                                                                 offsetof(DeviceTables, dequant8))
                                    : 0u)) +
                4u * static_cast<std::uint32_t>(e0)};
            const std::uint32_t wy_at{wx_at + next}, wb_at{wy_at + next};
            const float4 wx4{*reinterpret_cast<const float4*>(weights + wx_at)};
            const float4 wy4{*reinterpret_cast<const float4*>(weights + wy_at)};
            const float4 wb4{*reinterpret_cast<const float4*>(weights + wb_at)};
            const float4 ix4{*reinterpret_cast<const float4*>(inverses + wx_at)};
            const float4 iy4{*reinterpret_cast<const float4*>(inverses + wy_at)};
            const float4 ib4{*reinterpret_cast<const float4*>(inverses + wb_at)};
            const float qgsf{S.scale[p].x}, rq{S.scale[p].y};
            // The lane's LLF coefficients (the first m of its four, in the
            // rows fx < m) to where block_dc reads them; they are no items'.
            const int fx{e0 >> (n == 32 ? 5 : (n == 16 ? 4 : 3))};
            std::uint32_t keep0{~0u}, keep1{~0u};
            if ((e0 & (n - 1)) == 0 && fx < m) {
#pragma unroll
                for (int i{0}; i < 4; ++i) {
                    if (i < m) {
                        S.llf[0][op + 8 * fx + i] = f16_at(hx, i);
                        S.llf[1][op + 8 * fx + i] = f16_at(hy, i);
                        S.llf[2][op + 8 * fx + i] = f16_at(hb, i);
                    }
                }
                keep0 = m == 1 ? 0xffff0000u : 0u;
                keep1 = m == 4 ? 0u : ~0u;
            }
            int a0[4], a1[4], a2[4];
#pragma unroll
            for (int i{0}; i < 4; ++i) {
                const float wy{f4_at(wy4, i)};
                const float qy{__builtin_rintf(div_by_recip(f16_at(hy, i) * qgsf, wy, f4_at(iy4, i)))};
                const float y_round{div_by_recip(qy * wy, qgsf, rq)};
                a0[i] = static_cast<int>(__builtin_rintf(
                    div_by_recip((f16_at(hx, i) - yx * y_round) * qgsf, f4_at(wx4, i), f4_at(ix4, i))));
                a1[i] = static_cast<int>(qy);
                a2[i] = static_cast<int>(__builtin_rintf(
                    div_by_recip((f16_at(hb, i) - yb * y_round) * qgsf, f4_at(wb4, i), f4_at(ib4, i))));
            }
            const uint2 q0{pair(a0[0], a0[1]) & keep0, pair(a0[2], a0[3]) & keep1};
            const uint2 q1{pair(a1[0], a1[1]) & keep0, pair(a1[2], a1[3]) & keep1};
            const uint2 q2{pair(a2[0], a2[1]) & keep0, pair(a2[2], a2[3]) & keep1};
            cnt = nonzeros(q0.x, q0.y) | (nonzeros(q1.x, q1.y) << 8) | (nonzeros(q2.x, q2.y) << 16);
            *reinterpret_cast<uint2*>(out0 + at) = q0;
            *reinterpret_cast<uint2*>(out1 + at) = q1;
            *reinterpret_cast<uint2*>(out2 + at) = q2;
        }
        // The block's counts into lane 0 of its row of 16 lanes (row
        // shifts; lanes shifted in from outside the row read 0).
        cnt += static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(cnt), 0x101, 0xf, 0xf, true));
        cnt += static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(cnt), 0x102, 0xf, 0xf, true));
        cnt += static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(cnt), 0x104, 0xf, 0xf, true));
        cnt += static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(cnt), 0x108, 0xf, 0xf, true));
        if (in && (lane & 15) == 0) {
            atomicAdd(&S.nz[op][0], cnt & 0xffu);
            atomicAdd(&S.nz[op][1], (cnt >> 8) & 0xffu);
            atomicAdd(&S.nz[op][2], cnt >> 16);
        }
    }
    __syncthreads();

    if (w > 0) {
        // The DC values, beside wave 0's lists: waves 1, 2 and 3 take X, Y
        // and B (against Y's round trip).
        const int bx{tx * 8 + (lane & 7)}, by{ty * 8 + (lane >> 3)};
        if (bx < bw && by < bh) {
            const float scale_y{512.0f * prm.dc_scale};
            float v{block_dc(S, lane, w - 1)};
            float scale{w == 1 ? 4096.0f * prm.dc_scale : scale_y};
            if (w == 3) {
                const float qy{__builtin_rintf(block_dc(S, lane, 1) * scale_y)};
                const float y_dc_round{static_cast<float>(static_cast<int>(qy)) / scale_y};
                v = v - 1.0f * y_dc_round;
                scale = 256.0f * prm.dc_scale;
            }
            dc[static_cast<std::size_t>(w - 1) * nblk + static_cast<std::size_t>(by) * bw + bx] =
                static_cast<int>(__builtin_rintf(v * scale));
        }
    }
    if (tid < 64) {
        const int p{tid};
        const int bx{tx * 8 + (p & 7)}, by{ty * 8 + (p >> 3)};
        // This block's items for the tokenizer's lists, in item order Y, X,
        // B: with non-zeros (dense) or without (zero count).
        bool dense[3]{false, false, false}, zero[3]{false, false, false};
        if (bx < bw && by < bh) {
            const int own{S.own[p]};
            const int n{own >> 8}, op{own & 255};
            const int m{n / 8};
            const std::size_t b{static_cast<std::size_t>(by) * bw + bx};
            const unsigned int l2{n == 16 ? 2u : (n == 32 ? 4u : 0u)};
            for (int c{0}; c < 3; ++c) {
                const unsigned int cnt{S.nz[op][c]};
                nz_grid[c * nblk + b] = static_cast<std::uint8_t>((cnt + m * m - 1) >> l2);
                nz_count[c * nblk + b] = op == p ? static_cast<std::uint16_t>(cnt) : 0;
            }
            // Covered blocks' items have no tokens (emission reads no count
            // for them).
            if (op == p) {
#pragma unroll
                for (int j{0}; j < 3; ++j) {
                    const bool any{S.nz[op][j == 0 ? 1 : (j == 1 ? 0 : 2)] != 0};
                    dense[j] = any;
                    zero[j] = !any;
                }
            }
        }
        // Wave 0 appends the tile's items: prefix sums of the per-lane counts
        // (0..3, two ballots each), one reservation per list.
        if (list.items != nullptr) {
            const int nd{(dense[0] ? 1 : 0) + (dense[1] ? 1 : 0) + (dense[2] ? 1 : 0)};
            const int nzc{(zero[0] ? 1 : 0) + (zero[1] ? 1 : 0) + (zero[2] ? 1 : 0)};
            const std::uint64_t below{(1ull << p) - 1ull};
            const std::uint64_t d0{__ballot(nd & 1)}, d1{__ballot(nd & 2)};
            const std::uint64_t z0{__ballot(nzc & 1)}, z1{__ballot(nzc & 2)};
            const std::uint32_t dpre{static_cast<std::uint32_t>(__popcll(d0 & below) + 2 * __popcll(d1 & below))};
            const std::uint32_t zpre{static_cast<std::uint32_t>(__popcll(z0 & below) + 2 * __popcll(z1 & below))};
            const std::uint32_t dtot{static_cast<std::uint32_t>(__popcll(d0) + 2 * __popcll(d1))};
            const std::uint32_t ztot{static_cast<std::uint32_t>(__popcll(z0) + 2 * __popcll(z1))};
            std::uint32_t base{0};
            if (p < 2) {
                base = atomicAdd(&list.count[p], p == 0 ? dtot : ztot);
            }
            const std::uint32_t dbase{static_cast<std::uint32_t>(__shfl(static_cast<int>(base), 0, 64))};
            const std::uint32_t zbase{static_cast<std::uint32_t>(__shfl(static_cast<int>(base), 1, 64))};
            const std::uint32_t last{3u * geo.nblocks - 1u};
            const std::uint32_t b3{(static_cast<std::uint32_t>(by) * static_cast<std::uint32_t>(bw) +
                                    static_cast<std::uint32_t>(bx)) * 3u};
            std::uint32_t kd{dbase + dpre}, kz{zbase + zpre};
#pragma unroll
            for (int j{0}; j < 3; ++j) {
                if (dense[j]) {
                    list.items[kd++] = b3 + static_cast<std::uint32_t>(j);
                }
                if (zero[j]) {
                    list.items[last - kz++] = b3 + static_cast<std::uint32_t>(j);
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void tile_quantize_kernel(
    Geometry geo, FrameParams prm, const std::uint16_t* __restrict__ coeffs,
    const std::int8_t* __restrict__ acs, const std::int32_t* __restrict__ qf,
    const float* __restrict__ cfl_part, std::int16_t* __restrict__ ac,
    std::uint8_t* __restrict__ nz_grid, std::uint16_t* __restrict__ nz_count, ItemList list,
    std::int32_t* __restrict__ dc, std::int8_t* __restrict__ ytox, std::int8_t* __restrict__ ytob) {
    tile_quantize_kernel_body(Wg{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}, geo, prm, coeffs, acs, qf, cfl_part, ac,
                              nz_grid, nz_count, list, dc, ytox, ytob);
}

// ---------------------------------------------------------------------------
// Config-1 semantics (the reference's test path: dct.cu:43-101 forward DCT8
// over the whole frame, quant.cu:30-97 quantize_dct8): DCT8 everywhere, the
// uniform quant field, no colour-correlation maps; coefficient k of channel c
// is rintf(v * f) with f = ac_scale / w8[c][k] (ac_scale = raw quant field x
// global scale) or DC_INV_QUANT[c] x dc_scale at k = 0, and B is taken
// against Y's round trip qy / f_y.  Note the operation order: a product by a
// rounded quotient, unlike the VarDCT quantizer's quotient of a product.
// One workgroup per 32x32 region: XYB, gaborish, then per channel (Y first,
// whose quantized values B needs) a DCT8 row pass into LDS lines and a column
// pass that quantizes and stores.
__global__ __launch_bounds__(256) void dct8_uniform_kernel(
    Geometry geo, FrameParams prm, const std::uint8_t* __restrict__ luma, std::size_t luma_pitch,
    const std::uint8_t* __restrict__ chroma, std::size_t chroma_pitch, std::int16_t* __restrict__ ac,
    std::int32_t* __restrict__ dc, std::int8_t* __restrict__ acs_out, std::int32_t* __restrict__ qf_out,
    std::int8_t* __restrict__ ytox, std::int8_t* __restrict__ ytob) {
    __shared__ RegionShared S;
    const int tid{static_cast<int>(threadIdx.x)};
    const int nreg{static_cast<int>(geo.rw * geo.rh)};
    const int per_xcd{(nreg + 7) / 8};
    const int region{static_cast<int>(blockIdx.x & 7u) * per_xcd + static_cast<int>(blockIdx.x >> 3)};
    if (region >= nreg) {
        return;
    }
    const int rx{region % static_cast<int>(geo.rw)};
    const int ry{region / static_cast<int>(geo.rw)};
    const int W{static_cast<int>(geo.width)}, H{static_cast<int>(geo.height)};
    const int bw{static_cast<int>(geo.bw)}, bh{static_cast<int>(geo.bh)};
    const int bx0{rx * 4}, by0{ry * 4};
    const std::size_t nblk{geo.nblocks};
    const std::size_t cplane{nblk * 64};

    __shared__ alignas(16) float lines[16 * RowBuf8::BS];
    __shared__ std::int32_t qy[1024];  // Y's quantized values
    xyb_tile(S, luma, luma_pitch, chroma, chroma_pitch, rx * 32, ry * 32, W, H, tid);
    __syncthreads();
    float4 sharp[3];
    gaborish_tile(S, tid, sharp);
    __syncthreads();
    store_sharp(S, tid, sharp);
    __syncthreads();

    const float ac_scale{prm.qgsf_select};
    const float dcq[3]{4096.0f * prm.dc_scale, 512.0f * prm.dc_scale, 256.0f * prm.dc_scale};
    const int b{tid >> 3}, sub{tid & 7};
    const int bx{bx0 + (b & 3)}, by{by0 + (b >> 2)};
    const bool inside{tid < 128 && bx < bw && by < bh};
    const std::size_t blk{inside ? static_cast<std::size_t>(by) * bw + bx : 0};
    for (int ci{0}; ci < 3; ++ci) {
        const int c{ci == 0 ? 1 : (ci == 1 ? 0 : 2)};
        if (tid < 128) {
            float o[8];
            const int row{(b >> 2) * 8 + sub};
            dct_line<8, 8>(plane_of(S, c) + row * kSP, 0, o, (b & 3) * 8, sp_swz(row));
#pragma unroll
            for (int f{0}; f < 8; ++f) {
                lines[b * RowBuf8::BS + f * RowBuf8::RS + sub] = o[f];
            }
        }
        __syncthreads();
        if (tid < 128) {
            float o[8];
            dct_line<8, 8>(&lines[b * RowBuf8::BS + sub * RowBuf8::RS], 0, o);
#pragma unroll
            for (int f{0}; f < 8; ++f) {
                const int e{sub * 8 + f};
                const float fc{e == 0 ? dcq[c] : ac_scale / g_tables.dequant8[c][e]};
                float v{o[f]};
                if (c == 2) {
                    const float fy{e == 0 ? dcq[1] : ac_scale / g_tables.dequant8[1][e]};
                    v = v - 1.0f * (static_cast<float>(qy[b * 64 + e]) / fy);
                }
                const int q{static_cast<int>(__builtin_rintf(v * fc))};
                if (c == 1) {
                    qy[b * 64 + e] = q;
                }
                if (inside) {
                    if (e == 0) {
                        dc[c * nblk + blk] = q;
                        ac[c * cplane + blk * 64] = 0;
                    } else {
                        ac[c * cplane + blk * 64 + e] = static_cast<std::int16_t>(q);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (tid < 16) {
        const int x{bx0 + (tid & 3)}, y{by0 + (tid >> 2)};
        if (x < bw && y < bh) {
            acs_out[static_cast<std::size_t>(y) * bw + x] = 8;
            qf_out[static_cast<std::size_t>(y) * bw + x] = static_cast<std::int32_t>(prm.raw_quant_field);
        }
    }
    if (tid == 0 && (rx & 1) == 0 && (ry & 1) == 0) {
        const std::size_t t{static_cast<std::size_t>(ry / 2) * geo.cmw + rx / 2};
        ytox[t] = 0;
        ytob[t] = 0;
    }
}

}  // namespace cjx
