// The learned transform-selection / adaptive-quantization network: its
// training kernels (included into device.hip).
//
// Network (one row of 96 features per 32x32 region):
//   h = ReLU(W1 x + b1)  (64),  z = W2 h + b2  (7)
//   z[0], z[1]  root logits (split, DCT32) under a softmax
//   z[2..5]     quad q: DCT16 (> 0) or four DCT8s (< 0), sigmoid
//   z[6]        the region's mean log2 quant field
// Parameters (FP32 masters, laid out W1[64][96], b1[64], W2[7][64], b2[7]);
// the encoder runs FP16 copies of W1 and W2 (region kernel, FP32
// accumulation).  Labels per region (12 floats): root, quad[4], quant-field
// target, root mask, quad mask[4], unused; a mask of 0 drops the term.
// Loss: mean over regions of m_r CE(root) + sum_q m_q BCE(quad q) +
// lambda (z6 - target)^2.
//
// mlp_grad_kernel: a workgroup takes tiles of 32 regions: forward, loss
// gradient of the outputs, backward, and the gradient sums of its tiles into
// its row of a partial-gradient buffer.  mlp_reduce_kernel sums the rows
// (fixed order) into the batch's mean gradient and, with a learning rate,
// takes one Adam step.  The two large products (X W1^T and dH^T X) run on the
// matrix cores in FP32 (v_mfma_f32_16x16x4_f32 rounds as an fmaf chain), the
// rest in lanes; at batches of a few thousand regions the kernels are bound by
// one workgroup's chain of latencies (two reads of memory, 24 + 8 matrix steps,
// four barriers), so a tile is spread over eight waves and a wave reads four
// floats at a time, everything before the first use.  Gradient of 4,096
// regions 10 us, of 60,000 36 us (one thread per region or entry: 41, 145);
// evaluation of 1,000 and 100,000 rows 4.9 and 20.5 us (one thread per row:
// 168, 366).

namespace cjx {

constexpr int kMlpIn = 96;
constexpr int kMlpHid = 64;
constexpr int kMlpOut = 7;
constexpr int kMlpLabels = 12;
constexpr int kMlpParams = kMlpHid * kMlpIn + kMlpHid + kMlpOut * kMlpHid + kMlpOut;
constexpr int kMlpB1 = kMlpHid * kMlpIn;
constexpr int kMlpW2 = kMlpB1 + kMlpHid;
constexpr int kMlpB2 = kMlpW2 + kMlpOut * kMlpHid;
constexpr int kMlpTiles = 32;       // regions per tile
constexpr int kMlpThreads = 512;    // eight waves: (16 rows, 16 hidden units) each
constexpr int kMlpMaxWgs = 512;     // two resident workgroups per CU; more regions, more tiles each
// LDS pitches: the matrix cores' operands (16 rows at four consecutive
// columns, or four rows at 16 consecutive columns) fall into different banks.
constexpr int kMlpXPitch = 100;
constexpr int kMlpHPitch = 80;
constexpr int kMlpW2Pitch = 68;

struct MlpShared {
    alignas(16) float x[kMlpTiles][kMlpXPitch];
    alignas(16) float h[kMlpTiles][kMlpHPitch];   // activations
    alignas(16) float w2[kMlpOut + 1][kMlpW2Pitch];  // row 7: zeros
    float b2[kMlpOut + 1];
};

struct MlpGradShared {
    MlpShared f;
    float dh[kMlpTiles][kMlpHPitch];  // gradients at the hidden units
    float dz[kMlpTiles][8];
    float loss[kMlpThreads / 64];
};

__device__ __forceinline__ f4v mlp_step_mfma(float a, float b, f4v acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}

// Four floats from any float's address.
using f4u = float __attribute__((ext_vector_type(4), aligned(4)));

// The lane's share of the first layer (hidden unit j = 16 (w % 4) + l % 16,
// inputs 16 s + 4 (l / 16) + u: any order of the sum serves, this one reads
// four inputs at a time) and of the second's.
struct MlpParamsLane {
    f4u w[kMlpIn / 16];
    float b, w2, b2;
};

__device__ __forceinline__ MlpParamsLane mlp_read_params(const float* __restrict__ params) {
    const int t{static_cast<int>(threadIdx.x)}, lane{t & 63};
    const int j{16 * ((t >> 6) & 3) + (lane & 15)};
    MlpParamsLane p;
#pragma unroll
    for (int s{0}; s < kMlpIn / 16; ++s) {
        p.w[s] = *reinterpret_cast<const f4u*>(&params[j * kMlpIn + 16 * s + 4 * (lane >> 4)]);
    }
    p.b = params[kMlpB1 + j];
    p.w2 = t < kMlpOut * kMlpHid ? params[kMlpW2 + t] : 0.0f;
    p.b2 = t < kMlpOut ? params[kMlpB2 + t] : 0.0f;
    return p;
}

__device__ __forceinline__ void mlp_store_params(MlpShared& S, const MlpParamsLane& p) {
    const int t{static_cast<int>(threadIdx.x)};
    S.w2[t >> 6][t & 63] = p.w2;
    if (t < kMlpOut + 1) {
        S.b2[t] = p.b2;
    }
}

// Rows first .. first + 31 of x (zeros past n): four inputs per thread, the
// first 256 threads another four.
struct MlpRows {
    f4u v[2];
};
static_assert(kMlpTiles * kMlpIn == 6 * kMlpThreads, "inputs per thread");

__device__ __forceinline__ MlpRows mlp_read_rows(const float* __restrict__ x, std::uint32_t first, std::uint32_t n) {
    MlpRows rows{};
#pragma unroll
    for (int i{0}; i < 2; ++i) {
        const std::uint32_t e{4 * (static_cast<std::uint32_t>(i * kMlpThreads) + threadIdx.x)};
        const std::uint32_t r{e / kMlpIn};
        if (r < static_cast<std::uint32_t>(kMlpTiles) && r < n - first) {
            rows.v[i] = *reinterpret_cast<const f4u*>(&x[static_cast<std::size_t>(first) * kMlpIn + e]);
        }
    }
    return rows;
}

__device__ __forceinline__ void mlp_store_rows(MlpShared& S, const MlpRows& rows) {
#pragma unroll
    for (int i{0}; i < 2; ++i) {
        const int e{4 * (i * kMlpThreads + static_cast<int>(threadIdx.x))};
        if (e < kMlpTiles * kMlpIn) {
            *reinterpret_cast<f4v*>(&S.x[e / kMlpIn][e % kMlpIn]) = rows.v[i];
        }
    }
}

// h = ReLU(W1 x + b1) of the tile: wave w takes rows 16 (w / 4) .. + 15 and
// hidden units 16 (w % 4) .. + 15.
__device__ __forceinline__ void mlp_hidden(MlpShared& S, const MlpParamsLane& p) {
    const int t{static_cast<int>(threadIdx.x)}, lane{t & 63}, w{t >> 6};
    const int c{lane & 15}, g{lane >> 4};
    const float* const xr{&S.x[16 * (w >> 2) + c][4 * g]};
    f4v acc{p.b, p.b, p.b, p.b}, odd{};
#pragma unroll
    for (int s{0}; s < kMlpIn / 16; ++s) {
        const f4v a{*reinterpret_cast<const f4v*>(&xr[16 * s])};
        acc = mlp_step_mfma(a[0], p.w[s][0], acc);
        odd = mlp_step_mfma(a[1], p.w[s][1], odd);
        acc = mlp_step_mfma(a[2], p.w[s][2], acc);
        odd = mlp_step_mfma(a[3], p.w[s][3], odd);
    }
#pragma unroll
    for (int u{0}; u < 4; ++u) {
        S.h[16 * (w >> 2) + 4 * g + u][16 * (w & 3) + c] = fmaxf(acc[u] + odd[u], 0.0f);
    }
}

// Output o = t % 8 of row t / 16 in the lanes of each row of 16 (both halves):
// lane t sums hidden units 32 (t / 8 % 2) .., the halves then add.
__device__ __forceinline__ float mlp_output(const MlpShared& S) {
    const int t{static_cast<int>(threadIdx.x)};
    const int r{t >> 4}, o{t & 7}, half{(t >> 3) & 1};
    float s0{half == 0 ? S.b2[o] : 0.0f}, s1{0.0f};
#pragma unroll
    for (int q{0}; q < 32; q += 8) {
        const float4 wa{*reinterpret_cast<const float4*>(&S.w2[o][32 * half + q])};
        const float4 wb{*reinterpret_cast<const float4*>(&S.w2[o][32 * half + q + 4])};
        const float4 ha{*reinterpret_cast<const float4*>(&S.h[r][32 * half + q])};
        const float4 hb{*reinterpret_cast<const float4*>(&S.h[r][32 * half + q + 4])};
        s0 = __builtin_fmaf(wa.x, ha.x, s0);
        s1 = __builtin_fmaf(wb.x, hb.x, s1);
        s0 = __builtin_fmaf(wa.y, ha.y, s0);
        s1 = __builtin_fmaf(wb.y, hb.y, s1);
        s0 = __builtin_fmaf(wa.z, ha.z, s0);
        s1 = __builtin_fmaf(wb.z, hb.z, s1);
        s0 = __builtin_fmaf(wa.w, ha.w, s0);
        s1 = __builtin_fmaf(wb.w, hb.w, s1);
    }
    const float s{s0 + s1};
    return s + __shfl_xor(s, 8, 64);
}

__global__ __launch_bounds__(kMlpThreads) __attribute__((amdgpu_waves_per_eu(4))) void mlp_grad_kernel(const float* __restrict__ params,
                                                               const float* __restrict__ x,
                                                               const float* __restrict__ labels, std::uint32_t n,
                                                               float lambda, float* __restrict__ partial) {
    __shared__ MlpGradShared S;
    const int t{static_cast<int>(threadIdx.x)}, lane{t & 63}, w{t >> 6};
    const int c{lane & 15}, g{lane >> 4};
    const std::uint32_t tiles{(n + kMlpTiles - 1) / kMlpTiles};
    MlpRows rows{mlp_read_rows(x, blockIdx.x * static_cast<std::uint32_t>(kMlpTiles), n)};
    const MlpParamsLane p{mlp_read_params(params)};
    mlp_store_params(S.f, p);
    // Sums over the workgroup's tiles.  W1: hidden units 16 (w % 4) .., inputs
    // 16 (3 (w / 4) + k) ..; W2 entry t (t < 448), else hidden bias t - 448;
    // output bias t.
    f4v gw1[3]{};
    float gw2{0.0f}, gb2{0.0f}, loss{0.0f};
    for (std::uint32_t tile{blockIdx.x}; tile < tiles; tile += gridDim.x) {
        const std::uint32_t first{tile * static_cast<std::uint32_t>(kMlpTiles)};
        const std::uint32_t row{first + static_cast<std::uint32_t>(t >> 4)};
        // The row's labels (used after the forward pass).
        const int o{t & 7};
        float lab{0.0f}, mask{0.0f};
        if (row < n) {
            const float* const l{labels + static_cast<std::size_t>(row) * kMlpLabels};
            lab = o == 6 ? l[5] : (o >= 2 && o < 6 ? l[o - 1] : l[0]);
            mask = o == 6 ? 1.0f : (o >= 2 && o < 6 ? l[5 + o] : l[6]);
        }
        mlp_store_rows(S.f, rows);
        __syncthreads();
        mlp_hidden(S.f, p);
        if (tile + gridDim.x < tiles) {
            rows = mlp_read_rows(x, (tile + gridDim.x) * static_cast<std::uint32_t>(kMlpTiles), n);
        }
        __syncthreads();
        // Outputs and their loss gradient.
        {
            const float z{mlp_output(S.f)};
            const float other{__shfl_xor(z, 1, 64)};  // lanes 0, 1: the two root logits
            float dz{0.0f}, part{0.0f};
            if (o < 2) {
                const float z0{o == 0 ? z : other}, z1{o == 0 ? other : z};
                const float mx{fmaxf(z0, z1)};
                const float e0{expf(z0 - mx)}, e1{expf(z1 - mx)};
                const float p1{e1 / (e0 + e1)};
                const bool y32{lab > 0.5f};
                part = o == 0 ? mask * (mx + logf(e0 + e1) - (y32 ? z1 : z0)) : 0.0f;
                dz = o == 0 ? mask * ((1.0f - p1) - (y32 ? 0.0f : 1.0f)) : mask * (p1 - (y32 ? 1.0f : 0.0f));
            } else if (o < 6) {
                const float sp{z > 30.0f ? z : log1pf(expf(z))};
                part = mask * (sp - lab * z);
                dz = mask * (1.0f / (1.0f + expf(-z)) - lab);
            } else if (o == 6) {
                const float d{z - lab};
                part = lambda * d * d;
                dz = 2.0f * lambda * d;
            }
            if (row >= n) {
                dz = 0.0f;
                part = 0.0f;
            }
            if ((t & 8) == 0) {
                S.dz[t >> 4][o] = dz;
                loss += part;
            }
        }
        __syncthreads();
        // Hidden gradients: rows 8 k + w, hidden unit `lane` (the ReLU mask
        // from the activations).
#pragma unroll
        for (int k{0}; k < kMlpTiles / 8; ++k) {
            const int r{8 * k + w};
            float s{0.0f};
#pragma unroll
            for (int q{0}; q < kMlpOut; ++q) {
                s = __builtin_fmaf(S.f.w2[q][lane], S.dz[r][q], s);
            }
            S.dh[r][lane] = S.f.h[r][lane] > 0.0f ? s : 0.0f;
        }
        if (t < kMlpOut * kMlpHid) {
            float s{0.0f};
            for (int r{0}; r < kMlpTiles; ++r) {
                s = __builtin_fmaf(S.dz[r][t >> 6], S.f.h[r][lane], s);
            }
            gw2 += s;
        }
        if (t < kMlpOut) {
            float s{0.0f};
            for (int r{0}; r < kMlpTiles; ++r) {
                s += S.dz[r][t];
            }
            gb2 += s;
        }
        __syncthreads();
        if (t >= kMlpOut * kMlpHid) {
            float s{0.0f};
            for (int r{0}; r < kMlpTiles; ++r) {
                s += S.dh[r][lane];
            }
            gw2 += s;
        }
        // First layer's gradient: dH^T X.
#pragma unroll
        for (int s{0}; s < kMlpTiles / 4; ++s) {
            const float a{S.dh[4 * s + g][16 * (w & 3) + c]};
#pragma unroll
            for (int k{0}; k < 3; ++k) {
                gw1[k] = mlp_step_mfma(a, S.f.x[4 * s + g][16 * (3 * (w >> 2) + k) + c], gw1[k]);
            }
        }
        __syncthreads();  // the tile's arrays are read
    }
    float* const out{partial + static_cast<std::size_t>(blockIdx.x) * (kMlpParams + 1)};
#pragma unroll
    for (int k{0}; k < 3; ++k) {
#pragma unroll
        for (int u{0}; u < 4; ++u) {
            out[(16 * (w & 3) + 4 * g + u) * kMlpIn + 16 * (3 * (w >> 2) + k) + c] = gw1[k][u];
        }
    }
    out[t < kMlpOut * kMlpHid ? kMlpW2 + t : kMlpB1 + lane] = gw2;
    if (t < kMlpOut) {
        out[kMlpB2 + t] = gb2;
    }
    for (int off{32}; off > 0; off >>= 1) {
        loss += __shfl_xor(loss, off, 64);
    }
    if (lane == 0) {
        S.loss[w] = loss;
    }
    __syncthreads();
    if (t == 0) {
        float s{0.0f};
        for (int k{0}; k < kMlpThreads / 64; ++k) {
            s += S.loss[k];
        }
        out[kMlpParams] = s;
    }
}

// grad[p] = (sum over the rows of partial[p]) / n; loss[0] likewise.  With
// lr > 0, one Adam step (beta1 0.9, beta2 0.999, eps 1e-8; `step` counts
// from 1) on params with moments m, v.  A workgroup takes 64 columns: wave w
// sums rows w, w + 16, ..., eight loads at a time, and the first wave adds the
// sixteen sums: bound by the latency of the loads, 4.0 us for 128 rows, 6.0
// for 512 (one thread per column over all rows: 31 for 128, 440 for 1,875).
constexpr int kMlpSlices = 16;

__global__ __launch_bounds__(64 * kMlpSlices) void mlp_reduce_kernel(
    const float* __restrict__ partial, std::uint32_t rows, std::uint32_t n, float* __restrict__ grad,
    float* __restrict__ loss, float* __restrict__ params, float* __restrict__ m, float* __restrict__ v,
    std::uint32_t step, float lr) {
    __shared__ float sums[kMlpSlices][64];
    const std::uint32_t lane{threadIdx.x & 63u}, w{threadIdx.x >> 6};
    const std::uint32_t p{blockIdx.x * 64u + lane};
    const bool in{p <= static_cast<std::uint32_t>(kMlpParams)};
    float s{0.0f};
    if (in) {
        const float* const col{partial + p};
        std::uint32_t r{w};
        for (; r + 7 * kMlpSlices < rows; r += 8 * kMlpSlices) {
            float x[8];
#pragma unroll
            for (std::uint32_t k{0}; k < 8; ++k) {
                x[k] = col[static_cast<std::size_t>(r + k * kMlpSlices) * (kMlpParams + 1)];
            }
            s += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        }
        for (; r < rows; r += kMlpSlices) {
            s += col[static_cast<std::size_t>(r) * (kMlpParams + 1)];
        }
    }
    sums[w][lane] = s;
    __syncthreads();
    if (w != 0 || !in) {
        return;
    }
    float t[kMlpSlices];
#pragma unroll
    for (int k{0}; k < kMlpSlices; ++k) {
        t[k] = sums[k][lane];
    }
#pragma unroll
    for (int k{kMlpSlices / 2}; k > 0; k >>= 1) {
        for (int i{0}; i < k; ++i) {
            t[i] += t[i + k];
        }
    }
    const float g{t[0] / static_cast<float>(n)};
    if (p == static_cast<std::uint32_t>(kMlpParams)) {
        loss[0] = g;
        return;
    }
    grad[p] = g;
    if (lr > 0.0f) {
        const float b1{0.9f}, b2{0.999f};
        const float mp{b1 * m[p] + (1.0f - b1) * g};
        const float vp{b2 * v[p] + (1.0f - b2) * g * g};
        m[p] = mp;
        v[p] = vp;
        const float c1{1.0f - powf(b1, static_cast<float>(step))};
        const float c2{1.0f - powf(b2, static_cast<float>(step))};
        params[p] -= lr * (mp / c1) / (sqrtf(vp / c2) + 1e-8f);
    }
}

// Outputs z[n][7] of the FP32 network (evaluation of training runs): a
// workgroup takes tiles of 32 rows.
__global__ __launch_bounds__(kMlpThreads) void mlp_forward_kernel(const float* __restrict__ params,
                                                                  const float* __restrict__ x, std::uint32_t n,
                                                                  float* __restrict__ z) {
    __shared__ MlpShared S;
    const std::uint32_t tiles{(n + kMlpTiles - 1) / kMlpTiles};
    const int t{static_cast<int>(threadIdx.x)};
    MlpRows rows{mlp_read_rows(x, blockIdx.x * static_cast<std::uint32_t>(kMlpTiles), n)};
    const MlpParamsLane p{mlp_read_params(params)};
    mlp_store_params(S, p);
    for (std::uint32_t tile{blockIdx.x}; tile < tiles; tile += gridDim.x) {
        const std::uint32_t first{tile * static_cast<std::uint32_t>(kMlpTiles)};
        mlp_store_rows(S, rows);
        __syncthreads();
        mlp_hidden(S, p);
        if (tile + gridDim.x < tiles) {
            rows = mlp_read_rows(x, (tile + gridDim.x) * static_cast<std::uint32_t>(kMlpTiles), n);
        }
        __syncthreads();
        const float out{mlp_output(S)};
        const std::uint32_t row{first + static_cast<std::uint32_t>(t >> 4)};
        if ((t & 15) < kMlpOut && row < n) {
            z[static_cast<std::size_t>(row) * kMlpOut + (t & 15)] = out;
        }
    }
}

}  // namespace cjx
