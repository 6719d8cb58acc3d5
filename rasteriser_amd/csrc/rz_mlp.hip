// rz_mlp.hip — packing, inference and training kernels of the learned shader (rz_mlp.h).
//
// Training is minibatch Adam on FP32 master weights.  The forward pass rounds weights
// and activations to BF16 exactly where inference does (inputs, hidden activations),
// so the trained network is the one the matrix cores evaluate; gradients are FP32 and
// pass straight through the rounding.  Loss: mean over the batch of the squared error
// summed over the three channels.
#include "rz_device.h"
#include "rz_mlp.h"

namespace rz {

// ---------------------------------------------------------------------------------
// m, v: Adam's moments to clear (new weights), or null.
__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ W, uint16_t* __restrict__ packed,
                                                  float* __restrict__ m, float* __restrict__ v) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (m && i < kMlpParams) {
        m[i] = 0.f;
        v[i] = 0.f;
    }
    if (i < kFragL2) {
        const int h = i / 256, lane = (i / 4) % 64, j = i % 4;
        const int o = 16 * h + lane % 16, k = 4 * (lane / 16) + j;
        packed[i] = to_bf16(k < kMlpIn ? W[kOffW1 + o * kMlpIn + k] : 0.f);
    } else if (i < kFragL3) {
        // [h][t][lane][8]: A[m][8g + j] = W2[16h + m][u(t, g, j)]
        const int q = i - kFragL2, ht = q / 512, lane = (q / 8) % 64, j = q % 8;
        const int h = ht / 2, t = ht % 2;
        const int o = 16 * h + lane % 16, k = mlp_k32_unit(t, lane / 16, j);
        packed[i] = to_bf16(W[kOffW2 + o * kMlpHidden + k]);
    } else if (i < kFragEnd) {
        // [t][lane][8]: A[m][8g + j] = W3[m][u(t, g, j)] (rows 3..15 zero)
        const int q = i - kFragL3, t = q / 512, lane = (q / 8) % 64, j = q % 8;
        const int o = lane % 16, k = mlp_k32_unit(t, lane / 16, j);
        packed[i] = to_bf16(o < kMlpOut ? W[kOffW3 + o * kMlpHidden + k] : 0.f);
    } else if (i < kFragEnd + 144) {
        float* bias = reinterpret_cast<float*>(packed + kFragEnd);
        const int b = i - kFragEnd;
        bias[b] = b < 64 ? W[kOffB1 + b] : b < 128 ? W[kOffB2 + b - 64] : (b - 128 < kMlpOut ? W[kOffB3 + b - 128] : 0.f);
    }
}

// Inference over a feature array [n][12] -> [n][3] (the shading pass runs the same
// mlp_wave on fragments it computes itself).
__global__ __launch_bounds__(256) void k_mlp_infer(const float* __restrict__ x, int64_t n,
                                                   const uint16_t* __restrict__ packed, float* __restrict__ y) {
    __shared__ __align__(16) uint16_t s_net[kPackedBytes / 2];
    __shared__ __align__(16) uint16_t s_in[4][64 * 16];
    __shared__ __align__(16) float s_out[4][64 * 4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t i = (int64_t)blockIdx.x * 256 + tid;
    stage_net(packed, s_net, tid, 256);
#pragma unroll
    for (int k = 0; k < 16; ++k)
        s_in[wave][lane * 16 + k] = to_bf16((i < n && k < kMlpIn) ? x[i * kMlpIn + k] : 0.f);
    __syncthreads();
    mlp_wave(s_net, s_in[wave], s_out[wave], lane);
    __syncthreads();
    if (i < n)
        for (int c = 0; c < kMlpOut; ++c) y[i * kMlpOut + c] = s_out[wave][lane * 4 + c];
}

// ---------------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// One training step's gradient.  A workgroup of four waves takes 64 samples at a time
// (drawn at random from the training set), 16 to a wave, and keeps the summed parameter
// gradient of its samples in accumulators over all its chunks (chunk, chunk + grid, ...),
// so a step writes one partial gradient per workgroup.
//
// Every product runs on the matrix cores.  The forward pass is mlp_wave's (bf16 operands,
// f32 accumulation); its accumulators leave hidden unit 16h + 4g + j of sample col in lane
// (g, col), which is also row g of the B operand of an f32 16x16x4 product whose four k
// are the units 16h + 4g + j, g = 0..3: the backward product W2^T delta2 takes delta2 from
// the registers it was formed in.  The gradients contract over the samples, so the
// activations and deltas pass through LDS once ([sample][unit], rows of 80 words: the 64
// lanes of an operand read, 4 samples by 16 units, fall on 64 different banks); wave w
// forms rows 16w..16w+15 of gW2 and gW1 and columns 16w..16w+15 of gW3.  Deltas stay f32
// throughout (f32 matrix products: a bf16 split would need three products and its own
// error bound, and these take about 1 us of the step).
//
// What bounds it: one chunk's chain of dependent loads, products and barriers; one
// workgroup to a CU at 16,384 samples.  A step of 16,384 samples there: 154 us as scalar
// products from LDS in one wave a workgroup, 13.9 us in this form.
constexpr int kRow = 80;
constexpr int kWRow = 68;                                  // W2 rows in LDS (both its reads on different banks)
constexpr int kGradStride = (kMlpParams + 63) / 64 * 64;   // floats between partial gradients
constexpr int kGradBlocks = 256;                           // one workgroup per CU

__device__ __forceinline__ mlp_f4 mfma_f32(float a, float b, mlp_f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four floats (16-byte aligned) as a bf16 fragment, or zeros.
__device__ __forceinline__ mlp_s4 frag4(const float* w, bool keep = true) {
    const uint2 v = make_uint2(bf16x2(w[0], w[1]), bf16x2(w[2], w[3]));
    return __builtin_bit_cast(mlp_s4, make_uint2(keep ? v.x : 0u, keep ? v.y : 0u));
}

__global__ __launch_bounds__(256) void k_mlp_grad(const float* __restrict__ samples, int64_t n,
                                                  const float* __restrict__ W, float* __restrict__ gpart,
                                                  float* __restrict__ lpart, uint64_t seed, uint32_t step,
                                                  float inv_batch, uint32_t chunks) {
    __shared__ __align__(16) float sH1[64][kRow], sH2[64][kRow], sD1[64][kRow], sD2[64][kRow];
    __shared__ __align__(16) float sX[64][16];
    __shared__ float sDY[64][4];
    __shared__ float sLoss[4];
    __shared__ __align__(16) float sW1[kMlpHidden * kMlpIn + 4], sW2[kMlpHidden][kWRow], sW3[kMlpOut][kMlpHidden];
    __shared__ __align__(16) float sB1[kMlpHidden], sB2[kMlpHidden], sB3[4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, col = lane & 15;
    const int s = 16 * wave + col;   // the lane's sample within a chunk (the wave's four rows share it)
    // a chunk's sample: inputs 4g..4g+3 (g < 3), or the three targets (g = 3)
    float x[4];
    auto load = [&](uint32_t chunk) {
        const uint64_t gid = (uint64_t)chunk * 64 + s;
        const int64_t idx = (int64_t)(mix64(seed + 0x9E3779B97F4A7C15ull * ((uint64_t)step * 1048576u + gid + 1)) %
                                      (uint64_t)n);
        const float* smp = samples + idx * kMlpSampleFloats + 4 * g;
        x[0] = smp[0];
        x[1] = smp[1];
        x[2] = smp[2];
        x[3] = g < 3 ? smp[3] : 0.f;
    };
    load(blockIdx.x);
    // weights rounded to bf16 and biases into LDS, read once per workgroup (the fragments
    // below straight from global memory, about 200 narrow loads a wave: 14.2 against 13.9 us)
    for (int e = tid; e < kMlpHidden * kMlpIn; e += 256) sW1[e] = round_bf16(W[kOffW1 + e]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = 4 * (q * 256 + tid);
        const float4 w = *reinterpret_cast<const float4*>(W + kOffW2 + e);
        *reinterpret_cast<float4*>(&sW2[e >> 6][e & 63]) =
            make_float4(round_bf16(w.x), round_bf16(w.y), round_bf16(w.z), round_bf16(w.w));
    }
    if (tid < kMlpOut * kMlpHidden) sW3[tid >> 6][tid & 63] = round_bf16(W[kOffW3 + tid]);
    if (tid < kMlpHidden) {
        sB1[tid] = W[kOffB1 + tid];
        sB2[tid] = W[kOffB2 + tid];
    }
    if (tid < kMlpOut) sB3[tid] = W[kOffB3 + tid];
    __syncthreads();
    // weight fragments as packed for inference (k_mlp_pack), and the weights of the
    // backward pass
    mlp_s4 f1[4];
    mlp_s8 f2[4][2], f3[2];
    float w2t[4][4][4], w3[3][4][4], b1[4][4], b2[4][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        f1[h] = frag4(sW1 + (16 * h + col) * kMlpIn + 4 * g, g < 3);   // (g = 3 reads on past the row: 12 inputs)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const float* r = &sW2[16 * h + col][32 * t + 4 * g];   // units u(t, g, 0..3) and u(t, g, 4..7)
            f2[h][t] = __builtin_shufflevector(frag4(r), frag4(r + 16), 0, 1, 2, 3, 4, 5, 6, 7);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int unit = 16 * h + 4 * g + j;
            b1[h][j] = sB1[unit];
            b2[h][j] = sB2[unit];
#pragma unroll
            for (int c = 0; c < kMlpOut; ++c) w3[c][h][j] = sW3[c][unit];
#pragma unroll
            for (int k = 0; k < 4; ++k) w2t[h][j][k] = sW2[unit][16 * k + col];
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float* r = &sW3[col < kMlpOut ? col : 0][32 * t + 4 * g];
        f3[t] = __builtin_shufflevector(frag4(r, col < kMlpOut), frag4(r + 16, col < kMlpOut), 0, 1, 2, 3, 4, 5, 6, 7);
    }
    const float b3[3] = {sB3[0], sB3[1], sB3[2]};

    const mlp_f4 z4 = {0.f, 0.f, 0.f, 0.f};
    mlp_f4 gw2[4] = {z4, z4, z4, z4}, gw1 = z4, gw3 = z4;
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, loss = 0.f;
    for (uint32_t chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x) {   // (uniform)
        const mlp_s4 xb = frag4(x, g < 3);
        if (g < 3)
            *reinterpret_cast<float4*>(&sX[s][4 * g]) =
                make_float4(round_bf16(x[0]), round_bf16(x[1]), round_bf16(x[2]), round_bf16(x[3]));
        else
            *reinterpret_cast<float4*>(&sX[s][12]) = make_float4(0.f, 0.f, 0.f, 0.f);
        // forward: pre-activations kept for relu'
        float a1[4][4], a2[4][4];
        mlp_s4 h1[4], h2[4];
        auto layer = [&](const mlp_f4& acc, const float* b, float* a, mlp_s4& hb, float* row) {
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = acc[j] + b[j];
            const float r[4] = {fmaxf(a[0], 0.f), fmaxf(a[1], 0.f), fmaxf(a[2], 0.f), fmaxf(a[3], 0.f)};
            hb = frag4(r);
            *reinterpret_cast<float4*>(row) =
                make_float4(from_bf16((uint16_t)hb[0]), from_bf16((uint16_t)hb[1]), from_bf16((uint16_t)hb[2]),
                            from_bf16((uint16_t)hb[3]));
        };
#pragma unroll
        for (int h = 0; h < 4; ++h)
            layer(__builtin_amdgcn_mfma_f32_16x16x16bf16_1k(f1[h], xb, z4, 0, 0, 0), b1[h], a1[h], h1[h],
                  &sH1[s][16 * h + 4 * g]);
        {
            const mlp_s8 k0 = __builtin_shufflevector(h1[0], h1[1], 0, 1, 2, 3, 4, 5, 6, 7);
            const mlp_s8 k1 = __builtin_shufflevector(h1[2], h1[3], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int h = 0; h < 4; ++h)
                layer(mfma_k32(f2[h][1], k1, mfma_k32(f2[h][0], k0, z4)), b2[h], a2[h], h2[h], &sH2[s][16 * h + 4 * g]);
        }
        const mlp_f4 y = mfma_k32(f3[1], __builtin_shufflevector(h2[2], h2[3], 0, 1, 2, 3, 4, 5, 6, 7),
                                  mfma_k32(f3[0], __builtin_shufflevector(h2[0], h2[1], 0, 1, 2, 3, 4, 5, 6, 7), z4));
        // residuals in the lanes of row 0 (outputs 0..2), their scaled values to every row
        const float target[3] = {x[0], x[1], x[2]};   // (row 3's)
        if (chunk + gridDim.x < chunks) load(chunk + gridDim.x);   // the next chunk's, behind the backward pass
        float dy[3];
#pragma unroll
        for (int c = 0; c < kMlpOut; ++c) {
            const float r = y[c] + b3[c] - __shfl(target[c], 48 + col, 64);
            if (g == 0) loss += r * r;
            dy[c] = __shfl(2.f * r * inv_batch, col, 64);
            if (g == 0) sDY[s][c] = dy[c];
        }
        // backward through the activations
        float d2[4][4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float v = w3[0][h][j] * dy[0] + w3[1][h][j] * dy[1] + w3[2][h][j] * dy[2];
                d2[h][j] = a2[h][j] > 0.f ? v : 0.f;
            }
            *reinterpret_cast<float4*>(&sD2[s][16 * h + 4 * g]) = make_float4(d2[h][0], d2[h][1], d2[h][2], d2[h][3]);
        }
        mlp_f4 e[4] = {z4, z4, z4, z4};
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int k = 0; k < 4; ++k) e[k] = mfma_f32(w2t[h][j][k], d2[h][j], e[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            *reinterpret_cast<float4*>(&sD1[s][16 * k + 4 * g]) =
                make_float4(a1[k][0] > 0.f ? e[k][0] : 0.f, a1[k][1] > 0.f ? e[k][1] : 0.f,
                            a1[k][2] > 0.f ? e[k][2] : 0.f, a1[k][3] > 0.f ? e[k][3] : 0.f);
        __syncthreads();
        // parameter gradients over the chunk's 64 samples, four to a product
#pragma unroll 4
        for (int q = 0; q < 16; ++q) {
            const int r = 4 * q + g;
            const float p2 = sD2[r][16 * wave + col], p1 = sD1[r][16 * wave + col];
            const float py = col < kMlpOut ? sDY[r][col] : 0.f;
            gb2 += p2;
            gb1 += p1;
            gb3 += py;
#pragma unroll
            for (int t = 0; t < 4; ++t) gw2[t] = mfma_f32(p2, sH1[r][16 * t + col], gw2[t]);
            gw1 = mfma_f32(p1, sX[r][col], gw1);
            gw3 = mfma_f32(py, sH2[r][16 * wave + col], gw3);
        }
        __syncthreads();   // (the next chunk rewrites the activations)
    }

    auto rows4 = [](float v) {   // over the wave's four rows
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
    gb1 = rows4(gb1);
    gb2 = rows4(gb2);
    gb3 = rows4(gb3);
    float* out = gpart + (size_t)blockIdx.x * kGradStride;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int o = 16 * wave + 4 * g + j;
#pragma unroll
        for (int t = 0; t < 4; ++t) out[kOffW2 + o * kMlpHidden + 16 * t + col] = gw2[t][j];
        if (col < kMlpIn) out[kOffW1 + o * kMlpIn + col] = gw1[j];
        if (g == 0 && j < kMlpOut) out[kOffW3 + j * kMlpHidden + 16 * wave + col] = gw3[j];
    }
    if (g == 0) {
        out[kOffB1 + 16 * wave + col] = gb1;
        out[kOffB2 + 16 * wave + col] = gb2;
        if (wave == 0 && col < kMlpOut) out[kOffB3 + col] = gb3;
    }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) loss += __shfl_xor(loss, m, 64);
    if (lane == 0) sLoss[wave] = loss;
    __syncthreads();
    if (tid == 0) lpart[blockIdx.x] = (sLoss[0] + sLoss[1]) + (sLoss[2] + sLoss[3]);
}

// Sums the partial gradients and updates the weights: 64 parameters to a workgroup, its 16
// waves each summing every 16th partial (one thread per parameter over all of them: a
// serial chain of 256 loads, 69 us).  The last workgroup sums the loss.
constexpr int kAdamBlocks = kGradStride / 64;
__global__ __launch_bounds__(1024) void k_mlp_adam(float* __restrict__ W, float* __restrict__ m, float* __restrict__ v,
                                                   const float* __restrict__ gpart, int nparts,
                                                   const float* __restrict__ lpart, float* __restrict__ loss_out,
                                                   float lr, float c1, float c2) {
    __shared__ float s_sum[16][64];
    const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const bool params = blockIdx.x < kAdamBlocks;   // (uniform)
    const int e = blockIdx.x * 64 + lane;
    float g = 0.f;
    if (params) {
        if (e < kMlpParams) {
#pragma unroll 8
            for (int b = slice; b < nparts; b += 16) g += gpart[(size_t)b * kGradStride + e];
        }
    } else {
        for (int b = threadIdx.x; b < nparts; b += 1024) g += lpart[b];
    }
    s_sum[slice][lane] = g;
    __syncthreads();
    if (slice != 0) return;
    g = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) g += s_sum[k][lane];
    if (!params) {
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) g += __shfl_xor(g, k, 64);
        if (lane == 0) *loss_out = g;
    } else if (e < kMlpParams) {
        const float mm = 0.9f * m[e] + 0.1f * g;
        const float vv = 0.999f * v[e] + 0.001f * g * g;
        m[e] = mm;
        v[e] = vv;
        W[e] -= lr * (mm * c1) / (sqrtf(vv * c2) + 1e-8f);
    }
}

hipError_t launch_mlp_pack(const float* W, uint16_t* packed, float* m, float* v, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_pack, dim3((kFragEnd + 144 + 255) / 256), dim3(256), 0, s, W, packed, m, v);
    return hipGetLastError();
}

hipError_t launch_mlp_infer(const float* x, int64_t n, const uint16_t* packed, float* y, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_mlp_infer, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, n, packed, y);
    return hipGetLastError();
}

// Partial gradients of a step of `batch` samples, and the floats between them.
int mlp_grad_parts(int batch) { return batch / 64 < kGradBlocks ? batch / 64 : kGradBlocks; }
size_t mlp_grad_stride() { return kGradStride; }

hipError_t launch_mlp_step(const float* samples, int64_t n, float* W, float* m, float* v, float* gpart,
                           float* lpart, float* loss_out, int batch, uint64_t seed, uint32_t step, float lr,
                           float c1, float c2, hipStream_t s) {
    const int chunks = batch / 64, parts = mlp_grad_parts(batch);
    hipLaunchKernelGGL(k_mlp_grad, dim3(parts), dim3(256), 0, s, samples, n, (const float*)W, gpart, lpart, seed,
                       step, 1.0f / (float)(chunks * 64), (uint32_t)chunks);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mlp_adam, dim3(kAdamBlocks + 1), dim3(1024), 0, s, W, m, v, (const float*)gpart, parts,
                       (const float*)lpart, loss_out, lr, c1, c2);
    return hipGetLastError();
}

}  // namespace rz
