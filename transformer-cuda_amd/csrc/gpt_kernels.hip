// gpt_kernels.hip - the element-wise and reduction kernels of the GPT training-step harness
// around the attention path and the products (fp32): embedding, LayerNorm, column sums (LayerNorm
// parameter and position gradients), fused cross-entropy, and the fused gradient-clip + AdamW +
// zero-grad update.  GELU, residuals and the bias gradients are the products' (gpt_epilogue.hpp).
//
// Reference (behaviour, one kernel family each): src/kernels/embedding.cu (token + position
// gather, scatter-add backward), src/kernels/layernorm.cu:29-303 (biased variance, eps inside
// the square root), src/kernels/loss.cu:24-125 (mean cross-entropy, dlogits = (softmax - onehot) /
// (B*T)), src/optimizer.cu:117-154 (global-norm clip folded into AdamW with decoupled weight
// decay, then zero the gradient).
//
// LayerNorm runs one wave64 per row, cross-entropy one workgroup; reductions over rows (gamma, beta
// and position-embedding gradients) are two-stage and deterministic: partial sums over fixed row
// shares, then a sum of them in order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "gpt_kernels.hpp"

namespace tcamd {
namespace gpt {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;
constexpr int kRowsPerBlock = kBlock / kWave;

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int off = kWave / 2; off >= 1; off >>= 1) x += __shfl_xor(x, off, kWave);
    return x;
}
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
    for (int off = kWave / 2; off >= 1; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, kWave));
    return x;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
inline unsigned blocks_for(long long n, int per_block) {
    return static_cast<unsigned>((n + per_block - 1) / per_block);
}

// ---- embedding ------------------------------------------------------------------------
__global__ void embedding_fwd_kernel(const int* __restrict__ tokens,
                                     const float* __restrict__ tok_emb,
                                     const float* __restrict__ pos_emb, float* __restrict__ out,
                                     int BT, int T, int C) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<long long>(BT) * C) return;
    const int row = static_cast<int>(i / C), c = static_cast<int>(i % C);
    out[i] = tok_emb[static_cast<long long>(tokens[row]) * C + c] +
             pos_emb[static_cast<long long>(row % T) * C + c];
}

// d_tok_emb[token] += dx[row] (tokens repeat: atomic adds).
__global__ void embedding_tok_bwd_kernel(const int* __restrict__ tokens,
                                         const float* __restrict__ dx,
                                         float* __restrict__ d_tok_emb, int BT, int C) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<long long>(BT) * C) return;
    const int row = static_cast<int>(i / C), c = static_cast<int>(i % C);
    atomicAdd(&d_tok_emb[static_cast<long long>(tokens[row]) * C + c], dx[i]);
}

// ---- column sums: out[n] = sum_r x[r, n] (beta: out = sum + beta*out) -----------------
constexpr int kChunkRows = 128;

// partial[chunk][n] = sum over the chunk's rows; with ln_x != nullptr the summand is
// x[r,n] times the normalised input (ln_x[r,n] - mean[r]) * rstd[r] (the LayerNorm gamma
// gradient).  A block covers 64 columns (one wave's lanes, 256 contiguous bytes per row)
// and the chunk's rows split over its 4 waves, two rows in flight per thread; the 4 partial
// sums of a column meet in LDS.
constexpr int kColTile = kWave;
constexpr int kColLanes = kBlock / kColTile;
__global__ __launch_bounds__(kBlock) void colsum_partial_kernel(
    const float* __restrict__ x, int R, int N, const float* __restrict__ ln_x,
    const float* __restrict__ ln_mean, const float* __restrict__ ln_rstd,
    float* __restrict__ partial) {
    __shared__ float red[kColLanes][kColTile];
    const int c = threadIdx.x % kColTile, j = threadIdx.x / kColTile;
    const int n = blockIdx.x * kColTile + c;
    const int r0 = blockIdx.y * kChunkRows, r1 = min(R, r0 + kChunkRows);
    auto term = [&](int r) {
        const long long i = static_cast<long long>(r) * N + n;
        return ln_x != nullptr ? x[i] * ((ln_x[i] - ln_mean[r]) * ln_rstd[r]) : x[i];
    };
    float s0 = 0.0f, s1 = 0.0f;
    if (n < N) {
        int r = r0 + j;
        for (; r + kColLanes < r1; r += 2 * kColLanes) {
            s0 += term(r);
            s1 += term(r + kColLanes);
        }
        if (r < r1) s0 += term(r);
    }
    red[j][c] = s0 + s1;
    __syncthreads();
    if (j == 0 && n < N) {
        float t = red[0][c];
#pragma unroll
        for (int i = 1; i < kColLanes; ++i) t += red[i][c];
        partial[static_cast<long long>(blockIdx.y) * N + n] = t;
    }
}

// out[n] = sum over the nchunk partial rows: a block covers 16 columns, its 16 lanes per
// column stride over the chunks.
constexpr int kFinCols = 16;
constexpr int kFinLanes = kBlock / kFinCols;
__global__ __launch_bounds__(kBlock) void colsum_final_kernel(const float* __restrict__ partial,
                                                              int nchunk, int N,
                                                              float* __restrict__ out) {
    __shared__ float red[kFinLanes][kFinCols + 1];
    const int c = threadIdx.x % kFinCols, j = threadIdx.x / kFinCols;
    const int n = blockIdx.x * kFinCols + c;
    float s = 0.0f;
    if (n < N) {
        // four rows in flight: a lane's 32 dependent loads of the 512 LayerNorm partials took 11 us
        float t[4] = {};
        int k = j;
        for (; k + 3 * kFinLanes < nchunk; k += 4 * kFinLanes)
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] += partial[static_cast<long long>(k + i * kFinLanes) * N + n];
        for (; k < nchunk; k += kFinLanes) s += partial[static_cast<long long>(k) * N + n];
        s += (t[0] + t[1]) + (t[2] + t[3]);
    }
    red[j][c] = s;
    __syncthreads();
    if (j == 0 && n < N) {
        float t = red[0][c];
        for (int i = 1; i < kFinLanes; ++i) t += red[i][c];
        out[n] = t;
    }
}

// out[i] = sum_j x[j*n + i], the slices in order: a thread per V elements (V = 4: 16-byte
// accesses, n and the pointers' alignment allowing).  HBM-bound: the slices were just written,
// and the reads of four at a time are in flight together.
template <int V>
__global__ __launch_bounds__(kBlock) void slice_sum_kernel(const float* __restrict__ x,
                                                           int nslice, long long n,
                                                           float* __restrict__ out) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const long long i = (static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x) * V;
    if (i >= n) return;
    vec s = {};
#pragma unroll 4
    for (int j = 0; j < nslice; ++j) s += *reinterpret_cast<const vec*>(x + j * n + i);
    *reinterpret_cast<vec*>(out + i) = s;
}

// ---- LayerNorm ---------------------------------------------------------------------------
// HBM-bound passes over (rows, C).  A wave holds its row in registers, a lane V neighbouring
// columns of each of NV groups of 64 V, so that a row is read once and its loads are all in
// flight: forward 18.3 -> 11 us, backward with its parameter gradients 66 -> 28 us at 8192 x 768
// (a second read of the row for every pass over it, and two column-sum launches with 4-byte
// accesses, before).  Rows of more than 2048 columns, or of a number that V does not divide,
// take the kernels after these.
template <int V>
using vecf = float __attribute__((ext_vector_type(V)));

template <int V, int NV>
__global__ __launch_bounds__(kBlock) void layernorm_fwd_row_kernel(
    const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, float* __restrict__ y, float* __restrict__ mean_out,
    float* __restrict__ rstd_out, int R, int C, float eps) {
    const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    if (row >= R) return;
    const float* xr = x + static_cast<long long>(row) * C;
    vecf<V> v[NV];
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = V * (lane + kWave * i);
        v[i] = c < C ? *reinterpret_cast<const vecf<V>*>(xr + c) : vecf<V>{};
#pragma unroll
        for (int e = 0; e < V; ++e) s += v[i][e];
    }
    const float mean = wave_sum(s) / C;
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (V * (lane + kWave * i) < C)
#pragma unroll
            for (int e = 0; e < V; ++e) q = fmaf(v[i][e] - mean, v[i][e] - mean, q);
    }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / C + eps);
    float* yr = y + static_cast<long long>(row) * C;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = V * (lane + kWave * i);
        if (c >= C) continue;
        const vecf<V> g = *reinterpret_cast<const vecf<V>*>(gamma + c);
        const vecf<V> b = *reinterpret_cast<const vecf<V>*>(beta + c);
        vecf<V> o;
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = fmaf((v[i][e] - mean) * rstd, g[e], b[e]);
        *reinterpret_cast<vecf<V>*>(yr + c) = o;
    }
    if (lane == 0) {
        mean_out[row] = mean;
        rstd_out[row] = rstd;
    }
}

// dx as layernorm_bwd_kernel's, and the workgroup's share of dgamma = sum_r dy xhat and dbeta =
// sum_r dy as row blockIdx.x of partial (rows of 2 C: dgamma, dbeta).  Workgroups take rows in
// turn, so the grid bounds the partial rows.
template <int V, int NV>
__global__ __launch_bounds__(kBlock) void layernorm_bwd_row_kernel(
    const float* __restrict__ dy, const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ mean, const float* __restrict__ rstd, float* __restrict__ dx,
    float* __restrict__ partial, int R, int C, int accumulate) {
    __shared__ __attribute__((aligned(16))) float red[kRowsPerBlock][NV * V * kWave];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    vecf<V> dg[NV], db[NV], gm[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = V * (lane + kWave * i);
        dg[i] = vecf<V>{};
        db[i] = vecf<V>{};
        gm[i] = c < C ? *reinterpret_cast<const vecf<V>*>(gamma + c) : vecf<V>{};
    }
    for (int row = blockIdx.x * kRowsPerBlock + w; row < R; row += gridDim.x * kRowsPerBlock) {
        const long long base = static_cast<long long>(row) * C;
        const float mu = mean[row], rs = rstd[row];
        vecf<V> g[NV], xh[NV], old[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = V * (lane + kWave * i);
            const bool in = c < C;
            g[i] = in ? *reinterpret_cast<const vecf<V>*>(dy + base + c) : vecf<V>{};
            xh[i] = in ? *reinterpret_cast<const vecf<V>*>(x + base + c) : vecf<V>{};
            old[i] = in && accumulate ? *reinterpret_cast<const vecf<V>*>(dx + base + c) : vecf<V>{};
        }
        float sg = 0.0f, sgx = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float d = g[i][e];
                xh[i][e] = (xh[i][e] - mu) * rs;
                if (V * (lane + kWave * i) < C) dg[i][e] = fmaf(d, xh[i][e], dg[i][e]);
                db[i][e] += d;
                g[i][e] = d * gm[i][e];
                sg += g[i][e];
                sgx = fmaf(g[i][e], xh[i][e], sgx);
            }
        const float mg = wave_sum(sg) / C, mgx = wave_sum(sgx) / C;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = V * (lane + kWave * i);
            if (c >= C) continue;
            vecf<V> o;
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float d = rs * (g[i][e] - mg - xh[i][e] * mgx);
                o[e] = accumulate ? old[i][e] + d : d;
            }
            *reinterpret_cast<vecf<V>*>(dx + base + c) = o;
        }
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NV; ++i)
            *reinterpret_cast<vecf<V>*>(&red[w][V * (lane + kWave * i)]) = half == 0 ? dg[i] : db[i];
        __syncthreads();
        for (int c = threadIdx.x; c < C; c += kBlock) {
            float t = red[0][c];
#pragma unroll
            for (int j = 1; j < kRowsPerBlock; ++j) t += red[j][c];
            partial[(static_cast<long long>(blockIdx.x) * 2 + half) * C + c] = t;
        }
    }
}

__global__ __launch_bounds__(kBlock) void layernorm_fwd_kernel(
    const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, float* __restrict__ y, float* __restrict__ mean_out,
    float* __restrict__ rstd_out, int R, int C, float eps) {
    const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    if (row >= R) return;
    const float* xr = x + static_cast<long long>(row) * C;
    float s = 0.0f;
    for (int c = lane; c < C; c += kWave) s += xr[c];
    const float mean = wave_sum(s) / C;
    float v = 0.0f;
    for (int c = lane; c < C; c += kWave) {
        const float d = xr[c] - mean;
        v = fmaf(d, d, v);
    }
    const float rstd = 1.0f / sqrtf(wave_sum(v) / C + eps);
    float* yr = y + static_cast<long long>(row) * C;
    for (int c = lane; c < C; c += kWave) yr[c] = fmaf((xr[c] - mean) * rstd, gamma[c], beta[c]);
    if (lane == 0) {
        mean_out[row] = mean;
        rstd_out[row] = rstd;
    }
}

// dx = rstd * (g - mean(g) - xhat * mean(g * xhat)), g = dy * gamma; dx is added to
// (accumulate) or written.
__global__ __launch_bounds__(kBlock) void layernorm_bwd_kernel(
    const float* __restrict__ dy, const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ mean, const float* __restrict__ rstd, float* __restrict__ dx,
    int R, int C, int accumulate) {
    const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    if (row >= R) return;
    const long long base = static_cast<long long>(row) * C;
    const float mu = mean[row], rs = rstd[row];
    float sg = 0.0f, sgx = 0.0f;
    for (int c = lane; c < C; c += kWave) {
        const float g = dy[base + c] * gamma[c];
        sg += g;
        sgx = fmaf(g, (x[base + c] - mu) * rs, sgx);
    }
    const float mg = wave_sum(sg) / C, mgx = wave_sum(sgx) / C;
    for (int c = lane; c < C; c += kWave) {
        const float g = dy[base + c] * gamma[c];
        const float xh = (x[base + c] - mu) * rs;
        const float d = rs * (g - mg - xh * mgx);
        dx[base + c] = accumulate ? dx[base + c] + d : d;
    }
}

// ---- cross-entropy ----------------------------------------------------------------------
// One workgroup per row, the row in registers: THREADS x NV groups of four neighbouring logits,
// read once and replaced by their exponentials, which give both the sum and the gradient.
// HBM-bound: the logits read and the gradient written.  8192 x 50257: 1324 -> 660 us (3.3 GB
// at 5.0 TB/s; the kernel after it reads every row twice and takes each exponential twice).
template <int THREADS, int NV>
__global__ __launch_bounds__(THREADS) void cross_entropy_row_kernel(
    const float* __restrict__ logits, const int* __restrict__ targets,
    float* __restrict__ dlogits, float* __restrict__ row_loss, int V, float inv_rows) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows start anywhere
    __shared__ float red[2][THREADS / kWave];
    const int row = blockIdx.x;
    const int tid = threadIdx.x, lane = tid % kWave, w = tid / kWave;
    const float* z = logits + static_cast<long long>(row) * V;
    f4u v[NV];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = 4 * (tid + THREADS * i);
        if (c + 3 < V) {
            v[i] = *reinterpret_cast<const f4u*>(z + c);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = c + e < V ? z[c + e] : -INFINITY;
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, v[i][e]);
    mx = wave_max(mx);
    if (lane == 0) red[0][w] = mx;
    __syncthreads();
    mx = red[0][0];
#pragma unroll
    for (int i = 1; i < THREADS / kWave; ++i) mx = fmaxf(mx, red[0][i]);
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[i][e] = expf(v[i][e] - mx);
            s += v[i][e];
        }
    s = wave_sum(s);
    if (lane == 0) red[1][w] = s;
    __syncthreads();
    s = 0.0f;
#pragma unroll
    for (int i = 0; i < THREADS / kWave; ++i) s += red[1][i];
    const float inv = 1.0f / s;
    const int tgt = targets[row];
    float* dz = dlogits + static_cast<long long>(row) * V;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = 4 * (tid + THREADS * i);
        f4u o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = (v[i][e] * inv - (c + e == tgt ? 1.0f : 0.0f)) * inv_rows;
        if (c + 3 < V) {
            *reinterpret_cast<f4u*>(dz + c) = o;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < V) dz[c + e] = o[e];
        }
    }
    if (tid == 0) row_loss[row] = mx + logf(s) - z[tgt];
}

// Rows that do not fit registers.
// One workgroup per row: loss_row = logsumexp(z) - z[target]; dz = (softmax(z) - onehot)
// * inv_rows.  Row losses are summed by a second pass (deterministic).
__global__ __launch_bounds__(kBlock) void cross_entropy_kernel(
    const float* __restrict__ logits, const int* __restrict__ targets,
    float* __restrict__ dlogits, float* __restrict__ row_loss, int V, float inv_rows) {
    __shared__ float red[kBlock / kWave];
    const int row = blockIdx.x;
    const int tid = threadIdx.x, lane = tid % kWave, w = tid / kWave;
    const float* z = logits + static_cast<long long>(row) * V;
    // one pass for the maximum and the sum of exponentials (a thread's running sum is
    // rescaled when its maximum grows), then the thread sums are brought to the row maximum
    float tm = -INFINITY, ts = 0.0f;
    for (int i = tid; i < V; i += kBlock) {
        const float zi = z[i];
        if (zi > tm) {
            ts = ts * expf(tm - zi) + 1.0f;
            tm = zi;
        } else {
            ts += expf(zi - tm);
        }
    }
    float mx = wave_max(tm);
    if (lane == 0) red[w] = mx;
    __syncthreads();
    mx = red[0];
    for (int i = 1; i < kBlock / kWave; ++i) mx = fmaxf(mx, red[i]);
    __syncthreads();
    float s = tm == -INFINITY ? 0.0f : ts * expf(tm - mx);
    s = wave_sum(s);
    if (lane == 0) red[w] = s;
    __syncthreads();
    s = 0.0f;
    for (int i = 0; i < kBlock / kWave; ++i) s += red[i];
    const float lse = mx + logf(s);
    const int tgt = targets[row];
    float* dz = dlogits + static_cast<long long>(row) * V;
    for (int i = tid; i < V; i += kBlock) {
        const float p = expf(z[i] - lse);
        dz[i] = (p - (i == tgt ? 1.0f : 0.0f)) * inv_rows;
    }
    if (tid == 0) row_loss[row] = lse - z[tgt];
}

__global__ void mean_kernel(const float* __restrict__ x, int n, float* __restrict__ out) {
    __shared__ float red[kBlock / kWave];
    float s = 0.0f;
    for (int i = threadIdx.x; i < n; i += kBlock) s += x[i];
    s = wave_sum(s);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int i = 0; i < kBlock / kWave; ++i) t += red[i];
        *out = t / n;
    }
}

// ---- gradient norm + AdamW ------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void sumsq_partial_kernel(const float* __restrict__ g,
                                                               long long n,
                                                               float* __restrict__ partial) {
    __shared__ float red[kBlock / kWave];
    float s = 0.0f;
    for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < n;
         i += static_cast<long long>(gridDim.x) * kBlock)
        s = fmaf(g[i], g[i], s);
    s = wave_sum(s);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int i = 0; i < kBlock / kWave; ++i) t += red[i];
        partial[blockIdx.x] = t;
    }
}

__global__ void norm_final_kernel(const float* __restrict__ partial, int n,
                                  float* __restrict__ norm) {
    __shared__ float red[kBlock / kWave];
    float s = 0.0f;
    for (int i = threadIdx.x; i < n; i += kBlock) s += partial[i];
    s = wave_sum(s);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int i = 0; i < kBlock / kWave; ++i) t += red[i];
        *norm = sqrtf(t);
    }
}

__global__ void adamw_kernel(float* __restrict__ p, float* __restrict__ g, float* __restrict__ m,
                             float* __restrict__ v, const float* __restrict__ norm, long long n,
                             AdamWParams a) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float nrm = *norm;
    float gi = g[i];
    if (nrm > a.max_norm && nrm > 1e-6f) gi *= a.max_norm / nrm;
    const float mt = a.beta1 * m[i] + (1.0f - a.beta1) * gi;
    const float vt = a.beta2 * v[i] + (1.0f - a.beta2) * gi * gi;
    m[i] = mt;
    v[i] = vt;
    const float mh = mt / a.bc1, vh = vt / a.bc2;
    const float pi = p[i];
    p[i] = pi - a.lr * (mh / (sqrtf(vh) + a.eps) + a.weight_decay * pi);
    g[i] = 0.0f;
}

}  // namespace

void embedding_forward(const int* tokens, const float* tok_emb, const float* pos_emb, float* out,
                       int B, int T, int C, hipStream_t s) {
    const long long n = static_cast<long long>(B) * T * C;
    hipLaunchKernelGGL(embedding_fwd_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s,
                       tokens, tok_emb, pos_emb, out, B * T, T, C);
}

void embedding_backward(const int* tokens, const float* dx, float* d_tok_emb, float* d_pos_emb,
                        float* scratch, int B, int T, int C, hipStream_t s) {
    const long long n = static_cast<long long>(B) * T * C;
    hipLaunchKernelGGL(embedding_tok_bwd_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s,
                       tokens, dx, d_tok_emb, B * T, C);
    // d_pos_emb[t, c] = sum_b dx[b, t, c]: column sums of a (B, T*C) matrix
    column_sum(dx, B, T * C, d_pos_emb, scratch, s);
}

size_t column_sum_scratch(int R, int N) {
    return static_cast<size_t>((R + kChunkRows - 1) / kChunkRows) * N;
}

void column_sum(const float* x, int R, int N, float* out, float* scratch, hipStream_t s) {
    const int nchunk = (R + kChunkRows - 1) / kChunkRows;
    hipLaunchKernelGGL(colsum_partial_kernel, dim3(blocks_for(N, kColTile), nchunk),
                       dim3(kBlock), 0, s, x, R, N, nullptr, nullptr, nullptr, scratch);
    hipLaunchKernelGGL(colsum_final_kernel, dim3(blocks_for(N, kFinCols)), dim3(kBlock), 0, s,
                       scratch, nchunk, N, out);
}

void sum_slices(const float* x, int nslice, long long n, float* out, hipStream_t s) {
    if (n % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0)
        hipLaunchKernelGGL(slice_sum_kernel<4>, dim3(blocks_for(n, 4 * kBlock)), dim3(kBlock), 0,
                           s, x, nslice, n, out);
    else
        hipLaunchKernelGGL(slice_sum_kernel<1>, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s,
                           x, nslice, n, out);
}

// Groups of 4 x 64 columns that a row kernel holds: 0 where the row does not fit.
int ln_groups(int C) { return C % 4 == 0 && C <= 2048 ? (C + 255) / 256 : 0; }
// Workgroups of layernorm_bwd_row_kernel: two of its waves per SIMD.
int ln_bwd_blocks(int R) {
    return static_cast<int>(std::min<long long>((R + kRowsPerBlock - 1) / kRowsPerBlock, 512));
}

#define LN_DISPATCH(groups, LAUNCH)      \
    switch (groups) {                    \
        case 1: LAUNCH(1); break;        \
        case 2: LAUNCH(2); break;        \
        case 3: LAUNCH(3); break;        \
        case 4: LAUNCH(4); break;        \
        case 5:                          \
        case 6: LAUNCH(6); break;        \
        default: LAUNCH(8); break;       \
    }

void layernorm_forward(const float* x, const float* gamma, const float* beta, float* y,
                       float* mean, float* rstd, int R, int C, float eps, hipStream_t s) {
    const dim3 grid(blocks_for(R, kRowsPerBlock));
    const int groups = aligned16(gamma) && aligned16(beta) ? ln_groups(C) : 0;
    if (groups == 0) {
        hipLaunchKernelGGL(layernorm_fwd_kernel, grid, dim3(kBlock), 0, s, x, gamma, beta, y, mean,
                           rstd, R, C, eps);
        return;
    }
#define LN_FWD(NV)                                                                             \
    hipLaunchKernelGGL((layernorm_fwd_row_kernel<4, NV>), grid, dim3(kBlock), 0, s, x, gamma, \
                       beta, y, mean, rstd, R, C, eps)
    LN_DISPATCH(groups, LN_FWD)
#undef LN_FWD
}

size_t layernorm_backward_scratch(int R, int C) {
    return std::max(column_sum_scratch(R, C), static_cast<size_t>(ln_bwd_blocks(R)) * 2 * C);
}

void layernorm_backward(const float* dy, const float* x, const float* gamma, const float* mean,
                        const float* rstd, float* dx, float* dgamma_dbeta, float* scratch, int R,
                        int C, bool accumulate, hipStream_t s) {
    const int acc = accumulate ? 1 : 0;
    const int groups = aligned16(gamma) ? ln_groups(C) : 0;
    if (groups == 0) {
        hipLaunchKernelGGL(layernorm_bwd_kernel, dim3(blocks_for(R, kRowsPerBlock)), dim3(kBlock),
                           0, s, dy, x, gamma, mean, rstd, dx, R, C, acc);
        const int nchunk = (R + kChunkRows - 1) / kChunkRows;
        hipLaunchKernelGGL(colsum_partial_kernel, dim3(blocks_for(C, kColTile), nchunk),
                           dim3(kBlock), 0, s, dy, R, C, x, mean, rstd, scratch);
        hipLaunchKernelGGL(colsum_final_kernel, dim3(blocks_for(C, kFinCols)), dim3(kBlock), 0, s,
                           scratch, nchunk, C, dgamma_dbeta);
        column_sum(dy, R, C, dgamma_dbeta + C, scratch, s);
        return;
    }
    const int blocks = ln_bwd_blocks(R);
#define LN_BWD(NV)                                                                               \
    hipLaunchKernelGGL((layernorm_bwd_row_kernel<4, NV>), dim3(blocks), dim3(kBlock), 0, s, dy, \
                       x, gamma, mean, rstd, dx, scratch, R, C, acc)
    LN_DISPATCH(groups, LN_BWD)
#undef LN_BWD
    hipLaunchKernelGGL(colsum_final_kernel, dim3(blocks_for(2 * C, kFinCols)), dim3(kBlock), 0, s,
                       scratch, blocks, 2 * C, dgamma_dbeta);
}

void cross_entropy(const float* logits, const int* targets, float* dlogits, float* row_loss,
                   float* loss, int rows, int V, hipStream_t s) {
    const float inv_rows = 1.0f / static_cast<float>(rows);
    // the smallest register footprint that holds the row; 256 threads up to 16384 logits, beyond
    // that the 1024 that a row's loads need in flight.  16 groups are over the registers of 1024
    // threads: rows of 33000, 45000 and 53000 take 341, 420 and 477 us with them (4096 rows), 247,
    // 291 and 344 with 13
#define CE_ROW(THREADS, NV)                                                                    \
    hipLaunchKernelGGL((cross_entropy_row_kernel<THREADS, NV>), dim3(rows), dim3(THREADS), 0, s, \
                       logits, targets, dlogits, row_loss, V, inv_rows)
    if (V <= 1024) CE_ROW(256, 1);
    else if (V <= 4096) CE_ROW(256, 4);
    else if (V <= 8192) CE_ROW(256, 8);
    else if (V <= 16384) CE_ROW(256, 16);
    else if (V <= 32768) CE_ROW(1024, 8);
    else if (V <= 53248) CE_ROW(1024, 13);
    else if (V <= 65536) CE_ROW(1024, 16);
    else
        hipLaunchKernelGGL(cross_entropy_kernel, dim3(rows), dim3(kBlock), 0, s, logits, targets,
                           dlogits, row_loss, V, inv_rows);
#undef CE_ROW
    hipLaunchKernelGGL(mean_kernel, dim3(1), dim3(kBlock), 0, s, row_loss, rows, loss);
}

int adamw_norm_blocks() { return 1024; }

void clip_adamw_zero(float* params, float* grads, float* m, float* v, float* norm_scratch,
                     long long n, const AdamWParams& a, hipStream_t s) {
    const int nb = adamw_norm_blocks();
    hipLaunchKernelGGL(sumsq_partial_kernel, dim3(nb), dim3(kBlock), 0, s, grads, n,
                       norm_scratch + 1);
    hipLaunchKernelGGL(norm_final_kernel, dim3(1), dim3(kBlock), 0, s, norm_scratch + 1, nb,
                       norm_scratch);
    hipLaunchKernelGGL(adamw_kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, s, params,
                       grads, m, v, norm_scratch, n, a);
}

}  // namespace gpt
}  // namespace tcamd
