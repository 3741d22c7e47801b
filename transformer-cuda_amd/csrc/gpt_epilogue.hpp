// gpt_epilogue.hpp - what the training-step harness's products do with their sums, and the
// launch that chooses their tiles and slices (gpt_gemm.hpp).
#pragma once

#include "gemm_planes.hpp"
#include "gpt_kernels.hpp"

namespace tcamd {
namespace gpt {

using namespace gemm;

// gelu_tanh(x) = x s and its derivative s + 2 x s (1 - s) u', with s = 1 / (1 + exp(-2 u)) =
// (1 + tanh u) / 2, u = c (x + a x^3): one exponential and one reciprocal, and no cancellation
// of 1 + tanh u for negative x.
constexpr float kGeluC = 0.7978845608028654f;  // sqrt(2/pi)
constexpr float kGeluA = 0.044715f;
__device__ __forceinline__ float gelu_s(float x) {
    const float u = kGeluC * (x + kGeluA * x * x * x);
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.8853900817779268f * u));
}
__device__ __forceinline__ float gelu(float x) { return x * gelu_s(x); }
__device__ __forceinline__ float gelu_grad(float x) {
    const float s = gelu_s(x);
    return s + 2.0f * x * s * (1.0f - s) * (kGeluC * (1.0f + 3.0f * kGeluA * x * x));
}

// Element-wise epilogues of one product: Map turns the sum at flat index i, column col into the
// outputs.  pair: two columns per access where every buffer's rows are 8-byte aligned.
template <class Map>
struct EpiMap : Map {
    static constexpr bool kColumnSums = false;
    int pair;
    __device__ __forceinline__ void store1(long long, int row, int col, int, int N,
                                           float x) const {
        const size_t i = static_cast<size_t>(row) * N + col;
        float y[1] = {x};
        this->template apply<1>(i, col, y);
    }
    template <int J>
    __device__ __forceinline__ void store(long long b, int row, int col, int M, int N,
                                          const float (&x)[J]) const {
        if (J == 2 && pair) {
            if (col >= N) return;
            float y[2] = {x[0], x[J - 1]};
            this->template apply<2>(static_cast<size_t>(row) * N + col, col, y);
        } else {
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (col + j < N) store1(b, row, col + j, M, N, x[j]);
        }
    }
};

template <int J>
__device__ __forceinline__ void put(float* p, const float (&x)[J]) {
    if constexpr (J == 2) *reinterpret_cast<f32x2*>(p) = f32x2{x[0], x[1]};
    else *p = x[0];
}
template <int J>
__device__ __forceinline__ void get(const float* p, float (&x)[J]) {
    if constexpr (J == 2) {
        const f32x2 v = *reinterpret_cast<const f32x2*>(p);
        x[0] = v[0];
        x[1] = v[1];
    } else {
        x[0] = *p;
    }
}

struct MapBias {
    static constexpr int kArrays = 1;
    float* C;
    const float* bias;
    template <int J>
    __device__ __forceinline__ void apply(size_t i, int col, float (&x)[J]) const {
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] += bias[col + j];
        put<J>(C + i, x);
    }
};
struct MapBiasResidual {
    static constexpr int kArrays = 2;
    float* C;
    const float *bias, *residual;
    template <int J>
    __device__ __forceinline__ void apply(size_t i, int col, float (&x)[J]) const {
        float r[J];
        get<J>(residual + i, r);
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = r[j] + x[j] + bias[col + j];
        put<J>(C + i, x);
    }
};
struct MapBiasGelu {
    static constexpr int kArrays = 2;
    float *pre, *C;
    const float* bias;
    template <int J>
    __device__ __forceinline__ void apply(size_t i, int col, float (&x)[J]) const {
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] += bias[col + j];
        put<J>(pre + i, x);
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] = gelu(x[j]);
        put<J>(C + i, x);
    }
};
struct MapGeluBackward {
    static constexpr int kArrays = 2;
    float* C;
    const float* pre;
    template <int J>
    __device__ __forceinline__ void apply(size_t i, int, float (&x)[J]) const {
        float y[J];
        get<J>(pre + i, y);
#pragma unroll
        for (int j = 0; j < J; ++j) x[j] *= gelu_grad(y[j]);
        put<J>(C + i, x);
    }
};

// C and, as its row M, the column sums of op(B); slices `stride` floats apart.
struct EpiGradient : EpiAxpby {
    static constexpr bool kColumnSums = true;
    __device__ __forceinline__ void column_sum(long long batch, int col, int M, int N,
                                               float x) const {
        C[batch * sC + static_cast<size_t>(M) * N + col] = x;
    }
};

// Slices of K: at GPT-2 small the weight gradients (K = 8192 tokens, 36 tiles of 256 x 256 for
// the feed-forward ones) and the head's input gradient (K = 50257, 96 tiles) leave most CUs idle
// without them; with B*T = 256 every product does.  More than 16 slices of such outputs would
// cost more in partial sums than they fill.
constexpr int kMaxSlices = 16;
constexpr long long kMaxPartials = 1LL << 28;  // floats of partial results (1 GiB)

inline Plan plan(int M, int N, int K, int arrays = 1) {
    const long long out = (static_cast<long long>(M) + 1) * N;
    const long long most = kMaxPartials / out;
    const int slices = static_cast<int>(most < 1 ? 1 : most > kMaxSlices ? kMaxSlices : most);
    return pick_tile(M, N, 1, K, slices, arrays);
}

// The sums over the slices, in order, through a product's epilogue: a thread per J columns.
template <int J, class Epi>
__global__ __launch_bounds__(256) void slices_epilogue_kernel(const float* __restrict__ x,
                                                              int nslice, int M, int N, Epi epi) {
    const unsigned i = (blockIdx.x * 256u + threadIdx.x) * J;  // < 2^28: kMaxPartials
    const unsigned n = static_cast<unsigned>(M) * N;
    if (i >= n) return;
    float s[J] = {};
#pragma unroll 4
    for (int z = 0; z < nslice; ++z) {
        float v[J];
        get<J>(x + static_cast<size_t>(z) * n + i, v);
#pragma unroll
        for (int j = 0; j < J; ++j) s[j] += v[j];
    }
    const int row = static_cast<int>(i / N);
    epi.template store<J>(0, row, static_cast<int>(i - static_cast<unsigned>(row) * N), M, N, s);
}

inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; }

inline EpiAxpby plain(float* C, int N, long long sC) {
    return EpiAxpby{C, sC, 1.0f, 0.0f, N % 2 == 0 && sC % 2 == 0 && aligned8(C)};
}

// One product through Map; aligned: all of Map's row buffers start 8-byte aligned.
template <bool TA, bool TB, class Map>
void product_map(int M, int N, int K, const float* A, const float* B, const Map& map,
                 bool aligned, float* scratch, hipStream_t s) {
    const Plan p = plan(M, N, K, Map::kArrays);
    const Problem g{A, B, M, N, K, 0, 0, kGemmFull, p.kslice, 0, 0, 0, 0};
    const EpiMap<Map> epi{map, N % 2 == 0 && aligned};
    if (p.slices == 1) {
        launch_tile<TA, TB>(p.tile, g, 1, epi, s);
        return;
    }
    const long long mn = static_cast<long long>(M) * N;
    launch_tile<TA, TB>(p.tile, g, p.slices, plain(scratch, N, mn), s);
    if (epi.pair)
        hipLaunchKernelGGL((slices_epilogue_kernel<2, EpiMap<Map>>),
                           dim3(static_cast<unsigned>((mn + 511) / 512)), dim3(256), 0, s, scratch,
                           p.slices, M, N, epi);
    else
        hipLaunchKernelGGL((slices_epilogue_kernel<1, EpiMap<Map>>),
                           dim3(static_cast<unsigned>((mn + 255) / 256)), dim3(256), 0, s, scratch,
                           p.slices, M, N, epi);
}

// One product as it is.
template <bool TA, bool TB>
void product_plain(int M, int N, int K, const float* A, const float* B, float* C, float* scratch,
                   hipStream_t s) {
    const Plan p = plan(M, N, K);
    const Problem g{A, B, M, N, K, 0, 0, kGemmFull, p.kslice, 0, 0, 0, 0};
    const long long mn = static_cast<long long>(M) * N;
    launch_tile<TA, TB>(p.tile, g, p.slices, plain(p.slices > 1 ? scratch : C, N, mn), s);
    if (p.slices > 1) sum_slices(scratch, p.slices, mn, C, s);
}

}  // namespace gpt
}  // namespace tcamd
