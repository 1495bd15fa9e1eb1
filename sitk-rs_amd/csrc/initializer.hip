// The learned initializer: a small 3-D CNN that predicts an affine start for
// the registration from a downsampled image pair, trained and run by this
// library's own kernels. No counterpart in the reference, whose initializers
// are geometric (src/registration/initializer.rs: CenteredTransformInitializer).
//
// Network (input 64^3 x 2 channels, fixed and moving, z-scored, BF16):
//   conv1  2 -> 16, 3^3, stride 1, ReLU        64^3
//   conv2 16 -> 32, 3^3, stride 2, ReLU        32^3
//   conv3 32 -> 64, 3^3, stride 2, ReLU        16^3
//   conv4 64 -> 64, 3^3, stride 2, ReLU         8^3
//   conv5 64 ->128, 3^3, stride 2, ReLU         4^3
//   global average pool -> 128
//   fc1 128 -> 128, ReLU ; fc2 128 -> 12
// Zero 'same' padding. Outputs: the 9 entries of (A - I) and t / 10 mm of the
// affine x -> A (x - c) + t + c about the fixed image's centre c.
//
// Layout: activations channels-last [n][z][y][x][c] in BF16 (the input's two
// channels as one 4-byte word per voxel); conv weights [co][tap][ci] (tap =
// kz*9 + ky*3 + kx, the first layer's ci padded to 8 in the parameter vector).
// The convolutions' kernels are in conv3.hpp. The weight gradient is split
// over the output positions into fixed partial rows that a second kernel adds
// in a fixed order, so training is deterministic. Master weights, their
// gradients and Adam's moments are FP32; the MLP head (0.01% of the FLOPs) runs
// in FP32 on the vector units.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "common.hpp"
#include "conv3.hpp"
#include "image.hpp"
#include "metric.hpp"

namespace sitkhip {
namespace cnn {

constexpr int kLayers = 5;
constexpr int kEdge = 64;          // input edge
constexpr int kCin0 = 8;           // input channels of the parameter layout (2 used)
constexpr int kCin0Used = 2;       // input channels held in memory
constexpr int kFeat = 128;         // GAP features
constexpr int kHidden = 128;
constexpr int kOut = 12;
constexpr int kCh[kLayers + 1] = {kCin0, 16, 32, 64, 64, 128};
constexpr int kStride[kLayers] = {1, 2, 2, 2, 2};

// ------------------------------------------------------------------ BF16
__host__ __device__ inline uint16_t f2bf(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN
    u += 0x7fffu + ((u >> 16) & 1u);                       // round to nearest even
    return static_cast<uint16_t>(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t h) {
    const uint32_t u = static_cast<uint32_t>(h) << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// ------------------------------------------------------- small kernels
// Global average pool of the last conv output [n][64][128] and the MLP head,
// one workgroup per sample: lane t of 128 sums channel t's positions, then row t
// of W1, then (t < 12) row t of W2, each in order: the sums decide the rounding
// of the gradients' BF16 values, see conv_wgrad. All 256 lanes load W1, in whole
// rows, and half of its columns at a time goes to LDS.
constexpr int kHeadCols = kFeat / 2;
__global__ __launch_bounds__(256) void head_forward(const uint16_t *__restrict__ y,
                                                    const float *__restrict__ w1,
                                                    const float *__restrict__ b1,
                                                    const float *__restrict__ w2,
                                                    const float *__restrict__ b2,
                                                    float *__restrict__ feat, float *__restrict__ hid,
                                                    float *__restrict__ out) {
    __shared__ float f[kFeat], hh[kHidden], sw1[kHidden][kHeadCols + 1], sw2[kOut][kHidden + 1];
    const int b = blockIdx.x, t = threadIdx.x;
    float s = 0.0f;
    if (t < kFeat) {
        uint16_t v[64];
#pragma unroll
        for (int p = 0; p < 64; ++p) v[p] = y[(static_cast<size_t>(b) * 64 + p) * kFeat + t];
#pragma unroll
        for (int p = 0; p < 64; ++p) s += bf2f(v[p]);
        s *= 1.0f / 64.0f;
        f[t] = s;
        feat[b * kFeat + t] = s;
        s = b1[t];
    }
    for (int i = t; i < kOut * kHidden; i += 256) sw2[i / kHidden][i % kHidden] = w2[i];
    constexpr int kQuads = kHidden * kHeadCols / 4 / 256;  // per lane and half
    float4 w[2][kQuads];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int k = 0; k < kQuads; ++k) {
            const int i = t + 256 * k, row = i / (kHeadCols / 4), col = i % (kHeadCols / 4);
            w[h][k] = reinterpret_cast<const float4 *>(w1 + row * kFeat + h * kHeadCols)[col];
        }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kQuads; ++k) {
            const int i = t + 256 * k, row = i / (kHeadCols / 4), col = i % (kHeadCols / 4) * 4;
            sw1[row][col] = w[h][k].x;
            sw1[row][col + 1] = w[h][k].y;
            sw1[row][col + 2] = w[h][k].z;
            sw1[row][col + 3] = w[h][k].w;
        }
        __syncthreads();
        if (t < kHidden)
#pragma unroll 32
            for (int i = 0; i < kHeadCols; ++i) s += sw1[t][i] * f[h * kHeadCols + i];
    }
    if (t < kHidden) {
        s = fmaxf(s, 0.0f);
        hh[t] = s;
        hid[b * kHidden + t] = s;
    }
    __syncthreads();
    if (t < kOut) {
        float o = b2[t];
#pragma unroll 32
        for (int j = 0; j < kHidden; ++j) o += sw2[t][j] * hh[j];
        out[b * kOut + t] = o;
    }
}

// MLP head backward, per sample (one workgroup of 256 lanes): the hidden
// gradient dhid = relu'(hid) * W2' dout, the pooled features' dfeat = W1' dhid
// (128 lanes each, in order), and through the pool and the last convolution's
// ReLU the gradient of its 64 output positions.
__global__ __launch_bounds__(256) void head_backward_samples(
    const float *__restrict__ hid, const float *__restrict__ dout, const float *__restrict__ w1,
    const float *__restrict__ w2, const uint16_t *__restrict__ y, float *__restrict__ dhid,
    uint16_t *__restrict__ dy) {
    __shared__ float dh[kHidden];
    __shared__ uint16_t grad[kFeat];
    const int b = blockIdx.x, t = threadIdx.x & 127, h = threadIdx.x >> 7;
    if (h == 0) {
        float s = 0.0f;
#pragma unroll
        for (int o = 0; o < kOut; ++o) s += w2[o * kHidden + t] * dout[b * kOut + o];
        s = hid[b * kHidden + t] > 0.0f ? s : 0.0f;
        dh[t] = s;
        dhid[b * kHidden + t] = s;
    }
    __syncthreads();
    if (h == 0) {
        float s = 0.0f;
#pragma unroll 32
        for (int j = 0; j < kHidden; ++j) s += w1[j * kFeat + t] * dh[j];
        grad[t] = f2bf(s * (1.0f / 64.0f));
    }
    __syncthreads();
    const uint16_t g = grad[t];
#pragma unroll 8
    for (int p = h; p < 64; p += 2) {
        const size_t i = (static_cast<size_t>(b) * 64 + p) * kFeat + t;
        dy[i] = bf2f(y[i]) > 0.0f ? g : 0;
    }
}

// The head's weight gradients, sums over the batch in order: workgroup r <
// 128 takes row r of W1 (and b1[r]), workgroup 128 + o row o of W2 (and b2[o]).
// (One workgroup for the whole head, looping over samples and rows, took
// 363 us for 24 samples; the two kernels take 10.)
__global__ __launch_bounds__(128) void head_backward_weights(
    int n, const float *__restrict__ feat, const float *__restrict__ hid,
    const float *__restrict__ dout, const float *__restrict__ dhid, float *__restrict__ gw1,
    float *__restrict__ gb1, float *__restrict__ gw2, float *__restrict__ gb2) {
    const int t = threadIdx.x;
    const bool first = blockIdx.x < kHidden;
    const int r = first ? blockIdx.x : blockIdx.x - kHidden;
    const float *row = first ? dhid + r : dout + r;
    const float *col = first ? feat : hid;
    const int ld = first ? kHidden : kOut;
    float s = 0.0f, sb = 0.0f;
#pragma unroll 8
    for (int b = 0; b < n; ++b) {
        const float d = row[b * ld];
        s += d * col[b * kFeat + t];
        sb += d;
    }
    (first ? gw1 : gw2)[r * kFeat + t] = s;
    if (t == 0) (first ? gb1 : gb2)[r] = sb;
}
static_assert(kFeat == kHidden && kFeat == 128, "the head's kernels share their lane layout");

// Adam (Kingma & Ba 2015) on the flat FP32 parameters.
__global__ void adam_step(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                          float *__restrict__ v, size_t n, float lr, float b1, float b2, float eps,
                          float c1, float c2) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// BF16 copies of the conv layers' weights, all layers in one launch: w
// [co][27][ci] and, for the input gradient, transposed [ci][27][co].
struct CastLayer {
    const float *w;
    uint16_t *wb, *wt;
    int co, ci, begin;  // begin: the layer's first index over all layers
};
struct CastLayers {
    CastLayer l[kLayers];
    int total;
};
__global__ __launch_bounds__(256) void cast_weights(CastLayers L) {
    const int at = blockIdx.x * 256 + threadIdx.x;
    if (at >= L.total) return;
    int k = 0;
    while (k + 1 < kLayers && at >= L.l[k + 1].begin) ++k;
    const CastLayer &q = L.l[k];
    const int i = at - q.begin;
    const int c = i % q.ci, tap = (i / q.ci) % 27, o = i / (27 * q.ci);
    const uint16_t h = f2bf(q.w[i]);
    q.wb[i] = h;
    q.wt[(static_cast<size_t>(c) * 27 + tap) * q.co + o] = h;
}

// The 64^3 input volumes are read four voxels per lane.
constexpr int kVol = kEdge * kEdge * kEdge;
constexpr int kVolBlocks = kVol / (256 * 4);

// Sums over the 64 lanes of a wave in a fixed order, in every lane.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum and sum of squares of 1,024 voxels of volume blockIdx.y (FP64):
// part[(volume * kVolBlocks + block) * 2 ..].
__global__ __launch_bounds__(256) void moments_partials(const float *__restrict__ v,
                                                        double *__restrict__ part) {
    __shared__ double s[4][2];
    const float4 q = reinterpret_cast<const float4 *>(
        v + static_cast<size_t>(blockIdx.y) * kVol)[blockIdx.x * 256 + threadIdx.x];
    const double x[4] = {q.x, q.y, q.z, q.w};
    double a = 0.0, b = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a += x[k];
        b += x[k] * x[k];
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if ((threadIdx.x & 63) == 0) {
        s[threadIdx.x >> 6][0] = a;
        s[threadIdx.x >> 6][1] = b;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        part[(static_cast<size_t>(blockIdx.y) * kVolBlocks + blockIdx.x) * 2 + threadIdx.x] =
            (s[0][threadIdx.x] + s[1][threadIdx.x]) + (s[2][threadIdx.x] + s[3][threadIdx.x]);
}

// Volume blockIdx.x's normalisation from its partial sums (one wave, a fixed
// order): norm[2 b ..] = {mean, 1 / std} as floats.
__global__ __launch_bounds__(64) void moments_finish(const double *__restrict__ part,
                                                     float *__restrict__ norm) {
    part += static_cast<size_t>(blockIdx.x) * kVolBlocks * 2;
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int b = threadIdx.x; b < kVolBlocks; b += 64) {
        s1 += part[2 * b];
        s2 += part[2 * b + 1];
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    if (threadIdx.x == 0) {
        const double mean = s1 / kVol;
        const double var = fmax(s2 / kVol - mean * mean, 1e-12);
        norm[2 * blockIdx.x] = static_cast<float>(mean);
        norm[2 * blockIdx.x + 1] = static_cast<float>(1.0 / sqrt(var));
    }
}

// Slots first .. first + gridDim.y - 1 from their two volumes (fixed, moving:
// volumes 2b and 2b + 1 of `v`, normalisations 4b .. 4b + 3): voxel i of
// slot b is {(f - mean_f) / std_f, (m - mean_m) / std_m} as BF16, one word.
__global__ __launch_bounds__(256) void pack_slots(const float *__restrict__ v,
                                                  const float *__restrict__ norm,
                                                  uint32_t *__restrict__ slots) {
    const int b = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    const float4 *src = reinterpret_cast<const float4 *>(v + static_cast<size_t>(2 * b) * kVol);
    const float4 f = src[i], m = src[i + kVol / 4];
    const float *q = norm + 4 * b;
    auto word = [&](float x, float y) {
        return static_cast<uint32_t>(f2bf((x - q[0]) * q[1])) |
               (static_cast<uint32_t>(f2bf((y - q[2]) * q[3])) << 16);
    };
    reinterpret_cast<uint4 *>(slots + static_cast<size_t>(b) * kVol)[i] =
        make_uint4(word(f.x, m.x), word(f.y, m.y), word(f.z, m.z), word(f.w, m.w));
}

// --------------------------------------------------------------- the net
struct Net {
    int max_batch = 0;
    // parameter offsets (floats) in the flat buffers
    size_t off_w[kLayers], off_b[kLayers], off_w1, off_b1, off_w2, off_b2, nparams;
    DeviceBuffer<float> params, grads, adam_m, adam_v;
    long long adam_t = 0;
    DeviceBuffer<uint16_t> wb[kLayers], wt[kLayers];
    DeviceBuffer<uint16_t> act[kLayers + 1];   // act[0] = input slots (2 channels), act[l+1] = conv l output
    DeviceBuffer<uint16_t> dact[kLayers + 1];  // gradients w.r.t. act (masked); none for the input
    DeviceBuffer<float> partials;              // weight-gradient rows of every layer
    DeviceBuffer<float> bias_partials;         // [kBiasSplits][channels] of every layer
    size_t off_partial[kLayers], off_bias_partial[kLayers];
    DeviceBuffer<float> feat, hid, out, dout, dhid;
    bool weights_dirty = true;
};

static int out_edge(int layer) {  // edge of conv `layer`'s output (layer 0..4)
    int e = kEdge;
    for (int l = 0; l <= layer; ++l) e /= kStride[l];
    return e;
}
static size_t act_elems(int idx, int n) {  // idx 0 = input, idx l+1 = conv l output
    const int e = idx == 0 ? kEdge : out_edge(idx - 1);
    const int c = idx == 0 ? kCin0Used : kCh[idx];
    return static_cast<size_t>(n) * e * e * e * c;
}

// How a layer's output positions are split for the weight gradient: one part per
// 4,096 of them, at most 256, each a whole number of 32-position steps. Part of
// the order of a gradient's sums (conv_wgrad), so nothing else decides it.
struct WgradSplit {
    int positions, per, rows;
};
static WgradSplit wgrad_split(int layer, int n) {
    WgradSplit s;
    const int e = out_edge(layer);
    s.positions = n * e * e * e;
    const int want = std::min(256, std::max(1, s.positions / 4096));
    s.per = ((s.positions + want - 1) / want + 31) / 32 * 32;
    s.rows = (s.positions + s.per - 1) / s.per;
    return s;
}
// The most rows that batches up to n have.
static int wgrad_max_rows(int layer, int n) {
    const int e = out_edge(layer);
    return std::min(256, std::max(1, n * e * e * e / 4096));
}
static int wgrad_row_len(int layer) {
    return kCh[layer + 1] * 27 * (layer == 0 ? kCin0Used : kCh[layer]);
}

static void init_params(Net &net, uint64_t seed) {
    std::vector<float> h(net.nparams, 0.0f);
    uint64_t s = seed;
    auto next = [&]() {
        s += 0x9E3779B97F4A7C15ull;
        uint64_t z = s;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto normal = [&]() {
        const double u1 = (static_cast<double>(next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        const double u2 = (static_cast<double>(next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
    };
    for (int l = 0; l < kLayers; ++l) {
        const int ci = kCh[l], co = kCh[l + 1];
        const int ci_used = l == 0 ? 2 : ci;
        const double sd = std::sqrt(2.0 / (27.0 * ci_used));  // He initialisation
        for (int o = 0; o < co; ++o)
            for (int t = 0; t < 27; ++t)
                for (int c = 0; c < ci; ++c)
                    h[net.off_w[l] + (static_cast<size_t>(o) * 27 + t) * ci + c] =
                        c < ci_used ? static_cast<float>(sd * normal()) : 0.0f;
    }
    const double sd1 = std::sqrt(2.0 / kFeat), sd2 = std::sqrt(1.0 / kHidden) * 0.1;
    for (int i = 0; i < kHidden * kFeat; ++i) h[net.off_w1 + i] = static_cast<float>(sd1 * normal());
    for (int i = 0; i < kOut * kHidden; ++i) h[net.off_w2 + i] = static_cast<float>(sd2 * normal());
    net.params.upload(h.data(), h.size());
    sync();
    net.weights_dirty = true;
}

Net *create(int max_batch, uint64_t seed) {
    if (max_batch < 1 || max_batch > 256) fail(SITKHIP_ERR_INVALID_ARGUMENT, "batch must be 1..256");
    auto *net = new Net();
    try {
        net->max_batch = max_batch;
        size_t o = 0;
        for (int l = 0; l < kLayers; ++l) {
            net->off_w[l] = o;
            o += static_cast<size_t>(kCh[l + 1]) * 27 * kCh[l];
            net->off_b[l] = o;
            o += kCh[l + 1];
        }
        net->off_w1 = o; o += kHidden * kFeat;
        net->off_b1 = o; o += kHidden;
        net->off_w2 = o; o += kOut * kHidden;
        net->off_b2 = o; o += kOut;
        net->nparams = o;
        net->params.alloc(o);
        net->grads.alloc(o);
        net->adam_m.alloc(o);
        net->adam_v.alloc(o);
        HIP_OK(hipMemsetAsync(net->grads.ptr, 0, o * sizeof(float), backend().stream));
        HIP_OK(hipMemsetAsync(net->adam_m.ptr, 0, o * sizeof(float), backend().stream));
        HIP_OK(hipMemsetAsync(net->adam_v.ptr, 0, o * sizeof(float), backend().stream));
        for (int l = 0; l < kLayers; ++l) {
            const size_t n = static_cast<size_t>(kCh[l + 1]) * 27 * kCh[l];
            net->wb[l].alloc(n);
            net->wt[l].alloc(n);
        }
        for (int i = 0; i <= kLayers; ++i) {
            net->act[i].alloc(act_elems(i, max_batch));
            if (i > 0) net->dact[i].alloc(act_elems(i, max_batch));
        }
        HIP_OK(hipMemsetAsync(net->act[0].ptr, 0, net->act[0].bytes(), backend().stream));
        size_t partials = 0, bias_partials = 0;
        for (int l = 0; l < kLayers; ++l) {
            net->off_partial[l] = partials;
            partials += static_cast<size_t>(wgrad_max_rows(l, max_batch)) * wgrad_row_len(l);
            net->off_bias_partial[l] = bias_partials;
            bias_partials += static_cast<size_t>(kBiasSplits) * kCh[l + 1];
        }
        net->partials.alloc(partials);
        net->bias_partials.alloc(bias_partials);
        net->feat.alloc(static_cast<size_t>(max_batch) * kFeat);
        net->hid.alloc(static_cast<size_t>(max_batch) * kHidden);
        net->out.alloc(static_cast<size_t>(max_batch) * kOut);
        net->dout.alloc(static_cast<size_t>(max_batch) * kOut);
        net->dhid.alloc(static_cast<size_t>(max_batch) * kHidden);
        init_params(*net, seed);
    } catch (...) {
        delete net;
        throw;
    }
    return net;
}

static void refresh_weights(Net &net) {
    if (!net.weights_dirty) return;
    CastLayers L;
    L.total = 0;
    for (int l = 0; l < kLayers; ++l) {
        L.l[l] = {net.params.ptr + net.off_w[l], net.wb[l].ptr, net.wt[l].ptr, kCh[l + 1], kCh[l], L.total};
        L.total += kCh[l + 1] * 27 * kCh[l];
    }
    launch_kernel("cnn_cast_weights", cast_weights, dim3((L.total + 255) / 256), dim3(256), 0, L);
    check_launch("cast_weights");
    net.weights_dirty = false;
}

static void check_batch(const Net &net, int n) {
    if (n < 1 || n > net.max_batch)
        fail(SITKHIP_ERR_INVALID_ARGUMENT, "batch must be 1.." + std::to_string(net.max_batch));
}

static const float *param(const Net &net, size_t off) { return net.params.ptr + off; }

static const uint32_t *input_words(const Net &net) {
    return reinterpret_cast<const uint32_t *>(net.act[0].ptr);
}

// Workgroups of a launch that walks `items`: `per_cu` on every CU, or one each.
static unsigned resident(int per_cu, int items) {
    return static_cast<unsigned>(std::max(1, std::min(items, per_cu * backend().cu_count)));
}

// A kernel with more than 64 KB of dynamic LDS has to be told so.
template <typename F>
static void allow_lds(F kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
}

template <int LGDO, int CI, int CO, int R, int COW, bool HOLD>
static void launch_forward(Net &net, int layer, int n, int per_cu = 0) {
    using T = InTile<LGDO, CI, R, 1, 3>;
    auto kernel = conv_forward<LGDO, CI, CO, R, COW, HOLD>;
    const int chunks = T::chunks(n);
    allow_lds(kernel, T::kBytes);
    launch_kernel("cnn_conv_fwd", kernel, dim3(HOLD ? resident(per_cu, chunks) : chunks, CO / COW), dim3(kConvLanes),
                  T::kBytes, static_cast<const uint16_t *>(net.act[layer].ptr),
                  static_cast<const uint16_t *>(net.wb[layer].ptr),
                  param(net, net.off_b[layer]), net.act[layer + 1].ptr,
                  chunks);
    check_launch("cnn_conv_fwd");
}

template <int LGDO, int CI, int CO, int QY, int QZ, int CG, bool HOLD>
static void launch_dgrad(Net &net, int layer, int n) {
    constexpr int DO = 1 << LGDO;
    constexpr size_t lds = static_cast<size_t>(QZ + 1) * (QY + 1) * (DO + 1) * (2 * CO + 16);
    static_assert(lds <= 64 * 1024, "the staged dy fits the default limit");
    const int tiles = n * (DO / QY) * (DO / QZ);
    launch_kernel("cnn_conv_dgrad", conv_dgrad<LGDO, CI, CO, QY, QZ, CG, HOLD>,
                  dim3(HOLD ? resident(2, tiles) : tiles, CG), dim3(kConvLanes), lds,
                  static_cast<const uint16_t *>(net.dact[layer + 1].ptr),
                  static_cast<const uint16_t *>(net.wt[layer].ptr),
                  static_cast<const uint16_t *>(net.act[layer].ptr), net.dact[layer].ptr, tiles);
    check_launch("cnn_conv_dgrad");
}

template <int LGDO, int CI, int CO, int R, int ZP, int KZN, int COW, int CG>
static void launch_wgrad(Net &net, int layer, int n) {
    using T = InTile<LGDO, CI, R, ZP, KZN * ZP>;
    constexpr size_t lds = T::kBytes + static_cast<size_t>(T::P) * (2 * COW + 16);
    const WgradSplit s = wgrad_split(layer, n);
    auto kernel = conv_wgrad<LGDO, CI, CO, R, ZP, KZN, COW, CG>;
    allow_lds(kernel, lds);
    launch_kernel("cnn_conv_wgrad", kernel, dim3(s.rows, CG * (3 / KZN) * (CO / COW)), dim3(kConvLanes), lds,
                  static_cast<const uint16_t *>(net.act[layer].ptr),
                  static_cast<const uint16_t *>(net.dact[layer + 1].ptr),
                  net.partials.ptr + net.off_partial[layer], s.per, s.positions);
    check_launch("cnn_conv_wgrad");
}

void forward(Net &net, int n, float *out_host) {
    check_batch(net, n);
    refresh_weights(net);
    {
        const int chunks = C0Tile<kF0Rows>::chunks(n);
        launch_kernel("cnn_conv0_fwd", conv0_forward, dim3(resident(8, chunks)), dim3(kConvLanes), 0,
                      input_words(net), static_cast<const uint16_t *>(net.wb[0].ptr), kCin0,
                      param(net, net.off_b[0]), net.act[1].ptr, chunks);
        check_launch("conv0_forward");
    }
    launch_forward<5, 16, 32, 2, 32, true>(net, 1, n, 3);
    launch_forward<4, 32, 64, 2, 64, true>(net, 2, n, 2);
    launch_forward<3, 64, 64, 4, 64, false>(net, 3, n);
    launch_forward<2, 64, 128, 4, 64, false>(net, 4, n);
    launch_kernel("cnn_head", head_forward, dim3(n), dim3(256), 0,
                  static_cast<const uint16_t *>(net.act[kLayers].ptr), param(net, net.off_w1),
                  param(net, net.off_b1), param(net, net.off_w2), param(net, net.off_b2), net.feat.ptr,
                  net.hid.ptr, net.out.ptr);
    check_launch("cnn_head");
    if (out_host) {
        net.out.download(out_host, static_cast<size_t>(n) * kOut);
    }
    sync();
}

// Backward from dL/dout (host, n x 12) after forward() of the same batch:
// every parameter gradient into net.grads.
void backward(Net &net, int n, const float *dout_host) {
    check_batch(net, n);
    net.dout.upload(dout_host, static_cast<size_t>(n) * kOut);
    launch_kernel("cnn_head_bwd", head_backward_samples, dim3(n), dim3(256), 0,
                  static_cast<const float *>(net.hid.ptr), static_cast<const float *>(net.dout.ptr),
                  param(net, net.off_w1), param(net, net.off_w2),
                  static_cast<const uint16_t *>(net.act[kLayers].ptr), net.dhid.ptr,
                  net.dact[kLayers].ptr);
    launch_kernel("cnn_head_bwd", head_backward_weights, dim3(kHidden + kOut), dim3(128), 0, n,
                  static_cast<const float *>(net.feat.ptr), static_cast<const float *>(net.hid.ptr),
                  static_cast<const float *>(net.dout.ptr), static_cast<const float *>(net.dhid.ptr),
                  net.grads.ptr + net.off_w1, net.grads.ptr + net.off_b1, net.grads.ptr + net.off_w2,
                  net.grads.ptr + net.off_b2);
    check_launch("cnn_head_bwd");
    launch_wgrad<2, 64, 128, 4, 4, 1, 16, 3>(net, 4, n);
    launch_dgrad<2, 64, 128, 4, 4, 4, false>(net, 4, n);
    launch_wgrad<3, 64, 64, 8, 2, 1, 16, 3>(net, 3, n);
    launch_dgrad<3, 64, 64, 8, 1, 4, false>(net, 3, n);
    launch_wgrad<4, 32, 64, 8, 1, 1, 32, 3>(net, 2, n);
    launch_dgrad<4, 32, 64, 8, 1, 1, false>(net, 2, n);
    launch_wgrad<5, 16, 32, 4, 1, 1, 32, 1>(net, 1, n);
    launch_dgrad<5, 16, 32, 4, 1, 1, true>(net, 1, n);
    const WgradSplit s0 = wgrad_split(0, n);
    if (s0.per % (kW0Rows * 64) != 0) fail(SITKHIP_ERR_DRIVER, "first-layer splits are not whole chunks");
    launch_kernel("cnn_conv_wgrad", conv0_wgrad, dim3(s0.rows), dim3(kW0Lanes), 0, input_words(net),
                  static_cast<const uint16_t *>(net.dact[1].ptr), net.partials.ptr + net.off_partial[0],
                  s0.per, s0.positions);
    check_launch("conv0_wgrad");
    BiasLayers bias;
    for (int l = 0; l < kLayers; ++l)
        bias.l[l] = {net.dact[l + 1].ptr, net.bias_partials.ptr + net.off_bias_partial[l],
                     wgrad_split(l, n).positions, kCh[l + 1]};
    launch_kernel("cnn_bias_grad", bias_grad, dim3(kBiasSplits, kLayers), dim3(kConvLanes), 0, bias);
    check_launch("bias_grad");
    PartialJobs jobs;
    jobs.n = 0;
    unsigned blocks = 0;
    auto add = [&](const float *p, float *out, int rows, int len, int inner, int ld) {
        jobs.j[jobs.n++] = {p, out, rows, len, inner, ld, blocks};
        blocks += static_cast<unsigned>((len + kPartialLanes - 1) / kPartialLanes);
    };
    for (int l = 0; l < kLayers; ++l) {
        const int len = wgrad_row_len(l);
        add(net.partials.ptr + net.off_partial[l], net.grads.ptr + net.off_w[l], wgrad_split(l, n).rows, len,
            l == 0 ? kCin0Used : len, l == 0 ? kCin0 : len);
        add(net.bias_partials.ptr + net.off_bias_partial[l], net.grads.ptr + net.off_b[l], kBiasSplits,
            kCh[l + 1], kCh[l + 1], kCh[l + 1]);
    }
    launch_kernel("cnn_sum_partials", reduce_partials, dim3(blocks), dim3(kPartialLanes), 0, jobs);
    check_launch("reduce_partials");
    sync();
}

void adam(Net &net, float lr, float b1, float b2, float eps) {
    ++net.adam_t;
    const float c1 = 1.0f - std::pow(b1, static_cast<float>(net.adam_t));
    const float c2 = 1.0f - std::pow(b2, static_cast<float>(net.adam_t));
    LaunchScope scope("cnn_adam");
    hipLaunchKernelGGL(adam_step, dim3(grid_for(net.nparams, 256, 1024)), dim3(256), 0,
                       backend().stream, net.params.ptr, net.grads.ptr, net.adam_m.ptr,
                       net.adam_v.ptr, net.nparams, lr, b1, b2, eps, c1, c2);
    check_launch("adam_step");
    net.weights_dirty = true;
    sync();
}

// Input slots first .. first + n - 1 from 2n 64^3 float volumes already on
// the device, consecutive: slot b's fixed volume is volume 2b, its moving
// volume 2b + 1. The normalisations are computed on the device (no host round
// trip), every volume's in one launch.
static void pack(Net &net, int first, int n, const float *vols) {
    if (first < 0 || n < 1 || first + n > net.max_batch)
        fail(SITKHIP_ERR_INVALID_ARGUMENT, "slot out of range");
    uint32_t *dst = reinterpret_cast<uint32_t *>(net.act[0].ptr) + static_cast<size_t>(first) * kVol;
    const unsigned nv = static_cast<unsigned>(2 * n);
    DeviceBuffer<double> part(static_cast<size_t>(nv) * kVolBlocks * 2);
    DeviceBuffer<float> norm(static_cast<size_t>(nv) * 2);
    launch_kernel("cnn_moments", moments_partials, dim3(kVolBlocks, nv), dim3(256), 0, vols, part.ptr);
    check_launch("moments_partials");
    launch_kernel("cnn_moments", moments_finish, dim3(nv), dim3(64), 0,
                  static_cast<const double *>(part.ptr), norm.ptr);
    check_launch("moments_finish");
    launch_kernel("cnn_pack", pack_slots, dim3(kVolBlocks, static_cast<unsigned>(n)), dim3(256), 0, vols,
                  static_cast<const float *>(norm.ptr), dst);
    check_launch("pack_slots");
}

// The 64^3 grid spanning an image's physical extent (same origin corner and
// direction, spacing size * spacing / 64): each output voxel is the linear
// interpolation at the centre of the input block it covers.
static sitkhip_geometry grid64(const sitkhip_geometry &g) {
    sitkhip_geometry o = g;
    for (int d = 0; d < 3; ++d) {
        o.size[d] = kEdge;
        o.spacing[d] = g.spacing[d] * static_cast<double>(g.size[d]) / kEdge;
    }
    // keep the physical box: origin moves by half the spacing change
    for (int r = 0; r < 3; ++r) {
        double acc = g.origin[r];
        for (int c = 0; c < 3; ++c) acc += g.direction[r * 3 + c] * 0.5 * (o.spacing[c] - g.spacing[c]);
        o.origin[r] = acc;
    }
    return o;
}

// Slots first .. first + n - 1 from n image pairs: every image linearly
// resampled (identity map) onto the 64^3 grid spanning its own extent -- all
// 2n placements in one launch -- then z-scored and packed.
void set_inputs(Net &net, int first, int n, const Image *const *fixed, const Image *const *moving) {
    if (first < 0 || n < 1 || first + n > net.max_batch)
        fail(SITKHIP_ERR_INVALID_ARGUMENT, "slot out of range");
    const size_t nv = static_cast<size_t>(kEdge) * kEdge * kEdge;
    DeviceBuffer<float> vols(static_cast<size_t>(2 * n) * nv);
    PrepBatch prep;
    for (int b = 0; b < n; ++b) {
        for (int ch = 0; ch < 2; ++ch) {
            const Image *im = ch ? moving[b] : fixed[b];
            if (!im) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image");
            const sitkhip_geometry og = grid64(im->geom);
            prep.places.push_back({im->buf.ptr, im->geom, vols.ptr + static_cast<size_t>(2 * b + ch) * nv, og});
        }
    }
    enqueue_placements(prep);
    pack(net, first, n, vols.ptr);
    sync();  // the placement descriptors' host copies live as long as `prep`
}

void set_input(Net &net, int slot, const Image &fixed, const Image &moving) {
    const Image *f = &fixed, *m = &moving;
    set_inputs(net, slot, 1, &f, &m);
}

void set_input_raw(Net &net, int slot, const float *fixed_host, const float *moving_host) {
    const size_t nv = static_cast<size_t>(kEdge) * kEdge * kEdge;
    DeviceBuffer<float> v(2 * nv);
    HIP_OK(hipMemcpyAsync(v.ptr, fixed_host, nv * sizeof(float), hipMemcpyHostToDevice, backend().stream));
    HIP_OK(hipMemcpyAsync(v.ptr + nv, moving_host, nv * sizeof(float), hipMemcpyHostToDevice,
                          backend().stream));
    pack(net, slot, 1, v.ptr);
    sync();  // the caller's host arrays may go once this returns
}

}  // namespace cnn
}  // namespace sitkhip

// =================================================================== C ABI
using namespace sitkhip;

extern "C" {

int sitkhip_cnn_create(int max_batch, uint64_t seed, sitkhip_cnn *out) {
    return run_guarded([&] {
        if (!out) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null out-pointer");
        *out = reinterpret_cast<sitkhip_cnn>(cnn::create(max_batch, seed));
    });
}

void sitkhip_cnn_free(sitkhip_cnn h) { delete reinterpret_cast<cnn::Net *>(h); }

static cnn::Net &net_ref(sitkhip_cnn h) {
    auto n = reinterpret_cast<cnn::Net *>(h);
    if (!n) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null network");
    return *n;
}

int sitkhip_cnn_param_count(sitkhip_cnn h, size_t *n) {
    return run_guarded([&] {
        if (!n) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null out-pointer");
        *n = net_ref(h).nparams;
    });
}

int sitkhip_cnn_get_params(sitkhip_cnn h, float *out, size_t n) {
    return run_guarded([&] {
        cnn::Net &net = net_ref(h);
        if (!out || n != net.nparams) fail(SITKHIP_ERR_INVALID_ARGUMENT, "length mismatch");
        net.params.download(out, n);
        sync();
    });
}

int sitkhip_cnn_set_params(sitkhip_cnn h, const float *in, size_t n) {
    return run_guarded([&] {
        cnn::Net &net = net_ref(h);
        if (!in || n != net.nparams) fail(SITKHIP_ERR_INVALID_ARGUMENT, "length mismatch");
        net.params.upload(in, n);
        sync();
        net.weights_dirty = true;
    });
}

int sitkhip_cnn_get_grads(sitkhip_cnn h, float *out, size_t n) {
    return run_guarded([&] {
        cnn::Net &net = net_ref(h);
        if (!out || n != net.nparams) fail(SITKHIP_ERR_INVALID_ARGUMENT, "length mismatch");
        net.grads.download(out, n);
        sync();
    });
}

int sitkhip_cnn_set_input(sitkhip_cnn h, int slot, sitkhip_image fixed, sitkhip_image moving) {
    return run_guarded([&] {
        auto f = reinterpret_cast<Image *>(fixed);
        auto m = reinterpret_cast<Image *>(moving);
        if (!f || !m) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image");
        cnn::set_input(net_ref(h), slot, *f, *m);
    });
}

int sitkhip_cnn_set_inputs(sitkhip_cnn h, int first_slot, int n, const sitkhip_image *fixed,
                           const sitkhip_image *moving) {
    return run_guarded([&] {
        if (!fixed || !moving) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image array");
        cnn::set_inputs(net_ref(h), first_slot, n, reinterpret_cast<const Image *const *>(fixed),
                        reinterpret_cast<const Image *const *>(moving));
    });
}

int sitkhip_cnn_set_input_raw(sitkhip_cnn h, int slot, const float *fixed64, const float *moving64) {
    return run_guarded([&] {
        if (!fixed64 || !moving64) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null volume");
        cnn::set_input_raw(net_ref(h), slot, fixed64, moving64);
    });
}

int sitkhip_cnn_forward(sitkhip_cnn h, int batch, float *out) {
    return run_guarded([&] { cnn::forward(net_ref(h), batch, out); });
}

int sitkhip_cnn_backward(sitkhip_cnn h, int batch, const float *dout) {
    return run_guarded([&] {
        if (!dout) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null gradient");
        cnn::backward(net_ref(h), batch, dout);
    });
}

int sitkhip_cnn_adam(sitkhip_cnn h, float lr, float beta1, float beta2, float eps) {
    return run_guarded([&] { cnn::adam(net_ref(h), lr, beta1, beta2, eps); });
}

int sitkhip_cnn_train_step(sitkhip_cnn h, int batch, const float *targets, float lr, float *loss) {
    return run_guarded([&] {
        cnn::Net &net = net_ref(h);
        if (!targets) fail(SITKHIP_ERR_INVALID_ARGUMENT, "null targets");
        std::vector<float> out(static_cast<size_t>(batch) * cnn::kOut), d(out.size());
        cnn::forward(net, batch, out.data());
        double l = 0.0;
        const float scale = 2.0f / static_cast<float>(out.size());
        for (size_t i = 0; i < out.size(); ++i) {
            const float e = out[i] - targets[i];
            l += static_cast<double>(e) * e;
            d[i] = scale * e;
        }
        if (loss) *loss = static_cast<float>(l / static_cast<double>(out.size()));
        cnn::backward(net, batch, d.data());
        cnn::adam(net, lr, 0.9f, 0.999f, 1e-8f);
    });
}

// Activation `index` (0 = packed input, l + 1 = conv l output) of the last
// forward pass, or with `gradient` != 0 the gradient w.r.t. it from the last
// backward pass (conv outputs: after the ReLU mask), as floats.
int sitkhip_cnn_activation(sitkhip_cnn h, int index, int gradient, int batch, float *out, size_t n) {
    return run_guarded([&] {
        cnn::Net &net = net_ref(h);
        if (index < 0 || index > cnn::kLayers) fail(SITKHIP_ERR_INVALID_ARGUMENT, "bad index");
        cnn::check_batch(net, batch);
        const size_t held = cnn::act_elems(index, batch);
        const size_t len = index == 0 ? held / cnn::kCin0Used * cnn::kCin0 : held;
        if (!out || n != len) fail(SITKHIP_ERR_INVALID_ARGUMENT, "length mismatch");
        std::vector<uint16_t> hb(held, 0);
        if (!(index == 0 && gradient)) {  // (the input's gradient is not computed: zeros)
            (gradient ? net.dact[index] : net.act[index]).download(hb.data(), held);
            sync();
        }
        if (index > 0) {
            for (size_t i = 0; i < len; ++i) out[i] = cnn::bf2f(hb[i]);
            return;
        }
        for (size_t i = 0; i < len; ++i) {  // the unused channels read zero
            const size_t v = i / cnn::kCin0, c = i % cnn::kCin0;
            out[i] = c < static_cast<size_t>(cnn::kCin0Used)
                         ? cnn::bf2f(hb[v * cnn::kCin0Used + c]) : 0.0f;
        }
    });
}

}  // extern "C"
