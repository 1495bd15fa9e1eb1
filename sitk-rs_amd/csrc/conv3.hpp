// The 3-D convolutions of the learned initializer on the gfx950 BF16 matrix
// cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation): forward, input gradient
// and weight gradient of the stride-2 layers, and the two-channel first layer.
//
// Every kernel stages the voxels that a tile of output positions reads, zero
// padding included, in LDS once for all 27 taps, and builds its matrix
// operands from there. Voxels are channels-last, so a forward or input-
// gradient operand (K = channels) is one 16-byte LDS read; the weight
// gradient's K runs over positions, which channels-last does not keep
// together, and its operands come through ds_read_b64_tr_b16, which hands
// each lane four consecutive rows of its column out of a 4 x 16 block.
// Voxels are spaced 2 C + 16 bytes apart in LDS: with stride-2 positions that
// puts eight neighbouring rows' 32-byte pieces on different banks for
// C = 16, 32, 64 and 128.
//
// MFMA 16x16x32 lane layout: lane l supplies row (A) or column (B) l mod 16,
// K group 8 (l / 16) .. + 7, and receives D rows 4 (l / 16) .. + 3 of column
// l mod 16.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

namespace sitkhip {
namespace cnn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // a staged 16-byte piece

union Frag {
    uint4 u;
    bf16x8 v;
    uint16_t h[8];
    i16x4 t[2];
};

__device__ __forceinline__ bf16x8 zero_frag() {
    Frag f;
    f.u = make_uint4(0, 0, 0, 0);
    return f.v;
}
__device__ __forceinline__ bf16x8 load_frag(const void *p) {
    Frag f;
    f.u = *reinterpret_cast<const uint4 *>(p);
    return f.v;
}
// Two transposed LDS reads: elements 0..3 from `p`, 4..7 from `p + h`. Lane
// 16 g + i passes the address of row i / 4, columns 4 (i mod 4) .. + 3 of its
// group's 4 x 16 block and receives rows 0..3 of column i. All lanes take part.
__device__ __forceinline__ bf16x8 tr_frag(const char *p, int h) {
    typedef __attribute__((address_space(3))) i16x4 *lds_ptr;
    Frag f;
    f.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
    f.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + h));
    return f.v;
}
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 zero_acc() { return f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }

// Four floats to four BF16 (round to nearest even), one 8-byte word.
__device__ __forceinline__ uint2 pack_bf16(const float v[4]) {
    union {
        __bf16 h[4];
        uint2 u;
    } w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w.h[e] = static_cast<__bf16>(v[e]);
    return w.u;
}
__device__ __forceinline__ float bf16_at(const uint2 &w, int e) {
    const uint32_t p = e < 2 ? w.x : w.y;
    return __uint_as_float((e & 1) ? (p & 0xffff0000u) : (p << 16));
}

constexpr int kConvLanes = 256;

// ------------------------------------------------ input tiles, stride 2
// A chunk of output positions: ZP planes x R rows x all DO columns of one
// sample. It reads input planes 2 z0 - 1 + .. , rows 2 y0 - 1 .. 2 y0 + 2 R - 1
// and columns -1 .. DI - 1 (stride 2 never reaches past the high edge).
// PL planes are staged; plane q's input z is first_z + q * step_z.
template <int LGDO, int CI, int R, int ZP, int PL>
struct InTile {
    static constexpr int DO = 1 << LGDO, DI = 2 * DO;
    static constexpr int ROWS = 2 * R + 1, COLS = DI + 1, VS = 2 * CI + 16;
    static constexpr int P = ZP * R * DO;  // output positions
    static constexpr int ZC = DO / ZP, YC = DO / R;
    static constexpr int kBytes = PL * ROWS * COLS * VS;
    static constexpr int kPieces = PL * ROWS * DI * (CI / 8);  // 16 bytes each
    static constexpr int kPer = (kPieces + kConvLanes - 1) / kConvLanes;
    static_assert(P % 16 == 0 && (ZP == 1 || R == DO), "whole position tiles");

    __device__ static void chunk(int c, int &n, int &z0, int &y0) {
        y0 = (c % YC) * R;
        const int q = c / YC;
        z0 = (q % ZC) * ZP;
        n = q / ZC;
    }
    static int chunks(int n) { return n * ZC * YC; }
    // column -1 of every row: zero, never overwritten
    __device__ static void clear_edge(char *lds) {
        for (int i = threadIdx.x; i < PL * ROWS * (VS / 16); i += kConvLanes)
            *reinterpret_cast<uint4 *>(lds + (i / (VS / 16)) * COLS * VS + (i % (VS / 16)) * 16) =
                make_uint4(0, 0, 0, 0);
    }
    __device__ static void load(const uint16_t *__restrict__ x, int n, int first_z, int step_z,
                                int y0, u32x4 (&v)[kPer]) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            const int c8 = i % (CI / 8), xi = i / (CI / 8) % DI, q = i / (CI / 8 * DI);
            const int zi = first_z + (q / ROWS) * step_z, yi = 2 * y0 - 1 + q % ROWS;
            v[k] = u32x4{0, 0, 0, 0};
            if (i < kPieces && zi >= 0 && yi >= 0)
                v[k] = *reinterpret_cast<const u32x4 *>(
                    x + (((static_cast<size_t>(n) * DI + zi) * DI + yi) * DI + xi) * CI + c8 * 8);
        }
    }
    __device__ static void store(char *lds, const u32x4 (&v)[kPer]) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            const int c8 = i % (CI / 8), xi = i / (CI / 8) % DI, q = i / (CI / 8 * DI);
            if (i < kPieces)
                *reinterpret_cast<u32x4 *>(lds + (q * COLS + xi + 1) * VS + c8 * 16) = v[k];
        }
    }
    // Byte offset of output position p's first tap (kz = ky = kx = 0); `zs`
    // staged planes lie between two output planes.
    __device__ static constexpr int at(int p, int zs) {
        const int xo = p % DO, r = p / DO % R, zp = p / (DO * R);
        return ((zp * zs * ROWS + 2 * r) * COLS + 2 * xo) * VS;
    }
    __host__ __device__ static constexpr int tap(int kz, int ky, int kx) {
        return ((kz * ROWS + ky) * COLS + kx) * VS;
    }
};

// ------------------------------------------------------- forward, stride 2
// y = bf16(relu(w x + b)). D rows are output channels (A: weights), columns
// positions, so a lane ends with four consecutive channels of one position.
// The four waves split the channel tiles first, then the position tiles. HOLD:
// the wave's weights stay in registers and the workgroup walks many chunks;
// otherwise they stream from L2 (layers whose weights exceed the registers
// have few positions).
// Bound by its traffic in layer 1 (268 MB in, 67 MB out for 32 pairs: 4.6 TB/s)
// and by latency in layers 3-4 (few positions). Gathering the operands from
// global memory, with every lane's voxel address worked out per K step, took
// 203 us for layer 1 and 168 us for layers 2-4 of 32 pairs; this takes 74 and 61.
template <int LGDO, int CI, int CO, int R, int COW, bool HOLD>
__global__ __launch_bounds__(kConvLanes) void conv_forward(const uint16_t *__restrict__ x,
                                                           const uint16_t *__restrict__ wb,
                                                           const float *__restrict__ bias,
                                                           uint16_t *__restrict__ y, int nchunks) {
    using T = InTile<LGDO, CI, R, 1, 3>;
    constexpr int K = 27 * CI, STEPS = (K + 31) / 32;
    constexpr int RT = COW / 16, WR = RT < 4 ? RT : 4, NR = RT / WR;  // row tiles per wave
    constexpr int WP = 4 / WR, PT = T::P / 16 / WP;                   // position tiles per wave
    static_assert(PT >= 1 && PT * WP * 16 == T::P, "positions split over the waves");
    extern __shared__ char lds[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.y * COW + (w % WR) * NR * 16;
    const int pt0 = (w / WR) * PT;
    const uint16_t *wrow = wb + static_cast<size_t>(row0 + r16) * K + 8 * g;
    auto weights = [&](int nr, int s) {
        return (STEPS * 32 > K && s == STEPS - 1 && 32 * s + 8 * g >= K)
                   ? zero_frag()
                   : load_frag(wrow + static_cast<size_t>(nr) * 16 * K + 32 * s);
    };
    bf16x8 held[HOLD ? NR * STEPS : 1];
    if (HOLD) {
#pragma unroll
        for (int i = 0; i < NR * STEPS; ++i) held[i] = weights(i / STEPS, i % STEPS);
    }
    int base[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p)
        base[p] = T::at((pt0 + p) * 16 + r16, 2) + (CI == 16 ? 16 * (g & 1) : 16 * g);
    T::clear_edge(lds);
    u32x4 v[T::kPer];
    int c = blockIdx.x, n, z0, y0;
    if (c < nchunks) {
        T::chunk(c, n, z0, y0);
        T::load(x, n, 2 * z0 - 1, 1, y0, v);
    }
    for (; c < nchunks; c += gridDim.x) {
        T::chunk(c, n, z0, y0);
        __syncthreads();
        T::store(lds, v);
        __syncthreads();
        const int cn = c + gridDim.x;
        if (HOLD && cn < nchunks) {
            int n2, z2, y2;
            T::chunk(cn, n2, z2, y2);
            T::load(x, n2, 2 * z2 - 1, 1, y2, v);
        }
        f32x4 acc[NR][PT];
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int p = 0; p < PT; ++p) acc[i][p] = zero_acc();
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            int off;
            if constexpr (CI == 16) {  // two taps per step: this lane group's
                const int t0 = 2 * s, t1 = 2 * s + 1 < 27 ? 2 * s + 1 : t0;
                const int o0 = T::tap(t0 / 9, t0 / 3 % 3, t0 % 3), o1 = T::tap(t1 / 9, t1 / 3 % 3, t1 % 3);
                off = g < 2 ? o0 : o1;
            } else {
                const int t = 32 * s / CI;
                off = T::tap(t / 9, t / 3 % 3, t % 3) + 2 * (32 * s % CI);
            }
            bf16x8 b[PT];
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                b[p] = load_frag(lds + base[p] + off);
                // the padding tap's weights are zero; so is what they meet
                if (STEPS * 32 > K && s == STEPS - 1 && 32 * s + 8 * g >= K) b[p] = zero_frag();
            }
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const bf16x8 a = HOLD ? held[i * STEPS + s] : weights(i, s);
#pragma unroll
                for (int p = 0; p < PT; ++p) acc[i][p] = mfma(a, b[p], acc[i][p]);
            }
        }
        const size_t pos0 = ((static_cast<size_t>(n) * T::DO + z0) * T::DO + y0) * T::DO;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int co = row0 + 16 * i + 4 * g;
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = fmaxf(acc[i][p][e] + bias[co + e], 0.0f);
                *reinterpret_cast<uint2 *>(y + (pos0 + (pt0 + p) * 16 + r16) * CO + co) = pack_bf16(o);
            }
        }
        if (!HOLD) break;  // one chunk per workgroup: nothing to carry over
    }
}

// ------------------------------------------------ weight gradient, stride 2
// dW[co][tap][ci] = sum over positions of dy[m][co] x[m's tap][ci]. The
// positions are cut into splits of `per` (a multiple of 32, wgrad_split), one
// per blockIdx.x; a split's products are added 32 positions at a time in the
// positions' order into one partial row [CO][27 CI], and reduce_partials adds
// the rows in order. The order of a gradient's sums is kept for good: a
// training run amplifies the rounding of a sum (Adam divides each gradient by
// its own size) until two orders differ by several percent after four steps.
// So the chip is filled by splitting the outputs, kernel planes (KZN), channels
// (COW) and column tiles (CG groups) over blockIdx.y, and the staged chunk (P
// positions) is large, since a split's chunks come one after another. 24 pairs,
// layers 1 to 4: 70, 56, 49 and 24 us (without column groups 70, 65, 73 and 27;
// a second chunk on its way changed nothing), bound by the LDS reads and stores
// between two barriers. Rows of any positions, added in a tree, took 60, 37, 14
// and 9. The first kernels, which gathered each operand's positions from global
// memory one scalar at a time, took 5.6 ms for the five layers.
template <int LGDO, int CI, int CO, int R, int ZP, int KZN, int COW, int CG>
__global__ __launch_bounds__(kConvLanes, CI <= 32 ? 2 : 1) void conv_wgrad(const uint16_t *__restrict__ x,
                                                         const uint16_t *__restrict__ dy,
                                                         float *__restrict__ partial, int per, int total) {
    using T = InTile<LGDO, CI, R, ZP, KZN * ZP>;
    constexpr int DS = 2 * COW + 16;                       // bytes per staged dy position
    constexpr int STEPS = T::P / 32, RT = COW / 16;
    constexpr int NC = 9 * KZN * CI / 16 / CG, NJ = (NC + 3) / 4;  // column tiles, per wave
    constexpr int DYP = T::P * COW / 8, DYN = (DYP + kConvLanes - 1) / kConvLanes;
    static_assert(T::P % 32 == 0 && (KZN == 3 ? ZP == 1 : KZN == 1), "chunk shape");
    static_assert(9 * KZN * CI / 16 % CG == 0, "column groups of whole tiles");
    extern __shared__ char lds[];
    char *sdy = lds + T::kBytes;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, g = lane >> 4;
    constexpr int KZG = 3 / KZN;  // workgroups along blockIdx.y: column groups, planes, channels
    const int t0 = (blockIdx.y % CG) * NC;
    const int kz0 = (blockIdx.y / CG % KZG) * KZN, co0 = (blockIdx.y / (CG * KZG)) * COW;

    const int p0 = 8 * g + (i16 >> 2);  // this lane's row of the first 4 x 16 block
    const int xbase = T::at(p0, 1) + 8 * (i16 & 3), dbase = p0 * DS + 8 * (i16 & 3);
    constexpr int kXHalf = T::DO >= 8 ? 8 * T::VS : 2 * T::COLS * T::VS;     // position + 4
    int toff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int t = t0 + w + 4 * j, tap = t / (CI / 16), c = t % (CI / 16);
        toff[j] = T::tap((tap / 9) * ZP, tap / 3 % 3, tap % 3) + 32 * c;
    }
    f32x4 acc[NJ][RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j][r] = zero_acc();

    T::clear_edge(lds);
    u32x4 v[T::kPer], d[DYN];
    auto fetch = [&](int c) {
        int n, z0, y0;
        T::chunk(c, n, z0, y0);
        T::load(x, n, 2 * z0 - 1 + kz0, KZN == 3 ? 1 : 2, y0, v);
        const size_t pos0 = static_cast<size_t>(c) * T::P;
#pragma unroll
        for (int k = 0; k < DYN; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            if (i < DYP)
                d[k] = *reinterpret_cast<const u32x4 *>(dy + (pos0 + i / (COW / 8)) * CO + co0 +
                                                        (i % (COW / 8)) * 8);
        }
    };
    auto step = [&](int s) {
        bf16x8 a[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) a[r] = tr_frag(sdy + dbase + s * 32 * DS + 32 * r, 4 * DS);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (NC % 4 != 0 && w + 4 * j >= NC) continue;  // the same for the whole wave
            const bf16x8 b = tr_frag(lds + xbase + toff[j] + T::at(32 * s, 1), kXHalf);
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[j][r] = mfma(a[r], b, acc[j][r]);
        }
    };
    // the split's positions; its first and last chunk may be a neighbour's too
    const int begin = blockIdx.x * per, end = min(begin + per, total);
    const int c_end = (end + T::P - 1) / T::P;
    int c = begin / T::P;
    if (c < c_end) fetch(c);
    for (; c < c_end; ++c) {
        __syncthreads();
        T::store(lds, v);
#pragma unroll
        for (int k = 0; k < DYN; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            if (i < DYP)
                *reinterpret_cast<u32x4 *>(sdy + (i / (COW / 8)) * DS + (i % (COW / 8)) * 16) = d[k];
        }
        __syncthreads();
        if (c + 1 < c_end) fetch(c + 1);
        const int at = c * T::P;
        if (at >= begin && at + T::P <= end) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) step(s);
        } else {
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (at + 32 * s >= begin && at + 32 * s < end) step(s);
        }
    }
    float *out = partial + static_cast<size_t>(blockIdx.x) * (CO * 27 * CI);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int t = w + 4 * j;
        if (NC % 4 != 0 && t >= NC) continue;
        const int col = kz0 * 9 * CI + (t0 + t) * 16 + i16;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                out[static_cast<size_t>(co0 + 16 * r + 4 * g + e) * (27 * CI) + col] = acc[j][r][e];
    }
}

// ------------------------------------------------------------ bias gradient
// db[co] = sum of dy[m][co], every layer in one launch: a workgroup takes one
// of kBiasSplits runs of a layer's positions, lane (c, part) adds channel c of
// positions part, part + 256 / C, ..., the parts are added in order, and
// reduce_partials adds the runs in order (see conv_wgrad on the order). 24
// pairs, 265 MB: 52 us (5.1 TB/s; the first kernels 709).
struct BiasLayer {
    const uint16_t *dy;
    float *partial;  // [kBiasSplits][channels]
    int positions, channels;
};
struct BiasLayers {
    BiasLayer l[5];
};
constexpr int kBiasSplits = 256;
constexpr int kBiasLoads = 64;  // in flight per lane: the first layer has 1,024 waves for 201 MB

__global__ __launch_bounds__(kConvLanes) void bias_grad(BiasLayers L) {
    __shared__ float red[kConvLanes];
    const BiasLayer &q = L.l[blockIdx.y];
    const int C = q.channels, parts = kConvLanes / C;
    const int per = (q.positions + kBiasSplits - 1) / kBiasSplits;
    const int m0 = blockIdx.x * per, m1 = min(q.positions, m0 + per);
    const int c = threadIdx.x % C, part = threadIdx.x / C;
    const uint16_t *p = q.dy + c;
    float acc = 0.0f;
    int m = m0 + part;
    for (; m + (kBiasLoads - 1) * parts < m1; m += kBiasLoads * parts) {
        uint16_t v[kBiasLoads];
#pragma unroll
        for (int u = 0; u < kBiasLoads; ++u) v[u] = p[static_cast<size_t>(m + u * parts) * C];
#pragma unroll
        for (int u = 0; u < kBiasLoads; ++u) acc += __uint_as_float(static_cast<uint32_t>(v[u]) << 16);
    }
#pragma unroll 8
    for (; m < m1; m += parts) acc += __uint_as_float(static_cast<uint32_t>(p[static_cast<size_t>(m) * C]) << 16);
    red[threadIdx.x] = acc;
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < C) {
        float t = 0.0f;
        for (int k = 0; k < parts; ++k) t += red[k * C + threadIdx.x];
        q.partial[static_cast<size_t>(blockIdx.x) * C + threadIdx.x] = t;
    }
}

// ------------------------------------------------- input gradient, stride 2
// dx at input position 2 q + p (p a parity triple) sums, along each axis, the
// taps (k = 1, output q) for p = 0 and (k = 0, output q + 1), (k = 2, output
// q) for p = 1: eight dense products with 1, 2, 2, 4, 2, 4, 4 and 8 taps over
// the same staged dy, 27 in all, where one product over every input position
// would multiply zeros in seven of eight taps. The result is masked by the
// layer's input (its ReLU) as it is stored.
// CG > 1: the parity classes are spread over blockIdx.y (layers with few
// positions). One product over every position took 495 us a layer for layers
// 1-2 of 24 pairs and 78 for layers 3-4, its masks 0.18 ms more; this takes
// 90 / 53 and 14 / 13.
// HOLD: the wave's 27 weight operands stay in registers and the workgroup
// walks many tiles (layer 1: 157 us with a weight load ahead of each product,
// 91 held: 452 MB, 5.0 TB/s); layers 2-4, whose operands do not fit, read them
// from L2 (loading a class's together spilled: layer 2 took 79 us).
template <int LGDO, int CI, int CO, int QY, int QZ, int CG, bool HOLD>
__global__ __launch_bounds__(kConvLanes, 2) void conv_dgrad(const uint16_t *__restrict__ dy,
                                                         const uint16_t *__restrict__ wt,
                                                         const uint16_t *__restrict__ act,
                                                         uint16_t *__restrict__ dx, int ntiles) {
    constexpr int DO = 1 << LGDO, DI = 2 * DO, DS = 2 * CO + 16, KS = CO / 32;
    constexpr int Y1 = QY + 1, Z1 = QZ + 1, X1 = DO + 1;
    constexpr int P = QZ * QY * DO, WR = CI / 16 < 4 ? CI / 16 : 4, WP = 4 / WR, PT = P / 16 / WP;
    static_assert(CI / 16 == WR && PT >= 1, "one row tile per wave");
    constexpr int kPieces = Z1 * Y1 * X1 * (CO / 8), kPer = (kPieces + kConvLanes - 1) / kConvLanes;
    extern __shared__ char lds[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int ci0 = (w % WR) * 16;
    int base[PT], inside[PT];  // LDS bytes of the tile's position q; element offset of 2 q in dx
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int p = ((w / WR) * PT + t) * 16 + r16;
        const int qx = p % DO, qy = p / DO % QY, qz = p / (DO * QY);
        base[t] = ((qz * Y1 + qy) * X1 + qx) * DS + 16 * g;
        inside[t] = ((2 * qz * DI + 2 * qy) * DI + 2 * qx) * CI + ci0 + 4 * g;
    }
    const uint16_t *wrow = wt + static_cast<size_t>(ci0 + r16) * 27 * CO + 8 * g;
    bf16x8 held[HOLD ? 27 * KS : 1];
    if (HOLD) {
#pragma unroll
        for (int i = 0; i < 27 * KS; ++i) held[i] = load_frag(wrow + 32 * i);
    }
    auto origin = [&](int tile, size_t &n, int &z0, int &y0) {
        y0 = (tile % (DO / QY)) * QY;
        z0 = tile / (DO / QY) % (DO / QZ) * QZ;
        n = tile / ((DO / QY) * (DO / QZ));
    };
    u32x4 v[kPer];
    auto fetch = [&](int tile) {
        size_t n;
        int z0, y0;
        origin(tile, n, z0, y0);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            const int c8 = i % (CO / 8), xo = i / (CO / 8) % X1, q = i / (CO / 8 * X1);
            const int yo = y0 + q % Y1, zo = z0 + q / Y1;
            v[k] = u32x4{0, 0, 0, 0};
            if (i < kPieces && xo < DO && yo < DO && zo < DO)
                v[k] = *reinterpret_cast<const u32x4 *>(dy + (((n * DO + zo) * DO + yo) * DO + xo) * CO +
                                                        c8 * 8);
        }
    };
    // eight classes with 8, (4 2 1), (4 2), (4 2) taps per group
    const unsigned group = CG == 1 ? 0xffu : (0x50240b80u >> (8 * blockIdx.y)) & 0xffu;
    int tile = blockIdx.x;
    if (tile < ntiles) fetch(tile);
    for (; tile < ntiles; tile += gridDim.x) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * kConvLanes;
            if (i < kPieces)
                *reinterpret_cast<u32x4 *>(lds + i / (CO / 8) * DS + i % (CO / 8) * 16) = v[k];
        }
        __syncthreads();
        if (HOLD && tile + static_cast<int>(gridDim.x) < ntiles) fetch(tile + gridDim.x);
        size_t n;
        int z0, y0;
        origin(tile, n, z0, y0);
        const size_t corner = (((n * DI + 2 * z0) * DI + 2 * y0) * DI) * CI;
#pragma unroll
        for (int cls = 0; cls < 8; ++cls) {
            if (!((group >> cls) & 1u)) continue;
            const int pz = cls >> 2, py = (cls >> 1) & 1, px = cls & 1;
            const size_t at = corner + static_cast<size_t>((pz * DI + py) * DI + px) * CI;
            f32x4 acc[PT];
            uint2 y[PT];
#pragma unroll
            for (int t = 0; t < PT; ++t) {
                acc[t] = zero_acc();
                y[t] = *reinterpret_cast<const uint2 *>(act + at + inside[t]);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int tz = k >> 2, ty = (k >> 1) & 1, tx = k & 1;
                if (tz > pz || ty > py || tx > px) continue;
                // parity 1: first k = 0 at q + 1, then k = 2 at q
                const int tap = (pz ? 2 * tz : 1) * 9 + (py ? 2 * ty : 1) * 3 + (px ? 2 * tx : 1);
                const int off = (((pz - tz) * Y1 + (py - ty)) * X1 + (px - tx)) * DS;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const bf16x8 a = HOLD ? held[tap * KS + s] : load_frag(wrow + tap * CO + 32 * s);
#pragma unroll
                    for (int t = 0; t < PT; ++t)
                        acc[t] = mfma(a, load_frag(lds + base[t] + off + 64 * s), acc[t]);
                }
            }
#pragma unroll
            for (int t = 0; t < PT; ++t) {
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = bf16_at(y[t], e) > 0.0f ? acc[t][e] : 0.0f;
                *reinterpret_cast<uint2 *>(dx + at + inside[t]) = pack_bf16(o);
            }
        }
        if (!HOLD) break;  // one tile per workgroup: nothing to carry over
    }
}

// ----------------------------------------------------------- first layer
// 2 -> 16 channels, stride 1, 64^3. A voxel's two channels are one 4-byte
// word. A chunk is ROWS output rows (ROWS / 4 per wave) of one plane; it reads
// 3 planes x (ROWS + 2) rows x voxels -2 .. 65, zero outside the volume.
template <int ROWS, int LANES = kConvLanes>
struct C0Tile {
    static constexpr int COLS = 68, kVox = 3 * (ROWS + 2) * COLS, WAVE_ROWS = ROWS / 4;
    static constexpr int kPer = (kVox + LANES - 1) / LANES;

    static int chunks(int n) { return n * 64 * (64 / ROWS); }
    __device__ static void chunk(int c, size_t &n, int &z, int &y0) {
        y0 = (c % (64 / ROWS)) * ROWS;
        z = (c / (64 / ROWS)) & 63;
        n = static_cast<size_t>(c / (64 / ROWS)) >> 6;
    }
    __device__ static void load(const uint32_t *__restrict__ x, int c, uint32_t (&v)[kPer]) {
        size_t n;
        int z, y0;
        chunk(c, n, z, y0);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * LANES;
            const int xi = i % COLS - 2, row = i / COLS;
            const int yi = y0 + row % (ROWS + 2) - 1, zi = z + row / (ROWS + 2) - 1;
            v[k] = 0;
            if (i < kVox && (xi | yi | zi) >= 0 && xi < 64 && yi < 64 && zi < 64)
                v[k] = x[((n * 64 + zi) * 64 + yi) * 64 + xi];
        }
    }
    __device__ static void store(char *lds, const uint32_t (&v)[kPer]) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = threadIdx.x + k * LANES;
            if (i < kVox) *reinterpret_cast<uint32_t *>(lds + 4 * i) = v[k];
        }
    }
    // byte of voxel x - 2 of the row that tap (kz, ky) of this wave's first
    // output row reads
    __device__ static int row(int kz, int ky, int wave) {
        return (kz * (ROWS + 2) + wave * WAVE_ROWS + ky) * COLS * 4;
    }
};

// Forward: K = 27 taps x 2 channels = 54, zero-padded to two MFMA steps; an
// operand's eight K values are four voxel words. Rows are output channels, so
// a lane stores four consecutive channels of one position. The weights stay
// in registers over the workgroup's chunks, and the next chunk's voxels load
// while this one's are multiplied: 163 us for 32 pairs with one chunk per
// workgroup and voxels of 16 bytes, 79 now (301 MB: 3.8 TB/s).
constexpr int kF0Rows = 8;  // (chunks of four rows: 96 us)
__global__ __launch_bounds__(kConvLanes) void conv0_forward(const uint32_t *__restrict__ x,
                                                            const uint16_t *__restrict__ wb, int ld,
                                                            const float *__restrict__ bias,
                                                            uint16_t *__restrict__ y, int nchunks) {
    using T = C0Tile<kF0Rows>;
    __shared__ __attribute__((aligned(16))) char lds[4 * T::kVox];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    bf16x8 a[2];
    int off[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        Frag f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int tap = 16 * s + 4 * g + j, t = tap < 27 ? tap : 26;
            f.h[2 * j] = tap < 27 ? wb[(r * 27 + t) * ld] : static_cast<uint16_t>(0);
            f.h[2 * j + 1] = tap < 27 ? wb[(r * 27 + t) * ld + 1] : static_cast<uint16_t>(0);
            off[s][j] = T::row(t / 9, t / 3 % 3, w) + (r + t % 3 + 1) * 4;
        }
        a[s] = f.v;
    }
    float b4[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) b4[e] = bias[4 * g + e];
    uint32_t v[T::kPer];
    int c = blockIdx.x;
    if (c < nchunks) T::load(x, c, v);
    for (; c < nchunks; c += gridDim.x) {
        __syncthreads();
        T::store(lds, v);
        __syncthreads();
        if (c + static_cast<int>(gridDim.x) < nchunks) T::load(x, c + gridDim.x, v);
        size_t n;
        int z, y0;
        T::chunk(c, n, z, y0);
        uint16_t *row = y + (((n * 64 + z) * 64 + y0 + w * T::WAVE_ROWS) * 64 + r) * 16 + 4 * g;
#pragma unroll
        for (int t = 0; t < 4 * T::WAVE_ROWS; ++t) {  // 16 positions each, four to a row
            f32x4 acc = zero_acc();
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t q[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    q[j] = *reinterpret_cast<const uint32_t *>(lds + off[s][j] + (t / 4) * T::COLS * 4 +
                                                               64 * (t % 4));
                    if (16 * s + 4 * g + j >= 27) q[j] = 0;  // padding: zero weights meet zeros
                }
                Frag f;
                f.u = make_uint4(q[0], q[1], q[2], q[3]);
                acc = mfma(a[s], f.v, acc);
            }
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = fmaxf(acc[e] + b4[e], 0.0f);
            *reinterpret_cast<uint2 *>(row + 16 * 16 * t) = pack_bf16(o);
        }
    }
}

// Weight gradient, the positions 32 at a time in their order (see conv_wgrad):
// one split of `per` positions per workgroup, one 16-column tile per wave of the
// first kW0Tiles. The three kx taps of one (kz, ky) are 12 consecutive bytes of
// a staged row, read as two 8-byte pieces (voxels x - 1, x and x + 1, x + 2;
// the last voxel's products are dropped), four pieces to a tile. A transposed
// read takes 8-byte pieces on 8-byte boundaries, so the rows are staged twice,
// the second time one voxel earlier, and an even x reads there. At most 256
// splits, a workgroup per CU: eight waves stage, two chunks ahead. 24 pairs, 226
// MB: 70 us (3.2 TB/s; 1,024 rows of any positions took 52).
constexpr int kW0Lanes = 512;
constexpr int kW0Dy = 48;  // bytes per staged dy position (16 channels + 16)
constexpr int kW0Rows = 8;
constexpr int kW0Tiles = 5;
constexpr int kW0Copy = 4 * C0Tile<kW0Rows, kW0Lanes>::kVox;  // one staged copy of the rows
constexpr int kW0Lds = 2 * kW0Copy + kW0Rows * 64 * kW0Dy;
constexpr int kW0Out = 16 * 54;  // [16][27][2]

__global__ __launch_bounds__(kW0Lanes) void conv0_wgrad(const uint32_t *__restrict__ x,
                                                        const uint16_t *__restrict__ dy,
                                                        float *__restrict__ partial, int per, int total) {
    using T = C0Tile<kW0Rows, kW0Lanes>;
    constexpr int P = kW0Rows * 64;  // positions of a chunk; splits are whole chunks
    __shared__ __attribute__((aligned(16))) char lds[kW0Lds];
    char *sdy = lds + 2 * kW0Copy;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, g = lane >> 4, sub = i16 & 3;
    const int p0 = 8 * g + (i16 >> 2);  // this lane's row of the first 4 x 16 block
    const int piece = min(4 * w + sub, 17);
    // voxel x - 1 lies at word x + 1 of its row, in the second copy at word x
    const int xoff = T::row(piece / 6, piece / 2 % 3, 0) + (p0 & 1 ? 4 * (p0 + 1) : kW0Copy + 4 * p0) +
                     8 * (piece & 1);
    const int dbase = p0 * kW0Dy + 8 * sub;
    f32x4 acc = zero_acc();
    constexpr int kDyN = P * 2 / kW0Lanes;
    struct Chunk {
        uint32_t v[T::kPer];
        u32x4 d[kDyN];
    } even, odd;
    auto fetch = [&](Chunk &q, int c) {
        T::load(x, c, q.v);
#pragma unroll
        for (int k = 0; k < kDyN; ++k)
            q.d[k] = *reinterpret_cast<const u32x4 *>(dy + static_cast<size_t>(c) * P * 16 +
                                                      (threadIdx.x + k * kW0Lanes) * 8);
    };
    const int c_end = min(static_cast<int>(blockIdx.x + 1) * per, total) / P;
    auto run = [&](Chunk &q, int c) {
        if (c >= c_end) return;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < T::kPer; ++k) {
            const int i = threadIdx.x + k * kW0Lanes;
            if (i < T::kVox) {
                *reinterpret_cast<uint32_t *>(lds + 4 * i) = q.v[k];
                if (i > 0) *reinterpret_cast<uint32_t *>(lds + kW0Copy + 4 * (i - 1)) = q.v[k];
            }
        }
#pragma unroll
        for (int k = 0; k < kDyN; ++k) {
            const int i = threadIdx.x + k * kW0Lanes;
            *reinterpret_cast<u32x4 *>(sdy + (i >> 1) * kW0Dy + (i & 1) * 16) = q.d[k];
        }
        __syncthreads();
        if (c + 2 < c_end) fetch(q, c + 2);
        if (w >= kW0Tiles) return;  // these waves stage only
#pragma unroll
        for (int s = 0; s < P / 32; ++s) {
            const bf16x8 a = tr_frag(sdy + dbase + 32 * s * kW0Dy, 4 * kW0Dy);
            acc = mfma(a, tr_frag(lds + xoff + (s >> 1) * T::COLS * 4 + (s & 1) * 128, 16), acc);
        }
    };
    int c = blockIdx.x * per / P;
    if (c < c_end) fetch(even, c);
    if (c + 1 < c_end) fetch(odd, c + 1);
    for (; c < c_end; c += 2) {
        run(even, c);
        run(odd, c + 1);
    }
    if (w >= kW0Tiles) return;
    float *out = partial + static_cast<size_t>(blockIdx.x) * kW0Out;
    const int pi = 4 * w + (i16 >> 2), kx = 2 * (pi & 1) + ((i16 >> 1) & 1);  // this lane's column
    if (pi < 18 && kx < 3)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            out[(4 * g + e) * 54 + ((pi >> 1) * 3 + kx) * 2 + (i16 & 1)] = acc[e];
}

// ---------------------------------------------------------- partial rows
// Partial rows summed into the gradient vector in one launch, each value's rows
// in their order (see conv_wgrad), sixteen loads ahead (24 pairs: 12 us). Value i goes to
// out[(i / inner) * ld + i % inner] (the first layer's two used channels lie
// eight apart in the parameter vector).
struct PartialRows {
    const float *p;
    float *out;
    int rows, len, inner, ld;
    unsigned first_block;
};
constexpr int kMaxPartialJobs = 10;
struct PartialJobs {
    PartialRows j[kMaxPartialJobs];
    int n;
};
constexpr int kPartialLanes = 64;

__global__ __launch_bounds__(kPartialLanes) void reduce_partials(PartialJobs J) {
    int k = 0;
    while (k + 1 < J.n && blockIdx.x >= J.j[k + 1].first_block) ++k;
    const PartialRows &q = J.j[k];
    const int i = static_cast<int>(blockIdx.x - q.first_block) * kPartialLanes + threadIdx.x;
    if (i >= q.len) return;
    const float *p = q.p + i;
    float s = 0.0f;
    int r = 0;
    for (; r + 16 <= q.rows; r += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = p[static_cast<size_t>(r + u) * q.len];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += v[u];
    }
    for (; r < q.rows; ++r) s += p[static_cast<size_t>(r) * q.len];
    q.out[(i / q.inner) * q.ld + i % q.inner] = s;
}

}  // namespace cnn
}  // namespace sitkhip
