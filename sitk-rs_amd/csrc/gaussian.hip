// Recursive (Deriche/Farneback 4th-order IIR) Gaussian smoothing on the device,
// bit-exact against the reference's host filter.
//
// Reference: crates/sitk/src/filters/recursive_gaussian.rs:171-204 (axis loop),
// :472-528 (filter_line), crates/sitk/src/core/deriche.rs:187-347 (the 20
// coefficients), crates/sitk/src/cuda/ops/pyramid.rs:217-293 (device entry).
//
// Bit-exactness rests on three things, all kept here:
//   1. The recursion runs in FP64 with every multiply and add rounded separately
//      (this file is compiled with -ffp-contract=off) and in the reference's
//      left-to-right term order, one line per lane.
//   2. The coefficients are computed on the host with the platform libm, in the
//      reference's expression order, and handed to the kernel.
//   3. Intermediate axes stay FP64; the only narrowing is (float) of the last
//      smoothed axis' output, which equals the reference's single `as f32`.
//
// Layout: volumes are dimension-0 fastest. A smoothed axis is one launch. Lines
// along axes 1 and 2 are assigned to lanes by their dimension-0 coordinate, so
// every step of the recursion is one coalesced access across a wavefront; axis 0
// lines are contiguous, so there a lane reads and writes 16 bytes of its line at
// a time.
#include <hip/hip_runtime.h>

#include <array>
#include <algorithm>
#include <vector>

#include <cmath>
#include <cstring>
#include <mutex>

#include "common.hpp"
#include "image.hpp"

namespace sitkhip {

// The 20 coefficients in to_array order (deriche.rs:290-296):
// [n0..n3, d1..d4, m1..m4, bn1..bn4, bm1..bm4].
struct IirCoef {
    double c[20];
};

// ----------------------------------------------------------- host: coefficients
// Poles and the ZeroOrder Farneback column (deriche.rs:112-117, 135-140).
namespace {
constexpr double kW1 = 0.6681, kL1 = -1.3932, kW2 = 2.0787, kL2 = -1.3732;
constexpr double kA1 = 1.3530, kB1 = 1.8151, kA2 = -0.3531, kB2 = 0.0902;
}  // namespace

// ZeroOrder coefficients for index-space sigma `sigmad` (deriche.rs:187-280
// with compute_d_coefficients :304-319 and compute_n_coefficients :325-347).
// The same products and sums as the reference, in the same order.
IirCoef zero_order_coefficients(double sigmad) {
    const double cos1 = std::cos(kW1 / sigmad), cos2 = std::cos(kW2 / sigmad);
    const double sin1 = std::sin(kW1 / sigmad), sin2 = std::sin(kW2 / sigmad);
    const double e1 = std::exp(kL1 / sigmad), e2 = std::exp(kL2 / sigmad);

    const double d4 = e1 * e1 * e2 * e2;
    const double d3 = -2.0 * cos1 * e1 * e2 * e2 - 2.0 * cos2 * e2 * e1 * e1;
    const double d2 = 4.0 * cos2 * cos1 * e1 * e2 + e1 * e1 + e2 * e2;
    const double d1 = -2.0 * (e2 * cos2 + e1 * cos1);
    const double sd = 1.0 + d1 + d2 + d3 + d4;

    double n0 = kA1 + kA2;
    double n1 = e2 * (kB2 * sin2 - (kA2 + 2.0 * kA1) * cos2) +
                e1 * (kB1 * sin1 - (kA1 + 2.0 * kA2) * cos1);
    double n2 = ((kA1 + kA2) * cos2 * cos1 - kB1 * cos2 * sin1 - kB2 * cos1 * sin2) * 2.0 * e1 * e2 +
                kA2 * e1 * e1 + kA1 * e2 * e2;
    double n3 = e2 * e1 * e1 * (kB2 * sin2 - kA2 * cos2) + e1 * e2 * e2 * (kB1 * sin1 - kA1 * cos1);
    const double sn_raw = n0 + n1 + n2 + n3;

    // Unity DC gain.
    const double alpha0 = 2.0 * sn_raw / sd - n0;
    n0 = n0 / alpha0;
    n1 = n1 / alpha0;
    n2 = n2 / alpha0;
    n3 = n3 / alpha0;

    // Symmetric anti-causal numerator and the boundary coefficients.
    const double m1 = n1 - d1 * n0, m2 = n2 - d2 * n0, m3 = n3 - d3 * n0, m4 = -d4 * n0;
    const double sn = n0 + n1 + n2 + n3;
    const double sm = m1 + m2 + m3 + m4;

    IirCoef k;
    double *c = k.c;
    c[0] = n0; c[1] = n1; c[2] = n2; c[3] = n3;
    c[4] = d1; c[5] = d2; c[6] = d3; c[7] = d4;
    c[8] = m1; c[9] = m2; c[10] = m3; c[11] = m4;
    c[12] = d1 * sn / sd; c[13] = d2 * sn / sd; c[14] = d3 * sn / sd; c[15] = d4 * sn / sd;
    c[16] = d1 * sm / sd; c[17] = d2 * sm / sd; c[18] = d3 * sm / sd; c[19] = d4 * sm / sd;
    return k;
}

// ------------------------------------------------------------------- device
template <typename T>
__device__ __forceinline__ double widen(T v) { return static_cast<double>(v); }

template <typename T>
__device__ __forceinline__ T narrow(double v);
template <>
__device__ __forceinline__ double narrow<double>(double v) { return v; }
template <>
__device__ __forceinline__ float narrow<float>(double v) { return static_cast<float>(v); }

// The line geometry of one smoothed axis.
struct LineSet {
    long long nlines;
    int len;             // elements per line
    long long stride;    // element stride along the line
    long long n0, n01;   // for decoding a line index
    int axis;
};

__device__ __forceinline__ long long line_start(const LineSet &L, long long l) {
    if (L.axis == 0) return l * L.n0;                                 // l = i1 + i2*n1
    if (L.axis == 1) return (l % L.n0) + (l / L.n0) * L.n01;          // l = i0 + i2*n0
    return l;                                                         // l = i0 + i1*n0
}

// One line per lane, straight from global memory (axes 1 and 2: adjacent lanes
// touch adjacent addresses at every step).
//
// Causal pass: writes outs[k] to tmp. Anti-causal pass: walks back, and writes
// dst[k] = narrow(outs[k] + scratch[k]) as soon as scratch[k] exists -- the
// same single addition the reference's final loop performs (:525-527).
// tmp may alias dst when DstT is double (each element is read before it is
// overwritten, by the same lane).
template <typename SrcT, typename DstT>
__global__ __launch_bounds__(256) void iir_lines(const SrcT *__restrict__ src, double *tmp,
                                                 DstT *dst, LineSet L, IirCoef k) {
    const long long l = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (l >= L.nlines) return;
    const long long s0 = line_start(L, l);
    const long long st = L.stride;
    const int ln = L.len;
    const double *c = k.c;
    const double n0 = c[0], n1 = c[1], n2 = c[2], n3 = c[3];
    const double d1 = c[4], d2 = c[5], d3 = c[6], d4 = c[7];
    const double m1 = c[8], m2 = c[9], m3 = c[10], m4 = c[11];

    // ---- causal (recursive_gaussian.rs:476-493)
    const double v1 = widen(src[s0]);
    const double x1 = widen(src[s0 + st]);
    const double x2 = widen(src[s0 + 2 * st]);
    const double x3 = widen(src[s0 + 3 * st]);
    double o0 = v1 * n0 + v1 * n1 + v1 * n2 + v1 * n3;
    double o1 = x1 * n0 + v1 * n1 + v1 * n2 + v1 * n3;
    double o2 = x2 * n0 + x1 * n1 + v1 * n2 + v1 * n3;
    double o3 = x3 * n0 + x2 * n1 + x1 * n2 + v1 * n3;
    o0 -= v1 * c[12] + v1 * c[13] + v1 * c[14] + v1 * c[15];
    o1 -= o0 * d1 + v1 * c[13] + v1 * c[14] + v1 * c[15];
    o2 -= o1 * d1 + o0 * d2 + v1 * c[14] + v1 * c[15];
    o3 -= o2 * d1 + o1 * d2 + o0 * d3 + v1 * c[15];
    tmp[s0] = o0;
    tmp[s0 + st] = o1;
    tmp[s0 + 2 * st] = o2;
    tmp[s0 + 3 * st] = o3;
    // window: a = data[i-1], b = data[i-2], cc = data[i-3]; p1..p4 = outs[i-1..i-4]
    double a = x3, b = x2, cc = x1;
    double p1 = o3, p2 = o2, p3 = o1, p4 = o0;
    for (int i = 4; i < ln; ++i) {
        const double x = widen(src[s0 + i * st]);
        double o = x * n0 + a * n1 + b * n2 + cc * n3;
        o -= p1 * d1 + p2 * d2 + p3 * d3 + p4 * d4;
        tmp[s0 + i * st] = o;
        cc = b; b = a; a = x;
        p4 = p3; p3 = p2; p2 = p1; p1 = o;
    }

    // ---- anti-causal (recursive_gaussian.rs:495-522) and the roll-in (:525-527)
    const long long e = s0 + static_cast<long long>(ln - 1) * st;
    const double v2 = widen(src[e]);
    const double y1 = widen(src[e - st]);      // data[ln-2]
    const double y2 = widen(src[e - 2 * st]);  // data[ln-3]
    double s_1 = v2 * m1 + v2 * m2 + v2 * m3 + v2 * m4;          // scratch[ln-1]
    double s_2 = v2 * m1 + v2 * m2 + v2 * m3 + v2 * m4;          // data[ln-1] is v2
    double s_3 = y1 * m1 + v2 * m2 + v2 * m3 + v2 * m4;          // scratch[ln-3]
    double s_4 = y2 * m1 + y1 * m2 + v2 * m3 + v2 * m4;          // scratch[ln-4]
    s_1 -= v2 * c[16] + v2 * c[17] + v2 * c[18] + v2 * c[19];
    s_2 -= s_1 * d1 + v2 * c[17] + v2 * c[18] + v2 * c[19];
    s_3 -= s_2 * d1 + s_1 * d2 + v2 * c[18] + v2 * c[19];
    s_4 -= s_3 * d1 + s_2 * d2 + s_1 * d3 + v2 * c[19];
    dst[e] = narrow<DstT>(tmp[e] + s_1);
    dst[e - st] = narrow<DstT>(tmp[e - st] + s_2);
    dst[e - 2 * st] = narrow<DstT>(tmp[e - 2 * st] + s_3);
    dst[e - 3 * st] = narrow<DstT>(tmp[e - 3 * st] + s_4);
    // window for index j: data[j+1..j+4] = (w1, w2, w3, w4); scratch[j+1..j+4] = (q1..q4)
    double w2 = y2, w3 = y1, w4 = v2;    // data[ln-3], data[ln-2], data[ln-1]
    double q1 = s_4, q2 = s_3, q3 = s_2, q4 = s_1;
    for (int j = ln - 5; j >= 0; --j) {
        const double w1 = widen(src[s0 + (j + 1) * st]);  // data[j+1]
        double s = w1 * m1 + w2 * m2 + w3 * m3 + w4 * m4;
        s -= q1 * d1 + q2 * d2 + q3 * d3 + q4 * d4;
        dst[s0 + j * st] = narrow<DstT>(tmp[s0 + j * st] + s);
        w4 = w3; w3 = w2; w2 = w1;
        q4 = q3; q3 = q2; q2 = q1; q1 = s;
    }
}

// Two lanes per line, 32 lines per wavefront: lane l < 32 runs the causal
// recursion of line l forward while lane l + 32 runs the anti-causal recursion
// of the same line backward, in lock-step. At step i the causal lane produces
// outs[i] and the anti-causal lane scratch[n-1-i]. Until the middle each lane
// parks its values; after it, each lane takes its partner's value for the same
// element (parked n-1-i steps earlier) and writes the finished output outs[k] +
// scratch[k] (of an odd line's middle element both lanes hold their term at
// the same step). The causal outputs never leave the chip, so a line costs one
// read of its input per lane and one write of its output. Both recursions have
// the same shape,
//     v = (((x*c0 + a*c1) + b*c2) + cc*c3) - (((p1*d1 + p2*d2) + p3*d3) + p4*d4),
// with (c0..c3) = (n0..n3) for the causal lane and (m1..m4) for the anti-causal
// lane (whose x is data[j+1] for output j), so the loop is lane-uniform.
//
// The last kRegPairs * 16 values before the middle are parked in registers (a
// partner's come across the wave by ds_bpermute), the earlier ones in LDS: at
// 256 voxels a wave of 32 lines takes 24 KB of LDS instead of 64, so every
// line of a 256 x 256 x 160 volume is resident at once (five waves per CU; with
// all values in LDS two, and 98 / 72 / 44 us for the three axes; now 47 / 38 /
// 29: 2.7 / 4.4 / 4.3 TB/s). Four pairs leave 32 KB, which five waves of a CU
// do not fit, and took 61 / 51 / 30; six spill. The registers then allow two
// waves per SIMD; fewer pairs for more waves gained nothing on short lines.
//
// Steps run in blocks of eight whose inputs load one to two blocks ahead, into
// two register blocks used in turn (blocks of sixteen measured the same).
// ALONG0 (axis 0, whose lines are contiguous):
// a block's inputs are two or four 16-byte loads of the lane's own line, and
// its outputs 16-byte stores -- one step per instruction touched 64 cache
// lines for 4 or 8 bytes each and bound that axis.
constexpr int kPairLines = 32;
constexpr int kPD = 8;
constexpr int kRegPairs = 5;

// Steps [0, lds_steps) of a line of n voxels (n >= 8) are parked in LDS, the
// others before the middle in registers.
__host__ __device__ inline int reg_pairs(int n) {
    const int k = (n / 2 - 4) / (2 * kPD);
    return k < kRegPairs ? k : kRegPairs;
}
__host__ __device__ inline int lds_steps(int n) { return n / 2 - 2 * kPD * reg_pairs(n); }
inline size_t pair_lds_bytes(int n) {
    return static_cast<size_t>(2) * lds_steps(n) * kPairLines * sizeof(double);
}

// Sixteen bytes of a contiguous line, at the element's alignment.
template <typename T>
struct alignas(sizeof(T)) Vec16 {
    T v[16 / sizeof(T)];
};

template <typename SrcT, typename DstT, bool ALONG0>
__device__ __forceinline__ void iir_pair_body(const SrcT *__restrict__ src, DstT *__restrict__ dst,
                                              const LineSet &L, const IirCoef &k, unsigned block,
                                              double *lds) {
    const int lane = threadIdx.x;
    const int role = lane >> 5;  // 0 causal, 1 anti-causal
    const int li = lane & 31;
    long long line = static_cast<long long>(block) * kPairLines + li;
    const bool act = line < L.nlines;
    if (!act) line = L.nlines - 1;  // mirror a valid line; stores are suppressed
    const long long s0 = line_start(L, line);
    const long long st = ALONG0 ? 1 : L.stride;
    const int n = L.len;
    const double *c = k.c;
    const double d1 = c[4], d2 = c[5], d3 = c[6], d4 = c[7];
    const double c0 = role ? c[8] : c[0];
    const double c1 = role ? c[9] : c[1];
    const double c2 = role ? c[10] : c[2];
    const double c3 = role ? c[11] : c[3];
    const int park = lds_steps(n), pairs = reg_pairs(n), half = n / 2;
    double *mine = lds + role * park * kPairLines + li;
    const double *partner = lds + (1 - role) * park * kPairLines + li;

    double a, b, cc, p1, p2, p3, p4;
    double v[4];
    if (role == 0) {
        // causal boundary (recursive_gaussian.rs:476-487)
        const double n0 = c[0], n1 = c[1], n2 = c[2], n3 = c[3];
        const double v1 = widen(src[s0]);
        const double x1 = widen(src[s0 + st]);
        const double x2 = widen(src[s0 + 2 * st]);
        const double x3 = widen(src[s0 + 3 * st]);
        double o0 = v1 * n0 + v1 * n1 + v1 * n2 + v1 * n3;
        double o1 = x1 * n0 + v1 * n1 + v1 * n2 + v1 * n3;
        double o2 = x2 * n0 + x1 * n1 + v1 * n2 + v1 * n3;
        double o3 = x3 * n0 + x2 * n1 + x1 * n2 + v1 * n3;
        o0 -= v1 * c[12] + v1 * c[13] + v1 * c[14] + v1 * c[15];
        o1 -= o0 * d1 + v1 * c[13] + v1 * c[14] + v1 * c[15];
        o2 -= o1 * d1 + o0 * d2 + v1 * c[14] + v1 * c[15];
        o3 -= o2 * d1 + o1 * d2 + o0 * d3 + v1 * c[15];
        v[0] = o0; v[1] = o1; v[2] = o2; v[3] = o3;
        a = x3; b = x2; cc = x1;
        p1 = o3; p2 = o2; p3 = o1; p4 = o0;
    } else {
        // anti-causal boundary (recursive_gaussian.rs:496-510)
        const double m1 = c[8], m2 = c[9], m3 = c[10], m4 = c[11];
        const long long e = s0 + static_cast<long long>(n - 1) * st;
        const double v2 = widen(src[e]);
        const double y1 = widen(src[e - st]);
        const double y2 = widen(src[e - 2 * st]);
        double q1 = v2 * m1 + v2 * m2 + v2 * m3 + v2 * m4;
        double q2 = v2 * m1 + v2 * m2 + v2 * m3 + v2 * m4;
        double q3 = y1 * m1 + v2 * m2 + v2 * m3 + v2 * m4;
        double q4 = y2 * m1 + y1 * m2 + v2 * m3 + v2 * m4;
        q1 -= v2 * c[16] + v2 * c[17] + v2 * c[18] + v2 * c[19];
        q2 -= q1 * d1 + v2 * c[17] + v2 * c[18] + v2 * c[19];
        q3 -= q2 * d1 + q1 * d2 + v2 * c[18] + v2 * c[19];
        q4 -= q3 * d1 + q2 * d2 + q1 * d3 + v2 * c[19];
        v[0] = q1; v[1] = q2; v[2] = q3; v[3] = q4;  // scratch[n-1 .. n-4]
        a = y2; b = y1; cc = v2;                     // data[n-3], data[n-2], data[n-1]
        p1 = q4; p2 = q3; p3 = q2; p4 = q1;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) mine[i * kPairLines] = v[i];

    // the value read at step i sits at A + i * S; the output of step i at W + i * S
    const long long S = role ? -st : st;
    const SrcT *const A = src + (role ? s0 + static_cast<long long>(n) * st : s0);
    DstT *const W = dst + (role ? s0 + static_cast<long long>(n - 1) * st : s0);

    // The inputs of steps base .. base + 7. A block that would pass the line's
    // end reads inside it instead (its values are not used).
    auto load_block = [&](SrcT (&buf)[kPD], int base) {
        const bool in = base + kPD <= n;
        if constexpr (ALONG0) {
            constexpr int kV = 16 / sizeof(SrcT);
            // ascending addresses: the anti-causal lane's block is read reversed
            const SrcT *p = in ? (role ? A - base - (kPD - 1) : A + base) : src + s0;
            Vec16<SrcT> q[kPD / kV];
#pragma unroll
            for (int j = 0; j < kPD / kV; ++j) q[j] = *reinterpret_cast<const Vec16<SrcT> *>(p + j * kV);
#pragma unroll
            for (int j = 0; j < kPD; ++j) {
                const int r = kPD - 1 - j;
                buf[j] = role ? q[r / kV].v[r % kV] : q[j / kV].v[j % kV];
            }
        } else {
            const SrcT *p = A + static_cast<long long>(in ? base : n - 1) * S;
            const long long step = in ? S : 0;
#pragma unroll
            for (int j = 0; j < kPD; ++j) {
                buf[j] = *p;
                p += step;
            }
        }
    };
    auto store_block = [&](const DstT (&o)[kPD], int base) {
        if (!act) return;
        if constexpr (ALONG0) {
            constexpr int kV = 16 / sizeof(DstT);
            DstT *p = role ? W - base - (kPD - 1) : W + base;
#pragma unroll
            for (int j = 0; j < kPD / kV; ++j) {
                Vec16<DstT> q;
#pragma unroll
                for (int e = 0; e < kV; ++e) q.v[e] = role ? o[kPD - 1 - (j * kV + e)] : o[j * kV + e];
                *reinterpret_cast<Vec16<DstT> *>(p + j * kV) = q;
            }
        } else {
            DstT *p = W + base * S;
#pragma unroll
            for (int j = 0; j < kPD; ++j) {
                *p = o[j];
                p += S;
            }
        }
    };
    auto recur = [&](SrcT in) {
        const double x = widen(in);
        double o = x * c0 + a * c1 + b * c2 + cc * c3;
        o -= p1 * d1 + p2 * d2 + p3 * d3 + p4 * d4;
        cc = b; b = a; a = x;
        p4 = p3; p3 = p2; p2 = p1; p1 = o;
        return o;
    };
    // the input of one step, for what does not fill a block
    auto input = [&](int i) { return A[static_cast<long long>(i) * S]; };

    // ---- steps 4 .. park - 1 into LDS: first those past whole pairs of blocks
    const int odd_steps = (park - 4) % (2 * kPD);
    SrcT bufA[kPD], bufB[kPD];
    int base = 4 + odd_steps;
    load_block(bufA, base);
    {
        SrcT x[2 * kPD - 1];
#pragma unroll
        for (int j = 0; j < 2 * kPD - 1; ++j) x[j] = input(4 + (j < odd_steps ? j : 0));
#pragma unroll
        for (int j = 0; j < 2 * kPD - 1; ++j)
            if (j < odd_steps) mine[(4 + j) * kPairLines] = recur(x[j]);
    }
    for (; base < park; base += 2 * kPD) {
        load_block(bufB, base + kPD);
#pragma unroll
        for (int j = 0; j < kPD; ++j) mine[(base + j) * kPairLines] = recur(bufA[j]);
        load_block(bufA, base + 2 * kPD);
#pragma unroll
        for (int j = 0; j < kPD; ++j) mine[(base + kPD + j) * kPairLines] = recur(bufB[j]);
    }
    // ---- steps park .. n / 2 - 1 into registers
    double held[kRegPairs][2 * kPD];
#pragma unroll
    for (int r = 0; r < kRegPairs; ++r) {
        if (r < pairs) {
            load_block(bufB, base + kPD);
#pragma unroll
            for (int j = 0; j < kPD; ++j) held[r][j] = recur(bufA[j]);
            load_block(bufA, base + 2 * kPD);
#pragma unroll
            for (int j = 0; j < kPD; ++j) held[r][kPD + j] = recur(bufB[j]);
            base += 2 * kPD;
        }
    }
    // ---- an odd line's middle element: both lanes hold their term now
    if (n & 1) {
        const double o = recur(base + kPD <= n ? bufA[0] : input(base));
        const double q = __shfl_xor(o, 32, 64);
        if (role == 0 && act) W[static_cast<long long>(half) * S] = narrow<DstT>(o + q);
        ++base;
        load_block(bufA, base);
    }
    // ---- back through the registers
    auto run_back = [&](const SrcT (&buf)[kPD], const double (&q)[kPD], int at) {
        DstT o[kPD];
#pragma unroll
        for (int j = 0; j < kPD; ++j) o[j] = narrow<DstT>(recur(buf[j]) + q[j]);
        store_block(o, at);
    };
#pragma unroll
    for (int r = kRegPairs - 1; r >= 0; --r) {
        if (r < pairs) {
            double q[kPD];
#pragma unroll
            for (int j = 0; j < kPD; ++j) q[j] = __shfl_xor(held[r][2 * kPD - 1 - j], 32, 64);
            load_block(bufB, base + kPD);
            run_back(bufA, q, base);
#pragma unroll
            for (int j = 0; j < kPD; ++j) q[j] = __shfl_xor(held[r][kPD - 1 - j], 32, 64);
            load_block(bufA, base + 2 * kPD);
            run_back(bufB, q, base + kPD);
            base += 2 * kPD;
        }
    }
    // ---- back through LDS. The workgroup is this one wave: before the first
    // read of the partner's values only this wave's LDS writes need to have landed.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    for (; base + 2 * kPD <= n; base += 2 * kPD) {
        double q[kPD];
#pragma unroll
        for (int j = 0; j < kPD; ++j) q[j] = partner[(n - 1 - base - j) * kPairLines];
        load_block(bufB, base + kPD);
        run_back(bufA, q, base);
#pragma unroll
        for (int j = 0; j < kPD; ++j) q[j] = partner[(n - 1 - base - kPD - j) * kPairLines];
        load_block(bufA, base + 2 * kPD);
        run_back(bufB, q, base + kPD);
    }
    if (base < n) {  // the last steps, loaded together
        SrcT x[2 * kPD - 1];
        double q[2 * kPD - 1];
#pragma unroll
        for (int j = 0; j < 2 * kPD - 1; ++j) {
            const int i = base + j < n ? base + j : n - 1;
            x[j] = input(i);
            q[j] = partner[(n - 1 - i) * kPairLines];
        }
#pragma unroll
        for (int j = 0; j < 2 * kPD - 1; ++j) {
            if (base + j < n) {
                const double o = recur(x[j]);
                if (act) W[static_cast<long long>(base + j) * S] = narrow<DstT>(o + q[j]);
            }
        }
    }
}

template <typename SrcT, typename DstT, bool ALONG0>
__global__ __launch_bounds__(64, 2) void iir_pair_lines(const SrcT *__restrict__ src,
                                                        DstT *__restrict__ dst, LineSet L, IirCoef k) {
    extern __shared__ double lds[];  // [2][lds_steps][32]: role, step, line
    iir_pair_body<SrcT, DstT, ALONG0>(src, dst, L, k, blockIdx.x, lds);
}

// Many volumes' lines along one axis in one launch: workgroup b takes
// volume vol_of[b], lines (b - first_block) * 32 ... of it, with that
// volume's line geometry and coefficients; the per-line arithmetic is
// iir_pair_lines'.
struct BatchLines {
    const void *src;
    void *dst;
    LineSet L;
    IirCoef k;
    unsigned first_block;
};

template <typename SrcT, typename DstT, bool ALONG0>
__global__ __launch_bounds__(64, 2) void iir_pair_lines_batch(const BatchLines *__restrict__ vols,
                                                              const int *__restrict__ vol_of) {
    extern __shared__ double lds[];
    const BatchLines &v = vols[vol_of[blockIdx.x]];
    iir_pair_body<SrcT, DstT, ALONG0>(static_cast<const SrcT *>(v.src), static_cast<DstT *>(v.dst), v.L,
                                      v.k, blockIdx.x - v.first_block, lds);
}

static LineSet lines_for(const sitkhip_geometry &g, int axis) {
    LineSet L;
    long long n0 = static_cast<long long>(g.size[0]);
    long long n1 = static_cast<long long>(g.size[1]);
    long long n2 = static_cast<long long>(g.size[2]);
    long long n = n0 * n1 * n2;
    L.axis = axis;
    L.len = static_cast<int>(g.size[axis]);
    L.nlines = n / static_cast<long long>(g.size[axis]);
    L.n0 = n0;
    L.n01 = n0 * n1;
    L.stride = axis == 0 ? 1 : (axis == 1 ? n0 : n0 * n1);
    return L;
}

static size_t max_lds_per_block() {
    static size_t v = 0;
    if (!v) {
        int a = 0;
        HIP_OK(hipDeviceGetAttribute(&a, hipDeviceAttributeMaxSharedMemoryPerBlock,
                                     backend().device));
        v = static_cast<size_t>(a);
    }
    return v;
}

// Whether the two-lane kernel takes lines of n voxels.
static bool paired(size_t n) {
    return n >= 8 && n < (1u << 30) && pair_lds_bytes(static_cast<int>(n)) <= max_lds_per_block();
}
// A kernel with more than 64 KB of dynamic LDS has to be told so.
static void allow_lds(const void *kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        HIP_OK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(bytes)));
}

// tmp: an FP64 scratch volume the single-lane kernel needs for its causal
// outputs (it may alias dst when DstT is double); the two-lane kernel, used
// whenever its LDS fits, needs none.
template <typename SrcT, typename DstT>
static void launch_axis(const SrcT *src, double *tmp, DstT *dst, const sitkhip_geometry &g, int axis,
                        const IirCoef &k) {
    LineSet L = lines_for(g, axis);
    static const char *names[3] = {"gauss_iir_axis0", "gauss_iir_axis1", "gauss_iir_axis2"};
    if (paired(L.len)) {
        const size_t lds = pair_lds_bytes(L.len);
        const dim3 blocks(static_cast<unsigned>((L.nlines + kPairLines - 1) / kPairLines));
        auto kernel = axis == 0 ? iir_pair_lines<SrcT, DstT, true> : iir_pair_lines<SrcT, DstT, false>;
        allow_lds(reinterpret_cast<const void *>(kernel), lds);
        launch_kernel(names[axis], kernel, blocks, dim3(64), lds, src, dst, L, k);
    } else {
        unsigned blocks = static_cast<unsigned>((L.nlines + 255) / 256);
        launch_kernel(names[axis], iir_lines<SrcT, DstT>, dim3(blocks), dim3(256), 0, src, tmp, dst, L, k);
    }
    check_launch(names[axis]);
}

__global__ void copy_f32(const float *__restrict__ s, float *__restrict__ d, size_t n) {
    size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        d[i] = s[i];
}

// Refusals of recursive_gaussian (recursive_gaussian.rs:171-204): sigma >= 0
// on every axis, and a smoothed axis (sigma > 0) needs at least 4 voxels.
// Returns the smoothed axes in order.
static int smoothed_axes(const sitkhip_geometry &g, const double sigma[3], int axes[3]) {
    for (int d = 0; d < 3; ++d) {
        if (!(sigma[d] >= 0.0))
            fail(SITKHIP_ERR_INVALID_ARGUMENT, "recursive_gaussian: sigma must be >= 0");
    }
    int na = 0;
    for (int d = 0; d < 3; ++d) {
        if (sigma[d] <= 0.0) continue;
        if (g.size[d] < 4)
            fail(SITKHIP_ERR_UNSUPPORTED_GEOMETRY,
                 "recursive_gaussian: axis " + std::to_string(d) + " has " +
                     std::to_string(g.size[d]) + " voxels; the recursion needs at least 4");
        axes[na++] = d;
    }
    return na;
}

// Enqueues the smoothing of `src` (geometry g) into `dst` on the library
// stream. A and B are FP64 volumes of g's voxel count: A is used whenever an
// axis is smoothed, B when two or more are.
static void enqueue_smoothing(const float *src, float *dst, const sitkhip_geometry &g,
                              const double sigma[3], const int axes[3], int na, double *A,
                              double *B) {
    const size_t n = geometry_len(g);
    if (na == 0) {
        launch_kernel("copy_f32", copy_f32, dim3(grid_for(n, 256, 4096)), dim3(256), 0, src, dst, n);
        check_launch("copy_f32");
        return;
    }
    if (na == 1) {
        IirCoef k = zero_order_coefficients(sigma[axes[0]] / g.spacing[axes[0]]);
        launch_axis<float, float>(src, A, dst, g, axes[0], k);
        return;
    }
    // first smoothed axis: f32 -> A (causal outputs land in A itself)
    IirCoef k0 = zero_order_coefficients(sigma[axes[0]] / g.spacing[axes[0]]);
    launch_axis<float, double>(src, A, A, g, axes[0], k0);
    double *cur = A, *other = B;
    for (int a = 1; a < na - 1; ++a) {
        IirCoef k = zero_order_coefficients(sigma[axes[a]] / g.spacing[axes[a]]);
        launch_axis<double, double>(cur, other, other, g, axes[a], k);
        double *t = cur; cur = other; other = t;
    }
    IirCoef kl = zero_order_coefficients(sigma[axes[na - 1]] / g.spacing[axes[na - 1]]);
    launch_axis<double, float>(cur, other, dst, g, axes[na - 1], kl);
}

// recursive_gaussian (pyramid.rs:217-293 / recursive_gaussian.rs:171-204).
Image *recursive_gaussian(const Image &in, const double sigma[3], bool synchronous) {
    int axes[3];
    const int na = smoothed_axes(in.geom, sigma, axes);
    const sitkhip_geometry &g = in.geom;
    size_t n = in.len();
    Image *out = image_like(g);
    try {
        // FP64 intermediates of this call, from the caching allocator: freed
        // at return while the launches are still queued, a block is reused
        // only by later work on the same stream (or held back while work is
        // spread over several streams), so calls on different streams never
        // share one.
        DeviceBuffer<double> A(na >= 1 ? n : 1), B(na >= 2 ? n : 1);
        enqueue_smoothing(in.buf.ptr, out->buf.ptr, g, sigma, axes, na, A.ptr, B.ptr);
        if (synchronous) sync();
    } catch (...) {
        delete out;
        throw;
    }
    return out;
}

// ------------------------------------------------ smoothing without allocation
// The FP64 intermediates of sitkhip_recursive_gaussian_into: two volumes of at
// most kIntoMaxVoxels voxels (2 x 64 MiB), a static device array that every
// device the library runs on holds until the process ends. Host code never
// uses the array's name as an address: the device address of each device's
// copy is looked up once, when the backend is initialised on that device, and
// kept in g_scratch_addr.
constexpr size_t kIntoMaxVoxels = SITKHIP_GAUSSIAN_INTO_MAX_VOXELS;
static __device__ __align__(256) double scratch[2 * kIntoMaxVoxels];
constexpr int kMaxDevices = 64;
static double *g_scratch_addr[kMaxDevices] = {};

void gaussian_scratch_setup(int device) {
    if (device < 0 || device >= kMaxDevices)
        fail(SITKHIP_ERR_NO_DEVICE, "device index " + std::to_string(device) +
                                        " beyond the scratch table of " +
                                        std::to_string(kMaxDevices) + " devices");
    void *p = nullptr;
    HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_addr[device] = static_cast<double *>(p);
}

// recursive_gaussian into a caller's image through the static scratch: no
// device allocation. Every call on one device shares that device's scratch.
static void recursive_gaussian_into(const Image &in, const double sigma[3], Image &out) {
    int axes[3];
    const int na = smoothed_axes(in.geom, sigma, axes);
    if (!same_geometry(in.geom, out.geom))
        fail(SITKHIP_ERR_INVALID_ARGUMENT,
             "recursive_gaussian_into: the output image's geometry is not the input's");
    if (in.buf.ptr == out.buf.ptr)
        fail(SITKHIP_ERR_INVALID_ARGUMENT,
             "recursive_gaussian_into: the output image is the input image");
    const size_t n = in.len();
    if (n > kIntoMaxVoxels)
        fail(SITKHIP_ERR_INVALID_ARGUMENT,
             "recursive_gaussian_into: " + std::to_string(n) + " voxels exceed the " +
                 std::to_string(kIntoMaxVoxels) + " its scratch holds");
    const int dev = backend().device;
    double *base = (dev >= 0 && dev < kMaxDevices) ? g_scratch_addr[dev] : nullptr;
    if (!base)
        fail(SITKHIP_ERR_DRIVER, "recursive_gaussian_into: scratch not set up on device " +
                                     std::to_string(dev));
    enqueue_smoothing(in.buf.ptr, out.buf.ptr, in.geom, sigma, axes, na, base,
                      base + kIntoMaxVoxels);
    sync();
}

// ----------------------------------------------------------- batched volumes
// One axis of a batch's smoothing: every volume's lines, and which volume each
// workgroup takes.
struct AxisBatch {
    std::vector<BatchLines> vols;
    std::vector<int> vol_of;
    size_t lds = 0;
    void add(const void *src, void *dst, const sitkhip_geometry &g, int axis, double sigma) {
        BatchLines v;
        v.src = src;
        v.dst = dst;
        v.L = lines_for(g, axis);
        v.k = zero_order_coefficients(sigma / g.spacing[axis]);
        v.first_block = static_cast<unsigned>(vol_of.size());
        vol_of.insert(vol_of.end(), static_cast<size_t>((v.L.nlines + kPairLines - 1) / kPairLines),
                      static_cast<int>(vols.size()));
        lds = std::max(lds, pair_lds_bytes(v.L.len));
        vols.push_back(v);
    }
};

template <typename SrcT, typename DstT>
static void launch_axis_batch(const AxisBatch &b, const BatchLines *vols, const int *vol_of, int axis) {
    static const char *names[3] = {"gauss_iir_axis0", "gauss_iir_axis1", "gauss_iir_axis2"};
    auto kernel = axis == 0 ? iir_pair_lines_batch<SrcT, DstT, true> : iir_pair_lines_batch<SrcT, DstT, false>;
    allow_lds(reinterpret_cast<const void *>(kernel), b.lds);
    launch_kernel(names[axis], kernel, dim3(static_cast<unsigned>(b.vol_of.size())), dim3(64), b.lds, vols,
                  vol_of);
    check_launch(names[axis]);
}

// recursive_gaussian of many volumes, smoothing all three axes of each
// (sigma[i] > 0 on every axis): three launches per group of volumes whose
// FP64 intermediates fit a 1 GiB budget, the per-line arithmetic that of the
// one-volume path (so the results are the same bits). Volumes the paired-lane
// kernel cannot take (an axis shorter than 8 voxels, or lines whose LDS does
// not fit) go through recursive_gaussian one by one. Asynchronous.
std::vector<Image *> recursive_gaussian_batch(const std::vector<const Image *> &in,
                                              const std::vector<std::array<double, 3>> &sigma) {
    const size_t n = in.size();
    std::vector<Image *> out(n, nullptr);
    try {
        std::vector<size_t> group;
        size_t group_bytes = 0;
        auto flush = [&]() {
            if (group.empty()) return;
            std::vector<DeviceBuffer<double>> A(group.size()), B(group.size());
            AxisBatch axes[3];
            for (size_t j = 0; j < group.size(); ++j) {
                const size_t i = group[j];
                const sitkhip_geometry &g = in[i]->geom;
                A[j].alloc(in[i]->len());
                B[j].alloc(in[i]->len());
                out[i] = image_like(g);
                axes[0].add(in[i]->buf.ptr, A[j].ptr, g, 0, sigma[i][0]);
                axes[1].add(A[j].ptr, B[j].ptr, g, 1, sigma[i][1]);
                axes[2].add(B[j].ptr, out[i]->buf.ptr, g, 2, sigma[i][2]);
            }
            // the three axes' tables in one copy ahead of the three launches
            // (volumes first: they hold pointers)
            size_t at[3][2], bytes = 0;
            for (int k = 0; k < 2; ++k)
                for (int d = 0; d < 3; ++d) {
                    at[d][k] = bytes;
                    bytes += k == 0 ? axes[d].vols.size() * sizeof(BatchLines)
                                    : axes[d].vol_of.size() * sizeof(int);
                }
            std::vector<unsigned char> host(bytes);
            for (int d = 0; d < 3; ++d) {
                std::memcpy(host.data() + at[d][0], axes[d].vols.data(),
                            axes[d].vols.size() * sizeof(BatchLines));
                std::memcpy(host.data() + at[d][1], axes[d].vol_of.data(),
                            axes[d].vol_of.size() * sizeof(int));
            }
            DeviceBuffer<unsigned char> dev(bytes);
            dev.upload(host.data(), bytes);
            auto vols = [&](int d) { return reinterpret_cast<const BatchLines *>(dev.ptr + at[d][0]); };
            auto vol_of = [&](int d) { return reinterpret_cast<const int *>(dev.ptr + at[d][1]); };
            launch_axis_batch<float, double>(axes[0], vols(0), vol_of(0), 0);
            launch_axis_batch<double, double>(axes[1], vols(1), vol_of(1), 1);
            launch_axis_batch<double, float>(axes[2], vols(2), vol_of(2), 2);
            group.clear();
            group_bytes = 0;
        };
        for (size_t i = 0; i < n; ++i) {
            const sitkhip_geometry &gi = in[i]->geom;
            bool ok = true;
            for (int d = 0; d < 3; ++d) {
                if (!(sigma[i][d] > 0.0) || !paired(gi.size[d])) ok = false;
            }
            if (!ok) {
                out[i] = recursive_gaussian(*in[i], sigma[i].data(), false);
                continue;
            }
            const size_t bytes = in[i]->len() * 2 * sizeof(double);
            if (!group.empty() && group_bytes + bytes > (static_cast<size_t>(1) << 30)) flush();
            group.push_back(i);
            group_bytes += bytes;
        }
        flush();
    } catch (...) {
        for (Image *p : out) delete p;
        throw;
    }
    return out;
}
}  // namespace sitkhip

extern "C" int sitkhip_recursive_gaussian_batch(size_t n, const sitkhip_image *in,
                                                const double *sigma, sitkhip_image *out) {
    return sitkhip::run_guarded([&] {
        if (n == 0) return;
        if (!in || !sigma || !out) sitkhip::fail(SITKHIP_ERR_INVALID_ARGUMENT, "null array");
        std::vector<const sitkhip::Image *> imgs(n);
        std::vector<std::array<double, 3>> sig(n);
        for (size_t i = 0; i < n; ++i) {
            imgs[i] = reinterpret_cast<const sitkhip::Image *>(in[i]);
            if (!imgs[i]) sitkhip::fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image");
            for (int d = 0; d < 3; ++d) {
                sig[i][d] = sigma[3 * i + d];
                if (!(sig[i][d] >= 0.0))
                    sitkhip::fail(SITKHIP_ERR_INVALID_ARGUMENT, "recursive_gaussian: sigma must be >= 0");
            }
        }
        std::vector<sitkhip::Image *> res = sitkhip::recursive_gaussian_batch(imgs, sig);
        sitkhip::sync();
        for (size_t i = 0; i < n; ++i) out[i] = reinterpret_cast<sitkhip_image>(res[i]);
    });
}

extern "C" int sitkhip_recursive_gaussian_into(sitkhip_image in, const double sigma[3],
                                               sitkhip_image out) {
    return sitkhip::run_guarded([&] {
        auto src = reinterpret_cast<sitkhip::Image *>(in);
        auto dst = reinterpret_cast<sitkhip::Image *>(out);
        if (!src || !sigma || !dst)
            sitkhip::fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image or sigma");
        sitkhip::recursive_gaussian_into(*src, sigma, *dst);
    });
}

extern "C" int sitkhip_recursive_gaussian(sitkhip_image in, const double sigma[3],
                                          sitkhip_image *out) {
    return sitkhip::run_guarded([&] {
        auto img = reinterpret_cast<sitkhip::Image *>(in);
        if (!img || !sigma || !out)
            sitkhip::fail(SITKHIP_ERR_INVALID_ARGUMENT, "null image, sigma or out-pointer");
        *out = reinterpret_cast<sitkhip_image>(sitkhip::recursive_gaussian(*img, sigma, true));
    });
}
