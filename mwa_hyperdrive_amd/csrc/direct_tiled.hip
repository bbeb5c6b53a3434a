// Faster FP64 direct kernels for the common case: one beam shared by every tile (or no
// beam) and evenly spaced channels.
//
// k_tiles_mfma (points, Gaussians): a block owns up to 16 x 16 tile pairs and one chunk of
// channels. The baseline phase factorises over antennas,
//   e^{i theta_pq f/c} = e^{i theta_p f/c} e^{-i theta_q f/c},  theta_t = u_t L + v_t M + w_t N,
// (baseline uvw = tile1 - tile2, mdbook/src/defs/coords.md), so per component the block
// evaluates the phasors of its 32 tiles (middle channel and channel step) into LDS (64
// sincos shared by 256 baselines instead of 512), each lane forms its baseline's phasors from
// them, and the FP64 matrix cores multiply them by the coherencies. Diagonal tile blocks are
// paired so that 240 of 256 pairs are wanted ones. k_direct_tiled keeps the products on the vector
// ALUs: the precision path's FP32 Gaussians, and few components in FP64.
//
// k_rect_mfma does the same for pairs of a tile with its own beam and one of the shared beam.
//
// k_shapelets (shapelets, FP64): the coefficient sums are formed once per run of channels within a
// cell of the basis table. k_shapelet_chan_tiles (per-tile beams whose runs hold few channels),
// k_shapelet_chan_tiles32 and k_shapelet_chan32 (FP32): one wave per baseline, one or two channels per lane;
// the table positions x_pos = k f + 5000 of neighbouring channels fall in the same or adjacent table cells, so
// each coefficient's table reads coalesce across the wave instead of touching 64 unrelated cache lines.
#include "sm_internal.h"
#include "sm_jones.h"
#include "sm_math.h"
#include "sm_tiled.h"

namespace sm {

constexpr int kTG = 16;   // tiles per group
constexpr int kWin = 32;  // shapelet table window per wave and axis, cells
constexpr int kRows = 16; // shapelet table rows staged per wave
constexpr int kWinPair = 24;  // shapelet table window per wave and axis of the two-channel kernel, cells
constexpr int kCT = 32;   // components per LDS stage
// Channels per lane in k_direct_tiled. FP32 Gaussians, measured per timestep of 256 tiles,
// 384 channels and 10 000 Gaussians: 78.4 ms with 4, 76.2 ms with 6 (142 VGPRs), 115.9 ms with 8.
constexpr int kTiledNchGaussian = 6;
constexpr int kTiledNchPoint = 8;
static_assert(kTiledNchGaussian <= SM_NCH && kTiledNchPoint <= SM_NCH, "the padded channel count covers whole chunks of SM_NCH channels");

// The kernels below come in two arithmetic types T. double: the FP64 direct kernels. float:
// the precision path's kernels, in which the phases, their range reduction mod 2 pi, the table
// positions of shapelets and the Gaussian exponents are still formed in FP64, and everything
// after (phasor products, envelopes, coherency products, accumulation) runs in FP32.
template <class T> struct Vec4;
template <> struct Vec4<double> { using type = double4; };
template <> struct Vec4<float> { using type = float4; };

__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// e^x of an FP64 argument: FP64 exp, or the hardware base-2 exponential in FP32 (an argument
// below the FP32 range gives 0).
__device__ __forceinline__ void exp_of(double x, double &out) { out = exp(x); }
__device__ __forceinline__ void exp_of(double x, float &out) {
    out = __builtin_amdgcn_exp2f((float)(x * 1.4426950408889634));
}

// sin and cos of an FP64 phase in the kernel's arithmetic (the shapelet kernel's per-channel
// phases). FP64: table_sincos. FP32: x is reduced mod pi/2 in FP64 exactly as fast_sincos does,
// and the reduced |r| <= pi/4 goes through the Taylor series of sin to r^9 and of cos to r^10
// in FP32 (truncation below 2e-9, under the FP32 rounding).
__device__ __forceinline__ void sincos_phase(double x, double &s, double &c) { table_sincos(x, kSinCos32, s, c); }
__device__ __forceinline__ void sincos_phase(double x, float &s, float &c) {
    const double k = rint(x * 0.6366197723675814);
    double r = fma(-k, 1.5707963267948966, x);
    r = fma(-k, 6.123233995736766e-17, r);
    const float rf = (float)r, r2 = rf * rf;
    // coefficients (-1)^n / (2n+1)! and (-1)^n / (2n)!
    float ps = 2.7557319e-06f;
    ps = __builtin_fmaf(ps, r2, -1.9841270e-04f);
    ps = __builtin_fmaf(ps, r2, 8.3333333e-03f);
    ps = __builtin_fmaf(ps, r2, -1.6666667e-01f);
    const float sn = __builtin_fmaf(rf * r2, ps, rf);
    float pc = -2.7557319e-07f;
    pc = __builtin_fmaf(pc, r2, 2.4801587e-05f);
    pc = __builtin_fmaf(pc, r2, -1.3888889e-03f);
    pc = __builtin_fmaf(pc, r2, 4.1666667e-02f);
    pc = __builtin_fmaf(pc, r2, -0.5f);
    const float cn = __builtin_fmaf(r2, pc, 1.0f);
    const int q = (int)(long long)k & 3;
    const float a = (q & 1) ? cn : sn;  // sin x = sin r, cos r, -sin r, -cos r for q = 0..3
    const float b = (q & 1) ? sn : cn;  // cos x = cos r, -sin r, -cos r, sin r
    s = (q & 2) ? -a : a;
    c = ((q + 1) & 2) ? -b : b;
}

// FP32 kernels sum in two levels: a stage's components (at most 32) add into the inner
// accumulators, which are then added into the outer ones, so the rounding of a sum over N
// components grows like sqrt(N / stage) rather than sqrt(N). FP64 kernels sum in one level.
template <class T> struct TwoLevel { static constexpr bool on = false; };
template <> struct TwoLevel<float> { static constexpr bool on = true; };

template <class T, int N>
__device__ __forceinline__ void flush_stage(T (&acc)[N][8], T (&tot)[N][8]) {
    if (!TwoLevel<T>::on) return;
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            tot[k][e] += acc[k][e];
            acc[k][e] = T(0);
        }
}

template <class T> __device__ __forceinline__ T two_level_sum(T acc, T tot) { return TwoLevel<T>::on ? tot + acc : acc; }

template <class T> __device__ __forceinline__ const T *pick(const double *d, const float *f);
template <> __device__ __forceinline__ const double *pick<double>(const double *d, const float *) { return d; }
template <> __device__ __forceinline__ const float *pick<float>(const double *, const float *f) { return f; }

// Tile pairs on the vector units: a lane per pair, NCH channels. float: the precision path's Gaussians
// (phases and exponents in FP64). double: few components on many blocks with FP32 visibilities alone, where
// reading and adding to the visibilities is most of the time: a lane moves all 32 bytes of one, k_tiles_mfma's
// 8. 128 tiles, 768 channels, 1 and 7 Gaussians 66 and 82 us (5.9 TB/s), on k_tiles_mfma 100 and 108; 384
// channels, 2 points 39 and 44.
template <int KIND, int NCH, class T>
__global__ __launch_bounds__(256) void k_direct_tiled(const TiledArgs a) {
    using V4 = typename Vec4<T>::type;
    __shared__ V4 s_ph[kCT][32];
    __shared__ double s_uvw[32][3];
    const int total = a.npairs * a.nchunks;
    int b = blockIdx.x;
    if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
    const int chunk = b / a.npairs;
    int f0, cnt;
    chunk_range<NCH>(a.chunks, chunk, a.nchan, f0, cnt);
    const int4 pr = a.pairs[b - chunk * a.npairs];
    const int tid = threadIdx.x, r = tid >> 4, cq = tid & 15;
    if (tid < 32) {
        const int g = tid < 16 ? pr.y : pr.z;
        int t = g * kTG + (tid & 15);
        if (g < 0 || t >= a.ntiles) t = 0;
        s_uvw[tid][0] = a.tile_uvw[3 * t];
        s_uvw[tid][1] = a.tile_uvw[3 * t + 1];
        s_uvw[tid][2] = a.tile_uvw[3 * t + 2];
    }
    int p, q, sp, sq;
    bool valid;
    if (pr.x == 0) {
        p = pr.y * kTG + r;
        q = pr.z * kTG + cq;
        sp = r;
        sq = 16 + cq;
        valid = q < a.ntiles;
    } else if (r < cq) {
        p = pr.y * kTG + r;
        q = pr.y * kTG + cq;
        sp = r;
        sq = cq;
        valid = q < a.ntiles;
    } else if (r > cq && pr.z >= 0) {
        p = pr.z * kTG + cq;
        q = pr.z * kTG + r;
        sp = 16 + cq;
        sq = 16 + r;
        valid = q < a.ntiles;
    } else {
        p = 0;
        q = 1;
        sp = 0;
        sq = 1;
        valid = false;
    }
    __syncthreads();
    const double bu = s_uvw[sp][0] - s_uvw[sq][0];
    const double bv = s_uvw[sp][1] - s_uvw[sq][1];

    const double *__restrict__ freqs = a.freqs;
    const double F0 = freqs[f0];
    const double DF = freqs[f0 + 1] - F0;
    const double f0c = F0 / SM_VEL_C;
    const double dfc = DF / SM_VEL_C;
    const T *__restrict__ coh = pick<T>(a.coh, a.coh32);
    const double4 *__restrict__ lmn4 = a.lmn;
    const double4 *__restrict__ shape = a.shape;

    T acc[NCH][8], tot[NCH][8];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[k][e] = tot[k][e] = T(0);

    for (int c0 = 0; c0 < a.ncomp; c0 += kCT) {
        const int nc = a.ncomp - c0 < kCT ? a.ncomp - c0 : kCT;
        // Per-tile phasors (start, step) of this stage's components, phases reduced in FP64.
        for (int e = tid; e < kCT * 32; e += 256) {
            const int slot = e & 31, cc = e >> 5;
            double ps = 0.0, pc = 1.0, qs = 0.0, qc = 1.0;
            if (cc < nc) {
                const double4 l = lmn4[c0 + cc];
                const double th = s_uvw[slot][0] * l.x + s_uvw[slot][1] * l.y + s_uvw[slot][2] * l.z;
                table_sincos(th * f0c, kSinCos32, ps, pc);
                table_sincos(th * dfc, kSinCos32, qs, qc);
            }
            V4 ph;
            ph.x = (T)pc;
            ph.y = (T)ps;
            ph.z = (T)qc;
            ph.w = (T)qs;
            s_ph[cc][slot] = ph;
        }
        __syncthreads();
        for (int cc = 0; cc < nc; ++cc) {
            const int c = c0 + cc;
            const V4 A = s_ph[cc][sp];
            const V4 B = s_ph[cc][sq];
            T zr = A.x * B.x + A.y * B.y;
            T zi = A.y * B.x - A.x * B.y;
            const T rr = A.z * B.z + A.w * B.w;
            const T ri = A.w * B.z - A.z * B.w;
            T env = T(1), er = T(1), eg = T(1);
            if (KIND == KIND_GAUSSIAN) {
                const double4 g = shape[c];
                const double qf = g.x * (bu * bu) + g.y * (bu * bv) + g.z * (bv * bv);
                exp_of(qf * (F0 * F0), env);
                exp_of(qf * (DF * (2.0 * F0 + DF)), er);
                exp_of(qf * (2.0 * DF * DF), eg);
            }
            // The table is the Hermitian form (Re XX, Re XY, Im XY, Re YY) of J S J^H (see
            // TiledArgs), 32 contiguous bytes per channel. Per visibility: V_XX = sum C_XX z,
            // A = sum Re(C_XY) z, B = sum Im(C_XY) z, V_YY = sum C_YY z (8 FMAs per component
            // instead of 16); V_XY = A + i B and V_YX = A - i B are formed once at the end.
            const T *cc4 = coh + ((size_t)c * a.nchan_pad + f0) * 4;
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                T pr_ = zr, pi_ = zi;
                if (KIND == KIND_GAUSSIAN) {
                    pr_ *= env;
                    pi_ *= env;
                }
                const T cxx = cc4[k * 4], cxyr = cc4[k * 4 + 1], cxyi = cc4[k * 4 + 2], cyy = cc4[k * 4 + 3];
                acc[k][0] = fma_t(cxx, pr_, acc[k][0]);
                acc[k][1] = fma_t(cxx, pi_, acc[k][1]);
                acc[k][2] = fma_t(cxyr, pr_, acc[k][2]);
                acc[k][3] = fma_t(cxyr, pi_, acc[k][3]);
                acc[k][4] = fma_t(cxyi, pr_, acc[k][4]);
                acc[k][5] = fma_t(cxyi, pi_, acc[k][5]);
                acc[k][6] = fma_t(cyy, pr_, acc[k][6]);
                acc[k][7] = fma_t(cyy, pi_, acc[k][7]);
                const T nr = zr * rr - zi * ri;
                zi = zr * ri + zi * rr;
                zr = nr;
                if (KIND == KIND_GAUSSIAN) {
                    env *= er;
                    er *= eg;
                }
            }
        }
        flush_stage(acc, tot);
        __syncthreads();
    }
    if (!valid) return;
    if (a.tile_map != nullptr) {
        p = a.tile_map[p];
        q = a.tile_map[q];
    }
    const size_t nt = a.tile_map != nullptr ? (size_t)a.ntiles_bl : (size_t)a.ntiles;
    const size_t bl = (size_t)p * nt - (size_t)p * (p + 1) / 2 + (size_t)(q - p - 1);
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int f = f0 + k;
        if (k >= cnt) break;
        const size_t o = (size_t)f * a.nbl + bl;
        T s8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) s8[e] = two_level_sum(acc[k][e], tot[k][e]);
        // XX, XY = A + i B, YX = A - i B, YY.
        const T v[8] = {s8[0], s8[1], s8[2] - s8[5], s8[3] + s8[4], s8[2] + s8[5], s8[3] - s8[4], s8[6], s8[7]};
        float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v32[e] += (float)v[e];
        if (a.vis64 != nullptr) {
            double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v64[e] += (double)v[e];
        }
    }
}

// ------------------------------------------------------------------ FP64 tile pairs on MFMA
// One visibility is V^e = sum_c C^e_c z_c over the four real coefficients e of the Hermitian
// coherency: an N x K by K x 4 product with K the components and N the real and imaginary
// parts of the baselines' phasors. v_mfma_f64_4x4x4 computes four such 4 x 4 x 4 blocks: lane l
// supplies z of component l / 16 and baseline 4 (l % 4) + (l / 4) % 4 and C^{l % 4} of component
// l / 16, and accumulates e = l % 4 of baseline l / 4: a wave's stores are contiguous. The vector
// ALUs only form z.

// Lane `lane`'s value of v (every lane active), as a wave-uniform value.
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// A frequency over c in two doubles, kept in scalar registers (the same on every lane).
__device__ __forceinline__ TwoDouble over_c(double f) {
    const TwoDouble q = two_quotient(f, SM_VEL_C);
    return {readlane_f64(q.hi, 0), readlane_f64(q.lo, 0)};
}

// z of the chunk's channels from the middle one outwards in both directions: evenly spaced
// channels obey z_{k+1} = 2 cos(delta) z_k - z_{k-1}, one FMA per part, and starting in the middle
// keeps the recurrence's error growth to (NCH / 2)^2 roundings. (a0, b0) are the tiles' phasors at
// channel NCH / 2 - 1, (a1, b1) at one channel step's frequency. Neither phase may be rounded to one
// double (table_sincos_product): a run of two channels across a gap of the band starts NCH / 2 - 1 gaps
// above its first channel, where such a rounding is several times the first channel's, and the step's
// is carried back as often (100 and 300 MHz, tiles within 3 km: rms error of z 1.5e-12 with rounded
// phases, 1.9e-13 without, as on any other band; most of that is theta's own rounding).
template <int NCH>
__device__ __forceinline__ void chunk_phasors(double2 a0, double2 a1, double2 b0, double2 b1, double (&zr)[NCH],
                                              double (&zi)[NCH]) {
    constexpr int m = NCH / 2 - 1;
    zr[m] = fma(a0.x, b0.x, a0.y * b0.y);
    zi[m] = fma(a0.y, b0.x, -(a0.x * b0.y));
    const double rr = fma(a1.x, b1.x, a1.y * b1.y), ri = fma(a1.y, b1.x, -(a1.x * b1.y));
    zr[m + 1] = fma(zr[m], rr, -(zi[m] * ri));
    zi[m + 1] = fma(zr[m], ri, zi[m] * rr);
    const double c2 = 2.0 * rr;
#pragma unroll
    for (int k = m + 2; k < NCH; ++k) {
        zr[k] = fma(c2, zr[k - 1], -zr[k - 2]);
        zi[k] = fma(c2, zi[k - 1], -zi[k - 2]);
    }
#pragma unroll
    for (int k = m - 1; k >= 0; --k) {
        zr[k] = fma(c2, zr[k + 1], -zr[k + 2]);
        zi[k] = fma(c2, zi[k + 1], -zi[k + 2]);
    }
}

// z of the chunk's channels times a Gaussian's envelope e^{q f^2}, q = A u^2 + B u v + C v^2 (sh), by its
// ratios from channel to channel: q0, q1 and q2 are f^2 at the first channel and its first and second
// differences, qmin the q below which the envelope is 0 at every channel (e^-800 underflows).
template <int NCH, bool NARROW>
__device__ __forceinline__ void gaussian_envelopes(double4 sh, double bu, double bv, double qmin, double q0, double q1,
                                                   double q2, const double *s_exp, double (&zr)[NCH], double (&zi)[NCH]) {
    double qf = sh.x * (bu * bu) + sh.y * (bu * bv) + sh.z * (bv * bv);
    qf = qf < qmin ? qmin : qf;
    double env = table_exp(qf * q0, s_exp);
    // Descending channels give a positive exponent; the cap keeps 0 * er at 0.
    double er = table_exp(NARROW ? qf * q1 : fmin(qf * q1, 700.0), s_exp);
    const double eg = NARROW ? small_exp(qf * q2) : table_exp(qf * q2, s_exp);
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        zr[k] *= env;
        zi[k] *= env;
        env *= er;
        er *= eg;
    }
}

// What bounds it: FP64 issue. The matrix and vector FP64 instructions share one unit (16 FMAs
// and 16 MFMAs per wave, measured: 36 and 111 ns apart, 141 ns together), which sustains 75
// TFLOP/s on this MFMA against 62 on FMAs (the clock falls to 2.07 GHz under FMAs). A component
// visibility's 8 accumulating FMAs become 2/64 MFMAs and the phasor's 4-instruction rotation the 2
// FMAs of the recurrence. At 128 tiles, 768 channels: 5600 points 18.0 -> 13.7 ms (MFMA 53% and
// other VALU 34% of the cycles, at 2.05 GHz), 2000 Gaussians 12.9 -> 7.8 ms (their exponentials
// through table_exp: 10.1 -> 8.6 ms). Two waves per SIMD: the accumulators take 128 VGPRs. Four
// waves of half the accumulators spill and run slower (15.5 and 23.7 ms). Points in the 4-channel form
// are held to 128 VGPRs, two blocks a CU.
//
// A block owns R = NG * WR rows of one 16 x 16 tile-pair block and one chunk of at most NCH
// channels. WR waves split the rows (NG each); WC waves split the components (each takes every
// WC-th group of four of a stage), their sums meeting in LDS at the end. A chunk's coherencies are
// read NCH wide whatever its count (TiledArgs::coh); what the extra channels accumulate is dropped.
template <int KIND, int NCH, int NG, int WR, int WC, bool NARROW, bool SLICED>
__global__ __launch_bounds__(64 * WR * WC, KIND == KIND_POINT && NCH == 4 ? 4 : 2) void k_tiles_mfma(const TiledArgs a) {
    constexpr int R = NG * WR, SUB = kTG / R, NT = 64 * WR * WC;
    static_assert(kCT % (4 * WC) == 0, "a stage is whole groups of four components per wave");
    constexpr int KR = WC > 1 ? WC / NG : 1;  // channels reduced at a time (WC > 1)
    struct Stage {
        double2 p0[kCT][32], p1[kCT][32];  // tile phasors: the chunk's middle channel, one channel step
        double c[kCT][NCH * 4 + 4];        // coherencies; the padding puts components on distinct banks
    };
    union Lds {
        Stage st;
        double red[WC > 1 ? WC : 1][KR][NG][2][64];
    };
    __shared__ Lds L;
    __shared__ double2 s_uv[32];
    __shared__ double s_w[32];
    __shared__ double2 s_sc[64];
    __shared__ double s_exp[64];
    const int per_slice = a.npairs * a.nchunks * SUB;
    const int total = per_slice * (SLICED ? a.slices : 1);
    int b = blockIdx.x;
    if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
    const int slice = SLICED ? b / per_slice : 0;  // of the components
    b -= slice * per_slice;
    const int c_begin = slice * a.slice_len;
    const int c_end = SLICED ? min(a.ncomp, c_begin + a.slice_len) : a.ncomp;
    const int chunk = b / (a.npairs * SUB);
    int f0, cnt;
    chunk_range<NCH>(a.chunks, chunk, a.nchan, f0, cnt);
    const int rem = b - chunk * (a.npairs * SUB);
    const int row0 = (rem % SUB) * R;
    const int4 pr = a.pairs[rem / SUB];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wr = wave % WR, wc = wave / WR;
    const int cq = 4 * (lane & 3) + ((lane >> 2) & 3), ck = lane >> 4;
    if (tid < 32) {
        const int g = tid < 16 ? pr.y : pr.z;
        int t = g * kTG + (tid & 15);
        if (g < 0 || t >= a.ntiles) t = 0;
        s_uv[tid] = make_double2(a.tile_uvw[3 * t], a.tile_uvw[3 * t + 1]);
        s_w[tid] = a.tile_uvw[3 * t + 2];
    }
    if (tid < 64) {
        s_sc[tid] = make_double2(kSinCos32[2 * tid], kSinCos32[2 * tid + 1]);
        if (KIND == KIND_GAUSSIAN) s_exp[tid] = kExp64[tid];
    }
    // Tile slots of each (row, column): off-diagonal blocks pair group y's tile r with group
    // z's tile cq; diagonal blocks hold group y's pairs above the diagonal and group z's below.
    int sp[NG], sq[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int r = row0 + wr * NG + g;
        const bool lower = pr.x != 0 && r > cq;
        sp[g] = lower ? 16 + cq : r;
        sq[g] = pr.x == 0 ? 16 + cq : (lower ? 16 + r : cq);
    }
    // Slots this block reads: its rows and group z's columns, or (diagonal) all of them.
    const int nslot = pr.x == 0 ? R + 16 : 32;
    __syncthreads();
    const double *__restrict__ freqs = a.freqs;
    const double F0 = freqs[f0];
    const double DF = freqs[f0 + 1] - F0;
    constexpr int m = NCH / 2 - 1;
    const TwoDouble fm0 = over_c(F0 + m * DF), fm1 = over_c(DF);
    const double4 *__restrict__ lmn4 = a.lmn;
    const double4 *__restrict__ shape = a.shape;
    const double *__restrict__ coh = a.coh + (size_t)f0 * 4;
    const size_t cstride = (size_t)a.nchan_pad * 4;
    const double qmin = -800.0 / (F0 * F0), q0 = F0 * F0, q1 = DF * (2.0 * F0 + DF), q2 = 2.0 * DF * DF;

    double acc[NCH][NG][2];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[k][g][0] = acc[k][g][1] = 0.0;

    for (int c0 = c_begin; c0 < c_end; c0 += kCT) {
        const int nc = min(kCT, c_end - c0);
        const int nc4 = (nc + 3) & ~3;  // components past the last are staged as 0
        for (int e = tid; e < nc4 * (NCH * 2); e += NT) {
            const int cc = e / (NCH * 2), i = e % (NCH * 2);
            double2 v = make_double2(0.0, 0.0);
            if (cc < nc) v = reinterpret_cast<const double2 *>(coh + (size_t)(c0 + cc) * cstride)[i];
            *reinterpret_cast<double2 *>(&L.st.c[cc][2 * i]) = v;
        }
#pragma unroll 2
        for (int e = tid; e < nc4 * nslot; e += NT) {
            const int cc = e / nslot, i = e - cc * nslot;
            const int slot = pr.x != 0 ? i : (i < R ? row0 + i : i - R + 16);
            double s0 = 0.0, c0_ = 0.0, s1 = 0.0, c1 = 0.0;
            if (cc < nc) {
                const double4 l = lmn4[c0 + cc];
                const double2 uv = s_uv[slot];
                const double th = uv.x * l.x + uv.y * l.y + s_w[slot] * l.z;
                table_sincos_product(th, fm0, reinterpret_cast<const double *>(s_sc), s0, c0_);
                table_sincos_product(th, fm1, reinterpret_cast<const double *>(s_sc), s1, c1);
            }
            L.st.p0[cc][slot] = make_double2(c0_, s0);
            L.st.p1[cc][slot] = make_double2(c1, s1);
        }
        __syncthreads();
#pragma unroll 2
        for (int cs = 4 * wc; cs < nc; cs += 4 * WC) {
            const int cc = cs + ck;
            double A[NCH];
#pragma unroll
            for (int k = 0; k < NCH; ++k) A[k] = L.st.c[cc][4 * k + (lane & 3)];
            double4 sh = make_double4(0.0, 0.0, 0.0, 0.0);
            if (KIND == KIND_GAUSSIAN) sh = shape[min(c0 + cc, a.ncomp - 1)];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                double zr[NCH], zi[NCH];
                chunk_phasors<NCH>(L.st.p0[cc][sp[g]], L.st.p1[cc][sp[g]], L.st.p0[cc][sq[g]], L.st.p1[cc][sq[g]], zr,
                                   zi);
                if (KIND == KIND_GAUSSIAN) {
                    const double2 tp = s_uv[sp[g]], tq = s_uv[sq[g]];
                    const double bu = tp.x - tq.x, bv = tp.y - tq.y;
                    gaussian_envelopes<NCH, NARROW>(sh, bu, bv, qmin, q0, q1, q2, s_exp, zr, zi);
                }
#pragma unroll
                for (int k = 0; k < NCH; ++k) {
                    acc[k][g][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(zr[k], A[k], acc[k][g][0], 0, 0, 0);
                    acc[k][g][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(zi[k], A[k], acc[k][g][1], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    // Lane l holds (re, im) of coefficient l % 4 for baseline l / 4 of its row: lanes of A = sum
    // Re(C_XY) z and B = sum Im(C_XY) z exchange them (lane ^ 3) for XY = A + i B and YX = A - i B,
    // and each lane adds to one of the visibility's four entries, 512 contiguous bytes per wave. The
    // entries of several channels are read before the first is written, or each would wait for its
    // own: 2 points on 384 channels 114 -> 58 us, with 16 separate spans per wave instruction before.
    const int sc = lane >> 2, se = lane & 3;
    const size_t fstride = 4 * (SLICED ? (size_t)a.ntiles * (a.ntiles - 1) / 2 : (size_t)a.nbl);
    auto entry = [&](int g, size_t &o) {  // the lane's entry of row g at channel f0; whether there is one
        const int r = row0 + wr * NG + g;
        int p, q;
        bool valid;
        if (pr.x == 0) {
            p = pr.y * kTG + r;
            q = pr.z * kTG + sc;
            valid = q < a.ntiles;
        } else if (r < sc) {
            p = pr.y * kTG + r;
            q = pr.y * kTG + sc;
            valid = q < a.ntiles;
        } else {
            p = pr.z * kTG + sc;
            q = pr.z * kTG + r;
            valid = r > sc && pr.z >= 0 && q < a.ntiles;
        }
        if (!valid) p = 0, q = 1;
        if (!SLICED && a.tile_map != nullptr) {
            p = a.tile_map[p];
            q = a.tile_map[q];
        }
        const size_t nt = !SLICED && a.tile_map != nullptr ? (size_t)a.ntiles_bl : (size_t)a.ntiles;
        const size_t bl = (size_t)p * nt - (size_t)p * (p + 1) / 2 + (size_t)(q - p - 1);
        o = (f0 * (fstride / 4) + bl) * 4 + se;
        return valid;
    };
    float2 *const vis32 = reinterpret_cast<float2 *>(a.vis32);
    double2 *const vis64 = reinterpret_cast<double2 *>(a.vis64);
    auto value = [&](double re, double im) {
        const double ore = __shfl_xor(re, 3), oim = __shfl_xor(im, 3);
        return make_double2(se == 1 ? re - oim : (se == 2 ? ore + im : re), se == 1 ? im + ore : (se == 2 ? oim - re : im));
    };
    auto add = [&](bool on, size_t o, float2 t, double2 d, double re, double im) {
        const double2 v = value(re, im);
        const double vr = v.x, vi = v.y;
        if (!on) return;
        vis32[o] = make_float2(t.x + (float)vr, t.y + (float)vi);
        if (vis64 != nullptr) vis64[o] = make_double2(d.x + vr, d.y + vi);
    };
    if (SLICED) {
        static_assert(!SLICED || WC == 1, "one wave has a component's sums");
        // This slice's sums; k_tiles_finish adds the slices to the visibilities.
        double2 *const out = a.part + (size_t)slice * a.nchan * fstride;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            size_t o;
            const bool valid = entry(g, o);
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                const double2 v = value(acc[k][g][0], acc[k][g][1]);
                if (valid && k < cnt) out[o + k * fstride] = v;
            }
        }
    } else if (WC == 1) {
        constexpr int KB = 8;  // channels read at a time
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            size_t o;
            const bool valid = entry(g, o);
#pragma unroll
            for (int k0 = 0; k0 < NCH; k0 += KB) {
                float2 t[KB];
                double2 d[KB];
#pragma unroll
                for (int k = 0; k < KB; ++k) {
                    const bool on = valid && k0 + k < cnt;
                    t[k] = on ? vis32[o + (k0 + k) * fstride] : make_float2(0.0f, 0.0f);
                    d[k] = on && vis64 != nullptr ? vis64[o + (k0 + k) * fstride] : make_double2(0.0, 0.0);
                }
#pragma unroll
                for (int k = 0; k < KB; ++k)
                    add(valid && k0 + k < cnt, o + (k0 + k) * fstride, t[k], d[k], acc[k0 + k][g][0], acc[k0 + k][g][1]);
            }
        }
    } else {
        // The WC waves' sums of KR channels at a time, added in wave order, one (channel, row) per wave.
        static_assert(WC == 1 || (WR == 1 && WC == KR * NG && NCH % KR == 0), "one row and channel per adding wave");
        const int kr = wc / NG, gr = wc % NG;
        size_t o;
        const bool valid = entry(gr, o);
        float2 t[NCH / KR];
        double2 d[NCH / KR];
#pragma unroll
        for (int i = 0; i < NCH / KR; ++i) {
            const bool on = valid && i * KR + kr < cnt;
            t[i] = on ? vis32[o + (i * KR + kr) * fstride] : make_float2(0.0f, 0.0f);
            d[i] = on && vis64 != nullptr ? vis64[o + (i * KR + kr) * fstride] : make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int i = 0; i < NCH / KR; ++i) {
            if (i * KR >= cnt) break;
#pragma unroll
            for (int k = 0; k < KR; ++k)
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    L.red[wc][k][g][0][lane] = acc[i * KR + k][g][0];
                    L.red[wc][k][g][1][lane] = acc[i * KR + k][g][1];
                }
            __syncthreads();
            double re = 0.0, im = 0.0;
#pragma unroll
            for (int w = 0; w < WC; ++w) {
                re += L.red[w][kr][gr][0][lane];
                im += L.red[w][kr][gr][1][lane];
            }
            add(valid && i * KR + kr < cnt, o + (i * KR + kr) * fstride, t[i], d[i], re, im);
            __syncthreads();
        }
    }
}

// The component slices' sums, added in order to the visibilities: one thread per (channel, baseline,
// entry), baselines numbered over the kernel's tiles.
__global__ void k_tiles_finish(const TiledArgs a) {
    const size_t npl = (size_t)a.ntiles * (a.ntiles - 1) / 2, n = a.nchan * npl * 4;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int s = 0; s < a.slices; ++s) {
        const double2 v = a.part[s * n + i];
        re += v.x;
        im += v.y;
    }
    size_t o = i;
    if (a.tile_map != nullptr) {
        const size_t f = i / (npl * 4);
        int p, q;
        triangle_pair((int)(i / 4 - f * npl), a.ntiles, p, q);
        p = a.tile_map[p];
        q = a.tile_map[q];
        o = (f * a.nbl + (size_t)p * a.ntiles_bl - (size_t)p * (p + 1) / 2 + (size_t)(q - p - 1)) * 4 + (i & 3);
    }
    float2 &t = reinterpret_cast<float2 *>(a.vis32)[o];
    t = make_float2(t.x + (float)re, t.y + (float)im);
    if (a.vis64 != nullptr) {
        double2 &d = reinterpret_cast<double2 *>(a.vis64)[o];
        d = make_double2(d.x + re, d.y + im);
    }
}

// Tile-group pairs: off-diagonal (0, g0, g1) with g0 < g1, then diagonal groups paired from
// both ends (1, g, G-1-g), the middle one alone (1, g, -1) when G is odd.
std::vector<int4> tile_pairs(int ntiles) {
    const int G = (ntiles + kTG - 1) / kTG;
    std::vector<int4> out;
    for (int g0 = 0; g0 < G; ++g0)
        for (int g1 = g0 + 1; g1 < G; ++g1) out.push_back(make_int4(0, g0, g1, 0));
    for (int g = 0; g < G / 2; ++g) out.push_back(make_int4(1, g, G - 1 - g, 0));
    if (G % 2 == 1) out.push_back(make_int4(1, G / 2, -1, 0));
    return out;
}

template <int KIND, int NCH, int NG, int WR, int WC, bool NARROW, bool SLICED = false>
static hipError_t launch_tiles_form(TiledArgs a, hipStream_t stream) {
    if (WC == 1 && !SLICED && a.part != nullptr)
        return launch_tiles_form<KIND, NCH, NG, WR, WC, NARROW, WC == 1>(a, stream);
    a.nchunks = chunk_count(a.chunks, NCH, a.nchan);
    hipLaunchKernelGGL((k_tiles_mfma<KIND, NCH, NG, WR, WC, NARROW, SLICED>),
                       dim3((unsigned)(a.npairs * a.nchunks * (kTG / (NG * WR)) * a.slices)), dim3(64 * WR * WC), 0, stream, a);
    if (a.part != nullptr) {
        const size_t n = (size_t)a.nchan * a.ntiles * (a.ntiles - 1) * 2;
        hipLaunchKernelGGL(k_tiles_finish, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
    }
    return hipGetLastError();
}

// Whether part holds, or could be made to hold, `bytes` of slice sums.
static bool reserve_slices(DevBuf *part, size_t bytes) {
    if (part == nullptr) return false;
    if (part->ptr == nullptr || part->bytes < bytes) {
        size_t free_b = 0, total_b = 0;
        if (!part->borrowed && (hipMemGetInfo(&free_b, &total_b) != hipSuccess || bytes > (free_b + part->bytes) / 8)) {
            (void)hipGetLastError();
            return false;
        }
        if (part->reserve(bytes) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
    }
    return true;
}

// Components of a slice: whole stages.
static int slice_length(int ncomp, int slices) { return ((ncomp + slices - 1) / slices + kCT - 1) / kCT * kCT; }

// Which form: the one with the smallest estimated time. With k = ceil(blocks / 256) blocks for the CU
// with the most, n components take start + start_block k + n (comp + comp_block k) us, whether a CU holds
// one, two or three at once (from 8 on the constant part is one of a block: slices do not divide it); the
// constants are fits to the kernel times of every form and slice count at 393 sizes (9 to 256 tiles, 1 to
// 768 channels, 4 to 20000 components, points and Gaussians), each form's within 6% rms. The form taken is
// 0.6% slower than the fastest on average, and more than 10% slower at 5 sizes of 786. Two row groups of 16 channels share a Gaussian's exponentials and a phasor's set-up over the
// most channels (768 channels, 5600 points 13.7 ms, 2000 Gaussians 7.8 ms; four row groups of 8 channels
// 13.7 and 8.3 ms). Two row groups of 8 channels fill the chip sooner: 100 points and Gaussians on 24
// channels and 128 tiles 28 and 37 us, against 38 and 53 us. Splitting the components over eight waves
// costs 1.5 times the widest form's time on a full chip, but its blocks are 4 rows high: 32 tiles, 64
// channels, 100 points 16 us, 4 wide, against 39 us.
// A form whose waves hold whole components (all but the last two) may also run slices of the components,
// of at least 128, in blocks of their own: their FP64 sums are written, read and added to the
// visibilities, after one more launch (5 us; 4 TB/s, or 12 TB/s for sums that fit the last-level cache).
// 128 tiles, 27 of 32 channels: 5600 points 1012 -> 673 us, 2000 Gaussians 561 -> 402 us; calls of 10000
// points for 32 tiles and 32 channels 728 -> 175 us, 20000 for 48 tiles and 2 channels 1418 -> 270 us.
TilesChoice choose_tiles_form(bool g, const TiledArgs &a, bool may_slice) {
    struct Form {
        int nch, sub;
        double start, start_block, comp, comp_block;
    };
    static const Form kPoint[5] = {{16, 2, 7.2, 5.7, 0.088, 0.167},
                                   {8, 1, 7.8, 5.4, 0.080, 0.173},
                                   {8, 2, 6.2, 2.4, 0.070, 0.092},
                                   {8, 4, 3.8, 6.1, 0.008, 0.077},
                                   {4, 4, 5.6, 2.4, 0.024, 0.044}};
    static const Form kGaussian[5] = {{16, 2, 7.8, 6.7, 0.120, 0.272},
                                      {8, 1, 8.2, 6.5, 0.106, 0.308},
                                      {8, 2, 5.3, 3.3, 0.078, 0.167},
                                      {8, 4, 3.8, 6.8, 0.008, 0.119},
                                      {4, 4, 4.2, 4.5, 0.005, 0.0936}};
    const size_t n = (size_t)a.nchan * a.ntiles * (a.ntiles - 1) * 2;  // entries of a slice's sums
    const int most = may_slice ? (int)std::min<size_t>(16, a.part_limit / (sizeof(double2) * std::max<size_t>(n, 1))) : 1;
    TilesChoice best{-1, 1, 0.0};
    for (int i = 0; i < 5; ++i) {
        if (i == 0 && !a.even16) continue;
        const Form &f = g ? kGaussian[i] : kPoint[i];
        for (int s = 1; s == 1 || (i < 3 && s <= most && s <= a.ncomp / 128); ++s) {
            const int len = s > 1 ? slice_length(a.ncomp, s) : a.ncomp;
            if ((a.ncomp + len - 1) / len != s) continue;  // the last slices would be empty
            const double k = ceil((double)a.npairs * f.sub * chunk_count(a.chunks, f.nch, a.nchan) * s / 256.0);
            double t = f.start + f.start_block * k + len * fmax(f.comp + f.comp_block * k, (f.comp / 8.0 + f.comp_block) * k);
            const double bytes = (double)sizeof(double2) * n * s;
            if (s > 1) t += 5.0 + 2.0 * bytes / (bytes <= 2e8 ? 12e6 : 4e6);
            if (best.form < 0 || t < best.us) best = TilesChoice{i, s, t};
        }
    }
    return best;
}

// The FP32 kernel's blocks are three to a CU: with x = blocks / 256, n components take n (0.53, 0.55, 0.64)
// us for up to one, two and three a CU, then n (0.30 + 0.183 x) (32 to 256 tiles, x of 1 to 64, within 8%).
// The FP64 kernel's estimate is some 5% short at such sizes, so that 8% decide. us a timestep, FP32 and
// FP64: 128 tiles, 72 channels, 200 Gaussians 183 and 207, 1000 619 and 555; 96 channels, 1000 628 and 639,
// 5000 2752 and 2542; 230 tiles, 48 channels, 10000 10810 and 8250, 96 channels 15650 and 16180; 256 tiles,
// 36 channels, 5000 3245 and 4541.
bool fp64_gaussians_faster(const TiledArgs &a) {
    const double x = (double)a.npairs * chunk_count(a.chunks, kTiledNchGaussian, a.nchan) / 256.0;
    const double us32 = 15.0 + a.ncomp * (x > 3.0 ? 0.30 + 0.183 * x : (x > 2.0 ? 0.64 : (x > 1.0 ? 0.55 : 0.53)));
    return choose_tiles_form(true, a, true).us < 0.92 * us32;
}

template <int KIND, bool NARROW>
static hipError_t launch_tiles(const TiledArgs &a_in, DevBuf *part, hipStream_t stream) {
    constexpr bool g = KIND == KIND_GAUSSIAN;
    TilesChoice best = choose_tiles_form(g, a_in, part != nullptr);
    TiledArgs a = a_in;
    a.part = nullptr;
    const size_t n = (size_t)a.nchan * a.ntiles * (a.ntiles - 1) * 2;
    if (best.slices > 1 && !reserve_slices(part, sizeof(double2) * n * best.slices)) best = choose_tiles_form(g, a, false);
    a.slices = best.slices;
    if (a.slices > 1) a.part = part->as<double2>();
    a.slice_len = slice_length(a.ncomp, a.slices);
    switch (best.form) {
    case 0: return launch_tiles_form<KIND, 16, 2, 4, 1, NARROW>(a, stream);
    case 1: return launch_tiles_form<KIND, 8, 4, 4, 1, NARROW>(a, stream);
    case 2: return launch_tiles_form<KIND, 8, 2, 4, 1, NARROW>(a, stream);
    case 3: return launch_tiles_form<KIND, 8, 4, 1, 8, NARROW>(a, stream);
    default: return launch_tiles_form<KIND, 4, 4, 1, 8, NARROW>(a, stream);
    }
}

// 60 tiles, 400 channels: 14 Gaussians 29.9 us, on k_tiles_mfma 32.3, but 20 37.9 and 35.8; 20 points 25.7
// and 27.7, 28 30.1 and 30.8. 128 tiles, 64 channels (352 blocks), 7 Gaussians 18.3 and 16.6; 768 channels,
// 24 points 111 and 123; 81 tiles, 383 channels, 18 Gaussians 51.8 and 56.7.
bool few_components(bool g, const TiledArgs &a) {
    const long blocks = (long)a.npairs * chunk_count(a.chunks, g ? kTiledNchGaussian : kTiledNchPoint, a.nchan);
    return a.vis64 == nullptr && blocks >= 400 && a.ncomp <= (g ? 18 : (blocks < 600 ? 20 : 28));
}

hipError_t launch_direct_tiled(Kind kind, const TiledArgs &a_in, DevBuf *part, hipStream_t stream) {
    if (a_in.ncomp <= 0 || a_in.nbl <= 0 || a_in.nchan <= 0) return hipSuccess;
    TiledArgs a = a_in;
    if (a.coh32 != nullptr) {
        if (kind != KIND_GAUSSIAN) return hipErrorInvalidValue;  // FP32 points take the MFMA point path
        a.nchunks = chunk_count(a.chunks, kTiledNchGaussian, a.nchan);
        hipLaunchKernelGGL((k_direct_tiled<KIND_GAUSSIAN, kTiledNchGaussian, float>), dim3(a.npairs * a.nchunks),
                           dim3(256), 0, stream, a);
        return hipGetLastError();
    }
    if (few_components(kind == KIND_GAUSSIAN, a)) {
        a.nchunks = chunk_count(a.chunks, kind == KIND_GAUSSIAN ? kTiledNchGaussian : kTiledNchPoint, a.nchan);
        const dim3 grid(a.npairs * a.nchunks);
        if (kind == KIND_GAUSSIAN)
            hipLaunchKernelGGL((k_direct_tiled<KIND_GAUSSIAN, kTiledNchGaussian, double>), grid, dim3(256), 0, stream, a);
        else
            hipLaunchKernelGGL((k_direct_tiled<KIND_POINT, kTiledNchPoint, double>), grid, dim3(256), 0, stream, a);
        return hipGetLastError();
    }
    return kind == KIND_GAUSSIAN ? (a.narrow ? launch_tiles<KIND_GAUSSIAN, true>(a, part, stream)
                                             : launch_tiles<KIND_GAUSSIAN, false>(a, part, stream))
                                 : launch_tiles<KIND_POINT, true>(a, part, stream);
}

// ------------------------------------------------------------------ pairs with own beams
constexpr int kPJC = 8;  // components per LDS stage
constexpr int kPJN = 4;  // channels per lane

// 2x2 complex (A B^H)[i][j] = sum_k A[i][k] conj(B[j][k]) added to acc with phasor z:
// acc += z (A B^H).
template <class T>
__device__ __forceinline__ void acc_abh(const T *a, const T *b, T zr, T zi, T *acc) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            T mr = T(0), mi = T(0);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const T ar = a[4 * i + 2 * k], ai = a[4 * i + 2 * k + 1];
                const T br = b[4 * j + 2 * k], bi = b[4 * j + 2 * k + 1];
                mr = fma_t(ar, br, mr);
                mr = fma_t(ai, bi, mr);
                mi = fma_t(ai, br, mi);
                mi = fma_t(-ar, bi, mi);
            }
            const int e = 2 * (2 * i + j);
            acc[e] = fma_t(mr, zr, acc[e]);
            acc[e] = fma_t(-mi, zi, acc[e]);
            acc[e + 1] = fma_t(mr, zi, acc[e + 1]);
            acc[e + 1] = fma_t(mi, zr, acc[e + 1]);
        }
}

// 2x2 complex acc += A B^H.
template <class T> __device__ __forceinline__ void acc_ab(const T *a, const T *b, T *acc) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int e = 2 * (2 * i + j);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const T ar = a[4 * i + 2 * k], ai = a[4 * i + 2 * k + 1];
                const T br = b[4 * j + 2 * k], bi = b[4 * j + 2 * k + 1];
                acc[e] = fma_t(ar, br, acc[e]);
                acc[e] = fma_t(ai, bi, acc[e]);
                acc[e + 1] = fma_t(ai, br, acc[e + 1]);
                acc[e + 1] = fma_t(-ar, bi, acc[e + 1]);
            }
        }
}

// Points: the baseline phasor factorises over the two tiles, z = K_p conj(K_q), so the staged
// factors carry it: A = K_p J_p S (row slots) and B = K_q J_q (column slots) per channel, with
// K_t = exp(i theta_t f / c) formed in FP64 per (component, tile slot, channel), and each lane
// accumulates A B^H (32 FMAs per channel and component instead of 48). Gaussians keep z
// outside: their envelope depends on the baseline, not on the tiles.
template <int KIND, class T>
__global__ __launch_bounds__(256) void k_pair_jones(const PairJonesArgs a, int ngroups) {
    using V4 = typename Vec4<T>::type;
    __shared__ V4 s_ph[kPJC][32];
    // [component][channel][slot]: slots 0..15 hold J_p S of the row tiles, 16..31 J_q of the
    // column tiles; a wave's 16 column lanes read 16 consecutive slots.
    __shared__ T s_m[kPJC][kPJN][32][8];
    __shared__ double s_uvw[32][3];
    __shared__ int s_row[32];
    const int ngpairs = ngroups * (ngroups + 1) / 2;
    // Block = (component slice, channel chunk, tile-group pair), the pair fastest.
    const int per_slice = ngpairs * a.nchunks;
    const int slice = blockIdx.x / per_slice;
    const int in_slice = blockIdx.x - slice * per_slice;
    const int chunk = in_slice / ngpairs;
    const int slice_len = (a.ncomp + a.csplit - 1) / a.csplit;
    const int c_begin = slice * slice_len;
    const int c_end = a.ncomp < c_begin + slice_len ? a.ncomp : c_begin + slice_len;
    // Tile-group pair (g0 <= g1) of this block, in row-major order of the upper triangle.
    int2 gp = make_int2(0, 0);
    {
        int rem = in_slice - chunk * ngpairs, g0 = 0;
        while (rem >= ngroups - g0) {
            rem -= ngroups - g0;
            ++g0;
        }
        gp = make_int2(g0, g0 + rem);
    }
    int f0, cnt;
    chunk_range<kPJN>(a.chunks, chunk, a.nchan, f0, cnt);
    const int tid = threadIdx.x, r = tid >> 4, cq = tid & 15;
    if (tid < 32) {
        const int g = tid < 16 ? gp.x : gp.y;
        const int i = g * 16 + (tid & 15);
        const int t = a.tiles[i < a.ntiles_list ? i : a.ntiles_list - 1];
        s_uvw[tid][0] = a.tile_uvw[3 * t];
        s_uvw[tid][1] = a.tile_uvw[3 * t + 1];
        s_uvw[tid][2] = a.tile_uvw[3 * t + 2];
        s_row[tid] = a.beam.tile_rows[t];
    }
    const int ip = gp.x * 16 + r, iq = gp.y * 16 + cq;
    const bool valid = ip < a.ntiles_list && iq < a.ntiles_list && ip < iq;
    __syncthreads();
    const double bu = s_uvw[r][0] - s_uvw[16 + cq][0];
    const double bv = s_uvw[r][1] - s_uvw[16 + cq][1];
    const double F0 = a.freqs[f0];
    const double DF = a.freqs[f0 + 1] - F0;
    const double f0c = F0 / SM_VEL_C, dfc = DF / SM_VEL_C;

    T acc[kPJN][8], tot[kPJN][8];
#pragma unroll
    for (int k = 0; k < kPJN; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[k][e] = tot[k][e] = T(0);

    for (int c0 = c_begin; c0 < c_end; c0 += kPJC) {
        const int nc = c_end - c0 < kPJC ? c_end - c0 : kPJC;
        if (KIND != KIND_POINT) {
            // One phasor pair per (component, tile slot): 8 x 32 = 256 threads.
            const int cc = tid >> 5, slot = tid & 31;
            double ps = 0.0, pc = 1.0, qs = 0.0, qc = 1.0;
            if (cc < nc) {
                const double4 l = a.lmn[c0 + cc];
                const double th = s_uvw[slot][0] * l.x + s_uvw[slot][1] * l.y + s_uvw[slot][2] * l.z;
                table_sincos(th * f0c, kSinCos32, ps, pc);
                table_sincos(th * dfc, kSinCos32, qs, qc);
            }
            V4 ph;
            ph.x = (T)pc;
            ph.y = (T)ps;
            ph.z = (T)qc;
            ph.w = (T)qs;
            s_ph[cc][slot] = ph;
        }
        // J_p S (row slots) and J_q (column slots) per (component, slot, channel).
        for (int w = tid; w < kPJC * 32 * kPJN; w += 256) {
            const int k = w % kPJN, slot = (w / kPJN) & 31, cc = w / (kPJN * 32);
            const int f = f0 + k < a.nchan ? f0 + k : a.nchan - 1;
            T *o = s_m[cc][k][slot];
            if (cc >= nc) {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = T(0);
                continue;
            }
            const int c = c0 + cc;
            double j[8];
            load_jones(&a.beam.jones[((size_t)s_row[slot] * a.beam.n_ufreq + a.beam.freq_map[f]) * a.beam.n_dir +
                                     a.beam.dir_offset + c],
                       j);
            double ks = 0.0, kc = 1.0;  // the tile phasor K_t at this channel (points)
            if (KIND == KIND_POINT) {
                const double4 l = a.lmn[c];
                const double th = s_uvw[slot][0] * l.x + s_uvw[slot][1] * l.y + s_uvw[slot][2] * l.z;
                table_sincos(th * (a.freqs[f] / SM_VEL_C), kSinCos32, ks, kc);
            }
            if (slot < 16) {
                double sv[8];
                load_jones(reinterpret_cast<const JonesF64 *>(a.coh + ((size_t)c * a.nchan_pad + f) * 8), sv);
                // (J S)[i][l] = sum_k J[i][k] S[k][l]
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int l = 0; l < 2; ++l) {
                        double re = 0.0, im = 0.0;
#pragma unroll
                        for (int kk = 0; kk < 2; ++kk) {
                            const double jr = j[4 * i + 2 * kk], ji = j[4 * i + 2 * kk + 1];
                            const double sr = sv[4 * kk + 2 * l], si = sv[4 * kk + 2 * l + 1];
                            re += jr * sr - ji * si;
                            im += jr * si + ji * sr;
                        }
                        if (KIND == KIND_POINT) {
                            o[4 * i + 2 * l] = (T)(re * kc - im * ks);
                            o[4 * i + 2 * l + 1] = (T)(re * ks + im * kc);
                        } else {
                            o[4 * i + 2 * l] = (T)re;
                            o[4 * i + 2 * l + 1] = (T)im;
                        }
                    }
            } else if (KIND == KIND_POINT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[2 * e] = (T)(j[2 * e] * kc - j[2 * e + 1] * ks);
                    o[2 * e + 1] = (T)(j[2 * e] * ks + j[2 * e + 1] * kc);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (T)j[e];
            }
        }
        __syncthreads();
        if (KIND == KIND_POINT) {
            for (int cc = 0; cc < nc; ++cc)
#pragma unroll
                for (int k = 0; k < kPJN; ++k) acc_ab<T>(s_m[cc][k][r], s_m[cc][k][16 + cq], acc[k]);
        } else
        for (int cc = 0; cc < nc; ++cc) {
            const V4 A = s_ph[cc][r];
            const V4 B = s_ph[cc][16 + cq];
            T zr = A.x * B.x + A.y * B.y;
            T zi = A.y * B.x - A.x * B.y;
            const T rr = A.z * B.z + A.w * B.w;
            const T ri = A.w * B.z - A.z * B.w;
            T env = T(1), er = T(1), eg = T(1);
            if (KIND == KIND_GAUSSIAN) {
                const double4 g = a.shape[c0 + cc];
                const double qf = g.x * (bu * bu) + g.y * (bu * bv) + g.z * (bv * bv);
                exp_of(qf * (F0 * F0), env);
                exp_of(qf * (DF * (2.0 * F0 + DF)), er);
                exp_of(qf * (2.0 * DF * DF), eg);
            }
#pragma unroll
            for (int k = 0; k < kPJN; ++k) {
                T pr = zr, pi = zi;
                if (KIND == KIND_GAUSSIAN) {
                    pr *= env;
                    pi *= env;
                }
                acc_abh<T>(s_m[cc][k][r], s_m[cc][k][16 + cq], pr, pi, acc[k]);
                const T nr = zr * rr - zi * ri;
                zi = zr * ri + zi * rr;
                zr = nr;
                if (KIND == KIND_GAUSSIAN) {
                    env *= er;
                    er *= eg;
                }
            }
        }
        flush_stage(acc, tot);
        __syncthreads();
    }
    if (!valid) return;
    if (a.csplit > 1) {
        // This slice's sums into accum[f][pair][8]; pairs in upper-triangle order of the list.
        const int n = a.ntiles_list;
        const size_t npairs = (size_t)n * (n - 1) / 2;
        const size_t t = (size_t)ip * n - (size_t)ip * (ip + 1) / 2 + (size_t)(iq - ip - 1);
#pragma unroll
        for (int k = 0; k < kPJN; ++k) {
            if (k >= cnt) break;
            double *dst = a.accum + ((size_t)(f0 + k) * npairs + t) * 8;
#pragma unroll
            for (int e = 0; e < 8; ++e) unsafeAtomicAdd(&dst[e], (double)two_level_sum(acc[k][e], tot[k][e]));
        }
        return;
    }
    const int p = a.tiles[ip], q = a.tiles[iq];
    const size_t nt = (size_t)a.ntiles_bl;
    const size_t bl = (size_t)p * nt - (size_t)p * (p + 1) / 2 + (size_t)(q - p - 1);
#pragma unroll
    for (int k = 0; k < kPJN; ++k) {
        if (k >= cnt) break;
        const size_t o = (size_t)(f0 + k) * a.nbl + bl;
        float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v32[e] += (float)two_level_sum(acc[k][e], tot[k][e]);
        if (a.vis64 != nullptr) {
            double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v64[e] += (double)two_level_sum(acc[k][e], tot[k][e]);
        }
    }
}

// vis[f][bl(pair)] += accum[f][pair] (FP64, and its FP32 rounding), pairs in upper-triangle
// order of the tile list.
__global__ void k_pair_finish(int nchan, int n, const int *__restrict__ tiles, int ntiles_bl, int nbl,
                              const double *__restrict__ accum, JonesF32 *vis32, JonesF64 *vis64) {
    const size_t npairs = (size_t)n * (n - 1) / 2;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nchan * npairs) return;
    const int f = (int)(i / npairs);
    int ip, iq;
    triangle_pair((int)(i - (size_t)f * npairs), n, ip, iq);
    const size_t p = (size_t)tiles[ip], q = (size_t)tiles[iq];
    const size_t o = (size_t)f * nbl + p * ntiles_bl - p * (p + 1) / 2 + (q - p - 1);
    const double *src = accum + i * 8;
    float *v32 = reinterpret_cast<float *>(&vis32[o]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v32[e] += (float)src[e];
    if (vis64 != nullptr) {
        double *v64 = reinterpret_cast<double *>(&vis64[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v64[e] += src[e];
    }
}

__global__ void k_zero_accum(size_t n, double *x) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        x[i] = 0.0;
}

hipError_t launch_pair_jones(Kind kind, const PairJonesArgs &a_in, DevBuf *accum, hipStream_t stream) {
    PairJonesArgs a = a_in;
    if (a.ncomp <= 0 || a.ntiles_list < 2 || a.nchan <= 0) return hipSuccess;
    if (kind == KIND_SHAPELET) return hipErrorInvalidValue;
    const int G = (a.ntiles_list + 15) / 16;
    a.nchunks = chunk_count(a.chunks, kPJN, a.nchan);
    const long blocks = (long)(G * (G + 1) / 2) * a.nchunks;
    // About 2048 blocks (8 per CU), each slice at least 64 components.
    long split = (2048 + blocks - 1) / blocks;
    split = std::min<long>(split, std::max(1, a.ncomp / (8 * kPJC)));
    split = std::max(1L, std::min(split, 64L));
    const size_t npairs = (size_t)a.ntiles_list * (a.ntiles_list - 1) / 2;
    const size_t nacc = (size_t)a.nchan * npairs * 8;
    a.csplit = 1;
    a.accum = nullptr;
    if (split > 1 && accum != nullptr) {
        if (accum->reserve(sizeof(double) * nacc) == hipSuccess) {
            a.csplit = (int)split;
            a.accum = accum->as<double>();
            hipLaunchKernelGGL(k_zero_accum, dim3(1024), dim3(256), 0, stream, nacc, a.accum);
        } else {
            (void)hipGetLastError();  // no room for the partial sums: unsplit launch
        }
    }
    const long total = blocks * a.csplit;
    if (a.fp32) {
        if (kind == KIND_GAUSSIAN)
            hipLaunchKernelGGL((k_pair_jones<KIND_GAUSSIAN, float>), dim3((unsigned)total), dim3(256), 0, stream, a, G);
        else
            hipLaunchKernelGGL((k_pair_jones<KIND_POINT, float>), dim3((unsigned)total), dim3(256), 0, stream, a, G);
    } else if (kind == KIND_GAUSSIAN) {
        hipLaunchKernelGGL((k_pair_jones<KIND_GAUSSIAN, double>), dim3((unsigned)total), dim3(256), 0, stream, a, G);
    } else {
        hipLaunchKernelGGL((k_pair_jones<KIND_POINT, double>), dim3((unsigned)total), dim3(256), 0, stream, a, G);
    }
    if (a.csplit > 1) {
        const size_t n = (size_t)a.nchan * npairs;
        hipLaunchKernelGGL(k_pair_finish, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a.nchan,
                           a.ntiles_list, a.tiles, a.ntiles_bl, a.nbl, a.accum, a.vis32, a.vis64);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ row tiles x class 0
// Pairs of a row tile (outside class 0) with a class-0 column tile: V_pq = sum_c C_c z_c with the
// full coherency C = J_r S J_0^H of the row's class. Where the array orders the baseline the other
// way (q < p), V_qp = V_pq^H is stored, which holds because the instrumental coherency S is
// Hermitian (XY and YX are conjugates).
//
// FP64, k_rect_mfma: the tile-pair kernel's scheme (k_tiles_mfma) with the four complex entries of C
// as the second operand and 16 columns of one row in a matrix instruction, four per channel (re and
// im of z by re and im of C). A wave has one row and 16 CG columns, so a component's C, staged in LDS,
// serves CG groups; a block has WR rows, which share the columns' phasors. Slices of the components
// (blockIdx / per_slice) fill the chip when there are few row tiles; their sums meet in `part`.
// Bound by FP64 issue: per component and channel 128 pairs take 128 matrix cycles a SIMD, their
// phasors about 50. 26 rows by 230 columns, 96 channels: 50000 points 43.0 -> 27.6 ms, 10000 Gaussians
// 14.1 -> 7.6 ms, against one lane per column on the vector ALUs. The blocks of one XCD sharing C took
// 37.5 to 31 ms of points, reading it a stage ahead the rest. Measured slower: 8 rows a block (33.4 and
// 9.4 ms); 4 column groups (26.4 and 11.2 ms); three waves a SIMD (26.5 and 9.7 ms).
constexpr int kRectNch = 8;  // channels per chunk
constexpr int kRectC = 16;   // components per LDS stage
constexpr int kRectCG = 2;    // column groups per wave
constexpr int kRectWR = 4;   // rows, one wave each, per block

// Entry se of the baseline (row ri, column cj) at channel 0: its index in the visibilities, and
// whether the array has the baseline the other way round (then the transposed entry's, conjugated).
__device__ __forceinline__ size_t rect_entry(const RectArgs &a, int ri, int cj, int se, bool &flip) {
    const int p = a.row_tiles[ri], q = a.col_tiles[cj];
    flip = q < p;
    const int lo = flip ? q : p, hi = flip ? p : q;
    const size_t bl = (size_t)lo * a.ntiles_bl - (size_t)lo * (lo + 1) / 2 + (size_t)(hi - lo - 1);
    return bl * 4 + (flip ? ((se & 1) << 1) | (se >> 1) : se);
}

template <int KIND, bool NARROW>
__global__ __launch_bounds__(64 * kRectWR, 2) void k_rect_mfma(const RectArgs a, int per_slice, int slice_len, double2 *part) {
    constexpr int WR = kRectWR, NCH = kRectNch, CG = kRectCG, NC = 16 * CG, NS = WR + NC, NT = 64 * WR;
    static_assert(NCH * 4 == 32 && kRectC % 4 == 0, "half a wave reads a component's C");
    __shared__ double2 s_p0[kRectC][NS], s_p1[kRectC][NS];  // tile phasors: rows, then columns (see Stage of k_tiles_mfma)
    __shared__ double2 s_c[WR][kRectC][NCH * 4 + 4];        // C; the padding puts components on distinct banks
    __shared__ double2 s_uv[NS];
    __shared__ double s_w[NS];
    __shared__ double2 s_sc[64];
    __shared__ double s_exp[64];
    __shared__ int s_cls[WR];
    const int nrg = (a.n_row + WR - 1) / WR, ncg = (a.n_col + NC - 1) / NC;
    // Consecutive blocks of one XCD (blockIdx modulo 8) take the column groups of the same rows,
    // channels and components, which share their C in its L2.
    const int bid = blockIdx.x, per = gridDim.x >> 3;
    const int vb = bid < per * 8 ? (bid & 7) * per + (bid >> 3) : bid;
    const int slice = vb / per_slice, b = vb - slice * per_slice;
    const int chunk = b / (nrg * ncg), rem = b - chunk * (nrg * ncg);
    const int rg = rem / ncg, cg = rem - rg * ncg;
    int f0, cnt;
    chunk_range<NCH>(a.chunks, chunk, a.nchan, f0, cnt);
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    if (tid < NS) {
        const int t = tid < WR ? a.row_tiles[min(rg * WR + tid, a.n_row - 1)]
                               : a.col_tiles[min(cg * NC + tid - WR, a.n_col - 1)];
        s_uv[tid] = make_double2(a.tile_uvw[3 * t], a.tile_uvw[3 * t + 1]);
        s_w[tid] = a.tile_uvw[3 * t + 2];
        if (tid < WR) s_cls[tid] = a.row_cls[min(rg * WR + tid, a.n_row - 1)];
    }
    if (tid < 64) {
        s_sc[tid] = make_double2(kSinCos32[2 * tid], kSinCos32[2 * tid + 1]);
        if (KIND == KIND_GAUSSIAN) s_exp[tid] = kExp64[tid];
    }
    __syncthreads();
    const int rows = min(WR, a.n_row - rg * WR);  // rows of this block
    const bool row_ok = w < rows;
    const int cq = 4 * (lane & 3) + ((lane >> 2) & 3), ck = lane >> 4, se = lane & 3;
    const double F0 = a.freqs[f0], DF = a.freqs[f0 + 1] - F0;
    const TwoDouble fm0 = over_c(F0 + (NCH / 2 - 1) * DF), fm1 = over_c(DF);
    const double qmin = -800.0 / (F0 * F0), q0 = F0 * F0, q1 = DF * (2.0 * F0 + DF), q2 = 2.0 * DF * DF;
    const double4 *__restrict__ lmn4 = a.lmn;
    const double4 *__restrict__ shape = a.shape;
    const double2 *__restrict__ coh = reinterpret_cast<const double2 *>(a.coh_cls);

    double re[NCH][CG], im[NCH][CG];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
        for (int g = 0; g < CG; ++g) re[k][g] = im[k][g] = 0.0;

    const int c_end = min(a.ncomp, (slice + 1) * slice_len);
    // Each wave stages its row's C, read one stage ahead. Components past the last are staged as 0.
    constexpr int PER = kRectC * NCH * 4 / 64;
    const double2 *__restrict__ crow = coh + (size_t)s_cls[w] * a.ncomp * a.nchan_pad * 4 + (size_t)f0 * 4 + (lane & 31);
    const size_t cstride = (size_t)a.nchan_pad * 4;
    double2 cv[PER];
    auto read_c = [&](int c0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = c0 + 2 * i + (lane >> 5);
            cv[i] = row_ok && c < c_end ? crow[c * cstride] : make_double2(0.0, 0.0);
        }
    };
    read_c(slice * slice_len);
    for (int c0 = slice * slice_len; c0 < c_end; c0 += kRectC) {
        const int nc = min(kRectC, c_end - c0), nc4 = (nc + 3) & ~3;
#pragma unroll
        for (int i = 0; i < PER; ++i) s_c[w][2 * i + (lane >> 5)][lane & 31] = cv[i];
        for (int e = tid; e < nc4 * NS; e += NT) {
            const int cc = e / NS, slot = e - cc * NS;
            double s0 = 0.0, c0_ = 0.0, s1 = 0.0, c1 = 0.0;
            if (cc < nc) {
                const double4 l = lmn4[c0 + cc];
                const double2 uv = s_uv[slot];
                const double th = uv.x * l.x + uv.y * l.y + s_w[slot] * l.z;
                table_sincos_product(th, fm0, reinterpret_cast<const double *>(s_sc), s0, c0_);
                table_sincos_product(th, fm1, reinterpret_cast<const double *>(s_sc), s1, c1);
            }
            s_p0[cc][slot] = make_double2(c0_, s0);
            s_p1[cc][slot] = make_double2(c1, s1);
        }
        __syncthreads();
        if (row_ok) {
            read_c(c0 + kRectC);
            for (int cs = 0; cs < nc; cs += 4) {
                const int cc = cs + ck;
                double2 C[NCH];
#pragma unroll
                for (int k = 0; k < NCH; ++k) C[k] = s_c[w][cc][4 * k + se];
                double4 sh = make_double4(0.0, 0.0, 0.0, 0.0);
                if (KIND == KIND_GAUSSIAN) sh = shape[min(c0 + cc, a.ncomp - 1)];
#pragma unroll
                for (int g = 0; g < CG; ++g) {
                    const int sq = WR + 16 * g + cq;
                    double zr[NCH], zi[NCH];
                    chunk_phasors<NCH>(s_p0[cc][w], s_p1[cc][w], s_p0[cc][sq], s_p1[cc][sq], zr, zi);
                    if (KIND == KIND_GAUSSIAN) {
                        const double2 tp = s_uv[w], tq = s_uv[sq];
                        gaussian_envelopes<NCH, NARROW>(sh, tp.x - tq.x, tp.y - tq.y, qmin, q0, q1, q2, s_exp, zr, zi);
                    }
#pragma unroll
                    for (int k = 0; k < NCH; ++k) {
                        re[k][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(zr[k], C[k].x, re[k][g], 0, 0, 0);
                        im[k][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(zr[k], C[k].y, im[k][g], 0, 0, 0);
                    }
#pragma unroll
                    for (int k = 0; k < NCH; ++k) {
                        re[k][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(zi[k], -C[k].y, re[k][g], 0, 0, 0);
                        im[k][g] = __builtin_amdgcn_mfma_f64_4x4x4f64(zi[k], C[k].x, im[k][g], 0, 0, 0);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (!row_ok) return;
    const int ri = rg * WR + w;
    float2 *const vis32 = reinterpret_cast<float2 *>(a.vis32);
    double2 *const vis64 = reinterpret_cast<double2 *>(a.vis64);
    const size_t fstride = (size_t)a.nbl * 4;
#pragma unroll
    for (int g = 0; g < CG; ++g) {
        const int cj = cg * NC + 16 * g + (lane >> 2);
        if (cj >= a.n_col) continue;
        if (part != nullptr) {
            double2 *o = part + (((size_t)slice * a.nchan + f0) * a.n_row + ri) * a.n_col * 4 + (size_t)cj * 4 + se;
#pragma unroll
            for (int k = 0; k < NCH; ++k)
                if (k < cnt) o[(size_t)k * a.n_row * a.n_col * 4] = make_double2(re[k][g], im[k][g]);
        } else {
            bool flip;
            const size_t o = rect_entry(a, ri, cj, se, flip) + (size_t)f0 * a.nbl * 4;
            // Every channel's entries are read before the first is written.
            float2 t[NCH];
            double2 d[NCH];
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                t[k] = k < cnt ? vis32[o + k * fstride] : make_float2(0.0f, 0.0f);
                d[k] = k < cnt && vis64 != nullptr ? vis64[o + k * fstride] : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int k = 0; k < NCH; ++k) {
                if (k >= cnt) break;
                const double vi = flip ? -im[k][g] : im[k][g];
                vis32[o + k * fstride] = make_float2(t[k].x + (float)re[k][g], t[k].y + (float)vi);
                if (vis64 != nullptr) vis64[o + k * fstride] = make_double2(d[k].x + re[k][g], d[k].y + vi);
            }
        }
    }
}

// The slices' sums, added in order to the visibilities: one thread per (channel, row, column, entry).
__global__ void k_rect_finish(const RectArgs a, int slices, const double2 *__restrict__ part) {
    const size_t n = (size_t)a.nchan * a.n_row * a.n_col * 4;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int s = 0; s < slices; ++s) {
        const double2 v = part[s * n + i];
        re += v.x;
        im += v.y;
    }
    const int se = (int)(i & 3), cj = (int)((i >> 2) % a.n_col);
    const size_t rf = (i >> 2) / a.n_col;
    const int ri = (int)(rf % a.n_row), f = (int)(rf / a.n_row);
    bool flip;
    const size_t o = rect_entry(a, ri, cj, se, flip) + (size_t)f * a.nbl * 4;
    if (flip) im = -im;
    float2 &t = reinterpret_cast<float2 *>(a.vis32)[o];
    t = make_float2(t.x + (float)re, t.y + (float)im);
    if (a.vis64 != nullptr) {
        double2 &d = reinterpret_cast<double2 *>(a.vis64)[o];
        d = make_double2(d.x + re, d.y + im);
    }
}

// FP32 (phases in FP64), k_direct_rect: a block owns 4 row tiles (one per wave) and 64 column tiles
// (one per lane) for one channel chunk. Every lane of a wave shares its row's class, so C arrives
// through scalar loads as in k_direct_tiled.
constexpr int kRC = 16;  // components per LDS stage
constexpr int kRT = 4 + 64;  // tile slots per block: 4 rows, then 64 columns
// Channels per lane. 256 tiles, 384 channels: Gaussians 28.3 ms with 4, 26.8 ms with 6.
constexpr int kRectNchGaussian = 6;

__global__ __launch_bounds__(256) void k_direct_rect(const RectArgs a) {
    using T = float;
    constexpr int NCH = kRectNchGaussian;
    __shared__ float4 s_ph[kRC][kRT];
    __shared__ double s_uvw[kRT][3];
    const int nrg = (a.n_row + 3) / 4, ncg = (a.n_col + 63) / 64;
    const int b = blockIdx.x;
    const int chunk = b / (nrg * ncg);
    int f0, cnt;
    chunk_range<NCH>(a.chunks, chunk, a.nchan, f0, cnt);
    const int rem = b - chunk * (nrg * ncg);
    const int rg = rem / ncg, cg = rem - rg * ncg;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    if (tid < kRT) {
        int t;
        if (tid < 4) {
            const int i = rg * 4 + tid;
            t = a.row_tiles[i < a.n_row ? i : a.n_row - 1];
        } else {
            const int j = cg * 64 + tid - 4;
            t = a.col_tiles[j < a.n_col ? j : a.n_col - 1];
        }
        s_uvw[tid][0] = a.tile_uvw[3 * t];
        s_uvw[tid][1] = a.tile_uvw[3 * t + 1];
        s_uvw[tid][2] = a.tile_uvw[3 * t + 2];
    }
    const int ri = rg * 4 + w, cj = cg * 64 + lane;
    const bool row_ok = ri < a.n_row;
    const bool valid = row_ok && cj < a.n_col;
    const int cls = __builtin_amdgcn_readfirstlane(row_ok ? a.row_cls[ri] : 0);
    __syncthreads();
    const int sp = w, sq = 4 + lane;
    const double bu = s_uvw[sp][0] - s_uvw[sq][0];
    const double bv = s_uvw[sp][1] - s_uvw[sq][1];

    const double *__restrict__ freqs = a.freqs;
    const double F0 = freqs[f0];
    const double DF = freqs[f0 + 1] - F0;
    const double f0c = F0 / SM_VEL_C;
    const double dfc = DF / SM_VEL_C;
    const T *__restrict__ coh = a.coh_cls32 + (size_t)cls * a.ncomp * a.nchan_pad * 8;
    const double4 *__restrict__ lmn4 = a.lmn;
    const double4 *__restrict__ shape = a.shape;

    T acc[NCH][8], tot[NCH][8];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[k][e] = tot[k][e] = T(0);

    for (int c0 = 0; c0 < a.ncomp; c0 += kRC) {
        const int nc = a.ncomp - c0 < kRC ? a.ncomp - c0 : kRC;
        for (int e = tid; e < kRC * kRT; e += 256) {
            const int cc = e / kRT, slot = e - cc * kRT;
            double ps = 0.0, pc = 1.0, qs = 0.0, qc = 1.0;
            if (cc < nc) {
                const double4 l = lmn4[c0 + cc];
                const double th = s_uvw[slot][0] * l.x + s_uvw[slot][1] * l.y + s_uvw[slot][2] * l.z;
                table_sincos(th * f0c, kSinCos32, ps, pc);
                table_sincos(th * dfc, kSinCos32, qs, qc);
            }
            s_ph[cc][slot] = make_float4((float)pc, (float)ps, (float)qc, (float)qs);
        }
        __syncthreads();
        if (row_ok) {
            for (int cc = 0; cc < nc; ++cc) {
                const int c = c0 + cc;
                const float4 A = s_ph[cc][sp];
                const float4 B = s_ph[cc][sq];
                T zr = A.x * B.x + A.y * B.y;
                T zi = A.y * B.x - A.x * B.y;
                const T rr = A.z * B.z + A.w * B.w;
                const T ri_ = A.w * B.z - A.z * B.w;
                T env, er, eg;
                const double4 g = shape[c];
                const double qf = g.x * (bu * bu) + g.y * (bu * bv) + g.z * (bv * bv);
                exp_of(qf * (F0 * F0), env);
                exp_of(qf * (DF * (2.0 * F0 + DF)), er);
                exp_of(qf * (2.0 * DF * DF), eg);
                const T *cc8 = coh + ((size_t)c * a.nchan_pad + f0) * 8;
#pragma unroll
                for (int k = 0; k < NCH; ++k) {
                    const T pr_ = zr * env, pi_ = zi * env;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const T cr = cc8[k * 8 + 2 * e], ci = cc8[k * 8 + 2 * e + 1];
                        acc[k][2 * e] = fma_t(cr, pr_, acc[k][2 * e]);
                        acc[k][2 * e] = fma_t(-ci, pi_, acc[k][2 * e]);
                        acc[k][2 * e + 1] = fma_t(cr, pi_, acc[k][2 * e + 1]);
                        acc[k][2 * e + 1] = fma_t(ci, pr_, acc[k][2 * e + 1]);
                    }
                    const T nr = zr * rr - zi * ri_;
                    zi = zr * ri_ + zi * rr;
                    zr = nr;
                    env *= er;
                    er *= eg;
                }
            }
        }
        flush_stage(acc, tot);
        __syncthreads();
    }
    if (!valid) return;
    const int p = a.row_tiles[ri], q = a.col_tiles[cj];
    const bool flip = q < p;  // array baseline (q, p): store V_pq^H
    const int lo = flip ? q : p, hi = flip ? p : q;
    const size_t nt = (size_t)a.ntiles_bl;
    const size_t bl = (size_t)lo * nt - (size_t)lo * (lo + 1) / 2 + (size_t)(hi - lo - 1);
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
        const int f = f0 + k;
        if (k >= cnt) break;
        T v[8], w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = two_level_sum(acc[k][e], tot[k][e]);
        if (flip) {
            // (V^H)_ij = conj(V_ji): XX, YX, XY, YY with the imaginary parts negated.
            v[0] = w[0];
            v[1] = -w[1];
            v[2] = w[4];
            v[3] = -w[5];
            v[4] = w[2];
            v[5] = -w[3];
            v[6] = w[6];
            v[7] = -w[7];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = w[e];
        }
        const size_t o = (size_t)f * a.nbl + bl;
        float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v32[e] += (float)v[e];
        if (a.vis64 != nullptr) {
            double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v64[e] += (double)v[e];
        }
    }
}

template <int KIND, bool NARROW>
static hipError_t launch_rect(const RectArgs &a, DevBuf *part, hipStream_t stream) {
    constexpr int WR = kRectWR;
    const int per_slice = ((a.n_row + WR - 1) / WR) * ((a.n_col + 16 * kRectCG - 1) / (16 * kRectCG)) *
                          chunk_count(a.chunks, kRectNch, a.nchan);
    // Slices of at least 512 components: as many as fill whole rounds of the blocks that the 256 CUs hold
    // (two waves a SIMD), few for the traffic of their sums. No room for those: one.
    constexpr int kSlots = 2 * 256 * 4 / WR;
    const size_t n = (size_t)a.nchan * a.n_row * a.n_col * 4;  // entries of a slice's sums
    const int most = (int)std::min<size_t>(16, kSliceBytes / (sizeof(double2) * n));
    int slices = 1;
    double t_best = 0.0;
    for (int s = 1; s == 1 || (s <= most && s <= a.ncomp / 512); ++s) {
        const double t = (double)((per_slice * (long)s + kSlots - 1) / kSlots) / s + 0.02 * s * per_slice / kSlots;
        if (s == 1 || t < t_best) {
            slices = s;
            t_best = t;
        }
    }
    if (slices > 1 && !reserve_slices(part, sizeof(double2) * n * slices)) slices = 1;
    double2 *p = slices > 1 ? part->as<double2>() : nullptr;
    const int slice_len = ((a.ncomp + slices - 1) / slices + kRectC - 1) / kRectC * kRectC;
    hipLaunchKernelGGL((k_rect_mfma<KIND, NARROW>), dim3((unsigned)(per_slice * slices)), dim3(64 * WR), 0, stream, a,
                       per_slice, slice_len, p);
    if (p != nullptr)
        hipLaunchKernelGGL(k_rect_finish, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a, slices, p);
    return hipGetLastError();
}

hipError_t launch_direct_rect(Kind kind, const RectArgs &a, DevBuf *part, hipStream_t stream) {
    if (a.ncomp <= 0 || a.n_row <= 0 || a.n_col <= 0 || a.nchan <= 0) return hipSuccess;
    if (a.coh_cls32 == nullptr)
        return kind == KIND_GAUSSIAN ? (a.narrow ? launch_rect<KIND_GAUSSIAN, true>(a, part, stream)
                                                 : launch_rect<KIND_GAUSSIAN, false>(a, part, stream))
                                     : launch_rect<KIND_POINT, true>(a, part, stream);
    if (kind != KIND_GAUSSIAN) return hipErrorInvalidValue;  // FP32 points take the MFMA point path
    const long total = (long)((a.n_row + 3) / 4) * ((a.n_col + 63) / 64) * chunk_count(a.chunks, kRectNchGaussian, a.nchan);
    hipLaunchKernelGGL(k_direct_rect, dim3((unsigned)total), dim3(256), 0, stream, a);
    return hipGetLastError();
}

// ------------------------------------------------------------------ shapelets
// Per-tile beams: one wave per baseline, one channel per lane, the coefficients summed per channel.
template <class T> __device__ __forceinline__ void shapelet_chan_tiles(const ShapeletChanArgs &a) {
    const int nbx = (a.nbl + 3) / 4;
    const int total = nbx * a.ngroups;
    int b = blockIdx.x;
    if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
    const int group = b / nbx;
    const int bx = b - group * nbx;
    const int lane = threadIdx.x & 63;
    const int bl = bx * 4 + (int)(threadIdx.x >> 6);
    if (bl >= a.nbl) return;  // whole wave; the kernel has no barriers
    const int f_raw = group * 64 + lane;
    const bool valid = f_raw < a.nchan;
    const int f = valid ? f_raw : a.nchan - 1;
    const double freq = a.freqs[f];
    const double fc = freq / SM_VEL_C;
    const UVW uvw = a.uvw[bl];
    int2 rows = make_int2(0, 0);
    int uf = 0;
    int cls = -1;
    bool herm = false;
    rows = a.beam.bl_rows[bl];
    uf = a.beam.freq_map[f];
    if (a.beam.coh_cls != nullptr) {
        if (rows.y == a.beam.row0) {
            cls = a.beam.class_of_row[rows.x];
        } else if (rows.x == a.beam.row0) {
            cls = a.beam.class_of_row[rows.y];
            herm = true;
        }
    }
    const PackedCoeff *__restrict__ packed = a.packed;
    const T *__restrict__ sbf = pick<T>(a.sbf, a.sbf32);
    // Per-wave windows of the basis table (kRows rows x kWin cells per axis).
    __shared__ T wx_lds[4][kRows][kWin], wy_lds[4][kRows][kWin];
    const int wv = threadIdx.x >> 6;
    // The wave's lowest and highest channel frequency (invalid lanes repeat the last channel).
    double fmin_w = freq, fmax_w = freq;
    for (int o = 32; o > 0; o >>= 1) {
        fmin_w = fmin(fmin_w, __shfl_xor(fmin_w, o));
        fmax_w = fmax(fmax_w, __shfl_xor(fmax_w, o));
    }
    T acc[1][8] = {{0, 0, 0, 0, 0, 0, 0, 0}}, tot[1][8] = {{0, 0, 0, 0, 0, 0, 0, 0}};
    // The wave's baseline is uniform; the next component's coefficient range is loaded one
    // iteration ahead.
    const int blu = __builtin_amdgcn_readfirstlane(bl);
    // Shapelet UVs are read from bl_uv: forming them here takes registers that it does not have (256
    // tiles: more spills, 104 -> 110 ms per timestep).
    // The phase dot product, the UV in the component's frame (xk, yk) and the table window are
    // the same on every lane of the wave: lane l forms those of component 64 q + l once per
    // batch q of 64 components, and each component reads them from that lane. The window is
    // packed as first cell | width << 16 (both below SM_SBF_L < 2^15).
    double th_lane = 0.0, xk_lane = 0.0, yk_lane = 0.0;
    int wx_lane = 0, wy_lane = 0;
    auto load_batch = [&](int q) {
        const int cl = min((q << 6) + lane, a.ncomp - 1);
        const double4 l = a.lmn[cl];
        const double4 sh = a.shape[cl];
        const double2 suv = a.bl_uv[(size_t)cl * a.nbl + blu];
        th_lane = uvw.u * l.x + uvw.v * l.y + uvw.w * l.z;
        const double xk = (suv.x * sh.x + suv.y * sh.y) * sh.z;
        const double yk = (suv.x * sh.y - suv.y * sh.x) * sh.w;
        // The cells the wave touches: positions are monotone in frequency, so the extreme
        // channels bound them (the same expressions as each lane's position, so the same
        // roundings).
        const double xa = xk * fmin_w + SM_SBF_C, xb = xk * fmax_w + SM_SBF_C;
        const double ya = yk * fmin_w + SM_SBF_C, yb = yk * fmax_w + SM_SBF_C;
        const int ix0 = (int)fmin(fmax(floor(fmin(xa, xb)), 0.0), (double)(SM_SBF_L - 2));
        const int ix1 = (int)fmin(fmax(floor(fmax(xa, xb)), 0.0), (double)(SM_SBF_L - 2));
        const int iy0 = (int)fmin(fmax(floor(fmin(ya, yb)), 0.0), (double)(SM_SBF_L - 2));
        const int iy1 = (int)fmin(fmax(floor(fmax(ya, yb)), 0.0), (double)(SM_SBF_L - 2));
        xk_lane = xk;
        yk_lane = yk;
        wx_lane = ix0 | ((ix1 - ix0 + 2) << 16);
        wy_lane = iy0 | ((iy1 - iy0 + 2) << 16);
    };
    int4 pr_next = a.prange[0];
    for (int c = 0; c < a.ncomp; ++c) {
        const int4 pr4 = pr_next;
        pr_next = a.prange[c + 1 < a.ncomp ? c + 1 : c];
        if ((c & 63) == 0) load_batch(c >> 6);
        const int src = c & 63;
        const double theta = readlane_f64(th_lane, src);
        const double xk = readlane_f64(xk_lane, src), yk = readlane_f64(yk_lane, src);
        const int wxp = __builtin_amdgcn_readlane(wx_lane, src), wyp = __builtin_amdgcn_readlane(wy_lane, src);
        T zr, zi;
        sincos_phase(theta * fc, zi, zr);
        const double x_pos = xk * freq + SM_SBF_C;
        const double y_pos = yk * freq + SM_SBF_C;
        const double fx = floor(x_pos), fy = floor(y_pos);
        const int ix = (int)fmin(fmax(fx, 0.0), (double)(SM_SBF_L - 2));
        const int iy = (int)fmin(fmax(fy, 0.0), (double)(SM_SBF_L - 2));
        const T wx = (T)(x_pos - fx), wy = (T)(y_pos - fy);
        T er, ei;
        const int xw = wxp >> 16, yw = wyp >> 16;
        if (xw <= kWin && yw <= kWin && pr4.w <= kRows) {
            // Stage rows 0 .. pr4.w - 1 of both windows in this wave's LDS, then interpolate
            // from LDS: one 16-byte read per axis per coefficient instead of two gathers.
            const int bx0 = wxp & 0xffff, by0 = wyp & 0xffff;
            // Lane -> (row lane >> lw, cell lane & (2^lw - 1)), 2^lw the smallest power of two
            // of at least 4 cells covering both windows, so one pass stages 64 >> lw rows of both
            // axes (16 rows for windows of up to 4 cells). All loads first, then all LDS writes:
            // the loads are in flight together instead of one round trip per row. A lane past
            // the window or past row pr4.w - 1 reads an in-bounds cell (the window's last cell;
            // rows below kRows + 16 <= SM_SBF_N) that is never written. Byte offsets are 32-bit
            // (the table is 8 MB), from the uniform base.
            const int wm = max(xw, yw);
            const int lw = wm <= 4 ? 2 : (wm <= 8 ? 3 : (wm <= 16 ? 4 : 5));
            const int rstep = 64 >> lw;
            const int j = lane & ((1 << lw) - 1), rl = lane >> lw;
            const int jxc = min(j, xw - 1), jyc = min(j, yw - 1);
            static_assert(kRows + 16 <= SM_SBF_N, "staged rows must exist in the basis table");
            const unsigned ox = (unsigned)((rl * SM_SBF_L + bx0 + jxc) * sizeof(T));
            const unsigned oy = (unsigned)((rl * SM_SBF_L + by0 + jyc) * sizeof(T));
            const char *sbf_b = reinterpret_cast<const char *>(sbf);
            constexpr int kBatch = 2;  // row steps in flight at once (register budget)
            for (int i0 = 0; i0 < pr4.w; i0 += kBatch * rstep) {
                T tx[kBatch], ty[kBatch];
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int base = i0 + i * rstep;
                    const unsigned step = (unsigned)(base * SM_SBF_L * sizeof(T));
                    if (base < pr4.w) {
                        tx[i] = *reinterpret_cast<const T *>(sbf_b + (ox + step));
                        ty[i] = *reinterpret_cast<const T *>(sbf_b + (oy + step));
                    }
                }
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int base = i0 + i * rstep, r = base + rl;
                    if (base < pr4.w && r < pr4.w) {
                        if (j < xw) wx_lds[wv][r][j] = tx[i];
                        if (j < yw) wy_lds[wv][r][j] = ty[i];
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int jx = ix - bx0, jy = iy - by0;
            T part[2];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                const PackedCoeff *cp = packed + pr4.x + (pt ? pr4.y : 0);
                const int cnt = pt ? pr4.z : pr4.y;
                T accp = T(0);
#pragma unroll 2
                for (int k = 0; k < cnt; ++k) {
                    double val;
                    int n1, n2;
                    load_packed_uniform(cp + k, val, n1, n2);
                    const T xl = wx_lds[wv][n1][jx], xh = wx_lds[wv][n1][jx + 1];
                    const T yl = wy_lds[wv][n2][jy], yh = wy_lds[wv][n2][jy + 1];
                    const T u_value = xl + (xh - xl) * wx;
                    const T v_value = yl + (yh - yl) * wy;
                    accp += ((T)val * u_value) * v_value;
                }
                part[pt] = accp;
            }
            er = part[0];
            ei = part[1];
            // Every lane's reads are done before the next component's staging.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            // Rare (a window wider than the LDS copy): one coefficient at a time, which keeps
            // this path's registers below the staged path's.
            T part[2];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                const PackedCoeff *cp = packed + pr4.x + (pt ? pr4.y : 0);
                const int cnt = pt ? pr4.z : pr4.y;
                T accp = T(0);
#pragma unroll 1
                for (int k = 0; k < cnt; ++k) {
                    double val;
                    int n1, n2;
                    load_packed_uniform(cp + k, val, n1, n2);
                    const T *bx = sbf + n1 * SM_SBF_L + ix, *by = sbf + n2 * SM_SBF_L + iy;
                    const T u_value = bx[0] + (bx[1] - bx[0]) * wx;
                    const T v_value = by[0] + (by[1] - by[0]) * wy;
                    accp += ((T)val * u_value) * v_value;
                }
                part[pt] = accp;
            }
            er = part[0];
            ei = part[1];
        }
        const T pr = zr * er - zi * ei;
        const T pi = zr * ei + zi * er;
        T cj[8];
        if (cls >= 0) {
            class_coh(pick<T>(a.beam.coh_cls, a.coh_cls32) + (((size_t)cls * a.ncomp + c) * a.nchan_pad + f) * 8,
                      herm, cj);
        } else {
            // J_p S J_q^H of the instrumental flux S (FP64 table) and the two tiles' beams.
            const double *s = a.coh + ((size_t)c * a.nchan_pad + f) * 8;
            double sv[8], j1[8], j2[8], cd[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[e] = s[e];
            load_jones_t(&a.beam.jones[((size_t)rows.x * a.beam.n_ufreq + uf) * a.beam.n_dir + a.beam.dir_offset + c], j1);
            load_jones_t(&a.beam.jones[((size_t)rows.y * a.beam.n_ufreq + uf) * a.beam.n_dir + a.beam.dir_offset + c], j2);
            sandwich_t(j1, sv, j2, cd);
#pragma unroll
            for (int e = 0; e < 8; ++e) cj[e] = (T)cd[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[0][2 * e] = fma_t(cj[2 * e], pr, acc[0][2 * e]);
            acc[0][2 * e] = fma_t(-cj[2 * e + 1], pi, acc[0][2 * e]);
            acc[0][2 * e + 1] = fma_t(cj[2 * e], pi, acc[0][2 * e + 1]);
            acc[0][2 * e + 1] = fma_t(cj[2 * e + 1], pr, acc[0][2 * e + 1]);
        }
        if ((c & 15) == 15) flush_stage(acc, tot);
    }
    if (!valid) return;
    const size_t o = (size_t)f * a.nbl + bl;
    float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
    for (int e = 0; e < 8; ++e) v32[e] += (float)two_level_sum(acc[0][e], tot[0][e]);
    if (a.vis64 != nullptr) {
        double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v64[e] += (double)two_level_sum(acc[0][e], tot[0][e]);
    }
}

// Held to 128 VGPRs in FP64 (4 waves per SIMD, a few spilled values) instead of 164 (3 waves), and to 96
// in FP32 (5 waves) instead of 118: 256 tiles and 384 channels 129 -> 111 ms and 66.2 -> 57.8 ms.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_shapelet_chan_tiles(
    const ShapeletChanArgs a) {
    shapelet_chan_tiles<double>(a);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void k_shapelet_chan_tiles32(
    const ShapeletChanArgs a) {
    shapelet_chan_tiles<float>(a);
}

// Shared beam, FP32: one wave per baseline and 128 channels, two adjacent channels per lane
// (channels 2 l and 2 l + 1 of the group on lane l). The table cells are read for both channels
// at once: adjacent channels' positions differ by |k| df, below one cell (checked per component),
// so both fall in cells i0 and i0 + 1 with i0 the lower of their two cells. The staged window
// holds each cell's value and its difference to the next cell, formed once per component, and
// the lane reads T[i0], T[i0 + 1] - T[i0] and T[i0 + 2] - T[i0 + 1] per axis and coefficient
// (24 bytes for two channels, against 16 per channel reading two values). A channel in cell
// i0 interpolates
//   u = T[i0] + (T[i0+1] - T[i0]) w,
// as the single-channel form does, and one in cell i0 + 1 takes
//   u = (T[i0] + (T[i0+1] - T[i0])) + (T[i0+2] - T[i0+1]) w,
// equal to T[i0+1] + (T[i0+2] - T[i0+1]) w up to the rounding of T[i0] + (T[i0+1] - T[i0]).
// The coherency table is in the Hermitian form (Re XX, Re XY, Im XY, Re YY; J S J^H with one
// beam on both sides), so each channel accumulates with 8 FMAs per component.

// A staged basis-table cell: the value T[i] and the difference T[i + 1] - T[i].
struct __attribute__((aligned(8))) CellTD {
    float t, d;
};

__global__ __launch_bounds__(256) void k_shapelet_chan32(const ShapeletChanArgs a) {
    using T = float;
    const int ngroups = (a.nchan + 127) / 128;
    const int nbx = (a.nbl + 3) / 4;
    const int total = nbx * ngroups;
    int b = blockIdx.x;
    if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
    const int group = b / nbx;
    const int bx = b - group * nbx;
    const int lane = threadIdx.x & 63;
    const int bl = bx * 4 + (int)(threadIdx.x >> 6);
    if (bl >= a.nbl) return;  // whole wave; the kernel has no barriers
    const int fa_raw = group * 128 + 2 * lane;
    const bool valid_a = fa_raw < a.nchan, valid_b = fa_raw + 1 < a.nchan;
    const int fa = valid_a ? fa_raw : a.nchan - 1;
    const int fb = valid_b ? fa_raw + 1 : a.nchan - 1;
    const double freq_a = a.freqs[fa], freq_b = a.freqs[fb];
    const double fc_a = freq_a / SM_VEL_C, fc_b = freq_b / SM_VEL_C;
    const UVW uvw = a.uvw[bl];
    const PackedCoeff *__restrict__ packed = a.packed;
    const T *__restrict__ sbf = a.sbf32;
    const T *__restrict__ coh_t = a.coh32;
    // Per-wave windows of the basis table (kRows rows x kWinPair cells per axis), each cell
    // holding T[i] and T[i + 1] - T[i].
    __shared__ CellTD wx_lds[4][kRows][kWinPair], wy_lds[4][kRows][kWinPair];
    const int wv = threadIdx.x >> 6;
    // The wave's lowest and highest channel frequency and its largest step between a lane's
    // two channels (channels past the last repeat it).
    double fmin_w = fmin(freq_a, freq_b), fmax_w = fmax(freq_a, freq_b), dfmax_w = fabs(freq_b - freq_a);
    for (int o = 32; o > 0; o >>= 1) {
        fmin_w = fmin(fmin_w, __shfl_xor(fmin_w, o));
        fmax_w = fmax(fmax_w, __shfl_xor(fmax_w, o));
        dfmax_w = fmax(dfmax_w, __shfl_xor(dfmax_w, o));
    }
    T acc[2][8], tot[2][8];
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[ch][e] = tot[ch][e] = T(0);
    const int blu = __builtin_amdgcn_readfirstlane(bl);
    // Shapelet UVs: formed here from the baseline's tile XYZs and each component's (HA, Dec)
    // when those are given; else read from bl_uv.
    const bool uv_here = a.hadec != nullptr;
    double x1 = 0, y1 = 0, z1 = 0, x2 = 0, y2 = 0, z2 = 0;
    if (uv_here) {
        const int2 t = a.bl_tiles[blu];
        x1 = a.xyz[3 * t.x];
        y1 = a.xyz[3 * t.x + 1];
        z1 = a.xyz[3 * t.x + 2];
        x2 = a.xyz[3 * t.y];
        y2 = a.xyz[3 * t.y + 1];
        z2 = a.xyz[3 * t.y + 2];
    }
    const double4 *__restrict__ hd4 = reinterpret_cast<const double4 *>(a.hadec);
    // As in k_shapelet_chan_tiles32: the wave-uniform per-component values, formed by lane l for
    // component 64 q + l and read back by lane.
    double th_lane = 0.0, xk_lane = 0.0, yk_lane = 0.0;
    int wx_lane = 0, wy_lane = 0;
    auto load_batch = [&](int q) {
        const int cl = min((q << 6) + lane, a.ncomp - 1);
        const double4 l = a.lmn[cl];
        const double4 sh = a.shape[cl];
        const double2 suv =
            uv_here ? shapelet_uv(hd4[cl], x1, y1, z1, x2, y2, z2) : a.bl_uv[(size_t)cl * a.nbl + blu];
        th_lane = uvw.u * l.x + uvw.v * l.y + uvw.w * l.z;
        const double xk = (suv.x * sh.x + suv.y * sh.y) * sh.z;
        const double yk = (suv.x * sh.y - suv.y * sh.x) * sh.w;
        const double xa = xk * fmin_w + SM_SBF_C, xb = xk * fmax_w + SM_SBF_C;
        const double ya = yk * fmin_w + SM_SBF_C, yb = yk * fmax_w + SM_SBF_C;
        const int ix0 = (int)fmin(fmax(floor(fmin(xa, xb)), 0.0), (double)(SM_SBF_L - 2));
        const int ix1 = (int)fmin(fmax(floor(fmax(xa, xb)), 0.0), (double)(SM_SBF_L - 2));
        const int iy0 = (int)fmin(fmax(floor(fmin(ya, yb)), 0.0), (double)(SM_SBF_L - 2));
        const int iy1 = (int)fmin(fmax(floor(fmax(ya, yb)), 0.0), (double)(SM_SBF_L - 2));
        xk_lane = xk;
        yk_lane = yk;
        wx_lane = ix0 | ((ix1 - ix0 + 2) << 16);
        wy_lane = iy0 | ((iy1 - iy0 + 2) << 16);
    };
    int4 pr_next = a.prange[0];
    for (int c = 0; c < a.ncomp; ++c) {
        const int4 pr4 = pr_next;
        pr_next = a.prange[c + 1 < a.ncomp ? c + 1 : c];
        if ((c & 63) == 0) load_batch(c >> 6);
        const int src = c & 63;
        const double theta = readlane_f64(th_lane, src);
        const double xk = readlane_f64(xk_lane, src), yk = readlane_f64(yk_lane, src);
        const int wxp = __builtin_amdgcn_readlane(wx_lane, src), wyp = __builtin_amdgcn_readlane(wy_lane, src);
        T zr[2], zi[2];
        sincos_phase(theta * fc_a, zi[0], zr[0]);
        sincos_phase(theta * fc_b, zi[1], zr[1]);
        const double xpa = xk * freq_a + SM_SBF_C, xpb = xk * freq_b + SM_SBF_C;
        const double ypa = yk * freq_a + SM_SBF_C, ypb = yk * freq_b + SM_SBF_C;
        const double fxa = floor(xpa), fxb = floor(xpb), fya = floor(ypa), fyb = floor(ypb);
        const int ixa = (int)fmin(fmax(fxa, 0.0), (double)(SM_SBF_L - 2));
        const int ixb = (int)fmin(fmax(fxb, 0.0), (double)(SM_SBF_L - 2));
        const int iya = (int)fmin(fmax(fya, 0.0), (double)(SM_SBF_L - 2));
        const int iyb = (int)fmin(fmax(fyb, 0.0), (double)(SM_SBF_L - 2));
        const T wxa = (T)(xpa - fxa), wxb = (T)(xpb - fxb), wya = (T)(ypa - fya), wyb = (T)(ypb - fyb);
        const int xw = wxp >> 16, yw = wyp >> 16;
        // One component's coherencies for both channels (Hermitian form, 4 values each).
        T cq[2][4];
        {
            const T *s_a = coh_t + ((size_t)c * a.nchan_pad + fa) * 4;
            const T *s_b = coh_t + ((size_t)c * a.nchan_pad + fb) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                cq[0][e] = s_a[e];
                cq[1][e] = s_b[e];
            }
        }
        T er[2], ei[2];
        // Staged path: both windows, one extra cell for T[i0 + 2], fit the LDS copy, and the
        // two channels of a lane are less than half a cell apart on both axes (so their cells
        // differ by at most one, with a wide margin for rounding).
        const bool near = fabs(xk) * dfmax_w < 0.5 && fabs(yk) * dfmax_w < 0.5;
        if (near && xw + 1 <= kWinPair && yw + 1 <= kWinPair && pr4.w <= kRows) {
            const int bx0 = wxp & 0xffff, by0 = wyp & 0xffff;
            const int xs = xw + 1, ys = yw + 1;  // staged cells per axis
            // As in k_shapelet_chan_tiles32: lane -> (row lane >> lw, cell lane & (2^lw - 1)). A lane past
            // the window or past row pr4.w - 1 reads an in-bounds cell that is never written; the
            // last cell is at most SM_SBF_L, in the row or at the next row's first cell, and the
            // difference it enters is only multiplied by a zero weight when outside the row.
            // T[i + 1] comes from the next lane of the row; the difference formed with the next
            // row's lane at cell 2^lw - 1 >= xs - 1 is never read (the loop reads differences
            // at cells up to xs - 2).
            const int wm = max(xs, ys);
            const int lw = wm <= 4 ? 2 : (wm <= 8 ? 3 : (wm <= 16 ? 4 : 5));
            const int rstep = 64 >> lw;
            const int j = lane & ((1 << lw) - 1), rl = lane >> lw;
            const int jxc = min(j, xs - 1), jyc = min(j, ys - 1);
            static_assert(kRows + 16 < SM_SBF_N, "staged rows and the next row must exist in the basis table");
            const unsigned ox = (unsigned)((rl * SM_SBF_L + bx0 + jxc) * sizeof(T));
            const unsigned oy = (unsigned)((rl * SM_SBF_L + by0 + jyc) * sizeof(T));
            const char *sbf_b = reinterpret_cast<const char *>(sbf);
            constexpr int kBatch = 2;
            for (int i0 = 0; i0 < pr4.w; i0 += kBatch * rstep) {
                T tx[kBatch], ty[kBatch];
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int base = i0 + i * rstep;
                    const unsigned step = (unsigned)(base * SM_SBF_L * sizeof(T));
                    if (base < pr4.w) {
                        tx[i] = *reinterpret_cast<const T *>(sbf_b + (ox + step));
                        ty[i] = *reinterpret_cast<const T *>(sbf_b + (oy + step));
                    }
                }
#pragma unroll
                for (int i = 0; i < kBatch; ++i) {
                    const int base = i0 + i * rstep, r = base + rl;
                    if (base < pr4.w) {  // wave-uniform: every lane takes part in the shuffles
                        const T tx1 = __shfl_down(tx[i], 1), ty1 = __shfl_down(ty[i], 1);
                        if (r < pr4.w) {
                            if (j < xs) wx_lds[wv][r][j] = CellTD{tx[i], tx1 - tx[i]};
                            if (j < ys) wy_lds[wv][r][j] = CellTD{ty[i], ty1 - ty[i]};
                        }
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // Each channel's weights on (T[i0+1] - T[i0]) and (T[i0+2] - T[i0+1]).
            const int ix0l = min(ixa, ixb), iy0l = min(iya, iyb);
            const int jx = ix0l - bx0, jy = iy0l - by0;
            const bool xa_lo = ixa == ix0l, xb_lo = ixb == ix0l, ya_lo = iya == iy0l, yb_lo = iyb == iy0l;
            const T ax_a = xa_lo ? wxa : T(1), bx_a = xa_lo ? T(0) : wxa;
            const T ax_b = xb_lo ? wxb : T(1), bx_b = xb_lo ? T(0) : wxb;
            const T ay_a = ya_lo ? wya : T(1), by_a = ya_lo ? T(0) : wya;
            const T ay_b = yb_lo ? wyb : T(1), by_b = yb_lo ? T(0) : wyb;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                const PackedCoeff *cp = packed + pr4.x + (pt ? pr4.y : 0);
                const int cnt = pt ? pr4.z : pr4.y;
                T acc_a = T(0), acc_b = T(0);
#pragma unroll 4
                for (int k = 0; k < cnt; ++k) {
                    double val;
                    int n1, n2;
                    load_packed_uniform(cp + k, val, n1, n2);
                    const CellTD cx = wx_lds[wv][n1][jx], cy = wy_lds[wv][n2][jy];
                    const T dx12 = wx_lds[wv][n1][jx + 1].d, dy12 = wy_lds[wv][n2][jy + 1].d;
                    const T u_a = fma_t(dx12, bx_a, fma_t(cx.d, ax_a, cx.t));
                    const T u_b = fma_t(dx12, bx_b, fma_t(cx.d, ax_b, cx.t));
                    const T v_a = fma_t(dy12, by_a, fma_t(cy.d, ay_a, cy.t));
                    const T v_b = fma_t(dy12, by_b, fma_t(cy.d, ay_b, cy.t));
                    acc_a += ((T)val * u_a) * v_a;
                    acc_b += ((T)val * u_b) * v_b;
                }
                (pt ? ei : er)[0] = acc_a;
                (pt ? ei : er)[1] = acc_b;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            // Rare: one coefficient at a time from the table in memory, per channel.
            const int ixs[2] = {ixa, ixb}, iys[2] = {iya, iyb};
            const T wxs[2] = {wxa, wxb}, wys[2] = {wya, wyb};
#pragma unroll
            for (int ch = 0; ch < 2; ++ch) {
#pragma unroll
                for (int pt = 0; pt < 2; ++pt) {
                    const PackedCoeff *cp = packed + pr4.x + (pt ? pr4.y : 0);
                    const int cnt = pt ? pr4.z : pr4.y;
                    T accp = T(0);
#pragma unroll 1
                    for (int k = 0; k < cnt; ++k) {
                        double val;
                        int n1, n2;
                        load_packed_uniform(cp + k, val, n1, n2);
                        const T *bxp = sbf + n1 * SM_SBF_L + ixs[ch], *byp = sbf + n2 * SM_SBF_L + iys[ch];
                        const T u_value = bxp[0] + (bxp[1] - bxp[0]) * wxs[ch];
                        const T v_value = byp[0] + (byp[1] - byp[0]) * wys[ch];
                        accp += ((T)val * u_value) * v_value;
                    }
                    (pt ? ei : er)[ch] = accp;
                }
            }
        }
#pragma unroll
        for (int ch = 0; ch < 2; ++ch) {
            const T pr = zr[ch] * er[ch] - zi[ch] * ei[ch];
            const T pi = zr[ch] * ei[ch] + zi[ch] * er[ch];
            acc[ch][0] = fma_t(cq[ch][0], pr, acc[ch][0]);
            acc[ch][1] = fma_t(cq[ch][0], pi, acc[ch][1]);
            acc[ch][2] = fma_t(cq[ch][1], pr, acc[ch][2]);
            acc[ch][3] = fma_t(cq[ch][1], pi, acc[ch][3]);
            acc[ch][4] = fma_t(cq[ch][2], pr, acc[ch][4]);
            acc[ch][5] = fma_t(cq[ch][2], pi, acc[ch][5]);
            acc[ch][6] = fma_t(cq[ch][3], pr, acc[ch][6]);
            acc[ch][7] = fma_t(cq[ch][3], pi, acc[ch][7]);
        }
        if ((c & 15) == 15) flush_stage(acc, tot);
    }
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
        if (!(ch ? valid_b : valid_a)) continue;
        const size_t o = (size_t)(ch ? fb : fa) * a.nbl + bl;
        T s8[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) s8[e] = two_level_sum(acc[ch][e], tot[ch][e]);
        // XX, XY = A + i B, YX = A - i B, YY.
        const T v[8] = {s8[0], s8[1], s8[2] - s8[5], s8[3] + s8[4], s8[2] + s8[5], s8[3] - s8[4], s8[6], s8[7]};
        float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v32[e] += (float)v[e];
        if (a.vis64 != nullptr) {
            double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v64[e] += (double)v[e];
        }
    }
}

// J_p S J_q^H of component c at channel f, from the flux table (S) and the beams of rows p and q.
__device__ __forceinline__ void own_beam_coh(const ShapeletChanArgs &a, int2 rows, int c, int f, double o[8]) {
    double sv[8], j1[8], j2[8];
    load_jones_t(reinterpret_cast<const JonesF64 *>(a.coh + ((size_t)c * a.nchan_pad + f) * 8), sv);
    const size_t col = (size_t)a.beam.freq_map[f] * a.beam.n_dir + a.beam.dir_offset + c;
    load_jones_t(&a.beam.jones[(size_t)rows.x * a.beam.n_ufreq * a.beam.n_dir + col], j1);
    load_jones_t(&a.beam.jones[(size_t)rows.y * a.beam.n_ufreq * a.beam.n_dir + col], j2);
    sandwich_t(j1, sv, j2, o);
}

// Shapelets in FP64, with one beam on both sides (Hermitian coherencies) or none, or per-tile beams
// (PT: the class's coherency or J_p S J_q^H, 8 values). One lane per channel (SL
// slots of 64 / LB channels), LB baselines per wave.
//
// A component's basis-table positions x(f) = xk f + 5000 and y(f) are linear in frequency and the
// basis functions are interpolated linearly, so while both positions stay in one pair of table
// cells the envelope sum_k c_k B_n1(x) B_n2(y) is the same bilinear function of the two
// fractions, i.e. one quadratic in f. Along the band (x, y) walks monotonically through the
// table, so the cell pairs it visits ("segments") are numbered by the cell edges crossed since the
// lowest frequency, s = |ix - ixa| + |iy - iya|. Components are taken in batches of at most 32
// segments; per batch the wave
//   1. sums the coefficients once per segment and part (real, imaginary), one lane each, into the
//      quadratic's three coefficients, in FP64,
//   2. evaluates them at every channel (4 FMAs) with the phasor and the coherency.
// Where an x and a y edge are crossed within rounding of one channel, the channel and the lane that
// sums its segment may order them differently; the two bilinear forms then meet at that channel.
// Positions outside the table, or more than kShSeg segments, take the per-channel sums.
//
// The values of the next components are formed by one lane each and read back from LDS. The phasor
// is a sincos at the first slot, turned by the slots' common step by the recurrence
// z_{k+1} = 2 cos(delta) z_k - z_{k-1} (unevenly spaced channels: a sincos each).
//
// Bound by step 1, whose reads are scattered (16 bytes per lane, about 40 cycles of the address
// unit per wave instruction), and by the latency of step 2's chain at 3 - 4 waves per SIMD: of
// 13.5 ms on 1400 components, 128 tiles and 384 channels of 80 kHz, 4.9 ms are coefficient sums
// and 2.9 ms phasors. Summing the coefficients per channel, from table windows staged in LDS, took
// 21.7 ms there, and 4.0 against 0.9 ms on 24 channels of 40 kHz. Slower in step 1: windows staged
// in LDS (22 ms), the basis functions by their recurrence in registers (15.6 ms). Per-tile beams (500
// components, 256 tiles within 3 km, 96 channels of 80 kHz, so about three channels a run): 26.7 ms
// summing per channel, 24.4 ms here (24.8 ms with the registers for three waves and no spills).
constexpr int kShItems = 32;  // (component, baseline) pairs whose values are formed at a time
constexpr int kShSeg = 64;    // segment quadratics per wave
constexpr int kShCoef = 128;  // staged coefficients per wave

struct __attribute__((aligned(16))) ShVal {
    double xk, yk, theta, c2, rr, ri;
    int ixa, iya;    // cells at the lowest frequency
    int edges, off;  // edges crossed on x | on y << 16; segments of the pairs before this one
    int4 coef;       // launch_pack_coeffs' range
};

// Basis-table position of frequency f, rounded alike everywhere.
__device__ __forceinline__ double table_pos(double k, double f) { return fma(k, f, SM_SBF_C); }

__device__ __forceinline__ int cell_of(double pos) {
    return (int)fmin(fmax(floor(pos), 0.0), (double)(SM_SBF_L - 2));
}

// A table cell's value and its neighbour's, read together.
struct __attribute__((packed, aligned(8))) CellPair {
    double v, next;
};

template <int SL, int LB, int WPS, bool PT>
__global__ __launch_bounds__(256, WPS) void k_shapelets(const ShapeletChanArgs a) {
    constexpr int LPB = 64 / LB, SPAN = SL * LPB, VC = kShItems / LB;
    __shared__ ShVal s_val[4][kShItems];
    __shared__ __attribute__((aligned(16))) double s_seg[4][kShSeg][6];
    __shared__ PackedCoeff s_coef[4][kShCoef];
    __shared__ double2 s_sc[64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (threadIdx.x < 64) s_sc[lane] = make_double2(kSinCos32[2 * lane], kSinCos32[2 * lane + 1]);
    __syncthreads();
    const double *sc_tab = reinterpret_cast<const double *>(s_sc);
    const int ngroups = (a.nchan + SPAN - 1) / SPAN;
    const int nbx = (a.nbl + 4 * LB - 1) / (4 * LB);
    const int total = nbx * ngroups;
    int b = blockIdx.x;
    if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
    const int group = b / nbx;
    const int bl0 = ((b - group * nbx) * 4 + wv) * LB;  // the wave's first baseline
    if (bl0 >= a.nbl) return;                           // whole wave; no barriers below
    const int bsub = lane / LPB;  // this lane's baseline as a channel
    const int ch0 = group * SPAN + (lane & (LPB - 1));
    // Per-tile beams: the beam rows of the lane's baseline, and its class if one of them is class 0's.
    int2 rows = make_int2(0, 0);
    int cls = -1;
    bool herm = false;
    if (PT) {
        rows = a.beam.bl_rows[min(bl0 + bsub, a.nbl - 1)];
        if (a.beam.coh_cls != nullptr) {
            herm = rows.y != a.beam.row0;
            if (!herm || rows.x == a.beam.row0) cls = a.beam.class_of_row[herm ? rows.y : rows.x];
        }
    }
    double freq[SL], tk[SL];
#pragma unroll
    for (int k = 0; k < SL; ++k) freq[k] = a.freqs[min(ch0 + k * LPB, a.nchan - 1)];
    // The span's lowest and highest frequency, and whether its slots are one step apart.
    double fmin_w = freq[0], fmax_w = freq[0];
#pragma unroll
    for (int k = 1; k < SL; ++k) {
        fmin_w = fmin(fmin_w, freq[k]);
        fmax_w = fmax(fmax_w, freq[k]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        fmin_w = fmin(fmin_w, __shfl_xor(fmin_w, o));
        fmax_w = fmax(fmax_w, __shfl_xor(fmax_w, o));
    }
    const double step = __shfl(freq[SL > 1 ? 1 : 0] - freq[0], 0);
    bool rot = true;
#pragma unroll
    for (int k = 1; k < SL; ++k) rot = rot && (ch0 + k * LPB >= a.nchan || freq[k] - freq[k - 1] == step);
    rot = __all(rot);
    // Quadratics are in t = (f - fmin) / unit, t <= 1.
    const double unit = fmax_w > fmin_w ? fmax_w - fmin_w : 1.0;
#pragma unroll
    for (int k = 0; k < SL; ++k) tk[k] = (freq[k] - fmin_w) / unit;

    const PackedCoeff *__restrict__ packed = a.packed;
    const double *__restrict__ sbf = a.sbf;
    const char *__restrict__ sbf_b = reinterpret_cast<const char *>(a.sbf);
    const double *__restrict__ coh = a.coh;
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    double acc[SL][8];
#pragma unroll
    for (int k = 0; k < SL; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[k][e] = 0.0;

    for (int c0 = 0; c0 < a.ncomp; c0 += VC) {
        // Values of (component, baseline) pair `lane`, and the running count of segments.
        int upto = 0;  // segments of the pairs up to and with this lane's
        int coef_lo = 0, coef_hi = 0;
        bool fast = true;
        wave_sync();
        if (lane < kShItems) {
            const int c = min(c0 + lane / LB, a.ncomp - 1);
            const int obl = min(bl0 + lane % LB, a.nbl - 1);
            const int2 ot = a.bl_tiles != nullptr ? a.bl_tiles[obl] : make_int2(0, 0);
            const UVW uvw = a.uvw[obl];
            const double4 l = a.lmn[c], sh = a.shape[c];
            const double4 *__restrict__ hd4 = reinterpret_cast<const double4 *>(a.hadec);
            const double2 suv = a.hadec != nullptr
                                    ? shapelet_uv(hd4[c], a.xyz[3 * ot.x], a.xyz[3 * ot.x + 1], a.xyz[3 * ot.x + 2],
                                                  a.xyz[3 * ot.y], a.xyz[3 * ot.y + 1], a.xyz[3 * ot.y + 2])
                                    : a.bl_uv[(size_t)c * a.nbl + obl];
            ShVal v;
            v.xk = (suv.x * sh.x + suv.y * sh.y) * sh.z;
            v.yk = (suv.x * sh.y - suv.y * sh.x) * sh.w;
            v.theta = uvw.u * l.x + uvw.v * l.y + uvw.w * l.z;
            table_sincos(v.theta * (step / SM_VEL_C), sc_tab, v.ri, v.rr);
            v.c2 = 2.0 * v.rr;
            const double xa = table_pos(v.xk, fmin_w), xb = table_pos(v.xk, fmax_w);
            const double ya = table_pos(v.yk, fmin_w), yb = table_pos(v.yk, fmax_w);
            v.ixa = cell_of(xa);
            v.iya = cell_of(ya);
            const int nx = abs(cell_of(xb) - v.ixa), ny = abs(cell_of(yb) - v.iya);
            const double lo = 1.0, hi = (double)(SM_SBF_L - 2);
            fast = xa >= lo && xb >= lo && ya >= lo && yb >= lo && xa < hi && xb < hi && ya < hi && yb < hi &&
                   nx + ny + 1 <= kShSeg / LB;
            v.edges = fast ? nx | ny << 16 : 0;
            v.coef = a.prange[c];
            coef_lo = v.coef.x;
            coef_hi = v.coef.x + v.coef.y + v.coef.z;
            upto = fast ? nx + ny + 1 : 0;
            const int own = upto;
            for (int o = 1; o < kShItems; o <<= 1) {
                const int before = __shfl_up(upto, o);
                if (lane >= o) upto += before;
            }
            v.off = upto - own;
            s_val[wv][lane] = v;
        }
        wave_sync();
        const int nitem = min(VC, a.ncomp - c0) * LB;
        for (int i0 = 0; i0 < nitem;) {
            // The batch: pairs i0 .. i1 - 1, as many as 32 segments hold, or one component of up
            // to kShSeg (two passes), or one component without segments (direct).
            const int base = i0 > 0 ? __builtin_amdgcn_readlane(upto, i0 - 1) : 0;
            const unsigned long long over = __ballot(lane >= i0 && (!fast || upto - base > 32));
            int i1 = min((over != 0 ? __ffsll(over) - 1 : 64) / LB * LB, nitem);
            const bool direct = i1 <= i0 && __any(lane >= i0 && lane < i0 + LB && !fast);
            if (i1 <= i0) i1 = i0 + LB;
            if (!direct) {
                // 1. One segment and part per lane.
                const int nseg = __builtin_amdgcn_readlane(upto, i1 - 1) - base;
                const int cfirst = __builtin_amdgcn_readlane(coef_lo, i0);
                const int ncoef = __builtin_amdgcn_readlane(coef_hi, i1 - 1) - cfirst;
                const bool staged = ncoef <= kShCoef;
                if (staged) {
#pragma unroll
                    for (int j = 0; j < kShCoef; j += 64)
                        if (j + lane < ncoef)
                            reinterpret_cast<int4 *>(s_coef[wv])[j + lane] =
                                reinterpret_cast<const int4 *>(packed)[cfirst + j + lane];
                    wave_sync();
                }
                for (int sf = lane >> 1; __any(sf < nseg); sf += 32) {
                    if (sf >= nseg) continue;
                    const int part = lane & 1;
                    int it = i0;
                    for (int i = i0 + 1; i < i1; ++i)
                        it += __builtin_amdgcn_readlane(upto, i - 1) - base <= sf ? 1 : 0;
                    const ShVal &v = s_val[wv][it];
                    const int sg = sf - (v.off - base);
                    const double xk = v.xk, yk = v.yk;
                    const double xa = table_pos(xk, fmin_w), ya = table_pos(yk, fmin_w);
                    const double X = xk * unit, Y = yk * unit;
                    // Edges of x among the first sg crossed: edge i of x at t = (ux + i) / |X|.
                    const int nx = v.edges & 0xffff, ny = v.edges >> 16;
                    const double ux = X >= 0.0 ? v.ixa + 1 - xa : xa - v.ixa, uy = Y >= 0.0 ? v.iya + 1 - ya : ya - v.iya;
                    const double rx = fabs(X), ry = fabs(Y);
                    int ex = max(0, sg - ny);
                    const int ex_max = min(sg, nx);
                    ex = min(ex_max, max(ex, (int)((sg * rx + ux * ry - uy * rx) / fmax(rx + ry, 1e-300))));
                    while (ex > max(0, sg - ny) && (ux + (ex - 1)) * ry > (uy + (sg - ex)) * rx) --ex;
                    while (ex < ex_max && (uy + (sg - ex - 1)) * rx > (ux + ex) * ry) ++ex;
                    const int ix = X >= 0.0 ? v.ixa + ex : v.ixa - ex, iy = Y >= 0.0 ? v.iya + (sg - ex) : v.iya - (sg - ex);
                    const unsigned ox = 8u * (unsigned)ix, oy = 8u * (unsigned)iy;  // byte offsets, 32-bit: the table is 8 MB
                    const int4 cr = v.coef;
                    const int first = cr.x + (part ? cr.y : 0), cnt = part ? cr.z : cr.y;
                    double s00 = 0.0, s10 = 0.0, s01 = 0.0, s11 = 0.0;
                    // Four coefficients at a time, their eight table reads in flight together (the
                    // scheduling barrier keeps the compiler from waiting for each read in turn).
                    auto add4 = [&](const PackedCoeff *cp, int j) {
                        double val[4], x[4][2], y[4][2];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const PackedCoeff cf = cp[min(j + u, cnt - 1)];
                            val[u] = j + u < cnt ? cf.value : 0.0;
                            const CellPair tx = *reinterpret_cast<const CellPair *>(
                                sbf_b + (ox + __umul24((unsigned)cf.n1, 8u * SM_SBF_L)));
                            const CellPair ty = *reinterpret_cast<const CellPair *>(
                                sbf_b + (oy + __umul24((unsigned)cf.n2, 8u * SM_SBF_L)));
                            x[u][0] = tx.v;
                            x[u][1] = tx.next;
                            y[u][0] = ty.v;
                            y[u][1] = ty.next;
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const double vx = val[u] * x[u][0], vd = val[u] * (x[u][1] - x[u][0]);
                            const double yd = y[u][1] - y[u][0];
                            s00 = fma(vx, y[u][0], s00);
                            s01 = fma(vx, yd, s01);
                            s10 = fma(vd, y[u][0], s10);
                            s11 = fma(vd, yd, s11);
                        }
                    };
                    if (staged) {
#pragma unroll 1
                        for (int j = 0; j < cnt; j += 4) add4(s_coef[wv] + (first - cfirst), j);
                    } else {
#pragma unroll 1
                        for (int j = 0; j < cnt; j += 4) add4(packed + first, j);
                    }
                    // The bilinear form at fractions wx = wx0 + X t, wy = wy0 + Y t.
                    const double wx0 = fma(xk, fmin_w, SM_SBF_C - ix), wy0 = fma(yk, fmin_w, SM_SBF_C - iy);
                    const double a0 = fma(wx0, s10, s00), a1 = fma(wx0, s11, s01), d = fma(wy0, s11, s10);
                    double *o = s_seg[wv][sf] + 3 * part;
                    o[0] = fma(wy0, a1, a0);
                    o[1] = fma(Y, a1, X * d);
                    o[2] = (X * Y * s11);
                }
                wave_sync();
            }
            // 2. Channels.
#pragma unroll 1
            for (int i = i0; i < i1; i += LB) {
                const int c = c0 + i / LB;
                const ShVal &v = s_val[wv][i + bsub];
                double cq[SL][PT ? 8 : 4];
#pragma unroll
                for (int k = 0; k < SL; ++k) {
                    if (PT) {
                        const int f = min(ch0 + k * LPB, a.nchan - 1);
                        if (cls >= 0)
                            class_coh(a.beam.coh_cls + (((size_t)cls * a.ncomp + c) * a.nchan_pad + f) * 8, herm, cq[k]);
                        else
                            own_beam_coh(a, rows, c, f, cq[k]);
                        continue;
                    }
                    const double *q = coh + ((size_t)c * 2 * a.nchan_pad + min(ch0 + k * LPB, a.nchan - 1)) * 2;
                    cq[k][0] = q[0];
                    cq[k][1] = q[1];
                    cq[k][2] = q[2 * a.nchan_pad];
                    cq[k][3] = q[2 * a.nchan_pad + 1];
                }
                const double theta = v.theta, xk = v.xk, yk = v.yk;
                double er[SL], ei[SL];
                if (!direct) {
                    const double *sb = s_seg[wv][v.off - base];
                    const int ixa = v.ixa, iya = v.iya;
#pragma unroll
                    for (int k = 0; k < SL; ++k) {
                        const int sg = abs((int)table_pos(xk, freq[k]) - ixa) + abs((int)table_pos(yk, freq[k]) - iya);
                        const double *q = sb + 6 * sg;
                        er[k] = fma(tk[k], fma(tk[k], q[2], q[1]), q[0]);
                        ei[k] = fma(tk[k], fma(tk[k], q[5], q[4]), q[3]);
                    }
                } else {
                    // Rare: one coefficient at a time from the table in memory, per channel.
                    const int4 cr = v.coef;
#pragma unroll
                    for (int k = 0; k < SL; ++k) {
                        const double xp = table_pos(xk, freq[k]), yp = table_pos(yk, freq[k]);
                        const double wx = xp - floor(xp), wy = yp - floor(yp);
                        const double *bx = sbf + cell_of(xp), *by = sbf + cell_of(yp);
                        double sum[2];
#pragma unroll
                        for (int pt = 0; pt < 2; ++pt) {
                            const int first = cr.x + (pt ? cr.y : 0), cnt = pt ? cr.z : cr.y;
                            sum[pt] = 0.0;
#pragma unroll 1
                            for (int j = 0; j < cnt; ++j) {
                                const PackedCoeff cf = packed[first + j];
                                const double *tx = bx + cf.n1 * SM_SBF_L, *ty = by + cf.n2 * SM_SBF_L;
                                const double u = tx[0] + (tx[1] - tx[0]) * wx, w = ty[0] + (ty[1] - ty[0]) * wy;
                                sum[pt] += (cf.value * u) * w;
                            }
                        }
                        er[k] = sum[0];
                        ei[k] = sum[1];
                    }
                }
                double zr[SL], zi[SL];
                table_sincos(theta * (freq[0] / SM_VEL_C), sc_tab, zi[0], zr[0]);
                if (SL > 1) {
                    if (rot) {
                        const double rr = v.rr, ri = v.ri, c2 = v.c2;
                        zr[SL > 1 ? 1 : 0] = zr[0] * rr - zi[0] * ri;
                        zi[SL > 1 ? 1 : 0] = zr[0] * ri + zi[0] * rr;
#pragma unroll
                        for (int k = 2; k < SL; ++k) {
                            zr[k] = fma(c2, zr[k - 1], -zr[k - 2]);
                            zi[k] = fma(c2, zi[k - 1], -zi[k - 2]);
                        }
                    } else {
#pragma unroll
                        for (int k = 1; k < SL; ++k)
                            table_sincos(theta * (freq[k] / SM_VEL_C), sc_tab, zi[k], zr[k]);
                    }
                }
#pragma unroll
                for (int k = 0; k < SL; ++k) {
                    const double pr = zr[k] * er[k] - zi[k] * ei[k];
                    const double pi = zr[k] * ei[k] + zi[k] * er[k];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double cr = cq[k][PT ? 2 * e : e];
                        acc[k][2 * e] = fma(cr, pr, acc[k][2 * e]);
                        acc[k][2 * e + 1] = fma(cr, pi, acc[k][2 * e + 1]);
                        if (PT) {
                            const double ci = cq[k][PT ? 2 * e + 1 : 0];
                            acc[k][2 * e] = fma(-ci, pi, acc[k][2 * e]);
                            acc[k][2 * e + 1] = fma(ci, pr, acc[k][2 * e + 1]);
                        }
                    }
                }
            }
            wave_sync();
            i0 = i1;
        }
    }
    const int bl = bl0 + bsub;
    if (bl >= a.nbl) return;
#pragma unroll
    for (int k = 0; k < SL; ++k) {
        const int f = ch0 + k * LPB;
        if (f >= a.nchan) continue;
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[k][e];
        if (!PT) {
            // XX, XY = A + i B, YX = A - i B, YY.
            const double ar = v[2], ai = v[3], br = v[4], bi = v[5];
            v[2] = ar - bi;
            v[3] = ai + br;
            v[4] = ar + bi;
            v[5] = ai - br;
        }
        const size_t o = (size_t)f * a.nbl + bl;
        float *v32 = reinterpret_cast<float *>(&a.vis32[o]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v32[e] += (float)v[e];
        if (a.vis64 != nullptr) {
            double *v64 = reinterpret_cast<double *>(&a.vis64[o]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v64[e] += v[e];
        }
    }
}

template <int SL, int LB, int WPS, bool PT>
static hipError_t launch_shapelets_form(const ShapeletChanArgs &a, hipStream_t stream) {
    const long total = (long)((a.nbl + 4 * LB - 1) / (4 * LB)) * ((a.nchan + SL * 64 / LB - 1) / (SL * 64 / LB));
    hipLaunchKernelGGL((k_shapelets<SL, LB, WPS, PT>), dim3((unsigned)total), dim3(256), 0, stream, a);
    return hipGetLastError();
}

// The forms: fewer, wider groups share the phasors' start and the component's values among more
// channels; narrow ones hold fewer segments, the cost that grows with the table edges that a component
// crosses over a group's channels. Per-tile beams have a fourth, k_shapelet_chan_tiles, whose sums per
// channel cost the same wherever the edges lie. Each takes a time per group that is linear in those edges
// up to where most components leave the segments for the direct sums; the lines are fits, within 12%, to
// 200 components of 0.5 to 5 arcmin, 128 tiles within 0.5, 1.5 and 3 km, and 4 to 384 channels of 20 kHz
// to 1.28 MHz. The form taken is within 5% of the fastest at 77 of these 78 sizes (10% at the other). ms,
// forms 0 to 3, per-tile beams:
//   384 x 80 kHz, 500 m   4.6 4.9 5.5 7.7     24 x 80 kHz, 1500 m      0.93 0.79 0.62 1.36
//   384 x 80 kHz, 1500 m  6.6 6.3 6.7 7.8     12 x 1.28 MHz, 500 m     1.29 1.00 0.94 1.35
//   384 x 80 kHz, 3000 m  10.5 9.3 9.4 7.9    12 x 1.28 MHz, 1500 m    3.11 2.20 1.68 1.48
// A group's waves also start and write their visibilities once, which is what a few components cost (us,
// 128 tiles, 384 channels of 40 kHz, forms 0 to 3): one, shared beam 87 147 142, per-tile beams 105 175 169
// 96; 16, shared 286 356 378, per-tile 414 478 495 568. `start` holds it, in ms at 128 tiles.
int choose_shapelet_form(bool per_tile, int ncomp, int nchan, double step, double edges_per_hz) {
    struct Line {
        int span;  // channels of a group
        double start, at0, edge, most;
    };
    static const Line kShared[3] = {
        {64, 0.0122, 0.29, 0.092, 45.0}, {64, 0.022, 0.37, 0.071, 36.0}, {32, 0.0105, 0.25, 0.069, 20.0}};
    static const Line kOwn[4] = {{64, 0.014, 0.56, 0.099, 45.0}, {64, 0.026, 0.62, 0.075, 37.0},
                                 {32, 0.0123, 0.395, 0.069, 21.0}, {64, 0.0107, 1.29, 0.0132, 60.0}};
    int best = 0;
    double t_best = 0.0;
    for (int i = 0; i < (per_tile ? 4 : 3); ++i) {
        const Line &f = per_tile ? kOwn[i] : kShared[i];
        const double edges = edges_per_hz * step * std::min(nchan, f.span);
        const double each = (f.at0 + f.edge * fmin(edges, f.most)) / 200.0;
        const double t = ((nchan + f.span - 1) / f.span) * (f.start + ncomp * each);
        if (i == 0 || t < t_best) {
            best = i;
            t_best = t;
        }
    }
    return best;
}

template <bool PT> static hipError_t launch_shapelets(int form, const ShapeletChanArgs &a, hipStream_t stream) {
    switch (form) {
    case 0: return launch_shapelets_form<2, 2, 3, PT>(a, stream);
    case 1: return launch_shapelets_form<1, 1, 4, PT>(a, stream);
    default: return launch_shapelets_form<1, 2, 4, PT>(a, stream);
    }
}

// Mean table edges per Hz that a shapelet crosses, over up to 4096 of the (component, baseline) pairs.
__global__ __launch_bounds__(256) void k_shapelet_edges(size_t n, int nbl, const double4 *__restrict__ shape,
                                                        const double2 *__restrict__ bl_uv, double *out) {
    __shared__ double part[4];
    const size_t samples = n < 4096 ? n : 4096;
    double sum = 0.0;
    for (size_t i = threadIdx.x; i < samples; i += 256) {
        const size_t at = i * n / samples;
        const double4 sh = shape[at / nbl];
        const double2 uv = bl_uv[at];
        sum += fabs((uv.x * sh.x + uv.y * sh.y) * sh.z) + fabs((uv.x * sh.y - uv.y * sh.x) * sh.w);
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) *out = (part[0] + part[1] + part[2] + part[3]) / samples;
}

hipError_t launch_shapelet_edges(int ncomp, int nbl, const double4 *d_shape, const double2 *d_bl_uv, double *d_out,
                                 hipStream_t stream) {
    if (ncomp <= 0 || nbl <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_shapelet_edges, dim3(1), dim3(256), 0, stream, (size_t)ncomp * nbl, nbl, d_shape, d_bl_uv, d_out);
    return hipGetLastError();
}

hipError_t launch_shapelet_chan(bool per_tile, const ShapeletChanArgs &a, hipStream_t stream) {
    if (a.ncomp <= 0 || a.nbl <= 0 || a.nchan <= 0) return hipSuccess;
    const bool f32 = a.coh32 != nullptr;
    if (f32 && (a.sbf32 == nullptr || (per_tile && a.beam.coh_cls != nullptr && a.coh_cls32 == nullptr)))
        return hipErrorInvalidValue;
    const int form = choose_shapelet_form(per_tile, a.ncomp, a.nchan, a.step, a.edges_per_hz);
    if (!f32 && form < 3) return per_tile ? launch_shapelets<true>(form, a, stream) : launch_shapelets<false>(form, a, stream);
    // Per-tile beams: a.ngroups groups of 64 channels; FP32 shared beam: groups of 128 channels.
    const int total = ((a.nbl + 3) / 4) * (per_tile ? a.ngroups : (a.nchan + 127) / 128);
    hipLaunchKernelGGL(!per_tile ? k_shapelet_chan32 : (f32 ? k_shapelet_chan_tiles32 : k_shapelet_chan_tiles),
                       dim3(total), dim3(256), 0, stream, a);
    return hipGetLastError();
}

__global__ void k_to_f32(size_t n, const double *__restrict__ in, float *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

hipError_t launch_to_f32(size_t n, const double *d_in, float *d_out, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, n, d_in, d_out);
    return hipGetLastError();
}

// Tile UVWs from baseline UVWs: r_0 = 0, r_q = -uvw(0, q), so r_p - r_q = uvw(p, q) for
// UVWs that are differences of tile UVWs, as xyzs_to_cross_uvws produces.
__global__ void k_tile_uvw_from_baselines(int ntiles, const UVW *__restrict__ uvw, double *__restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntiles) return;
    if (t == 0) {
        out[0] = out[1] = out[2] = 0.0;
        return;
    }
    const UVW b = uvw[t - 1];  // baseline (0, t)
    out[3 * t] = -b.u;
    out[3 * t + 1] = -b.v;
    out[3 * t + 2] = -b.w;
}

hipError_t launch_tile_uvw_from_baselines(int ntiles, const UVW *d_uvw, double *d_out, hipStream_t stream) {
    hipLaunchKernelGGL(k_tile_uvw_from_baselines, dim3((ntiles + 255) / 256), dim3(256), 0, stream, ntiles, d_uvw,
                       d_out);
    return hipGetLastError();
}

}  // namespace sm
