// FP64 kernels of the per-direction ("plain") calibration path for gfx950.
//
//   dd_kernel               MetaData::GenerateDDMatrix (model/cpu/MetaData.cc:166-203)
//   rotate_average_f64      CpuLeapCalibrator::RotateVisibilities (CpuLeapCalibrator.cc:181-217)
//   assemble_ad_kernel      pinv(A) = G+ A^T from the Gram pseudo-inverse
//   cal1, delta_sum, cal and inversion_small kernels
//                           the inversion of CpuLeapCalibrator::PhaseRotate (:159-178)
//   gram_* kernels          G+ = pinv(A^T A) (MetaData.cc:111, :123)
//
// Layouts in HBM: visibilities MS-native [row][channel][pol] complex (c128 or
// c64); uvw [row][3] f64; avgData [direction][baseline][pol] complex128;
// Ad stored transposed as AdT [K][N] (row k = column k of Ad); cal [direction][N].
#include "batched_common.h"
#include "inversion_common.h"
#include "leap_internal.h"

#include <type_traits>

namespace leap {
namespace {

constexpr int kBlock = 256;       // 4 wave64 per workgroup
// ---------------------------------------------------------------------------
// dd matrices, one thread per direction; dd row-major [d][3][3].
// ---------------------------------------------------------------------------
__global__ void dd_kernel(double ra0, double dec0, const double* __restrict__ dirs, uint32_t D,
                          double* __restrict__ dd) {
#pragma clang fp contract(off)
    const uint32_t d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= D) return;
    const double ang1 = kPi / 2.0 - dec0;
    const double ang2 = dirs[2 * d] - ra0;
    const double ang3 = -kPi / 2.0 + dirs[2 * d + 1];
    double s1, c1, s2, c2, s3, c3;
    sincos(ang1, &s1, &c1);
    sincos(ang2, &s2, &c2);
    sincos(ang3, &s3, &c3);
    const double m1[9] = {1, 0, 0, 0, c1, -s1, 0, s1, c1};
    const double m2[9] = {c2, s2, 0, -s2, c2, 0, 0, 0, 1};
    const double m3[9] = {1, 0, 0, 0, c3, -s3, 0, s3, c3};
    double t[9];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            t[i * 3 + j] = m3[i * 3 + 0] * m2[j] + m3[i * 3 + 1] * m2[3 + j] + m3[i * 3 + 2] * m2[6 + j];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            dd[9 * d + i * 3 + j] = t[i * 3 + 0] * m1[j] + t[i * 3 + 1] * m1[3 + j] + t[i * 3 + 2] * m1[6 + j];
}

// ---------------------------------------------------------------------------
// rotate_average_f64: every (row, channel) sample of a baseline rotated by
// exp(i * shift), shift = sf(row) / lambda(channel), for up to ND directions at once
// and summed per direction; a sample whose rotated polarisations hold a NaN is skipped.
// No atomics and no write-back to the cube; the sum order depends on the set's shape
// alone, so a direction's result has the same bits whatever ND and the number of pols
// kept (PO: 1 for calibrations, which use pol 0 only; P otherwise).
//
// One pass serves ND directions because the cube is what a single direction waits for
// (5.9 TB/s on complex64, 6.0 to 6.2 on complex128, 4.2 ms for 26 GB), while a direction's
// own work is some 34 instructions per sample.  256 stations, 32 t, 384 ch, 4 pols: 4
// directions of the complex64 cube (13 GB) take 2.35 ms in one pass against 8.87 in four,
// 2 of the complex128 cube 4.36 against 8.34; 16 directions of 128 stations, 14 t, 48 ch
// (355 MB) 0.13 ms in two passes against 1.10 in sixteen, bound by the arithmetic.  There a wave
// has some ten samples a lane, and its sums over the lanes took 0.04 ms while their step sizes were
// variables and every value was picked by comparisons.
// A wave owns its samples of one baseline and holds ND sums per pol in registers:
//  - shift is the correctly rounded quotient: q = sf * r, r = RN(1 / lambda), then
//    fma(fma(-q, lambda, sf), r, q) (Markstein 1990), 3 instructions against a division's 11
//  - exp(i shift) from the 64-entry table in LDS (phasor_table)
//  - the rotated sample goes into the sums as four FMAs
// Samples that are not finite, a baseline's chunk of rows where a shift is not below 2^25 rad
// (looked at once a row and direction) and channels without a finite wavelength take the plain
// form (division, sincos, rotate every pol, look for a NaN), exactly as the reference does it.
// ---------------------------------------------------------------------------
constexpr double kMaxShift = 67108864.0;  // 2^26 rad, far inside the phasor table's range
constexpr double kMaxLambda = 0x1p900;    // longer ones (a channel at 0 Hz) are divided by
constexpr uint32_t kRowChunk = 32;          // rows whose shift factors a wave keeps in LDS
constexpr uint32_t kLambdaLds = 1024;       // channels whose wavelengths sit in LDS

template <typename T, int P>
struct VisLoad {
    T v[2 * P];
    VisLoad() = default;
    __device__ inline explicit VisLoad(const T* __restrict__ p) { load(p); }
    __device__ inline void load(const T* __restrict__ p) {
        typedef T T2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const T2 x = reinterpret_cast<const T2*>(p)[q];
            v[2 * q] = x.x;
            v[2 * q + 1] = x.y;
        }
    }
    // 0 * x is NaN exactly for infinities and NaNs.
    __device__ inline bool finite() const {
        T z = T(0);
#pragma unroll
        for (int q = 0; q < 2 * P; ++q) z = fma(T(0), v[q], z);
        return z == T(0);
    }
};

// Sums of N values over a wave: every step halves the values a lane holds while there is
// more than one, so N + 4 exchanges do instead of 6 N.  The lane's value is number
// wave_sum_index<N>(lane); each is summed over the lanes in the same tree whatever N.
template <int N, int M = 32>
__device__ inline double wave_sum_n(const double (&v)[N], uint32_t lane) {
    constexpr int H = N > 1 ? N / 2 : 1;  // the step's sizes are constants, so v stays in registers
    double s[H];
    if constexpr (N > 1) {
        const bool up = lane & M;
#pragma unroll
        for (int j = 0; j < H; ++j) {
            const double send = up ? v[j] : v[j + H], keep = up ? v[j + H] : v[j];
            s[j] = keep + __shfl_xor(send, M, 64);
        }
    } else {
        s[0] = v[0] + __shfl_xor(v[0], M, 64);
    }
    if constexpr (M > 1) return wave_sum_n<H, M / 2>(s, lane);
    return s[0];
}

template <int N>
__device__ inline uint32_t wave_sum_index(uint32_t lane) {
    return lane / (64 / N);  // the upper half of the values goes to the lanes with bit 32, and so on
}

constexpr int pow2_at_least(int n) {
    int p = 1;
    while (p < n) p *= 2;
    return p;
}

// Grid: (groups of directions fastest, baselines) x solution intervals; waves of a baseline:
// wpb (1: the workgroup's waves take one baseline each).  lambda2: (lambda, RN(1 / lambda)).
// avg[interval][direction][baseline][PO].
// Sixteen waves of a baseline (1,024 threads, 128 registers) with up to four directions a pass.
constexpr int max_threads(bool wide, int nd) { return wide || nd > 4 ? 256 : 1024; }

template <typename T, int P, int PO, int ND, bool kWide>
__global__ __launch_bounds__(max_threads(kWide, ND)) void rotate_average_f64(
    const T* __restrict__ vis, const double* __restrict__ uvw, const double* __restrict__ dd, uint32_t D,
    uint32_t groups, uint32_t wpb, uint32_t T_steps, uint32_t nbl, uint32_t C,
    const double2* __restrict__ lambda2, double* __restrict__ avg, uint64_t* __restrict__ started) {
#pragma clang fp contract(off)
    dev::stamp(started);
    constexpr int NV = pow2_at_least(2 * PO * ND);
    __shared__ double2 s_lambda[kLambdaLds];
    __shared__ double2 s_table[dev::kPhasorTable];
    // kWide, for 64-byte samples (4 complex128 pols) of which pol 0 is kept: a lane loading its own
    // sample strides the wave's four loads by 64 bytes and leaves the reuse of their lines to the
    // L1, which the waves in flight overflow.  So the wave loads its 64 samples as 256 consecutive
    // 16-byte units, a pol a lane, and hands the pol-0 units over through LDS.
    static_assert(!kWide || (PO == 1 && P * sizeof(T) == 32), "wide loads: four 16-byte pols, pol 0 kept");
    __shared__ double2 s_pol0[kWide ? 4 * 64 : 1];
    extern __shared__ double s_dyn[];  // shift factors [wave][row][ND], then partial sums [wave][NV]
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    double* s_sf = s_dyn + size_t(wave) * (kRowChunk * ND);
    double* s_red = s_dyn + size_t(waves) * (kRowChunk * ND);
    const bool in_lds = C <= kLambdaLds;
    if (in_lds)
        for (uint32_t c = threadIdx.x; c < C; c += blockDim.x) s_lambda[c] = lambda2[c];
    dev::phasor_table_init(s_table);
    __syncthreads();
    const uint32_t group = blockIdx.x % groups, block = blockIdx.x / groups;
    const uint32_t per_group = (D + groups - 1) / groups;
    const uint32_t d0 = group * per_group;
    const uint32_t active = min(per_group, D - d0);  // the host leaves no group empty
    const uint32_t bl = wpb == 1 ? block * waves + wave : block;
    const uint32_t part = wpb == 1 ? 0 : wave;  // this wave's share of the baseline's samples
    const size_t rows0 = size_t(blockIdx.y) * T_steps * nbl;
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) acc[q] = 0.0;

    if (bl < nbl) {
        // the largest |1 / lambda|, at an end of the band: one look at a row's shift factors stands for
        // its samples' shifts
        const double r_max = fmax(fabs(lambda2[0].y), fabs(lambda2[C - 1].y));
        const uint32_t step_t = 64 * wpb / C, step_c = 64 * wpb % C;
        for (uint32_t t0 = 0; t0 < T_steps; t0 += kRowChunk) {
            const uint32_t tn = min(kRowChunk, T_steps - t0);
            dev::wave_fence();  // the previous chunk's factors have been read
            bool far = false;
            for (uint32_t i = lane; i < tn * ND; i += 64) {
                const uint32_t t = i / ND, d = i % ND;
                const size_t row = rows0 + size_t(t0 + t) * nbl + bl;
                const double* dz = dd + size_t(min(d0 + d, D - 1)) * 9 + 6;
                const double u = uvw[3 * row], v = uvw[3 * row + 1], w = uvw[3 * row + 2];
                const double wrot = dz[0] * u + dz[1] * v + dz[2] * w;  // (dd * uvw).z, MetaData.cc:227
                s_sf[i] = -kTwoPi * (wrot - w);                        // CpuLeapCalibrator.cc:190
                far |= !(fabs(s_sf[i]) * r_max < 0.5 * kMaxShift);
            }
            dev::wave_fence();
            const bool near = !__any(far);
            // samples lane + 64 * (part + k * wpb) of the chunk, in (row, channel) order
            const size_t at0 = rows0 + size_t(t0) * nbl + bl;
            auto at = [&](uint32_t t, uint32_t c) { return vis + ((at0 + size_t(t) * nbl) * C + c) * (2 * P); };
            auto advance = [&](uint32_t& t, uint32_t& c) {
                t += step_t;
                c += step_c;
                if (c >= C) {
                    c -= C;
                    ++t;
                }
            };
            uint32_t t = (64 * part + lane) / C, c = (64 * part + lane) % C;
            VisLoad<T, P> next;                                  // !kWide: this lane's next sample
            uint32_t tu[kWide ? 4 : 1], cu[kWide ? 4 : 1];       // kWide: row and channel of unit 64 j + lane's sample
            double2 unit[kWide ? 4 : 1];
            auto load_units = [&] {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    unit[j] = make_double2(0.0, 0.0);
                    if (tu[j] < tn) unit[j] = reinterpret_cast<const double2*>(at(tu[j], cu[j]))[lane & 3];
                    advance(tu[j], cu[j]);
                }
            };
            if constexpr (kWide) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    tu[j] = (64 * part + 16 * j + lane / 4) / C;
                    cu[j] = (64 * part + 16 * j + lane / 4) % C;
                }
                load_units();
            } else if (t < tn) {
                next.load(at(t, c));
            }
            for (uint32_t first = 64 * part; kWide ? first < tn * C : t < tn; first += 64 * wpb) {
                double v[2 * PO];
                VisLoad<T, P> x;
                bool plain = true;
                if constexpr (kWide) {
                    bool bad = false;
                    dev::wave_fence();  // the batch before has been read
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        bad |= fma(0.0, unit[j].x, 0.0 * unit[j].y) != 0.0;  // also where it is NaN
                        if ((lane & 3) == 0) s_pol0[wave * 64 + 16 * j + lane / 4] = unit[j];
                    }
                    dev::wave_fence();
                    const double2 p0 = s_pol0[wave * 64 + lane];
                    load_units();
                    const bool look = __any(bad);  // one of the wave's 64 samples is not finite
                    if (t >= tn) break;            // the chunk's last samples need not fill the wave
                    v[0] = p0.x;
                    v[1] = p0.y;
                    if (look) plain = VisLoad<T, P>(at(t, c)).finite();
                } else {
                    x = next;
                    plain = x.finite();
#pragma unroll
                    for (int q = 0; q < 2 * PO; ++q) v[q] = double(x.v[q]);
                }
                const double* sf = s_sf + t * ND;
                const double2 l = in_lds ? s_lambda[c] : lambda2[c];
                const uint32_t ts = t, cs0 = c;
                advance(t, c);
                if constexpr (!kWide)
                    if (t < tn) next.load(at(t, c));
                plain = plain && near && fabs(l.x) < kMaxLambda;
                if (plain) {
#pragma unroll
                    for (int d = 0; d < ND; ++d) {
                        if ((d & 1) == 0 && uint32_t(d) >= active) break;
                        const double q = sf[d] * l.y;
                        const double shift = fma(fma(-q, l.x, sf[d]), l.y, q);  // sf / lambda, :195
                        const double2 e = dev::phasor_table(s_table, shift);
#pragma unroll
                        for (int q = 0; q < PO; ++q) {  // (a + ib)(cs + i sn), :198, :208-214
                            double* o = acc + 2 * (d * PO + q);
                            o[0] = fma(-v[2 * q + 1], e.y, fma(v[2 * q], e.x, o[0]));
                            o[1] = fma(v[2 * q + 1], e.x, fma(v[2 * q], e.y, o[1]));
                        }
                    }
                } else {
                    if constexpr (kWide) x.load(at(ts, cs0));
#pragma unroll 1
                    for (int d = 0; d < ND; ++d) {
                        double sn, cs, r[2 * P];
                        sincos(sf[d] / l.x, &sn, &cs);
                        bool nan = false;
#pragma unroll
                        for (int q = 0; q < P; ++q) {
                            const double a = double(x.v[2 * q]), b = double(x.v[2 * q + 1]);
                            r[2 * q] = a * cs - b * sn;
                            r[2 * q + 1] = a * sn + b * cs;
                            nan |= __builtin_isnan(r[2 * q]) || __builtin_isnan(r[2 * q + 1]);  // :201-206
                        }
#pragma unroll
                        for (int k = 0; k < ND; ++k)  // sums indexed by constants stay in registers
                            if (k == d && !nan)
#pragma unroll
                                for (int q = 0; q < 2 * PO; ++q) acc[2 * k * PO + q] += r[q];
                    }
                }
            }
        }
    }
    double s = wave_sum_n<NV>(acc, lane);
    const uint32_t v = wave_sum_index<NV>(lane);
    const bool first = lane % (64 / NV) == 0;
    if (wpb != 1) {  // the baseline's waves in order
        if (first) s_red[wave * NV + v] = s;
        __syncthreads();
        if (wave != 0) return;
        s = s_red[v];
        for (uint32_t w = 1; w < waves; ++w) s += s_red[w * NV + v];
    }
    const uint32_t d = v / (2 * PO);
    if (first && bl < nbl && d < active)
        avg[((size_t(blockIdx.y) * D + d0 + d) * nbl + bl) * (2 * PO) + v % (2 * PO)] = s;
}

// ---------------------------------------------------------------------------
// Ad assembly: AdT[k][i] = G+(i, a1_k) - G+(i, a2_k) for k < K-1 and
// AdT[K-1][i] = G+(i, c); G+ is symmetric, so G+(i, a) = Gp[a * N + i].
// ---------------------------------------------------------------------------
__global__ void assemble_ad_kernel(const double* __restrict__ Gp, int32_t N,
                                   const int2* __restrict__ pairs, int32_t n_pairs,
                                   int32_t constraint, double* __restrict__ AdT) {
    const int32_t k = blockIdx.x;
    if (k < n_pairs) {
        const int2 p = pairs[k];
        for (int32_t i = threadIdx.x; i < N; i += blockDim.x)
            AdT[size_t(k) * N + i] = Gp[size_t(p.x) * N + i] - Gp[size_t(p.y) * N + i];
    } else {
        for (int32_t i = threadIdx.x; i < N; i += blockDim.x)
            AdT[size_t(k) * N + i] = constraint < N ? Gp[size_t(constraint) * N + i] : 0.0;
    }
}

// ---------------------------------------------------------------------------
// Inversion of every direction d:
//   phase[k]  = arg(avg[d][I1[k]][pol 0]) for the rows k of A1, 0 at its constraint row
//   cal1[d]   = Ad1 * phase
//   delta[n]  = arg(exp(-2 pi i (cal1[a1_n] - cal1[a2_n])) * avg[d][n][pol 0]) for the rows
//               n of A (row n of avgData, as the reference indexes it; A * cal1 in gather
//               form, exact because each row of A is e_a1 - e_a2), 0 at its constraint row
//   cal[d]    = Ad * delta + cal1[d]
// The products go through Ad = G+ A^T: A^T y is each antenna's signed sum of its rows'
// values, and G+ applied to it is N x N, so a direction costs its rows and N^2 instead of
// K N with K about N^2 / 2.  The constraint's value is 0 and A^T y sums to 0 over each
// component, so G+ may be taken without the ones of the constraint's component (Gx), whose
// column of the constraint antenna is zero too: that antenna's sum is not needed.
// Latency-bound below some 50 directions, three launches of 5 to 8 us; 64 directions of 128
// antennas (8128 rows) take 24 us, where the split-K product with the K x N pseudo-inverse
// and the kernels around it took 150.
// ---------------------------------------------------------------------------

// Antenna j's signed sum of its rows' phases, 0 for the constraint.
__device__ inline double antenna_phase(const double* __restrict__ a_d, uint32_t nbl, uint32_t P, const PhaseRows& r,
                                       int32_t j) {
    double b = 0.0;
    if (j != r.constraint)
        for (int32_t e = r.csr_off[j]; e < r.csr_off[j + 1]; ++e) {
            const int32_t v = r.csr_ent[e];
            int32_t idx = r.I[v >> 1];
            if (idx < 0) idx += int32_t(nbl);  // VectorRangeSelect wrap (math/cpu/vector.h:97-104)
            const double* a = a_d + size_t(idx) * (2 * P);
            const double ph = atan2(a[1], a[0]);
            b += (v & 1) ? -ph : ph;
        }
    return b;
}

// cal1: one workgroup per (direction, 64 antennas), eight groups of 64 lanes taking every
// eighth column each; every workgroup forms the direction's antenna sums for itself (one
// arg per antenna when A1 is a star).
constexpr int32_t kCal1Groups = 8;
constexpr int32_t kCal1Chunk = 2048;  // antenna sums in LDS at once

__global__ __launch_bounds__(64 * kCal1Groups) void cal1_kernel(const double* __restrict__ avg, uint32_t nbl,
                                                                uint32_t P, const PhaseRows r,
                                                                double* __restrict__ cal1,
                                                                uint64_t* __restrict__ started) {
    dev::stamp(started);
    __shared__ double s_b[kCal1Chunk];
    __shared__ double s_part[kCal1Groups][64];
    const uint32_t d = blockIdx.x;
    const int32_t lane = threadIdx.x % 64, group = threadIdx.x / 64;
    const int32_t i = blockIdx.y * 64 + lane, ic = min(i, r.N - 1);
    const double* a_d = avg + size_t(d) * nbl * (2 * P);
    double acc = 0.0;
    for (int32_t j0 = 0; j0 < r.N; j0 += kCal1Chunk) {
        const int32_t jn = min(kCal1Chunk, r.N - j0);
        __syncthreads();
        for (int32_t j = threadIdx.x; j < jn; j += 64 * kCal1Groups) {
            s_b[j] = antenna_phase(a_d, nbl, P, r, j0 + j);
        }
        __syncthreads();
#pragma unroll 8
        for (int32_t j = group; j < jn; j += kCal1Groups) acc = fma(r.Gx[size_t(j0 + j) * r.N + ic], s_b[j], acc);
    }
    s_part[group][lane] = acc;
    __syncthreads();
    if (group != 0 || i >= r.N) return;
    for (int g = 1; g < kCal1Groups; ++g) acc += s_part[g][lane];
    cal1[size_t(d) * r.N + i] = acc;
}

// sums[d][a] = A^T delta: one wave per (direction, antenna) over the antenna's rows.  Each
// row's delta is formed by both of its antennas, which costs less than a launch and an array
// between them up to a few million rows in all (256 directions of 256 antennas: 125 us).
__global__ __launch_bounds__(kBlock) void delta_sum_kernel(const double* __restrict__ avg, uint32_t nbl, uint32_t P,
                                                           const PhaseRows r, const double* __restrict__ cal1,
                                                           double* __restrict__ sums) {
#pragma clang fp contract(off)
    const uint32_t d = blockIdx.x, lane = threadIdx.x % 64;
    const int32_t a = int32_t(blockIdx.y * (kBlock / 64) + threadIdx.x / 64);
    if (a >= r.N) return;  // whole waves
    double acc = 0.0;
    if (a != r.constraint)
        for (int32_t e = r.csr_off[a] + int32_t(lane); e < r.csr_off[a + 1]; e += 64) {
            const int32_t v = r.csr_ent[e];
            const double t = dev::delta_phase(avg, nbl, P, r.pairs, r.K, r.N, cal1, d, v >> 1);
            acc += (v & 1) ? -t : t;
        }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) sums[size_t(d) * r.N + a] = acc;
}

// cal[d][a] = Gx[a][:] . sums[d] + cal1[d][a]: one wave per (direction, antenna).
__global__ __launch_bounds__(kBlock) void cal_kernel(const double* __restrict__ Gx, int32_t N,
                                                     const double* __restrict__ sums, const double* __restrict__ cal1,
                                                     double* __restrict__ cal) {
    const uint32_t d = blockIdx.x, lane = threadIdx.x % 64;
    const int32_t a = int32_t(blockIdx.y * (kBlock / 64) + threadIdx.x / 64);
    if (a >= N) return;  // whole waves
    const double* row = Gx + size_t(a) * N;
    const double* x = sums + size_t(d) * N;
    double acc = 0.0;
#pragma unroll 4
    for (int32_t j = int32_t(lane); j < N; j += 64) acc = fma(row[j], x[j], acc);
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) cal[size_t(d) * N + a] = acc + cal1[size_t(d) * N + a];
}

// The three kernels above for one direction a workgroup, where a direction's rows and antennas fit one:
// each thread forms one row's delta, each wave sums the antennas' rows from LDS.  Sums in the same
// order, so the same bits.  Six stations, one direction: a call 36 us with the three launches, 32 with
// one; 45 antennas (990 rows), 512 directions 342 and 333.
constexpr int32_t kSmallWaves = 16, kSmallRows = 64 * kSmallWaves, kSmallAntennas = 64;

__global__ __launch_bounds__(kSmallRows) void inversion_small_kernel(const double* __restrict__ avg, uint32_t nbl,
                                                                     uint32_t P, const PhaseRows r1, const PhaseRows r,
                                                                     double* __restrict__ cal,
                                                                     uint64_t* __restrict__ started) {
#pragma clang fp contract(off)
    dev::stamp(started);
    __shared__ double s_b[kSmallAntennas], s_cal1[kSmallAntennas], s_sums[kSmallAntennas];
    __shared__ double s_part[kCal1Groups][64];
    __shared__ double s_delta[kSmallRows];
    const uint32_t d = blockIdx.x;
    const int32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const double* a_d = avg + size_t(d) * nbl * (2 * P);
    if (int32_t(threadIdx.x) < r1.N) s_b[threadIdx.x] = antenna_phase(a_d, nbl, P, r1, threadIdx.x);
    __syncthreads();
    if (wave < kCal1Groups) {
        double acc = 0.0;
        const int32_t ic = min(lane, r1.N - 1);
        for (int32_t j = wave; j < r1.N; j += kCal1Groups) acc = fma(r1.Gx[size_t(j) * r1.N + ic], s_b[j], acc);
        s_part[wave][lane] = acc;
    }
    __syncthreads();
    if (wave == 0 && lane < r1.N) {
        double acc = s_part[0][lane];
        for (int g = 1; g < kCal1Groups; ++g) acc += s_part[g][lane];
        s_cal1[lane] = acc;
    }
    __syncthreads();
    const int32_t n = int32_t(threadIdx.x);
    if (n < r.K - 1) s_delta[n] = dev::delta_phase(avg, nbl, P, r.pairs, r.K, 0, s_cal1, d, n);
    __syncthreads();
    for (int32_t a = wave; a < r.N; a += kSmallWaves) {
        double acc = 0.0;
        if (a != r.constraint)
            for (int32_t e = r.csr_off[a] + lane; e < r.csr_off[a + 1]; e += 64) {
                const int32_t v = r.csr_ent[e];
                const double t = s_delta[v >> 1];
                acc += (v & 1) ? -t : t;
            }
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (lane == 0) s_sums[a] = acc;
    }
    __syncthreads();
    for (int32_t a = wave; a < r.N; a += kSmallWaves) {
        double acc = lane < r.N ? fma(r.Gx[size_t(a) * r.N + lane], s_sums[lane], 0.0) : 0.0;
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (lane == 0) cal[size_t(d) * r.N + a] = acc + s_cal1[a];
    }
}

// ---------------------------------------------------------------------------
// Moore-Penrose inverse of the Gram matrix G = A^T A (N x N), for A the baseline
// rows e_a1 - e_a2 plus the constraint row e_c.  G is a graph Laplacian L plus
// e_c e_c^T, formed exactly (small integers).  Over the components S of the baseline
// graph (an unused antenna is one of its own), with J the matrix of ones:
//   c in S:      G_SS 1 = e_c, so G+_SS = X + J with X the inverse of L_SS without
//                row and column c (zero there): the ones are exact and X is a well
//                conditioned inverse (about |S| against |S|^2 for G_SS itself)
//   c not in S:  G+_SS = (L_SS + J / |S|)^-1 - J / |S|
// and zero between components.  So the matrix M to invert is L with the identity in
// row and column c and J / |S| added over the components without c; it is block
// diagonal, the zeros between blocks stay exact below, and it is inverted whole,
// without sorting the antennas.
//
// M^-1 by block sweeps (Gauss-Jordan on 32 x 32 blocks without pivoting, which a
// positive definite matrix does not need): the sweep of block k with P = M_kk^-1
// takes M_ij to M_ij - M_ik P M_kj, M_ik to M_ik P, M_kk to -P; after every block
// has been swept the matrix is -M^-1.  A launch per sweep: each workgroup owns one
// 32 x 32 tile of the lower triangle and its mirror image, inverts M_kk for itself
// (32 rank-1 steps with one barrier each, which are most of a sweep's time) and
// writes the other of two buffers, so a sweep reads only what the previous one left.
// Latency-bound: 10 us a sweep whatever N, one sweep per 32 antennas, both matrices
// (A, A1) of a metadata in the same launches.  One workgroup per component doing a
// left-looking Cholesky, as before, took 2.8 ms per matrix at 128 antennas and
// 14.5 ms at 256 on a single CU.
// ---------------------------------------------------------------------------
constexpr int32_t kGramTile = 32;
constexpr int32_t kGramRows = 4096;  // antennas whose counts sit in LDS at once

// Column a of M: counts of the rows joining a to every antenna (LDS integers, so
// repeated baselines add up in any order), a's degree on the diagonal, 1 / |S| on a's
// component when it has no constraint.
__global__ __launch_bounds__(kBlock) void gram_matrix_kernel(const GramPinv* __restrict__ mats, int32_t N) {
    __shared__ int32_t s_count[kGramRows];
    const GramPinv m = mats[blockIdx.y];
    const int32_t a = blockIdx.x;
    const int32_t e0 = m.csr_off[a], e1 = m.csr_off[a + 1];
    const double shift = m.shift[a];
    const int32_t comp = m.comp[a];
    for (int32_t r0 = 0; r0 < N; r0 += kGramRows) {
        const int32_t rn = min(kGramRows, N - r0);
        for (int32_t i = threadIdx.x; i < rn; i += kBlock) s_count[i] = 0;
        __syncthreads();
        for (int32_t e = e0 + int32_t(threadIdx.x); e < e1; e += kBlock) {
            const int32_t v = m.csr_ent[e];  // 2 k + (a is antenna2 of row k)
            const int2 p = m.pairs[v >> 1];
            const int32_t other = ((v & 1) ? p.x : p.y) - r0;
            if (other >= 0 && other < rn) atomicAdd(&s_count[other], 1);
        }
        __syncthreads();
        for (int32_t i = threadIdx.x; i < rn; i += kBlock) {
            const int32_t r = r0 + i;
            double x = r == a ? double(e1 - e0) : -double(s_count[i]);
            if (m.comp[r] == comp) x += shift;
            if (r == m.constraint || a == m.constraint) x = r == a ? 1.0 : 0.0;
            m.buf[0][size_t(a) * N + r] = x;
        }
        __syncthreads();
    }
}

// Sweep of block k; grid (lower-triangle tiles, matrices).  Thread t owns row t / 8,
// columns 4 (t % 8) .. + 3 of each tile.  The last sweep writes G+ itself, and G+ without
// the ones of the constraint's component (X above) where it is asked for.
__global__ __launch_bounds__(kBlock) void gram_sweep_kernel(const GramPinv* __restrict__ mats, int32_t N, int32_t k,
                                                            int32_t last) {
    constexpr int32_t B = kGramTile, LD = B + 2;  // rows of 34 doubles: 16-byte aligned, banks shifted by 4
    __shared__ double s_p[B][LD], s_l[B][LD], s_r[B][LD], s_q[B][LD];
    __shared__ double s_row[2][B], s_col[2][B];
    const GramPinv m = mats[blockIdx.y];
    const double* src = m.buf[k & 1];
    double* dst = m.buf[(k & 1) ^ 1];
    // tile (bi, bj), bi >= bj, from the triangular index
    int32_t bi = int32_t((sqrtf(8.0f * float(blockIdx.x) + 1.0f) - 1.0f) * 0.5f);
    while (bi * (bi + 1) / 2 > int32_t(blockIdx.x)) --bi;
    while ((bi + 1) * (bi + 2) / 2 <= int32_t(blockIdx.x)) ++bi;
    const int32_t bj = int32_t(blockIdx.x) - bi * (bi + 1) / 2;
    const int32_t r = int32_t(threadIdx.x) / 8, c = int32_t(threadIdx.x) % 8 * 4;
    // element (i, j) of the padded matrix: the identity past N
    auto at = [&](int32_t i, int32_t j) {
        return i < N && j < N ? src[size_t(i) * N + j] : (i == j ? 1.0 : 0.0);
    };
    double p[4], x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        p[q] = at(k * B + r, k * B + c + q);
        x[q] = at(bi * B + r, bj * B + c + q);
        s_l[r][c + q] = at(bi * B + r, k * B + c + q);  // M_ik
        s_r[r][c + q] = at(k * B + r, bj * B + c + q);  // M_kj
    }
    // -P = -M_kk^-1 by rank-1 sweeps; the next pivot's row and column are published in
    // the buffer that the step before has finished reading.
    if (r == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) s_row[0][c + q] = p[q];
    if (c == 0) s_col[0][r] = p[0];
    for (int32_t s = 0; s < B; ++s) {
        __syncthreads();
        const int b = s & 1;
        const double pivot = s_row[b][s];
        if (!(pivot > 0.0) && blockIdx.x == 0 && threadIdx.x == 0) *m.status = 1;
        const double inv = 1.0 / pivot;
        const double f = s_col[b][r] * inv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double row = s_row[b][c + q];
            const bool on_col = c + q == s;
            if (r == s) p[q] = on_col ? -inv : row * inv;
            else p[q] = on_col ? f : fma(-f, row, p[q]);
        }
        if (s + 1 < B) {
            if (r == s + 1)
#pragma unroll
                for (int q = 0; q < 4; ++q) s_row[b ^ 1][c + q] = p[q];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c + q == s + 1) s_col[b ^ 1][r] = p[q];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) s_p[r][c + q] = -p[q];
    __syncthreads();
    if (bi == k && bj == k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = p[q];
    } else {
        // q = P M_kj (bj != k), or M_ik P (bj == k) which is the tile itself
        const double(*u)[LD] = bj == k ? s_l : s_p;
        const double(*v)[LD] = bj == k ? s_p : s_r;
        double y[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
        for (int32_t l = 0; l < B; ++l) {
            const double ul = u[r][l];
#pragma unroll
            for (int q = 0; q < 4; ++q) y[q] = fma(ul, v[l][c + q], y[q]);
        }
        if (bi == k || bj == k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = y[q];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) s_q[r][c + q] = y[q];
            __syncthreads();
#pragma unroll 8
            for (int32_t l = 0; l < B; ++l) {
                const double ul = s_l[r][l];
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = fma(-ul, s_q[l][c + q], x[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int32_t i = bi * B + r, j = bj * B + c + q;
        if (i >= N || j > i) continue;  // the mirror image of (i, j) is (j, i)
        const size_t ij = size_t(i) * N + j, ji = size_t(j) * N + i;
        if (!last) {
            dst[ij] = dst[ji] = x[q];
            continue;
        }
        const bool joined = m.comp[i] == m.comp[j];
        double v = -x[q] - (joined ? m.shift[i] : 0.0);
        if (i == m.constraint && j == m.constraint) v = 0.0;
        if (m.Gx) m.Gx[ij] = m.Gx[ji] = v;
        if (joined && m.constraint < N && m.comp[i] == m.comp[m.constraint]) v += 1.0;
        m.Gp[ij] = m.Gp[ji] = v;
    }
}

template <typename T, int P, int PO, int ND>
void launch_rotate_nd(hipStream_t s, const RotateF64& a) {
    const uint32_t groups = (a.D + ND - 1) / ND;
    const uint32_t waves = a.wpb == 1 ? 4 : a.wpb;
    const uint64_t blocks = uint64_t(groups) * (a.wpb == 1 ? (a.nbl + 3) / 4 : a.nbl);
    require(blocks < (1ull << 31) && a.intervals < 65536, LEAP_ERR_RANGE, "too many workgroups for one launch");
    constexpr int NV = pow2_at_least(2 * PO * ND);
    const size_t lds = size_t(waves) * (kRowChunk * ND + NV) * sizeof(double);
    auto launch = [&](auto wide) {
        rotate_average_f64<T, P, PO, ND, decltype(wide)::value>
            <<<dim3(uint32_t(blocks), a.intervals), 64 * waves, lds, s>>>(static_cast<const T*>(a.vis), a.uvw, a.dd, a.D,
                                                                         groups, a.wpb, a.T, a.nbl, a.C, a.lambda2,
                                                                         a.avg, a.started);
        LEAP_HIP(hipGetLastError());
    };
    // Wide loads up to 4 directions, where the visibilities are the bound; with 8 their registers
    // cost half the waves (16 directions on 355 MB: 220 us against 130).
    if constexpr (PO == 1 && P * sizeof(T) == 32 && ND <= 4) {
        if (waves <= 4) return launch(std::true_type{});
    }
    launch(std::false_type{});
}

template <typename T, int P>
void launch_rotate_pols(hipStream_t s, const RotateF64& a, uint32_t nd) {
    if (a.pols_out == 1) {
        switch (nd) {
            case 1: return launch_rotate_nd<T, P, 1, 1>(s, a);
            case 2: return launch_rotate_nd<T, P, 1, 2>(s, a);
            case 4: return launch_rotate_nd<T, P, 1, 4>(s, a);
            default: return launch_rotate_nd<T, P, 1, 8>(s, a);
        }
    }
    if constexpr (P > 1) {
        if (nd == 1) return launch_rotate_nd<T, P, P, 1>(s, a);
        return launch_rotate_nd<T, P, P, 2>(s, a);
    }
}

template <typename T>
void launch_rotate_typed(hipStream_t s, const RotateF64& a, uint32_t nd) {
    switch (a.P) {
        case 1: return launch_rotate_pols<T, 1>(s, a, nd);
        case 2: return launch_rotate_pols<T, 2>(s, a, nd);
        case 3: return launch_rotate_pols<T, 3>(s, a, nd);
        case 4: return launch_rotate_pols<T, 4>(s, a, nd);
        default: throw Error(LEAP_ERR_NOT_IMPLEMENTED, "unsupported polarisation count");
    }
}

}  // namespace

void launch_dd(hipStream_t s, double ra0, double dec0, const double* d_dirs, uint32_t D, double* d_dd) {
    if (D == 0) return;
    dd_kernel<<<(D + 63) / 64, 64, 0, s>>>(ra0, dec0, d_dirs, D, d_dd);
    LEAP_HIP(hipGetLastError());
}

void launch_rotate_f64(hipStream_t s, const RotateF64& in) {
    if (in.nbl == 0 || in.D == 0 || in.intervals == 0) return;
    RotateF64 a = in;
    // Waves of a baseline, from the set's shape alone: one where the baselines alone are
    // 4 waves per SIMD, four below, sixteen where even those leave most SIMDs empty and a
    // baseline has samples for all of them.
    a.wpb = a.nbl >= 4096 ? 1 : a.nbl < 512 && uint64_t(a.T) * a.C >= 4096 ? 16 : 4;
    // Directions per pass: as many as D has, up to 8, but no more than leaves 4 waves per SIMD
    // (splitting the directions over workgroups shortens each wave's chain instead).
    const uint64_t waves = uint64_t(a.nbl) * a.wpb * a.intervals;
    uint32_t nd = a.pols_out != 1 ? 2 : a.wpb > 4 ? 4 : 8;
    while (nd > 1 && (nd / 2 >= a.D || waves * ((a.D + nd - 1) / nd) < 4096)) nd /= 2;
    if (a.vis_dtype == LEAP_VIS_C64)
        launch_rotate_typed<float>(s, a, nd);
    else
        launch_rotate_typed<double>(s, a, nd);
}

void launch_gram_pinv(hipStream_t s, const GramPinv* d_mats, uint32_t n_mats, int32_t N) {
    if (n_mats == 0 || N == 0) return;
    gram_matrix_kernel<<<dim3(uint32_t(N), n_mats), kBlock, 0, s>>>(d_mats, N);
    LEAP_HIP(hipGetLastError());
    const int32_t blocks = (N + kGramTile - 1) / kGramTile;
    for (int32_t k = 0; k < blocks; ++k) {
        gram_sweep_kernel<<<dim3(uint32_t(blocks) * (blocks + 1) / 2, n_mats), kBlock, 0, s>>>(d_mats, N, k,
                                                                                              k + 1 == blocks);
        LEAP_HIP(hipGetLastError());
    }
}

void launch_assemble_ad(hipStream_t s, const double* Gp, int32_t N, const int2* pairs, int32_t n_pairs,
                        int32_t constraint, double* AdT) {
    assemble_ad_kernel<<<n_pairs + 1, kBlock, 0, s>>>(Gp, N, pairs, n_pairs, constraint, AdT);
    LEAP_HIP(hipGetLastError());
}

void launch_cal1(hipStream_t s, const leap_metadata& md, const double* avg, uint32_t avg_pols, uint32_t D,
                 double* cal1, uint64_t* started) {
    if (D == 0) return;
    const PhaseRows r = md.rows_of_A1();
    cal1_kernel<<<dim3(D, uint32_t(r.N + 63) / 64), 64 * kCal1Groups, 0, s>>>(avg, md.nbl, avg_pols, r, cal1, started);
    LEAP_HIP(hipGetLastError());
}

void launch_inversion_f64(hipStream_t s, const leap_metadata& md, const double* avg, uint32_t avg_pols, uint32_t D,
                          double* cal1, double* sums, double* cal, uint64_t* started) {
    if (D == 0) return;
    const PhaseRows r = md.rows_of_A();
    if (r.N <= kSmallAntennas && r.K - 1 <= kSmallRows) {
        inversion_small_kernel<<<D, kSmallRows, 0, s>>>(avg, md.nbl, avg_pols, md.rows_of_A1(), r, cal, started);
        LEAP_HIP(hipGetLastError());
        return;
    }
    launch_cal1(s, md, avg, avg_pols, D, cal1, started);
    const dim3 grid(D, uint32_t(r.N + kBlock / 64 - 1) / (kBlock / 64));
    delta_sum_kernel<<<grid, kBlock, 0, s>>>(avg, md.nbl, avg_pols, r, cal1, sums);
    LEAP_HIP(hipGetLastError());
    cal_kernel<<<grid, kBlock, 0, s>>>(r.Gx, r.N, sums, cal1, cal);
    LEAP_HIP(hipGetLastError());
}

}  // namespace leap
