// FP64 rotate/average from the cube by folded channel blocks, a wave at a time (gfx950): the route
// of batched pol-0 calls that take the Horner channel sums and name no tile.
//
// For a row and direction the sum over channels is exp(i sf kappa0) P(z) with
// P(z) = sum_c v_c z^c, z = exp(i theta), theta = sf dkappa, sf = -2 pi ((dd uvw).z - w)
// (CpuLeapCalibrator.cc:181-217 rotates every sample by itself).  It is taken in blocks of eight
// channels about their middle: with s = 1/2, 3/2, 5/2, 7/2 and the pairs v+, v- at the middle +- s,
//   p = sum_s (v+ + v-) cos(s theta) + i (v+ - v-) sin(s theta)
// and P(z) = z^(7/2) H, where H runs over the blocks by Horner's rule in w = z^8.  The pairs' sums and
// differences are formed once per sample for all directions and the eight cosines and sines once
// per row and direction, so a channel costs 2.5 FMAs a direction where Horner's rule over the
// channels costs four.  A (row, channel) with a non-finite pol is left out for every direction.
//
// Decomposition: a wave holds four rows, one in each 16 lanes; a lane holds ND directions of its row
// (16 ND directions a wave) and loads one of 16 channels of it, chunks of K samples a lane ahead
// in registers.  Lane n of a row folds its sample with its mirror's of the same eight channels, and the
// FMAs take the folded pairs from lanes 4 to 7 and 12 to 15 by DPP row broadcasts: samples do not
// pass through LDS, nothing is shared between waves but the phasor table, and there is no barrier
// in the loop.  The rows are RT timesteps of BB baselines (RT BB = 4): timesteps of one baseline where the
// set has few baselines, one timestep of four where it has enough; with few baselines the four
// waves of a workgroup take turns at one baseline's timesteps.
//
// The residual loss (Q) also keeps every row's sums, q[row][d] = (e0 P(z), e0 z P'(z)), so that its
// adjoint does not read the cube: z P'(z) = z^(7/2) (7/2 H + G) with G <- w G + 8 w H + p',
// p' = sum_s s ((v+ - v-) cos(s theta) + i (v+ + v-) sin(s theta)), beside H <- w H + p.
//
// With up to 32 directions it runs at the cube's bytes (256 stations, 32 t, 384 channels of
// complex64: 8 directions 2.27 ms, 32 directions 2.36 ms, 5.5 TB/s; 64 directions 3.56 ms, where its
// instructions cost more than the cube; Horner's rule over the channels took 2.41 ms and 5.35 ms).  128 antennas, 14 t, 48
// channels of complex128, 64 directions: 93 us, three quarters of it issued FP64 instructions.
// Row sums of 16 directions (128 stations, 64 t, 192 channels of complex64) 714 us against 849.
#include "batched_common.h"

#include <algorithm>
#include <type_traits>

namespace leap {
namespace {

using namespace dev;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;       // waves of a workgroup
constexpr int kLanes = 16;      // lanes of a row
constexpr int kRows = 64 / kLanes;
constexpr uint32_t kMaxND = 4, kMaxNDQ = 2;  // directions of a lane, with row sums

// Samples of a chunk per lane: those loaded ahead hold 8 to 32 registers.
constexpr int samples_ahead(int sample_bytes) { return sample_bytes > 16 ? 2 : 4; }

// Waves per SIMD that the registers of ND directions a lane allow.
constexpr int waves_per_simd(bool c128, int nd, bool q) {
    return nd > 2 || (nd > 1 && c128 && q) ? 2 : nd > 1 || c128 || q ? 3 : 4;
}

struct WaveArgs {
    const double* uvw;
    const double* dd;
    uint32_t D, dirs_per_block, T, nbl, C, bb_log2, split, pols_out;
    double kappa0, dkappa;
    double* avg;  // [interval][D][nbl][pols_out]
    double* q;    // [row][D][4]
    uint64_t* started;
};

// x of lane 7 - n in lane n of every eight lanes.
__device__ inline float half_mirror(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, true));
}
__device__ inline double half_mirror(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x141, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x141, 0xf, 0xf, true));
}

// h += sum_s a_s e_s.x + i b_s e_s.y over the four pairs in lanes HALF ? 12..15 : 4..7 of each 16 lanes,
// every lane with its own e_s = (cos, sin).  All lanes of the wave call it.  A lane's value written by
// a vector instruction may be read by DPP two wait states later: the leading s_nop.
#define LEAP_PAIR(N, C_, S_)                                                    \
    "v_fmac_f64_dpp %0, %2, " C_ " row_newbcast:" N " row_mask:0xf bank_mask:0xf\n"  \
    "v_fmac_f64_dpp %1, %3, " C_ " row_newbcast:" N " row_mask:0xf bank_mask:0xf\n"  \
    "v_fmac_f64_dpp %0, -%5, " S_ " row_newbcast:" N " row_mask:0xf bank_mask:0xf\n" \
    "v_fmac_f64_dpp %1, %4, " S_ " row_newbcast:" N " row_mask:0xf bank_mask:0xf\n"
template <int HALF>
__device__ inline void add_pairs(C2<double>& h, C2<double> a, C2<double> b, const C2<double> (&e)[4]) {
    if constexpr (HALF)
        asm volatile("s_nop 1\n" LEAP_PAIR("12", "%6", "%7") LEAP_PAIR("13", "%8", "%9") LEAP_PAIR("14", "%10", "%11")
                         LEAP_PAIR("15", "%12", "%13")
                     : "+v"(h.x), "+v"(h.y)
                     : "v"(a.x), "v"(a.y), "v"(b.x), "v"(b.y), "v"(e[0].x), "v"(e[0].y), "v"(e[1].x), "v"(e[1].y),
                       "v"(e[2].x), "v"(e[2].y), "v"(e[3].x), "v"(e[3].y));
    else
        asm volatile("s_nop 1\n" LEAP_PAIR("4", "%6", "%7") LEAP_PAIR("5", "%8", "%9") LEAP_PAIR("6", "%10", "%11")
                         LEAP_PAIR("7", "%12", "%13")
                     : "+v"(h.x), "+v"(h.y)
                     : "v"(a.x), "v"(a.y), "v"(b.x), "v"(b.y), "v"(e[0].x), "v"(e[0].y), "v"(e[1].x), "v"(e[1].y),
                       "v"(e[2].x), "v"(e[2].y), "v"(e[3].x), "v"(e[3].y));
}
#undef LEAP_PAIR

template <typename VT, int P, int ND, bool Q>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(waves_per_simd(sizeof(VT) == 8, ND, Q), 8))) void horner_wave_kernel(
    const VT* __restrict__ vis, const WaveArgs a) {
#pragma clang fp contract(off)
    constexpr int K = samples_ahead(2 * P * int(sizeof(VT)));
    constexpr uint32_t CC = kLanes * K;  // channels of a chunk
    stamp(a.started);
    __shared__ double2 s_table[kPhasorTable];
    __shared__ C2<double> s_part[kWaves][ND][64];
    phasor_table_init(s_table);
    __syncthreads();
    const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t blocks = (a.D + a.dirs_per_block - 1) / a.dirs_per_block;
    // (baselines, direction block), blocks fastest
    const uint32_t item = a.split ? blockIdx.x : blockIdx.x * kWaves + wave;
    const uint32_t BB = 1u << a.bb_log2, RT = kRows >> a.bb_log2;
    const uint32_t bl0 = (item / blocks) * BB;
    if (bl0 >= a.nbl) return;  // never in a split workgroup
    const uint32_t d0 = (item % blocks) * a.dirs_per_block;
    const uint32_t d_end = min(a.D, d0 + a.dirs_per_block);
    const size_t rows0 = size_t(blockIdx.y) * a.T * a.nbl;
    const uint32_t t_first = a.split ? wave * RT : 0, t_step = a.split ? kWaves * RT : RT;

    // this lane's row of a step, (timestep offset, baseline), and its directions
    const uint32_t row = lane / kLanes, l = lane % kLanes;
    const uint32_t my_t = row >> a.bb_log2, my_bl = bl0 + (row & (BB - 1));
    auto direction = [&](int j) { return d0 + l + j * kLanes; };
    double dz[ND][3];
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        const double* r = a.dd + size_t(min(direction(j), a.D - 1)) * 9 + 6;
        dz[j][0] = r[0];
        dz[j][1] = r[1];
        dz[j][2] = r[2];
    }

    // Loads past the set's rows or channels are clamped into it, so that every load goes to its registers
    // without a branch: such rows are not accumulated and such channels are folded as zero.
    struct Raw {
        VT x[2 * P];
    };
    Raw raw[K];
    const VT* base;
    auto row_at = [&](uint32_t t0) {
        const size_t r = rows0 + size_t(min(t0 + my_t, a.T - 1)) * a.nbl + min(my_bl, a.nbl - 1);
        base = vis + r * (size_t(a.C) * (2 * P));
    };
    auto load = [&](uint32_t c0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            typedef std::conditional_t<sizeof(VT) == 8, f64x2, f32x2> U;
            const U* p = reinterpret_cast<const U*>(base + size_t(min(c0 + kLanes * k + l, a.C - 1)) * (2 * P));
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const U u = p[q];
                raw[k].x[2 * q] = u.x;
                raw[k].x[2 * q + 1] = u.y;
            }
        }
    };
    C2<double> sum[K], dif[K];  // in lanes 4 to 7 and 12 to 15
    auto fold = [&](uint32_t c0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            VT f = VT(0);  // NaN where a pol is not finite
#pragma unroll
            for (int q = 0; q < 2 * P; ++q) f = fma(VT(0), raw[k].x[q], f);
            const bool ok = f == VT(0) && c0 + kLanes * k + l < a.C;
            const VT x = ok ? raw[k].x[0] : VT(0), y = ok ? raw[k].x[1] : VT(0);
            const double mx = half_mirror(x), my = half_mirror(y);
            sum[k] = {double(x) + mx, double(y) + my};
            dif[k] = {double(x) - mx, double(y) - my};
        }
    };
    double u, v, w;
    auto load_uvw = [&](uint32_t t) {
        u = v = w = 0.0;
        if (t < a.T && my_bl < a.nbl) {
            const double* r = a.uvw + (rows0 + size_t(t) * a.nbl + my_bl) * 3;
            u = r[0];
            v = r[1];
            w = r[2];
        }
    };

    C2<double> acc[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) acc[j] = {0.0, 0.0};
    const uint32_t last = (a.C - 1) / CC * CC;  // first channel of the last chunk
    const double weight = 0.5 + double(l % 4);  // s of the lane's pair
    row_at(t_first);
    load(last);
    load_uvw(t_first + my_t);
    for (uint32_t t0 = t_first; t0 < a.T; t0 += t_step) {
        double sf[ND];
        C2<double> e[ND][4], zb[ND], h[ND], g[Q ? ND : 1];
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            sf[j] = shift_factor(dz[j], u, v, w);
            const double theta = sf[j] * a.dkappa;
            const double2 half = phasor_table(s_table, 0.5 * theta), eight = phasor_table(s_table, 8.0 * theta);
            zb[j] = {eight.x, eight.y};
            e[j][0] = {half.x, half.y};
            const C2<double> z = cmul(e[j][0], e[j][0]);
#pragma unroll
            for (int s = 1; s < 4; ++s) e[j][s] = cmul(e[j][s - 1], z);
            h[j] = {0.0, 0.0};
            if constexpr (Q) g[j] = {0.0, 0.0};
        }
        const bool row_ok = t0 + my_t < a.T && my_bl < a.nbl;
        load_uvw(t0 + t_step + my_t);
        for (int32_t c0 = int32_t(last); c0 >= 0; c0 -= CC) {
            fold(uint32_t(c0));
            const bool next_row = c0 == 0;
            if (next_row) row_at(t0 + t_step);
            if (!next_row || t0 + t_step < a.T) load(next_row ? last : uint32_t(c0) - CC);
#pragma unroll
            for (int k = K - 1; k >= 0; --k) {
                auto block = [&](auto half) {
                    if (uint32_t(c0) + kLanes * k + 8 * half >= a.C) return;
#pragma unroll
                    for (int j = 0; j < ND; ++j) {
                        h[j] = horner_step(h[j], zb[j], C2<double>{0.0, 0.0});
                        if constexpr (Q) {
                            g[j] = horner_step(g[j], zb[j], C2<double>{8.0 * h[j].x, 8.0 * h[j].y});
                            add_pairs<half>(g[j], C2<double>{weight * dif[k].x, weight * dif[k].y},
                                            C2<double>{weight * sum[k].x, weight * sum[k].y}, e[j]);
                        }
                        add_pairs<half>(h[j], sum[k], dif[k], e[j]);
                    }
                };
                block(std::integral_constant<int, 1>());
                block(std::integral_constant<int, 0>());
            }
        }
        if (row_ok) {
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                const double2 e0 = phasor_table(s_table, sf[j] * a.kappa0);
                const C2<double> mid = cmul(C2<double>{e0.x, e0.y}, e[j][3]);  // e0 z^(7/2)
                const C2<double> r = cmul(mid, h[j]);
                acc[j].x += r.x;
                acc[j].y += r.y;
                if constexpr (Q) {
                    if (direction(j) < d_end) {
                        const C2<double> r1 = cmul(mid, C2<double>{fma(3.5, h[j].x, g[j].x), fma(3.5, h[j].y, g[j].y)});
                        f64x2* o = reinterpret_cast<f64x2*>(a.q) +
                                   ((rows0 + size_t(t0 + my_t) * a.nbl + my_bl) * a.D + direction(j)) * 2;
                        o[0] = f64x2{r.x, r.y};
                        o[1] = f64x2{r1.x, r1.y};
                    }
                }
            }
        }
    }
    // the timesteps of a baseline lie BB rows apart
    for (uint32_t m = BB * kLanes; m < 64; m *= 2) {
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            acc[j].x += __shfl_xor(acc[j].x, m, 64);
            acc[j].y += __shfl_xor(acc[j].y, m, 64);
        }
    }
    if (a.split) {  // the sums of the workgroup's waves
#pragma unroll
        for (int j = 0; j < ND; ++j) s_part[wave][j][lane] = acc[j];
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int j = 0; j < ND; ++j)
            for (int i = 1; i < kWaves; ++i) {
                acc[j].x += s_part[i][j][lane].x;
                acc[j].y += s_part[i][j][lane].y;
            }
    }
    if (my_t != 0 || my_bl >= a.nbl) return;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        const uint32_t d = direction(j);
        if (d >= d_end) continue;
        double* o = a.avg + ((size_t(blockIdx.y) * a.D + d) * a.nbl + my_bl) * (2 * a.pols_out);
        o[0] = acc[j].x;
        o[1] = acc[j].y;
        for (uint32_t q = 2; q < 2 * a.pols_out; ++q) o[q] = 0.0;  // pols not accumulated
    }
}

template <typename VT, int P, bool Q, int ND>
void launch_one(hipStream_t s, const void* vis, uint32_t intervals, uint32_t blocks, WaveArgs a) {
    // Baselines of a wave: four while that leaves three waves per SIMD, halved (for as many more
    // timesteps at a time) until it does; below two the timesteps of a baseline go over four waves.
    uint32_t bb = 2;
    auto waves = [&](uint32_t log2) { return uint64_t((a.nbl + (1u << log2) - 1) >> log2) * blocks * intervals; };
    while (bb > 0 && waves(bb) < 3072 && (uint32_t(kRows) >> bb) < a.T) --bb;
    a.bb_log2 = bb;
    a.split = bb == 0 && waves(0) < 2048 && a.T > kRows;
    const uint64_t items = uint64_t((a.nbl + (1u << bb) - 1) >> bb) * blocks;
    const uint64_t groups = a.split ? items : (items + kWaves - 1) / kWaves;
    require(groups < (1ull << 31) && intervals < 65536, LEAP_ERR_RANGE, "too many workgroups for one launch");
    horner_wave_kernel<VT, P, ND, Q>
        <<<dim3(uint32_t(groups), intervals), 64 * kWaves, 0, s>>>(static_cast<const VT*>(vis), a);
    LEAP_HIP(hipGetLastError());
}

template <typename VT, int P, bool Q>
void launch_nd(hipStream_t s, uint32_t nd, const void* vis, uint32_t intervals, uint32_t blocks, const WaveArgs& a) {
    switch (nd) {
        case 1: return launch_one<VT, P, Q, 1>(s, vis, intervals, blocks, a);
        case 2: return launch_one<VT, P, Q, 2>(s, vis, intervals, blocks, a);
        default: break;
    }
    if constexpr (!Q) {
        if (nd == 3) return launch_one<VT, P, Q, 3>(s, vis, intervals, blocks, a);
        return launch_one<VT, P, Q, 4>(s, vis, intervals, blocks, a);
    }
}

template <typename VT, bool Q>
void launch_pols(hipStream_t s, uint32_t nd, const void* vis, uint32_t P, uint32_t intervals, uint32_t blocks,
                 const WaveArgs& a) {
    switch (P) {
        case 1: return launch_nd<VT, 1, Q>(s, nd, vis, intervals, blocks, a);
        case 2: return launch_nd<VT, 2, Q>(s, nd, vis, intervals, blocks, a);
        case 3: return launch_nd<VT, 3, Q>(s, nd, vis, intervals, blocks, a);
        case 4: return launch_nd<VT, 4, Q>(s, nd, vis, intervals, blocks, a);
        default: throw Error(LEAP_ERR_NOT_IMPLEMENTED, "unsupported polarisation count");
    }
}

}  // namespace

// Directions of a lane: the fewest direction blocks of at most 16 max_nd directions, evenly filled;
// more and narrower ones while the set's baselines make fewer than 2,048 waves of them.
static uint32_t directions_per_lane(uint32_t D, uint32_t nbl, uint32_t intervals, uint32_t max_nd) {
    const uint32_t slots = (D + kLanes - 1) / kLanes;  // 16 directions
    uint32_t blocks = (slots + max_nd - 1) / max_nd;
    uint32_t nd = (slots + blocks - 1) / blocks;
    while (nd > 1 && uint64_t(nbl) * intervals * blocks < 2048) {
        --nd;
        blocks = (slots + nd - 1) / nd;
    }
    return nd;
}

int32_t horner_wave_tile(uint32_t D, uint32_t nbl, uint32_t intervals) {
    const uint32_t nd = directions_per_lane(D, nbl, intervals, kMaxND);
    return int32_t(kLanes * nd * 10 + nd);
}

void launch_horner_wave(hipStream_t s, const HornerWave& h) {
    if (h.nbl == 0 || h.D == 0 || h.intervals == 0 || h.T == 0) return;
    const uint32_t nd = directions_per_lane(h.D, h.nbl, h.intervals, h.q ? kMaxNDQ : kMaxND);
    const uint32_t blocks = (h.D + kLanes * nd - 1) / (kLanes * nd);
    const WaveArgs a{h.uvw, h.dd, h.D, (h.D + blocks - 1) / blocks, h.T, h.nbl, h.C, 0, 0, h.pols_out,
                     h.f0 / kSpeedOfLight, h.df / kSpeedOfLight, h.avg, h.q, h.started};
    const bool c64 = h.vis_dtype == LEAP_VIS_C64;
    if (h.q)
        (c64 ? launch_pols<float, true> : launch_pols<double, true>)(s, nd, h.vis, h.P, h.intervals, blocks, a);
    else
        (c64 ? launch_pols<float, false> : launch_pols<double, false>)(s, nd, h.vis, h.P, h.intervals, blocks, a);
}

}  // namespace leap
