// FP64 Horner rotate/average from the cube, a wave at a time (gfx950): the route of
// batched pol-0 calls that take the Horner channel sums and name no tile.
//
// For a row and direction the sum over channels is exp(i sf kappa0) P(z) with
// P(z) = sum_c v_c z^c, z = exp(i sf dkappa), sf = -2 pi ((dd uvw).z - w), evaluated as two
// interleaved Horner chains P(z) = P_even(z^2) + z P_odd(z^2): four FMAs per channel and
// direction (CpuLeapCalibrator.cc:181-217 rotates every sample by itself).  A (row, channel)
// with a non-finite pol is left out for every direction.
//
// Decomposition: a wave holds RW = 64 / L rows at a time, L lanes a row with ND directions
// each.  The rows are RT timesteps of BB baselines (RT BB = RW): many timesteps of one
// baseline where the set has few baselines, one timestep of many where it has enough, so
// that short observations and short solution intervals leave no lane without a row.  Chunks
// of CC channels of each row (128 or 256 samples, from the last channels down) are loaded a
// chunk ahead into registers, lanes over samples, and handed to the direction lanes through
// wave-private LDS as FP64 pol 0, zero where a pol is not finite.  Nothing is shared between
// waves but the phasor table, so there is no barrier in the loop: each wave's loads hide
// behind the chains of the others on its SIMD.  A lane reads a channel once (16 bytes, the
// same for the lanes of a row) for 4 ND FMAs; with ND = 2 the LDS returns what the four SIMDs
// consume.
//
// The workgroup-wide tiles of kernels_batched.hip copy with global_load_lds behind two
// barriers a chunk and pad a row's channels to whole chunks and its timesteps to the rows in
// flight, which costs most where rows are short.  128 antennas, 48 channels: 14 timesteps, 64
// directions 117 us against 169 on complex128 (95 against 137 on complex64); one timestep, 16
// directions 10 us against 47.  256 stations, 32 t, 384 channels of complex64: 8 directions 2.41 ms
// against 3.49 (5.4 TB/s), 64 directions 5.35 against 5.34 (39 TFLOP/s, bound by the FMAs).
#include "batched_common.h"

#include <type_traits>

namespace leap {
namespace {

using namespace dev;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// Samples of a chunk per lane: those loaded ahead hold 16 or 32 registers.
constexpr int samples_ahead(int sample_bytes) { return sample_bytes > 16 ? 2 : 4; }
constexpr int kWaves = 4;      // waves of a workgroup, independent of each other

struct WaveArgs {
    const double* uvw;
    const double* dd;
    uint32_t D, dirs_per_block, T, nbl, C, bb_log2, pols_out;
    double kappa0, dkappa;
    double* avg;  // [interval][D][nbl][pols_out]
};

// Waves per SIMD: four, three where a chunk of 64-byte samples ahead takes 32 registers, two
// where a lane carries four directions.
constexpr int waves_per_simd(int sample_bytes, int nd) { return nd > 2 ? 2 : sample_bytes > 32 ? 3 : 4; }

template <typename VT, int P, int L, int ND>
__global__ __launch_bounds__(64 * kWaves)
__attribute__((amdgpu_waves_per_eu(waves_per_simd(2 * P * int(sizeof(VT)), ND), 8))) void horner_wave_kernel(const VT* __restrict__ vis, const WaveArgs a) {
#pragma clang fp contract(off)
    constexpr int RW = 64 / L;
    constexpr int K = samples_ahead(2 * P * int(sizeof(VT)));
    constexpr int CC = 64 * K / RW;
    static_assert(CC % 2 == 0, "chunks hold whole channel pairs");
    constexpr int PAD = L < 16 ? 1 : 0;  // a 16-lane group of a read spans rows: other banks
    __shared__ C2<double> s_v[kWaves][RW][CC + PAD];
    __shared__ double2 s_table[kPhasorTable];
    phasor_table_init(s_table);
    __syncthreads();
    const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    auto& v = s_v[wave];
    const uint32_t blocks = (a.D + a.dirs_per_block - 1) / a.dirs_per_block;
    const uint32_t item = blockIdx.x * kWaves + wave;  // (baselines, direction block), blocks fastest
    const uint32_t BB = 1u << a.bb_log2, RT = RW >> a.bb_log2;
    const uint32_t bl0 = (item / blocks) * BB;
    if (bl0 >= a.nbl) return;
    const uint32_t d0 = (item % blocks) * a.dirs_per_block;
    const uint32_t d_end = min(a.D, d0 + a.dirs_per_block);
    const size_t rows0 = size_t(blockIdx.y) * a.T * a.nbl;

    // this lane's row of a step, (timestep offset, baseline), and its directions
    const uint32_t row = lane / L, l = lane % L;
    const uint32_t my_t = row >> a.bb_log2, my_bl = bl0 + (row & (BB - 1));
    double dz[ND][3];
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        const double* r = a.dd + size_t(min(d0 + l + j * L, a.D - 1)) * 9 + 6;
        dz[j][0] = r[0];
        dz[j][1] = r[1];
        dz[j][2] = r[2];
    }

    // The samples of a chunk are (row i / CC, channel i % CC) for i = lane + 64 k: the lane's first
    // one and, for k > 0, that many rows (or, in wide chunks, channels) further.  The rows' bits of
    // k do not overlap the lane's, so a sample's address is the lane's plus a uniform step.
    struct Raw {
        VT x[2 * P];
    };
    Raw raw[K];
    const uint32_t r_lane = CC >= 64 ? 0 : lane / CC, c_lane = CC >= 64 ? lane : lane % CC;
    const uint32_t t_lane = r_lane >> a.bb_log2, bl_lane = bl0 + (r_lane & (BB - 1));
    const VT* p_lane = vis + ((rows0 + size_t(t_lane) * a.nbl + bl_lane) * a.C + c_lane) * (2 * P);
    auto load = [&](uint32_t t0, uint32_t c0) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            constexpr int per_row = CC >= 64 ? CC / 64 : 1;
            const uint32_t rk = CC >= 64 ? k / per_row : k * (64 / CC), ck = CC >= 64 ? 64 * (k % per_row) : 0;
            const uint32_t tk = t0 + (rk >> a.bb_log2), bk = rk & (BB - 1);  // uniform
            if (tk + t_lane < a.T && bk + bl_lane < a.nbl && c0 + ck + c_lane < a.C) {
                const VT* p = p_lane + ((size_t(tk) * a.nbl + bk) * a.C + c0 + ck) * (2 * P);
                typedef std::conditional_t<sizeof(VT) == 8, f64x2, f32x2> U;
#pragma unroll
                for (int q = 0; q < P; ++q) {
                    const U u = reinterpret_cast<const U*>(p)[q];
                    raw[k].x[2 * q] = u.x;
                    raw[k].x[2 * q + 1] = u.y;
                }
            } else {
#pragma unroll
                for (int q = 0; q < 2 * P; ++q) raw[k].x[q] = VT(0);
            }
        }
    };
    auto hand_over = [&] {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t i = lane + 64 * k;
            VT z = VT(0);  // NaN where a pol is not finite
#pragma unroll
            for (int q = 0; q < 2 * P; ++q) z = fma(VT(0), raw[k].x[q], z);
            const bool ok = z == VT(0);
            v[i / CC][i % CC] = {ok ? double(raw[k].x[0]) : 0.0, ok ? double(raw[k].x[1]) : 0.0};
        }
    };
    double u, v_, w;
    auto load_uvw = [&](uint32_t t) {
        u = v_ = w = 0.0;
        if (t < a.T && my_bl < a.nbl) {
            const double* r = a.uvw + (rows0 + size_t(t) * a.nbl + my_bl) * 3;
            u = r[0];
            v_ = r[1];
            w = r[2];
        }
    };

    C2<double> acc[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) acc[j] = {0.0, 0.0};
    const uint32_t last = (a.C - 1) / CC * CC;  // first channel of the last chunk
    load(0, last);
    load_uvw(my_t);
    for (uint32_t t0 = 0; t0 < a.T; t0 += RT) {
        double sf[ND];
        C2<double> z[ND], z2[ND], he[ND], ho[ND];
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            sf[j] = shift_factor(dz[j], u, v_, w);
            const double2 e = phasor_table(s_table, sf[j] * a.dkappa);
            z[j] = {e.x, e.y};
            z2[j] = cmul(z[j], z[j]);
            he[j] = {0.0, 0.0};
            ho[j] = {0.0, 0.0};
        }
        const bool row_ok = t0 + my_t < a.T && my_bl < a.nbl;
        load_uvw(t0 + RT + my_t);
        for (int32_t c0 = int32_t(last); c0 >= 0; c0 -= CC) {
            wave_fence();  // the chunk before has been read
            hand_over();
            wave_fence();
            if (c0 > 0)
                load(t0, uint32_t(c0) - CC);
            else if (t0 + RT < a.T)
                load(t0 + RT, last);
            // a row's last channel may pair with the zero past it
            const int32_t pairs = int32_t(min(uint32_t(CC), a.C - uint32_t(c0)) + 1) / 2;
#pragma unroll 2
            for (int32_t k = pairs - 1; k >= 0; --k) {
                const C2<double> ve = v[row][2 * k], vo = v[row][2 * k + 1];
#pragma unroll
                for (int j = 0; j < ND; ++j) {
                    he[j] = horner_step(he[j], z2[j], ve);
                    ho[j] = horner_step(ho[j], z2[j], vo);
                }
            }
        }
        if (row_ok) {
#pragma unroll
            for (int j = 0; j < ND; ++j) {
                const double2 e0 = phasor_table(s_table, sf[j] * a.kappa0);
                const C2<double> zo = cmul(z[j], ho[j]);
                const C2<double> r = cmul(C2<double>{e0.x, e0.y}, C2<double>{he[j].x + zo.x, he[j].y + zo.y});
                acc[j].x += r.x;
                acc[j].y += r.y;
            }
        }
    }
    // the timesteps of a baseline lie BB L lanes apart
    for (uint32_t m = BB * L; m < 64; m *= 2) {
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            acc[j].x += __shfl_xor(acc[j].x, m, 64);
            acc[j].y += __shfl_xor(acc[j].y, m, 64);
        }
    }
    if (my_t != 0 || my_bl >= a.nbl) return;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        const uint32_t d = d0 + l + j * L;
        if (d >= d_end) continue;
        double* o = a.avg + ((size_t(blockIdx.y) * a.D + d) * a.nbl + my_bl) * (2 * a.pols_out);
        o[0] = acc[j].x;
        o[1] = acc[j].y;
        for (uint32_t q = 2; q < 2 * a.pols_out; ++q) o[q] = 0.0;  // pols not accumulated
    }
}

template <typename VT, int P, int L, int ND>
void launch_one(hipStream_t s, const void* vis, uint32_t intervals, uint32_t blocks, WaveArgs a) {
    constexpr uint32_t RW = 64 / L;
    // Baselines of a wave: as many as its rows while that leaves 8 waves per SIMD, halved
    // (for as many more timesteps at a time) until it does.
    uint32_t bb = 0;
    while ((2u << bb) <= RW) ++bb;
    auto waves = [&](uint32_t log2) { return uint64_t((a.nbl + (1u << log2) - 1) >> log2) * blocks * intervals; };
    while (bb > 0 && waves(bb) < 8192 && (RW >> bb) < a.T) --bb;
    a.bb_log2 = bb;
    const uint64_t items = uint64_t((a.nbl + (1u << bb) - 1) >> bb) * blocks;
    const uint64_t groups = (items + kWaves - 1) / kWaves;
    require(groups < (1ull << 31) && intervals < 65536, LEAP_ERR_RANGE, "too many workgroups for one launch");
    horner_wave_kernel<VT, P, L, ND>
        <<<dim3(uint32_t(groups), intervals), 64 * kWaves, 0, s>>>(static_cast<const VT*>(vis), a);
    LEAP_HIP(hipGetLastError());
}

template <typename VT, int P>
void launch_tile(hipStream_t s, int32_t tile, const void* vis, uint32_t intervals, uint32_t blocks, const WaveArgs& a) {
    switch (tile) {
        case 82: return launch_one<VT, P, 4, 2>(s, vis, intervals, blocks, a);
        case 162: return launch_one<VT, P, 8, 2>(s, vis, intervals, blocks, a);
        case 322: return launch_one<VT, P, 16, 2>(s, vis, intervals, blocks, a);
        case 642: return launch_one<VT, P, 32, 2>(s, vis, intervals, blocks, a);
        case 1282: return launch_one<VT, P, 64, 2>(s, vis, intervals, blocks, a);
        default: return launch_one<VT, P, 64, 4>(s, vis, intervals, blocks, a);
    }
}

template <typename VT>
void launch_pols(hipStream_t s, int32_t tile, const void* vis, uint32_t P, uint32_t intervals, uint32_t blocks,
                 const WaveArgs& a) {
    switch (P) {
        case 1: return launch_tile<VT, 1>(s, tile, vis, intervals, blocks, a);
        case 2: return launch_tile<VT, 2>(s, tile, vis, intervals, blocks, a);
        case 3: return launch_tile<VT, 3>(s, tile, vis, intervals, blocks, a);
        case 4: return launch_tile<VT, 4>(s, tile, vis, intervals, blocks, a);
        default: throw Error(LEAP_ERR_NOT_IMPLEMENTED, "unsupported polarisation count");
    }
}

}  // namespace

// Directions per wave: 8, 16, 32, 64 or 128 at two a lane, or 256 at four.  A step of a wave costs
// about 8 C instructions a lane for the chains, 0.03 of that for each row it hands over (more rows
// at narrower tiles) and 150 for the phasors, and covers whole direction slots; the cheapest tile
// for D directions among those that give 4 waves per SIMD (else the narrowest tile: with 300
// baselines, 128 t and 90 channels, 64 directions take 248 us in 300 waves, 82 in 2,400).
int32_t horner_wave_tile(uint32_t D, uint32_t nbl, uint32_t C, uint32_t intervals) {
    constexpr struct {
        int32_t tile;
        uint32_t db, rw;
    } tiles[] = {{82, 8, 16}, {162, 16, 8}, {322, 32, 4}, {642, 64, 2}, {1282, 128, 1}, {2564, 256, 1}};
    int32_t best = 82;
    double best_cost = 0.0;
    for (const auto& t : tiles) {
        const uint64_t blocks = (D + t.db - 1) / t.db;
        if (t.db > 8 && uint64_t(nbl) * blocks * intervals < 4096) break;
        const double lanes = t.tile % 10 == 4 ? 1.9 : 1.0;  // four directions a lane: a little less than twice
        const double cost = double(blocks) * lanes / t.rw * (8.0 * C * (1.0 + 0.03 * t.rw) + 150.0);
        if (best_cost == 0.0 || cost < best_cost) {
            best_cost = cost;
            best = t.tile;
        }
    }
    return best;
}

void launch_horner_wave(hipStream_t s, const HornerWave& h) {
    if (h.nbl == 0 || h.D == 0 || h.intervals == 0 || h.T == 0) return;
    const int32_t tile = horner_wave_tile(h.D, h.nbl, h.C, h.intervals);
    const uint32_t db = uint32_t(tile / 10), blocks = (h.D + db - 1) / db;
    const WaveArgs a{h.uvw, h.dd, h.D, (h.D + blocks - 1) / blocks, h.T, h.nbl, h.C, 0, h.pols_out,
                     h.f0 / kSpeedOfLight, h.df / kSpeedOfLight, h.avg};
    if (h.vis_dtype == LEAP_VIS_C64)
        launch_pols<float>(s, tile, h.vis, h.P, h.intervals, blocks, a);
    else
        launch_pols<double>(s, tile, h.vis, h.P, h.intervals, blocks, a);
}

}  // namespace leap
