// Host -> device staging of host-resident visibilities.
//
// Pageable host memory is copied in chunks through two pinned buffers: worker
// threads fill a buffer in pieces, in order, and each piece is sent on the
// context's copy stream while the next ones are filled.  (Sent buffer by buffer, a cube that
// fits one was first copied whole and then sent: 180 MB in 4.8 ms; 3.3 ms in pieces.)
// For the packed pol-0 path the workers apply the
// reference's skip rule (CpuLeapCalibrator.cc:201-214: a (row, channel) with a
// non-finite polarisation is left out, here written as 0) and keep pol 0
// only, so a quarter of a 4-pol cube crosses the bus.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "leap_internal.h"

namespace leap {

namespace {

constexpr size_t kChunkBytes = size_t(256) << 20;  // per pinned buffer

unsigned worker_count() {
    const unsigned hc = std::thread::hardware_concurrency();
    return std::max(1u, std::min(16u, hc ? hc : 1u));
}

constexpr size_t kPieceBytes = size_t(8) << 20;    // a copy on the bus: 0.15 ms
constexpr size_t kBlockBytes = size_t(512) << 10;  // taken by a worker at a time

// fill(begin, end) over the units [0, n) of unit_bytes each, in blocks that the workers and the calling
// thread take in order; ready(begin, end) on the calling thread for each piece, in order, once filled.
template <typename Fill, typename Ready>
void fill_in_pieces(size_t n, size_t unit_bytes, Fill&& fill, Ready&& ready) {
    const size_t block = std::max<size_t>(1, kBlockBytes / unit_bytes), per_piece = kPieceBytes / kBlockBytes;
    const size_t blocks = (n + block - 1) / block, pieces = (blocks + per_piece - 1) / per_piece;
    std::atomic<size_t> next{0};
    std::vector<std::atomic<size_t>> filled(pieces);
    for (auto& f : filled) f.store(0, std::memory_order_relaxed);
    auto work = [&] {  // one block; false when none is left
        const size_t b = next.fetch_add(1, std::memory_order_relaxed);
        if (b >= blocks) return false;
        fill(b * block, std::min(n, (b + 1) * block));
        filled[b / per_piece].fetch_add(1, std::memory_order_release);
        return true;
    };
    struct Pool {  // joined also when ready throws
        std::vector<std::thread> threads;
        ~Pool() {
            for (auto& t : threads) t.join();
        }
    } pool;
    const size_t helpers = std::min<size_t>(worker_count(), blocks) - 1;
    pool.threads.reserve(helpers);
    try {
        for (size_t i = 0; i < helpers; ++i)
            pool.threads.emplace_back([&work] {
                while (work()) {
                }
            });
    } catch (const std::system_error&) {  // fewer helpers, or none
    }
    for (size_t p = 0; p < pieces; ++p) {
        const size_t b0 = p * per_piece, b1 = std::min(blocks, b0 + per_piece);
        while (filled[p].load(std::memory_order_acquire) < b1 - b0)
            if (!work()) std::this_thread::yield();
        ready(b0 * block, std::min(n, b1 * block));
    }
}

void ensure_staging(leap_ctx* ctx) {
    if (ctx->pinned_bytes >= kChunkBytes) return;
    for (int b = 0; b < 2; ++b) {
        if (ctx->h2d_pending[b]) LEAP_HIP(hipEventSynchronize(ctx->ev_h2d[b]));
        ctx->h2d_pending[b] = false;
        if (ctx->h_pinned[b]) LEAP_HIP(hipHostFree(ctx->h_pinned[b]));
        ctx->h_pinned[b] = nullptr;
    }
    ctx->pinned_bytes = 0;
    for (int b = 0; b < 2; ++b) LEAP_HIP(hipHostMalloc(&ctx->h_pinned[b], kChunkBytes, hipHostMallocDefault));
    ctx->pinned_bytes = kChunkBytes;
}

// The copy stream starts after the work already queued on ctx->stream.
void fork_copy_stream(leap_ctx* ctx) {
    LEAP_HIP(hipEventRecord(ctx->ev_copy_fork, ctx->stream));
    LEAP_HIP(hipStreamWaitEvent(ctx->copy_stream, ctx->ev_copy_fork, 0));
}

// Later work on ctx->stream starts after the copies.
void join_copy_stream(leap_ctx* ctx) {
    LEAP_HIP(hipEventRecord(ctx->ev_copy_join, ctx->copy_stream));
    LEAP_HIP(hipStreamWaitEvent(ctx->stream, ctx->ev_copy_join, 0));
}

// A staging call that ends early leaves no copy in flight: its pieces' event is recorded after the last
// one only, and the next call fills the same pinned buffers.
struct EndsEarly {
    leap_ctx* ctx;
    bool done = false;
    ~EndsEarly() {
        if (done) return;
        (void)hipStreamSynchronize(ctx->copy_stream);
        ctx->h2d_pending[0] = ctx->h2d_pending[1] = false;
    }
};

// The pinned buffer b is free once its previous copy has completed.
void acquire(leap_ctx* ctx, int b) {
    if (ctx->h2d_pending[b]) {
        LEAP_HIP(hipEventSynchronize(ctx->ev_h2d[b]));
        ctx->h2d_pending[b] = false;
    }
}

// Part of the pinned buffer b to the device; sent(b) after its last one.
void send(leap_ctx* ctx, int b, size_t offset, void* device_dst, size_t bytes) {
    LEAP_HIP(hipMemcpyAsync(device_dst, static_cast<const char*>(ctx->h_pinned[b]) + offset, bytes,
                            hipMemcpyHostToDevice, ctx->copy_stream));
    ctx->last_stage_bytes += bytes;
    ctx->h2d_pending[b] = true;
}

void sent(leap_ctx* ctx, int b) { LEAP_HIP(hipEventRecord(ctx->ev_h2d[b], ctx->copy_stream)); }

template <typename VT>
void pack_pol0_host(const VT* src, uint32_t P, size_t begin, size_t end, VT* out) {
    for (size_t i = begin; i < end; ++i) {
        const VT* p = src + i * 2 * P;
        bool finite = true;
        for (uint32_t k = 0; k < 2 * P; ++k) finite = finite && std::isfinite(p[k]);
        out[2 * i] = finite ? p[0] : VT(0);
        out[2 * i + 1] = finite ? p[1] : VT(0);
    }
}

}  // namespace

void stage_copy(leap_ctx* ctx, const void* host_src, size_t bytes, void* device_dst) {
    if (bytes == 0) return;
    ensure_staging(ctx);
    EndsEarly call{ctx};
    fork_copy_stream(ctx);
    const char* src = static_cast<const char*>(host_src);
    char* dst = static_cast<char*>(device_dst);
    int b = 0;
    for (size_t off = 0; off < bytes; off += kChunkBytes, b ^= 1) {
        const size_t len = std::min(kChunkBytes, bytes - off);
        acquire(ctx, b);
        char* pin = static_cast<char*>(ctx->h_pinned[b]);
        fill_in_pieces(
            len, 1, [&](size_t lo, size_t hi) { std::memcpy(pin + lo, src + off + lo, hi - lo); },
            [&](size_t lo, size_t hi) { send(ctx, b, lo, dst + off + lo, hi - lo); });
        sent(ctx, b);
    }
    join_copy_stream(ctx);
    call.done = true;
}

void stage_pol0(leap_ctx* ctx, const void* host_vis, int32_t vis_dtype, uint32_t P, size_t n, double* device_dst) {
    if (n == 0) return;
    ensure_staging(ctx);
    const bool c64 = vis_dtype == LEAP_VIS_C64;
    const size_t out_elem = c64 ? 8 : 16;  // pol 0 in the source precision
    const size_t per_chunk = kChunkBytes / out_elem;
    if (c64)
        for (int b = 0; b < 2; ++b) ctx->d_widen[b].reserve(kChunkBytes);
    EndsEarly call{ctx};
    fork_copy_stream(ctx);
    int b = 0;
    for (size_t e0 = 0; e0 < n; e0 += per_chunk, b ^= 1) {
        const size_t m = std::min(per_chunk, n - e0);
        acquire(ctx, b);
        if (c64) {
            const float* src = static_cast<const float*>(host_vis) + e0 * 2 * P;
            float* pin = static_cast<float*>(ctx->h_pinned[b]);
            // the device staging buffer b is free once its previous widen kernel has run
            if (ctx->widen_pending[b]) LEAP_HIP(hipStreamWaitEvent(ctx->copy_stream, ctx->ev_widened[b], 0));
            fill_in_pieces(
                m, out_elem, [&](size_t lo, size_t hi) { pack_pol0_host(src, P, lo, hi, pin); },
                [&](size_t lo, size_t hi) {
                    send(ctx, b, lo * out_elem, ctx->d_widen[b].as<char>() + lo * out_elem, (hi - lo) * out_elem);
                });
            sent(ctx, b);
            LEAP_HIP(hipStreamWaitEvent(ctx->stream, ctx->ev_h2d[b], 0));
            launch_widen_c64(ctx->stream, ctx->d_widen[b].ptr, m, device_dst + 2 * e0);
            LEAP_HIP(hipEventRecord(ctx->ev_widened[b], ctx->stream));
            ctx->widen_pending[b] = true;
        } else {
            const double* src = static_cast<const double*>(host_vis) + e0 * 2 * P;
            double* pin = static_cast<double*>(ctx->h_pinned[b]);
            fill_in_pieces(
                m, out_elem, [&](size_t lo, size_t hi) { pack_pol0_host(src, P, lo, hi, pin); },
                [&](size_t lo, size_t hi) {
                    send(ctx, b, lo * out_elem, device_dst + 2 * (e0 + lo), (hi - lo) * out_elem);
                });
            sent(ctx, b);
        }
    }
    join_copy_stream(ctx);
    call.done = true;
}

}  // namespace leap
