// Host transfers of per-cell and per-node arrays (transfer.hpp).
//
// A full readback of 4.2 M cells moved 67 MB into pageable memory and then
// converted and reordered it on one thread, 29 ms beside a 0.33 ms step; now
// the kernels below write the reordered doubles over the bus (50 GB/s into
// pinned memory, measured), chunk by chunk, and the threads' copies into the
// caller's fresh pages (4 GB/s on one thread, 40 on 16) run behind it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "context.hpp"
#include "transfer.hpp"

namespace lbfs {

// caller cell c0 + k of a chunk of m cells: its record as four doubles, in rows
// of m (soa) or one after the other
__global__ __launch_bounds__(256) void k_export_cells(const float4 *__restrict__ src, const int *__restrict__ inv, int c0,
                                                      int m, double add0, int aos, double *__restrict__ out)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m) return;
    const float4 s = src[inv[c0 + k]];
    const double v[4] = {add0 + (double)s.x, (double)s.y, (double)s.z, (double)s.w};
    if (aos) {
        double2 *o = reinterpret_cast<double2 *>(out) + 2 * (size_t)k;
        o[0] = make_double2(v[0], v[1]);
        o[1] = make_double2(v[2], v[3]);
    } else {
#pragma unroll
        for (int t = 0; t < 4; t++) out[(size_t)t * m + k] = v[t];
    }
}

__global__ __launch_bounds__(256) void k_import_cells(const double *__restrict__ in, const int *__restrict__ inv, int c0,
                                                      int m, float4 *__restrict__ dst)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m) return;
    const double2 *p = reinterpret_cast<const double2 *>(in) + 2 * (size_t)k;
    const double2 a = p[0], b = p[1];
    dst[inv[c0 + k]] = make_float4((float)a.x, (float)a.y, (float)b.x, (float)b.y);
}

// value k of the chunk: component of node n0 + k / 3, in up to three rows of
// 3 m values
__global__ __launch_bounds__(256) void k_export_nodes(MemArgs m, int n0, int count, int rows, const float4 *r0,
                                                      const float4 *r1, const float4 *r2, int origin_row,
                                                      double *__restrict__ out)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= 3 * count) return;
    const int n = n0 + k / 3, c = k % 3;
    const float4 *row[3] = {r0, r1, r2};
#pragma unroll
    for (int q = 0; q < 3; q++) {
        if (q >= rows) break;
        const float4 v = row[q][n];
        double x = (double)(c == 0 ? v.x : (c == 1 ? v.y : v.z));
        if (q == origin_row) {
            const float4 o = m.node_origin[n];
            x = (double)(c == 0 ? o.x : (c == 1 ? o.y : o.z)) + x;
        }
        out[(size_t)q * 3 * count + k] = x;
    }
}

void Staging::release()
{
    for (double *&b : buf) {
        if (b) (void)hipHostFree(b);
        b = nullptr;
    }
    for (hipEvent_t &e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    bytes = 0;
}

namespace {

constexpr size_t CHUNK_BYTES = (size_t)8 << 20;   // per staging buffer
constexpr size_t PIECE_BYTES = (size_t)256 << 10; // a thread's copy

struct Piece {
    void *dst;
    const void *src;
    size_t bytes;
};

// threads that copy pieces beside the calling one, for one transfer; as many as
// the transfer's bytes keep busy, none if they cannot be started
class CopyTeam {
    std::vector<std::thread> th;
    std::mutex mx;
    std::condition_variable work, done;
    const std::vector<Piece> *pieces = nullptr;
    std::atomic<size_t> next{0};
    int round = 0, busy = 0;
    bool stop = false;

    void take(const std::vector<Piece> &p)
    {
        for (size_t k; (k = next.fetch_add(1)) < p.size();) std::memcpy(p[k].dst, p[k].src, p[k].bytes);
    }
    void loop()
    {
        int seen = 0;
        std::unique_lock<std::mutex> lk(mx);
        for (;;) {
            work.wait(lk, [&] { return stop || round != seen; });
            if (stop) return;
            seen = round;
            const std::vector<Piece> &p = *pieces;
            lk.unlock();
            take(p);
            lk.lock();
            if (--busy == 0) done.notify_one();
        }
    }

public:
    explicit CopyTeam(size_t bytes)
    {
        const size_t hw = std::max(1u, std::thread::hardware_concurrency());
        const size_t n = std::min<size_t>(std::min<size_t>(hw, 16), bytes >> 20);
        try {
            for (size_t k = 1; k < n; k++) th.emplace_back([this] { loop(); });
        } catch (const std::system_error &) {
        }
    }
    ~CopyTeam()
    {
        {
            std::lock_guard<std::mutex> lk(mx);
            stop = true;
        }
        work.notify_all();
        for (std::thread &t : th) t.join();
    }
    // copies every segment, in pieces
    void copy(const std::vector<Piece> &segments)
    {
        std::vector<Piece> p;
        for (const Piece &s : segments)
            for (size_t o = 0; o < s.bytes; o += PIECE_BYTES)
                p.push_back({(char *)s.dst + o, (const char *)s.src + o, std::min(PIECE_BYTES, s.bytes - o)});
        next = 0;
        if (!th.empty() && p.size() > 1) {
            {
                std::lock_guard<std::mutex> lk(mx);
                pieces = &p;
                busy = (int)th.size();
                round++;
            }
            work.notify_all();
            take(p);
            std::unique_lock<std::mutex> lk(mx);
            done.wait(lk, [&] { return busy == 0; });
        } else {
            take(p);
        }
    }
};

#define HIPCHK(expr)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess) return ctx->fail(LBFS_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

// Readies the staging buffers of a transfer of `chunks` chunks of up to `bytes`
// (grown if a larger transfer comes): a single chunk needs one, whose allocation
// is most of a small mesh's first readback.  False where pinned memory cannot be
// had; the transfer then goes through pageable memory.
bool staging(lbfs_ctx *ctx, size_t bytes, size_t chunks)
{
    Staging &s = ctx->staging;
    if (s.bytes < bytes) s.release();
    const size_t size = std::max(bytes, s.bytes);
    for (size_t k = 0; k < std::min<size_t>(2, chunks); k++) {
        hipError_t e = hipSuccess;
        if (!s.ev[k]) e = hipEventCreateWithFlags(&s.ev[k], hipEventDisableTiming);
        if (e == hipSuccess && !s.buf[k]) e = hipHostMalloc((void **)&s.buf[k], size, hipHostMallocDefault);
        if (e != hipSuccess) {
            (void)hipGetLastError();  // (the next launch's check would report it again)
            s.release();
            return false;
        }
    }
    s.bytes = size;
    return true;
}

// the device's records in pageable memory
int pageable(lbfs_ctx *ctx, const float4 *src, size_t n, std::vector<float4> &h)
{
    h.resize(n);
    HIPCHK(hipMemcpyAsync(h.data(), src, sizeof(float4) * n, hipMemcpyDeviceToHost, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return LBFS_OK;
}

int read_cells_pageable(lbfs_ctx *ctx, const float4 *src, double add0, const CellArrays &out)
{
    std::vector<float4> h;
    const int rc = pageable(ctx, src, (size_t)ctx->lay.n_cells, h);
    if (rc) return rc;
    for (int i = 0; i < ctx->lay.n_cells; i++) {
        const size_t c = (size_t)ctx->lay.perm[i];
        const double v[4] = {add0 + (double)h[i].x, (double)h[i].y, (double)h[i].z, (double)h[i].w};
        for (int t = 0; t < 4; t++) (out.aos ? out.aos[4 * c + t] : out.soa[t][c]) = v[t];
    }
    return LBFS_OK;
}

int write_cells_pageable(lbfs_ctx *ctx, const double *src, float4 *dst)
{
    const size_t n = (size_t)ctx->lay.n_cells;
    std::vector<float4> h(n);
    for (size_t i = 0; i < n; i++) {
        const double *v = src + 4 * (size_t)ctx->lay.perm[i];
        h[i] = make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
    }
    HIPCHK(hipMemcpyAsync(dst, h.data(), sizeof(float4) * n, hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return LBFS_OK;
}

int read_nodes_pageable(lbfs_ctx *ctx, double *const out[3])
{
    const MemArgs &m = ctx->mem;
    const float4 *const src[3] = {m.X, m.U, m.F};
    std::vector<float4> h, o;
    for (int q = 0; q < 3; q++) {
        if (!out[q]) continue;
        int rc = pageable(ctx, src[q], (size_t)m.n_nodes, h);
        if (!rc && q == 0) rc = pageable(ctx, m.node_origin, (size_t)m.n_nodes, o);
        if (rc) return rc;
        for (int n = 0; n < m.n_nodes; n++) {
            const double v[3] = {(double)h[n].x, (double)h[n].y, (double)h[n].z};
            const double c[3] = {q ? 0.0 : (double)o[n].x, q ? 0.0 : (double)o[n].y, q ? 0.0 : (double)o[n].z};
            for (int t = 0; t < 3; t++) out[q][3 * (size_t)n + t] = q ? v[t] : c[t] + v[t];
        }
    }
    return LBFS_OK;
}

// n items of `item` bytes out: launch(i0, m, buf) enqueues the kernel that
// fills buf, segments(i0, m, buf) lists where its parts go; pageable() does the
// whole transfer without pinned memory
int stream_out(lbfs_ctx *ctx, size_t n, size_t item, const std::function<hipError_t(int, int, double *)> &launch,
               const std::function<std::vector<Piece>(int, int, const double *)> &segments,
               const std::function<int()> &pageable)
{
    const size_t per = std::max<size_t>(1, CHUNK_BYTES / item);
    const size_t chunks = (n + per - 1) / per;
    if (!staging(ctx, std::min(n, per) * item, chunks)) return pageable();
    Staging &s = ctx->staging;
    CopyTeam team(n * item);
    auto start = [&](size_t k) -> hipError_t {
        const size_t i0 = k * per, m = std::min(per, n - i0);
        const hipError_t e = launch((int)i0, (int)m, s.buf[k & 1]);
        return e != hipSuccess ? e : hipEventRecord(s.ev[k & 1], ctx->stream);
    };
    for (size_t k = 0; k < std::min<size_t>(2, chunks); k++) HIPCHK(start(k));
    for (size_t k = 0; k < chunks; k++) {
        HIPCHK(hipEventSynchronize(s.ev[k & 1]));
        const size_t i0 = k * per, m = std::min(per, n - i0);
        team.copy(segments((int)i0, (int)m, s.buf[k & 1]));
        if (k + 2 < chunks) HIPCHK(start(k + 2));
    }
    return LBFS_OK;
}

}  // namespace

int read_cells(lbfs_ctx *ctx, const float4 *src, double add0, const CellArrays &out)
{
    return stream_out(
        ctx, (size_t)ctx->lay.n_cells, 32,
        [&](int c0, int m, double *buf) {
            hipLaunchKernelGGL(k_export_cells, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, src, ctx->cell_inv, c0, m,
                               add0, out.aos ? 1 : 0, buf);
            return hipGetLastError();
        },
        [&](int c0, int m, const double *buf) {
            std::vector<Piece> p;
            if (out.aos) {
                p.push_back({out.aos + 4 * (size_t)c0, buf, 32 * (size_t)m});
            } else {
                for (int t = 0; t < 4; t++) p.push_back({out.soa[t] + c0, buf + (size_t)t * m, 8 * (size_t)m});
            }
            return p;
        },
        [&] { return read_cells_pageable(ctx, src, add0, out); });
}

int read_nodes(lbfs_ctx *ctx, double *X, double *U, double *F)
{
    const MemArgs &m = ctx->mem;
    const float4 *row[3] = {nullptr, nullptr, nullptr};
    double *dst[3] = {nullptr, nullptr, nullptr};
    int rows = 0;
    const float4 *const src[3] = {m.X, m.U, m.F};
    double *const arr[3] = {X, U, F};
    for (int q = 0; q < 3; q++)
        if (arr[q]) {
            row[rows] = src[q];
            dst[rows++] = arr[q];
        }
    if (!rows) return LBFS_OK;
    return stream_out(
        ctx, (size_t)m.n_nodes, 24 * (size_t)rows,
        [&](int n0, int count, double *buf) {
            hipLaunchKernelGGL(k_export_nodes, dim3((3 * count + 255) / 256), dim3(256), 0, ctx->stream, m, n0, count, rows,
                               row[0], row[1], row[2], X ? 0 : -1, buf);
            return hipGetLastError();
        },
        [&](int n0, int count, const double *buf) {
            std::vector<Piece> p;
            for (int q = 0; q < rows; q++)
                p.push_back({dst[q] + 3 * (size_t)n0, buf + (size_t)q * 3 * count, 24 * (size_t)count});
            return p;
        },
        [&] { return read_nodes_pageable(ctx, arr); });
}

int write_cells(lbfs_ctx *ctx, const double *src, float4 *dst)
{
    const size_t n = (size_t)ctx->lay.n_cells, per = CHUNK_BYTES / 32, chunks = (n + per - 1) / per;
    if (!staging(ctx, std::min(n, per) * 32, chunks)) return write_cells_pageable(ctx, src, dst);
    Staging &s = ctx->staging;
    CopyTeam team(n * 32);
    for (size_t k = 0; k < chunks; k++) {
        const size_t c0 = k * per, m = std::min(per, n - c0);
        // (the buffer's chunk before the last one has been read)
        if (k >= 2) HIPCHK(hipEventSynchronize(s.ev[k & 1]));
        team.copy({{s.buf[k & 1], src + 4 * c0, 32 * m}});
        hipLaunchKernelGGL(k_import_cells, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, ctx->stream, s.buf[k & 1],
                           ctx->cell_inv, (int)c0, (int)m, dst);
        HIPCHK(hipGetLastError());
        HIPCHK(hipEventRecord(s.ev[k & 1], ctx->stream));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return LBFS_OK;
}

}  // namespace lbfs
