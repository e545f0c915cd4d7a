// Where host and device meet: small results and inputs, fills, copies of
// graphs, and arrays on their way to the caller.
//
// A pass over a small AIG is bound by these and not by its kernels: a copy of
// four bytes into pageable memory with its synchronisation costs 25 to 40 us,
// each fill a launch.  So a small result is written by a kernel into pinned
// memory of the context, followed by a sequence number that the host waits for
// (8 us); a small input travels in a kernel's arguments, without a wait; several
// fills, or the four arrays of a graph, take one launch.  Arrays of a whole AIG
// come through pinned staging, large ones by a few threads so that the copies
// out of it overlap the transfers.
#include "gls_internal.h"
#include "dev_common.h"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

namespace {

constexpr size_t MAIL_BYTES = 64 << 10, MAIL_FLAG = MAIL_BYTES;   // the sequence number follows the results
constexpr size_t STAGE_SMALL = 2 << 20, STAGE_SLOT = 4 << 20;
constexpr int STAGE_SLOTS = 4;

struct MailPiece {
    const uint8_t *src;
    uint32_t bytes, off;
};
struct MailArgs {
    MailPiece p[FETCH_PIECES];
    int n;
    uint8_t *out;
    uint32_t seq;
};

__global__ void __launch_bounds__(256) k_mail(MailArgs a) {
    for (int i = 0; i < a.n; i++) {
        const MailPiece p = a.p[i];
        uint8_t *out = a.out + p.off;
        uint32_t done = 0;
        if (((uintptr_t)p.src & 3u) == 0) {
            done = p.bytes & ~3u;
            for (uint32_t k = 4 * threadIdx.x; k < done; k += 4 * blockDim.x)
                *(uint32_t *)(out + k) = *(const uint32_t *)(p.src + k);
        }
        for (uint32_t k = done + threadIdx.x; k < p.bytes; k += blockDim.x) out[k] = p.src[k];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store((uint32_t *)(a.out + MAIL_FLAG), a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

constexpr size_t PUT_BYTES = 256;
struct PutArgs {
    uint32_t w[PUT_BYTES / 4];
};

__global__ void __launch_bounds__(64) k_put(PutArgs a, uint32_t words, uint32_t *dst) {
    if (threadIdx.x < words) dst[threadIdx.x] = a.w[threadIdx.x];
}

struct FillArgs {
    Fills::Seg s[FILL_SEGS];
    int n;
};

__global__ void __launch_bounds__(256) k_fills(FillArgs a) {
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    for (int i = 0; i < a.n; i++) {
        const Fills::Seg s = a.s[i];
        uint8_t *p = (uint8_t *)s.p;
        const uint32_t w = s.byte * 0x01010101u;
        size_t done = 0;
        if (((uintptr_t)p & 15u) == 0) {
            done = s.bytes & ~(size_t)15;
            for (size_t k = 16 * tid; k < done; k += 16 * stride) *(uint4 *)(p + k) = make_uint4(w, w, w, w);
        }
        for (size_t k = done + tid; k < s.bytes; k += stride) p[k] = (uint8_t)s.byte;
    }
}

__global__ void __launch_bounds__(256) k_copy_graph(DevGraph src, DevGraph dst) {
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    // the pool's blocks are aligned and hold 16 bytes beyond their size
    auto copy = [&](uint32_t *d, const uint32_t *s, size_t words) {
        for (size_t k = tid; k < (words + 3) / 4; k += stride) ((uint4 *)d)[k] = ((const uint4 *)s)[k];
    };
    copy(dst.f0, src.f0, src.nObjs);
    copy(dst.f1, src.f1, src.nObjs);
    copy(dst.level, src.level, src.nObjs);
    copy(dst.pos, src.pos, src.nPOs);
}

// f0, f1, pos one after the other
__global__ void __launch_bounds__(256) k_stage(DevGraph g, uint32_t *out) {
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    const size_t n = g.nObjs, total = 2 * n + g.nPOs;
    for (size_t k = tid; k < total; k += stride) out[k] = k < n ? g.f0[k] : k < 2 * n ? g.f1[k - n] : g.pos[k - 2 * n];
}

int grid_of(size_t items) { return (int)std::min<size_t>(std::max<size_t>((items + 255) / 256, 1), 4096); }

// waits until the kernel with this sequence number, and what was queued before
// it, has run
int mail_wait(gls_ctx *ctx, uint32_t seq) {
    const std::atomic<uint32_t> *flag = reinterpret_cast<const std::atomic<uint32_t> *>(ctx->mail + MAIL_FLAG);
    const auto limit = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
    for (uint32_t i = 1;; i++) {
        if (flag->load(std::memory_order_acquire) == seq) return GLS_OK;
        if ((i & 255u) == 0 && std::chrono::steady_clock::now() > limit) break;
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
        __builtin_ia32_pause();
#endif
    }
    // a long wait, or an error to report
    GLS_HIP(ctx, hipStreamSynchronize(ctx->stream));
    std::atomic_thread_fence(std::memory_order_acquire);
    return GLS_OK;
}

bool mail_ready(gls_ctx *ctx) {
    if (ctx->mail) return true;
    void *p = nullptr;
    if (hipHostMalloc(&p, MAIL_BYTES + 64, hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    ctx->mail = static_cast<uint8_t *>(p);
    memset(ctx->mail + MAIL_FLAG, 0, 64);
    return true;
}

uint8_t *stage_of(gls_ctx *ctx, size_t bytes) {
    if (ctx->stage_bytes >= bytes) return ctx->stage;
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    ctx->stage = nullptr;
    ctx->stage_bytes = 0;
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    ctx->stage = static_cast<uint8_t *>(p);
    ctx->stage_bytes = bytes;
    return ctx->stage;
}

// The context's device is the calling thread's current one while this lives:
// a program may copy or fetch on a thread that works on another device.
struct OnDevice {
    int was = -1, now;
    explicit OnDevice(int device) : now(device) {
        if (hipGetDevice(&was) != hipSuccess) was = -1;
        if (was != now) (void)hipSetDevice(now);
    }
    ~OnDevice() {
        if (was >= 0 && was != now) (void)hipSetDevice(was);
    }
    OnDevice(const OnDevice &) = delete;
};

uint32_t lit_in(uint32_t l, int32_t conv) { return (conv == GLS_LIT_CULS && l < 2) ? 1u - l : l; }

void take(uint32_t *dst, const uint32_t *src, size_t n, int32_t conv) {
    if (conv != GLS_LIT_CULS) memcpy(dst, src, sizeof(uint32_t) * n);
    else
        for (size_t i = 0; i < n; i++) dst[i] = lit_in(src[i], conv);
}

} // namespace

void transfer_free(gls_ctx *ctx) {
    if (ctx->mail) (void)hipHostFree(ctx->mail);
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    ctx->mail = ctx->stage = nullptr;
    ctx->stage_bytes = 0;
}

int fetch(gls_ctx *ctx, std::initializer_list<FetchPiece> pieces) {
    size_t total = 0;
    for (const FetchPiece &p : pieces) total += (p.bytes + 15) & ~(size_t)15;
    if (total <= MAIL_BYTES && pieces.size() <= (size_t)FETCH_PIECES && mail_ready(ctx)) {
        MailArgs a = {};
        uint32_t off = 0;
        for (const FetchPiece &p : pieces) {
            a.p[a.n++] = MailPiece{static_cast<const uint8_t *>(p.src), (uint32_t)p.bytes, off};
            off += ((uint32_t)p.bytes + 15u) & ~15u;
        }
        a.out = ctx->mail;
        a.seq = ++ctx->mail_seq;
        k_mail<<<1, 256, 0, ctx->stream>>>(a);
        GLS_HIP(ctx, hipGetLastError());
        GLS_TRY(mail_wait(ctx, a.seq));
        int i = 0;
        for (const FetchPiece &p : pieces) memcpy(p.dst, ctx->mail + a.p[i++].off, p.bytes);
        return GLS_OK;
    }
    for (const FetchPiece &p : pieces)
        GLS_HIP(ctx, hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, ctx->stream));
    GLS_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return GLS_OK;
}

// Every copy is ordered on the context stream: the stream is non-blocking, so
// copies on the legacy default stream would not wait for its kernels.
int stream_copy(gls_ctx *ctx, void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    if (kind == hipMemcpyDeviceToHost && bytes <= MAIL_BYTES) return fetch(ctx, {{dst, src, bytes}});
    if (kind == hipMemcpyHostToDevice && bytes <= PUT_BYTES && bytes % 4 == 0 && ((uintptr_t)dst & 3u) == 0) {
        PutArgs a;
        memcpy(a.w, src, bytes);
        k_put<<<1, 64, 0, ctx->stream>>>(a, (uint32_t)(bytes / 4), static_cast<uint32_t *>(dst));
        GLS_HIP(ctx, hipGetLastError());
        return GLS_OK;
    }
    GLS_HIP(ctx, hipMemcpyAsync(dst, src, bytes, kind, ctx->stream));
    GLS_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return GLS_OK;
}

int Fills::run() {
    if (n == 0) return GLS_OK;
    FillArgs a;
    size_t most = 0;
    for (int i = 0; i < n; i++) {
        a.s[i] = s[i];
        most = std::max(most, s[i].bytes);
    }
    a.n = n;
    n = 0;
    k_fills<<<grid_of((most + 15) / 16), 256, 0, ctx->stream>>>(a);
    GLS_HIP(ctx, hipGetLastError());
    return GLS_OK;
}

int dev_graph_copy(gls_ctx *ctx, const DevGraph &src, const DevGraph &dst) {
    const OnDevice on(ctx->device);
    k_copy_graph<<<grid_of(((size_t)std::max(src.nObjs, src.nPOs) + 3) / 4), 256, 0, ctx->stream>>>(src, dst);
    GLS_HIP(ctx, hipGetLastError());
    return GLS_OK;
}

// Arrays of the device copy to the caller's (any of them may be null).  Up to
// STAGE_SMALL bytes: one kernel into the staging and one copy out of it;
// more: pieces of STAGE_SLOT bytes on up to four threads, each with its part of
// the staging.  Through pageable copies into arrays of the handle first, 92 MB
// took 20 ms.  Without pinned memory to be had they are what is left.
int dev_graph_fetch(gls_ctx *ctx, const DevGraph &g, uint32_t *f0, uint32_t *f1, uint32_t *pos, int32_t conv) {
    const OnDevice on(ctx->device);
    const size_t n = g.nObjs, words = 2 * n + g.nPOs;
    if (4 * words <= STAGE_SMALL && mail_ready(ctx)) {
        uint32_t *stage = reinterpret_cast<uint32_t *>(stage_of(ctx, STAGE_SMALL));
        if (stage) {
            k_stage<<<grid_of(words), 256, 0, ctx->stream>>>(g, stage);
            MailArgs a = {};
            a.out = ctx->mail;
            a.seq = ++ctx->mail_seq;
            k_mail<<<1, 256, 0, ctx->stream>>>(a);
            GLS_HIP(ctx, hipGetLastError());
            GLS_TRY(mail_wait(ctx, a.seq));
            if (f0) take(f0, stage, n, conv);
            if (f1) take(f1, stage + n, n, conv);
            if (pos) take(pos, stage + 2 * n, g.nPOs, conv);
            return GLS_OK;
        }
    }
    struct Chunk {
        uint32_t *dst;
        const uint32_t *src;
        size_t words;
    };
    std::vector<Chunk> chunks;
    auto add = [&](uint32_t *dst, const uint32_t *src, size_t count) {
        for (size_t k = 0; dst && k < count; k += STAGE_SLOT / 4)
            chunks.push_back(Chunk{dst + k, src + k, std::min(count - k, STAGE_SLOT / 4)});
    };
    add(f0, g.f0, n);
    add(f1, g.f1, n);
    add(pos, g.pos, g.nPOs);
    uint8_t *stage = stage_of(ctx, STAGE_SLOT * STAGE_SLOTS);
    if (!stage) {
        for (const Chunk &c : chunks)
            GLS_HIP(ctx, hipMemcpyAsync(c.dst, c.src, sizeof(uint32_t) * c.words, hipMemcpyDeviceToHost, ctx->stream));
        GLS_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (conv == GLS_LIT_CULS)
            for (const Chunk &c : chunks) take(c.dst, c.dst, c.words, conv);
        return GLS_OK;
    }
    const int workers = (int)std::min<size_t>(STAGE_SLOTS, chunks.size());
    std::atomic<int> bad{0};
    auto work = [&](int w) {
        uint32_t *slot = reinterpret_cast<uint32_t *>(stage + STAGE_SLOT * (size_t)w);
        hipEvent_t e = nullptr;
        hipError_t r = hipSetDevice(ctx->device);
        if (r == hipSuccess) r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        for (size_t i = w; r == hipSuccess && i < chunks.size(); i += workers) {
            const Chunk &c = chunks[i];
            r = hipMemcpyAsync(slot, c.src, sizeof(uint32_t) * c.words, hipMemcpyDeviceToHost, ctx->stream);
            if (r == hipSuccess) r = hipEventRecord(e, ctx->stream);
            if (r == hipSuccess) r = hipEventSynchronize(e);
            if (r == hipSuccess) take(c.dst, slot, c.words, conv);
        }
        if (e) (void)hipEventDestroy(e);
        if (r != hipSuccess) bad = (int)r;
    };
    std::vector<std::thread> threads;
    int started = 1;
    try {
        threads.reserve(workers);
        for (; started < workers; started++) threads.emplace_back(work, started);
    } catch (const std::exception &) {
        // no thread to be had: its part is done here
    }
    work(0);
    for (int w = started; w < workers; w++) work(w);
    for (std::thread &t : threads) t.join();
    if (bad) return gls_fail(ctx, GLS_ERR_HIP, "array fetch: %s", hipGetErrorString((hipError_t)bad.load()));
    return GLS_OK;
}
