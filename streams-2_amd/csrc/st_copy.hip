// st_copy.hip -- ghosted fields between the solver's pitched layout on the
// device and the reference layout on the host, through pinned staging.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "st_solver.h"

namespace st {

// Staging for fields of up to nbytes: a pair of buffers per host thread, the
// threads one per 4 MiB of field, eight at most (32 MiB in all, whatever the
// field).  Buffers of 2 MiB: a copy leaves the link idle for about 13 us, so
// 1422 MB take 108 ms in 256 KiB pieces, 46 ms at 1 MiB, 36 ms at 2 MiB and
// 31 ms at 4 MiB, for which twice the pinned memory was not taken.  A solver
// without pinned memory still copies, through pageable staging of its calls.
void stage_create(CopyStage &cs, size_t nbytes) {
    size_t th = nbytes / kStagePerThread;
    cs.threads = th < 1 ? 1 : (th > kStageThreads ? kStageThreads : (int)th);
    const size_t share = (nbytes + 2 * cs.threads - 1) / (2 * cs.threads);
    cs.bytes = ((share < kStageBuffer ? share : kStageBuffer) + 4095) & ~(size_t)4095;
    if (hipHostMalloc((void **)&cs.mem, 2 * cs.threads * cs.bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        cs.mem = nullptr;
    }
    for (int q = 0; q < 2 * cs.threads; q++)
        if (hipEventCreateWithFlags(&cs.ev[q], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            cs.ev[q] = nullptr;
            stage_destroy(cs);
            return;
        }
}
void stage_destroy(CopyStage &cs) {
    for (auto &e : cs.ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (cs.mem) (void)hipHostFree(cs.mem);
    cs.mem = nullptr;
}

namespace {
struct Job {
    st_solver *s;
    char *dev, *host;
    size_t dpitch, hpitch;       // bytes of a row on either side
    size_t rows, hvar, rows_var; // all rows, rows of one variable and the host's bytes of it
    size_t per, chunks;          // rows of a chunk
    bool in;                     // host to device
    char *mem;
    size_t bytes;
    hipEvent_t *ev;              // null: wait for the stream
    std::atomic<size_t> next{0};
    std::atomic<int> err{0};

    char *row(size_t r) const { return host + (r / rows_var) * hvar + (r % rows_var) * hpitch; }
    void pack(char *b, size_t c) const {
        const size_t r0 = c * per, r1 = r0 + per < rows ? r0 + per : rows;
        for (size_t r = r0; r < r1; r++, b += dpitch) {
            std::memcpy(b, row(r), hpitch);
            std::memset(b + hpitch, 0, dpitch - hpitch);
        }
    }
    void unpack(const char *b, size_t c) const {
        const size_t r0 = c * per, r1 = r0 + per < rows ? r0 + per : rows;
        for (size_t r = r0; r < r1; r++, b += dpitch) std::memcpy(row(r), b, hpitch);
    }
    bool ok(hipError_t e) {
        if (e != hipSuccess) err.store((int)e);
        return e == hipSuccess;
    }
    bool issue(char *b, size_t c, int q) {
        const size_t r0 = c * per, n = (r0 + per < rows ? per : rows - r0) * dpitch;
        char *d = dev + r0 * dpitch;
        return ok(in ? hipMemcpyAsync(d, b, n, hipMemcpyHostToDevice, s->stream)
                     : hipMemcpyAsync(b, d, n, hipMemcpyDeviceToHost, s->stream)) &&
               (!ev || ok(hipEventRecord(ev[q], s->stream)));
    }
    bool wait(int q) { return ok(ev ? hipEventSynchronize(ev[q]) : hipStreamSynchronize(s->stream)); }
    // Two buffers a thread: one on the link while the other is re-spaced.
    // Every chunk is waited for before its buffer or this thread goes away: out
    // says whether one may be in flight, also where its event could not be
    // recorded or waited for.
    void run(int t) {
        char *b[2] = {mem + 2 * t * bytes, mem + (2 * t + 1) * bytes};
        bool out[2] = {false, false};
        size_t held[2] = {0, 0};
        for (int q = 0; err.load() == 0; q ^= 1) {
            const size_t c = next.fetch_add(1);
            const bool more = c < chunks;
            if (more) {
                if (out[q]) {  // in: the buffer's last chunk
                    if (!wait(2 * t + q)) break;
                    out[q] = false;
                }
                if (in) pack(b[q], c);
                out[q] = true;
                if (!issue(b[q], c, 2 * t + q)) break;
                held[q] = c;
            }
            if (!in && out[q ^ 1]) {
                if (!wait(2 * t + (q ^ 1))) break;
                out[q ^ 1] = false;
                unpack(b[q ^ 1], held[q ^ 1]);
            }
            if (!more && !(out[0] && !in) && !(out[1] && !in)) break;
        }
        if (out[0] || out[1]) (void)hipStreamSynchronize(s->stream);
    }
};
}  // namespace

// nvars ghosted variables of es-byte values.  Chunks of whole rows move over
// the link while others are re-spaced; a fresh host array is also first
// touched by these threads.  Fields under 8 MiB stay with the calling thread:
// their copy takes some 0.1 ms a MiB and starting a thread about as long.
// Against one pageable copy and one re-spacing thread a variable, out to a
// fresh array: 32x24x16 (1 MB) 0.58 -> 0.08 ms, 128x96x64 (38 MB) 5.6 -> 1.6,
// 512x256x256 (1422 MB) 237 -> 36.  Returns once the copies have completed.
hipError_t copy_rows(st_solver *s, void *dst, const void *src, size_t es, int nvars, hipMemcpyKind kind) {
    const Geo &g = s->g;
    Job j;
    j.s = s;
    j.in = kind == hipMemcpyHostToDevice;
    j.dev = (char *)(j.in ? dst : const_cast<void *>(src));
    j.host = (char *)(j.in ? const_cast<void *>(src) : dst);
    j.dpitch = (size_t)g.sx * es;
    j.hpitch = (size_t)g.rx * es;
    j.rows_var = (size_t)g.sy * g.sz;
    j.rows = j.rows_var * nvars;
    j.hvar = (size_t)g.nref * es;
    CopyStage *cs = s->stage;
    const size_t total = j.rows * j.dpitch;
    std::vector<char> tmp;
    std::unique_lock<std::mutex> lk;
    int threads = 1;
    if (cs && cs->mem && cs->bytes >= j.dpitch) {
        threads = (int)(total / kStagePerThread);
        threads = threads < 1 ? 1 : (threads > cs->threads ? cs->threads : threads);
        j.mem = cs->mem;
        j.bytes = cs->bytes;
        j.ev = cs->ev;
        lk = std::unique_lock<std::mutex>(cs->mu);
    } else {
        j.bytes = j.dpitch > kStageBuffer ? j.dpitch : kStageBuffer;
        j.ev = nullptr;
        try {
            tmp.resize(2 * j.bytes);
        } catch (const std::bad_alloc &) {
            return hipErrorOutOfMemory;
        }
        j.mem = tmp.data();
    }
    // at least two chunks a thread, so that both buffers work
    const size_t fit = j.bytes / j.dpitch, share = (j.rows + 2 * threads - 1) / (2 * threads);
    j.per = share < fit ? share : fit;
    j.chunks = (j.rows + j.per - 1) / j.per;
    std::vector<std::thread> pool;
    if (threads > 1) {
        try {
            pool.reserve(threads - 1);
            for (int t = 1; t < threads; t++)
                pool.emplace_back([&j, t, dev = s->device]() {
                    if (j.ok(hipSetDevice(dev))) j.run(t);
                });
        } catch (const std::exception &) {  // fewer threads: the others take the chunks
        }
    }
    j.run(0);
    for (auto &t : pool) t.join();
    if (j.err.load()) return (hipError_t)j.err.load();
    return hipStreamSynchronize(s->stream);
}

}  // namespace st
