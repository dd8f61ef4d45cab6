// The staged field copies (st_copy.hip) on a stand-in of the runtime whose
// copies wait in a queue until the stream or an event behind them is waited
// for, and whose calls can be made to fail: fields come through whole, and
// after an error no copy is left behind that could still touch the staging or
// the caller's array.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../streams-2_amd/csrc/st_solver.h"

namespace {
struct Op {
    void *dst;
    const void *src;
    size_t n;
};
std::mutex mu;
std::vector<Op> queue;  // of the one stream, in order
size_t done = 0;        // operations that have run
size_t mark[64];        // where each event was recorded
int events = 0;
enum Call { kCopy, kRecord, kEventWait, kCalls };
int left[kCalls];       // calls of a kind until one fails (< 0: none does)
bool fails(Call c) { return left[c] >= 0 && left[c]-- == 0; }
void run_to(size_t end) {
    for (; done < end; done++) std::memcpy(queue[done].dst, queue[done].src, queue[done].n);
}
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t)&mark[events++];
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    if (fails(kCopy)) return hipErrorInvalidValue;
    queue.push_back({d, s, n});
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    if (fails(kRecord)) return hipErrorInvalidHandle;
    *(size_t *)e = queue.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> lk(mu);
    if (fails(kEventWait)) return hipErrorInvalidHandle;
    run_to(*(size_t *)e);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    run_to(queue.size());
    return hipSuccess;
}
}

#define CHECK(c)                                                                                        \
    do {                                                                                                \
        if (!(c)) {                                                                                     \
            std::printf("%dx%dx%d in %d call %d after %d: %s\n", nx, ny, nz, in, call, after, #c);      \
            return 1;                                                                                   \
        }                                                                                               \
    } while (0)

static int run(int nx, int ny, int nz, int in, int call, int after) {
    st_solver s{};
    st::Geo &g = s.g;
    g.nx = nx; g.ny = ny; g.nz = nz; g.ng = 3;
    g.rx = nx + 6; g.sy = ny + 6; g.sz = nz + 6;
    g.sx = (g.rx + 15) / 16 * 16;
    g.sxy = g.sx * g.sy;
    g.nvol = (long long)g.sxy * g.sz;
    g.nref = (long long)g.rx * g.sy * g.sz;
    events = 0;
    st::stage_create(s.own_stage, 5 * sizeof(double) * (size_t)g.nvol);
    s.stage = &s.own_stage;
    std::vector<double> host(5 * g.nref), dev(5 * g.nvol), want;
    for (size_t t = 0; t < host.size(); t++) host[t] = in ? (double)t + 1.0 : 0.0;
    for (size_t t = 0; t < dev.size(); t++) dev[t] = in ? -1.0 : (double)t + 1.0;
    for (int &l : left) l = -1;
    if (call < kCalls) left[call] = after;
    const hipError_t e = in ? st::copy_rows(&s, dev.data(), host.data(), 8, 5, hipMemcpyHostToDevice)
                            : st::copy_rows(&s, host.data(), dev.data(), 8, 5, hipMemcpyDeviceToHost);
    const size_t flight = queue.size() - done;
    const bool failed = call < kCalls && left[call] < 0;
    queue.clear();
    done = 0;
    st::stage_destroy(s.own_stage);
    CHECK(flight == 0);
    CHECK((e != hipSuccess) == failed);
    if (failed) return 0;
    for (int m = 0; m < 5; m++)
        for (size_t r = 0; r < (size_t)g.sy * g.sz; r++)
            for (int i = 0; i < g.sx; i++) {
                const double d = dev[m * g.nvol + r * g.sx + i];
                if (i < g.rx) CHECK(d == host[m * g.nref + r * g.rx + i]);
                else if (in) CHECK(d == 0.0);
            }
    return 0;
}

int main() {
    int bad = 0;
    for (int in = 0; in < 2; in++) {
        // one thread, and several
        bad += run(13, 9, 7, in, kCalls, 0) + run(70, 90, 80, in, kCalls, 0);
        for (int call = 0; call < kCalls; call++)
            for (int after = 0; after < 8; after++)
                bad += run(13, 9, 7, in, call, after) + run(70, 90, 80, in, call, after);
    }
    return bad ? 1 : 0;
}
