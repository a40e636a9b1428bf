// kvd_batch.h -- the buffers of batched calls (prefill, batched decode), the list
// of idle ones a model keeps, and device allocation that gives those back before
// it fails.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

namespace kvd {

// logits of a batched step leave through pinned slots (logits_to_host)
constexpr int LOGIT_SLOTS = 4;
constexpr size_t LOGIT_SLOT_BYTES = (size_t)1 << 20;

// One set of buffers: [tokens][...] rows, GEMM operands, score grids.  A call leases
// one from its model and gives it back when its stream has drained (BatchLease),
// so sessions that prefill one after the other share one, and threads that run at
// once have one each.
struct Batch {
    bool flt = false;                    // holds the float attention's partials too: serves both modes
    int pmax = 0;                        // serves this pmax and below
    void *buf = nullptr;
    size_t bytes = 0;                    // of buf
    int TB = 0, mcb = 0;                 // tokens per attention batch, chunk capacity per q-head
    float *x0, *x1, *q, *k, *v, *qr, *ao, *ap, *hh, *dn, *rope, *part, *part_ml;
    int8_t *planes; int *sh, *counter, *zs;
    int64_t *vacc, *vacc_s;
    int64_t *gpart; int *gcnt;           // GEMM split-K partial slices and tile arrival counters
    // batched decode over sessions (allocated on first use): logits rows,
    // greedy tokens, per-token token / position / per-layer page tables
    void *dbuf = nullptr;
    float *logits; int *next, *toks, *tpos; float *const **tpages;
    int2 *work; int nwork = 0, wcap = 0;   // full-context layers' (token, chunk) work items
    void *hstage = nullptr;              // pinned: toks/tpos/tpages/work as uploaded, then:
    int *hnext = nullptr;                // the greedy tokens
    uint8_t *hslots = nullptr;           // LOGIT_SLOTS pieces of logits on their way to the caller
    hipEvent_t slot_ev[LOGIT_SLOTS] = {};
    bool serves(bool f, int p) const { return (flt || !f) && pmax >= p; }
    void release() {
        if (buf) hipFree(buf);
        if (dbuf) hipFree(dbuf);
        if (hstage) hipHostFree(hstage);
        for (hipEvent_t e : slot_ev) if (e) hipEventDestroy(e);
        *this = Batch{};
    }
};
constexpr size_t MAX_IDLE_BATCHES = 4;       // kept by a model; more go back to the device at once

// A model's idle sets, whole (every counter and total at zero).  Their memory is
// the process's to take back: dev_malloc frees the idle sets of all models.
class BatchSets {
    std::mutex mu;
    Batch idle[MAX_IDLE_BATCHES];            // [0, n), oldest first
    size_t n = 0;
    struct Registry { std::mutex mu; std::vector<BatchSets *> all; };
    static Registry &registry() { static Registry *r = new Registry; return *r; }   // outlives every model
    Batch remove(size_t i) {
        const Batch b = idle[i];
        std::copy(idle + i + 1, idle + n, idle + i);
        idle[--n] = Batch{};
        return b;
    }
    bool release_idle() {
        for (bool any = false;; any = true) {
            Batch b;
            {
                std::lock_guard<std::mutex> lk(mu);
                if (!n) return any;
                b = remove(0);
            }
            b.release();
        }
    }
public:
    BatchSets() {
        Registry &r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        r.all.push_back(this);
    }
    BatchSets(const BatchSets &) = delete;
    ~BatchSets() {
        Registry &r = registry();
        { std::lock_guard<std::mutex> lk(r.mu); r.all.erase(std::find(r.all.begin(), r.all.end(), this)); }
        release_idle();
    }
    // the smallest set that serves the call (a short call leaves the large ones
    // to the calls that need them), or an empty one for it
    Batch take(bool f, int p) {
        std::lock_guard<std::mutex> lk(mu);
        size_t best = n;
        for (size_t i = 0; i < n; i++)
            if (idle[i].serves(f, p) && (best == n || idle[i].bytes < idle[best].bytes)) best = i;
        if (best < n) return remove(best);
        Batch b;
        b.flt = f; b.pmax = p;
        return b;
    }
    // a whole set comes back; past the bound the oldest goes
    void give(const Batch &b) {
        Batch drop;
        {
            std::lock_guard<std::mutex> lk(mu);
            if (n == MAX_IDLE_BATCHES) drop = remove(0);
            idle[n++] = b;
        }
        drop.release();
    }
    static bool reclaim() {
        Registry &r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        bool any = false;
        for (BatchSets *s : r.all) any |= s->release_idle();
        return any;
    }
};

// hipMalloc, once more without the idle sets where the device is full
template <class T> hipError_t dev_malloc(T **p, size_t n) {
    hipError_t e = hipMalloc((void **)p, n);
    if (e == hipErrorOutOfMemory && BatchSets::reclaim()) {
        (void)hipGetLastError();             // the first attempt's, or a later launch check would report it
        e = hipMalloc((void **)p, n);
    }
    return e;
}

}  // namespace kvd
