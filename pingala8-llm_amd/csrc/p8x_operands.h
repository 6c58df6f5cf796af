// p8x_operands.h -- device memory of the prompt GEMM's decoded fp16 weight operands. They live within one call, so the
// calls of all tensors on a GPU share it. A call that gets none runs the kernel that decodes as it multiplies
// (k_mm): the same bits, slower. Templated on the device calls (HipApi in p8x_gemm.hip), so that the rules can be tested
// without a GPU.
#pragma once
#include <cstddef>
#include <mutex>

namespace p8x {

// A buffer of at least `need` bytes in *p (*have: its size), or false with the old one kept: running out of memory is no
// error here, and leaves none behind for the next launch's check. The new buffer is allocated before the old one is
// given back; the device is synchronized before that, since calls in flight may still use it.
template <class Api>
bool try_grow(void **p, size_t *have, size_t need) {
    if (*have >= need) return true;
    void *q = nullptr;
    if (!Api::alloc(&q, need)) {
        Api::clear_error();
        return false;
    }
    if (*p) {
        if (!Api::synchronize()) {
            Api::clear_error();
            Api::release(q);
            return false;
        }
        Api::release(*p);
    }
    *p = q;
    *have = need;
    return true;
}

// What the last kernel of a call that uses the buffer is given: its first workgroup stores n in *word (host memory), which
// tells that the launches before it have ended.
struct OperandMark {
    unsigned long long *word = nullptr, n = 0;
};

// A buffer that the calls on one GPU share. One call holds it at a time (its lock spans the call's launches), and a word
// in host memory, which the kernel behind those that read the buffer writes, tells when the GPU is done with it. (An event
// recorded there took 1.5 to 3 us a call, 33.0 -> 34.5 / 36.0 for 300 tokens of 1024 x 4096; given to the launch as its
// stop event, it took 30 us of a first call after a pause.) A call on the stream that used it last is ordered behind that
// use (a stream's work has ended before its handle is another's: hipStreamDestroy waits for it; Api::ordered says which
// handles name one stream); a call on any other stream gets it only once that use has ended, and nothing otherwise: it
// neither waits for another stream nor makes its own wait. Calls under stream capture get nothing, since a graph may be
// replayed beside anything. The memory is given back when the last tensor that can use it is released.
template <class Api>
class OperandBuffer {
public:
    class Lease {
    public:
        explicit Lease(void *p_ = nullptr) : p(p_) {}
        Lease(Lease &&o) : p(o.p), b(o.b), st(o.st), on(o.on) { o.p = nullptr; o.b = nullptr; }
        Lease(const Lease &) = delete;
        Lease &operator=(const Lease &) = delete;
        ~Lease() { if (b) b->done(st, on); }
        OperandMark mark() const { return OperandMark{b->word, b->seq}; }
        void launched() { on = true; }   // the kernel with the mark is on the stream, behind those that use the buffer
        void *p;   // null: no buffer

    private:
        friend class OperandBuffer;
        OperandBuffer *b = nullptr;
        typename Api::Stream st{};
        bool on = false;
    };

    void add_user() {
        std::lock_guard<std::mutex> lk(mu);
        ++users;
    }
    void drop_user() {
        std::lock_guard<std::mutex> lk(mu);
        failed = 0;   // memory came free
        if (--users || !buf) return;
        Api::release(buf);   // waits for the device
        buf = nullptr;
        bytes = 0;
        used = false;   // the word stays
    }
    // at set-up: the buffer is there for later calls of up to `need` bytes, if the memory is
    void reserve(size_t need) {
        std::lock_guard<std::mutex> lk(mu);
        failed = 0;
        (void)provide(need);
    }
    Lease take(size_t need, typename Api::Stream st) {
        Lease l;
        if (Api::capturing(st)) return l;
        mu.lock();
        const bool ready = !used || Api::ordered(st, last) || __atomic_load_n(word, __ATOMIC_ACQUIRE) == seq;
        if (!ready || !provide(need)) {
            mu.unlock();
            return l;
        }
        ++seq;
        l.p = buf;
        l.b = this;
        l.st = st;
        return l;
    }

private:
    bool provide(size_t need) {
        if (failed && need >= failed) return false;   // not tried again on every call
        if (word || Api::host_word(&word)) {
            if (try_grow<Api>(&buf, &bytes, need)) return true;
        }
        failed = need;
        return false;
    }
    void done(typename Api::Stream st, bool on) {
        last = st;
        used = on;
        if (!on) (void)Api::synchronize();   // a launch failed, no mark covers those before it
        mu.unlock();
    }

    std::mutex mu;
    void *buf = nullptr;
    size_t bytes = 0, failed = 0;
    unsigned long long *word = nullptr, seq = 0;   // the mark of the last use
    typename Api::Stream last{};
    bool used = false;   // launches of the last use may still run
    int users = 0;
};

// The buffers of a GPU: one, and up to three more from when calls on as many streams have overlapped (their first use
// allocates them). A call that finds them all in use on other streams gets none. Four, as HIP gives a process four hardware
// queues: us a call of 4096 x 14336, classes 2-4, 1500 tokens on 1, 2 and 3 streams 199, 177 and 187 with a buffer per
// tensor, 199, 177 and 244 with two in all.
template <class Api>
class OperandPool {
public:
    void add_user() { for (auto &x : b) x.add_user(); }
    void drop_user() { for (auto &x : b) x.drop_user(); }
    void reserve(size_t need) { b[0].reserve(need); }
    typename OperandBuffer<Api>::Lease take(size_t need, typename Api::Stream st) {
        for (auto &x : b) {
            auto l = x.take(need, st);
            if (l.p) return l;
        }
        return typename OperandBuffer<Api>::Lease();
    }

private:
    OperandBuffer<Api> b[4];
};

// The operands of calls that may not allocate: buffers of fixed sizes, allocated when the first tensor that needs one is
// prepared and given back with the last of all, so a captured call's pointer holds as long as its tensor. Calls that share
// them are ordered by the caller.
template <class Api>
class FixedOperands {
public:
    static constexpr size_t kSizes[] = {(size_t)16 << 20, (size_t)64 << 20, (size_t)192 << 20};

    void add_user(size_t need) {
        std::lock_guard<std::mutex> lk(mu);
        ++users;
        for (int i = 0; i < kN; ++i)
            if (need <= kSizes[i]) {
                if (!buf[i] && !Api::alloc(&buf[i], kSizes[i])) {
                    Api::clear_error();
                    buf[i] = nullptr;
                }
                return;
            }
    }
    void drop_user() {
        std::lock_guard<std::mutex> lk(mu);
        if (--users) return;
        for (void *&b : buf) {
            if (b) Api::release(b);
            b = nullptr;
        }
    }
    void *get(size_t need) {   // null: none
        std::lock_guard<std::mutex> lk(mu);
        for (int i = 0; i < kN; ++i)
            if (need <= kSizes[i] && buf[i]) return buf[i];
        return nullptr;
    }

private:
    static constexpr int kN = sizeof kSizes / sizeof *kSizes;
    std::mutex mu;
    void *buf[kN] = {};
    int users = 0;
};

}  // namespace p8x
