// host_stage.h — how the drop-ins on host arrays bring their operands to the device and their results back.
// Included by host_dropins.hip inside its unnamed namespace.
//
// A copy from or to ordinary host memory goes through the runtime's own staging, one block after the other: 256 KB 106 us,
// 4 MB 153 us in and 245 us out, where the same from pinned memory takes 12.6 and 81 us (55 GB/s and 6 us).  The caller's
// arrays cannot be pinned, so a call packs its inputs into a pinned block of the library's own, in the order they have on the
// device, and sends it in a few copies that grow (256 KB, 512 KB, ... 4 MB): while one travels the next is filled.  Results
// come back the same way in copies that shrink, each unpacked while the next travels.  One thread moves 30 GB/s of memory
// that is in no cache, so HELPERS threads of the library pack and unpack beside the caller's (1, 2, 3 and 6: 3.5, 2.5, 2.4 and
// 2.5 ms for the nine calls of a layer, a loss and an update; 4.9 through the runtime).  What bounds it: the link, in one
// direction at a time (88 MB, 1.6 ms).
//
// The helpers touch nothing but memory: they are given pieces of at most 64 KB, take them by counting up one number, and
// mark each when it is done.  The caller takes pieces as well and waits only for pieces that somebody has taken, so a
// helper that is asleep, late or was never created (no more processors, no threads left, a forked child) costs time and nothing
// else.  Between calls they look for work for 100 us and then sleep.
//
// Results are unpacked as their bytes arrive.  A call that fails leaves the arrays that it updates in place as they were, so that
// it can be made again: when a copy back fails they are filled again with what they held.  Where one round holds the inputs, that
// is still in the pinned block, and the results come back through another (unpacked behind the last copy instead, the nine calls took
// 2.59 ms for 2.37); otherwise each piece of such an array is copied to a log as it is packed, which costs 1 to 2 %
// (results held in ordinary memory until the last copy: nine calls 8.5 ms for 4.1).
#pragma once

constexpr int HELPERS = 3;
constexpr size_t PIECE = (size_t)64 << 10;
constexpr size_t PIN_MAX = (size_t)32 << 20;         // bytes of a pinned block at most; longer transfers go in rounds of this
constexpr int MAX_PIECES = 2 * (int)(PIN_MAX / PIECE) + 256;
constexpr size_t SEND_MIN = (size_t)256 << 10, SEND_MAX = (size_t)4 << 20;
constexpr int MAX_SENDS = 32;                        // copies of a round

// A host array of a call and where it lies in the call's block.  rows: the array is `rows`[i] * row_bytes behind host for i =
// 0 .., row_bytes each, and contiguous in the block.
struct Part {
    char *host;
    size_t at, bytes;
    const int *rows;
    size_t row_bytes;
    char *log;                           // where what the array held is copied to while it is packed, or NULL
};

// memcpy past the caches: what the device reads next, or results that are larger than a cache (18.9 MB unpacked in 344 us, with
// memcpy 450)
void copy_past(char *to, const char *from, size_t n) {
    if (n < 256) { memcpy(to, from, n); return; }
    const size_t head = (16 - ((uintptr_t)to & 15)) & 15;
    memcpy(to, from, head);
    to += head;
    from += head;
    n -= head;
    for (; n >= 64; n -= 64, to += 64, from += 64) {
        __m128i v[4];
        for (int i = 0; i < 4; i++) v[i] = _mm_loadu_si128((const __m128i *)(from + 16 * i));
        for (int i = 0; i < 4; i++) _mm_stream_si128((__m128i *)(to + 16 * i), v[i]);
    }
    memcpy(to, from, n);
    _mm_sfence();
}

// `bytes` bytes from byte `from` of a part on; to the block or back
void move_part(const Part &p, size_t from, size_t bytes, char *block, bool in, bool past) {
    const auto copy = [past](char *to, const char *from, size_t n) {
        if (past) copy_past(to, from, n);
        else memcpy(to, from, n);
    };
    if (!p.rows) {
        if (in) copy(block, p.host + from, bytes);
        else copy(p.host + from, block, bytes);
        return;
    }
    while (bytes) {
        const size_t r = from / p.row_bytes, o = from - r * p.row_bytes, n = p.row_bytes - o < bytes ? p.row_bytes - o : bytes;
        char *h = p.host + (size_t)p.rows[r] * p.row_bytes + o;
        if (in) copy(block, h, n);
        else copy(h, block, n);
        block += n;
        from += n;
        bytes -= n;
    }
}

struct Piece {
    const Part *part;
    size_t from, bytes;
    char *block;
    bool in, past;                       // to the block or back; past the caches
};

enum : unsigned char { TO_DO, PACKED, DONE };       // PACKED: may be sent, the log is still to come

struct Helpers {
    pthread_t thread[HELPERS];
    int n;                                // created
    int mode;                             // g_ctx.host_stage at the time
    pid_t pid;                            // of the process that created them
    pthread_mutex_t lock;
    pthread_cond_t wake;
    bool stop;                            // under the lock
    std::atomic<int> asleep;
    std::atomic<unsigned> calls;          // goes up with each round of pieces: a helper that has slept looks again
    // the round at hand: pieces below `ready` may be taken; `next` counts them out (its upper half is the round's number, so that
    // a helper that was late for a round takes nothing of the one behind it)
    std::atomic<unsigned long long> next;
    std::atomic<int> ready;
    std::atomic<int> active;              // between the start of a round and its end
    Piece piece[MAX_PIECES];
    std::atomic<unsigned char> done[MAX_PIECES];
};
Helpers *g_helpers = nullptr;

// takes and moves one piece of the round; false if there is none to take
bool one_piece(Helpers *h) {
    unsigned long long n = h->next.load(std::memory_order_acquire);
    for (;;) {
        if ((int)(n & 0xffffffffu) >= h->ready.load(std::memory_order_acquire)) return false;
        if (h->next.compare_exchange_weak(n, n + 1, std::memory_order_acq_rel, std::memory_order_acquire)) break;
    }
    const int i = (int)(n & 0xffffffffu);
    const Piece &p = h->piece[i];
    move_part(*p.part, p.from, p.bytes, p.block, p.in, p.past);
    if (p.in && p.part->log) {
        h->done[i].store(PACKED, std::memory_order_release);
        move_part(*p.part, p.from, p.bytes, p.part->log + p.from, true, true);
    }
    h->done[i].store(DONE, std::memory_order_release);
    return true;
}

// The pieces 0 .. pieces - 1 become a round, of which the first `ready` may be taken; the round's number.
unsigned long long start_pieces(Helpers *h, int pieces, int ready) {
    // no helper may still be looking at the round before
    const unsigned long long number = (h->next.load(std::memory_order_relaxed) >> 32) + 1;
    h->ready.store(0, std::memory_order_seq_cst);
    h->next.store(number << 32, std::memory_order_seq_cst);
    h->ready.store(ready, std::memory_order_seq_cst);
    if (pieces > 4 && h->n > 0) {
        h->active.store(1);
        h->calls.fetch_add(1);
        if (h->asleep.load() > 0) {
            pthread_mutex_lock(&h->lock);
            pthread_cond_broadcast(&h->wake);
            pthread_mutex_unlock(&h->lock);
        }
    }
    return number;
}

// Takes what is left of a round (after an error nothing more is), and waits for the pieces that helpers have taken.
void end_pieces(Helpers *h, int pieces, unsigned long long number, bool ok) {
    int taken = pieces;
    if (ok) while (one_piece(h)) { }
    else taken = std::min(pieces, (int)(h->next.exchange((number << 32) | 0x7fffffffu) & 0x7fffffffu));
    for (int i = 0; i < taken; i++)
        while (h->done[i].load(std::memory_order_acquire) != DONE) __builtin_ia32_pause();
    h->active.store(0);
}

void *helper_main(void *arg) {
    Helpers *h = (Helpers *)arg;
    unsigned seen = h->calls.load(std::memory_order_acquire);
    int idle = 0;
    for (;;) {
        if (one_piece(h)) { idle = 0; continue; }
        if (h->active.load(std::memory_order_acquire)) idle = 0;           // pieces of this round are still to come
        if (++idle < 800) {                               // about 100 us
            for (int i = 0; i < 8; i++) __builtin_ia32_pause();
            continue;
        }
        idle = 0;
        pthread_mutex_lock(&h->lock);
        h->asleep.fetch_add(1);
        while (!h->stop && h->calls.load() == seen) pthread_cond_wait(&h->wake, &h->lock);
        seen = h->calls.load();
        h->asleep.fetch_sub(1);
        const bool stop = h->stop;
        pthread_mutex_unlock(&h->lock);
        if (stop) return nullptr;
    }
}

void stop_helpers() {
    Helpers *h = g_helpers;
    if (!h || h->pid != getpid()) return;                 // (a forked child has no threads to stop)
    pthread_mutex_lock(&h->lock);
    h->stop = true;
    pthread_cond_broadcast(&h->wake);
    pthread_mutex_unlock(&h->lock);
    for (int i = 0; i < h->n; i++) pthread_join(h->thread[i], nullptr);
    pthread_cond_destroy(&h->wake);
    pthread_mutex_destroy(&h->lock);
    free(h);
    g_helpers = nullptr;
}
// (threads that run when the library's code goes away would crash)
__attribute__((destructor)) void stop_helpers_at_exit() { stop_helpers(); }

// The helpers' state, created with its threads on first use; NULL without memory for it.
Helpers *helpers() {
    if (g_helpers && g_helpers->mode != g_ctx.host_stage) stop_helpers();
    if (g_helpers) return g_helpers;
    Helpers *h = (Helpers *)calloc(1, sizeof(Helpers));
    if (!h) return nullptr;
    pthread_mutex_init(&h->lock, nullptr);
    pthread_cond_init(&h->wake, nullptr);
    h->pid = getpid();
    h->mode = g_ctx.host_stage;
    cpu_set_t cpus;
    const int have = sched_getaffinity(0, sizeof(cpus), &cpus) == 0 ? CPU_COUNT(&cpus) : 1;
    sigset_t all, old;                                    // the program's signals are not for them
    sigfillset(&all);
    pthread_sigmask(SIG_SETMASK, &all, &old);
    while (h->mode != 1 && h->n < HELPERS && h->n + 1 < have && pthread_create(&h->thread[h->n], nullptr, helper_main, h) == 0) h->n++;
    pthread_sigmask(SIG_SETMASK, &old, nullptr);
    return g_helpers = h;
}

// ---- the blocks ----
struct Pinned {
    char *host, *dev;                                // its address here and on the device
    size_t bytes;
};
Pinned g_pin = {}, g_pin_back = {};                  // the second for results of elementwise calls and of calls that update arrays
hipEvent_t g_sent[MAX_SENDS] = {};
char *g_log = nullptr;                               // old values of arrays that a call updates
size_t g_log_bytes = 0;
constexpr size_t LOG_KEPT = (size_t)256 << 20;       // a longer one does not outlive its call

// pinned memory for min(bytes, PIN_MAX) and the events of a round; false where there is none
bool pinned(Pinned &p, size_t bytes) {
    if (g_ctx.host_stage == 2) return false;
    if (!g_sent[MAX_SENDS - 1])
        for (auto &e : g_sent)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) { e = nullptr; (void)hipGetLastError(); return false; }
    size_t want = (size_t)1 << 20;
    while (want < bytes && want < PIN_MAX) want *= 2;
    if (p.host && p.bytes >= want) return true;
    if (p.host) (void)hipHostFree(p.host);                 // (between calls nothing travels)
    p = Pinned{};
    void *h = nullptr, *d = nullptr;
    if (hipHostMalloc(&h, want, hipHostMallocMapped) != hipSuccess) { (void)hipGetLastError(); return false; }
    if (hipHostGetDevicePointer(&d, h, 0) != hipSuccess) { (void)hipGetLastError(); (void)hipHostFree(h); return false; }
    p = Pinned{(char *)h, (char *)d, want};
    return true;
}

char *log_space(size_t bytes) {
    if (bytes <= g_log_bytes) return g_log;
    free(g_log);
    g_log = (char *)malloc(bytes);
    g_log_bytes = g_log ? bytes : 0;
    if (!g_log) mi355_fail("no host memory for %zu bytes of old values", bytes);
    return g_log;
}
void free_log() {
    free(g_log);
    g_log = nullptr;
    g_log_bytes = 0;
}

// A copy between the pinned block and the device's: 16 bytes at a time, over the link at 50 GB/s from 1 MB on.  By a kernel, not
// a copy engine: the engine waits 9 us for the kernel before it and lets the one behind it wait as long (16 MB in pieces of 1 MB:
// 442 us in and 440 out, by kernels 375 and 332).
__global__ __launch_bounds__(256) void stage_copy_kernel(v4i *__restrict__ to, const v4i *__restrict__ from, unsigned n) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
        __builtin_nontemporal_store(__builtin_nontemporal_load(from + i), to + i);
}
hipError_t stage_copy(char *to, const char *from, size_t bytes) {
    const unsigned n = (unsigned)ceil_div(bytes, 16);
    hipLaunchKernelGGL(stage_copy_kernel, dim3(std::min(512u, (n + 255) / 256)), dim3(256), 0, g_ctx.stream, (v4i *)to, (const v4i *)from, n);
    return hipGetLastError();
}

void free_stage() {
    stop_helpers();
    for (Pinned *p : {&g_pin, &g_pin_back}) {
        if (p->host) (void)hipHostFree(p->host);
        *p = Pinned{};
    }
    free_log();
    for (auto &e : g_sent) { if (e) (void)hipEventDestroy(e); e = nullptr; }
}

// The operands of one call: laid out one behind the other in a block of device memory, in the order in which they are added.
// The inputs have to be neighbours, and the results (what lies between two of them travels with them).
class Stage {
public:
    // each returns the part's number
    int in(const void *host, size_t bytes) { return add((void *)host, bytes, true, false); }
    int out(void *host, size_t bytes) { return add(host, bytes, false, true); }
    int inout(void *host, size_t bytes) { return add(host, bytes, true, true); }
    int rows_inout(void *host, const int *rows, size_t n, size_t row_bytes) {
        const int i = add(host, n * row_bytes, true, true);
        p_[i].rows = rows;
        p_[i].row_bytes = row_bytes;
        return i;
    }
    template <typename T>
    T *dev(int i) const { return (T *)(dev_ + p_[i].at); }

    // the part is a result from here on, and belongs to this array
    void becomes(int i, void *host) { p_[i].host = (char *)host; in_[i] = false; out_[i] = true; }

    ~Stage() { if (g_log_bytes > LOG_KEPT) free_log(); }

    // device memory, and the inputs on their way to it
    bool send() {
        dev_ = (char *)slot(0, total_);
        if (!dev_) return false;
        size_t updated = 0;
        for (int i = 0; i < n_; i++)
            if (in_[i] && out_[i]) updated += p_[i].bytes;
        // (no pinned memory: each array by itself, and the log)
        pin_ = helpers() && pinned(g_pin, total_) ? &g_pin : nullptr;
        back_ = pin_ && updated && total_ <= pin_->bytes && pinned(g_pin_back, total_) ? &g_pin_back : pin_;
        if (updated && back_ == pin_) {
            char *log = log_space(updated);
            if (!log) return false;
            for (int i = 0; i < n_; i++)
                if (in_[i] && out_[i]) {
                    p_[i].log = log;
                    log += p_[i].bytes;
                }
        }
        return move(true);
    }
    // brings the results to their arrays; those that are inputs too are as before the call unless it returns true
    bool receive() {
        copies_ = 0;
        if (move(false)) return true;
        for (int i = 0; i < n_; i++)
            if (in_[i] && out_[i]) unpack(helpers(), p_[i], p_[i].log ? p_[i].log : g_pin.host + (p_[i].at - sent_));
        return false;
    }

    // Elementwise calls on parts of n floats: the arrays go through in chunks of values, and the kernel of a chunk reads the pinned block
    // of the inputs and writes that of the results itself, one launch in the place of a copy, the operation and a copy; what has come
    // back is unpacked while later chunks are packed and travel.  chunk(in, out, count): in[i], out[i] are the addresses of
    // part i's values; 0 if it was launched.  Longer arrays than a block holds go in rounds.
    // 1: done.  0: nothing has been done (no pinned memory, or arrays that overlap other than value by value); the call takes
    // the other way.  -1: failed; the arrays that are inputs and results, of one part or of two, are as before the call, and so
    // are those that it only writes unless every chunk was launched and the results of one did not come back.
    // Of arrays that are only written nothing is kept that could be put back.  Where a call has any, nothing is unpacked before the
    // last chunk is launched; what that takes from the overlap the threads spend on packing, which is then done sooner.  Longer ones than a block
    // holds would be written in one round with the chunks of the next still to be launched: those take the other way.
    // us, by way of the device / so: Adam step of [2048][768] 968 / 887, of [3072][1024] 2030 / 1800, SwiGLU backward of [2048][256] 281 /
    // 252, forward 187 / 171, axpby of [768][256] 92 / 82.  Bound by the link, whose 57 GB/s are those of both directions together (two
    // copies of 64 MB, one each way, take as long at once as one after the other), and by 7 us between the kernels of two chunks.
    template <typename F>
    int stream(size_t n, const F &chunk) {
        int ins = 0;
        size_t updated = 0;
        bool old[MAX];                    // inputs that results are written over
        bool only = false;                // a result that lies over no input
        for (int i = 0; i < n_; i++) {
            if (p_[i].rows || p_[i].bytes != n * sizeof(float)) return 0;
            ins += in_[i];
            old[i] = in_[i] && out_[i];
            for (int j = 0; j < n_; j++) {
                if (i == j || !out_[j]) continue;
                const char *a = p_[i].host, *b = p_[j].host;
                if (a == b ? out_[i] : a < b + p_[j].bytes && b < a + p_[i].bytes) return 0;
                old[i] |= a == b;
            }
            if (old[i]) updated += p_[i].bytes;
            bool over = in_[i];
            for (int j = 0; j < n_; j++) over |= in_[j] && p_[j].host == p_[i].host;
            only |= out_[i] && !over;
        }
        Helpers *h = helpers();
        if (!h) return 0;
        const size_t most = PIN_MAX / (sizeof(float) * n_) & ~(size_t)4095;
        const size_t len = std::min(most, (n + 63) & ~(size_t)63), stride = len * sizeof(float);     // values of a round
        if (only && len < n) return 0;
        if (!pinned(g_pin, stride * n_) || !pinned(g_pin_back, stride * n_)) return 0;
        const bool logged = updated && len < n;
        if (logged) {
            char *log = log_space(updated);
            if (!log) return -1;
            for (int i = 0; i < n_; i++)
                if (old[i]) {
                    p_[i].log = log;
                    log += p_[i].bytes;
                }
        }
        copies_ = 0;
        int chunks = 0;
        for (size_t r0 = 0; r0 < n; r0 += len) {
            const size_t cnt = std::min(len, n - r0);
            // the ends of the chunks: they grow, and shrink again
            size_t cut[MAX_SENDS];
            int sends = 0;
            const size_t least = SEND_MIN / sizeof(float) / ins, largest = SEND_MAX / sizeof(float) / ins;
            for (size_t at = 0, c = least; at < cnt; sends++) {
                at += std::min(std::min(c, largest), std::max(least, (cnt - at) / 2)) & ~(size_t)1023;
                c *= 2;
                if (at > cnt || sends + 1 == MAX_SENDS) at = cnt;
                cut[sends] = at;
            }
            // the pieces in the order in which they are taken: a chunk's results two chunks behind its inputs, or behind all inputs
            const int lag = only ? sends : 2;
            int pieces = 0, packed[MAX_SENDS], last[MAX_SENDS], back_from[MAX_SENDS];       // first and last + 1 to pack, first to unpack
            auto add_pieces = [&](int s, bool in) {
                const size_t from = s ? cut[s - 1] : 0;
                for (int i = 0; i < n_; i++) {
                    if (!(in ? in_[i] : out_[i])) continue;
                    for (size_t at = from * sizeof(float); at < cut[s] * sizeof(float); at += PIECE) {
                        h->done[pieces].store(TO_DO, std::memory_order_relaxed);
                        h->piece[pieces++] = Piece{&p_[i], r0 * sizeof(float) + at, std::min(cut[s] * sizeof(float) - at, PIECE),
                                                   (in ? g_pin.host : g_pin_back.host) + i * stride + at, in, in || p_[i].bytes > (size_t)1 << 20};
                    }
                }
            };
            for (int s = 0; s < sends + lag; s++) {
                if (s < sends) {
                    packed[s] = pieces;
                    add_pieces(s, true);
                    last[s] = pieces;
                }
                if (s >= lag) {
                    back_from[s - lag] = pieces;
                    add_pieces(s - lag, false);
                }
            }
            const unsigned long long number = start_pieces(h, pieces, back_from[0]);
            hipError_t e = hipSuccess;
            int rc = 0, sent = 0, come = 0, ok = 0;
            while (come < sends && e == hipSuccess && rc == 0) {
                bool idle = true;
                if (sent < sends) {
                    ok = std::max(ok, packed[sent]);
                    // (an array's old values are in the log before any of it is written again)
                    while (ok < last[sent]) {
                        const unsigned char d = h->done[ok].load(std::memory_order_acquire);
                        if (d == TO_DO || (logged && d != DONE)) break;
                        ok++;
                    }
                    if (ok == last[sent]) {
                        const size_t from = sent ? cut[sent - 1] : 0;
                        float *in[MAX], *out[MAX];
                        for (int i = 0; i < n_; i++) {
                            in[i] = (float *)(g_pin.dev + i * stride) + from;
                            out[i] = (float *)(g_pin_back.dev + i * stride) + from;
                        }
                        // (or what g_ctx.host_stage_fail makes of it)
                        rc = ++chunks == -g_ctx.host_stage_fail ? mi355_fail("chunk %d launch: refused", chunks) : chunk(in, out, cut[sent] - from);
                        if (rc == 0) e = hipEventRecord(g_sent[sent], g_ctx.stream);
                        sent++;
                        idle = false;
                    }
                }
                if (e == hipSuccess && rc == 0 && come < (only && sent < sends ? 0 : sent)) {
                    const hipError_t q = hipEventQuery(g_sent[come]);
                    if (q == hipErrorNotReady) {
                        (void)hipGetLastError();
                    } else {
                        e = back(q);
                        if (e == hipSuccess) {
                            come++;
                            h->ready.store(come < sends ? back_from[come] : pieces, std::memory_order_release);
                        }
                        idle = false;
                    }
                }
                if (idle && !one_piece(h)) __builtin_ia32_pause();
            }
            const bool good = e == hipSuccess && rc == 0;
            end_pieces(h, pieces, number, good);
            if (good) continue;
            if (e != hipSuccess) fail("D2H", e);
            else (void)hipStreamSynchronize(g_ctx.stream);
            const size_t written = (r0 + (come ? cut[come - 1] : 0)) * sizeof(float);
            for (int i = 0; i < n_; i++)
                if (old[i]) {
                    Part p = p_[i];
                    p.bytes = written;
                    unpack(h, p, logged ? p.log : g_pin.host + i * stride);
                }
            return -1;
        }
        return 1;
    }

private:
    static constexpr int MAX = 8;
    Part p_[MAX];
    bool in_[MAX], out_[MAX];
    int n_ = 0;
    size_t total_ = 0;
    char *dev_ = nullptr;
    const Pinned *pin_ = nullptr, *back_ = nullptr;         // what the inputs and the results go through; NULL: nothing
    size_t sent_ = 0;           // where the inputs begin
    int copies_ = 0;            // of this receive()

    int add(void *host, size_t bytes, bool in, bool out) {
        p_[n_] = Part{(char *)host, total_, bytes, nullptr, 0, nullptr};
        in_[n_] = in;
        out_[n_] = out;
        total_ += (bytes + 255) & ~(size_t)255;
        return n_++;
    }
    bool fail(const char *what, hipError_t e) const {
        mi355_fail("%s copy: %s", what, hipGetErrorString(e));
        (void)hipStreamSynchronize(g_ctx.stream);          // nothing of the call is in the blocks any more
        return false;
    }

    bool move(bool in) {
        const char *what = in ? "H2D" : "D2H";
        size_t lo = total_, hi = 0;
        for (int i = 0; i < n_; i++)
            if (in ? in_[i] : out_[i]) {
                lo = std::min(lo, p_[i].at);
                hi = std::max(hi, p_[i].at + p_[i].bytes);
            }
        if (lo >= hi) return true;
        if (in) sent_ = lo;
        const Pinned *pin = in ? pin_ : back_;
        Helpers *h = helpers();
        if (!pin || !h) return move_unpinned(in, what);
        for (size_t beg = lo; beg < hi; beg += pin->bytes) {
            if (in && beg > lo) {                          // the block is filled again: the last round has to have left it
                const hipError_t e = hipStreamSynchronize(g_ctx.stream);
                if (e != hipSuccess) return fail(what, e);
            }
            if (!round(in, what, h, *pin, beg, std::min(hi, beg + pin->bytes))) return false;
        }
        return true;
    }

    // a whole part from host memory at `from` to its array
    static void unpack(Helpers *h, const Part &p, char *from) {
        if (!h) { move_part(p, 0, p.bytes, from, false, true); return; }
        for (size_t at = 0; at < p.bytes;) {
            int pieces = 0;
            for (; pieces < MAX_PIECES && at < p.bytes; at += PIECE) {
                h->done[pieces].store(TO_DO, std::memory_order_relaxed);
                h->piece[pieces++] = Piece{&p, at, std::min(p.bytes - at, PIECE), from + at, false, true};
            }
            end_pieces(h, pieces, start_pieces(h, pieces, pieces), true);
        }
    }

    // a copy that has come back, or what g_ctx.host_stage_fail makes of it
    hipError_t back(hipError_t e) { return e == hipSuccess && ++copies_ == g_ctx.host_stage_fail ? hipErrorUnknown : e; }

    // bytes beg .. end - 1 of the device block, through the pinned one
    bool round(bool in, const char *what, Helpers *h, const Pinned &pin, size_t beg, size_t end) {
        // the ends of the copies
        size_t cut[MAX_SENDS];
        int sends = 0;
        for (size_t at = beg, c = SEND_MIN; at < end; sends++) {
            if (in) {
                at += c;
                c = std::min(2 * c, SEND_MAX);
            } else {
                at += std::min(SEND_MAX, std::max(SEND_MIN, ((end - at) / 2 + 0xffff) & ~(size_t)0xffff));
            }
            if (at > end || sends + 1 == MAX_SENDS) at = end;
            cut[sends] = at;
        }
        const bool past = in || end - beg > (size_t)1 << 20;        // (small results stay in the caches for their reader)
        // the pieces, none across the end of a copy; last[s]: pieces up to the end of copy s
        int pieces = 0, last[MAX_SENDS], s = 0;
        for (int i = 0; i < n_; i++) {
            if (!(in ? in_[i] : out_[i])) continue;
            size_t at = std::max(p_[i].at, beg);
            const size_t stop = std::min(p_[i].at + p_[i].bytes, end);
            while (at < stop) {
                while (at >= cut[s]) last[s++] = pieces;
                const size_t n = std::min(std::min(stop, cut[s]) - at, PIECE);
                h->done[pieces].store(TO_DO, std::memory_order_relaxed);
                h->piece[pieces++] = Piece{&p_[i], at - p_[i].at, n, pin.host + (at - beg), in, past};
                at += n;
            }
        }
        while (s < sends) last[s++] = pieces;
        const unsigned long long number = start_pieces(h, pieces, in ? pieces : 0);
        hipError_t e = hipSuccess;
        if (in) {
            int ok = 0;
            size_t from = beg;
            for (s = 0; s < sends;) {
                while (ok < pieces && h->done[ok].load(std::memory_order_acquire) != TO_DO) ok++;
                if (ok >= last[s]) {
                    e = stage_copy(dev_ + from, pin.dev + (from - beg), cut[s] - from);
                    if (e != hipSuccess) break;
                    from = cut[s++];
                } else if (!one_piece(h)) {
                    __builtin_ia32_pause();
                }
            }
        } else {
            size_t from = beg;
            for (s = 0; s < sends && e == hipSuccess; s++) {
                e = stage_copy(pin.dev + (from - beg), dev_ + from, cut[s] - from);
                if (e == hipSuccess) e = hipEventRecord(g_sent[s], g_ctx.stream);
                from = cut[s];
            }
            for (s = 0; s < sends && e == hipSuccess;) {
                e = back(hipEventQuery(g_sent[s]));
                if (e == hipSuccess) {
                    h->ready.store(last[s++], std::memory_order_release);
                } else if (e == hipErrorNotReady) {
                    (void)hipGetLastError();
                    e = hipSuccess;
                    if (!one_piece(h)) __builtin_ia32_pause();
                }
            }
        }
        end_pieces(h, pieces, number, e == hipSuccess);
        return e == hipSuccess || fail(what, e);
    }

    // without pinned memory: each array by itself, through the runtime's staging
    bool move_unpinned(bool in, const char *what) {
        for (int i = 0; i < n_; i++) {
            if (!(in ? in_[i] : out_[i])) continue;
            const Part &p = p_[i];
            if (in && p.log) move_part(p, 0, p.bytes, p.log, true, true);
            const size_t step = p.rows ? p.row_bytes : p.bytes;
            for (size_t r = 0; r * step < p.bytes; r++) {
                char *host = p.host + (p.rows ? (size_t)p.rows[r] * step : 0), *dev = dev_ + p.at + r * step;
                hipError_t e = in ? hipMemcpyAsync(dev, host, step, hipMemcpyHostToDevice, g_ctx.stream)
                                  : hipMemcpyAsync(host, dev, step, hipMemcpyDeviceToHost, g_ctx.stream);
                if (e == hipSuccess && !in) e = back(hipStreamSynchronize(g_ctx.stream));
                if (e != hipSuccess) return fail(what, e);
            }
        }
        return true;
    }
};
