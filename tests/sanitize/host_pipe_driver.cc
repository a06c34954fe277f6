// Host pipeline driver (test infrastructure, built by tests/test_host_pipe_cpu.py): runs HostPipe on streams that are host
// threads, so that a "kernel" can be held as long as a scenario needs, without a GPU. Usage: driver <scenario>.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "host_pipe.h"

// ---------------------------------------------------------------- streams and events on host threads
struct ihipStream_t {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> queue;
    uint64_t queued = 0, done = 0;
    bool ending = false;
    std::thread worker{[this] {
        std::unique_lock<std::mutex> lock(mu);
        for (;;) {
            cv.wait(lock, [&] { return ending || !queue.empty(); });
            if (queue.empty()) return;
            std::function<void()> f = std::move(queue.front());
            queue.pop_front();
            lock.unlock();
            f();
            lock.lock();
            done++;
            cv.notify_all();
        }
    }};
    void push(std::function<void()> f) {
        std::lock_guard<std::mutex> lock(mu);
        queue.push_back(std::move(f));
        queued++;
        cv.notify_all();
    }
    void sync() {
        std::unique_lock<std::mutex> lock(mu);
        const uint64_t upto = queued;
        cv.wait(lock, [&] { return done >= upto; });
    }
    ~ihipStream_t() {
        {
            std::lock_guard<std::mutex> lock(mu);
            ending = true;
            cv.notify_all();
        }
        worker.join();
    }
};
struct ihipEvent_t {
    std::mutex mu;
    std::condition_variable cv;
    uint64_t recorded = 0, reached = 0;
    void wait(uint64_t upto) {
        std::unique_lock<std::mutex> lock(mu);
        cv.wait(lock, [&] { return reached >= upto; });
    }
    uint64_t last() {
        std::lock_guard<std::mutex> lock(mu);
        return recorded;
    }
};

static std::atomic<bool> fail_events{false};

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) { *s = new ihipStream_t; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { s->sync(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    uint64_t k;
    {
        std::lock_guard<std::mutex> lock(e->mu);
        k = ++e->recorded;
    }
    s->push([e, k] {
        std::lock_guard<std::mutex> lock(e->mu);
        e->reached = k;
        e->cv.notify_all();
    });
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int) {
    const uint64_t k = e->last();
    s->push([e, k] { e->wait(k); });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    e->wait(e->last());
    return fail_events ? hipErrorUnknown : hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t s) {
    s->push([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) {
    return hipErrorUnknown;
}
}

// ---------------------------------------------------------------- scenarios
using sa::HostPipe;

#define EXPECT(x)                                                    \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s\n", __LINE__, #x);              \
            std::fflush(stdout);                                     \
            std::_Exit(1);                                           \
        }                                                            \
    } while (0)

// A kernel that is held until open() is called.
struct Gate {
    std::mutex mu;
    std::condition_variable cv;
    bool opened = false;
    void open() {
        std::lock_guard<std::mutex> lock(mu);
        opened = true;
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> lock(mu);
        cv.wait(lock, [&] { return opened; });
    }
};

constexpr size_t ROW = 1024, PITCH = ROW + 8, HOST = ROW + 5;   // bytes of a row, on the device, on the host
constexpr uint64_t ROWS = 8192, SHOTS = 4 * ROWS + 77;          // batches of 8 MiB and a ragged last one

static std::vector<uint8_t> inputs(uint32_t seed) {
    std::vector<uint8_t> v(SHOTS * HOST);
    for (size_t i = 0; i < v.size(); i++) v[i] = (uint8_t)((i * 2654435761u + seed) >> 13);
    return v;
}

// A conversion of SHOTS rows (the "kernel" adds 1 to each byte) in batches of ROWS; before(batch) runs when the batch's
// inputs are queued, held(batch) as part of its kernel.
template <class Before, class Held>
static void convert(HostPipe &pipe, hipStream_t stream, const std::vector<uint8_t> &in, std::vector<uint8_t> &out,
                    Before before, Held held) {
    pipe.begin(stream, true, 2 * ROWS * PITCH, ROWS * PITCH, ROWS * PITCH);
    for (uint64_t s0 = 0, b = 0; s0 < SHOTS; s0 += ROWS, b++) {
        const uint64_t n = std::min(ROWS, SHOTS - s0);
        size_t cap;
        uint8_t *const d_in = pipe.next_slot(&cap), *const d_out = d_in + ROWS * PITCH;
        pipe.input(d_in, PITCH, in.data() + s0 * HOST, HOST, ROW, n);
        before(b);
        stream->push([=] {
            held(b);
            for (uint64_t r = 0; r < n; r++)
                for (size_t k = 0; k < ROW; k++) d_out[r * PITCH + k] = (uint8_t)(d_in[r * PITCH + k] + 1);
            for (uint64_t r = 0; r < n; r++) std::memset(d_out + r * PITCH + ROW, 0xEE, PITCH - ROW);
        });
        std::vector<HostPipe::Part> parts;
        parts.push_back({d_out, PITCH, ROW, out.data() + s0 * HOST, HOST, -1L});
        pipe.submit(parts, n);
    }
    pipe.finish();
}

static void check_rows(const std::vector<uint8_t> &in, const std::vector<uint8_t> &out) {
    for (uint64_t r = 0; r < SHOTS; r++) {
        for (size_t k = 0; k < ROW; k++) EXPECT(out[r * HOST + k] == (uint8_t)(in[r * HOST + k] + 1));
        for (size_t k = ROW; k < HOST; k++) EXPECT(out[r * HOST + k] == 0x5A);
    }
}

static void nothing(uint64_t) {}

static void rows() {
    HostPipe pipe;
    hipStream_t stream;
    (void)hipStreamCreateWithFlags(&stream, 0);
    for (uint32_t call = 0; call < 3; call++) {
        const auto in = inputs(call);
        std::vector<uint8_t> out(SHOTS * HOST, 0x5A);
        convert(pipe, stream, in, out, nothing, [](uint64_t b) {
            if (b % 2) std::this_thread::sleep_for(std::chrono::milliseconds(3));
        });
        check_rows(in, out);
    }
    (void)hipStreamDestroy(stream);
}

// A call ends while another call's kernel is held, and its threads with it.
static void callers() {
    HostPipe a, b;
    hipStream_t sa, sb;
    (void)hipStreamCreateWithFlags(&sa, 0);
    (void)hipStreamCreateWithFlags(&sb, 0);
    Gate gate, held;
    const auto ia = inputs(1), ib = inputs(2);
    std::vector<uint8_t> oa(SHOTS * HOST, 0x5A), ob(SHOTS * HOST, 0x5A);
    std::thread other([&] {
        convert(a, sa, ia, oa, nothing, [&](uint64_t k) {
            if (k == 1) {
                held.open();
                gate.wait();
            }
        });
    });
    held.wait();
    std::this_thread::sleep_for(std::chrono::milliseconds(50));   // the other call queues all it can
    convert(b, sb, ib, ob, nothing, nothing);
    check_rows(ib, ob);
    gate.open();
    other.join();
    check_rows(ia, oa);
    (void)hipStreamDestroy(sa);
    (void)hipStreamDestroy(sb);
}

// A batch's input is copied and queued while the kernel of the batch before is held.
static void overlap() {
    HostPipe pipe;
    hipStream_t stream;
    (void)hipStreamCreateWithFlags(&stream, 0);
    Gate gate;
    const auto in = inputs(3);
    std::vector<uint8_t> out(SHOTS * HOST, 0x5A);
    convert(pipe, stream, in, out, [&](uint64_t b) { if (b == 1) gate.open(); },
            [&](uint64_t b) { if (b == 0) gate.wait(); });
    check_rows(in, out);
    (void)hipStreamDestroy(stream);
}

// An error ends a call with an exception, a call that unwinds in the middle ends too, and the pipeline goes on.
static void errors() {
    HostPipe pipe;
    hipStream_t stream;
    (void)hipStreamCreateWithFlags(&stream, 0);
    const auto in = inputs(4);
    std::vector<uint8_t> out(SHOTS * HOST, 0x5A);
    for (int k = 0; k < 2; k++) {
        bool thrown = false;
        fail_events = k == 0;
        try {
            convert(pipe, stream, in, out, [&](uint64_t b) { if (k && b == 2) throw std::runtime_error("in a call"); }, nothing);
        } catch (const std::runtime_error &) {
            thrown = true;
        }
        pipe.drain_noexcept();
        fail_events = false;
        EXPECT(thrown);
    }
    std::fill(out.begin(), out.end(), 0x5A);
    convert(pipe, stream, in, out, nothing, nothing);
    check_rows(in, out);
    (void)hipStreamDestroy(stream);
}

// Rows of bits that become bytes: every remainder, tight and strided rows, with a newline, in one batch and on threads.
static void bits() {
    HostPipe pipe;
    hipStream_t stream;
    (void)hipStreamCreateWithFlags(&stream, 0);
    for (size_t n = 1; n < 80; n++) {
        for (int form = 0; form < 4; form++) {
            const size_t row = (n + 7) / 8, pitch = row + (form & 1), stride = n + (form < 2 ? 0 : 3);
            const uint64_t rows = n % 13 == 5 ? (3 << 20) / n : 1 + n % 7;
            const long newline = form == 3 ? (long)n : -1L;
            const uint8_t base = form == 1 ? 0 : '0';
            pipe.begin(stream, false, rows * pitch, rows * pitch);
            size_t cap;
            uint8_t *const dev = pipe.next_slot(&cap);
            for (uint64_t i = 0; i < rows * pitch; i++) dev[i] = (uint8_t)((i * 2654435761u + n) >> 11);
            std::vector<uint8_t> out(rows * stride - (stride - n) + (newline >= 0 ? 1 : 0), 0x5A);
            pipe.submit({{dev, pitch, row, out.data(), stride, newline, n, base}}, rows);
            pipe.finish();
            for (uint64_t r = 0; r < rows; r++) {
                for (size_t k = 0; k < n; k++) EXPECT(out[r * stride + k] == base + ((dev[r * pitch + k / 8] >> (k % 8)) & 1));
                for (size_t k = n; k < stride && r * stride + k < out.size(); k++)
                    EXPECT(out[r * stride + k] == (k == n && newline >= 0 ? '\n' : 0x5A));
            }
        }
    }
    (void)hipStreamDestroy(stream);
}

int main(int argc, char **argv) {
    const std::map<std::string, void (*)()> all = {{"rows", rows}, {"callers", callers}, {"overlap", overlap}, {"errors", errors}, {"bits", bits}};
    if (argc != 2 || !all.count(argv[1])) return 2;
    all.at(argv[1])();
    std::printf("ok\n");
    return 0;
}
