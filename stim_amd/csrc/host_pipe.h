// Double-buffered delivery of batch outputs from device memory to the caller's host rows.
//
// A call that returns rows in host memory runs in batches. Batch i's kernels write into device slot
// i % 2; a copy engine moves the slot's rows to pinned host buffer i % 2 on a second stream, a chunk of rows at
// a time; host threads copy each chunk that has arrived from the pinned buffer to the caller's rows (pageable,
// any row stride), or expand its bits to one byte per entry (a transfer of an eighth of the bytes). So the
// host copy of a chunk runs while the next one crosses PCIe, also in a call of one batch, and while
// batch i's rows travel, batch i + 1's kernels run into the other slot. 131,071 rows of 274 bytes (36 MB, 0.63 ms
// at the link's 57 GB/s) into new numpy arrays, whose pages are touched for the first time here: 1.16 ms (1.35 in processes
// whose new arrays find no large pages), and 1.1 to 1.6 ms with one transfer and then one copy of the whole batch; 20,001 rows
// of 1,798 entries as bytes 1.3 to 1.5 instead of 1.8 ms. Inputs in host memory (m2d) take the same way in: 50,001 records of
// 181 bytes converted in 0.70 ms, where a pitched copy from pageable memory took 9 us for each row, 460 ms; 600,001 of them,
// seven batches, in 3.9 ms (5.8 where an input's helpers wait behind those of the output before it).
// Per slot, three orderings keep the buffers consistent:
//   - the DMA of batch i waits for batch i's kernels (event `produced`, a wait on the copy stream);
//   - batch i + 2's kernels wait for batch i's DMA out of the slot (the last event `arrived`, a wait on the
//     compute stream: the host does not block);
//   - batch i + 2's DMA into the pinned buffer waits for the host copy of batch i out of it (a join of
//     that batch's host threads, before the DMA is queued).
// Both streams have the default priority.
#pragma once

#include <hip/hip_runtime.h>
#include <immintrin.h>
#include <sched.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <utility>
#include <vector>

namespace sa {

// Copies `rows` rows of `width` bytes between pitched buffers. Contiguous rows (both pitches equal to
// the width) go as one linear copy: the runtime splits a pitched copy into per-row transfers, which
// costs microseconds per row.
inline hipError_t copy_rows_async(void *dst, size_t dst_pitch, const void *src, size_t src_pitch, size_t width,
                                  size_t rows, hipMemcpyKind kind, hipStream_t stream) {
    if (width == 0 || rows == 0) return hipSuccess;
    if (dst_pitch == width && src_pitch == width) return hipMemcpyAsync(dst, src, width * rows, kind, stream);
    return hipMemcpy2DAsync(dst, dst_pitch, src, src_pitch, width, rows, kind, stream);
}

// The bits of a byte as eight bytes.
constexpr std::array<uint64_t, 256> bit_bytes() {
    std::array<uint64_t, 256> t{};
    for (uint32_t b = 0; b < 256; b++)
        for (uint32_t k = 0; k < 8; k++) t[b] |= (uint64_t)((b >> k) & 1) << (8 * k);
    return t;
}
inline constexpr std::array<uint64_t, 256> BIT_BYTES = bit_bytes();

// Expands `n` bits of src to bytes base + bit.
inline void expand_bits(const uint8_t *src, uint8_t *dst, size_t n, uint8_t base) {
    const uint64_t add = 0x0101010101010101ull * base;
    size_t i = 0;
    for (; i + 8 <= n; i += 8) {
        const uint64_t v = BIT_BYTES[src[i >> 3]] + add;
        std::memcpy(dst + i, &v, 8);
    }
    if (i == n) return;
    uint64_t v = BIT_BYTES[src[i >> 3]] + add;
    for (; i < n; i++, v >>= 8) dst[i] = (uint8_t)v;
}

// Expands `rows` rows of `n` bits at src (stride `src_stride`) to bytes base + bit at dst, rows without a gap between them:
// 32 bits at a time, a row's last ones with a whole store too where the rows after it, written later, take what is too
// much. A call of 60,000 rows of 25 bits takes 111 us, 143 with eight bits at a time, and 120 where the device
// expands them and the bytes cross the link; 30,000 rows of 120 bits 80, 112 and 200.
__attribute__((target("avx2"))) inline void expand_tight_rows(const uint8_t *src, size_t src_stride, uint8_t *dst, size_t n,
                                                              uint8_t base, uint64_t rows) {
    const __m256i pick = _mm256_setr_epi8(0, 0, 0, 0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 2, 2, 2, 2, 2, 2, 2, 2, 3, 3, 3, 3, 3, 3, 3, 3);
    const __m256i bits = _mm256_set1_epi64x((long long)0x8040201008040201ull), one = _mm256_set1_epi8(1);
    const __m256i add = _mm256_set1_epi8((char)base);
    const uint8_t *const end = dst + rows * n;
    auto expand = [&](uint32_t w) __attribute__((target("avx2"), always_inline)) {
        const __m256i x = _mm256_and_si256(_mm256_shuffle_epi8(_mm256_set1_epi32((int)w), pick), bits);
        return _mm256_add_epi8(_mm256_and_si256(_mm256_cmpeq_epi8(x, bits), one), add);
    };
    for (uint64_t r = 0; r < rows; r++, src += src_stride) {
        size_t i = 0;
        for (; i + 32 <= n; i += 32, dst += 32) {
            uint32_t w;
            std::memcpy(&w, src + (i >> 3), 4);
            _mm256_storeu_si256(reinterpret_cast<__m256i *>(dst), expand(w));
        }
        const size_t left = n - i;
        if (!left) continue;
        const uint8_t *const q = src + (i >> 3);
        uint32_t w = q[0];
        if (left > 8) w |= (uint32_t)q[1] << 8;
        if (left > 16) w |= (uint32_t)q[2] << 16;
        if (left > 24) w |= (uint32_t)q[3] << 24;
        if ((size_t)(end - dst) >= 32) {
            _mm256_storeu_si256(reinterpret_cast<__m256i *>(dst), expand(w));
        } else {
            alignas(32) uint8_t last[32];
            _mm256_store_si256(reinterpret_cast<__m256i *>(last), expand(w));
            std::memcpy(dst, last, left);
        }
        dst += left;
    }
}

// Packs `n` bytes into bits (1 where the byte is not 0), padding bits 0.
inline void pack_bytes(const uint8_t *src, uint8_t *dst, size_t n) {
    size_t i = 0;
    for (; i + 16 <= n; i += 16) {
        const __m128i x = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + i));
        const uint16_t m = (uint16_t)~_mm_movemask_epi8(_mm_cmpeq_epi8(x, _mm_setzero_si128()));
        std::memcpy(dst + (i >> 3), &m, 2);
    }
    for (; i < n; i += 8) {
        uint8_t b = 0;
        for (size_t k = 0; k < 8 && i + k < n; k++) b |= (uint8_t)((src[i + k] != 0) << k);
        dst[i >> 3] = b;
    }
}

// Idle host threads of the process, lent to one pipeline at a time and given back when its calls end; a thread without
// work for a second ends. Starting threads anew for each batch took about 15 us each, as much as a 1 MB transfer.
class HostThreads {
   public:
    static HostThreads &get() {
        static HostThreads *threads = new HostThreads;   // never destroyed: a thread may still be idle at exit
        return *threads;
    }
    // Runs f on up to n threads, each its own (none waits for a thread that runs something else); returns how many.
    int run(const std::function<void()> &f, int n) {
        int got = 0;
        bool wake = false;
        std::unique_lock<std::mutex> lock(mu_);
        try {
            for (; got < n; got++) {
                if (idle_ > (int)queue_.size()) {
                    queue_.push_back(f);
                    wake = true;
                } else if (alive_ < MOST) {
                    std::thread([this, f] { serve(f); }).detach();
                    alive_++;
                } else {
                    break;
                }
            }
        } catch (const std::exception &) {
            // No further thread or no memory: those that run are enough.
        }
        lock.unlock();
        if (wake) cv_.notify_one();   // the others by each other: the caller has kernels to launch
        return got;
    }

   private:
    static constexpr int MOST = 256;   // 32 calls' worth at once; further calls copy on their own threads
    void serve(std::function<void()> f) {
        f();
        f = nullptr;
        std::unique_lock<std::mutex> lock(mu_);
        for (;;) {
            idle_++;
            cv_.wait_for(lock, std::chrono::seconds(1), [&] { return !queue_.empty(); });
            idle_--;
            if (queue_.empty()) break;
            f = std::move(queue_.front());
            queue_.pop_front();
            const bool more = !queue_.empty();
            lock.unlock();
            if (more) cv_.notify_one();
            f();
            f = nullptr;
            lock.lock();
        }
        alive_--;
    }
    std::mutex mu_;
    std::condition_variable cv_;
    std::deque<std::function<void()>> queue_;   // at most one entry per idle thread
    int alive_ = 0, idle_ = 0;
};

// The threads that copy for one pipeline during a call, and their work: up to three jobs, each a number of shares that are
// taken one after another. The shares of an output become available a piece at a time, as the transfer's chunks arrive: one
// thread at a time waits for the next chunk, of the older output first. The call's own thread takes part while it waits
// for a job. A pipeline has threads of its own, so that no call waits behind another call's kernel, and an input is
// copied by all of them while an output is still on its way.
class Crew : public std::enable_shared_from_this<Crew> {
   public:
    enum { INPUT = 0, OUTPUT = 1, JOBS = 3 };   // INPUT, and one output per slot

    // Posts job `j` (which is done) for at least `helpers` threads beside the caller: shares 0 .. total - 1, available
    // at once, or `piece` more each time arrive(number of the piece) returns, and with the last of `pieces` the rest.
    void post(int j, int helpers, int total, std::function<void(int)> share, int pieces = 0, int piece = 0,
              std::function<hipError_t(int)> arrive = nullptr) {
        const std::function<void()> member = [self = shared_from_this()] { self->serve(); };
        int need;
        {
            std::lock_guard<Spin> lock(mu_);
            Job &job = jobs_[j];
            job.share = std::move(share);
            job.arrive = std::move(arrive);
            job.total = total;
            job.pieces = pieces;
            job.piece = piece;
            job.arrived = 0;
            job.available = pieces ? 0 : total;
            job.next = 0;
            job.order = orders_++;
            job.error = hipSuccess;
            in_call_ = true;
            need = std::max(0, helpers - members_);
            members_ += need;
            version_++;
        }
        cv_.notify_all();
        if (!need) return;
        const int got = HostThreads::get().run(member, need);
        if (got < need) {
            std::lock_guard<Spin> lock(mu_);
            members_ -= need - got;
        }
    }

    // Takes part in job j until it is done.
    hipError_t finish(int j) {
        std::unique_lock<Spin> lock(mu_);
        while (active(jobs_[j])) {
            if (!step(lock, j)) wait(lock);
        }
        return std::exchange(jobs_[j].error, hipSuccess);
    }

    // Withdraws what nobody has started and waits for the rest.
    void cancel() {
        std::unique_lock<Spin> lock(mu_);
        for (Job &job : jobs_) job.total = job.available = job.next;
        version_++;
        for (Job &job : jobs_) {
            while (active(job)) wait(lock);
            job.error = hipSuccess;
        }
    }

    // The call has ended (every job is done): its threads go unless another call of the pipeline follows within LINGER, and
    // nothing waits for that.
    void end_call() {
        std::lock_guard<Spin> lock(mu_);
        in_call_ = false;
    }

   private:
    // A program's calls follow each other: giving the threads back at once and borrowing them anew costs each call 15 us.
    static constexpr std::chrono::milliseconds LINGER{2};

    // Held for a few instructions at a time, by up to nine threads that a chunk's arrival sets going at once: a mutex puts
    // most of them to sleep there (36 MB of rows in 1.30 instead of 1.16 ms).
    struct Spin {
        std::atomic_flag held = ATOMIC_FLAG_INIT;
        void lock() {
            for (int tries = 0; held.test_and_set(std::memory_order_acquire); tries++) {
                if (tries % 64 == 63) std::this_thread::yield();
                else _mm_pause();
            }
        }
        void unlock() { held.clear(std::memory_order_release); }
    };

    struct Job {
        std::function<void(int)> share;
        std::function<hipError_t(int)> arrive;
        int total = 0, pieces = 0, piece = 0, arrived = 0, available = 0, next = 0;
        int running = 0;         // threads in a share
        bool waiting = false;    // a thread waits for its next piece
        uint64_t order = 0;
        hipError_t error = hipSuccess;
    };

    static bool active(const Job &job) { return job.next < job.total || job.running || job.waiting; }

    // Takes one share, the input's first, then the older output's, or waits for one piece. The call's own thread names the
    // job that it needs next (a member: -1) and leaves newer ones alone, and the outputs while it needs an input, which
    // kernels wait for; it takes older ones (36 MB of rows in 1.30 instead of 1.17 ms if it only takes the job's own).
    bool step(std::unique_lock<Spin> &lock, int needed) {
        auto skip = [&](int j) {
            return needed >= 0 && j != needed && (needed == INPUT || jobs_[j].order > jobs_[needed].order);
        };
        int by_age[JOBS] = {INPUT, OUTPUT, OUTPUT + 1};
        if (jobs_[OUTPUT + 1].order < jobs_[OUTPUT].order) std::swap(by_age[1], by_age[2]);
        for (int j : by_age) {
            Job &job = jobs_[j];
            if (skip(j) || job.next >= job.available) continue;
            const int i = job.next++;
            job.running++;
            lock.unlock();
            job.share(i);
            lock.lock();
            job.running--;
            if (!active(job)) version_++;
            return true;
        }
        bool waiting = false;
        for (const Job &job : jobs_) waiting = waiting || job.waiting;
        for (int j : by_age) {
            Job &job = jobs_[j];
            if (waiting || skip(j) || job.available >= job.total) continue;
            job.waiting = true;
            lock.unlock();
            const hipError_t e = job.arrive(job.arrived);
            lock.lock();
            job.waiting = false;
            if (e == hipSuccess) {
                job.available = ++job.arrived < job.pieces ? std::min(job.total, job.available + job.piece) : job.total;
            } else {
                job.error = e;
                job.total = job.available = job.next;
            }
            version_++;
            return true;
        }
        return false;
    }

    // Waits until something changes (true): polling while some job is under way (a chunk, or another thread's share, is
    // about to end; waking eight sleepers for each chunk costs more), and asleep, for LINGER at most, while there is none.
    bool wait(std::unique_lock<Spin> &lock) {
        const uint64_t seen = version_;
        bool soon = false;
        for (const Job &job : jobs_) soon = soon || active(job);
        if (!soon) return cv_.wait_for(lock, LINGER, [&] { return version_ != seen; });
        lock.unlock();
        for (int polls = 0; version_ == seen; polls++) {
            if (polls < 1000) std::this_thread::yield();
            else std::this_thread::sleep_for(std::chrono::microseconds(20));   // a long kernel
        }
        lock.lock();
        return true;
    }

    void serve() {
        std::unique_lock<Spin> lock(mu_);
        while (step(lock, -1) || wait(lock) || in_call_) {}
        members_--;
    }

    // What waiting threads poll lies apart from what the others write.
    alignas(64) std::atomic<uint64_t> version_{0};
    alignas(64) Spin mu_;
    Job jobs_[JOBS];
    std::condition_variable_any cv_;
    uint64_t orders_ = 0;
    int members_ = 0;
    bool in_call_ = false;
};

class HostPipe {
   public:
    // One output of a batch: `rows` rows of `row` bytes at `dev` (stride `dev_stride`, little more than `row`; the
    // buffer holds rows * dev_stride bytes) go to `host`
    // (stride `host_stride`); when `newline_at` >= 0 each host row also gets '\n' at that byte. With `bits`, a row
    // holds that many bits, which become bytes base + bit on the host.
    struct Part {
        const uint8_t *dev;
        size_t dev_stride;
        size_t row;
        uint8_t *host;
        size_t host_stride;
        long newline_at;
        size_t bits = 0;
        uint8_t base = 0;
    };

    HostPipe() = default;
    HostPipe(const HostPipe &) = delete;
    HostPipe &operator=(const HostPipe &) = delete;
    ~HostPipe() {
        drain_noexcept();
        for (int s = 0; s < 2; s++) {
            if (dev_[s]) (void)hipFree(dev_[s]);
            if (pin_[s]) (void)hipHostFree(pin_[s]);
            if (pin_in_[s]) (void)hipHostFree(pin_in_[s]);
            if (produced_[s]) (void)hipEventDestroy(produced_[s]);
            if (consumed_[s]) (void)hipEventDestroy(consumed_[s]);
            for (hipEvent_t e : arrived_[s]) {
                if (e) (void)hipEventDestroy(e);
            }
        }
        if (copy_) (void)hipStreamDestroy(copy_);
    }

    // Host threads per batch copy: the CPUs this process may run on, at most 8.
    static int host_threads() {
        cpu_set_t set;
        int n = 1;
        if (sched_getaffinity(0, sizeof(set), &set) == 0) n = CPU_COUNT(&set);
        return std::max(1, std::min(n, 8));
    }

    // Prepares a call on `compute` of one batch or several: the device slots hold at least `dev_bytes`, the pinned
    // buffers at least `host_bytes`, the pinned input buffers `in_bytes` (the first of each for one batch). Nothing
    // of an earlier call is in flight (finish() or drain ended it).
    void begin(hipStream_t compute, bool several, size_t dev_bytes, size_t host_bytes, size_t in_bytes = 0) {
        compute_ = compute;
        several_ = several;
        chk(hipGetDevice(&device_), "device");
        if (!copy_) {
            chk(hipStreamCreateWithFlags(&copy_, hipStreamNonBlocking), "copy stream");
            for (int s = 0; s < 2; s++) {
                chk(hipEventCreateWithFlags(&produced_[s], hipEventDisableTiming), "event");
                chk(hipEventCreateWithFlags(&consumed_[s], hipEventDisableTiming), "event");
                for (hipEvent_t &e : arrived_[s]) chk(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
            }
        }
        for (int s = 0; s < (several ? 2 : 1); s++) {
            if (dev_cap_[s] < dev_bytes) {
                if (dev_[s]) chk(hipFree(dev_[s]), "hipFree");
                dev_[s] = nullptr;
                dev_cap_[s] = 0;
                chk(hipMalloc(reinterpret_cast<void **>(&dev_[s]), dev_bytes), "hipMalloc (host pipeline slot)");
                dev_cap_[s] = dev_bytes;
            }
            pinned(pin_[s], pin_cap_[s], host_bytes);
            pinned(pin_in_[s], pin_in_cap_[s], in_bytes);
        }
        for (int s = 0; s < 2; s++) used_[s] = in_used_[s] = false;
        in_at_ = 0;
        batch_ = 0;
        pending_ = -1;
        nthreads_ = host_threads();
    }

    // Device slot of the next batch, with its capacity. The compute stream first waits until the DMA
    // of the batch that last used the slot has read it.
    uint8_t *next_slot(size_t *cap) {
        const int s = batch_ & 1;
        if (used_[s]) chk(hipStreamWaitEvent(compute_, arrived_[s][batches_[s].chunks - 1], 0), "wait for slot");
        *cap = dev_cap_[s];
        return dev_[s];
    }

    // Queues the copy of `rows` host rows into device rows of `pitch` bytes on the compute stream, through the batch's
    // pinned input buffer: rows of `row` bytes, or, with `bytes`, of that many bytes to pack into bits (row = packed
    // bytes). Inputs of a batch are queued before its kernels, each at its own offset of the buffer.
    void input(uint8_t *dev, size_t pitch, const uint8_t *host, size_t host_stride, size_t row, uint64_t rows,
               size_t bytes = 0) {
        const int s = batch_ & 1;
        if (!row || !rows) return;
        if (in_used_[s] && in_at_ == 0) chk(hipEventSynchronize(consumed_[s]), "input buffer");
        if (in_at_ + pitch * rows > pin_in_cap_[s]) throw std::logic_error("host pipeline input exceeds its pinned buffer");
        uint8_t *const pin = pin_in_[s] + in_at_;
        in_at_ += pitch * rows;
        auto copy = [=](uint64_t r0, uint64_t r1) {
            if (bytes) {
                for (uint64_t r = r0; r < r1; r++) pack_bytes(host + r * host_stride, pin + r * pitch, bytes);
            } else if (host_stride == row && pitch == row) {
                std::memcpy(pin + r0 * row, host + r0 * row, (r1 - r0) * row);
            } else {
                for (uint64_t r = r0; r < r1; r++) std::memcpy(pin + r * pitch, host + r * host_stride, row);
            }
        };
        const size_t total = std::max(row, bytes) * rows;
        const int k = (int)std::max<uint64_t>(1, std::min<uint64_t>(nthreads_, total >> 20));
        if (k > 1) {
            crew_->post(Crew::INPUT, k - 1, k, [&, k](int t) { copy(rows * t / k, rows * (t + 1) / k); });
            (void)crew_->finish(Crew::INPUT);
        } else {
            copy(0, rows);
        }
        chk(hipMemcpyAsync(dev, pin, pitch * rows, hipMemcpyHostToDevice, compute_), "copy from pinned buffer");
        if (several_) {
            chk(hipEventRecord(consumed_[s], compute_), "record");
            in_used_[s] = true;
        } else {
            in_flight_ = true;
        }
    }

    // Queues the DMA of the batch whose kernels were just queued (a chunk of rows after another), and has
    // the batch's host threads take the chunks as they arrive.
    void submit(const std::vector<Part> &parts, uint64_t rows) {
        const int s = batch_ & 1;
        size_t need = 0, host_bytes = 0;
        for (const Part &p : parts) {
            need += p.dev_stride * rows;
            host_bytes += (p.bits ? p.bits : p.row) * rows;
        }
        if (need > pin_cap_[s]) throw std::logic_error("host pipeline batch exceeds its pinned buffer");
        join(s);
        Batch &b = batches_[s];
        b.parts.clear();
        b.rows = rows;
        b.chunks = (int)std::max<uint64_t>(1, std::min<uint64_t>({(uint64_t)MAX_CHUNKS, host_bytes / CHUNK_BYTES, rows}));
        // Threads only where each gets at least 1 MiB; a smaller batch is copied by the caller, at the next
        // submit() or finish().
        b.nthreads = (int)std::min<uint64_t>(nthreads_, host_bytes >> 20);
        b.shares = (int)std::max<uint64_t>(1, std::min<uint64_t>(b.nthreads, host_bytes / b.chunks / SHARE_BYTES));
        // A call of one small batch has nothing to overlap: its transfer follows the kernels on their own stream, without
        // events (1613 shots of 121 results converted, packed: 52 us with a second stream, 33 without).
        b.direct = !several_ && b.chunks == 1 && b.nthreads <= 1;
        const hipStream_t out = b.direct ? compute_ : copy_;
        if (b.direct) {
            in_flight_ = true;
        } else {
            chk(hipEventRecord(produced_[s], compute_), "record");
            chk(hipStreamWaitEvent(copy_, produced_[s], 0), "wait for kernels");
        }
        size_t off = 0;
        for (const Part &p : parts) {
            Part q = p;
            q.dev = pin_[s] + off;
            b.parts.push_back(q);
            off += p.dev_stride * rows;
        }
        for (int c = 0; c < b.chunks; c++) {
            const uint64_t r0 = rows * c / b.chunks, r1 = rows * (c + 1) / b.chunks;
            for (size_t i = 0; i < parts.size(); i++) {
                const Part &p = parts[i];
                // Whole device rows, padding included: the runtime splits a pitched copy into per-row transfers.
                if (p.row && r1 > r0)
                    chk(hipMemcpyAsync(const_cast<uint8_t *>(b.parts[i].dev) + r0 * p.dev_stride, p.dev + r0 * p.dev_stride,
                                       (r1 - r0) * p.dev_stride, hipMemcpyDeviceToHost, out),
                        "copy to pinned buffer");
            }
            if (!b.direct) chk(hipEventRecord(arrived_[s][c], copy_), "record");
        }
        used_[s] = !b.direct;
        if (pending_ >= 0) copy_small(pending_);
        pending_ = -1;
        if (b.nthreads > 1) start(s);
        else pending_ = s;
        in_at_ = 0;
        batch_++;
    }

    // Delivers the last batch and waits for every host copy.
    void finish() {
        if (pending_ >= 0) copy_small(pending_);
        pending_ = -1;
        join(0);
        join(1);
        if (in_flight_) chk(hipStreamSynchronize(compute_), "copies on the compute stream");
        in_flight_ = false;
        crew_->end_call();
    }

    // Ends whatever is in flight without reporting errors (used when a call is unwinding).
    void drain_noexcept() {
        crew_->cancel();
        crew_->end_call();
        for (int s = 0; s < 2; s++) {
            if (in_used_[s]) (void)hipEventSynchronize(consumed_[s]);
        }
        if (copy_) (void)hipStreamSynchronize(copy_);
        if (in_flight_) (void)hipStreamSynchronize(compute_);
        in_flight_ = false;
        pending_ = -1;
        in_at_ = 0;
    }

   private:
    static constexpr int MAX_CHUNKS = 16;
    static constexpr size_t CHUNK_BYTES = (size_t)2 << 20;   // host bytes per chunk, at least
    static constexpr size_t SHARE_BYTES = (size_t)1 << 20;   // of a chunk, at least (start())

    struct Batch {
        std::vector<Part> parts;   // dev = pinned source rows, at the device rows' stride
        uint64_t rows = 0;
        int chunks = 1, nthreads = 1;
        int shares = 1;                // of a chunk before the last
        bool direct = false;           // transferred on the compute stream
    };

    static void chk(hipError_t e, const char *what) {
        if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
    }

    static void pinned(uint8_t *&p, size_t &cap, size_t bytes) {
        if (cap >= bytes) return;
        if (p) chk(hipHostFree(p), "hipHostFree");
        p = nullptr;
        cap = 0;
        chk(hipHostMalloc(reinterpret_cast<void **>(&p), bytes, hipHostMallocDefault), "hipHostMalloc (host pipeline buffer)");
        cap = bytes;
    }

    static void copy_rows(const Batch &b, uint64_t r0, uint64_t r1) {
        for (const Part &p : b.parts) {
            if (!p.row && p.newline_at < 0) continue;
            const uint8_t *src = p.dev + r0 * p.dev_stride;
            uint8_t *dst = p.host + r0 * p.host_stride;
            if (p.host_stride == p.row && p.dev_stride == p.row && p.newline_at < 0 && !p.bits) {
                std::memcpy(dst, src, (r1 - r0) * p.row);
                continue;
            }
            static const bool avx2 = __builtin_cpu_supports("avx2");
            if (p.bits && p.host_stride == p.bits && p.newline_at < 0 && avx2) {
                expand_tight_rows(src, p.dev_stride, dst, p.bits, p.base, r1 - r0);
                continue;
            }
            for (uint64_t r = r0; r < r1; r++, src += p.dev_stride, dst += p.host_stride) {
                if (p.bits) expand_bits(src, dst, p.bits, p.base);
                else std::memcpy(dst, src, p.row);
                if (p.newline_at >= 0) dst[p.newline_at] = '\n';
            }
        }
    }

    // A batch too small for threads: waits for its last chunk and copies it here.
    void copy_small(int s) {
        Batch &b = batches_[s];
        if (b.direct) {
            chk(hipStreamSynchronize(compute_), "copy to pinned buffer");
            in_flight_ = false;
        } else {
            chk(hipEventSynchronize(arrived_[s][b.chunks - 1]), "copy to pinned buffer");
        }
        copy_rows(b, 0, b.rows);
    }

    // Has the crew take the batch's shares as the chunks arrive. A share is 1 MiB or more, since threads that touch new
    // pages close by wait for each other (39 MB into new arrays: 2.1 ms with eight shares to each chunk of 2 MiB, 1.45 with
    // two); the last chunk, which nothing follows, is shared by all.
    void start(int s) {
        Batch &b = batches_[s];
        const int early = (b.chunks - 1) * b.shares;
        auto share = [&b, early](int i) {
            const int c = i < early ? i / b.shares : b.chunks - 1;
            const uint64_t of = i < early ? b.shares : b.nthreads, part = i < early ? i % b.shares : i - early;
            const uint64_t a = b.rows * c / b.chunks, n = b.rows * (c + 1) / b.chunks - a;
            copy_rows(b, a + n * part / of, a + n * (part + 1) / of);
        };
        auto arrive = [this, s](int c) {
            const hipError_t e = hipSetDevice(device_);
            return e == hipSuccess ? hipEventSynchronize(arrived_[s][c]) : e;
        };
        crew_->post(Crew::OUTPUT + s, b.nthreads, early + b.nthreads, share, b.chunks, b.shares, arrive);
    }

    void join(int s) { chk(crew_->finish(Crew::OUTPUT + s), "copy to pinned buffer"); }

    hipStream_t compute_ = nullptr, copy_ = nullptr;
    int device_ = 0;
    hipEvent_t produced_[2] = {nullptr, nullptr}, consumed_[2] = {nullptr, nullptr};
    hipEvent_t arrived_[2][MAX_CHUNKS] = {};
    uint8_t *dev_[2] = {nullptr, nullptr};
    uint8_t *pin_[2] = {nullptr, nullptr};
    uint8_t *pin_in_[2] = {nullptr, nullptr};
    size_t dev_cap_[2] = {0, 0}, pin_cap_[2] = {0, 0}, pin_in_cap_[2] = {0, 0};
    bool used_[2] = {false, false}, in_used_[2] = {false, false};
    size_t in_at_ = 0;   // bytes of the next batch's pinned input buffer in use
    Batch batches_[2];
    std::shared_ptr<Crew> crew_ = std::make_shared<Crew>();   // its threads may leave after the pipeline is gone
    uint64_t batch_ = 0;
    int pending_ = -1;
    int nthreads_ = 1;
    bool several_ = false;
    bool in_flight_ = false;   // copies of this call on the compute stream that no event marks
};

}  // namespace sa
