// Threads that move bytes between the caller's arrays and the host-pointer path's staging slots (host_path.hip).  Host code only.
#pragma once
#include <sched.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <immintrin.h>
#include <mutex>
#include <stddef.h>
#include <system_error>
#include <thread>

namespace acc950 {

// Stores that go past the caches: for bytes that this program does not read again soon -- a staging slot, which the device fetches, or a
// result larger than the caches.  An ordinary store would first fetch the line it is about to overwrite, half as much memory traffic again.
__attribute__((target("avx2"))) inline void stream_copy(char* dst, const char* src, size_t bytes)
{
    const size_t head = (32 - ((size_t)dst & 31)) & 31;
    if (bytes < 4096 + head) { std::memcpy(dst, src, bytes); return; }
    std::memcpy(dst, src, head);
    dst += head; src += head; bytes -= head;
    for (; bytes >= 128; bytes -= 128, dst += 128, src += 128) {
        const __m256i a = _mm256_loadu_si256((const __m256i*)src), b = _mm256_loadu_si256((const __m256i*)(src + 32)),
                      c = _mm256_loadu_si256((const __m256i*)(src + 64)), d = _mm256_loadu_si256((const __m256i*)(src + 96));
        _mm256_stream_si256((__m256i*)dst, a);
        _mm256_stream_si256((__m256i*)(dst + 32), b);
        _mm256_stream_si256((__m256i*)(dst + 64), c);
        _mm256_stream_si256((__m256i*)(dst + 96), d);
    }
    std::memcpy(dst, src, bytes);
    _mm_sfence();
}
inline void copy_bytes(char* dst, const char* src, size_t bytes, bool past_caches)
{
    static const bool wide = __builtin_cpu_supports("avx2");
    if (past_caches && wide) stream_copy(dst, src, bytes);
    else std::memcpy(dst, src, bytes);
}

// A fixed set of threads, started at the first large copy.  One copy at a time is dealt out (callers take turns); the calling thread takes
// a share itself.  While a large call is under way (Busy) the threads look for the next copy without sleeping for a while after each
// one: a call is a dozen or two copies of 1 to 8 MB, 15 to 100 us each, and waking six sleeping threads takes half as long again.  A pause
// longer than that -- a long kernel, the end of the call -- finds them asleep, and the next copy wakes them.
// As many of them take part as this process has cores beside the caller's (its affinity mask, looked at once per large call), and on fewer than four cores they
// always sleep: a waiting thread would take the time of one that copies, or of the runtime's (six threads awake whatever the cores, us on 16 / 4 / 2 / 1 cores: 4096x4096x512
// fp16 to fp32 1683 / 1707 / 7433 / 26185; threads that always sleep 1805 / 1887 / 2445 / 3295; this way 1667 / 1685 / 1705 / 2148).
// The threads live until the process ends.
class CopyPool {
public:
    static constexpr int kThreads = 6;
    static constexpr size_t kParallelFrom = (size_t)256 << 10; // smaller copies are the calling thread's alone
    static constexpr int kAwakeUs = 150;  // how long a thread looks for the next copy before it sleeps
    static constexpr int kPauses = 1000;  // how often a caller looks whether the threads are done before it yields (15 to 50 ns each)

    class Busy {
    public:
        Busy(CopyPool& pool, bool large) : pool_(large ? &pool : nullptr)
        {
            if (!pool_) return;
            pool_->look_at_cores();
            ++pool_->busy_;
            ++pool_->alarm_;
            pool_->wake(); // (up by the time the first piece is to be copied)
        }
        ~Busy() { if (pool_) --pool_->busy_; }
        Busy(const Busy&) = delete;
        Busy& operator=(const Busy&) = delete;

    private:
        CopyPool* pool_;
    };

    void copy(char* dst, const char* src, size_t bytes, bool past_caches)
    {
        if (bytes < kParallelFrom) { std::memcpy(dst, src, bytes); return; }
        std::lock_guard<std::mutex> turn(turn_);
        const int helpers = start_workers();
        if (!helpers) { copy_bytes(dst, src, bytes, past_caches); return; }
        Job job;
        job.dst = dst; job.src = src; job.bytes = bytes; job.past_caches = past_caches;
        job.per = ((bytes + helpers) / (helpers + 1) + 4095) & ~(size_t)4095;
        job.left = (bytes + job.per - 1) / job.per;
        job_ = &job;
        ++generation_;
        wake();
        work(job); // the caller's share
        await([&] { return job.left == 0; });
        // (a thread that is still looking at the job counts itself in before it does: none is once the count is zero)
        job_ = nullptr;
        await([&] { return inside_ == 0; });
    }
    int started() const { return started_; }

private:
    struct Job {
        char* dst;
        const char* src;
        size_t bytes, per;
        bool past_caches;
        std::atomic<size_t> next{0}, left{0};
    };
    void wake()
    {
        if (!asleep_) return; // (a thread counts itself asleep before it looks for a reason not to for the last time: one of the two sees the other)
        { std::lock_guard<std::mutex> lock(m_); } // (who has looked is asleep by now; told while the lock is held, they wake up to wait for it, 5 us of every copy)
        wake_.notify_all();
    }
    // waits for what another thread is about to do: a moment awake, then giving its core to whom it may belong
    template <typename Done>
    static void await(Done&& done)
    {
        for (int n = 0; n < kPauses; ++n) {
            if (done()) return;
            __builtin_ia32_pause();
        }
        while (!done()) std::this_thread::yield();
    }
    void look_at_cores()
    {
        cpu_set_t set;
        int cores = 1;
        if (sched_getaffinity(0, sizeof set, &set) == 0) cores = CPU_COUNT(&set);
        else if (const unsigned n = std::thread::hardware_concurrency()) cores = (int)n; // (more cores than the mask has room for)
        allowed_ = cores - 1 < kThreads ? cores - 1 : kThreads;
        awake_ = cores >= 4;
    }
    // starts the threads that are allowed and not there yet; returns how many take part
    int start_workers()
    {
        if (allowed_ < 0) look_at_cores();
        while (started_ < allowed_) {
            try {
                std::thread([this, i = started_.load()] { loop(i); }).detach();
            } catch (const std::system_error&) { // (the process has no more threads to give: those that are there do)
                break;
            }
            ++started_;
        }
        return started_ < allowed_ ? started_.load() : allowed_.load();
    }
    // takes pieces of the job until none is left
    static void work(Job& job)
    {
        for (;;) {
            const size_t off = job.next++ * job.per;
            if (off >= job.bytes) return;
            copy_bytes(job.dst + off, job.src + off, job.bytes - off < job.per ? job.bytes - off : job.per, job.past_caches);
            --job.left;
        }
    }
    void loop(int index)
    {
        unsigned long long seen = 0;
        unsigned heard = 0;
        auto last = std::chrono::steady_clock::now();
        for (unsigned looks = 0;; ++looks) {
            if (generation_ != seen) {
                seen = generation_;
                if (index < allowed_) {
                    ++inside_;
                    if (Job* job = job_) work(*job);
                    --inside_;
                }
                last = std::chrono::steady_clock::now();
                continue;
            }
            if (busy_ && awake_ && index < allowed_ && (looks % 32 || std::chrono::steady_clock::now() - last < std::chrono::microseconds(kAwakeUs))) {
                __builtin_ia32_pause();
                continue;
            }
            std::unique_lock<std::mutex> lock(m_);
            ++asleep_;
            wake_.wait(lock, [&] { return generation_ != seen || (alarm_ != heard && index < allowed_); });
            --asleep_;
            heard = alarm_;
            last = std::chrono::steady_clock::now();
        }
    }
    std::mutex turn_, m_;
    std::condition_variable wake_;
    std::atomic<int> started_{0}, allowed_{-1};
    std::atomic<Job*> job_{nullptr};
    std::atomic<unsigned long long> generation_{0};
    std::atomic<int> inside_{0}, busy_{0}, asleep_{0};
    std::atomic<unsigned> alarm_{0};
    std::atomic<bool> awake_{true};
};

} // namespace acc950
