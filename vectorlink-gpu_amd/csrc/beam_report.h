// The host's side of the beam loop's progress checks.  Nothing here needs the HIP runtime: what of it is used comes in as
// Gpu, which has
//   static void *pinned(size_t)  host memory that the GPU writes to, or null
//   int state()                  of the call's stream: 0 has ended, 1 still runs, below 0 an error
//   bool drain()                 waits for the stream; false: an error, what runs there may go on
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <chrono>
#include <mutex>
#include <thread>

struct BeamReport {
    int changed, sketch_rows, error, refused_at;  // as in BeamCtrl, after the checking iteration
    int check;                        // written last: iterations run up to that check
};

// Pinned host memory for the reports: one page of slots for the whole process, made with the first call that can and kept;
// a call borrows a slot.  With every slot lent out (64 calls at once) or no page to be had, a call waits for its stream at
// every check and fetches the flags instead.  A slot is given back when nothing that may write to it is left on the stream:
// a call that ends early, with launches still on their way, waits for them here (they use its workspace as well), and one
// whose stream cannot be waited for keeps the slot for good.
template <class Gpu>
class ReportSlot {
public:
    explicit ReportSlot(Gpu gpu) : gpu_(gpu) {
        std::lock_guard<std::mutex> hold(mutex_);
        if (!page_) page_ = static_cast<Slot *>(Gpu::pinned(kSlots * sizeof(Slot)));
        for (int i = 0; page_ && i < kSlots; ++i)
            if (!((lent_ >> i) & 1)) {
                lent_ |= 1ull << i;
                index_ = i;
                page_[i].report.check = page_[i].report.refused_at = 0;
                break;
            }
    }
    ~ReportSlot() {
        if (running_ && !gpu_.drain()) return;
        if (index_ < 0) return;
        std::lock_guard<std::mutex> hold(mutex_);
        lent_ &= ~(1ull << index_);
    }
    ReportSlot(const ReportSlot &) = delete;
    ReportSlot &operator=(const ReportSlot &) = delete;

    BeamReport *get() const { return index_ < 0 ? nullptr : &page_[index_].report; }
    void forget() {  // the last report, with no launch left that reports
        page_[index_].report.refused_at = 0;
        __atomic_store_n(&page_[index_].report.check, 0, __ATOMIC_RELAXED);
    }
    void launching() { running_ = true; }  // before anything of the call goes to the stream
    void drained() { running_ = false; }   // the stream has been waited for

    // Waits until the launch behind the check after iteration t has reported: 0, or below 0 (-1: the stream has ended
    // without a report, others as state()).  The stream is asked now and then, so that a launch that failed ends the wait.
    // A wait of a short call is some 60 us and looks all the time; from kLook on it lets other threads have the core
    // between two looks, and from kYield on it sleeps between them (a build's waits are 2 to 15 ms, and the next launch is
    // on the stream already).
    int wait(int t) const {
        using Clock = std::chrono::steady_clock;
        const BeamReport *r = get();
        const auto start = Clock::now();
        auto asked = start;
        for (;;) {
            for (int i = 0; i < 64; ++i) {
                if (__atomic_load_n(&r->check, __ATOMIC_ACQUIRE) == t) return 0;
                __builtin_ia32_pause();
            }
            const auto now = Clock::now();
            if (now - start < kLook) continue;
            if (now - asked > kAsk) {
                asked = now;
                const int s = gpu_.state();
                if (s < 0) return s;
                if (s == 0) return __atomic_load_n(&r->check, __ATOMIC_ACQUIRE) == t ? 0 : -1;
            }
            if (now - start < kYield) std::this_thread::yield();
            else std::this_thread::sleep_for(kSleep);
        }
    }

private:
    static constexpr int kSlots = 64;
    static constexpr std::chrono::microseconds kLook{200}, kYield{2000}, kSleep{20}, kAsk{2000};
    struct alignas(64) Slot { BeamReport report; };
    static inline std::mutex mutex_;
    static inline Slot *page_ = nullptr;
    static inline uint64_t lent_ = 0;
    Gpu gpu_;
    int index_ = -1;
    bool running_ = false;
};
