// stage.h -- pinned staging for the calls that move arrays between the host
// and the device.
//
// What bounded them: a copy to ordinary host memory goes through the runtime
// at 10-20 GB/s and 20-60 us a call (128 KB: 62 us; 7.4 MB: 422 us), where
// pinned memory takes 10 and 141 us.  So arrays pass through slots of a
// pinned buffer, the host's copy of one slot running beside the device's
// transfer of the next.  Slots of 512 KB: 17 us of transfer each, about the
// host's time for the same bytes.  The state of 266240 beads: 935 -> 277 us,
// of 312: 38 -> 15; features and labels of 20336 beads 715 -> 490.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace mte {

constexpr size_t STAGE_SLOT = 512 * 1024;
constexpr int STAGE_SLOTS = 8;
constexpr size_t STAGE_IDLE_MAX = 4;   // buffers kept per device while engines exist

struct StageBuf {
    char *mem = nullptr, *dev = nullptr;   // the same bytes as the host and as kernels address them
    hipEvent_t ev[STAGE_SLOTS] = {};
};

// The process's buffers, per device.  A call holds one buffer from its first
// transfer until it returns, so engines on several threads use different
// ones; idle ones are kept for the next call (STAGE_IDLE_MAX per device) and
// freed with the device's last engine.
class StagePool {
  public:
    static StagePool &get() {
        static StagePool *p = new StagePool();   // not destroyed: engines may outlive static destructors
        return *p;
    }
    void add_user(int device) {
        std::lock_guard<std::mutex> lock(mu_);
        dev_[device].users++;
    }
    void drop_user(int device) {   // with the device current
        std::vector<StageBuf> gone;
        {
            std::lock_guard<std::mutex> lock(mu_);
            Dev &d = dev_[device];
            if (--d.users == 0) gone.swap(d.idle);
        }
        for (StageBuf &b : gone) destroy(b);
    }
    // A buffer of the current device `device`; mem null when there is no
    // pinned memory left.
    StageBuf take(int device) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            std::vector<StageBuf> &idle = dev_[device].idle;
            if (!idle.empty()) {
                const StageBuf b = idle.back();
                idle.pop_back();
                return b;
            }
        }
        StageBuf b;
        bool ok = hipHostMalloc((void **)&b.mem, STAGE_SLOT * STAGE_SLOTS, hipHostMallocMapped | hipHostMallocCoherent) ==
                      hipSuccess &&
                  hipHostGetDevicePointer((void **)&b.dev, b.mem, 0) == hipSuccess;
        for (int i = 0; i < STAGE_SLOTS && ok; i++)
            ok = hipEventCreateWithFlags(&b.ev[i], hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            destroy(b);
            (void)hipGetLastError();
            b = StageBuf{};
        }
        return b;
    }
    void give(int device, StageBuf b) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            Dev &d = dev_[device];
            if (d.users > 0 && d.idle.size() < STAGE_IDLE_MAX) {
                d.idle.push_back(b);
                return;
            }
        }
        destroy(b);
    }

  private:
    struct Dev {
        int users = 0;
        std::vector<StageBuf> idle;
    };
    static void destroy(StageBuf &b) {
        for (hipEvent_t e : b.ev)
            if (e) (void)hipEventDestroy(e);
        if (b.mem) (void)hipHostFree(b.mem);
    }
    std::mutex mu_;
    std::map<int, Dev> dev_;
};

// One call's transfers on `stream`, in order.  Host memory given to to_host
// is written by finish() at the latest, host memory given to to_device has
// been read by then.  finish() waits for the stream.  Without
// a pinned buffer the copies are made directly.
class Stage {
  public:
    Stage(int device, hipStream_t stream) : device_(device), stream_(stream), buf_(StagePool::get().take(device)) {}
    ~Stage() {
        if (!buf_.mem) return;
        if (open_) (void)hipStreamSynchronize(stream_);   // an error path: transfers may still use the buffer
        StagePool::get().give(device_, buf_);
    }
    Stage(const Stage &) = delete;
    Stage &operator=(const Stage &) = delete;

    // Only what fits half a slot is staged (128 KB: 14 us, directly 58): the
    // runtime's own uploads reach 28 GB/s from 512 KB on, more than the host's
    // copies beside the launches do (7.7 MB: 270 us directly, 420 staged).
    hipError_t to_device(void *dst, const void *src, size_t n) {
        if (!buf_.mem || n > STAGE_SLOT / 2) return hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, stream_);
        char *p;
        hipError_t s = slot(&p);
        if (s != hipSuccess) return s;
        std::memcpy(p, src, n);
        if ((s = hipMemcpyAsync(dst, p, n, hipMemcpyHostToDevice, stream_)) != hipSuccess) return s;
        return sent(nullptr, 0, false);
    }
    hipError_t to_host(void *dst, const void *src, size_t n) {
        if (!buf_.mem) return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, stream_);
        for (size_t o = 0; o < n; o += STAGE_SLOT) {
            const size_t m = std::min(STAGE_SLOT, n - o);
            char *p;
            hipError_t s = slot(&p);
            if (s != hipSuccess) return s;
            if ((s = hipMemcpyAsync(p, (const char *)src + o, m, hipMemcpyDeviceToHost, stream_)) != hipSuccess) return s;
            if ((s = sent((char *)dst + o, m, n > STAGE_SLOT)) != hipSuccess) return s;
        }
        return hipSuccess;
    }
    // A kernel's output: `launch(p, o, m)` enqueues the kernel that writes
    // bytes [o, o + m) of the array to p, a slot's device address.  `step` is the
    // largest m, at most STAGE_SLOT.
    template <class Launch>
    hipError_t produce(void *dst, size_t n, size_t step, const Launch &launch) {
        for (size_t o = 0; o < n; o += step) {
            const size_t m = std::min(step, n - o);
            char *p;
            hipError_t s = slot(&p);
            if (s != hipSuccess) return s;
            if ((s = launch(buf_.dev + (p - buf_.mem), o, m)) != hipSuccess) return s;
            if ((s = sent((char *)dst + o, m, n > step)) != hipSuccess) return s;
        }
        return hipSuccess;
    }
    bool pinned() const { return buf_.mem != nullptr; }
    hipError_t finish() {
        hipError_t s = hipSuccess;
        for (int i = 0; i < STAGE_SLOTS && s == hipSuccess; i++) s = settle((next_ + i) % STAGE_SLOTS);
        if (s == hipSuccess && open_) s = hipStreamSynchronize(stream_);
        if (s == hipSuccess) open_ = false;
        return s;
    }

  private:
    struct Slot {
        void *dst = nullptr;   // where its bytes go once transferred (null: to the device)
        size_t n = 0;
        bool busy = false, marked = false;
    };
    // Waits until the slot's transfer is over and empties it.
    hipError_t settle(int i) {
        Slot &t = slot_[i];
        if (!t.busy) return hipSuccess;
        const hipError_t s = t.marked ? hipEventSynchronize(buf_.ev[i]) : hipStreamSynchronize(stream_);
        if (s != hipSuccess) return s;
        if (!t.marked) open_ = false;
        if (t.dst) std::memcpy(t.dst, buf_.mem + i * STAGE_SLOT, t.n);
        t = Slot{};
        return hipSuccess;
    }
    hipError_t slot(char **p) {
        *p = buf_.mem + next_ * STAGE_SLOT;
        return settle(next_);
    }
    hipError_t sent(void *dst, size_t n, bool mark) {
        slot_[next_].dst = dst;
        slot_[next_].n = n;
        slot_[next_].busy = true;
        slot_[next_].marked = mark;
        open_ = true;
        const int i = next_;
        next_ = (next_ + 1) % STAGE_SLOTS;
        return mark ? hipEventRecord(buf_.ev[i], stream_) : hipSuccess;
    }
    int device_;
    hipStream_t stream_;
    StageBuf buf_;
    Slot slot_[STAGE_SLOTS];
    int next_ = 0;
    bool open_ = true;   // work of this call may still be running
};

}  // namespace mte
