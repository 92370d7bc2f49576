// Host bookkeeping for kernels whose workgroups wait for each other (lu!'s and
// ldlt!'s panels): such a launch ends only if all its workgroups get a place
// on their CUs while the others already there spin. Whatever else runs beside
// it ends by itself, so what can keep a workgroup out for good is other
// waiting launches alone: three lu! calls on one 32-CU stream mask, or two
// ldlt! calls, whose panels (one workgroup a CU) share the same 32 CUs, could
// each become partly resident and wait until the spin bound. A call takes its
// places here first, for as long as it runs, and where it gets none runs the
// form of the panel that does not wait (the same bits).
#pragma once
#include <cstddef>
#include <cstdint>
#include <list>
#include <mutex>
#include <vector>

namespace mfk {

// One call: at most `groups` waiting workgroups at a time, of which a CU holds
// `per_cu`, on `cus` CUs.
struct WaitingCall {
    int64_t groups, per_cu, cus;
};

// Workgroups are dealt to the eight XCDs in turn whatever room each has, so
// the first XCD's share is what has to fit its CUs (three 9-workgroup panels
// put six workgroups on the four CUs a 32-CU mask has there).
constexpr int64_t kXcds = 8;

// Whether every call's launches end: one does if an XCD's CUs hold everybody's
// share of waiting workgroups together, all of them taken to be on those CUs;
// once it has ended, its places are free for the rest. A workgroup that needs
// a whole CU counts each of the others as a whole one too.
inline bool waiting_calls_end(std::vector<WaitingCall> calls) {
    for (bool ended = true; ended && !calls.empty();) {
        ended = false;
        for (size_t i = 0; i < calls.size() && !ended; ++i) {
            double need = 0.0;
            for (const WaitingCall &c : calls) need += (double)((c.groups + kXcds - 1) / kXcds) / (calls[i].per_cu == 1 ? 1 : c.per_cu);
            if (need <= (double)(calls[i].cus / kXcds)) {
                calls.erase(calls.begin() + (std::ptrdiff_t)i);
                ended = true;
            }
        }
    }
    return calls.empty();
}

// The places of one call, given back at its end. Every call of the process on
// a device counts; another process's cannot be seen.
class WaitingPlaces {
  public:
    static constexpr int kDevices = 64;
    WaitingPlaces() = default;
    WaitingPlaces(const WaitingPlaces &) = delete;
    WaitingPlaces &operator=(const WaitingPlaces &) = delete;
    ~WaitingPlaces() {
        if (!held_) return;
        std::lock_guard<std::mutex> g(lock());
        calls(device_).erase(at_);
    }
    bool take(int device, const WaitingCall &call) {
        if (held_ || device < 0 || device >= kDevices) return false;
        std::lock_guard<std::mutex> g(lock());
        std::list<WaitingCall> &all = calls(device);
        std::vector<WaitingCall> with(all.begin(), all.end());
        with.push_back(call);
        if (!waiting_calls_end(std::move(with))) return false;
        at_ = all.insert(all.end(), call);
        device_ = device;
        return held_ = true;
    }

  private:
    static std::mutex &lock() { static std::mutex m; return m; }
    static std::list<WaitingCall> &calls(int device) { static std::list<WaitingCall> all[kDevices]; return all[device]; }
    std::list<WaitingCall>::iterator at_{};
    int device_ = 0;
    bool held_ = false;
};

}  // namespace mfk
