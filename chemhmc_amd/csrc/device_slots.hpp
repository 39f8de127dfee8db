// What a process keeps once per GPU for callers that take turns there: a mutex and a value of its own for every
// device, so that callers on different devices never wait for each other.
#pragma once
#include <mutex>

namespace chmc {

template <typename T, int MaxDevices>
class DeviceSlots {
public:
    struct Slot {
        std::mutex mu;
        T value{};
    };
    // the slot of a device, nullptr if there is none
    Slot* of(int device) { return device >= 0 && device < MaxDevices ? &slots_[device] : nullptr; }

private:
    Slot slots_[MaxDevices];
};

}  // namespace chmc
