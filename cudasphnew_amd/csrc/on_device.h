// on_device.h -- a handle's device made current for the length of a scope.
#pragma once

#include <hip/hip_runtime.h>

namespace sph {

// Memory and events belong to the device that is current when they are
// created, a kernel runs on its stream's.  What a handle creates after its
// creation is created under this: the caller may be a thread whose current
// device is another one (0 in a new thread).  Costs one read of the current
// device where they agree.
class OnDevice {
    int back = -1;

  public:
    explicit OnDevice(int device) {
        int now = device;
        if (hipGetDevice(&now) == hipSuccess && now != device && hipSetDevice(device) == hipSuccess) back = now;
    }
    ~OnDevice() {
        if (back >= 0) (void)hipSetDevice(back);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;
};

}  // namespace sph
