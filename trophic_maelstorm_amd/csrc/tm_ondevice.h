// tm_ondevice.h -- a device made current, and the one before it again.
#pragma once
#include <hip/hip_runtime.h>

namespace tmk {

class OnDevice {
public:
    explicit OnDevice(int device)
    {
        if (hipGetDevice(&before_) != hipSuccess) before_ = device;
        ok_ = before_ == device || hipSetDevice(device) == hipSuccess;
        if (before_ == device || !ok_) before_ = -1;
    }
    ~OnDevice() { if (before_ >= 0) (void)hipSetDevice(before_); }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;
    bool ok() const { return ok_; }

private:
    int before_ = -1;
    bool ok_ = false;
};

}  // namespace tmk
