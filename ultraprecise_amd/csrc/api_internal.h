// api_internal.h -- helpers shared by the C ABI translation units
// (updec_api.hip, vm.hip, segsum.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/updec.h"
#include "planner.h"

namespace updec {

// the calling thread's current device is `dev` while this lives
class OnDevice {
  public:
    explicit OnDevice(int dev)
    {
        if (hipGetDevice(&was_) != hipSuccess || was_ == dev) was_ = -1;
        else (void)hipSetDevice(dev);
    }
    ~OnDevice()
    {
        if (was_ >= 0) (void)hipSetDevice(was_);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;

  private:
    int was_ = -1;
};

// while this lives the calling thread may allocate although a stream is being
// captured (an allocation is no part of what a capture records)
class AllocWhileCapturing {
  public:
    AllocWhileCapturing() { exchange(); }
    ~AllocWhileCapturing() { exchange(); }
    AllocWhileCapturing(const AllocWhileCapturing&) = delete;
    AllocWhileCapturing& operator=(const AllocWhileCapturing&) = delete;

  private:
    void exchange()
    {
        if (ok_) ok_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess;
    }
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool ok_ = true;
};

// record the calling thread's error message, return `code`
int api_fail(int code, const std::string& msg);
// compute units of the current device (cached)
int api_device_cus();
// column descriptors -> planner types (and names)
std::vector<ColumnType> api_types(const updec_column_desc* cols, int n, std::vector<std::string>* names);
// parse -> AlignOptimize -> plan; mode AUTO picks faithful inside the envelope
bool api_make_plan(const std::string& text, const std::vector<std::string>& names,
                   const std::vector<ColumnType>& types, int mode, Plan* out, std::string* err);
// device address of the segmented SUM's fixed scratch on the current device
// (segsum.hip), looked up once per device
int segsum_scratch_setup();

}  // namespace updec
