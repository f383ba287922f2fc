// tsu_host.h -- host helpers shared by the runtime files (internal).
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/tsuner.h"
#include "tsu_device.h"

namespace tsu {

// Run constants from the reference parameters (tsu_api.cpp).
void make_dev_params(const tsu_sim_params* p, const tsu_scheme* s, DevParams* P);
// Validates a scheme; on failure records the message and returns the code.
int validate_scheme(const tsu_scheme* s);
// Records msg as the calling thread's last error and returns code.
int set_error(int code, const std::string& msg);
// Held by every call on a handle but the waits for its stream: a call's
// launches and copies follow one another on the handle's streams with nothing
// of another thread's call between them.  A transfer reuses one buffer piece by
// piece, and the halves of an ensemble step beside its stream until they are
// joined.  Calls nest (recursive).
class HandleGuard {
public:
    HandleGuard(std::recursive_mutex& m, int device) : lock_(m)
    {
        if (hipGetDevice(&prev_) != hipSuccess) prev_ = -1;
        (void)hipSetDevice(device);
    }
    ~HandleGuard()
    {
        if (prev_ >= 0) (void)hipSetDevice(prev_);
    }

private:
    std::lock_guard<std::recursive_mutex> lock_;
    int prev_ = -1;
};
// FP64 values on their way to or from a handle's FP32 planes (device memory,
// at most 32 MB, allocated by the first transfer that is converted there and
// kept with the handle).
struct Staging {
    double* buf = nullptr;
    long long cap = 0;   // doubles
};
void free_staging(Staging* g);
// The five state planes of nv cells each, or of a download all five or one of
// them, between the host and a device state of the precision, ordered on the
// stream; a download is complete on return, an upload once the stream is.
int upload_planes(Staging* g, const double* host, void* state, int precision, long long nv, hipStream_t s);
int download_planes(Staging* g, const void* state, double* host, int precision, long long nv, int first, int planes,
                    hipStream_t s);
// Tile height for one launch of the stage kernel over grids of (npx, npy)
// cells (tsu_api.cpp).
int choose_tile_rows(const std::vector<std::pair<int, int>>& grids, bool sed, int precision, int device);

}  // namespace tsu
