// Internal host-side definitions shared by the C ABI translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>
#include <set>

struct mz_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::set<void*> allocs;  // device buffers owned by the context, freed at mz_ctx_free
    // scratch kept between calls of the synchronous entry points (MzScratch), freed at mz_ctx_free
    std::mutex scratch_mu;
    void *scratch_dev = nullptr, *scratch_pin = nullptr;
    size_t scratch_dev_bytes = 0, scratch_pin_bytes = 0;
};

// Device and pinned host scratch of one synchronous call (the stream is idle again when it returns): the context's own,
// grown as needed, or buffers of the call's own where a size is beyond what the context keeps, or where another
// thread is using the context's.
class MzScratch {
public:
    static constexpr size_t KEEP_DEV = (size_t)192 << 20, KEEP_PIN = (size_t)4 << 20;  // most a context keeps
    MzScratch(mz_ctx* c, size_t dev_bytes, size_t pin_bytes);
    ~MzScratch();
    MzScratch(const MzScratch&) = delete;
    MzScratch& operator=(const MzScratch&) = delete;
    int status() const { return status_; }  // MZ_OK or the failed allocation's code
    char* dev = nullptr;
    char* pin = nullptr;

private:
    mz_ctx* c_;
    int status_ = 0;
    bool own_dev_ = false, own_pin_ = false;  // freed at the call's end
    std::unique_lock<std::mutex> lock_;
};

struct mz_graph {
    hipGraph_t graph;
    hipGraphExec_t exec;
};

// set the thread-local error message and return `code`
int mz_fail(int code, const char* fmt, ...);
// MZ_OK, or MZ_ERR_HIP with the runtime's message
int mz_hip(hipError_t e, const char* what);
// zero-filled device allocation owned by the context
int mz_ctx_alloc(mz_ctx* c, size_t bytes, void** p);

// IEEE binary16 conversions (round to nearest even), host side
uint16_t mz_f2h_host(float x);
float mz_h2f_host(uint16_t h);
