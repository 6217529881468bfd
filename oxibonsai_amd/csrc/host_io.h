// host_io.h — moving the host buffers of a call to and from the device (host_io.hip).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace oxb {

// The host buffers of one call: begin, upload for every input, the call's launches, download for every output, and finish,
// after which the outputs are there.  All of it runs under the library's lock and enqueues on the stream in use.
//
// Until finish returns the device may read the inputs and write the outputs where they lie (buffers of pinned_alloc).  A
// call that fails on the way leaves that to the destructor, which waits for the stream: nothing touches the caller's
// buffers or the staging memory once the entry point has returned.
class IoCall {
public:
    IoCall() = default;
    IoCall(const IoCall&) = delete;
    IoCall& operator=(const IoCall&) = delete;
    ~IoCall();
    int begin();
    int upload(void* d_dst, const void* src, size_t bytes);
    int download(void* dst, const void* d_src, size_t bytes);
    int finish(const char* what);

private:
    bool open = false;
};

// Pinned host memory for results (oxb_hip_host_alloc): a download into it needs no second copy on the host.
void* pinned_alloc(size_t bytes);  // nullptr where the bound is reached or there is no such memory
bool pinned_free(void* p);
void io_shutdown();

}  // namespace oxb
