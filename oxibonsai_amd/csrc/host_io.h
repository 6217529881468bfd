// host_io.h — moving the host buffers of a call to and from the device (host_io.hip).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace oxb {

// All of these run under the library's lock and enqueue on the stream in use.
//
// A call that takes host buffers: io_begin, io_upload for every input, its launches, io_download for every output, and
// io_finish, after which the outputs are there.  (A call that fails on the way leaves the rest to the next io_begin.)
int io_begin();
// src is free for the caller to reuse when this returns.
int io_upload(void* d_dst, const void* src, size_t bytes);
int io_download(void* dst, const void* d_src, size_t bytes);
int io_finish(const char* what);

// Pinned host memory for results (oxb_hip_host_alloc): a download into it needs no second copy on the host.
void* pinned_alloc(size_t bytes);  // nullptr where the bound is reached or there is no such memory
bool pinned_free(void* p);
void io_shutdown();

}  // namespace oxb
