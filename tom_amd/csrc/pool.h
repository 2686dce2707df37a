// Device workspaces of the calls, kept between calls.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <initializer_list>

namespace tomhip {

// hipMalloc on the current device, for memory of any lifetime: where it fails
// the workspaces that wait for a next call are freed and it is tried again
// (throws like TOMHIP_CHECK(hipMalloc)). Freed with hipFree.
void* device_malloc(size_t bytes);

// A device workspace of at least `bytes` on the current device, for work on
// stream s (throws like device_malloc).
void* work_get(size_t bytes, hipStream_t s);
template <typename T>
void work_get(T** p, size_t bytes, hipStream_t s) {
  *p = static_cast<T*>(work_get(bytes, s));
}
// Gives a workspace back; what is queued on s so far may still use it. Null
// is ignored.
void work_put(const void* p, hipStream_t s) noexcept;
// Gives *p back and takes a workspace of `bytes` in its place. Where that
// fails *p is null: no pointer to a workspace that has been given back stays.
template <typename T>
void work_renew(T** p, size_t bytes, hipStream_t s) {
  work_put(*p, s);
  *p = nullptr;
  work_get(p, bytes, s);
}
// Gives workspaces of the current device back that any of its streams may
// still use: waits for the device, and where that is refused (while a stream
// is being captured) they go to the driver instead of the next call.
void work_put_all(std::initializer_list<const void*> ps) noexcept;

// Frees what waits for a next call on the device.
void work_trim(int device);

// Contexts of a device, counted: the last one to go frees what is kept.
void work_device_up(int device);
void work_device_down(int device) noexcept;

}  // namespace tomhip
