// Copies of large fields between the device and the caller's (pageable) FP64 host arrays.
#pragma once
#include <hip/hip_runtime.h>
#include <memory>

namespace flusi {

// One pool of pinned staging memory per device, shared by the contexts on it;
// it is freed with the last of them.
class HostCopyPool;
std::shared_ptr<HostCopyPool> host_copy_pool(int device);

// n reals: device element type T (float or double), host doubles; the pool's
// device holds them, whichever is current for the caller.  Ordered after the
// stream's earlier work; complete on return, with its outcome in `result`.
// False: no staging memory (or none yet: a small copy in does not make it at
// once), nothing copied; the plain copy needs none.
bool host_copy_pays(const void* host, long n, size_t elem);  // else a plain copy is as good
template <typename T>
bool host_copy_out(HostCopyPool& pool, const T* dev, double* host, long n, hipStream_t s, hipError_t& result);
template <typename T>
bool host_copy_in(HostCopyPool& pool, const double* host, T* dev, long n, hipStream_t s, hipError_t& result);

}  // namespace flusi
