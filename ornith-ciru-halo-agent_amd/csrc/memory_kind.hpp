// Which memory a kernel's device-scope atomics may be used on.
#pragma once
#include <hip/hip_runtime_api.h>

namespace ornith {

// Memory that a kernel on `device` reaches with device-scope atomics: that
// device's own allocations.  Pinned host and managed memory, and a peer's
// memory behind xGMI (cached apart in each XCD's L2, and only certain to be
// coherent when the kernel ends), take plain stores.
inline bool device_atomics_reach(const hipPointerAttribute_t& at, int device) {
    return at.type == hipMemoryTypeDevice && !at.isManaged && at.device == device;
}

}  // namespace ornith
