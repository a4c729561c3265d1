// Size rule of the device blocks that the runtime keeps (pt_runtime.hip).
// Plain C++: it runs on the host only.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace pt {

// No request above this reaches the driver: nothing that large exists, and
// every size at or below it can be rounded up without leaving size_t.
constexpr size_t kMaxBlockBytes = (size_t)PTRDIFF_MAX;

// The size a request of at most kMaxBlockBytes is rounded up to: a multiple
// of 512 bytes and of a sixteenth to an eighth of itself.
inline size_t block_class(size_t bytes)
{
    size_t step = 512;
    while (step <= bytes / 16) step *= 2;
    return (bytes + step - 1) / step * step;
}

}  // namespace pt
