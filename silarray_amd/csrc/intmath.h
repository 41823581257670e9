#pragma once

#include <cstdint>

namespace silgpu {

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace silgpu
