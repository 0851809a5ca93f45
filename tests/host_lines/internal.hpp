// Host stand-in for the library's internal header: what the kernel arguments name.
#pragma once
#include <cstdint>

namespace ifem {
constexpr int kMaxP = 3, kMaxNG = 5;
struct DevFunction {
  int type = 0;
};
} // namespace ifem
