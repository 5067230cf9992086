// LdsLimit over a HIP runtime of four devices that counts the calls: each device's
// limit is raised once, a failed call is tried again, devices do not share state.
#include "../../tinyinfer_amd/csrc/lds_limit.hpp"

#include <cstdio>
#include <cstdlib>

static int current = 0, calls[100] = {}, fail = 0;
extern "C" hipError_t hipGetDevice(int* dev) {
  *dev = current;
  return hipSuccess;
}
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute attr, int value) {
  if (attr != hipFuncAttributeMaxDynamicSharedMemorySize || value != 160 * 1024) std::exit(2);
  ++calls[current];
  return fail ? hipErrorInvalidValue : hipSuccess;
}

int main() {
  tia::LdsLimit limit;
  const int kernel = 0;
  auto raise = [&](int dev) {
    current = dev;
    return limit.raise(&kernel, 160 * 1024);
  };
  for (int round = 0; round < 3; ++round)
    for (int dev = 0; dev < 4; ++dev)
      if (raise(dev) != hipSuccess) return 1;
  for (int dev = 0; dev < 4; ++dev)
    if (calls[dev] != 1) return std::printf("device %d: %d calls\n", dev, calls[dev]), 1;
  fail = 1;
  if (raise(5) != hipErrorInvalidValue || raise(5) != hipErrorInvalidValue) return 1;
  fail = 0;
  if (raise(5) != hipSuccess || raise(5) != hipSuccess || calls[5] != 3) return 1;
  if (raise(70) != hipSuccess || raise(70) != hipSuccess || calls[70] != 2) return 1;  // past the record: every time
  return 0;
}
