// Workgroups per CU of a few kernels by the LDS that a launch asks for, worked out once for each.
//
// The layers of a network come in several image sizes and take turns, so one remembered size per kernel is forgotten at every
// layer, and asked for again in front of its launch: three pairs of convolutions (4 images of 28x28x128, 14x14x256, 7x7x512) in
// turn took 83.6 us under RowSync and 86.3 under TileSync, 81.9 and 84.3 with this (78.2 and 80.7 each by itself again and again).
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace cusync {
namespace rt {

// KIB: the most LDS of a launch, in KiB.  Not thread-safe.
template<int KERNELS, int KIB>
class OccupancyTable {
public:
  // ask(bytes) gives the workgroups per CU of launches with that much LDS; below 0 after an error, which is not remembered.
  template<class Ask>
  int perCU(int kernel, size_t lds, Ask ask) {
    const size_t kib = (lds + 1023) / 1024;
    if (kib > (size_t)KIB) return 0;
    int8_t& known = known_[kernel][kib];
    if (known == 0) {
      const int n = ask(kib * 1024);
      if (n < 0) return n;
      known = (int8_t)((n < 126 ? n : 126) + 1);
    }
    return known - 1;
  }

private:
  int8_t known_[KERNELS][KIB + 1] = {};      // one more than the workgroups per CU; 0: not asked yet
};

}  // namespace rt
}  // namespace cusync
