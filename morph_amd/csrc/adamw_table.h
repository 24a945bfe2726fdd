// The device-resident descriptor table of an AdamW group with many tensors.
//
// adamw.hip's and nonfinite.hip's launches carry their descriptors in the 4 KiB of
// kernel arguments: 48 tensors an AdamW launch, 160 a detector launch.  A group of
// hundreds of small tensors (norms and biases) then takes ten launches of 5 us for a few
// us of memory traffic.  What does not change from step to step (state, sizes, constant
// sets, clocks, which block belongs to which tensor) can lie in device memory, filled
// once; the kernel arguments then hold only the gradients' addresses, kTableRefs to a
// launch.  326 tensors of 3072: 10 launches, 50 us of kernels -> 2 launches, 10.5 us.
// A launch that fits the kernel arguments stays there: it needs no table.
//
// Layout: TableRow[count], then one int32 row index per AdamW block, then one per
// detector block.
#pragma once

#include <stdint.h>

namespace morph {

struct TableRow {
  float* p;
  float* m;
  float* v;
  void* out;
  int64_t n;
  int32_t hp, clock;
  int32_t first_block, det_first;  // of this tensor, among all of the table's
  int32_t reserved[2];
};
static_assert(sizeof(TableRow) == 64, "one row per 64 bytes");

constexpr int kTableRefs = 400;           // gradients per launch: 3200 bytes of kernel arguments
constexpr int kDetectorBytes = 16 * 1024; // gradient bytes per detector workgroup

}  // namespace morph
