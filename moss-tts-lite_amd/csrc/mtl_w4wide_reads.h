// Where w4_wide_kernel reads the weight and its staged metadata: byte offsets within each
// buffer.  Plain C++ without HIP types, so that a host program can walk every read.
#pragma once

namespace mtl {

// The strip that is read in the place of `strip`: the column tiles round N up to 256 columns,
// and strips past N repeat the last one.  These offsets travel as the scalar offset of a buffer
// load, which the load's range check need not cover, so they have to lie inside by themselves.
constexpr int wide_strip(int strip, int nstrips) { return strip < nstrips ? strip : nstrips - 1; }

constexpr int wide_weight_at(int strip, int kblocks, int block) {
  return (strip * kblocks + block) * 1024;                       // 1 KB follows
}

// g = 256 has one record for two blocks (krec = kblocks / 2), any other group one per block.
constexpr int wide_scale_at(int strip, int krec, int kblocks, int block, int mb) {
  return (strip * krec + (krec == kblocks ? block : block >> 1)) * 32 * mb;   // 32 mb bytes follow
}

constexpr int wide_zero_at(int strip, int zchunks, int chunk) {
  return (strip * zchunks + chunk) * 1024;                       // 1 KB follows
}

}  // namespace mtl
