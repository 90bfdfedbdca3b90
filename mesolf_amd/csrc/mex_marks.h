// Marks of a MEX call: which of its bitmaps, and which of its kernel sets, hold
// values that the BF16 split form (mex_split.hip) leaves to the FP32 form
// (k_mex_mfma).  They lie at the start of the call's scratch, zero when that is
// made and never cleared.  A mark holds the number of the call it was made in.
// The number is counted on the device: it is one more than that of
// the last finished call, so a sequence of launches that is replayed as it
// was recorded gets a new one each time.  k_mex_split_prep makes the marks;
// k_mex_split reads the count and passes the number on to k_mex_mfma, whose last
// launch of the call moves the count.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mlf {

constexpr int kMexHeadWords = 64;

struct MexMarks {
  uint32_t* w = nullptr;  // head words, then one word per bitmap; null: no marks

  __device__ uint32_t* finished() const { return w; }      // number of the last finished call
  __device__ uint32_t* current() const { return w + 1; }   // number of the call, for k_mex_mfma
  __device__ uint32_t* any() const { return w + 2; }       // a mark was made
  __device__ uint64_t* set() const { return reinterpret_cast<uint64_t*>(w + 4); }  // a kernel set is marked
  __device__ uint32_t* image(int i) const { return w + kMexHeadWords + i; }

  __device__ static uint64_t set_mark(uint32_t call, int ordinal) { return (uint64_t)ordinal << 32 | call; }
  // Kernel set `ordinal` of the call, or bitmap i, is the FP32 form's.
  __device__ bool set_marked(uint32_t call, int ordinal) const { return *set() == set_mark(call, ordinal); }
  __device__ bool image_marked(uint32_t call, int i) const { return *image(i) == call; }
};

}  // namespace mlf
