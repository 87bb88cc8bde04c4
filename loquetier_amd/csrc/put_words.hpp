// Small host tables on the device without a copy: their words travel in the launch's own arguments.
#pragma once
#include "smlm_common.hpp"

namespace smlm {

// A copy of a few words from pageable host memory makes the host wait (15 us and more, and for everything queued before
// it); a launch takes 4 and waits for nothing: its argument block goes to the device anyhow.  Whole add_lora forward and
// backward of three sequences of 200 rows, six such copies and a plan launch before, one launch now: 378 -> 278 us.
template <int N>
struct PutArgs {
  uint32_t* dst;
  int n;
  uint32_t words[N];
};
template <int N>
__global__ __launch_bounds__(256) void put_words_kernel(PutArgs<N> a) {
  for (int i = threadIdx.x; i < a.n; i += 256) a.dst[i] = a.words[i];
}
constexpr int kPutSmall = 128, kPutLarge = 896;  // (a launch takes up to 4 KiB of arguments)

}  // namespace smlm
