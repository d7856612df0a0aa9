// Tuned paged decode instantiations for bf16_t pools, K and V by streaming loads.
#include "decode_sched.h"

namespace llkv {
Kernels tuned_kernels_bf16_stream(int D, int G, bool append) { return tuned<bf16_t, true>(D, G, append); }
}  // namespace llkv
