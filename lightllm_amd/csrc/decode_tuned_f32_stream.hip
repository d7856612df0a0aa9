// Tuned paged decode instantiations for float pools, K and V by streaming loads.
#include "decode_sched.h"

namespace llkv {
Kernels tuned_kernels_f32_stream(int D, int G, bool append) { return tuned<float, true>(D, G, append); }
}  // namespace llkv
