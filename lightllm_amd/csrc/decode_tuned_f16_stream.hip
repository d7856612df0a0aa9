// Tuned paged decode instantiations for _Float16 pools, K and V by streaming loads.
#include "decode_sched.h"

namespace llkv {
Kernels tuned_kernels_f16_stream(int D, int G, bool append) { return tuned<_Float16, true>(D, G, append); }
}  // namespace llkv
