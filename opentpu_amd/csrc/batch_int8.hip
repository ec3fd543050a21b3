// The batch MM's kernels for int8 weights.
#include "batch_impl.h"

namespace otpu {
namespace bt {
template bool launch_fmt<OTPU_INT8>(const Args& a, int nsub, int mt, hipStream_t s);
}  // namespace bt
}  // namespace otpu
