// The batch MM's kernels for int4 weights.
#include "batch_impl.h"

namespace otpu {
namespace bt {
template bool launch_fmt<OTPU_INT4>(const Args& a, int nsub, int mt, hipStream_t s);
}  // namespace bt
}  // namespace otpu
