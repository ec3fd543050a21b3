// The prefill MM's kernels for fp4 weights.
#include "prefill_impl.h"

namespace otpu {
namespace pf {
template bool launch_fmt<OTPU_FP4>(const Args& a, int ms, hipStream_t s);
}  // namespace pf
}  // namespace otpu
