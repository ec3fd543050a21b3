// The prefill MM's kernels for int4 weights.
#include "prefill_impl.h"

namespace otpu {
namespace pf {
template bool launch_fmt<OTPU_INT4>(const Args& a, int ms, hipStream_t s);
}  // namespace pf
}  // namespace otpu
