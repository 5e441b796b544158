#include "hxq_rows_impl.h"

namespace hxq {
namespace rw {
template int launch_rows<0>(const Call &, int, bool, const Plan &, hipStream_t);
template int launch_grouped<0>(const Call &, const Grouped &, bool, int, hipStream_t);
}  // namespace rw
}  // namespace hxq
