#include "hxq_rows_impl.h"

namespace hxq {
namespace rw {
template int launch_rows<0>(const Call &, int, bool, const Plan &, hipStream_t);
}  // namespace rw
}  // namespace hxq
