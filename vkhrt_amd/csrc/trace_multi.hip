// Traversal kernels for TLASes of several BVH modes (instantiations of trace_impl.hpp).
#include "trace_impl.hpp"

namespace vk {
using Variant0 = GeoMulti;
VKHRT_INSTANTIATE_TRACE(Variant0)
}  // namespace vk
