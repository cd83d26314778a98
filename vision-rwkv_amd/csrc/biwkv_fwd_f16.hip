// Bi-WKV forward kernels for __half I/O.
#include "biwkv_fwd_impl.h"
namespace vrwkv {
namespace biwkv_fwd_detail {
template int biwkv_fwd_launch_io<__half>(const Plan&, const ParamVec&, const ParamVec&, const void*, const void*, const void*, void*, float*, int, int, int, hipStream_t);
}
}
#ifdef VRWKV_STAMPS
VRWKV_DEFINE_STAMP_SETTER(f16)
#endif
