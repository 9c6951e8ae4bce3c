// Decode-kernel instantiations for query type F32 and FP8 E4M3 caches (paged
// 5-D layout, head sizes that are multiples of 16, every block size).  One
// translation unit per type pair keeps the kernel matrix compiling in
// parallel.
#include "paged_decode_impl.h"

namespace pkv {
template hipError_t launch_decode_typed<F32, FP8>(const DecodeArgs&, int, int, hipStream_t, bool*);
}  // namespace pkv
