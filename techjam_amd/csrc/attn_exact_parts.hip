// The key-part instances of the exact-attention kernel, in a translation unit
// of their own: beside them the compiler schedules the one-sweep kernels it
// shares its inlined tile with differently (head_dim 128 fp16, 6 x 12 padded
// heads of 1777: 109.8 -> 110.5 us).
#include "attn_exact_kernel.h"

namespace tj {
namespace {

template <typename T>
int dispatch(const AttnArgs& a, int64_t D, hipStream_t stream) {
  switch (D) {
    case 32: return launch_parts<T, 32>(a, stream);
    case 64: return launch_parts<T, 64>(a, stream);
    case 128: return launch_parts<T, 128>(a, stream);
    default: return launch_parts<T, 256>(a, stream);
  }
}

}  // namespace

int dispatch_parts_f32(const AttnArgs& a, int64_t D, hipStream_t stream) { return dispatch<float>(a, D, stream); }
int dispatch_parts_f16(const AttnArgs& a, int64_t D, hipStream_t stream) { return dispatch<half_t>(a, D, stream); }

}  // namespace tj
