// The extend (prefill) kernels of one head_dim (DK_HEAD_DIM, set by the build: 64, 128 or
// 256) and their symbol table.
#include "dk_extend.h"

#ifndef DK_HEAD_DIM
#error "compile once per head_dim with -DDK_HEAD_DIM=64, 128 or 256"
#endif

namespace dk {
namespace {
template <class T, bool KV8>
const void* sym(bool cap) {
  return cap ? reinterpret_cast<const void*>(&dk_extend<T, DK_HEAD_DIM, KV8, true>)
             : reinterpret_cast<const void*>(&dk_extend<T, DK_HEAD_DIM, KV8, false>);
}
}  // namespace

template <int D>
const void* extend_symbol(bool bf16, bool kv8, bool cap) {
  if (bf16) return kv8 ? sym<BF16, true>(cap) : sym<BF16, false>(cap);
  return kv8 ? sym<F16, true>(cap) : sym<F16, false>(cap);
}
template const void* extend_symbol<DK_HEAD_DIM>(bool, bool, bool);
}  // namespace dk
