// Row passes (x) of kWGC8 for one group of lengths (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
template <> RowsFn rows_lo<kWGC8>(int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return launch_rows<N, kWGC8>;
    OFD_GEN_ROWS_LO(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace gen
}  // namespace ofd
