// Row passes (x) of kWT3S for one group of lengths (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
template <> RowsFn rows_lo<kWT3S>(int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return launch_rows<N, kWT3S>;
    OFD_GEN_ROWS_LO(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace gen
}  // namespace ofd
