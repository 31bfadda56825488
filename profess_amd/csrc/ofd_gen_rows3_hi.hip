// Row passes (x) of kWT3 for one group of lengths (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
template <> RowsFn rows_hi<kWT3>(int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return launch_rows<N, kWT3>;
    OFD_GEN_ROWS_HI(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace gen
}  // namespace ofd
