// Row passes (x with the inner part of y) of kWT3S for one group of lengths (ofd_yz_impl.h).
#include "ofd_yz_impl.h"

namespace ofd {
namespace yz {
template <> YzRowsFn yz_rows_lo<kWT3S>(int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return launch_rows<N, kWT3S>;
    OFD_YZ_ROWS_LO(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace yz
}  // namespace ofd
