// The y + z pass of one group of z lengths (ofd_yz_impl.h).
#include "ofd_yz_impl.h"

namespace ofd {
namespace yz {
YzFn yz_a(int n) {
  switch (n) {
#define X(N, A, B, T_) \
  case N: return launch_yz<N>;
    OFD_YZ_COLS_A(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace yz
}  // namespace ofd
