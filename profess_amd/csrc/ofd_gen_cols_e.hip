// Column passes (y, z) of one group of lengths (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
ColFns cols_e(int n) {
  switch (n) {
#define X(N, A, B, T_) \
  case N: return {launch_cols<N>, launch_z<N>};
    OFD_GEN_E(X)
#undef X
    default: return {nullptr, nullptr};
  }
}
}  // namespace gen
}  // namespace ofd
