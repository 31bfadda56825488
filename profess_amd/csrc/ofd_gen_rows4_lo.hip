// Row passes (x) of kWT4 for one group of lengths (ofd_gen_impl.h).
#include "ofd_gen_impl.h"

namespace ofd {
namespace gen {
template <> RowsFn rows_lo<kWT4>(int m) {
  switch (m) {
#define X(N, A, B, T_) \
  case N: return launch_rows<N, kWT4>;
    OFD_GEN_ROWS_LO(X)
#undef X
    default: return nullptr;
  }
}
}  // namespace gen
}  // namespace ofd
