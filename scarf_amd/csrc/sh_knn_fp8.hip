// The FP8 (E4M3) instantiations of the kNN screen and threshold kernels.
#include "sh_knn_screen.h"

namespace sh {

using Table = KnnTable<OpFP8, true, 64, 128>;
KnnOps knn_ops_fp8() {
  return {Table::screen, Table::bound, Table::collect, Table::screen_resident,
          Table::scan_resident};
}

}  // namespace sh
