// The BF16 instantiations of the kNN screen and threshold kernels.
#include "sh_knn_screen.h"

namespace sh {

using Table = KnnTable<OpBF16, false, 16, 32, 48, 64, 80, 96, 112, 128>;
KnnOps knn_ops_bf16() {
  return {Table::screen, Table::bound, Table::collect, Table::screen_resident,
          Table::scan_resident};
}

}  // namespace sh
