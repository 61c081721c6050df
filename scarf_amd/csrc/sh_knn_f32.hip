// The FP32 instantiations of the kNN screen and threshold kernels.
#include "sh_knn_screen.h"

namespace sh {

using Table = KnnTable<OpF32, false, 8, 16, 24, 32, 40, 48, 56, 64, 72, 80, 88, 96, 104, 112, 120,
                       128, 136>;
KnnOps knn_ops_f32() {
  return {Table::screen, Table::bound, Table::collect, Table::screen_resident,
          Table::scan_resident};
}

}  // namespace sh
