// Prints the decode GEMV's plans (csrc/qmv_mfma.h) for the problems read from standard input, one line
// "M K N group_size bits matrices" each: waves, load steps, rounds, rows per launch, activation rows' chunks a
// lane stages, rows per workgroup of several tiles (0: one tile each).  Host code only, for 256 CUs.
#include <stdio.h>

#include "../../mlx-gen_amd/csrc/qmv_mfma.h"

namespace mlxq {
int64_t device_cu_count() { return 256; }
}  // namespace mlxq

int main() {
  long long M, K, N;
  int gs, bits, nmat;
  while (scanf("%lld %lld %lld %d %d %d", &M, &K, &N, &gs, &bits, &nmat) == 6) {
    mlxq::QmvPlan p = {};
    if (!mlxq::qmv_plan(M, K, gs, bits, nmat, p)) {
      printf("none\n");
      continue;
    }
    mlxq::QmvArgs a = {};
    a.M = M;
    a.K = K;
    a.N = N;
    if (nmat == 2) a.wq2 = reinterpret_cast<const uint32_t*>(1);
    const int staged = p.mr * ((p.steps * p.ring * (512 / bits) / 8 + 63) / 64);
    const bool built = mlxq::qmv_multi_built(bits, gs, p.steps, p.mr, nmat, p.ring);
    printf("%d %d %d %d %d %d\n", p.waves, p.steps, p.ring, p.rows, staged, built ? mlxq::qmv_multi_rows(a, p) : 0);
  }
}
