// bdh_launch_gemm_f32 refuses what its kernel would overwrite; the refusal comes before anything touches a device.
#include <cstdio>

#include "../burn_dragon_amd/csrc/gemm_f32.h"

int main() {
  static float C[64];
  for (int reads_c = 0; reads_c < 2; ++reads_c) {
    bdh_ctx ctx;
    GemmF32 g;
    g.A = g.B = C;
    g.C = C;
    g.M = 8; g.N = 4; g.K = 4;
    g.lda = g.ldb = g.ldc = 4;
    g.rows_per = 4;
    g.c_outer = 32;
    g.accumulate = reads_c == 0;
    g.decay_state = reads_c == 1;
    const int rc = bdh_launch_gemm_f32(&ctx, g, false, false, GemmPlan{}, nullptr);
    if (rc != BDH_E_UNSUPPORTED) return std::printf("case %d: %d\n", reads_c, rc), 1;
  }
  std::puts("ok");
  return 0;
}
