// The register kernel (ffn_mfma_reg.h) with units of up to 64 token rows.
#include "ffn_mfma_reg.h"

namespace stmoe {

// Whether launch_mfma_reg has a kernel for a launch.
bool reg_takes(int act_dtype, int wtag, int mode, const GemmParams& p, int64_t max_rows) {
  if ((wtag != WF_Q8_0_P && wtag != WF_Q4_1_P && wtag != WF_FP8_F32D_P) || (act_dtype != STMOE_F16 && act_dtype != STMOE_BF16)) return false;
  if ((p.offsets ? p.E > 64 : p.E != 1) || p.kred % 256 != 0 || p.lda % 8 != 0 || p.ldo % 4 != 0 ||
      p.n_out % (mode == MODE_GATEUP ? 128 : 256) != 0 || max_rows >= ((int64_t)1 << 20) || p.kred >= ((int64_t)1 << 31))
    return false;
  // token rows are addressed with 32-bit byte offsets from the activation base
  const int64_t src_rows = p.perm ? (max_rows + p.k_top - 1) / p.k_top : max_rows;
  return src_rows * p.lda * 2 < (int64_t)1 << 32;
}
int launch_mfma_reg(int act_dtype, int wtag, int mode, const GemmParams& p, int64_t max_rows, int tile_rows, int fewer_rows, hipStream_t st) {
  if (max_rows == 0) return STMOE_OK;
  if (!reg_takes(act_dtype, wtag, mode, p, max_rows))
    return set_error(STMOE_ERR_UNSUPPORTED, "mfma reg kernel: needs packed weights, 16-bit activations, at most 64 experts, K %% 256 == 0 and output features in whole tiles");
  if (tile_rows < 1 || tile_rows > kRegWideRows)
    return set_error(STMOE_ERR_SHAPE, "mfma reg kernel: units of %d token rows", tile_rows);
  if (tile_rows > kRegUnitRows) return launch_reg_wide(act_dtype, wtag, mode, p, tile_rows, fewer_rows, st);
  return launch_reg_mt<kRegUnitRows / 16>(act_dtype, wtag, mode, p, tile_rows, 0, st);
}

}  // namespace stmoe
