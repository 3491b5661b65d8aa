// The register kernel (ffn_mfma_reg.h) with units of up to 96 token rows.
#include "ffn_mfma_reg.h"

namespace stmoe {

int launch_reg_wide(int act_dtype, int wtag, int mode, const GemmParams& p, int tile_rows, int fewer_rows, hipStream_t st) {
  return launch_reg_mt<kRegWideRows / 16>(act_dtype, wtag, mode, p, tile_rows, fewer_rows, st);
}

}  // namespace stmoe
