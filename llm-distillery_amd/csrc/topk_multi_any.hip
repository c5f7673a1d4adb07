// Forward KL against several prepared teachers on rows off the 16-byte grid or not a whole number of chunks long: the
// ROWS_ANY and ROWS_EXACT instantiations of the kernels in topk_div.hpp (see topk_multi.hip for the entry point).
#include "topk_div.hpp"

namespace dl {
int launch_fkl_any_multi(int logits_dtype, const TopkParams& p, int64_t ws_bytes, hipStream_t st, bool ws_cleared, bool off_grid) {
  return logits_dtype == DL_F32 ? launch_fkl<TagF32, true, ROWS_ANY>(p, ws_bytes, st, ws_cleared, off_grid)
         : logits_dtype == DL_BF16 ? launch_fkl<TagBF16, true, ROWS_ANY>(p, ws_bytes, st, ws_cleared, off_grid)
                                   : launch_fkl<TagF16, true, ROWS_ANY>(p, ws_bytes, st, ws_cleared, off_grid);
}
}  // namespace dl
