// Forward KL against one sparse teacher on rows off the 16-byte grid or not a whole number of chunks long: the
// ROWS_ANY and ROWS_EXACT instantiations of the kernels in topk_div.hpp.
#include "topk_div.hpp"

namespace dl {
int launch_fkl_any(int logits_dtype, const TopkParams& p, int64_t ws_bytes, hipStream_t st, bool off_grid) {
  return logits_dtype == DL_F32 ? launch_fkl<TagF32, false, ROWS_ANY>(p, ws_bytes, st, false, off_grid)
         : logits_dtype == DL_BF16 ? launch_fkl<TagBF16, false, ROWS_ANY>(p, ws_bytes, st, false, off_grid)
                                   : launch_fkl<TagF16, false, ROWS_ANY>(p, ws_bytes, st, false, off_grid);
}
}  // namespace dl
