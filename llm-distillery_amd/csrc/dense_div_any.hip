// Divergences against a dense teacher on rows off the 16-byte grid or not a whole number of 8-column units long.
#include "dense_kernels.hpp"

namespace dl {

template <int KIND, class TagS, class TagT, int NU>
static bool launch_any_kind(const DenseParams& p, hipStream_t st) {
  const int64_t units = p.V / 8;      // the columns behind them ride along whatever the shape
  if (units <= 256 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 256, NU, true>(p, st);
  else if (units <= 512 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 512, NU, true>(p, st);
  else if (units <= 1024 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 1024, NU, true>(p, st);
  else return false;
  return true;
}
template <class TagS, class TagT, int NU>
static bool launch_any_pair(const DenseParams& p, hipStream_t st) {
  if (p.kind == DL_FKL) return launch_any_kind<DL_FKL, TagS, TagT, NU>(p, st);
  if (p.kind == DL_RKL) return launch_any_kind<DL_RKL, TagS, TagT, NU>(p, st);
  return launch_any_kind<DL_JSD, TagS, TagT, NU>(p, st);
}

bool launch_dense_any(const DenseParams& p, hipStream_t st) {
  if (p.s_dtype == F32 && p.t_dtype == F32) return launch_any_pair<TagF32, TagF32, 4>(p, st);
  if (p.s_dtype == BF16 && p.t_dtype == BF16) return launch_any_pair<TagBF16, TagBF16, 8>(p, st);
  if (p.s_dtype == F16 && p.t_dtype == F16) return launch_any_pair<TagF16, TagF16, 8>(p, st);
  if (p.s_dtype == BF16 && p.t_dtype == F32) return launch_any_pair<TagBF16, TagF32, 4>(p, st);
  if (p.s_dtype == F16 && p.t_dtype == F32) return launch_any_pair<TagF16, TagF32, 4>(p, st);
  if (p.s_dtype == F32 && p.t_dtype == BF16) return launch_any_pair<TagF32, TagBF16, 4>(p, st);
  if (p.s_dtype == F32 && p.t_dtype == F16) return launch_any_pair<TagF32, TagF16, 4>(p, st);
  return false;
}

void launch_dense_split_any(const DenseParams& p, const DenseSplit& x, int nt, hipStream_t st) {
  launch_dense_split_pair<true>(p, x, nt, st);
}

}  // namespace dl
