// Kernels and C entry point for divergences against a dense teacher stored in memory.
#include "dense_kernels.hpp"

namespace dl {

// Rows too wide for the registers, 16-byte aligned: the same sweeps, every one of them over global
// memory with 16-byte loads, two units per thread in flight (2-3 reads of both rows; all but the first
// come from L2 / the memory-side cache as far as the rows of the workgroups in flight fit there).
template <class TagS, class TagT, int NT>
struct StreamRows {
  static constexpr bool ONLINE = true;       // every sweep reads both rows: maxima and sums share one
  const char* srow;
  const char* trow;
  int64_t nunits;
  __device__ __forceinline__ void store(char* grow, int64_t u, const float* g, Columns<8>) const { Unit<TagS>::store(grow, u, g); }
  template <class Tag>
  static __device__ __forceinline__ void fetch(Unit<Tag>& x, const char* row, int64_t u) {
#pragma unroll
    for (int k = 0; k < Unit<Tag>::NC; ++k) x.c[k] = *reinterpret_cast<const u32x4*>(row + (u * Unit<Tag>::NC + k) * 16);
  }
  template <class F>
  __device__ __forceinline__ void sweep(F f) {
    constexpr int U = 2;
    for (int64_t u0 = threadIdx.x; u0 < nunits; u0 += (int64_t)U * NT) {
      Unit<TagS> s[U];
      Unit<TagT> t[U];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int64_t u = u0 + (int64_t)j * NT;
        if (u < nunits) { fetch(s[j], srow, u); fetch(t[j], trow, u); }
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int64_t u = u0 + (int64_t)j * NT;
        if (u < nunits) {
          float a[8], b[8];
          s[j].unpack(a);
          t[j].unpack(b);
          f(u, a, b, Columns<8>{});
        }
      }
    }
  }
};

template <int KIND, class TagS, class TagT, int NT>
__global__ __launch_bounds__(NT) void dense_stream_vec_kernel(const DenseParams p) {
  __shared__ float red[64];
  const int64_t r = xcd_banded_row(blockIdx.x);
  if (r >= p.n_rows) return;
  const int tid = threadIdx.x;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * TagS::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  if (trow < 0) {
    if (grow) zero_row<TagS, NT>(grow, p.V / TagS::epc);
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  StreamRows<TagS, TagT, NT> rows{reinterpret_cast<const char*>(p.logits) + r * p.row_stride * TagS::bytes,
                                  reinterpret_cast<const char*>(p.t_logits) + trow * p.t_stride * TagT::bytes, p.V / 8};
  const DenseStats st = dense_stats<KIND, NT>(rows, p.inv_T_s, p.inv_T_t, red);
  if (tid == 0 && p.row_loss) p.row_loss[r] = st.loss;
  if (grow) dense_grad_sweep<KIND, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
}

// Rows too wide for both to sit in registers, but not for the student's alone: the student row is
// read from HBM once and kept on the CU, half of it in registers (NUS / 2 units per thread) and half
// in LDS (128 KiB; all of it in registers leaves too few for the sweeps: the compiler spills).  The
// teacher row is streamed through a ring of D units per thread in every sweep (its later reads come
// from L2 as far as the rows in flight fit there).  Against streaming both rows this saves one or
// two reads of the student row.
template <class TagS, class TagT, int NT, int NUS>
struct StudentRegRows {
  static constexpr bool ONLINE = true;       // every sweep reads the teacher row: maxima and sums share one
  static constexpr int D = Unit<TagT>::NC == 1 ? 4 : 2;      // teacher units in flight per thread
  static constexpr int NR = NUS / 2;                         // student units in registers; the rest in LDS
  static constexpr int NC = Unit<TagS>::NC;
  static constexpr size_t LDS_BYTES = (size_t)(NUS - NR) * NC * NT * 16;
  Unit<TagS> s[NR];
  u32x4* lds;
  const char* trow;
  int64_t nunits;
  __device__ __forceinline__ void store(char* grow, int64_t u, const float* g, Columns<8>) const { Unit<TagS>::store(grow, u, g); }
  __device__ __forceinline__ void load(const char* srow, const char* trow_, int64_t nu, u32x4* lds_) {
    trow = trow_;
    nunits = nu;
    lds = lds_;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (u < nunits) s[i].load(srow, u);
      else s[i].fill_neg_inf();
    }
#pragma unroll
    for (int i = NR; i < NUS; ++i) {         // every thread reads back only what it wrote: no barrier needed
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      Unit<TagS> x;
      if (u < nunits) x.load(srow, u);
      else x.fill_neg_inf();
#pragma unroll
      for (int k = 0; k < NC; ++k) lds[((i - NR) * NC + k) * NT + threadIdx.x] = x.c[k];
    }
  }
  template <class F>
  __device__ __forceinline__ void sweep(F f) {
    Unit<TagT> t[D];
#pragma unroll
    for (int d = 0; d < D && d < NUS; ++d) {
      const int64_t u = (int64_t)d * NT + threadIdx.x;
      if (u < nunits) StreamRows<TagS, TagT, NT>::fetch(t[d], trow, u);
    }
#pragma unroll
    for (int i = 0; i < NUS; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (u < nunits) {
        float a[8], b[8];
        if (i < NR) {
          s[i].unpack(a);
        } else {
          Unit<TagS> x;
#pragma unroll
          for (int k = 0; k < NC; ++k) x.c[k] = lds[((i - NR) * NC + k) * NT + threadIdx.x];
          x.unpack(a);
        }
        t[i % D].unpack(b);
        f(u, a, b, Columns<8>{});
      }
      if (i + D < NUS) {                     // refill the slot just used
        const int64_t un = (int64_t)(i + D) * NT + threadIdx.x;
        if (un < nunits) StreamRows<TagS, TagT, NT>::fetch(t[i % D], trow, un);
      }
      // no memory access moves across this point: without it the compiler issues the loads of all
      // units up front and spills the registers that hold them
      asm volatile("" ::: "memory");
    }
  }
};

template <int KIND, class TagS, class TagT, int NT, int NUS>
__global__ __launch_bounds__(NT) void dense_student_reg_kernel(const DenseParams p) {
  extern __shared__ __align__(16) u32x4 student_half[];
  __shared__ float red[64];
  const int64_t r = xcd_banded_row(blockIdx.x);
  if (r >= p.n_rows) return;
  const int tid = threadIdx.x;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * TagS::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  if (trow < 0) {
    if (grow) zero_row<TagS, NT>(grow, p.V / TagS::epc);
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  StudentRegRows<TagS, TagT, NT, NUS> rows;
  rows.load(reinterpret_cast<const char*>(p.logits) + r * p.row_stride * TagS::bytes,
            reinterpret_cast<const char*>(p.t_logits) + trow * p.t_stride * TagT::bytes, p.V / 8, student_half);
  const DenseStats st = dense_stats<KIND, NT>(rows, p.inv_T_s, p.inv_T_t, red);
  if (tid == 0 && p.row_loss) p.row_loss[r] = st.loss;
  if (grow) dense_grad_sweep<KIND, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
}

// Any size, any alignment, any dtype pair: four scalar passes over global memory.
template <int NT>
__global__ __launch_bounds__(NT) void dense_stream_kernel(const DenseParams p) {
  __shared__ float red[64];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t V = p.V;
  const int sb = p.s_dtype == F32 ? 4 : 2, tb = p.t_dtype == F32 ? 4 : 2;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * sb : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  if (trow < 0) {
    if (grow) for (int64_t j = tid; j < V; j += NT) store_from_float(grow, p.s_dtype, j, 0.f);
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  const char* srow = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * sb;
  const char* trw = reinterpret_cast<const char*>(p.t_logits) + trow * p.t_stride * tb;
  const int kind = p.kind;
  const float a_s = p.inv_T_s * LOG2E, a_t = p.inv_T_t * LOG2E;
  float ms = -INFINITY, mt = -INFINITY;
  for (int64_t j = tid; j < V; j += NT) {
    const float s = load_as_float(srow, p.s_dtype, j), t = load_as_float(trw, p.t_dtype, j);
    mt = fmaxf(mt, t);
    ms = fmaxf(ms, (kind == DL_RKL && t == -INFINITY) ? -INFINITY : s);
  }
  block_max2<NT>(ms, mt, red);
  const float bs = ms * a_s, bt = mt * a_t;
  float ss = 0.f, stt = 0.f;
  for (int64_t j = tid; j < V; j += NT) {
    const float s = load_as_float(srow, p.s_dtype, j), t = load_as_float(trw, p.t_dtype, j);
    ss += (kind == DL_RKL && t == -INFINITY) ? 0.f : fast_exp2(fmaf(s, a_s, -bs));
    stt += fast_exp2(fmaf(t, a_t, -bt));
  }
  block_sum2<NT>(ss, stt, red);
  const float ls = bs + fast_log2(ss), lt = bt + fast_log2(stt);
  float x = 0.f, y = 0.f;
  for (int64_t j = tid; j < V; j += NT) {
    const float lp = fmaf(load_as_float(srow, p.s_dtype, j), a_s, -ls);
    const float lq = fmaf(load_as_float(trw, p.t_dtype, j), a_t, -lt);
    if (kind == DL_FKL) fkl_term(lp, lq, x);
    else if (kind == DL_RKL) rkl_term(lp, lq, x);
    else jsd_term(lp, lq, x, y);
  }
  block_sum2<NT>(x, y, red);
  const float loss = kind == DL_JSD ? 0.5f * LN2 * (x + y) : x * LN2;
  const float aux = x * LN2;
  if (tid == 0 && p.row_loss) p.row_loss[r] = loss;
  if (grow) {
    const float c = p.inv_T_s * p.grad_scale;
    for (int64_t j = tid; j < V; j += NT) {
      const float lp = fmaf(load_as_float(srow, p.s_dtype, j), a_s, -ls);
      const float lq = fmaf(load_as_float(trw, p.t_dtype, j), a_t, -lt);
      store_from_float(grow, p.s_dtype, j, dense_grad(kind, lp, lq, aux) * c);
    }
  }
}

template <int KIND, class TagS, class TagT, int NU>
static bool launch_dense_kind(const DenseParams& p, hipStream_t st) {
  const int64_t units = p.V / 8;
  constexpr int NUS = 256 / (16 * Unit<TagS>::NC);      // the student row alone: 256 bytes of registers per thread
  const dim3 grid(xcd_banded_grid(p.n_rows));
  if (units <= 256 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 256, NU, false>(p, st);
  else if (units <= 512 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 512, NU, false>(p, st);
  else if (units <= 1024 * NU) launch_dense_reg_nt<KIND, TagS, TagT, 1024, NU, false>(p, st);
  else if (units <= 1024 * NUS) {
    // more than 64 KiB of dynamic LDS has to be requested per kernel, once per device (the call is slow)
    constexpr size_t lds = StudentRegRows<TagS, TagT, 1024, NUS>::LDS_BYTES;
    static thread_local int allowed_on = -1;
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (allowed_on != dev) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(&dense_student_reg_kernel<KIND, TagS, TagT, 1024, NUS>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return false;
      allowed_on = dev;
    }
    hipLaunchKernelGGL((dense_student_reg_kernel<KIND, TagS, TagT, 1024, NUS>), grid, dim3(1024), lds, st, p);
  }
  else hipLaunchKernelGGL((dense_stream_vec_kernel<KIND, TagS, TagT, 1024>), grid, dim3(1024), 0, st, p);
  return true;
}

template <class TagS, class TagT, int NU>
static bool launch_dense_reg(const DenseParams& p, hipStream_t st) {
  if (p.kind == DL_FKL) return launch_dense_kind<DL_FKL, TagS, TagT, NU>(p, st);
  if (p.kind == DL_RKL) return launch_dense_kind<DL_RKL, TagS, TagT, NU>(p, st);
  return launch_dense_kind<DL_JSD, TagS, TagT, NU>(p, st);
}

// Register path for the dtype pairs that occur: teacher stored like the student, or in fp32, or a 16-bit teacher
// against a student that the caller has already cast to fp32 (as the reference does with its logits).
static bool launch_dense_pair(const DenseParams& p, hipStream_t st) {
  if (p.s_dtype == F32 && p.t_dtype == F32) return launch_dense_reg<TagF32, TagF32, 4>(p, st);
  if (p.s_dtype == BF16 && p.t_dtype == BF16) return launch_dense_reg<TagBF16, TagBF16, 8>(p, st);
  if (p.s_dtype == F16 && p.t_dtype == F16) return launch_dense_reg<TagF16, TagF16, 8>(p, st);
  if (p.s_dtype == BF16 && p.t_dtype == F32) return launch_dense_reg<TagBF16, TagF32, 4>(p, st);
  if (p.s_dtype == F16 && p.t_dtype == F32) return launch_dense_reg<TagF16, TagF32, 4>(p, st);
  if (p.s_dtype == F32 && p.t_dtype == BF16) return launch_dense_reg<TagF32, TagBF16, 4>(p, st);
  if (p.s_dtype == F32 && p.t_dtype == F16) return launch_dense_reg<TagF32, TagF16, 4>(p, st);
  return false;
}

// Units per thread of the split kernels for a dtype pair (0: the pair has no register kernel).
static int dense_split_units(int s_dtype, int t_dtype) {
  if (s_dtype == t_dtype) return s_dtype == F32 ? 4 : 8;
  return t_dtype == F32 ? 6 : s_dtype == F32 ? 4 : 0;
}
// How a row of V columns is cut: threads per part and parts (parts == 0: not cut).  Measured (forward KL, 512 and
// 8192 rows, 32000 to 262144 columns, fp32 pairs, 16-bit pairs and a 16-bit student against an fp32 teacher):
//   * a row that half a workgroup's registers hold (512 threads) stays whole (4096 x 20000 bf16 against fp32, which take
//     1024 threads whole: 167 us, two parts of 256: 126);
//   * with a 16-bit student up to four parts of 256 threads beat half as many of 512 (more workgroups per CU to
//     hide the exchange behind), beyond that the partners to wait for cost more than they bring: parts of 512
//     threads, at most 8; fp32 students (a part of 256 threads holds 8192 columns only) take parts of 512 from the start;
//   * wider still, pairs with an fp32 row take parts of 1024 threads (beyond 8 of those, and beyond 262144
//     columns of a 16-bit pair, one workgroup per row streams the row from the caches);
//   * on fewer than 1024 rows the cut pays only from 256 KiB of row pair upwards (one workgroup per row keeps
//     the CUs busy by itself below that, and has no partners to wait for).
//   * JSD, whose parts meet twice and have one more launch behind them: a pair that 1024 threads hold stays whole below
//     1536 rows of 16-bit pairs and 3072 rows of others; a pair that they do not hold is always cut.  From these lines on the
//     cut was ahead at every width when both forms made the log ratios twice.  Now that they are kept, the two meet elsewhere,
//     earlier for wide rows (whole and cut, us): 16-bit pairs of 33000 / 40960 / 50257 / 65536 columns, 512 rows 37 / 41 / 54 / 70 and
//     46 / 49 / 57 / 62, 1024 rows 70 / 81 / 102 / 126 and 71 / 77 / 94 / 106, 1536 rows 103 / 118 / 149 / 182 and 96 / 107 / 132 / 147;
//     16392 / 24000 / 32768 columns, fp32 2048 rows 100 / 130 / 169 and 108 / 132 / 161, 3072 rows 148 / 186 / 240 and 148 / 186 /
//     230; bf16 against fp32 1536 rows 62 / 85 / 103 and 60 / 76 / 103 (28000: 98 and 101), 3072 rows 120 / 161 / 203 and 102 / 132 /
//     197; fp32 against bf16 1536 rows 77 / 102 / 135 and 86 / 102 / 126, 3072 rows 140 / 186 / 237 and 146 / 178 / 219 (16392
//     columns of this pair are ahead whole to 4096 rows: 178 and 185).
// `forced_nt` (256 / 512 / 1024, a tuning hook) fixes the thread count and cuts wherever two parts or more come out.
struct DenseCut { int nt, parts; };
static DenseCut dense_split_cut(int kind, int s_dtype, int t_dtype, int64_t n_rows, int64_t V, int forced_nt = 0) {
  const int nu = dense_split_units(s_dtype, t_dtype);
  if (nu == 0 || V < 8) return {0, 0};
  const int64_t units = (V + 7) / 8;
  const auto parts_of = [&](int nt) { return (units + (int64_t)nt * nu - 1) / ((int64_t)nt * nu); };
  const auto cut_of = [&](int nt) {
    const int64_t parts = parts_of(nt);
    return parts >= 2 && parts <= DENSE_MAX_PARTS && (nt != 1024 || t_dtype == F32 || s_dtype == F32) ? DenseCut{nt, (int)parts} : DenseCut{0, 0};
  };
  if (forced_nt) return cut_of(forced_nt);
  const int whole_nu = s_dtype == t_dtype && s_dtype != F32 ? 8 : 4;      // units per thread of the kernels that hold a row whole
  if (units <= 512 * whole_nu) return {0, 0};
  if (kind == DL_JSD) {
    if (units <= 1024 * whole_nu && n_rows < (whole_nu == 8 ? 1536 : 3072)) return {0, 0};
  } else {
    const int64_t pair_bytes = V * ((s_dtype == F32 ? 4 : 2) + (t_dtype == F32 ? 4 : 2));
    if (n_rows < 1024 && pair_bytes < 256 * 1024) return {0, 0};
  }
  if (parts_of(256) <= 4 && s_dtype != F32) return cut_of(256);      // (fp32 students: 8192 columns per such part only)
  if (parts_of(512) <= DENSE_MAX_PARTS) return cut_of(512);
  return cut_of(1024);
}

}  // namespace dl

extern "C" int64_t dl_div_dense_workspace_bytes(int kind, int logits_dtype, int t_dtype, int64_t n_rows, int64_t V) {
  if (n_rows <= 0 || V <= 0) return 0;
  // enough for every cut the flags of dl_div_dense_ws may ask for
  int parts = 0;
  for (int nt : {0, 256, 512, 1024}) parts = std::max(parts, dl::dense_split_cut(kind, logits_dtype, t_dtype, n_rows, V, nt).parts);
  return parts ? dl::DenseSplit::bytes(kind, n_rows, parts) : 0;
}

extern "C" int dl_div_dense(int kind, const void* logits, int logits_dtype, int64_t row_stride, int64_t n_rows,
                            int64_t V, const int32_t* row_map, const void* t_logits, int t_dtype, int64_t t_stride,
                            int64_t n_teacher_rows, float inv_T_student, float inv_T_teacher, float grad_scale,
                            float* row_loss, void* grad, int64_t grad_stride, void* stream) {
  return dl_div_dense_ws(kind, logits, logits_dtype, row_stride, n_rows, V, row_map, t_logits, t_dtype, t_stride,
                         n_teacher_rows, inv_T_student, inv_T_teacher, grad_scale, row_loss, grad, grad_stride, nullptr, 0, 0,
                         stream);
}

extern "C" int dl_div_dense_ws(int kind, const void* logits, int logits_dtype, int64_t row_stride, int64_t n_rows,
                               int64_t V, const int32_t* row_map, const void* t_logits, int t_dtype, int64_t t_stride,
                               int64_t n_teacher_rows, float inv_T_student, float inv_T_teacher, float grad_scale,
                               float* row_loss, void* grad, int64_t grad_stride, void* workspace, int64_t workspace_bytes,
                               int flags, void* stream) {
  using namespace dl;
  if (!logits || (!t_logits && n_teacher_rows > 0)) return DL_ERR_NULL;      // no teacher rows: every row is masked
  if (kind < DL_FKL || kind > DL_JSD || logits_dtype < DL_F32 || logits_dtype > DL_F16 || t_dtype < DL_F32 ||
      t_dtype > DL_F16)
    return DL_ERR_DTYPE;
  if (n_rows < 0 || V <= 0 || n_teacher_rows < 0 || row_stride < V || t_stride < V || (grad && grad_stride < V))
    return DL_ERR_SHAPE;
  if (n_rows > 0x7fffffffLL || V > 0x7fffffffLL) return DL_ERR_LIMIT;
  if (n_rows == 0) return DL_OK;
  const int sb = logits_dtype == DL_F32 ? 4 : 2, tb = t_dtype == DL_F32 ? 4 : 2;
  auto ok16 = [](const void* ptr, int64_t stride, int eb) {
    return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && (stride * eb) % 16 == 0;
  };
  const bool vec = V % 8 == 0 && ok16(logits, row_stride, sb) && ok16(t_logits, t_stride, tb) &&
                   (!grad || ok16(grad, grad_stride, sb));
  DenseParams p{kind, logits, logits_dtype, row_stride, n_rows, V, row_map, t_logits, t_dtype, t_stride,
                n_teacher_rows, inv_T_student, inv_T_teacher, grad_scale, row_loss, grad, grad_stride};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool elem = reinterpret_cast<uintptr_t>(logits) % sb == 0 && reinterpret_cast<uintptr_t>(t_logits) % tb == 0 &&
                    (!grad || reinterpret_cast<uintptr_t>(grad) % sb == 0);
  if (!elem) return DL_ERR_ALIGN;
  // rows cut into column parts, where a workspace for their exchange came along
  const int hook = (flags >> DL_TOPK_PARTS_SHIFT) & 15;      // 1 / 2: parts of 256 / 512 threads wherever the row can be cut
  const DenseCut cut = dense_split_cut(kind, logits_dtype, t_dtype, n_rows, V, hook == 1 ? 256 : hook == 2 ? 512 : hook == 3 ? 1024 : 0);
  if (cut.parts && workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
      workspace_bytes >= DenseSplit::bytes(kind, n_rows, cut.parts) && n_rows * cut.parts <= 0x7fffffffLL) {
    const DenseSplit x(kind, workspace, n_rows, cut.parts, (flags & DL_TOPK_NO_WAIT) ? 0 : DENSE_SPIN_LIMIT, (V + 7) / 8,
                       (int64_t)cut.nt * dense_split_units(logits_dtype, t_dtype));
    if (vec) launch_dense_split_pair<false>(p, x, cut.nt, st);
    else launch_dense_split_any(p, x, cut.nt, st);
    return hipGetLastError() == hipSuccess ? DL_OK : DL_ERR_LAUNCH;
  }
  if (!(vec ? launch_dense_pair(p, st) : launch_dense_any(p, st)))
    hipLaunchKernelGGL((dense_stream_kernel<1024>), dim3((unsigned)n_rows), dim3(1024), 0, st, p);
  return hipGetLastError() == hipSuccess ? DL_OK : DL_ERR_LAUNCH;
}
