// Kernels for divergences against a dense teacher stored in memory, rows (or column parts of rows) held in registers:
// dense_div.hip instantiates them for rows on the 16-byte grid, dense_div_any.hip for the others.
#pragma once
#include "dense_div.hpp"
#include <algorithm>

namespace dl {

struct DenseParams {
  int kind;
  const void* logits; int s_dtype; int64_t row_stride; int64_t n_rows; int64_t V;
  const int32_t* row_map;
  const void* t_logits; int t_dtype; int64_t t_stride; int64_t n_trows;
  float inv_T_s, inv_T_t, grad_scale;
  float* row_loss; void* grad; int64_t grad_stride;
};

// Both rows in registers: NU units of 8 columns per thread.  ANY: rows that may start on any element, of any length.
// The units then start at the student row's first 16-byte boundary, so that its accesses (and those of the gradient
// and of a teacher row of the same phase: every unmasked row of contiguous tensors) are aligned; where a row's phase
// differs, the same 16-byte accesses are unaligned, which global memory takes.  The columns ahead of the first unit
// (up to 7) and behind the last (up to 7) sit one per thread in the first threads of the workgroup (s_rest / t_rest,
// -inf in the others: adds nothing to any statistic), so that the sweeps over the units are those of aligned rows,
// with no bound inside them and no branch around a load.
// Measured, forward KL: 2044 x 101719 bf16 with a tenth of the rows masked 1391 -> 257 us (101720 columns: 255 us),
// 8192 x 50257 bf16 805 -> 490 us (50264: 488 us), 8192 x 32003 fp32 677 -> 538 us, 2000 x 100277 fp32 against bf16
// 1858 -> 526 us, 5 x 151665 fp16 234 -> 34 us.  (With units from the row's first element the unaligned stores cost
// 308 us on the first of these and 569 on the second; with a bounds check and an element-wise alternative at every
// chunk, as before, each load waited for the one before it.)
// BLOCKED (two fp32 rows): which 8 columns make up a unit is free as long as student, teacher and
// gradient agree, and nothing but the loads and stores ever asks.  A unit of 8 consecutive fp32 columns is two
// chunks side by side, so that a wave's load instruction touches every other 16 bytes: half of each line, and the
// next instruction the other half.  Instead the 128 chunks of 64 consecutive units (one wave's worth) are dealt
// chunk c to lane c % 64, first and second chunk of a unit 64 chunks apart (n apart in a last block of n < 64
// units): every load and store instruction of a wave then covers 1 KiB in one piece.
template <class TagS, class TagT, int NT, int NU, bool ANY = false>
struct RegRows {
  static constexpr bool ONLINE = false;      // sweeps cost no memory traffic: maxima first, then sums
  static constexpr bool CENTRED = ANY;       // reverse KL: gradient about the mean of the log ratios as they are rounded
  static constexpr bool BLOCKED = TagS::bytes == 4 && TagT::bytes == 4;
  Unit<TagS> s[NU];
  Unit<TagT> t[NU];
  int64_t nunits;
  int head, rest;        // ANY: columns ahead of the units, and those plus the ones behind
  float s_rest, t_rest;  // one of them, if tid < rest
  // its number, counted from the first unit's first column
  __device__ __forceinline__ int64_t rest_column() const {
    const int tid = (int)threadIdx.x;
    return tid < head ? (int64_t)(tid - head) : nunits * 8 + (tid - head);
  }
  // byte offset of chunk k of unit u in a BLOCKED row
  __device__ __forceinline__ int64_t blocked_at(int64_t u, int k) const {
    const int64_t b = u >> 6;
    const int64_t nb = min((int64_t)64, nunits - (b << 6));
    return ((b << 7) + k * nb + (u & 63)) * 16;
  }
  // 32-bit offsets behind a uniform base: 64-bit addresses of all loads in flight would cost their registers again
  template <class Tag>
  __device__ __forceinline__ void load_any(Unit<Tag>& x, const char* row, int u) const {
#pragma unroll
    for (int k = 0; k < Unit<Tag>::NC; ++k) {
      const unsigned at = BLOCKED ? (unsigned)blocked_at(u, k) : (unsigned)(u * Unit<Tag>::NC + k) * 16u;
      if constexpr (BLOCKED || Unit<Tag>::NC == 1) x.c[k] = load16_stream_any(row + at);
      else x.c[k] = load16_unaligned(row + at);
    }
  }
  __device__ __forceinline__ void load(const char* srow, const char* trow, int64_t nu, int head_ = 0, int tail_ = 0) {
    nunits = nu;
    head = head_;
    rest = head_ + tail_;
    s_rest = t_rest = -INFINITY;
    if constexpr (ANY) {
      if ((int)threadIdx.x < rest) {
        s_rest = load_as_float(srow, TagS::id, rest_column());
        t_rest = load_as_float(trow, TagT::id, rest_column());
      }
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (u < nunits) {
        if constexpr (ANY) { load_any<TagS>(s[i], srow, (int)u); load_any<TagT>(t[i], trow, (int)u); }
        else if constexpr (BLOCKED) {
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int64_t at = blocked_at(u, k);
            s[i].c[k] = load16_stream(srow + at);
            t[i].c[k] = load16_stream(trow + at);
          }
        }
        else { s[i].load(srow, u); t[i].load(trow, u); }
      } else {
        s[i].fill_neg_inf(); t[i].fill_neg_inf();
      }
    }
  }
  template <class N>
  __device__ __forceinline__ void store(char* grow, int64_t u, const float* g, N) const {
    if constexpr (ANY && N::value == 1) store_from_float(grow, TagS::id, rest_column(), g[0]);
    else if constexpr (ANY) {
#pragma unroll
      for (int k = 0; k < Unit<TagS>::NC; ++k) {
        const unsigned at = BLOCKED ? (unsigned)blocked_at((int)u, k) : (unsigned)((int)u * Unit<TagS>::NC + k) * 16u;
        const u32x4 v = Chunk<TagS>::pack(g + k * Chunk<TagS>::N);
        if constexpr (BLOCKED || Unit<TagS>::NC == 1) store16_stream_any(grow + at, v);
        else store16_unaligned(grow + at, v);
      }
    }
    else if constexpr (BLOCKED) {
#pragma unroll
      for (int k = 0; k < 2; ++k) store16_stream(grow + blocked_at(u, k), Chunk<TagS>::pack(g + k * 4));
    }
    else Unit<TagS>::store(grow, u, g);
  }
  template <class F>
  __device__ __forceinline__ void sweep(F f) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (u < nunits) {
        float a[8], b[8];
        s[i].unpack(a);
        t[i].unpack(b);
        f(u, a, b, Columns<8>{});
      }
    }
    if constexpr (ANY) {
      if ((int)threadIdx.x < rest) {
        float a[1] = {s_rest}, b[1] = {t_rest};
        f(nunits, a, b, Columns<1>{});
      }
    }
  }
  // The same, and what f leaves in its arguments goes back into the registers (fp32 rows: bit moves).
  // The branch is per wave, not per lane (lanes beyond the row hold -inf, which f must take): a value
  // rewritten under a per-lane branch would get a second register beside the one that the idle lanes keep.
  static constexpr bool EXACT_STASH = TagS::bytes == 4 && TagT::bytes == 4;
  template <class F>
  __device__ __forceinline__ void sweep_rewrite(F f) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (__builtin_amdgcn_readfirstlane((int)((u & ~(int64_t)63) < nunits))) {
        float a[8], b[8];
        s[i].unpack(a);
        t[i].unpack(b);
        f(u, a, b, Columns<8>{});
        s[i].repack(a);
        t[i].repack(b);
      }
    }
    if constexpr (ANY) {
      if ((int)threadIdx.x < rest) f(nunits, &s_rest, &t_rest, Columns<1>{});
    }
  }
  // JSD on the other pairs: the divergence sweep keeps a column's log ratio to the mixture, in fp32, for the gradient: in the
  // teacher's registers where those are fp32, else in registers of its own (a 16-bit teacher's are then free).
  static constexpr bool RATIO_STASH = !EXACT_STASH, RATIO_IN_T = TagT::bytes == 4;
  float ratio[RATIO_STASH && !RATIO_IN_T ? NU : 1][8];
  float ratio_rest;
  // f(s, t, d): sets d, the values to keep (per wave, as sweep_rewrite)
  template <class F>
  __device__ __forceinline__ void sweep_keep(F f) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (__builtin_amdgcn_readfirstlane((int)((u & ~(int64_t)63) < nunits))) {
        float a[8], b[8], d[8];
        s[i].unpack(a);
        t[i].unpack(b);
        f(a, b, d, Columns<8>{});
        if constexpr (RATIO_IN_T) t[i].repack(d);
        else {
#pragma unroll
          for (int e = 0; e < 8; ++e) ratio[i][e] = d[e];
        }
      }
    }
    if constexpr (ANY) {
      if ((int)threadIdx.x < rest) f(&s_rest, &t_rest, &ratio_rest, Columns<1>{});
    }
  }
  // f(u, s, d): the kept values beside the student's
  template <class F>
  __device__ __forceinline__ void sweep_kept(F f) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int64_t u = (int64_t)i * NT + threadIdx.x;
      if (u < nunits) {
        float a[8], d[8];
        s[i].unpack(a);
        if constexpr (RATIO_IN_T) t[i].unpack(d);
        else {
#pragma unroll
          for (int e = 0; e < 8; ++e) d[e] = ratio[i][e];
        }
        f(u, a, d, Columns<8>{});
      }
    }
    if constexpr (ANY) {
      if ((int)threadIdx.x < rest) f(nunits, &s_rest, &ratio_rest, Columns<1>{});
    }
  }
  // Maxima of both rows from the raw bit patterns, for two 16-bit rows: non-negative 16-bit floats
  // order like their patterns read as signed integers and every negative one reads as a negative
  // integer, so the packed integer maximum is the row's maximum whenever that is not negative (half
  // an instruction per element instead of two).  False -- for every thread alike -- when a row's
  // maximum is negative or the types are not 16-bit: the caller then takes the maxima from the values.
  static constexpr bool RAW_MAXIMA = TagS::bytes == 2 && TagT::bytes == 2;
  static __device__ __forceinline__ int raw_of(int id, float v) {      // the 16-bit pattern of v, which is exact in it, as a signed integer
    return id == BF16 ? __float_as_int(v) >> 16 : (int)__builtin_bit_cast(short, (_Float16)v);
  }
  __device__ __forceinline__ bool raw_maxima(float& ms, float& mt, float* red) {
    if constexpr (!RAW_MAXIMA) return false;
    typedef short i16x2 __attribute__((ext_vector_type(2)));
    i16x2 a = {(short)-32768, (short)-32768}, b = a;
#pragma unroll
    for (int i = 0; i < NU; ++i) {      // units beyond the row hold -inf: negative patterns
      forget(s[i].c[0]);
      forget(t[i].c[0]);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const unsigned ws = s[i].c[0][d], wt = t[i].c[0][d];      // by value: a bit cast straight from a vector element reads element 0
        a = __builtin_elementwise_max(a, __builtin_bit_cast(i16x2, ws));
        b = __builtin_elementwise_max(b, __builtin_bit_cast(i16x2, wt));
      }
    }
    int ia = max((int)a.x, (int)a.y), ib = max((int)b.x, (int)b.y);
    if constexpr (ANY) {                // -inf where the thread holds no such column
      ia = max(ia, raw_of(TagS::id, s_rest));
      ib = max(ib, raw_of(TagT::id, t_rest));
    }
    float fa = (float)ia, fb = (float)ib;      // exact, order-preserving
    block_max2<NT>(fa, fb, red);
    if (fa < 0.f || fb < 0.f) return false;
    const auto value = [](int id, unsigned bits) {
      return id == BF16 ? __uint_as_float(bits << 16) : (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
    };
    ms = value(TagS::id, (unsigned)(int)fa);
    mt = value(TagT::id, (unsigned)(int)fb);
    return true;
  }
};

// What JSD keeps of its divergence sweep for the gradient (see dense_stats).
template <class Rows, bool GRAD>
constexpr int JSD_KEEP = Rows::EXACT_STASH ? JSD_KEEP_BOTH : GRAD ? JSD_KEEP_RATIO : JSD_KEEP_NOTHING;

// JSD with a gradient: four waves per SIMD are asked for (128 registers): with the kept ratios the 16-bit pairs off the grid
// would take a few more, one workgroup fewer per CU (8192 x 32100 bf16: 386 us against 252).  The instances of 1024 threads
// for 16-bit pairs spill 5 to 7 registers so, those of 512 off the grid and the column parts of 512 one or two (8 to 32 bytes
// a lane); with the ratios made again they took 108 and none, and 8 to 15 % longer (128 x 50257 bf16 25.4 -> 23.4 us, 512 x
// 40960 45.7 -> 43.8, 4096 x 65536 411 -> 354).  GRAD = false: a call without a
// gradient, for which nothing is kept (JSD only: what a call's gradient costs the other kinds is a branch).
template <int KIND, class TagS, class TagT, int NT, int NU, bool ANY = false, bool GRAD = true>
__global__ __launch_bounds__(NT, KIND == DL_JSD && GRAD ? 4 : 1) void dense_reg_kernel(const DenseParams p) {
  __shared__ float red[64];
  const int64_t r = xcd_banded_row(blockIdx.x);
  if (r >= p.n_rows) return;
  const int tid = threadIdx.x;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * TagS::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  if (trow < 0) {
    if (grow) {
      if constexpr (ANY) zero_row_any<TagS, NT>(grow, p.V);
      else zero_row<TagS, NT>(grow, p.V / TagS::epc);
    }
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  RegRows<TagS, TagT, NT, NU, ANY> rows;
  const char* srow = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * TagS::bytes;
  const char* tl = reinterpret_cast<const char*>(p.t_logits) + trow * p.t_stride * TagT::bytes;
  const int head = ANY ? elements_to_grid<TagS>(srow, p.V) : 0;
  const int64_t nunits = (p.V - head) / 8;
  rows.load(srow + head * TagS::bytes, tl + head * TagT::bytes, nunits, head, ANY ? (int)(p.V - head - nunits * 8) : 0);
  if (ANY && grow) grow += head * TagS::bytes;
  if constexpr (KIND == DL_JSD) {
    constexpr int KEEP = JSD_KEEP<RegRows<TagS, TagT, NT, NU, ANY>, GRAD>;
    const DenseStats st = dense_stats<KIND, NT, KEEP>(rows, p.inv_T_s, p.inv_T_t, red);
    if (tid == 0 && p.row_loss) p.row_loss[r] = st.loss;
    if (GRAD && grow) dense_jsd_grad_kept<KEEP, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
  } else {
    const DenseStats st = dense_stats<KIND, NT>(rows, p.inv_T_s, p.inv_T_t, red);
    if (tid == 0 && p.row_loss) p.row_loss[r] = st.loss;
    if (grow) dense_grad_sweep<KIND, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
  }
}

// One launch over rows that NT threads hold whole.  JSD of pairs that keep the log ratio: without a gradient the kernel that
// keeps nothing (2048 x 12000 fp32 against bf16 32.5 us with the ratios kept, 29.2 without; 512 x 50257 bf16 42.5, 40.5).
template <int KIND, class TagS, class TagT, int NT, int NU, bool ANY>
static void launch_dense_reg_nt(const DenseParams& p, hipStream_t st) {
  const dim3 grid(xcd_banded_grid(p.n_rows)), block(NT);
  if constexpr (KIND == DL_JSD && RegRows<TagS, TagT, NT, NU, ANY>::RATIO_STASH) {
    if (!p.grad) {
      hipLaunchKernelGGL((dense_reg_kernel<KIND, TagS, TagT, NT, NU, ANY, false>), grid, block, 0, st, p);
      return;
    }
  }
  hipLaunchKernelGGL((dense_reg_kernel<KIND, TagS, TagT, NT, NU, ANY>), grid, block, 0, st, p);
}

// ---------------------------------------------------------------------------------------
// Rows cut into column parts.  A workgroup that holds a whole pair of rows is
// 512 or 1024 threads wide, so one or two of them fill a CU and nothing overlaps their load,
// arithmetic and store phases.  Here a row pair is cut into P <= 8 parts of 256 (or 512) threads x NU units
// instead; four (two) parts of different rows share a CU and hide each other's phases, and each part still
// reads its columns once.  The parts of a row exchange (maxima, sums of exponentials, divergence sum on the part's
// own biases) through a 32-byte record per part in a caller-provided workspace: relaxed device-scope stores
// and loads, validated by a tag over the five words; the wait is bounded, and a part that gives up -- it has
// written nothing yet, also when the gradient goes over the logits -- puts itself on a list that a second
// launch finishes from the then complete records.  Every part combines the records in part order: all parts
// of a row arrive at the same bits, and so does the second launch.  Parts of a row sit 8 workgroup ids
// apart, i.e. on one XCD back to back.
// JSD needs the row's normalisers inside a logarithm, and the divergence again in its gradient: its parts meet a second
// time, over (KL(P || M), KL(Q || M)) of their columns, in a second record each.  A part that gave up at either meeting is
// finished by two launches: the first makes the second records of all listed parts, the second finds every record complete.
// Those two keep nothing for the gradient: their body is a real call, and with the ratios its stack grew from 192 to 268
// bytes a lane.  The runtime gives a queue scratch for the largest it has met, and every launch that uses any then waits
// longer: with them in a process, all calls that cut rows, of any pair, took 4 us more (64 x 50257 fp32 26.3 -> 30.2).
// Against streaming such rows from memory (four scalar passes off the 16-byte grid): 4013 x 98922 bf16 against fp32
// 3600 -> 897 us, 327 x 125715 fp32 against bf16 428 -> 143 us, 4096 x 128256 bf16 1064 -> 916 us.
// ---------------------------------------------------------------------------------------
struct DenseRecord { unsigned ms, mt, ss, st, w, tag, pad0, pad1; };
constexpr int DENSE_MAX_PARTS = 8;
constexpr int DENSE_SPIN_LIMIT = 20000;

struct DenseSplit {
  DenseRecord* records;      // n_rows * parts
  DenseRecord* second;       // JSD: n_rows * parts more, right behind
  unsigned* retry_count;     // then a counter (16 bytes) and n_rows * parts list slots
  unsigned* retry_list;
  int parts;
  int spin_limit;
  int64_t part_units;        // units of 8 columns per part (the last part takes what is left)
  static int64_t n_records(int kind, int64_t n_rows, int parts) { return n_rows * parts * (kind == DL_JSD ? 2 : 1); }
  static int64_t bytes(int kind, int64_t n_rows, int parts) {
    return n_records(kind, n_rows, parts) * (int64_t)sizeof(DenseRecord) + n_rows * parts * 4 + 16;
  }
  // The row is cut evenly, in whole waves of units: a last part that holds a few columns would still take a
  // workgroup, and its partners would wait for it like for a full one.
  DenseSplit(int kind, void* ws, int64_t n_rows, int parts_, int spin, int64_t units, int64_t most_units) {
    part_units = ((units + parts_ - 1) / parts_ + 63) / 64 * 64;
    if (part_units > most_units || (parts_ - 1) * part_units >= units) part_units = most_units;
    records = reinterpret_cast<DenseRecord*>(ws);
    second = records + n_rows * parts_;
    char* base = reinterpret_cast<char*>(ws) + n_records(kind, n_rows, parts_) * (int64_t)sizeof(DenseRecord);
    retry_count = reinterpret_cast<unsigned*>(base);
    retry_list = reinterpret_cast<unsigned*>(base + 16);
    parts = parts_;
    spin_limit = spin;
  }
};

__device__ __forceinline__ unsigned dense_record_tag(unsigned a, unsigned b, unsigned c, unsigned d, unsigned e) {
  return a ^ ((b << 5) | (b >> 27)) ^ ((c << 11) | (c >> 21)) ^ ((d << 17) | (d >> 15)) ^ ((e << 23) | (e >> 9)) ^ 0x5eed4321u;
}
__device__ __forceinline__ void dense_record_publish(DenseRecord* w, float ms, float mt, float ss, float st, float wv) {
  const unsigned a = __float_as_uint(ms), b = __float_as_uint(mt), c = __float_as_uint(ss), d = __float_as_uint(st),
                 e = __float_as_uint(wv);
  __hip_atomic_store(&w->ms, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->mt, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->ss, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->st, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->w, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->tag, dense_record_tag(a, b, c, d, e), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Bounded wait for a partner's record; false = gave up after `limit` polls.  A cleared record is invalid.
__device__ __forceinline__ bool dense_record_collect(DenseRecord* w, int limit, float* out) {
  for (int spins = 0; spins < limit; ++spins) {
    const unsigned a = __hip_atomic_load(&w->ms, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned b = __hip_atomic_load(&w->mt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned c = __hip_atomic_load(&w->ss, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned d = __hip_atomic_load(&w->st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned e = __hip_atomic_load(&w->w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned t = __hip_atomic_load(&w->tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t == dense_record_tag(a, b, c, d, e)) {
      out[0] = __uint_as_float(a); out[1] = __uint_as_float(b); out[2] = __uint_as_float(c);
      out[3] = __uint_as_float(d); out[4] = __uint_as_float(e);
      return true;
    }
    __builtin_amdgcn_s_sleep(4);
  }
  return false;
}

// Publishes this part's record `w` (fresh) and collects the others' into xch; false (for every thread alike): a partner did
// not answer in time, the part has put itself on the list.
__device__ __forceinline__ bool dense_exchange(const DenseSplit& x, DenseRecord* ws, int64_t r, int h, bool publish, int limit,
                                               const float (&mine)[5], float (*xch)[DENSE_MAX_PARTS], int* xok) {
  const int tid = threadIdx.x, P = x.parts;
  if (tid == 0 && publish) dense_record_publish(ws + h, mine[0], mine[1], mine[2], mine[3], mine[4]);
  if (tid < P) {
    float rec[5] = {mine[0], mine[1], mine[2], mine[3], mine[4]};
    const int ok = (tid == h) || dense_record_collect(ws + tid, limit, rec);
#pragma unroll
    for (int k = 0; k < 5; ++k) xch[k][tid] = rec[k];
    xok[tid] = ok;
  }
  __syncthreads();
  bool all_ok = true;
  for (int j = 0; j < P; ++j) all_ok = all_ok && (xok[j] != 0);
  if (!all_ok && tid == 0) x.retry_list[atomicAdd(x.retry_count, 1u)] = (unsigned)(r * P + h);
  return all_ok;
}

// RETRY: SPLIT_FIRST the launch over all parts; SPLIT_FINISH over the listed ones, every record complete; SPLIT_SECOND
// (JSD) over the listed ones before that, up to their second record.
constexpr int SPLIT_FIRST = 0, SPLIT_FINISH = 1, SPLIT_SECOND = 2;

template <int KIND, class TagS, class TagT, int NT, int NU, int RETRY, bool ANY, bool GRAD>
__device__ __forceinline__ void dense_split_part(const DenseParams& p, const DenseSplit& x, int64_t r, int h, float* red,
                                                 float (*xch)[DENSE_MAX_PARTS], int* xok) {
  const int tid = threadIdx.x;
  const int P = x.parts;
  const int64_t u0 = (int64_t)h * x.part_units;                        // first unit of this part
  const char* srow = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * TagS::bytes;
  const int lead = ANY ? elements_to_grid<TagS>(srow, p.V) : 0;         // columns ahead of the row's first unit
  const int64_t row_units = (p.V - lead) / 8;
  const int64_t nu = max((int64_t)0, min(x.part_units, row_units - u0)); // its units
  const int head = h == 0 ? lead : 0;                                   // and its columns ahead of them and behind
  const int tail = ANY && h == P - 1 ? (int)(p.V - lead - row_units * 8) : 0;
  const int64_t first = lead + min(u0, row_units) * 8;                  // column of the first unit
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + (r * p.grad_stride + first) * TagS::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  if (trow < 0) {
    if (grow) {
      if constexpr (ANY) zero_row_any<TagS, NT>(grow - head * TagS::bytes, head + nu * 8 + tail);
      else zero_row<TagS, NT>(grow, nu * 8 / TagS::epc);
    }
    if (tid == 0 && h == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  using Rows = RegRows<TagS, TagT, NT, NU, ANY>;
  constexpr int KEEP = JSD_KEEP<Rows, GRAD && RETRY == SPLIT_FIRST>;
  Rows rows;
  rows.load(srow + first * TagS::bytes, reinterpret_cast<const char*>(p.t_logits) + (trow * p.t_stride + first) * TagT::bytes, nu,
            head, tail);
  const float a_s = p.inv_T_s * LOG2E, a_t = p.inv_T_t * LOG2E;
  float ms = -INFINITY, mt = -INFINITY;
  bool have = false;
  if constexpr (KIND != DL_RKL && Rows::RAW_MAXIMA) have = rows.raw_maxima(ms, mt, red);
  if (!have) {
    rows.sweep([&](int64_t, const float* s, const float* t, auto n) {
#pragma unroll
      for (int e = 0; e < decltype(n)::value; ++e) {
        mt = fmaxf(mt, t[e]);
        ms = fmaxf(ms, (KIND == DL_RKL && t[e] == -INFINITY) ? -INFINITY : s[e]);
      }
    });
    block_max2<NT>(ms, mt, red);
  }
  // A part that holds no finite logit (a masked stretch of the vocabulary): bias 0 keeps 2^(-inf - bias) = 0.  One masked
  // with the lowest value of its type or nearly so counts as such (MASKED_BELOW).
  if (ms * a_s < MASKED_BELOW) ms = -INFINITY;
  if (mt * a_t < MASKED_BELOW) mt = -INFINITY;
  const float bs = ms == -INFINITY ? 0.f : ms * a_s, bt = mt == -INFINITY ? 0.f : mt * a_t;
  float ss = 0.f, stt = 0.f, w = 0.f;
  rows.sweep([&](int64_t, const float* s, const float* t, auto n) {
#pragma unroll
    for (int e = 0; e < decltype(n)::value; ++e) {
      const float xs = fmaf(s[e], a_s, -bs), xt = fmaf(t[e], a_t, -bt);
      const float es = fast_exp2(xs), et = fast_exp2(xt);
      stt += et;
      if (KIND == DL_RKL) {
        const bool on = t[e] != -INFINITY;
        ss += on ? es : 0.f;
        w += (on && es > 0.f) ? es * (xs - xt) : 0.f;
      } else {
        ss += es;
        if (KIND == DL_FKL) w += et > 0.f ? et * (xt - xs) : 0.f;
      }
    }
  });
  if constexpr (KIND == DL_JSD) block_sum2<NT>(ss, stt, red);
  else block_sum3<NT>(ss, stt, w, red);

  const int limit = RETRY == SPLIT_FIRST ? x.spin_limit : 0x7fffffff;
  if (!dense_exchange(x, x.records + r * P, r, h, RETRY == SPLIT_FIRST, limit, {ms, mt, ss, stt, w}, xch, xok)) return;
  // the row's statistics from the parts', in part order (the same bits in every part)
  float Ms = xch[0][0], Mt = xch[1][0];
  for (int j = 1; j < P; ++j) { Ms = fmaxf(Ms, xch[0][j]); Mt = fmaxf(Mt, xch[1][j]); }
  float S = 0.f, T = 0.f, W = 0.f;
  for (int j = 0; j < P; ++j) {
    const float pms = xch[0][j], pmt = xch[1][j], pss = xch[2][j], pst = xch[3][j];
    // shifts of the part's biases to the row's (log2 domain, >= 0); a part without a finite maximum summed nothing on that
    // side (and where the other side has mass there, its terms are those of logits below MASKED_BELOW: their bias is nothing to them)
    float ds, dt;
    if constexpr (KIND == DL_RKL && Rows::CENTRED) {
      ds = pms == -INFINITY ? 0.f : Ms * a_s - pms * a_s;
      dt = pmt == -INFINITY ? 0.f : Mt * a_t - pmt * a_t;
    } else {
      ds = pms == -INFINITY ? 0.f : (Ms - pms) * a_s;
      dt = pmt == -INFINITY ? 0.f : (Mt - pmt) * a_t;
    }
    const float fs = fast_exp2(-ds), ft = fast_exp2(-dt);
    // a part whose mass is nothing to the row's adds nothing, whatever the other side's logits are there
    const float pw = (KIND == DL_FKL ? ft : fs) > 0.f ? xch[4][j] : 0.f;
    if (KIND == DL_FKL) W += ft * (pw - (dt - ds) * pst);
    if (KIND == DL_RKL) W += fs * (pw - (ds - dt) * pss);
    S += pss * fs;
    T += pst * ft;
  }
  DenseStats st;
  st.a_s = a_s; st.a_t = a_t;
  const float l2s = fast_log2(S), l2t = fast_log2(T);
  st.ls = (Ms == -INFINITY ? 0.f : Ms * a_s) + l2s;
  st.lt = (Mt == -INFINITY ? 0.f : Mt * a_t) + l2t;
  st.tmax = Mt;
  if constexpr (KIND == DL_JSD) {
    float kp = 0.f, kq = 0.f;
    dense_jsd_sums<KEEP>(rows, st, kp, kq);
    block_sum2<NT>(kp, kq, red);
    DenseRecord* ws2 = x.second + r * P;
    if (RETRY == SPLIT_SECOND) {
      if (tid == 0) dense_record_publish(ws2 + h, kp, kq, 0.f, 0.f, 0.f);
      return;
    }
    __syncthreads();      // the first meeting's records have been read
    if (!dense_exchange(x, ws2, r, h, RETRY == SPLIT_FIRST, limit, {kp, kq, 0.f, 0.f, 0.f}, xch, xok)) return;
    float X = 0.f, Y = 0.f;
    for (int j = 0; j < P; ++j) { X += xch[0][j]; Y += xch[1][j]; }
    st.loss = 0.5f * LN2 * (X + Y);
    st.aux = X * LN2;
  } else {
    st.loss = (KIND == DL_FKL ? W / T - l2t + l2s : W / S - l2s + l2t) * LN2;
    st.aux = KIND == DL_RKL && Rows::CENTRED ? rkl_centre(W / S, st, Ms * a_s, Mt * a_t) : st.loss;
  }
  if (tid == 0 && h == 0 && p.row_loss) p.row_loss[r] = st.loss;
  if (GRAD && grow) {
    if constexpr (KIND == DL_JSD && KEEP != JSD_KEEP_NOTHING) dense_jsd_grad_kept<KEEP, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
    else dense_grad_sweep<KIND, TagS>(rows, st, p.inv_T_s * p.grad_scale, grow);
  }
}

template <int KIND, class TagS, class TagT, int NT, int NU, bool ANY, bool GRAD = true>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
void dense_split_kernel(const DenseParams p, const DenseSplit x) {
  __shared__ float red[64];
  __shared__ float xch[5][DENSE_MAX_PARTS];
  __shared__ int xok[DENSE_MAX_PARTS];
  const unsigned P = (unsigned)x.parts;
  const unsigned grp = blockIdx.x / (8u * P), t_in = blockIdx.x % (8u * P);
  const int64_t r = (int64_t)grp * 8 + (t_in & 7u);
  if (r >= p.n_rows) return;
  dense_split_part<KIND, TagS, TagT, NT, NU, SPLIT_FIRST, ANY, GRAD>(p, x, r, (int)(t_in >> 3), red, xch, xok);
}

// One listed part, as a real call: the loop around it then costs the body no registers.
template <int KIND, class TagS, class TagT, int NT, int NU, int RETRY, bool ANY>
__device__ __attribute__((noinline)) void dense_split_part_again(const DenseParams& p, const DenseSplit& x, unsigned at, float* red,
                                                                 float (*xch)[DENSE_MAX_PARTS], int* xok) {
  dense_split_part<KIND, TagS, TagT, NT, NU, RETRY, ANY, true>(p, x, (int64_t)(at / (unsigned)x.parts), (int)(at % (unsigned)x.parts), red, xch, xok);
}

// The parts that gave up waiting, a fixed grid striding over their list (normally empty).
template <int KIND, class TagS, class TagT, int NT, int NU, int RETRY, bool ANY>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
void dense_split_retry_kernel(const DenseParams p, const DenseSplit x) {
  __shared__ float red[64];
  __shared__ float xch[5][DENSE_MAX_PARTS];
  __shared__ int xok[DENSE_MAX_PARTS];
  const unsigned n = *x.retry_count;
#pragma unroll 1
  for (unsigned e = blockIdx.x; e < n; e += gridDim.x) {
    dense_split_part_again<KIND, TagS, TagT, NT, NU, RETRY, ANY>(p, x, x.retry_list[e], red, xch, xok);
    __syncthreads();
  }
}

template <int NT>
__global__ __launch_bounds__(NT) void dense_clear_kernel(u32x4* ws, int64_t n16) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i < n16) ws[i] = u32x4{0u, 0u, 0u, 0u};
}

template <int KIND, class TagS, class TagT, int NT, int NU, bool ANY>
static void launch_dense_split_kind(const DenseParams& p, const DenseSplit& x, hipStream_t st) {
  const int64_t n16 = DenseSplit::n_records(KIND, p.n_rows, x.parts) * 2 + 1;      // records, then the retry counter
  hipLaunchKernelGGL((dense_clear_kernel<256>), dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st,
                     reinterpret_cast<u32x4*>(x.records), n16);
  const dim3 grid((unsigned)((p.n_rows + 7) / 8 * 8 * x.parts));
  constexpr bool KEEPS = KIND == DL_JSD && RegRows<TagS, TagT, NT, NU, ANY>::RATIO_STASH;      // see launch_dense_reg_nt
  if (KEEPS && !p.grad) hipLaunchKernelGGL((dense_split_kernel<KIND, TagS, TagT, NT, NU, ANY, !KEEPS>), grid, dim3(NT), 0, st, p, x);
  else hipLaunchKernelGGL((dense_split_kernel<KIND, TagS, TagT, NT, NU, ANY>), grid, dim3(NT), 0, st, p, x);
  const dim3 again((unsigned)std::min<int64_t>(p.n_rows * x.parts, 256));
  if constexpr (KIND == DL_JSD)
    hipLaunchKernelGGL((dense_split_retry_kernel<KIND, TagS, TagT, NT, NU, SPLIT_SECOND, ANY>), again, dim3(NT), 0, st, p, x);
  hipLaunchKernelGGL((dense_split_retry_kernel<KIND, TagS, TagT, NT, NU, SPLIT_FINISH, ANY>), again, dim3(NT), 0, st, p, x);
}
template <class TagS, class TagT, int NT, int NU, bool ANY>
static void launch_dense_split_nt(const DenseParams& p, const DenseSplit& x, hipStream_t st) {
  if (p.kind == DL_FKL) launch_dense_split_kind<DL_FKL, TagS, TagT, NT, NU, ANY>(p, x, st);
  else if (p.kind == DL_RKL) launch_dense_split_kind<DL_RKL, TagS, TagT, NT, NU, ANY>(p, x, st);
  else launch_dense_split_kind<DL_JSD, TagS, TagT, NT, NU, ANY>(p, x, st);
}
template <class TagS, class TagT, int NU, bool ANY>
static void launch_dense_split(const DenseParams& p, const DenseSplit& x, int nt, hipStream_t st) {
  if (nt == 256) launch_dense_split_nt<TagS, TagT, 256, NU, ANY>(p, x, st);
  else if (nt == 512) launch_dense_split_nt<TagS, TagT, 512, NU, ANY>(p, x, st);
  else if constexpr (TagT::bytes == 4 || TagS::bytes == 4) launch_dense_split_nt<TagS, TagT, 1024, NU, ANY>(p, x, st);      // 16-bit pairs reach 262144 columns with parts of 512 threads
}
template <bool ANY>
static void launch_dense_split_pair(const DenseParams& p, const DenseSplit& x, int nt, hipStream_t st) {
  if (p.s_dtype == F32 && p.t_dtype == F32) launch_dense_split<TagF32, TagF32, 4, ANY>(p, x, nt, st);
  else if (p.s_dtype == BF16 && p.t_dtype == BF16) launch_dense_split<TagBF16, TagBF16, 8, ANY>(p, x, nt, st);
  else if (p.s_dtype == F16 && p.t_dtype == F16) launch_dense_split<TagF16, TagF16, 8, ANY>(p, x, nt, st);
  else if (p.s_dtype == BF16 && p.t_dtype == F32) launch_dense_split<TagBF16, TagF32, 6, ANY>(p, x, nt, st);
  else if (p.s_dtype == F16 && p.t_dtype == F32) launch_dense_split<TagF16, TagF32, 6, ANY>(p, x, nt, st);
  else if (p.s_dtype == F32 && p.t_dtype == BF16) launch_dense_split<TagF32, TagBF16, 4, ANY>(p, x, nt, st);
  else launch_dense_split<TagF32, TagF16, 4, ANY>(p, x, nt, st);
}

// Rows off the 16-byte grid or not a whole number of units long (V >= 8), for every dtype pair that has register
// kernels (dense_div_any.hip).  launch_dense_any: one workgroup per row; false where no workgroup holds the pair.
bool launch_dense_any(const DenseParams& p, hipStream_t st);
void launch_dense_split_any(const DenseParams& p, const DenseSplit& x, int nt, hipStream_t st);

}  // namespace dl
