// Forward / reverse KL against a sparse (top-K) teacher: loss and gradient in one sweep.
//
// Forward KL needs the full-vocabulary log-sum-exp of the student row, so the row is pulled
// into registers with 16-byte non-temporal loads (read from HBM once), reduced, and the gradient
//     d kl / d logit_j = (softmax(z)_j - sum_k q_k [j == idx_k]) * inv_T * scale
// is produced from the same registers: a dense softmax sweep, then K sparse corrections after a
// workgroup barrier.  The K teacher entries (id, log-prob, gathered student logit) live in LDS.
//
// A 128256-entry bf16 row is 250 KB, half of a CU's register file, so a workgroup that holds a
// whole row runs alone on its CU and its load / arithmetic / store phases cannot overlap.  The
// split kernel therefore cuts a row into P column parts, one workgroup each; several parts of
// different rows share a CU and hide each other's phases.  The parts of a row exchange their
// (max, sum-exp, partial loss) through a small workspace in global memory; the wait on the
// partner is bounded, and a part that gives up recomputes the row statistics on its own.
//
// Reverse KL (student renormalised over the K ids) touches only the K gathered logits; its
// gradient row is a zero fill plus K sparse values.
//
// Rows that do not fit take the streaming kernel, which reads the row twice.
// This header holds the kernels and their launchers; topk_div.hip instantiates them for one stored
// teacher (dl_div_topk), topk_multi.hip for several unmerged teachers (dl_fkl_multi_teacher).
#pragma once
#include "distill_common.hpp"
#include "distill_hip.h"
#include <algorithm>

namespace dl {

// Several teachers handed over unmerged (dl_fkl_multi_teacher): teacher j holds Kt entries per row in
// val[j] / idx[j]; an entry's mass is exp(val + logw[j]); its id goes through id_map (teacher id ->
// student id, negative = dropped).
struct MultiTeacher {
  int n; int Kt;
  const void* val[DL_MAX_TEACHERS]; const void* idx[DL_MAX_TEACHERS];
  float logw[DL_MAX_TEACHERS];
  const int32_t* id_map; int64_t Vt;
};

// The same teachers prepared for the loss kernels (multi_prep_kernel): per teacher row the surviving
// entries as (student id, log of the renormalised mass), dealt into one bucket per column part of
// the loss kernel's row split, in stored order (teacher 0 first).  Bucket h of a row holds its first
// `cap0` entries in first[(row * parts + h) * cap0 ...] -- the part's workgroup fetches all cap0 slots
// by lane before it knows the count, and keeps what lies below it: the slots behind are never written
// -- and whatever exceeds cap0 in the row's share of `more`, buckets back to back.  head[row * 16 + h] = entries of bucket h (h < 8),
// [8] = entries of the row, [9] = float bits of the sum of the renormalised masses (1 up to rounding).
struct TeacherBuckets {
  const uint2* first; const uint2* more; const int* head;
  int cap0; int E;
};

struct TopkParams {
  const void* logits; int64_t row_stride; int64_t n_rows; int64_t V;
  const int32_t* row_map;
  const void* t_val; int t_val_dtype; const void* t_idx; int t_idx_itype; int K;
  int64_t n_trows; const int32_t* t_cnt;
  float inv_T_s, inv_T_t, grad_scale;
  float* row_loss; void* grad; int64_t grad_stride;
  void* workspace; int parts; int spin_limit; int flags;
  TeacherBuckets bk;    // MULTI kernels only; K is then the number of entries a bucket may hold, rounded up to whole slots
};

constexpr int MAX_PARTS = 16;             // parts a row may be cut into (parts of 256 x 4 chunks)
constexpr int MAX_COARSE_PARTS = 8;       // of 256 x 16 chunks
constexpr int REST_HEADS = 16;            // a part has up to 7 columns ahead of its first 16-byte boundary and 7 behind its last

// What one part of a split row tells the others: three floats and a tag that depends on all of
// them.  The four words are written and read with relaxed device-scope accesses (they bypass the
// non-coherent cache levels; no cache-wide flush or invalidate); a reader accepts a record only
// when the tag matches, so no ordering between the words is needed.  A cleared record is invalid.
struct PartStats { unsigned m, s, b, tag; };
__device__ __forceinline__ unsigned part_tag(unsigned m, unsigned s, unsigned b) {
  return m ^ ((s << 7) | (s >> 25)) ^ ((b << 13) | (b >> 19)) ^ 0x5eed1234u;
}
__device__ __forceinline__ void part_publish(PartStats* w, float m, float s, float b) {
  const unsigned um = __float_as_uint(m), us = __float_as_uint(s), ub = __float_as_uint(b);
  __hip_atomic_store(&w->m, um, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->s, us, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->b, ub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&w->tag, part_tag(um, us, ub), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Bounded wait for a partner's record; false = gave up after `limit` polls.
__device__ __forceinline__ bool part_collect(PartStats* w, int limit, float& m, float& s, float& b) {
  for (int spins = 0; spins < limit; ++spins) {
    const unsigned um = __hip_atomic_load(&w->m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned us = __hip_atomic_load(&w->s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned ub = __hip_atomic_load(&w->b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned ut = __hip_atomic_load(&w->tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (ut == part_tag(um, us, ub)) {
      m = __uint_as_float(um); s = __uint_as_float(us); b = __uint_as_float(ub);
      return true;
    }
    __builtin_amdgcn_s_sleep(4);
  }
  return false;
}

// Workspace of a split launch: n_rows * parts records, then a counter and the list of (row, part)
// numbers that gave up waiting for a partner and are finished by a second launch.
struct RetryList {
  unsigned* count;
  unsigned* entries;
  __host__ __device__ RetryList(void* workspace, int64_t n_rows, int parts) {
    char* base = reinterpret_cast<char*>(workspace) + n_rows * parts * (int64_t)sizeof(PartStats);
    count = reinterpret_cast<unsigned*>(base);
    entries = reinterpret_cast<unsigned*>(base + 16);
  }
  __host__ __device__ static int64_t bytes(int64_t n_rows, int parts) {
    return n_rows * parts * (int64_t)(sizeof(PartStats) + 4) + 16;
  }
};

// LDS carve-up shared by the kernels of this file.  The id array is padded to a multiple of 16
// with -1 so that it can be scanned four ids per read.
struct TopkLds {
  float* red;        // reduction scratch, 64 floats
  float* xm; float* xs; float* xb; int* xok;    // per-part statistics of a split row, MAX_PARTS each
  int* idx;          // Kp  vocabulary id or -1
  float* t;          // Kp  scaled teacher logit -> teacher log-probability over the K entries
  float* q;          // Kp  teacher probability
  float* z;          // Kp  gathered student logit
  // in-register corrections (kernels that keep the row in registers; owners == 0 elsewhere):
  float* val;        // Kp  final gradient value at the entry's column
  int* next;         // Kp  next entry owned by the same thread, or -1
  int* head;         // CORRECTION_HEADS list heads: first entry of a chunk's list, or -1
  unsigned* own;     // one per thread: bit i set = chunk i of the thread holds an entry
  int* rest;         // REST_HEADS list heads: entries on the part's columns beside its 16-byte chunks (ROWS_ANY)
  int Kp;
  __device__ TopkLds(unsigned char* base, int K, int owners = 0) {
    Kp = (K + 15) & ~15;
    red = reinterpret_cast<float*>(base);
    xm = red + 64; xs = xm + MAX_PARTS; xb = xs + MAX_PARTS; xok = reinterpret_cast<int*>(xb + MAX_PARTS);
    idx = reinterpret_cast<int*>(base + 512);
    t = reinterpret_cast<float*>(idx + Kp);
    q = t + Kp;
    z = q + Kp;
    val = z + Kp;
    next = reinterpret_cast<int*>(val + Kp);
    head = next + Kp;
    own = reinterpret_cast<unsigned*>(head + (owners ? CORRECTION_HEADS : 0));
    rest = reinterpret_cast<int*>(own + owners);
  }
  __host__ __device__ static size_t bytes(int K, int owners = 0) {
    const size_t Kp = (size_t)((K + 15) & ~15);
    return 512 + Kp * 16 + (owners ? Kp * 8 + (size_t)CORRECTION_HEADS * 4 + (size_t)owners * 4 + REST_HEADS * 4 : 0);
  }
};

// Teacher entries of one row held in registers between issue and use: J entries per thread,
// entry k = tid + j * NT.  Issuing their (tiny) loads before the row's 16 big ones, and the
// dependent gathers right behind those, keeps three global-memory latencies off the critical path.
template <int J>
struct TeacherEntries {
  int id[J];
  float tv[J];
  float z[J];
};

template <int NT, int J>
__device__ __forceinline__ void teacher_issue(const TopkParams& p, int64_t trow, TeacherEntries<J>& t) {
  const int K = p.K;
  const int cnt = p.t_cnt ? min(p.t_cnt[trow], K) : K;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k = threadIdx.x + j * NT;
    int64_t id = -1;
    float v = -INFINITY;
    if (k < cnt) {
      const int64_t at = trow * (int64_t)K + k;
      id = load_index(p.t_idx, p.t_idx_itype, at);
      v = load_as_float(p.t_val, p.t_val_dtype, at);       // independent of the id: both loads fly together
    }
    const bool ok = id >= 0 && id < p.V && v > -INFINITY;      // an entry of zero mass is no entry
    t.id[j] = ok ? (int)id : -1;
    t.tv[j] = ok ? v * p.inv_T_t : -INFINITY;
  }
}

template <class Tag, int J>
__device__ __forceinline__ void teacher_gather(const char* row, int lo, int hi, TeacherEntries<J>& t) {
#pragma unroll
  for (int j = 0; j < J; ++j)
    t.z[j] = (t.id[j] >= lo && t.id[j] < hi) ? load_as_float(row, Tag::id, t.id[j]) : 0.f;
}

// Prepared teachers (TeacherBuckets): the first J * NT = cap0 entries of this part's bucket, one per
// lane and slot, fetched by position alone (slots behind the count hold whatever was there); the bucket's and the row's entry
// counts and the row's mass sum come along as same-address loads.
struct BucketHead { int n; int total; float qsum; int more_at; };

template <int NT, int J>
__device__ __forceinline__ void bucket_issue(const TopkParams& p, int64_t trow, int h, int P, TeacherEntries<J>& t,
                                             BucketHead& hd) {
  const uint2* first = p.bk.first + (trow * P + h) * (int64_t)p.bk.cap0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const uint2 e = first[threadIdx.x + j * NT];
    t.id[j] = (int)e.x;
    t.tv[j] = __uint_as_float(e.y);
  }
  const int* head = p.bk.head + trow * 16;
  hd.n = min(max(head[h], 0), p.bk.E);    // counts are clamped to what the workspace and LDS were laid out for
  hd.total = head[8];
  hd.qsum = __int_as_float(head[9]);
  hd.more_at = 0;                         // where this bucket's overflow starts in the row's share of `more`
  for (int g = 0; g < h; ++g) hd.more_at += max(min(head[g], p.bk.E) - p.bk.cap0, 0);
  hd.more_at = min(hd.more_at, p.bk.E - max(hd.n - p.bk.cap0, 0));
}

// The columns [lo, hi) of a part: the ones of its 16-byte chunks are [lob, hib); a part of a row off the 16-byte grid
// (ANY) has up to 7 columns ahead of them and 7 behind.  Entries are linked into the list of the chunk their column lies
// in, or into the list of the one column beside the chunks.
struct PartCols {
  int lo, hi, lob, hib;
  __device__ __forceinline__ bool beside(int id) const { return id < lob || id >= hib; }      // of an id inside [lo, hi)
  __device__ __forceinline__ int rest_of(int id) const { return id < lob ? id - lo : (lob - lo) + (id - hib); }
};
template <class Tag, int NT, int NCH, bool ANY>
__device__ __forceinline__ void link_entry(const TopkLds& s, const PartCols& pc, int k, int id) {
  if (ANY && pc.beside(id)) s.next[k] = atomicExch(&s.rest[pc.rest_of(id)], k);
  else correction_link<Tag, NT, NCH>(s.head, s.own, s.next, k, id - pc.lob);
}
template <class Tag, int NT, int NCH, bool ANY>
__device__ __forceinline__ int first_entry(const TopkLds& s, const PartCols& pc, int id) {
  if (ANY && pc.beside(id)) return s.rest[pc.rest_of(id)];
  return s.head[correction_head_slot<Tag, NT, NCH>(id - pc.lob)];
}

// Registers -> LDS, then the teacher's log-sum-exp; same result layout as stage_teacher.
// The gathered student logits t.z are the last loads of the workgroup to arrive (they queue behind the
// row's own loads), so they are touched last: everything before overlaps with the row in flight.
template <int NT, int J>
__device__ __forceinline__ float teacher_finish(const TopkLds& s, const TeacherEntries<J>& t) {
  float tmax = -INFINITY;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k = threadIdx.x + j * NT;
    if (k < s.Kp) s.idx[k] = t.id[j];
    tmax = fmaxf(tmax, t.tv[j]);
  }
  tmax = block_max<NT>(tmax, s.red);     // barrier inside: LDS entries visible afterwards
  float tlse = tmax;
  if (tmax != -INFINITY) {
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) part += expf(t.tv[j] - tmax);
    tlse = tmax + logf(block_sum<NT>(part, s.red));
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = threadIdx.x + j * NT;
      if (k < s.Kp) {
        const float lt = t.tv[j] - tlse;
        s.t[k] = lt;
        s.q[k] = expf(lt);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k = threadIdx.x + j * NT;
    if (k < s.Kp) s.z[k] = t.z[j];      // read back by this thread only
  }
  return tlse;
}

// Stage the teacher row: ids, scaled log-probs, and the student logits at the ids that fall into
// the column range [lo, hi) this workgroup owns.  Returns the log-sum-exp of the scaled teacher
// entries (-inf if the row has none); afterwards s.t holds the teacher log-probabilities and s.q
// the probabilities (0 for padding and ignored entries).
template <class Tag, int NT>
__device__ __forceinline__ float stage_teacher(const TopkParams& p, const TopkLds& s, int64_t trow,
                                               const char* row, int lo, int hi) {
  const int K = p.K;
  const int cnt = p.t_cnt ? min(p.t_cnt[trow], K) : K;
  float tmax = -INFINITY;
  for (int k = threadIdx.x; k < s.Kp; k += NT) {
    const int64_t at = trow * (int64_t)K + k;
    const int64_t id = k < cnt ? load_index(p.t_idx, p.t_idx_itype, at) : -1;
    const bool in = id >= 0 && id < p.V;
    const float tv = in ? load_as_float(p.t_val, p.t_val_dtype, at) * p.inv_T_t : -INFINITY;
    const bool ok = in && tv > -INFINITY;                  // an entry of zero mass is no entry
    s.idx[k] = ok ? (int)id : -1;
    s.t[k] = tv;
    s.z[k] = (ok && id >= lo && id < hi) ? load_as_float(row, Tag::id, id) : 0.f;
    tmax = fmaxf(tmax, tv);
  }
  tmax = block_max<NT>(tmax, s.red);     // barrier inside: LDS entries visible afterwards
  if (tmax == -INFINITY) return tmax;
  float part = 0.f;
  for (int k = threadIdx.x; k < s.Kp; k += NT) part += expf(s.t[k] - tmax);
  const float tlse = tmax + logf(block_sum<NT>(part, s.red));
  for (int k = threadIdx.x; k < s.Kp; k += NT) {      // own entries only: no barrier needed yet
    const float lt = s.t[k] - tlse;
    s.t[k] = lt;
    s.q[k] = expf(lt);
  }
  return tlse;
}

// Partial forward-KL sums over the ids inside [lo, hi):  B = sum q_k (t_k - z_k * inv_T)  and, over
// all ids, Q = sum q_k.  The row value is  sum over parts of B  +  lse * Q.
template <int NT>
__device__ __forceinline__ void fkl_partials(const TopkParams& p, const TopkLds& s, int lo, int hi, float& B,
                                             float& Q) {
  B = 0.f; Q = 0.f;
  for (int k = threadIdx.x; k < s.Kp; k += NT) {
    const int id = s.idx[k];
    if (id >= 0) {
      const float q = s.q[k];
      Q += q;
      if (id >= lo && id < hi) B += q * (s.t[k] - s.z[k] * p.inv_T_s);
    }
  }
  block_sum2<NT>(B, Q, s.red);
}

// Sum of the masses q[e] of the entries on a chunk list that name column `want`, given the largest of
// them (`big` > 0): order-independent.  Every mass is scaled by a power of two taken from the largest
// (exact), rounded to an integer below 2^30 and added as such, so the sum is the same whatever order
// the list was linked in, and good to 2^-30 of the largest term per term.
__device__ __forceinline__ float mass_on_column(const int* next, const int* col, const float* q, int first, int want,
                                                float big) {
  const int shift = 30 - __builtin_amdgcn_frexp_expf(big);      // big * 2^shift in [2^29, 2^30)
  long long acc = 0;
  for (int e = first; e >= 0; e = next[e])
    if (col[e] == want) acc += (long long)__float2int_rn(ldexpf(q[e], shift));
  const float hi = (float)(int)(acc >> 24), lo = (float)(int)(acc & 0xffffff);      // acc < 2^41: both parts exact in fp32
  return ldexpf(fmaf(hi, 16777216.f, lo), -shift);
}

// Prepared teachers, the K-wide part of the row's loss.  Several entries of a row may carry the same
// student id (the same token in two teachers, two teacher ids mapped onto one student id); the
// mixture's mass on the id is their sum Q_id, and the row's forward KL is
//     sum_id Q_id (log Q_id - s_id)  =  sum_k q_k (log Q_id(k) - s_id(k)).
// All entries of a bucket lie inside the part's columns [lo, hi).  They are linked into the lists of
// the 16-byte chunks their columns lie in (the lists the gradient sweep uses anyway); the thread of
// entry k then finds the other entries of its column on that list and sums their masses in fixed
// point, independent of the list's order.  Entries beyond the bucket's first cap0 (rare: the ids of a
// row crowd into one part) are fetched here, from the row's overflow share.
// Leaves q in s.q, Q_id(k) in s.val[k], z in s.z[k]; returns the number of LDS entry slots in use
// (a multiple of NT); B as fkl_partials.
template <class Tag, int NT, int NCH, int J, bool ANY>
__device__ __forceinline__ int bucket_finish(const TopkParams& p, const TopkLds& s, const TeacherEntries<J>& te,
                                             const BucketHead& hd, int64_t trow, const char* row, const PartCols& pc, float& B) {
  const int lo = pc.lo, hi = pc.hi;
  const int nk = max(J * NT, (hd.n + NT - 1) / NT * NT);
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int k = threadIdx.x + j * NT;
    const bool ok = k < hd.n && te.id[j] >= lo && te.id[j] < hi;      // what lies behind the bucket's count was never written
    s.idx[k] = ok ? te.id[j] : -1;
    s.t[k] = te.tv[j];
    s.q[k] = ok ? expf(te.tv[j]) : 0.f;
    s.z[k] = te.z[j];
  }
  if (nk > J * NT) {
    const uint2* more = p.bk.more + trow * (int64_t)p.bk.E + hd.more_at;
    for (int k = J * NT + threadIdx.x; k < nk; k += NT) {
      uint2 e{0xffffffffu, 0xff800000u};
      if (k < hd.n) e = more[k - J * NT];
      const int id = (int)e.x;
      const bool ok = id >= lo && id < hi;
      const float lq = __uint_as_float(e.y);
      s.idx[k] = ok ? id : -1;
      s.t[k] = lq;
      s.q[k] = ok ? expf(lq) : 0.f;
      s.z[k] = ok ? load_as_float(row, Tag::id, id) : 0.f;
    }
  }
  __syncthreads();                                         // every wave's share of the lists is cleared
  for (int k = threadIdx.x; k < nk; k += NT) {
    const int id = s.idx[k];                               // this thread's own store
    if (id >= 0) link_entry<Tag, NT, NCH, ANY>(s, pc, k, id);
  }
  __syncthreads();
  B = 0.f;
  for (int k = threadIdx.x; k < nk; k += NT) {
    const int id = s.idx[k];
    if (id < 0) continue;
    const int first = first_entry<Tag, NT, NCH, ANY>(s, pc, id);
    int same = 0;
    float big = 0.f;
    for (int e = first; e >= 0; e = s.next[e]) {
      const bool mine = s.idx[e] == id;
      same += mine ? 1 : 0;
      big = fmaxf(big, mine ? s.q[e] : 0.f);
    }
    const float q = s.q[k];
    float Qid = q, l = s.t[k];
    if (same > 1 && big > 0.f) {
      Qid = mass_on_column(s.next, s.idx, s.q, first, id, big);
      l = logf(Qid);
    }
    s.val[k] = Qid;
    B += q * (l - s.z[k] * p.inv_T_s);
  }
  B = block_sum<NT>(B, s.red);
  return nk;
}

// Teacher mass on the id of entry k, summed over every entry that carries the same id.
__device__ __forceinline__ float mass_on_id(const TopkLds& s, int k, int id) {
  int same = 0;
  const int4* ids = reinterpret_cast<const int4*>(s.idx);
#pragma unroll 4
  for (int j = 0; j < s.Kp / 4; ++j) {
    const int4 v = ids[j];
    same += (v.x == id) + (v.y == id) + (v.z == id) + (v.w == id);
  }
  if (same == 1) return s.q[k];
  float q = 0.f;                        // duplicates inside a row are rare: slow path
  for (int j = 0; j < s.Kp; ++j) q += (s.idx[j] == id) ? s.q[j] : 0.f;
  return q;
}

// Sparse corrections of the dense softmax row already written by this workgroup, for the ids
// inside [lo, hi).  b is the row's log2-sum-exp2, a = inv_T * log2(e), c = inv_T * scale.
template <class Tag, int NT>
__device__ __forceinline__ void fkl_sparse_fix(const TopkLds& s, void* grow, int lo, int hi,
                                               float a, float b, float c, bool ids_unique) {
  for (int k = threadIdx.x; k < s.Kp; k += NT) {
    const int id = s.idx[k];
    if (id < lo || id >= hi) continue;
    const float q = ids_unique ? s.q[k] : mass_on_id(s, k, id);
    store_from_float(grow, Tag::id, id, (fast_exp2(fmaf(s.z[k], a, -b)) - q) * c);
  }
}

// The same corrections for a row (part) held in registers, applied by the threads that hold the
// columns before they store them (correction_link / correction_apply).  Entry threads leave the
// student probability at the entry's column in s.val and link the entry into its owner's list; the
// owner subtracts the teacher mass -- of all entries of that column, should ids repeat, which it
// sees from the chunk's list: no scan over the row's ids.
template <class Tag, int NT, int NCH, bool ANY>
__device__ __forceinline__ void fkl_link_corrections(const TopkLds& s, const PartCols& pc, float a, float b) {
  for (int k = threadIdx.x; k < s.Kp; k += NT) {
    const int id = s.idx[k];
    if (id < pc.lo || id >= pc.hi) continue;
    s.val[k] = fast_exp2(fmaf(s.z[k], a, -b));
    link_entry<Tag, NT, NCH, ANY>(s, pc, k, id);
  }
}
// The entries beside the part's chunks only (kernels that write the others behind their dense stores).
template <int NT>
__device__ __forceinline__ void fkl_link_rest(const TopkLds& s, const PartCols& pc) {
  for (int k = threadIdx.x; k < s.Kp; k += NT) {
    const int id = s.idx[k];
    if (id >= pc.lo && id < pc.hi && pc.beside(id)) s.next[k] = atomicExch(&s.rest[pc.rest_of(id)], k);
  }
}

// Full-row statistics straight from global memory (two uses: the streaming kernel, and a split
// part whose partner did not answer in time).  Returns the row maximum and sum 2^((x - max) a).
// MODE 0: element by element.  MODE 1: rows on the 16-byte grid, a whole number of chunks long.
// MODE 2: any row: its 16-byte chunks by vector loads, the elements before and behind them one by one.
template <class Tag, int NT, int MODE>
__device__ __forceinline__ void row_stats_streamed(const char* row, int64_t V, float a, float* red, float& mx,
                                                   float& sm) {
  using C = Chunk<Tag>;
  float m = -INFINITY;
  sm = 0.f;
  const auto one = [&](float f) {
    if (f > m) { sm *= fast_exp2((m - f) * a); m = f; }
    if (f * a > MASKED_BELOW) sm += fast_exp2(fmaf(f, a, -m * a));
  };
  if (MODE != 0) {
    const RowSplit<Tag> sp(row, V, MODE == 2);
    const char* body = row + (int64_t)sp.head * Tag::bytes;
    for (int64_t ch = threadIdx.x; ch < sp.nbody; ch += NT) {
      float f[C::N];
      C::unpack(*reinterpret_cast<const u32x4*>(body + ch * 16), f);
      float cm = f[0];
#pragma unroll
      for (int e = 1; e < C::N; ++e) cm = fmaxf(cm, f[e]);
      if (cm > m) { sm *= fast_exp2((m - cm) * a); m = cm; }
      const float mb = m * a;
      if (mb > MASKED_BELOW) {
#pragma unroll
        for (int e = 0; e < C::N; ++e) sm += fast_exp2(fmaf(f[e], a, -mb));
      }
    }
    if (MODE == 2 && (int)threadIdx.x < sp.leftovers()) one(load_as_float(row, Tag::id, sp.column(threadIdx.x)));
  } else {
    for (int64_t j = threadIdx.x; j < V; j += NT) one(load_as_float(row, Tag::id, j));
  }
  mx = block_max<NT>(m, red);
  sm = (m == -INFINITY) ? 0.f : sm * fast_exp2((m - mx) * a);
  sm = block_sum<NT>(sm, red);
}

// How the rows of a register kernel lie in memory (template parameter RAG):
//   ROWS_WHOLE  on the 16-byte grid (base and pitch), a whole number of chunks long
//   ROWS_ANY    anywhere (element-aligned), any length
// The chunks of a ROWS_ANY part start at its first 16-byte boundary, so that its loads (and the stores of a gradient row
// of the same phase: every row of contiguous tensors) are aligned; a gradient row of another phase takes the same stores
// unaligned.  The up to 7 columns ahead of the chunks and 7 behind them sit one per thread in the first threads of the
// workgroup (x_rest, -inf in the others: adds nothing to any statistic).  The sweeps are then those of whole rows: no
// bound and no branch inside them, and every shape that serves whole rows serves these, in their time: 16384 x 20003
// bf16, K = 100, 351 -> 271 us (20008 columns: 265 us), 8192 x 151665 1096 -> 955 us, 4093 x 50257 with a tenth of the
// rows masked 227 -> 174 us (unaligned accesses from the row's first column and an element-wise last chunk inside the
// sweeps, with fewer shapes to choose from, before).
//   ROWS_EXACT  ROWS_ANY that keeps the logits in the registers (KEEP_LOGITS) where the other two leave 16-bit
//               probabilities there: a second exponential per element, one rounding less, and no probability is lost for being
//               2^-39 of the row's largest.  For the two-byte rows off the 16-byte grid (base or pitch) that had no other
//               kernel than the streaming one, which makes every probability in fp32, where now one workgroup of 512 threads or
//               more holds the row: a whole number of chunks long, or wider than 512 x 16 chunks without a workspace (8192 x
//               50304 bf16, K = 100, pitch 50307: 386 us streamed, 344 us so, 327 us from 16 bits).  Rows that end inside
//               a chunk have always had their probabilities held in 16 bits, in two column parts or on the grid.
constexpr int ROWS_WHOLE = 0, ROWS_ANY = 1, ROWS_EXACT = 2;

// ---------------------------------------------------------------------------------------
// Forward KL, (part of) a row resident in registers: NT threads x NCH 16-byte chunks per thread.
// SPLIT: P = p.parts workgroups per row.  Consecutive workgroup ids are dealt round-robin to the 8
// XCDs, each of which dispatches its share in order, so the parts of a row are placed 8 ids apart:
// they land on the same XCD back to back (partners start together and meet through one L2).
// Within a group of 8*P ids, id t serves row 8*group + t % 8, part t / 8.
// ---------------------------------------------------------------------------------------
// J > 0: the K <= J * NT teacher entries travel in registers (loads issued ahead of the row's);
// J == 0: any K, staged by a plain loop.
// RETRY: second launch over the parts that gave up waiting in the first (see split_retry_list):
// every record of the row is published by then, so nothing is waited for.
// MULTI: the row's teachers arrive prepared in buckets (TopkParams::bk), J * NT = cap0 entries in registers.
// RAG: how the rows lie in memory (ROWS_WHOLE / ROWS_ANY / ROWS_EXACT above).
template <class Tag, int NT, int NCH, bool SPLIT, int J, bool RETRY, bool MULTI, int RAG = ROWS_WHOLE>
__device__ __forceinline__ void fkl_topk_part(const TopkParams& p, const TopkLds& s, int64_t r, int h) {
  static_assert(!MULTI || J > 0, "the head of a bucket travels in registers");
  constexpr bool ANY = RAG != ROWS_WHOLE, KEEP_LOGITS = RAG == ROWS_EXACT;
  using C = Chunk<Tag>;
  const int tid = threadIdx.x;
  const int P = SPLIT ? p.parts : 1;
  const int64_t c0 = (int64_t)h * NT * NCH;                       // the part starts c0 chunks into the row
  PartCols pc;
  pc.lo = pc.lob = (int)(c0 * C::N);
  pc.hi = (int)min(p.V, (int64_t)pc.lo + NT * NCH * C::N);
  const int lo = pc.lo, hi = pc.hi;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * Tag::bytes : nullptr;
  char* gpart = grow ? grow + c0 * 16 : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  const auto zero_part = [&]() {
    if constexpr (ANY) zero_row_any<Tag, NT>(gpart, hi - lo);
    else zero_row<Tag, NT>(gpart, (hi - lo) / C::N);
  };
  if (trow < 0) {
    if (gpart) zero_part();
    if (tid == 0 && h == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  const char* row = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * Tag::bytes;
  const char* rpart = row + c0 * 16;
  const int head = ANY ? elements_to_grid<Tag>(rpart, hi - lo) : 0;
  const int nch = (hi - lo - head) / C::N;                        // chunks of this part
  pc.lob = lo + head;
  pc.hib = pc.lob + nch * C::N;
  const int rest = ANY ? head + (hi - pc.hib) : 0;                // columns beside them
  const int rest_col = tid < head ? lo + tid : pc.hib + (tid - head);
  const char* rbody = rpart + head * Tag::bytes;

  correction_clear<NT>(s.head, s.own);      // lists of corrections, filled after the row statistics
  if constexpr (ANY) {
    if (tid < REST_HEADS) s.rest[tid] = -1;
  }
  TeacherEntries<(J > 0 ? J : 1)> te;
  BucketHead hd{};
  if constexpr (MULTI) bucket_issue<NT, J>(p, trow, h, P, te, hd);
  else if constexpr (J > 0) teacher_issue<NT, J>(p, trow, te);
  float x_rest = -INFINITY;
  if constexpr (ANY) {
    if (tid < rest) x_rest = load_as_float(row, Tag::id, rest_col);
  }
  u32x4 reg[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int64_t c = ChunkMap<NT, NCH>::chunk(i, tid);
    // cached, not streaming, loads: the gather of the logits at the teacher ids that follows then
    // finds its lines in L2 instead of fetching them a second time (0.47 GB less per 32768 rows of K = 200)
    reg[i] = c < nch ? *reinterpret_cast<const u32x4*>(rbody + c * 16) : C::neg_inf();
  }

  // teacher side while the row is in flight
  float tlse = 0.f, B = 0.f, Q = 0.f;
  int nk = s.Kp;                      // LDS entry slots in use
  if constexpr (MULTI) {
    teacher_gather<Tag, J>(row, lo, hi, te);
    if (hd.total > 0) nk = bucket_finish<Tag, NT, NCH, J, ANY>(p, s, te, hd, trow, row, pc, B);
    tlse = hd.total > 0 ? 0.f : -INFINITY;
    Q = hd.qsum;
  } else if constexpr (J > 0) {
    teacher_gather<Tag, J>(row, lo, hi, te);
    tlse = teacher_finish<NT, J>(s, te);
  } else {
    tlse = stage_teacher<Tag, NT>(p, s, trow, row, lo, hi);
  }
  if (tlse == -INFINITY) {            // no usable teacher entry: the row contributes nothing
    if (gpart) zero_part();
    if (tid == 0 && h == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  if constexpr (!MULTI) fkl_partials<NT>(p, s, lo, hi, B, Q);

  const float a = p.inv_T_s * LOG2E;
  float mx = x_rest;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    float f[C::N];
    forget(reg[i]);
    C::unpack(reg[i], f);
#pragma unroll
    for (int e = 0; e < C::N; ++e) mx = fmaxf(mx, f[e]);
  }
  mx = block_max<NT>(mx, s.red);
  // Second sweep: 2^(x a - max a + bias) takes the place of x in the registers; the gradient is
  // that value times a row constant, so each element costs one exp2, not two.  (Not with KEEP_LOGITS, see above.)
  constexpr float BIAS = KEEP_LOGITS ? 0.f : C::stash_bias;
  // A part that holds only -inf logits, or only masked ones: every 2^(.) below is 0, not NaN.  (MASKED_BELOW; for two-byte
  // logits already where the rounding of x a - bias could carry a stashed value past fp16's infinity: they are thousands apart there.)
  float mb = mx * a;
  const bool masked = SPLIT ? mb < (Tag::bytes == 2 ? -0x1p20f : MASKED_BELOW) : mx == -INFINITY;
  if (masked) { mb = 0.f; mx = -INFINITY; }
  const float mb_own = mb - BIAS;
  float sm = ANY ? fast_exp2(fmaf(x_rest, a, -mb_own)) : 0.f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    float f[C::N];
    forget(reg[i]);
    C::unpack(reg[i], f);
#pragma unroll
    for (int e = 0; e < C::N; ++e) {
      f[e] = fast_exp2(fmaf(f[e], a, -mb_own));
      sm += f[e];
    }
    if constexpr (!KEEP_LOGITS) reg[i] = C::stash(f);
    forget(reg[i]);         // pins the schedule chunk by chunk: no pile-up of unpacked values
  }
  sm = block_sum<NT>(sm * __builtin_exp2f(-BIAS), s.red);      // exact: a power of two

  if (SPLIT) {
    // publish this part's statistics, collect the others'
    PartStats* ws = reinterpret_cast<PartStats*>(p.workspace) + r * P;
    if (tid == 0 && !RETRY) part_publish(ws + h, mx, sm, B);
    if (tid < P) {
      float om = mx, os = sm, ob = B;
      const int ok = (tid == h) || part_collect(ws + tid, RETRY ? 0x7fffffff : p.spin_limit, om, os, ob);
      s.xm[tid] = om; s.xs[tid] = os; s.xb[tid] = ob; s.xok[tid] = ok;
    }
    __syncthreads();
    bool all_ok = true;
    for (int j = 0; j < P; ++j) all_ok = all_ok && (s.xok[j] != 0);
    if (!all_ok) {
      // A partner did not answer in time.  Nothing has been written yet: this part puts itself on
      // the retry list and leaves; its own record is published, so the partners can finish.
      if (tid == 0) {
        RetryList list(p.workspace, p.n_rows, P);
        list.entries[atomicAdd(list.count, 1u)] = (unsigned)(r * P + h);
      }
      return;
    }
    float M = s.xm[0];
    for (int j = 1; j < P; ++j) M = fmaxf(M, s.xm[j]);
    float S = 0.f, Bt = 0.f;
    for (int j = 0; j < P; ++j) { S += s.xs[j] * fast_exp2((s.xm[j] - M) * a); Bt += s.xb[j]; }
    mb = M * a; sm = S; B = Bt;
  }
  const float b = mb + fast_log2(sm);      // log2-sum-exp2 of the scaled row
  if (tid == 0 && h == 0 && p.row_loss) p.row_loss[r] = B + (b * LN2) * Q;

  if (gpart) {
    const float c = p.inv_T_s * p.grad_scale;
    const float kc = SPLIT && masked ? 0.f : fast_exp2(mb_own - b) * c;       // stashed value -> gradient (a masked part's: 0)
    // 16 chunks of 4-byte logits leave no registers for placing the corrections during the sweep
    // (it spills): those shapes write them behind the dense stores instead.
    constexpr bool IN_REGISTERS = !(Tag::bytes == 4 && NCH == 16);
    if constexpr (MULTI) {
      // the lists exist since bucket_finish, s.val holds the mixture's mass on the entry's id: every
      // entry of a column carries the column's final value, whichever of them the owner meets
      for (int k = tid; k < nk; k += NT) {
        const int id = s.idx[k];
        if (id >= lo && id < hi) s.val[k] = fast_exp2(fmaf(s.z[k], a, -b)) - s.val[k];
      }
      __syncthreads();
    } else if (IN_REGISTERS) {
      fkl_link_corrections<Tag, NT, NCH, ANY>(s, pc, a, b);
      __syncthreads();
    } else if (ANY) {
      fkl_link_rest<NT>(s, pc);
      __syncthreads();
    }
    char* gbody = gpart + head * Tag::bytes;
    const unsigned mine = IN_REGISTERS ? s.own[tid] : 0u;
    const bool may_repeat = !MULTI && (p.flags & DL_TOPK_UNIQUE_IDS) == 0;
    const auto mass = [&](int k) { return MULTI ? 0.f : s.q[k]; };
    const auto value = [&](int k, float q) { return (s.val[k] - q) * c; };
    unsigned repeats = 0u;            // chunks in which an id occurs more than once
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int64_t ch = ChunkMap<NT, NCH>::chunk(i, tid);
      if (ch < nch) {
        float f[C::N];
        forget(reg[i]);
        if constexpr (KEEP_LOGITS) {
          C::unpack(reg[i], f);
#pragma unroll
          for (int e = 0; e < C::N; ++e) f[e] = fast_exp2(fmaf(f[e], a, -b)) * c;
        } else {
          C::unstash(reg[i], f);
#pragma unroll
          for (int e = 0; e < C::N; ++e) f[e] *= kc;
        }
        if (mine & (1u << i))
          if (correction_apply<Tag, NT, NCH>(s.head, s.next, s.idx, pc.lob, i, f, mass, value)) repeats |= 1u << i;
        if constexpr (ANY) store16_stream_any(gbody + ch * 16, C::pack(f));
        else store16_stream(gbody + ch * 16, C::pack(f));
      }
    }
    if constexpr (ANY) {
      // a column beside the chunks: its dense value less the mass of the entries on its list
      if (tid < rest) {
        const int first = s.rest[tid];
        float g = fast_exp2(fmaf(x_rest, a, -b));
        if (first >= 0) g = MULTI ? s.val[first] : g - correction_exact_sum(s.next, s.idx, first, rest_col, [&](int k) { return s.q[k]; });
        store_from_float(grow, Tag::id, rest_col, g * c);
      }
    }
    if (may_repeat && repeats)
      correction_repeats<Tag, NT, NCH>(s.head, s.next, s.idx, pc.lob, repeats, NCH, mass, value,
                                  [&](int column, float v) { store_from_float(grow, Tag::id, column, v); });
    if (!IN_REGISTERS) {
      __syncthreads();      // dense stores are ordered before the sparse corrections
      if constexpr (MULTI) {
        for (int k = tid; k < nk; k += NT) {
          const int id = s.idx[k];
          if (id >= pc.lob && id < pc.hib) store_from_float(grow, Tag::id, id, s.val[k] * c);      // entries of one column: the same value
        }
      } else {
        fkl_sparse_fix<Tag, NT>(s, grow, pc.lob, pc.hib, a, b, c, (p.flags & DL_TOPK_UNIQUE_IDS) != 0);
      }
    }
  }
}

template <class Tag, int NT, int NCH, bool SPLIT, int J, bool MULTI = false, int RAG = ROWS_WHOLE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
void fkl_topk_reg_kernel(const TopkParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TopkLds s(smem, p.K, NT);
  const int P = SPLIT ? p.parts : 1;
  const unsigned grp = SPLIT ? blockIdx.x / (8u * P) : 0u, t_in = SPLIT ? blockIdx.x % (8u * P) : 0u;
  const int64_t r = SPLIT ? (int64_t)grp * 8 + (t_in & 7u) : xcd_banded_row(blockIdx.x);
  const int h = SPLIT ? (int)(t_in >> 3) : 0;
  if (r >= p.n_rows) return;
  fkl_topk_part<Tag, NT, NCH, SPLIT, J, false, MULTI, RAG>(p, s, r, h);
}

// One listed part, as a real call: the loop around it then costs the body no registers.
template <class Tag, int NT, int NCH, int J, bool MULTI, int RAG>
__device__ __attribute__((noinline)) void fkl_topk_part_again(const TopkParams& p, const TopkLds& s, unsigned at) {
  fkl_topk_part<Tag, NT, NCH, true, J, true, MULTI, RAG>(p, s, (int64_t)(at / (unsigned)p.parts), (int)(at % (unsigned)p.parts));
}

// The parts on the retry list, a fixed grid striding over it (normally the list is empty and
// every workgroup leaves after one load).
template <class Tag, int NT, int NCH, int J, bool MULTI = false, int RAG = ROWS_WHOLE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
void fkl_topk_retry_kernel(const TopkParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TopkLds s(smem, p.K, NT);
  const RetryList list(p.workspace, p.n_rows, p.parts);
  const unsigned n = *list.count;
#pragma unroll 1
  for (unsigned e = blockIdx.x; e < n; e += gridDim.x) {
    fkl_topk_part_again<Tag, NT, NCH, J, MULTI, RAG>(p, s, list.entries[e]);
    __syncthreads();      // LDS is reused by the next entry
  }
}

// ---------------------------------------------------------------------------------------
// Forward KL, streaming: any V, any alignment; the row is read twice (second read mostly L2 / MALL).
// MODE as for row_stats_streamed; MODE 2 needs the gradient row to sit on the 16-byte grid as the
// logits row does (same address modulo 16), so that the chunks of both line up.
// ---------------------------------------------------------------------------------------
template <class Tag, int NT, int MODE>
__global__ __launch_bounds__(NT) void fkl_topk_stream_kernel(const TopkParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TopkLds s(smem, p.K);
  using C = Chunk<Tag>;
  const int64_t r = xcd_banded_row(blockIdx.x);
  if (r >= p.n_rows) return;
  const int tid = threadIdx.x;
  const int64_t V = p.V;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * Tag::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  const char* row = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * Tag::bytes;
  const RowSplit<Tag> sp(row, V, MODE == 2);
  float tlse = -INFINITY;
  if (trow >= 0) tlse = stage_teacher<Tag, NT>(p, s, trow, row, 0, (int)V);
  if (tlse == -INFINITY) {
    if (grow) {
      if (MODE != 0) {
        zero_row<Tag, NT>(grow + (int64_t)sp.head * Tag::bytes, sp.nbody);
        if (MODE == 2 && tid < sp.leftovers()) store_from_float(grow, Tag::id, sp.column(tid), 0.f);
      } else {
        for (int64_t j = tid; j < V; j += NT) store_from_float(grow, Tag::id, j, 0.f);
      }
    }
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  float B, Q;
  fkl_partials<NT>(p, s, 0, (int)V, B, Q);
  const float a = p.inv_T_s * LOG2E;
  float mx, sm;
  row_stats_streamed<Tag, NT, MODE>(row, V, a, s.red, mx, sm);
  const float b = mx * a + fast_log2(sm);
  if (tid == 0 && p.row_loss) p.row_loss[r] = B + (b * LN2) * Q;

  if (grow) {
    const float c = p.inv_T_s * p.grad_scale;
    if (MODE != 0) {
      const char* body = row + (int64_t)sp.head * Tag::bytes;
      char* gbody = grow + (int64_t)sp.head * Tag::bytes;
      for (int64_t ch = tid; ch < sp.nbody; ch += NT) {
        float f[C::N];
        C::unpack(*reinterpret_cast<const u32x4*>(body + ch * 16), f);
#pragma unroll
        for (int e = 0; e < C::N; ++e) f[e] = fast_exp2(fmaf(f[e], a, -b)) * c;
        store16_stream(gbody + ch * 16, C::pack(f));
      }
      if (MODE == 2 && tid < sp.leftovers()) {
        const int64_t j = sp.column(tid);
        store_from_float(grow, Tag::id, j, fast_exp2(fmaf(load_as_float(row, Tag::id, j), a, -b)) * c);
      }
    } else {
      for (int64_t j = tid; j < V; j += NT)
        store_from_float(grow, Tag::id, j, fast_exp2(fmaf(load_as_float(row, Tag::id, j), a, -b)) * c);
    }
    __syncthreads();
    fkl_sparse_fix<Tag, NT>(s, grow, 0, (int)V, a, b, c, (p.flags & DL_TOPK_UNIQUE_IDS) != 0);
  }
}

// ---------------------------------------------------------------------------------------
// Reverse KL on the teacher's support: K gathered logits per row, gradient = zero row + K values.
// ---------------------------------------------------------------------------------------
// The K-wide part of a row.  Returns false if the row has no usable teacher entry (then nothing else is valid); else every
// entry k has its id (-1: none), the student's mass on it within the support in s.q and the log ratio to the teacher's in
// s.z, and rkl is the row's divergence: the gradient at an entry's column is c * q (z - rkl).  Ends in a barrier; an
// entry's values are written by thread k % NT.  J > 0: K <= J * NT entries in registers, all loads of a kind in flight together.
// The logits stay as they were read and are scaled inside a fused multiply-add: a product rounded by itself would put half an
// ulp of a number of the logits' size into every exponent (fp32 logits around 15, T = 1.4, 64 x 8001, K = 400: the gradient's
// error against float64 1.2e-6 so, 1.9e-6 with the product rounded).
template <class Tag, int NT, int J>
__device__ __forceinline__ bool rkl_on_support(const TopkParams& p, const TopkLds& s, int64_t r, int64_t trow, float& rkl) {
  if (trow < 0) return false;
  const int tid = threadIdx.x, K = p.K;
  const char* row = reinterpret_cast<const char*>(p.logits) + r * p.row_stride * Tag::bytes;
  if constexpr (J > 0) {
    const int cnt = p.t_cnt ? min(p.t_cnt[trow], K) : K;
    int id[J];
    float t[J], z[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = tid + j * NT;
      int64_t i = -1;
      float v = -INFINITY;
      if (k < cnt) {
        const int64_t at = trow * (int64_t)K + k;
        i = load_index(p.t_idx, p.t_idx_itype, at);
        v = load_as_float(p.t_val, p.t_val_dtype, at);
      }
      const bool in = i >= 0 && i < p.V;
      t[j] = in ? v * p.inv_T_t : -INFINITY;
      id[j] = in && t[j] > -INFINITY ? (int)i : -1;          // an entry of zero mass is no entry
    }
    float tmax = -INFINITY, zm = -INFINITY;
#pragma unroll
    for (int j = 0; j < J; ++j) z[j] = id[j] >= 0 ? load_as_float(row, Tag::id, id[j]) : 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      tmax = fmaxf(tmax, t[j]);
      if (id[j] >= 0) zm = fmaxf(zm, z[j] * p.inv_T_s);
    }
    block_max2<NT>(tmax, zm, s.red);
    if (tmax == -INFINITY) return false;
    float ts = 0.f, zs = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      ts += expf(t[j] - tmax);
      zs += id[j] >= 0 ? expf(fmaf(z[j], p.inv_T_s, -zm)) : 0.f;
    }
    block_sum2<NT>(ts, zs, s.red);
    const float tlse = tmax + logf(ts), slse = zm + logf(zs);
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int k = tid + j * NT;
      const float sp = fmaf(z[j], p.inv_T_s, -slse), d = sp - (t[j] - tlse), rk = expf(sp);
      if (id[j] >= 0) part = fmaf(rk, d, part);
      if (k < s.Kp) { s.idx[k] = id[j]; s.q[k] = rk; s.z[k] = d; }
    }
    rkl = block_sum<NT>(part, s.red);
    return true;
  } else {
    if (stage_teacher<Tag, NT>(p, s, trow, row, 0, (int)p.V) == -INFINITY) return false;
    // student renormalised over the staged ids
    float zm = -INFINITY;
    for (int k = tid; k < s.Kp; k += NT)
      if (s.idx[k] >= 0) zm = fmaxf(zm, s.z[k] * p.inv_T_s);
    zm = block_max<NT>(zm, s.red);
    float part = 0.f;
    for (int k = tid; k < s.Kp; k += NT)
      if (s.idx[k] >= 0) part += expf(fmaf(s.z[k], p.inv_T_s, -zm));
    const float slse = zm + logf(block_sum<NT>(part, s.red));
    part = 0.f;
    for (int k = tid; k < s.Kp; k += NT) {
      if (s.idx[k] >= 0) {
        const float sp = fmaf(s.z[k], p.inv_T_s, -slse);
        const float d = sp - s.t[k];
        const float rk = expf(sp);
        part = fmaf(rk, d, part);
        s.q[k] = rk;      // student mass on the support
        s.z[k] = d;       // log ratio
      }
    }
    rkl = block_sum<NT>(part, s.red);     // barriers inside publish s.q / s.z
    return true;
  }
}

// One launch: every workgroup makes its row's values and then writes the row.
// MODE 1: gradient rows on the 16-byte grid, a whole number of chunks long.  MODE 2: any other gradient row: its 16-byte
// chunks by vector stores (the teacher ids counted from the first of them), the columns before and behind them one by one.
template <class Tag, int NT, int MODE, int J>
__global__ __launch_bounds__(NT) void rkl_topk_kernel(const TopkParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TopkLds s(smem, p.K, NT);
  using C = Chunk<Tag>;
  const int64_t r = xcd_banded_row(blockIdx.x);
  if (r >= p.n_rows) return;
  const int tid = threadIdx.x;
  char* grow = p.grad ? reinterpret_cast<char*>(p.grad) + r * p.grad_stride * Tag::bytes : nullptr;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  const RowSplit<Tag> sp(grow, p.V, MODE == 2 && grow);              // the row that is written decides
  char* gbody = grow + (int64_t)sp.head * Tag::bytes;
  correction_clear<NT>(s.head, s.own);
  if (MODE == 2 && tid < REST_HEADS) s.rest[tid] = -1;
  // Every store comes after the K logits have been gathered (rkl_on_support ends in a barrier), so
  // the gradient may be written over the logits.
  float rkl;
  if (!rkl_on_support<Tag, NT, J>(p, s, r, trow, rkl)) {
    if (grow) {
      zero_row<Tag, NT>(gbody, sp.nbody);
      if (MODE == 2 && tid < sp.leftovers()) store_from_float(grow, Tag::id, sp.column(tid), 0.f);
    }
    if (tid == 0 && p.row_loss) p.row_loss[r] = 0.f;
    return;
  }
  if (tid == 0 && p.row_loss) p.row_loss[r] = rkl;
  if (grow) {
    const float c = p.inv_T_s * p.grad_scale;
    for (int k = tid; k < s.Kp; k += NT) {
      const int id = s.idx[k];
      if (id < 0) continue;
      // placed by the thread that writes the column's chunk, or one of the columns beside the body
      const int64_t idb = (int64_t)id - sp.head;
      if (idb >= 0 && idb < sp.nbody * C::N) correction_link<Tag, NT>(s.head, s.own, s.next, k, (int)idb);
      else if (MODE == 2) s.next[k] = atomicExch(&s.rest[idb < 0 ? id : sp.head + (int)(idb - sp.nbody * C::N)], k);
    }
    // the row of zeros, each chunk written once with the support's values already in place
    __syncthreads();
    const unsigned mine = s.own[tid];
    const int64_t nch = sp.nbody;
    const auto term = [&](int k) { return s.q[k] * (s.z[k] - rkl); };
    const auto value = [&](int, float g) { return g * c; };
    unsigned repeats = 0u;
    int n_own = 0;
    for (int64_t ch = tid, i = 0; ch < nch; ch += NT, ++i) {
      float f[C::N];
#pragma unroll
      for (int e = 0; e < C::N; ++e) f[e] = 0.f;
      if (mine & (1u << (i & 31)))
        if (correction_apply<Tag, NT>(s.head, s.next, s.idx, sp.head, (int)i, f, term, value)) repeats |= 1u << (i & 31);
      store16_stream(gbody + ch * 16, C::pack(f));
      n_own = (int)i + 1;
    }
    if (repeats)
      correction_repeats<Tag, NT>(s.head, s.next, s.idx, sp.head, repeats, n_own, term, value,
                                  [&](int column, float v) { store_from_float(grow, Tag::id, column, v); });
    if (MODE == 2 && tid < sp.leftovers()) {
      // a list each: where these few threads looked through all entries of the row, a chain of K reads stood behind its
      // stores (64 x 50257 bf16, K = 200 and 1000: 28 and 83 us with plain sums, 39 and 187 with exact ones; 16.5 and 26 so)
      const int first = s.rest[tid], j = (int)sp.column(tid);
      const float g = first >= 0 ? correction_exact_sum(s.next, s.idx, first, j, term) : 0.f;
      store_from_float(grow, Tag::id, j, g * c);
    }
  }
}

// Two launches, through a workspace of K (id, q (z - rkl)) pairs per row: the values of the rows, then nothing but the
// stores, in the order of the gradient's addresses (many rows: several turns of the two, see rkl_fill_rows).  A workgroup that makes a row's values and then writes the row is a
// chain of dependent round trips ahead of its stores, and 2048 rows are written at a time, spread over the whole buffer.
// Bound by the stores: a bare fill of 8192 x 128256 bf16 takes 300 us at best (7.0 TB/s: 4 KiB per workgroup, every XCD in an
// eighth of the buffer of its own), 314 with 16 KiB per workgroup, 345 with the workgroups dealt round the XCDs in
// address order, 320-455 from persistent grids.  Measured with the row's values (K = 200): 448 us in one launch, 359 so, of
// which 34 for the values; 384 with slabs of 16 KiB instead of 8, 420 with the correction lists of the register kernels
// instead of a slab in LDS and the workgroups in address order.  4096 x 128256 fp32, K = 20: 434 -> 331 us.
template <class Tag, int NT, int J>
__global__ __launch_bounds__(NT) void rkl_values_kernel(const TopkParams p, int64_t row0) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TopkLds s(smem, p.K);
  const int64_t r = row0 + blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t trow = teacher_row(p.row_map, r, p.n_trows);
  uint2* out = reinterpret_cast<uint2*>(p.workspace) + (int64_t)blockIdx.x * p.K;
  float rkl = 0.f;
  const bool live = rkl_on_support<Tag, NT, J>(p, s, r, trow, rkl);
  if (tid == 0 && p.row_loss) p.row_loss[r] = live ? rkl : 0.f;
  for (int k = tid; k < p.K; k += NT)
    out[k] = live ? uint2{(unsigned)s.idx[k], __float_as_uint(s.q[k] * (s.z[k] - rkl))} : uint2{~0u, 0u};
}

// Item b is part b % parts of row row0 + b / parts: SLAB bytes of the row's body (and with part 0 the columns beside the body:
// MODE 2).  The part is made in LDS: zeroed, the pairs that name one of its columns (out of all K pairs of the row, from
// L2) written into place, and stored in one piece; a bit per column tells a repeated id, whose pairs are then added up.
constexpr int RKL_FILL_NT = 256, RKL_FILL_NCH = 2, RKL_SLAB = RKL_FILL_NT * RKL_FILL_NCH * 16;
template <class Tag, int MODE>
__global__ __launch_bounds__(RKL_FILL_NT) void rkl_fill_kernel(const TopkParams p, int64_t row0, int64_t rows, unsigned parts) {
  using C = Chunk<Tag>;
  constexpr int NT = RKL_FILL_NT, NCH = RKL_FILL_NCH, COLS = RKL_SLAB / Tag::bytes, WORDS = COLS / 32 + 1;
  __shared__ __align__(16) u32x4 slab[NT * NCH];
  __shared__ unsigned named[WORDS];                                  // a bit per column; the last word: the columns beside the body
  __shared__ unsigned twice[WORDS];                                  // set: by more than one pair
  __shared__ float beside[REST_HEADS];
  __shared__ int repeats;
  const int tid = threadIdx.x;
  const unsigned item = xcd_eighth(blockIdx.x, gridDim.x);
  const int64_t at = item / parts, r = row0 + at;
  const int h = (int)(item % parts);
  if (at >= rows) return;
  const uint2* ent = reinterpret_cast<const uint2*>(p.workspace) + at * p.K;
  uint2 mine = tid < p.K ? ent[tid] : uint2{~0u, 0u};
#pragma unroll
  for (int i = 0; i < NCH; ++i) slab[i * NT + tid] = u32x4{0u, 0u, 0u, 0u};
  for (int i = tid; i < WORDS; i += NT) { named[i] = 0u; twice[i] = 0u; }
  if (tid == 0) repeats = 0;
  if (MODE == 2 && tid < REST_HEADS) beside[tid] = 0.f;
  char* grow = reinterpret_cast<char*>(p.grad) + r * p.grad_stride * Tag::bytes;
  const RowSplit<Tag> sp(grow, p.V, MODE == 2);
  const int c0 = h * NT * NCH;                                       // first chunk of the part
  const int nch = (int)min((int64_t)NT * NCH, sp.nbody - c0);        // its chunks (behind a row's head there may be none left: <= 0)
  const int lo = sp.head + c0 * C::N, hi = lo + max(nch, 0) * C::N;
  const int behind = sp.head + (int)sp.nbody * C::N;
  const float c = p.inv_T_s * p.grad_scale;
  // place of column `id`: inside the part, behind it (>= COLS) among the columns beside the body, or -1
  const auto place_of = [&](int id) {
    if (id >= lo && id < hi) return id - lo;
    if (MODE == 2 && h == 0 && id >= 0 && id < sp.head) return COLS + id;
    if (MODE == 2 && h == 0 && id >= behind) return COLS + sp.head + (id - behind);
    return -1;
  };
  const auto put = [&](int at, float g) {
    if (MODE == 2 && at >= COLS) beside[at - COLS] = g;
    else store_from_float(slab, Tag::id, at, g);
  };
  __syncthreads();
  for (int k = tid; k < p.K; k += NT) {
    if (k >= NT) mine = ent[k];
    const int at = place_of((int)mine.x);
    if (at < 0) continue;
    const unsigned bit = 1u << (at & 31);
    if (atomicOr(&named[at >> 5], bit) & bit) {
      atomicOr(&twice[at >> 5], bit);
      repeats = 1;
    } else {
      put(at, __uint_as_float(mine.y) * c);
    }
  }
  __syncthreads();
  if (repeats) {                                                     // every pair of a repeated id writes the same sum
    for (int k = tid; k < p.K; k += NT) {
      const int id = (int)ent[k].x, at = place_of(id);
      if (at < 0 || !(twice[at >> 5] & (1u << (at & 31)))) continue;
      put(at, exact_sum([&](auto f) {
        for (int q = 0; q < p.K; ++q) {
          const uint2 e = ent[q];
          if ((int)e.x == id) f(__uint_as_float(e.y));
        }
      }) * c);
    }
    __syncthreads();
  }
  char* gpart = grow + (int64_t)lo * Tag::bytes;
#pragma unroll
  for (int i = 0; i < NCH; ++i)
    if (i * NT + tid < nch) store16_stream(gpart + (i * NT + tid) * 16, slab[i * NT + tid]);
  if (MODE == 2 && h == 0 && tid < sp.leftovers()) store_from_float(grow, Tag::id, sp.column(tid), beside[tid]);
}

// clears the `ready` words of the split kernel's workspace (a template only so that it may live in a header)
template <int NT>
__global__ __launch_bounds__(NT) void clear_workspace_kernel(u32x4* ws, int64_t n16) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i < n16) ws[i] = u32x4{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------------------------------
// host dispatch
// ---------------------------------------------------------------------------------------
// Register slots for the entries of a row: J of fkl_topk_reg_kernel.  One stored teacher: 1 or 3 slots
// of NT entries, else 0 (staged by a loop).  Prepared teachers (MULTI): the slots the buckets were laid
// out for, cap0 / NT (1, 2, 4 or 8: bucket_slots).
template <int NT, bool MULTI>
static int entry_slots(const TopkParams& p) {
  if (MULTI) return p.bk.cap0 / NT;
  const int Kp = (p.K + 15) & ~15;
  return Kp <= NT ? 1 : Kp <= 3 * NT ? 3 : 0;
}

// Launches kernel template KERNEL<J, MULTI> for the slot count of this call.
#define DL_LAUNCH_BY_SLOTS(KERNEL_J, grid)                                                                      \
  {                                                                                                             \
    const int j = entry_slots<NT, MULTI>(p);                                                                    \
    const size_t lds = TopkLds::bytes(p.K, NT);                                                                 \
    if constexpr (MULTI) {                                                                                      \
      if (j == 1) hipLaunchKernelGGL((KERNEL_J(1)), dim3(grid), dim3(NT), lds, st, p);                          \
      if constexpr (2 * NT <= DL_MAX_TOPK)                                                                      \
        if (j == 2) hipLaunchKernelGGL((KERNEL_J(2)), dim3(grid), dim3(NT), lds, st, p);                        \
      if constexpr (4 * NT <= DL_MAX_TOPK)                                                                      \
        if (j == 4) hipLaunchKernelGGL((KERNEL_J(4)), dim3(grid), dim3(NT), lds, st, p);                        \
      if constexpr (8 * NT <= DL_MAX_TOPK)                                                                      \
        if (j == 8) hipLaunchKernelGGL((KERNEL_J(8)), dim3(grid), dim3(NT), lds, st, p);                        \
    } else {                                                                                                    \
      if (j == 1) hipLaunchKernelGGL((KERNEL_J(1)), dim3(grid), dim3(NT), lds, st, p);                          \
      else if (j == 3) hipLaunchKernelGGL((KERNEL_J(3)), dim3(grid), dim3(NT), lds, st, p);                     \
      else hipLaunchKernelGGL((KERNEL_J(0)), dim3(grid), dim3(NT), lds, st, p);                                 \
    }                                                                                                           \
  }

template <class Tag, int NT, int NCH, bool SPLIT, bool MULTI, int RAG>
static void launch_reg_j(const TopkParams& p, unsigned grid, hipStream_t st) {
#define DL_REG_KERNEL(J) fkl_topk_reg_kernel<Tag, NT, NCH, SPLIT, J, MULTI, RAG>
  DL_LAUNCH_BY_SLOTS(DL_REG_KERNEL, grid)
#undef DL_REG_KERNEL
}

template <class Tag, int NT, int NCH, bool MULTI, int RAG>
static void launch_retry_j(const TopkParams& p, unsigned grid, hipStream_t st) {
#define DL_RETRY_KERNEL(J) fkl_topk_retry_kernel<Tag, NT, NCH, J, MULTI, RAG>
  DL_LAUNCH_BY_SLOTS(DL_RETRY_KERNEL, grid)
#undef DL_RETRY_KERNEL
}
#undef DL_LAUNCH_BY_SLOTS

static int launch_status() { return hipGetLastError() == hipSuccess ? DL_OK : DL_ERR_LAUNCH; }

template <class Tag, int NT, int NCH, bool MULTI, int RAG>
static int launch_reg(const TopkParams& p, hipStream_t st) {
  launch_reg_j<Tag, NT, NCH, false, MULTI, RAG>(p, xcd_banded_grid(p.n_rows), st);
  return launch_status();
}

// 16-byte words at the head of the exchange workspace that must be zero when the split kernels start:
// one PartStats per (row, part), then the retry counter
static int64_t split_clear_words(int64_t n_rows, int parts) { return n_rows * parts + 1; }

// `cleared`: an earlier launch on the same stream has already zeroed those words
template <class Tag, int NT, int NCH, bool MULTI, int RAG>
static int launch_split(TopkParams p, int parts, hipStream_t st, bool cleared) {
  p.parts = parts;
  const int64_t n16 = split_clear_words(p.n_rows, parts);
  if (!cleared)
    hipLaunchKernelGGL(clear_workspace_kernel<256>, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<u32x4*>(p.workspace), n16);
  launch_reg_j<Tag, NT, NCH, true, MULTI, RAG>(p, (unsigned)((p.n_rows + 7) / 8 * 8 * parts), st);
  launch_retry_j<Tag, NT, NCH, MULTI, RAG>(p, (unsigned)std::min<int64_t>(p.n_rows * parts, 256), st);
  return launch_status();
}

// Number of column parts a row of `nch` 16-byte chunks is cut into (1 = one workgroup per row).
// Rows of up to 1024 x 16 chunks are cut into parts of 256 x 16 chunks, as many as hold columns (a
// part without columns would have no maximum to publish); `forced` (the DL_TOPK_PARTS field of the
// call's flags) = 1, 2 or 4 overrides that for such rows where every part still gets columns.
static int split_parts(int64_t nch, int forced, bool fine = false) {
  if (fine && nch > 256 * 4 && nch <= (int64_t)MAX_PARTS * 256 * 4) return (int)((nch + 256 * 4 - 1) / (256 * 4));
  if (nch <= 512 * 16) return 1;
  const int parts = (int)((nch + 256 * 16 - 1) / (256 * 16));      // 3 .. MAX_COARSE_PARTS parts of 256 x 16 chunks
  if (nch > 1024 * 16) return parts;
  if (forced == 1 || forced == 2 || (forced == 4 && parts == 4)) return forced;
  return parts;
}

// The register kernel that serves rows of `nch` 16-byte chunks of `bytes`-wide logits: threads per
// workgroup, chunks per thread, column parts per row (parts > 1: the split kernels, which need the
// exchange workspace: `split_ok`).  NT == 0: none (rows too wide: the streaming kernel).
struct FklShape { int NT, NCH, parts; };
static FklShape fkl_shape(int64_t nch, int bytes, int forced_parts, bool split_ok, bool fine = false, bool thirteen = false) {
  if (nch > (int64_t)MAX_COARSE_PARTS * 256 * 16) return {0, 0, 0};
  if (fine && split_ok && nch > 256 * 4 && nch <= (int64_t)MAX_PARTS * 256 * 4) return {256, 4, split_parts(nch, forced_parts, true)};
  if (nch <= 256 * 4) return {256, 4, 1};
  if (nch <= 256 * 8) return {256, 8, 1};
  // 4-byte logits: 8 chunks per thread from twice the threads keep the corrections in registers
  if (nch <= 256 * 16) return bytes == 4 ? FklShape{512, 8, 1} : FklShape{256, 16, 1};
  // two-byte rows of up to 53248 columns (the 50k vocabularies): 13 chunks per thread.  A workgroup's waves are
  // filled one after the other and the full ones set its time: 13 sweeps instead of 16
  // (16384 x 50304 bf16: 64.6 -> 68.3 % of the HBM peak, 51200 columns: 69 %)
  if (thirteen && bytes != 4 && nch <= 512 * 13) return {512, 13, 1};
  if (nch <= 512 * 16) return {512, 16, 1};
  const int parts = split_parts(nch, forced_parts);
  // The widest rows in half as many parts of 512 threads: fewer partners to wait for.  Measured at 8192
  // rows: four-byte rows of 6 to 8 parts of 256 threads gain 4-11 % that way, two-byte rows of 8 parts
  // 4 %; two-byte rows of 5 to 7 parts lose up to 8 % (the last, partly filled part gets larger).
  if (split_ok && nch > 1024 * 16 && (bytes == 4 ? parts >= 6 : parts == 8)) return {512, 16, (parts + 1) / 2};
  if (parts == 2 && split_ok) return {512, 16, 2};
  if (parts >= 3 && split_ok) {
    // rows that do not fill their parts: as few chunks per thread as hold the row (13 to 15), the parts then equally
    // full -- every wave of every part carries the same share, and that share sets the row's time
    const int64_t per_thread = (nch + (int64_t)parts * 256 - 1) / ((int64_t)parts * 256);
    if (thirteen && per_thread < 16) return {256, per_thread < 13 ? 13 : (int)per_thread, parts};
    return {256, 16, parts};
  }
  if (nch <= 1024 * 16) return {1024, 16, 1};      // no workspace: one workgroup per row
  return {0, 0, 0};
}

// MULTI has no streaming form: the caller checks fkl_shape first.
// RAG = ROWS_ANY: the shapes of whole rows of ceil(V / chunk) chunks; off_grid: not on the 16-byte grid (ROWS_EXACT).
template <class Tag, bool MULTI, int RAG = ROWS_WHOLE>
static int launch_fkl(const TopkParams& p, int64_t ws_bytes, hipStream_t st, bool ws_cleared = false, bool off_grid = false) {
  const int64_t nch = (p.V + Tag::epc - 1) / Tag::epc;
  const int forced = (p.flags >> DL_TOPK_PARTS_SHIFT) & 15;
  const bool fine = !MULTI && (p.flags & DL_TOPK_FINE_PARTS) != 0 &&
                    ws_bytes >= RetryList::bytes(p.n_rows, split_parts(nch, forced, true));
  // the shape a workspace would allow; without room for that shape's records, the shape that needs none
  const FklShape wish = fkl_shape(nch, Tag::bytes, forced, true, fine, !MULTI);
  const bool split_ok = p.workspace && ws_bytes >= RetryList::bytes(p.n_rows, wish.parts) && p.n_rows * wish.parts <= 0x7fffffffLL;
  const FklShape sh = wish.parts <= 1 || split_ok ? wish : fkl_shape(nch, Tag::bytes, forced, false, fine, !MULTI);
  if constexpr (RAG == ROWS_ANY && Tag::bytes == 2) {
    if (off_grid && sh.parts == 1 && (p.V % Tag::epc == 0 || sh.NT == 1024)) {
      if constexpr (!MULTI)
        if (sh.NT == 512 && sh.NCH == 13) return launch_reg<Tag, 512, 13, MULTI, ROWS_EXACT>(p, st);
      if (sh.NT == 512 && sh.NCH == 16) return launch_reg<Tag, 512, 16, MULTI, ROWS_EXACT>(p, st);
      if (sh.NT == 1024) return launch_reg<Tag, 1024, 16, MULTI, ROWS_EXACT>(p, st);
    }
  }
  switch (sh.NT * 100 + sh.NCH) {
    case 256 * 100 + 4:
      if constexpr (!MULTI)
        if (sh.parts > 1) return launch_split<Tag, 256, 4, MULTI, RAG>(p, sh.parts, st, ws_cleared);
      return launch_reg<Tag, 256, 4, MULTI, RAG>(p, st);
    case 256 * 100 + 8: return launch_reg<Tag, 256, 8, MULTI, RAG>(p, st);
    case 512 * 100 + 8:
      if constexpr (Tag::bytes == 4) return launch_reg<Tag, 512, 8, MULTI, RAG>(p, st);
      break;
    case 256 * 100 + 16:
      if (sh.parts > 1) return launch_split<Tag, 256, 16, MULTI, RAG>(p, sh.parts, st, ws_cleared);
      if constexpr (Tag::bytes != 4) return launch_reg<Tag, 256, 16, MULTI, RAG>(p, st);
      break;
    case 512 * 100 + 13:
      if constexpr (Tag::bytes != 4 && !MULTI) return launch_reg<Tag, 512, 13, MULTI, RAG>(p, st);
      break;
    case 256 * 100 + 13:
      if constexpr (!MULTI) return launch_split<Tag, 256, 13, MULTI, RAG>(p, sh.parts, st, ws_cleared);
      break;
    case 256 * 100 + 14:
      if constexpr (!MULTI) return launch_split<Tag, 256, 14, MULTI, RAG>(p, sh.parts, st, ws_cleared);
      break;
    case 256 * 100 + 15:
      if constexpr (!MULTI) return launch_split<Tag, 256, 15, MULTI, RAG>(p, sh.parts, st, ws_cleared);
      break;
    case 512 * 100 + 16:
      return sh.parts > 1 ? launch_split<Tag, 512, 16, MULTI, RAG>(p, sh.parts, st, ws_cleared) : launch_reg<Tag, 512, 16, MULTI, RAG>(p, st);
    case 1024 * 100 + 16: return launch_reg<Tag, 1024, 16, MULTI, RAG>(p, st);
    default: break;
  }
  if (MULTI) return DL_ERR_LIMIT;
  // too wide for the register kernels.  Rows off the 16-byte grid: the streaming kernel moves their chunks by aligned
  // vector accesses if logits and gradient rows share their address modulo 16 (the same pitch from 16-byte aligned
  // bases, or the gradient written over the logits)
  const dim3 grid(xcd_banded_grid(p.n_rows));
  if constexpr (RAG == ROWS_WHOLE) {
    hipLaunchKernelGGL((fkl_topk_stream_kernel<Tag, 1024, 1>), grid, dim3(1024), TopkLds::bytes(p.K), st, p);
  } else {
    const bool same_phase = !p.grad || (reinterpret_cast<uintptr_t>(p.logits) % 16 == reinterpret_cast<uintptr_t>(p.grad) % 16 &&
                                        ((p.row_stride - p.grad_stride) * Tag::bytes) % 16 == 0);
    if (same_phase) hipLaunchKernelGGL((fkl_topk_stream_kernel<Tag, 1024, 2>), grid, dim3(1024), TopkLds::bytes(p.K), st, p);
    else hipLaunchKernelGGL((fkl_topk_stream_kernel<Tag, 1024, 0>), grid, dim3(1024), TopkLds::bytes(p.K), st, p);
  }
  return launch_status();
}

// The ROWS_ANY instantiations of launch_fkl live in translation units of their own (topk_div_any.hip,
// topk_multi_any.hip), so that they compile beside the others.
int launch_fkl_any(int logits_dtype, const TopkParams& p, int64_t ws_bytes, hipStream_t st, bool off_grid);
int launch_fkl_any_multi(int logits_dtype, const TopkParams& p, int64_t ws_bytes, hipStream_t st, bool ws_cleared, bool off_grid);

// Reverse KL.  Parts of a row for the two-launch form; 0: one launch.  Narrow rows give a workgroup of the one-launch form
// little to write behind its K values, and a part of the two-launch form many pairs to look through for each of its columns
// (8192 x 32000 bf16, K = 200: 115 us in one launch, 120 in two; 16384 x 12000: 116, 123).  From 96 KiB per row on two
// launches pay where there is enough to write to cover the second one (2048 x 50304 bf16 49 -> 44 us, 1024 x 36696 fp32 43 ->
// 36; 1024 x 50304 bf16 28 against 29), from 195 KiB on always: few rows leave most of the chip idle in one launch (32 x
// 128256 bf16 32 -> 29 us, 512 rows 36 -> 29).  Below 160 KB, many rows of some thousand entries stay in one launch: each
// part of 8 KiB looks through all of them, and the values' launch holds up to 512 in registers only (16384 x 50304 bf16, K =
// 768 / 1000 / 1025 / 1300: 577 / 608 / 656 / 825 us in one launch, 577 / 657 / 734 / 816 in two; 16384 x 99000, K = 1000 1161
// and 1026).  At K = 2048 one launch has LDS for two workgroups per CU only: 32768 x 65536 bf16 2978 against 2416.
static int64_t rkl_fill_parts(int logits_dtype, int64_t n_rows, int64_t V, int K) {
  const int64_t row_bytes = V * (logits_dtype == F32 ? 4 : 2);
  if (row_bytes < 96 * 1024) return 0;
  if (row_bytes < 200000 && n_rows * row_bytes < (128LL << 20)) return 0;
  if (row_bytes < 160000 && n_rows > 2048 && K > 768 && K <= 1792) return 0;
  return (row_bytes / 16 + RKL_FILL_NT * RKL_FILL_NCH - 1) / (RKL_FILL_NT * RKL_FILL_NCH);
}
// The pairs of all rows at once would be read from beyond L2 once there are more than about 24 MB of them, in the middle of
// the stores (fill alone, 8192 x 128256 bf16: 320 us at K = 100 to 300, 500 at 400, 576 at 500, 762 at 1000).  The rows are
// therefore taken a few thousand at a time, values and stores in turn, over the same 16 MiB.  Inputs that no cache holds, one
// launch / all rows at once / by 16 MiB: 32768 x 128256 bf16, K = 200 1765 / 1954 / 1413 us, K = 500 1976 / 2579 / 1637; 8192
// rows, K = 500 513 / 660 / 413; 16384 x 128256 fp32, K = 300 1778 / 2022 / 1319.  4 and 8 MiB measure 1-30 % more than 16, 24
// MiB up to 20 % more.
constexpr int64_t RKL_WORKSPACE_MOST = 16LL << 20;
// Rows per turn (0: one launch for all rows)
static int64_t rkl_fill_rows(int logits_dtype, int64_t n_rows, int64_t V, int K) {
  const int64_t parts = rkl_fill_parts(logits_dtype, n_rows, V, K);
  if (!parts) return 0;
  const int64_t threads = ((1LL << 32) / RKL_FILL_NT - 8) / parts;      // a launch takes fewer than 2^32 threads
  const int64_t most = std::min(threads, RKL_WORKSPACE_MOST / (K * (int64_t)sizeof(uint2)));
  const int64_t turns = (n_rows + most - 1) / most;
  return (n_rows + turns - 1) / turns;
}
static int64_t rkl_workspace_bytes(int logits_dtype, int64_t n_rows, int64_t V, int K) {
  return rkl_fill_rows(logits_dtype, n_rows, V, K) * K * (int64_t)sizeof(uint2);
}

template <class Tag>
static hipError_t launch_rkl(const TopkParams& p, int64_t ws_bytes, bool aligned, hipStream_t st) {
  // the logits are only gathered from; what is written decides: MODE 2 takes any gradient row
  const int64_t need = p.grad && p.workspace ? rkl_workspace_bytes(Tag::id, p.n_rows, p.V, p.K) : 0;
  const bool two = need > 0 && ws_bytes >= need;
  const int J = p.K <= 256 ? 1 : p.K <= 512 ? 2 : 0;
  if (two) {
    const int64_t step = rkl_fill_rows(Tag::id, p.n_rows, p.V, p.K);
    const unsigned parts = (unsigned)rkl_fill_parts(Tag::id, p.n_rows, p.V, p.K);
    for (int64_t row0 = 0; row0 < p.n_rows; row0 += step) {
      const int64_t n = std::min(step, p.n_rows - row0);
      const dim3 rows((unsigned)n), by(256);
      if (J == 1) hipLaunchKernelGGL((rkl_values_kernel<Tag, 256, 1>), rows, by, TopkLds::bytes(p.K), st, p, row0);
      else if (J == 2) hipLaunchKernelGGL((rkl_values_kernel<Tag, 256, 2>), rows, by, TopkLds::bytes(p.K), st, p, row0);
      else hipLaunchKernelGGL((rkl_values_kernel<Tag, 256, 0>), rows, by, TopkLds::bytes(p.K), st, p, row0);
      const dim3 grid((unsigned)((n * parts + 7) / 8 * 8)), block(RKL_FILL_NT);
      if (aligned) hipLaunchKernelGGL((rkl_fill_kernel<Tag, 1>), grid, block, 0, st, p, row0, n, parts);
      else hipLaunchKernelGGL((rkl_fill_kernel<Tag, 2>), grid, block, 0, st, p, row0, n, parts);
    }
    return hipGetLastError();
  }
#define DL_LAUNCH_RKL(MODE, J) \
  hipLaunchKernelGGL((rkl_topk_kernel<Tag, 256, MODE, J>), dim3(xcd_banded_grid(p.n_rows)), dim3(256), TopkLds::bytes(p.K, 256), st, p)
  if (aligned) { if (J == 1) DL_LAUNCH_RKL(1, 1); else if (J == 2) DL_LAUNCH_RKL(1, 2); else DL_LAUNCH_RKL(1, 0); }
  else { if (J == 1) DL_LAUNCH_RKL(2, 1); else if (J == 2) DL_LAUNCH_RKL(2, 2); else DL_LAUNCH_RKL(2, 0); }
#undef DL_LAUNCH_RKL
  return hipGetLastError();
}

// Polls a part of a split row waits for its partners' records before it defers itself to the second launch.
constexpr int SPIN_LIMIT = 20000;

}  // namespace dl

