// FastTree tree-structured decode attention for gfx950 (MI355X): the two device kernels
// and the C ABI declared in include/fasttree_hip.h.
//
// Stage 1 computes, for every virtual node (a set of <= Q_TILE requests that share one run
// of KV tokens) and every KV head, the soft-max partial of those requests' query heads
// over that run.  All query rows of a vnode (requests x GQA group) form the N side of
// 16x16x32 MFMA tiles; the gathered K rows are the M side of S^T = K Q^T and the gathered
// V rows are read back from LDS transposed (ds_read_b64_tr_b16) as the M side of
// O^T = V^T P^T, so the probabilities go from the first contraction's accumulators
// straight into the second contraction's B operand without leaving registers.
//
// Stage 2 merges each request's partials with their log-sum-exp weights: D/4 lanes per (request,
// head), and several waves per list where whole lists would leave the machine idle.
//
// Reference for the arithmetic: kernel_bench/fasttree.py:299-413 (stage 1), :482-546
// (stage 2), :582-642 (the call that chains them).

#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <stdint.h>
#include <type_traits>

#include "../../include/fasttree_hip.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWave * kWavesPerBlock;
constexpr int kTileTokens = 32;          // KV tokens per inner step (two 16-token MFMA row blocks)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// ---------------------------------------------------------------------------------------
// Element-type traits: the 16-bit storage type only matters at the MFMA call and where
// fp32 probabilities / outputs are rounded to it.
// ---------------------------------------------------------------------------------------
struct F16 {
  static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ unsigned pack2(float lo, float hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(unsigned, v);
  }
  // what packing lo and hi rounded off, packed
  static __device__ __forceinline__ unsigned pack2_rest(float lo, float hi, unsigned packed) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 v = __builtin_bit_cast(h2, packed);
    return pack2(__builtin_fmaf((float)v[0], -1.f, lo), __builtin_fmaf((float)v[1], -1.f, hi));   // (one mixed instruction each)
  }
  // the lower (i = 0) or upper of a packed pair
  static __device__ __forceinline__ float of_pair(unsigned packed, int i) { return (float)__builtin_bit_cast(_Float16, (unsigned short)(packed >> (16 * i))); }
  // acc + lo + hi of a packed pair, in fp32
  static __device__ __forceinline__ float add_pair(unsigned packed, float acc) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 one = {(_Float16)1.f, (_Float16)1.f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, packed), one, acc, false);
  }
};
struct BF16 {
  static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ unsigned pack2(float lo, float hi) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    b2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(unsigned, v);
  }
  // what packing lo and hi rounded off, packed
  static __device__ __forceinline__ unsigned pack2_rest(float lo, float hi, unsigned packed) {
    return pack2(lo - __builtin_bit_cast(float, packed << 16), hi - __builtin_bit_cast(float, packed & 0xffff0000u));
  }
  static __device__ __forceinline__ float of_pair(unsigned packed, int i) { return __builtin_bit_cast(float, i ? packed & 0xffff0000u : packed << 16); }
  static __device__ __forceinline__ float add_pair(unsigned packed, float acc) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const b2 one = {(__bf16)1.f, (__bf16)1.f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, packed), one, acc, false);
  }
};

// Wave-wide exchange helpers.  v_permlane{16,32}_swap exchanges the odd 16-lane rows
// (upper 32-lane half) of its first operand with the even rows (lower half) of its second;
// fed the same value twice it yields (value of the even row / lower half, value of the odd
// row / upper half) in every lane.  The two results are copied into scalars before they are
// reinterpreted: a bit cast applied directly to an element of the returned vector reads
// element 0 for both.
struct LanePair { float lo, hi; };
__device__ __forceinline__ LanePair halves16(float x) {
  const unsigned a = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  return {__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1)};
}
__device__ __forceinline__ LanePair halves32(float x) {
  const unsigned a = __builtin_bit_cast(unsigned, x);
  auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  return {__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1)};
}
__device__ __forceinline__ float xor16_max(float x) { LanePair h = halves16(x); return fmaxf(h.lo, h.hi); }
__device__ __forceinline__ float xor32_max(float x) { LanePair h = halves32(x); return fmaxf(h.lo, h.hi); }
__device__ __forceinline__ float xor16_sum(float x) { LanePair h = halves16(x); return h.lo + h.hi; }
__device__ __forceinline__ float xor32_sum(float x) { LanePair h = halves32(x); return h.lo + h.hi; }
__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }
// x of the lane numbered `from` (0..63, may differ from lane to lane; every lane of the wave takes part).
__device__ __forceinline__ int lane_value(int x, int from) { return __builtin_amdgcn_ds_bpermute(4 * from, x); }
// The lane's number, opaque to the compiler: what is derived from it stays where it is used.  (In a
// kernel whose loops hold several kinds of work the compiler would otherwise compute every kind's
// lane addresses ahead of all of them and spill them: scratch reloads inside a stream of direct
// loads wait for the stream.)
__device__ __forceinline__ int lane_here() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  __builtin_assume(lane >= 0 && lane < 64);
  return lane;
}
// Orders this wave's LDS traffic around a point where lanes read what other lanes of the
// same wave wrote.  LDS executes one wave's instructions in order, so no wait is needed;
// the fences only stop the compiler from moving accesses across.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ float scale_from(float m_part, float m_all) {
  return (m_part == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_part - m_all);
}

// x / d for 0 <= x < 2^31 by a multiplication: mul = ceil(2^(31 + shift) / d) with shift = ceil(log2 d), whose
// excess over the exact factor is less than 2^-31 of it.  (The compiler's division by a value it does not know is
// some 25 instructions, and what runs once per block is fetched cold.)
struct Divisor {
  unsigned mul, shift;
  __host__ __device__ constexpr int operator()(int x) const { return (int)((unsigned)(((uint64_t)(2u * (unsigned)x) * mul) >> 32) >> shift); }
};
__host__ __device__ constexpr Divisor divisor(int d) {
  unsigned shift = 0;
  while ((int64_t(1) << shift) < d) ++shift;
  return Divisor{(unsigned)(((uint64_t(1) << (31 + shift)) + d - 1) / d), shift};
}
static_assert(divisor(1)(INT32_MAX) == INT32_MAX && divisor(64)(INT32_MAX) == INT32_MAX / 64 && divisor(7)(INT32_MAX) == INT32_MAX / 7 &&
              divisor(3)(INT32_MAX - 1) == (INT32_MAX - 1) / 3 && divisor(65535)(65534) == 0 && divisor(65535)(65535) == 1);

struct Stage1Args {
  const char* q;
  const char* k;
  const char* v;
  int64_t sq0, sq1, sk0, sk1, sv0, sv1;  // element strides
  const int32_t* kv_entries;
  const int32_t* kv_offs;
  const int32_t* kv_lens;
  const int32_t* q_entries;
  const int32_t* q_offs;
  const int32_t* q_lens;
  int vnode_begin, vnode_count;    // vnodes served by wide blocks (or the whole range for the per-wave-staging kernel)
  int narrow_begin, narrow_count;  // vnodes of at most 16 rows
  int narrow_share;                // waves that share one narrow vnode: 1, 2 or 4
  int wide_rows;                   // query rows the planner's tile gives a wide vnode (host hint for wide_chunks)
  int wide_chunks;                 // blocks per (wide vnode, kv head); block c serves row pieces c, c + wide_chunks, ..
  int block_slots;                 // blocks of the fused kernel the device runs at a time
  int join_rows;                   // most query rows neighbouring wide vnodes of one run are joined to (per block)
  // block programs written by the host (or null): four ints per program -- the wide vnodes
  // [first, end) of the wide range, then first and count of its narrow vnodes in the narrow range
  // (count < 0: they are served before the wide vnodes, else after them)
  const int32_t* prog_table;
  int num_programs;
  int narrow_in_programs;          // narrow vnodes (from narrow_begin) that programs serve
  // one record of kNarrowRecord ints per vnode of the narrow range, written by the host (or null):
  // what a wave needs to start on the vnode in one memory round trip instead of two -- the vnode's
  // four list entries, the requests of its rows and the pool slots of its first 32 tokens
  const int32_t* narrow_table;
  // one record of kProgRecord ints per program, written by the host (or null): what the block needs to
  // start on the program's first wide vnode -- see kProgRecord
  const int32_t* prog_records;
  int real_dim;                    // head dimension of the tensors; smaller than the kernel's D only for head_dim 16,
                                   // which the per-wave staging kernels compute as a zero-padded 32-dim contraction
  int g;
  int hkv;
  Divisor by_g, by_hkv, by_chunks;
  float scale_log2;  // sm_scale * log2(e)
  float* mid_o;
  int64_t so0, so1;
  float* mid_lse;
  int64_t sl0;
  // gathered (no-sharing) mode: vnode = (request, split) over a padded per-request cache
  const int32_t* cache_seqlens;
  int max_seqlen, kv_split, nsplit;
};

// How a kernel instance finds its vnode's slices.
struct VnodeView {
  int q_off;       // first scratch row
  int q_len;       // requests in this vnode
  int kv_len;      // tokens in the run
  int64_t kv_base; // tree mode: index into kv_entries; gathered mode: first cache row
};

// What every lane of the wave holds alike (read from LDS, or divided: integer division runs on vector
// registers) as scalars: loops over it then are scalar loops, and addresses made from it take no vector
// registers.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ VnodeView uniform(const VnodeView& w) {
  VnodeView u;
  u.q_off = __builtin_amdgcn_readfirstlane(w.q_off);
  u.q_len = __builtin_amdgcn_readfirstlane(w.q_len);
  u.kv_len = __builtin_amdgcn_readfirstlane(w.kv_len);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)w.kv_base), hi = __builtin_amdgcn_readfirstlane((unsigned)(w.kv_base >> 32));
  u.kv_base = (int64_t)(((uint64_t)hi << 32) | lo);
  return u;
}

// What a block of the fused kernel needs before it can ask for its record.  These are arguments of their own ahead of
// Stage1Args: built with -amdgpu-kernarg-preload-count, leading scalar arguments are in registers when a wave starts, and
// the record is asked for at once and not after a memory round trip for the arguments, which nothing has read before.  So are
// those of the kernels of narrow vnodes alone, of whole paths and of the merge; .2 us a launch (whole calls: 4 requests of a
// short prompt 6.44 -> 6.23 us, 16 of 32/32 heads 15.98 -> 15.60, 64 of 16/1 heads of 256 17.10 -> 16.56, 64 on a shared prefix
// 29.0 -> 28.6, a long document 42.8 -> 42.4).
#define FT_FIRST_PARAMETERS                                                                                        \
  const int32_t *first_table, const int32_t *first_records, const int32_t *first_narrow, int first_wide_blocks, int first_hkv, \
      unsigned first_mul, unsigned first_shift, int first_share, int first_items
#define FT_FIRST First{first_table, first_records, first_narrow, first_wide_blocks, first_hkv, Divisor{first_mul, first_shift}, first_share, first_items}
struct First {
  const int32_t *prog_table, *prog_records, *narrow_table;
  int wide_blocks, hkv;
  Divisor by_hkv;
  int narrow_share, narrow_items;
};
constexpr int kFirstBytes = sizeof(First);
static_assert(kFirstBytes == 3 * 8 + 6 * 4 && kFirstBytes % 8 == 0, "the parameters lie as the struct does");

// The kernel's arguments, read anew from where the launch put them, by code that one path of a kernel runs:
// what a path has read as a reference to the kernel's own parameter is held in scalar registers from its start
// on, beside what the other paths hold, and spilled into lanes of vector registers: 688 reads of such lanes in
// the fused kernel for the planner's lists (head_dim 128), 95 where each path reads its own arguments; a narrow
// wave of a single tile executed 777 vector instructions, 570 in the kernel without wide code.  387 requests with
// 28-token leaves, 32/32 heads: 65.4 -> 61.2 us; 240 of 32/8 heads with 160 tokens 53.8 -> 49.5; the 400-request
// tree in the reference's lists 63.2 -> 61.1.
__device__ __forceinline__ const Stage1Args& args_again() {
  auto p = (const __attribute__((address_space(4))) Stage1Args*)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + kFirstBytes);
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+s"(p));
#endif
  return *(const Stage1Args*)p;
}

// The plan's lists and tables, which no kernel writes, as the constant address space: reads at an address that
// is the same for the whole wave are scalar loads wherever they stand.
typedef const int32_t __attribute__((address_space(4)))* PlanInts;
__device__ __forceinline__ PlanInts plan_ints(const int32_t* p) { return (PlanInts)(uintptr_t)p; }

template <bool GATHERED>
__device__ __forceinline__ VnodeView load_vnode(const Stage1Args& a, int vnode) {
  VnodeView w;
  if constexpr (GATHERED) {
    int req = vnode / a.nsplit, split = vnode - req * a.nsplit;
    int len = plan_ints(a.cache_seqlens)[req] - split * a.kv_split;
    w.kv_len = len < 0 ? 0 : (len > a.kv_split ? a.kv_split : len);
    w.kv_base = (int64_t)req * a.max_seqlen + (int64_t)split * a.kv_split;
    w.q_off = vnode;
    w.q_len = 1;
  } else {
    w.q_off = plan_ints(a.q_offs)[vnode];
    w.q_len = plan_ints(a.q_lens)[vnode];
    w.kv_len = plan_ints(a.kv_lens)[vnode];
    w.kv_base = plan_ints(a.kv_offs)[vnode];
  }
  return w;
}

// Per-wave LDS staging of one 32-token tile.  Row pitches are chosen for the two read
// patterns: K rows are read 16 B per lane by 16 different rows at a time (pitch = 4 dwords
// mod 64 banks), V rows are read by ds_read_b64_tr_b16, where 16 lanes cover 4 rows x 32 B
// (pitch = 8 dwords mod 32 banks).
template <int D> struct TileGeom {
  static constexpr int kRowBytes = D * 2;
  static constexpr int kPitchK = kRowBytes + 16;
  static constexpr int kPitchV = kRowBytes + 32;
  static constexpr int kBytesK = kTileTokens * kPitchK;
  static constexpr int kBytesV = kTileTokens * kPitchV;
  static constexpr int kBytes = kBytesK + kBytesV;     // per wave
  static constexpr int kLanesPerRow = D / 8;           // 16-byte chunks in a row
  static constexpr int kRowsPerLoad = kWave / kLanesPerRow;
  static constexpr int kLoads = kTileTokens / kRowsPerLoad;
};

// Running soft-max state of one wave for NQB blocks of 16 query rows.  Accumulators are
// O^T tiles: lane l holds o[qb][db][j] = O[row 16*qb + l%16][dim 16*db + 4*(l/16) + j].
template <int D, int NQB> struct WaveState {
  f32x4 o[NQB][D / 16];
  float m[NQB];  // running max of scaled scores, log2 domain, identical in the 4 lanes of a row
  float l[NQB];  // running sum of this lane's own probabilities (reduced over lanes at the end)
};

// Query fragments of one wave (B operand of S^T = K Q^T): qf[qb][ks] holds, for row
// row0 + 16*qb + lane%16, the 8 dims 32*ks + 8*(lane/16) .. +7.  Rows past the vnode are zero.
template <int D, int NQB, bool GATHERED>
__device__ __forceinline__ void load_q_frags(const Stage1Args& a, const VnodeView& vn, int kvh, int row0,
                                             u32x4 (&qf)[NQB][D / 32]) {
  constexpr int KS = D / 32;
  const int lane = threadIdx.x & 63;
  const int p = lane & 15, c = lane >> 4;
  const int rows_total = vn.q_len * a.g;
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
    const int r = row0 + 16 * qb + p;
    const bool ok = r < rows_total;
    const int ri = ok ? r / a.g : 0;
    const int rj = ok ? r - ri * a.g : 0;
    const int64_t entry = ok ? (GATHERED ? (int64_t)(vn.q_off / a.nsplit) : (int64_t)a.q_entries[vn.q_off + ri]) : 0;
    const char* src = a.q + 2 * (entry * a.sq0 + (int64_t)(kvh * a.g + rj) * a.sq1 + 8 * c);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 z = {0u, 0u, 0u, 0u};
      qf[qb][ks] = ok && 32 * ks + 8 * c < a.real_dim ? *reinterpret_cast<const u32x4*>(src + 64 * ks) : z;
    }
  }
}

template <int D, int NQB>
__device__ __forceinline__ void reset_state(WaveState<D, NQB>& st) {
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
    st.m[qb] = -INFINITY;
    st.l[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) st.o[qb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// every lane of a row gets the row's full probability sum
template <int D, int NQB>
__device__ __forceinline__ void finish_state(WaveState<D, NQB>& st) {
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) st.l[qb] = xor32_sum(xor16_sum(st.l[qb]));
}

// One 32-token step of a wave: scores of its NQB*16 rows against the tile staged at
// (ldsK, ldsV), online soft-max update, P.V.  `valid` (>= 1) is how many of the 32 tokens exist.
template <typename E, int D, int NQB>
__device__ __forceinline__ void tile_step(const char* ldsK, const char* ldsV, int valid, float sc,
                                          const u32x4 (&qf)[NQB][D / 32], WaveState<D, NQB>& st) {
  using G = TileGeom<D>;
  constexpr int KS = D / 32, DB = D / 16;
  const int lane = threadIdx.x & 63;
  const int p = lane & 15, c = lane >> 4;

  // ---- S^T = K Q^T : s[tb][qb][j] = score(token 16*tb + 4*c + j, row 16*qb + p)
  f32x4 s[2][NQB];
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) s[tb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 kf = *reinterpret_cast<const u32x4*>(ldsK + (16 * tb + p) * G::kPitchK + 64 * ks + 16 * c);
#pragma unroll
      for (int qb = 0; qb < NQB; ++qb) s[tb][qb] = E::mfma(kf, qf[qb][ks], s[tb][qb]);
    }
  }

  // tokens past the end of the run score -inf (wave-uniform branch: only a run's last tile)
  if (valid < kTileTokens) {
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * tb + 4 * c + j >= valid) {
#pragma unroll
          for (int qb = 0; qb < NQB; ++qb) s[tb][qb][j] = -INFINITY;
        }
  }

  // Online soft-max with a lazily updated reference: a row's reference m only moves when the
  // row's running maximum exceeds it by more than kSlack (log2 units), so probabilities stay
  // below 2^kSlack -- exact in any case, since numerator and denominator share the reference --
  // and the accumulators are rescaled rarely instead of on almost every tile.
  constexpr float kSlack = 8.f;
  u32x4 pf[NQB];
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
    float mx = fmaxf(fmaxf(fmaxf(s[0][qb][0], s[0][qb][1]), fmaxf(s[0][qb][2], s[0][qb][3])),
                     fmaxf(fmaxf(s[1][qb][0], s[1][qb][1]), fmaxf(s[1][qb][2], s[1][qb][3])));
    mx = xor32_max(xor16_max(mx)) * sc;      // sc > 0; finite: the tile holds at least one token
    const float m_old = st.m[qb];
    const bool grow = mx > m_old + kSlack;   // also true on the first tile (m_old = -inf)
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float m_new = grow ? mx : m_old;
      const float alpha = __builtin_amdgcn_exp2f(m_old - m_new);
      st.l[qb] *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) st.o[qb][db] *= alpha;
      st.m[qb] = m_new;
    }
    const float neg_m = -st.m[qb];
    float x[8];
    float sum = 0.f;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[4 * tb + j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tb][qb][j], sc, neg_m));
        sum += x[4 * tb + j];
      }
    st.l[qb] += sum;
    pf[qb] = u32x4{E::pack2(x[0], x[1]), E::pack2(x[2], x[3]), E::pack2(x[4], x[5]), E::pack2(x[6], x[7])};
  }

  // ---- O^T += V^T P^T : A operand rows = dims 16*db + p, k slots = the 8 tokens this lane's P holds
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    const char* va = ldsV + (4 * c + (p >> 2)) * G::kPitchV + 2 * (16 * db + 4 * (p & 3));
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(va));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(va + 16 * G::kPitchV));
    const u32x2 lo2 = __builtin_bit_cast(u32x2, lo), hi2 = __builtin_bit_cast(u32x2, hi);
    const u32x4 vf = {lo2[0], lo2[1], hi2[0], hi2[1]};
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) st.o[qb][db] = E::mfma(vf, pf[qb], st.o[qb][db]);
  }
}

// One wave attends NQB*16 query rows to tokens [tile0*32, ...) in steps of tile_step_n tiles,
// staging each tile in its own LDS area.  Rows travel global -> registers -> LDS; the next tile
// is in flight while a tile is consumed.  (Used for head_dim 16 only, as a zero-padded 32.)
template <typename E, int D, int NQB, bool GATHERED>
__device__ __forceinline__ void wave_attend(const Stage1Args& a, const VnodeView& vn, int kvh, int row0,
                                            int tile0, int tile_step_n, char* lds, WaveState<D, NQB>& st) {
  using G = TileGeom<D>;
  const int lane = threadIdx.x & 63;
  char* ldsK = lds;
  char* ldsV = lds + G::kBytesK;

  u32x4 qf[NQB][D / 32];
  load_q_frags<D, NQB, GATHERED>(a, vn, kvh, row0, qf);
  reset_state<D, NQB>(st);

  const int ntiles = (vn.kv_len + kTileTokens - 1) / kTileTokens;
  if (tile0 >= ntiles) return;

  // rows by 16-byte chunks, coalesced per row
  const int ld_row = lane / G::kLanesPerRow, ld_chunk = lane % G::kLanesPerRow;
  const char* kbase = a.k + 2 * ((int64_t)kvh * a.sk1) + 16 * ld_chunk;
  const char* vbase = a.v + 2 * ((int64_t)kvh * a.sv1) + 16 * ld_chunk;
  auto load_slots = [&](int tile, int (&slot)[G::kLoads]) {
#pragma unroll
    for (int i = 0; i < G::kLoads; ++i) {
      const int t = tile * kTileTokens + i * G::kRowsPerLoad + ld_row;
      slot[i] = -1;
      if (tile < ntiles && t < vn.kv_len) slot[i] = GATHERED ? t : a.kv_entries[vn.kv_base + t];
    }
  };
  auto load_rows = [&](const int (&slot)[G::kLoads], u32x4 (&kreg)[G::kLoads], u32x4 (&vreg)[G::kLoads]) {
#pragma unroll
    for (int i = 0; i < G::kLoads; ++i) {
      u32x4 z = {0u, 0u, 0u, 0u};
      kreg[i] = z;
      vreg[i] = z;
      if (slot[i] >= 0 && 8 * ld_chunk < a.real_dim) {   // (chunks past a 16-dim row stay zero)
        const int64_t srow = GATHERED ? (vn.kv_base + slot[i]) : (int64_t)slot[i];
        kreg[i] = *reinterpret_cast<const u32x4*>(kbase + 2 * srow * a.sk0);
        vreg[i] = *reinterpret_cast<const u32x4*>(vbase + 2 * srow * a.sv0);
      }
    }
  };
  auto stage = [&](const u32x4 (&kreg)[G::kLoads], const u32x4 (&vreg)[G::kLoads]) {
#pragma unroll
    for (int i = 0; i < G::kLoads; ++i) {
      const int row = i * G::kRowsPerLoad + ld_row;
      *reinterpret_cast<u32x4*>(ldsK + row * G::kPitchK + 16 * ld_chunk) = kreg[i];
      *reinterpret_cast<u32x4*>(ldsV + row * G::kPitchV + 16 * ld_chunk) = vreg[i];
    }
    wave_lds_fence();
  };

  int slot[G::kLoads];
  u32x4 kreg[G::kLoads], vreg[G::kLoads];
  load_slots(tile0, slot);
  load_rows(slot, kreg, vreg);
  for (int tile = tile0; tile < ntiles; tile += tile_step_n) {
    stage(kreg, vreg);
    if (tile + tile_step_n < ntiles) {
      load_slots(tile + tile_step_n, slot);
      load_rows(slot, kreg, vreg);
    }
    tile_step<E, D, NQB>(ldsK, ldsV, vn.kv_len - tile * kTileTokens, a.scale_log2, qf, st);
    wave_lds_fence();
  }
  finish_state<D, NQB>(st);
}

// (PADDED: the kernel's D may be more than the tensors' head dimension)
template <int D, int NQB, bool PADDED = false>
__device__ __forceinline__ void write_partials(const Stage1Args& a, const VnodeView& vn, int kvh, int row0,
                                               const WaveState<D, NQB>& st, int ngroups = NQB) {
  constexpr int DB = D / 16;
  const int lane = lane_here();
  const int p = lane & 15, c = lane >> 4;
  const int rows_total = vn.q_len * a.g;
#pragma unroll
  for (int qb = 0; qb < NQB; ++qb) {
    const int r = row0 + 16 * qb + p;
    if (qb >= ngroups || r >= rows_total) continue;
    const int ri = a.by_g(r), rj = r - ri * a.g;
    const int64_t row = vn.q_off + ri;
    const int head = kvh * a.g + rj;
    const float l = st.l[qb];
    const float inv = l > 0.f ? 1.f / l : 0.f;
    float* dst = a.mid_o + row * a.so0 + (int64_t)head * a.so1 + 4 * c;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      if (!PADDED || 16 * db < a.real_dim) *reinterpret_cast<f32x4*>(dst + 16 * db) = st.o[qb][db] * inv;
    if (c == 0) a.mid_lse[row * a.sl0 + head] = l > 0.f ? (__builtin_amdgcn_logf(l) + st.m[qb]) * kLn2 : -INFINITY;
  }
}

// Merge of the four waves' states of one block (each over the same rows, different tokens)
// into wave 0, pairwise through LDS: waves {2,3} -> {0,1}, then wave 1 -> wave 0.
template <int D, int NQB>
__device__ __forceinline__ void merge_waves(float* xchg, WaveState<D, NQB>& st) {
  constexpr int NV = NQB * (D / 16) * 4 + 2 * NQB;  // floats of state per lane
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int half = 2; half >= 1; half >>= 1) {
    __syncthreads();
    if (wave >= half && wave < 2 * half) {
      float* dst = xchg + (size_t)(wave - half) * NV * kWave + lane;
      int n = 0;
#pragma unroll
      for (int qb = 0; qb < NQB; ++qb) {
        dst[(n++) * kWave] = st.m[qb];
        dst[(n++) * kWave] = st.l[qb];
#pragma unroll
        for (int db = 0; db < D / 16; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j) dst[(n++) * kWave] = st.o[qb][db][j];
      }
    }
    __syncthreads();
    if (wave < half) {
      const float* src = xchg + (size_t)wave * NV * kWave + lane;
      int n = 0;
#pragma unroll
      for (int qb = 0; qb < NQB; ++qb) {
        const float m2 = src[(n++) * kWave];
        const float l2 = src[(n++) * kWave];
        const float m = fmaxf(st.m[qb], m2);
        const float a1 = scale_from(st.m[qb], m), a2 = scale_from(m2, m);
        st.l[qb] = st.l[qb] * a1 + l2 * a2;
        st.m[qb] = m;
#pragma unroll
        for (int db = 0; db < D / 16; ++db)
#pragma unroll
          for (int j = 0; j < 4; ++j) st.o[qb][db][j] = st.o[qb][db][j] * a1 + src[(n++) * kWave] * a2;
      }
    }
  }
}

// SPLIT_WAVES = true : one block per (vnode, kv head); its 4 waves take every 4th KV tile and
//                      their states are merged through LDS (wide vnodes, long runs).
// SPLIT_WAVES = false: one wave per (vnode, kv head), 4 vnodes per block (narrow vnodes).
template <typename E, int D, int NQB, bool SPLIT_WAVES, bool GATHERED>
__global__ void __launch_bounds__(kBlock) stage1_kernel(Stage1Args a) {
  using G = TileGeom<D>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int kvh = blockIdx.y;
  char* my_lds = smem + wave * G::kBytes;

  if constexpr (!SPLIT_WAVES) {
    const int local = blockIdx.x * kWavesPerBlock + wave;
    if (local >= a.vnode_count) return;
    const VnodeView vn = load_vnode<GATHERED>(a, a.vnode_begin + local);
    const int rows_total = vn.q_len * a.g;
    for (int row0 = 0; row0 < rows_total; row0 += 16 * NQB) {
      WaveState<D, NQB> st;
      wave_attend<E, D, NQB, GATHERED>(a, vn, kvh, row0, 0, 1, my_lds, st);
      write_partials<D, NQB, true>(a, vn, kvh, row0, st);
    }
  } else {
    const VnodeView vn = load_vnode<GATHERED>(a, a.vnode_begin + blockIdx.x);
    const int rows_total = vn.q_len * a.g;
    for (int row0 = 0; row0 < rows_total; row0 += 16 * NQB) {
      WaveState<D, NQB> st;
      wave_attend<E, D, NQB, GATHERED>(a, vn, kvh, row0, wave, kWavesPerBlock, my_lds, st);
      merge_waves<D, NQB>(reinterpret_cast<float*>(smem), st);
      if (wave == 0) write_partials<D, NQB, true>(a, vn, kvh, row0, st);
      __syncthreads();  // staging LDS is reused by the next row chunk
    }
  }
}

// ---------------------------------------------------------------------------------------
// Wide vnodes: four waves per block and two blocks per compute unit, so that two waves share a
// SIMD and one wave's waits are filled by the other's instructions.
//
// What bounds a launch is the start, the waits and the end of its blocks, with the matrix pipes far
// from full: 1.07 PFLOP/s where two blocks of 192 rows on each unit read one run of 8192 tokens (the
// pipes busy 49 % of the cycles at 2090 MHz; a large library matrix product reaches 1.21), and .60
// in a decode step of 400 requests, whose blocks run for some 30 steps (24 %, 2633 MHz).  48 query
// rows per wave read a K or V operand from LDS once for three row groups and spread a tile's loads
// and barrier over 1.5 times the rows: a step of 96 rows takes .52 us against .69 with 32x32x16
// instructions and 32 rows per wave, 192 rows .86 (head_dim 128, 8 runs of 8 heads).
// 48 rows take 96 accumulator and 48 query registers of the 256 a wave has.
// ---------------------------------------------------------------------------------------
constexpr int kWideWaves = 4;
constexpr int kWideBlock = kWave * kWideWaves;
constexpr int kWaveSlotsPerCu = 8;                // waves of these kernels a compute unit holds
// 16-row groups a wave serves per pass, and query rows a block does
template <int D> struct WideRows {
  static constexpr int kGroups = D <= 128 ? 3 : 2;
  static constexpr int kBlock = 16 * kGroups * kWideWaves;
};
constexpr int kDeftRows = 32 * kWideWaves;        // (the comparison engine's kernel: 32 rows per wave)

// The XOR that places the 16-byte chunks of a row in LDS.  A K operand is read by 16 rows x 4 chunks in 16-byte
// words, of which rows 0-3 and 12-15 of one chunk go together with rows 4-11 of the next; a V operand, transposed, by
// 16 rows x 2 chunks in 8-byte words, 8 rows at a time: either has to hit all 64 banks.  Rows of 256 bytes and more
// start at the same bank, and their two low bits move a row by 4 chunks; shorter ones fill the banks between them.
// The next two bits, negated, set the quarters apart in both.  (The 400-request tree at head_dim 128: no conflicts
// counted in 4.5 million cycles of LDS access; with the two pairs of bits swapped, which suits the 32-row operands of
// 32x32x16 instructions, 4.0 million of 8.5: 62.4 -> 61.5 us.  Either serves those too.)
template <int D> __device__ __forceinline__ constexpr int chunk_swizzle(int row) {
  return (D >= 128 ? (row & 3) << 2 : D == 64 ? (row & 2) << 1 : 0) | (-(row >> 2) & 3);
}

// LDS layout of the wide kernel: rows of 2*D bytes back to back (no padding), 64-token super
// tiles of two 32-token tiles, a ring of kBufs buffers, then the rings of slot indices.  A row's 16-byte chunks are stored XOR-permuted: chunk c of row r sits in slot
// c ^ swz(r) (chunk_swizzle above).  Loads go global -> LDS directly; one wave instruction fills a 1 KB
// group of consecutive rows.
template <int D> struct WideGeom {
  static constexpr int kRowBytes = 2 * D;
  static constexpr int kChunks = D / 8;                  // 16-byte chunks per row
  static constexpr int kSub = 2;
  static constexpr int kTokens = kSub * kTileTokens;     // 64
  static constexpr int kBufs = 2;
  static constexpr int kTileBytes = kTileTokens * kRowBytes;
  static constexpr int kBytesK = kTokens * kRowBytes;
  static constexpr int kBytes = 2 * kBytesK;             // K + V of one buffer
  static constexpr int kRing = kBufs * kBytes;
  static constexpr int kGroupRows = kWave / kChunks;     // rows per 1 KB load group
  static constexpr int kGroups = kTokens / kGroupRows;   // groups per matrix and super tile
  static constexpr int kUnits = 2 * kGroups / kWideWaves;                       // loads per wave and super tile
  static constexpr int kSlots = kGroups >= kWideWaves ? kGroups / kWideWaves : 1;  // distinct rows among them
  static constexpr int kIdxBytes = kWideWaves * 4 * 4 * kTokens;                   // per wave: the slot indices of four super tiles
  static constexpr int kLds = kRing + kIdxBytes;
  static __device__ __forceinline__ int swz(int row) { return chunk_swizzle<D>(row); }
};

// State of one wave for 32 query rows (32x32x16 tiles).  o[db][j] = O[row lane%32][dim 32*db + 8*(j/4) +
// 4*(lane/32) + j%4]; m = soft-max reference (scaled scores, log2 domain); l = this lane's own
// share of the row sum until finish_state().
template <int D> struct WideState {
  f32x16 o[D / 32];
  float m;
  float l;
};

template <int D>
__device__ __forceinline__ void reset_state(WideState<D>& st) {
  st.m = -INFINITY;
  st.l = 0.f;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int j = 0; j < 16; ++j) st.o[db][j] = 0.f;
}

// The record of a block program (kProgRecord ints): entries 0..3 are kv_off, kv_len, q_off and q_len of the
// program's first wide vnode (if it has one, with or without the rest), entry 4 says whether the rest is there (the
// vnode exists and has at most 128 requests), entries kProgRecRequests.. the requests of its scratch rows, entries
// kProgRecSlots.. the pool slots of its first 64 tokens (the last token repeated past the end of a shorter run).
// With it a block knows after one memory round trip what it otherwise learns in three (its table entry, the
// vnode's list entries, the request and slot lists) before it can ask for query and K/V rows.
constexpr int kProgRecord = 256;
constexpr int kProgRecRequests = 8;
constexpr int kProgRecSlots = kProgRecRequests + 128;
static_assert(kProgRecSlots + 64 <= kProgRecord);

// Query fragments of a wave's 32 rows, loaded in two steps so that other loads can be put between the two
// dependent ones: the address of a lane's row (needs the request id of the row, one load), then the
// fragments.  qf[ks]: row row0 + lane%32, dims 16*ks + 8*(lane/32) .. +7; zero past the vnode (src == nullptr).
__device__ __forceinline__ const char* q_row_address32(const Stage1Args& a, const VnodeView& vn, int kvh, int row0) {
  const int lane = threadIdx.x & 63;
  const int r = row0 + (lane & 31), h = lane >> 5;
  if (r >= vn.q_len * a.g) return nullptr;
  const int ri = a.by_g(r);
  const int rj = r - ri * a.g;
  const int64_t entry = (int64_t)a.q_entries[vn.q_off + ri];
  return a.q + 2 * (entry * a.sq0 + (int64_t)(kvh * a.g + rj) * a.sq1 + 8 * h);
}
template <int D>
__device__ __forceinline__ void load_q_frags32(const char* src, u32x4 (&qf)[D / 16]) {
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    u32x4 z = {0u, 0u, 0u, 0u};
    qf[ks] = src ? *reinterpret_cast<const u32x4*>(src + 32 * ks) : z;
  }
}

// Per-lane LDS byte addresses of the operand reads inside tile 0 of the current buffer, for
// contraction step / dim block 0.  Thanks to the XOR layout the address for step ks (dim block
// db) is the base with 32*ks (64*db) XOR-ed in; the second tile of the super tile is a constant
// offset away and buffer b of the ring is b * kBytes further (the ring starts on a multiple of the
// row size).
struct WideLane {
  unsigned k;     // K operand: row lane%32, chunk lane/32 (step ks: chunk 2*ks + lane/32)
  unsigned v_lo;  // transposed V read: tokens 4*(lane/32) + 0..3 (+16 for u = 1), dims 0..31
  unsigned v_hi;  // same, tokens + 8
};

template <int D>
__device__ __forceinline__ void init_lane(WideLane& la, unsigned ring) {
  using W = WideGeom<D>;
  const int lane = threadIdx.x & 63;
  const int p32 = lane & 31, h = lane >> 5, p = lane & 15, gi = (lane >> 4) & 1;
  la.k = ring + p32 * W::kRowBytes + 16 * ((h & (W::kChunks - 1)) ^ W::swz(p32));
  const int row_lo = 4 * h + (p >> 2), row_hi = row_lo + 8;
  const int chunk = (2 * gi + ((p & 3) >> 1)) & (W::kChunks - 1);
  la.v_lo = ring + W::kBytesK + row_lo * W::kRowBytes + 16 * (chunk ^ W::swz(row_lo)) + 8 * (p & 1);
  la.v_hi = ring + W::kBytesK + row_hi * W::kRowBytes + 16 * (chunk ^ W::swz(row_hi)) + 8 * (p & 1);
}

// Byte offset of an object of the block's dynamic LDS segment within LDS.
__device__ __forceinline__ unsigned lds_offset(const void* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

__device__ __forceinline__ WideLane at_buffer(const WideLane& la0, unsigned buffer_offset) {
  return WideLane{la0.k + buffer_offset, la0.v_lo + buffer_offset, la0.v_hi + buffer_offset};
}

// 16 bytes per lane from global memory straight into LDS at lds_base + 16 * lane (lds_base is
// wave uniform).  Written as assembly on purpose: for the builtin the compiler cannot tell which
// later LDS reads touch the landing bytes and makes every one of them wait for all such loads
// in flight, which serialises the stream with the arithmetic.  Completion is awaited by hand
// with wait_direct_loads<N>() before the block barrier that publishes a buffer.
__device__ __forceinline__ void load_direct16(const char* src, unsigned lds_base) {
  // (M0 holds the LDS address: bound as an operand, so the compiler writes it and knows it is live)
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "{m0}"(lds_base) : "memory");
}
// The same for 4 bytes per lane at base + offset (base wave uniform), landing at lds_base + 4 * lane.
// A vector memory instruction may read a scalar register five wait states after a vector instruction wrote it (a
// spilled base comes back by v_readlane), and inside assembly the compiler does not see to that.
__device__ __forceinline__ void load_direct4(const void* base, unsigned offset, unsigned lds_base) {
  asm volatile("s_nop 4\n\tglobal_load_lds_dword %0, %1" ::"v"(offset), "s"(base), "{m0}"(lds_base) : "memory");
}
// Wait until at most N of this wave's vector-memory operations are still in flight (they finish
// in order).
template <int N>
__device__ __forceinline__ void wait_direct_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ u32x4 lds_read16(unsigned addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>((uintptr_t)addr);
}
__device__ __forceinline__ unsigned lds_read4(unsigned addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) unsigned*>((uintptr_t)addr);
}
__device__ __forceinline__ u32x2 lds_read_tr8(unsigned addr) {
  const i16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      reinterpret_cast<__attribute__((address_space(3))) i16x4*>((uintptr_t)addr));
  return __builtin_bit_cast(u32x2, v);
}

// The soft-max reference m of a row is updated lazily: only when the row's running maximum
// exceeds it by more than kSlack (log2 units).  Probabilities therefore stay below 2^kSlack --
// exact in any case, since numerator and denominator share the reference -- and the
// accumulators are rescaled rarely (in practice once, on a run's first tile).
constexpr float kSlack = 8.f;

// A tile step without a per-query mask (every row of the vnode attends every token of the run).
struct NoMask {
  __device__ __forceinline__ void operator()(f32x16&) const {}
};

// One 32-token step for the wave's 32 rows on the tile `off` bytes into the current buffer.
// S^T = K Q^T: A = K rows (token lane%32, 8 dims per lane), B = Q; accumulator register j of a
// lane is token 8*(j/4) + 4*(lane/32) + j%4.  Registers 8u .. 8u+7 are exactly the 8 k-slots a
// lane feeds to the u-th P.V contraction, whose A operand (V^T) comes from two transposed LDS
// reads of 4 consecutive tokens each.  valid < 32 only on a run's last, partial tile.  `mask`
// is applied to the raw scores (it overwrites those of tokens the lane's row does not attend).
template <typename E, int D, typename Mask = NoMask>
__device__ __forceinline__ void tile_step32(const WideLane& la, unsigned off, int valid, float sc,
                                            const u32x4 (&qf)[D / 16], WideState<D>& st, const Mask& mask = Mask()) {
  using W = WideGeom<D>;
  constexpr int KS = D / 16, DB = D / 32, NV = 2 * DB;

  // the K operands are requested eight contraction steps at a time, before the first of those
  // steps needs one (all of them at once up to head_dim 128)
  const unsigned kb = la.k + off;
  constexpr int KB = KS < 8 ? KS : 8;
  f32x16 s;
#pragma unroll
  for (int j = 0; j < 16; ++j) s[j] = 0.f;
#pragma unroll
  for (int k0 = 0; k0 < KS; k0 += KB) {
    u32x4 kf[KB];
#pragma unroll
    for (int ks = 0; ks < KB; ++ks) kf[ks] = lds_read16(kb ^ (32u * (k0 + ks)));
    // (keeps the scheduler from sinking each read next to its use, which would expose the full
    // LDS latency eight times in a row)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KB; ++ks) s = E::mfma32(kf[ks], qf[k0 + ks], s);
  }

  if (valid < kTileTokens) {  // wave uniform
    asm volatile("" ::: "memory");  // keeps this a branch: as selects it would run on every tile
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = (8 * (j >> 2) + 4 * h + (j & 3) >= valid) ? -INFINITY : s[j];
  }
  mask(s);

  // the V^T operands do not depend on the probabilities: request them now, so that they arrive
  // under the soft-max arithmetic (they take the registers the K operands just left); at
  // head_dim 256 only those of the first 16 tokens, the others after the first half of P.V
  const unsigned vlo = la.v_lo + off, vhi = la.v_hi + off;
  constexpr int VH = D > 128 ? DB : NV;   // operands requested ahead of the soft-max
  u32x4 vf[VH];
  auto read_v = [&](int i) {
    const int u = i / DB, db = i % DB;
    const u32x2 lo = lds_read_tr8((vlo ^ (64u * db)) + u * 16 * W::kRowBytes);
    const u32x2 hi = lds_read_tr8((vhi ^ (64u * db)) + u * 16 * W::kRowBytes);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  };
#pragma unroll
  for (int i = 0; i < VH; ++i) vf[i] = read_v(i);
  __builtin_amdgcn_sched_barrier(0);
  float mx = max3(s[0], s[1], s[2]);
#pragma unroll
  for (int j = 3; j < 15; j += 2) mx = max3(mx, s[j], s[j + 1]);
  mx = xor32_max(fmaxf(mx, s[15])) * sc;  // sc > 0; finite: the tile holds at least one token
  const bool grow = mx > st.m + kSlack;   // also true on a run's first tile (m = -inf)
  if (__builtin_amdgcn_ballot_w64(grow)) {
    const float m_new = grow ? mx : st.m;
    const float alpha = __builtin_amdgcn_exp2f(st.m - m_new);
    st.l *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db) st.o[db] *= alpha;
    st.m = m_new;
  }

  const float neg_m = -st.m;
  float x[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) x[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j], sc, neg_m));
  u32x4 pf[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    pf[u] = u32x4{E::pack2(x[8 * u + 0], x[8 * u + 1]), E::pack2(x[8 * u + 2], x[8 * u + 3]),
                  E::pack2(x[8 * u + 4], x[8 * u + 5]), E::pack2(x[8 * u + 6], x[8 * u + 7])};
  // the row sum is taken over the probabilities as P.V will see them (rounded to the storage
  // type), two per instruction
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) st.l = E::add_pair(pf[u][i], st.l);

#pragma unroll
  for (int i = 0; i < VH; ++i) st.o[i % DB] = E::mfma32(vf[i], pf[i / DB], st.o[i % DB]);
  if constexpr (VH < NV) {
    u32x4 vg[NV - VH];
#pragma unroll
    for (int i = VH; i < NV; ++i) vg[i - VH] = read_v(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = VH; i < NV; ++i) st.o[i % DB] = E::mfma32(vg[i - VH], pf[i / DB], st.o[i % DB]);
  }
}

template <int D>
__device__ __forceinline__ void finish_state(WideState<D>& st) {
  st.l = xor32_sum(st.l);
}

// (ROUND16: the normalised output is rounded to fp16 on its way to the fp32 scratch)
template <int D, bool ROUND16 = false>
__device__ __forceinline__ void write_partials32(const Stage1Args& a, const VnodeView& vn, int kvh, int row0,
                                                 const WideState<D>& st) {
  const int lane = threadIdx.x & 63;
  const int r = row0 + (lane & 31), h = lane >> 5;
  if (r >= vn.q_len * a.g) return;
  const int ri = r / a.g, rj = r - ri * a.g;
  const int64_t row = vn.q_off + ri;
  const int head = kvh * a.g + rj;
  const float inv = st.l > 0.f ? 1.f / st.l : 0.f;
  float* dst = a.mid_o + row * a.so0 + (int64_t)head * a.so1 + 4 * h;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      f32x4 v = {st.o[db][4 * jj] * inv, st.o[db][4 * jj + 1] * inv, st.o[db][4 * jj + 2] * inv,
                 st.o[db][4 * jj + 3] * inv};
      if constexpr (ROUND16) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (float)(_Float16)v[e];
      }
      *reinterpret_cast<f32x4*>(dst + 32 * db + 8 * jj) = v;
    }
  if (h == 0) a.mid_lse[row * a.sl0 + head] = st.l > 0.f ? (__builtin_amdgcn_logf(st.l) + st.m) * kLn2 : -INFINITY;
}

// Per-lane LDS byte addresses of a wave's 16x16x32 operand reads inside a 32-token tile (of a wide
// block's ring: tile 0 of the first buffer), for contraction step / dim block 0.  The XOR layout makes the address for step ks
// (dim block db) the base with 64*ks (32*db) XOR-ed in; the second 16 tokens of a tile, the second
// tile of a super tile and the second buffer are constant offsets away.
struct WideLane16 {
  unsigned k;   // K operand: token lane%16, chunk lane/16 (step ks: chunk 4*ks + lane/16)
  unsigned v;   // transposed V read: tokens 4*(lane/16) .. +3, dims 4*(lane%4) .. +3
};
template <int D>
__device__ __forceinline__ WideLane16 init_lane16(unsigned k_tile, unsigned v_tile) {
  using W = WideGeom<D>;
  const int lane = lane_here(), p = lane & 15, c = lane >> 4;
  const int vr = 4 * c + (p >> 2);
  return WideLane16{k_tile + p * W::kRowBytes + 16 * ((c & (W::kChunks - 1)) ^ W::swz(p)),
                    v_tile + vr * W::kRowBytes + 16 * ((((p & 3) >> 1) & (W::kChunks - 1)) ^ W::swz(vr)) + 8 * (p & 1)};
}

// A 32-token step for a wave's NQ 16-row groups, in three parts.
//
// Scores: S^T = K Q^T: A = K rows (token lane%16, 8 dims per lane), B = Q; s[tb][qb][j] of a lane is
// the score of token 16*tb + 4*(lane/16) + j and row 16*qb + lane%16, so the eight scores of a
// row group are exactly the k-slots the lane feeds to the P.V contraction: probabilities never
// leave registers.  kb: the lane's K address in the tile (see WideLane16).  read_all(): called once every
// K operand of the tile has been requested, ahead of the last matrix instructions.
struct Nothing { __device__ __forceinline__ void operator()() const {} };
template <typename E, int D, int NQ, typename F = Nothing>
__device__ __forceinline__ void tile_scores(unsigned kb, const u32x4 (&qf)[NQ][D / 32], f32x4 (&s)[2][NQ], F read_all = F()) {
  using W = WideGeom<D>;
  constexpr int KS = D / 32;
  constexpr int KB = KS < 4 ? KS : 4;     // contraction steps whose K operands are requested together
#pragma unroll
  for (int tb = 0; tb < 2; ++tb)
#pragma unroll
    for (int qb = 0; qb < NQ; ++qb) s[tb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k0 = 0; k0 < KS; k0 += KB) {
    u32x4 kf[KB][2];
#pragma unroll
    for (int ks = 0; ks < KB; ++ks)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) kf[ks][tb] = lds_read16((kb ^ (64u * (k0 + ks))) + tb * 16 * W::kRowBytes);
    // (keeps the scheduler from sinking each read next to its use, which would expose the full
    // LDS latency time and again)
    __builtin_amdgcn_sched_barrier(0);
    if (k0 + KB == KS) read_all();
#pragma unroll
    for (int ks = 0; ks < KB; ++ks)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) s[tb][qb] = E::mfma(kf[ks][tb], qf[qb][k0 + ks], s[tb][qb]);
  }
}

// The V^T operands of the dim blocks d0 .. of a tile: two transposed LDS reads of 4 consecutive tokens each.
template <int D> struct VOperands {
  static constexpr int kBatch = D / 16 < 8 ? D / 16 : 8;     // dim blocks requested together
  u32x4 f[kBatch];
  __device__ __forceinline__ void request(unsigned vb, int d0) {
#pragma unroll
    for (int db = 0; db < kBatch; ++db) {
      const u32x2 lo = lds_read_tr8(vb ^ (32u * (d0 + db)));
      const u32x2 hi = lds_read_tr8((vb ^ (32u * (d0 + db))) + 16 * WideGeom<D>::kRowBytes);
      f[db] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
};

// Scores to probabilities, online.  valid < 32 only on a run's last, partial tile.  The check whether a
// row's soft-max reference has to move (see kSlack) needs no exchange between the four lanes that
// share the row: each compares its own eight scores, and only when some lane of the wave finds one
// too large are the maxima exchanged and the accumulators rescaled.  REST: what rounding the probabilities to the
// storage type leaves over goes to `rest`.
template <typename E, int D, int NQ, bool REST = false>
__device__ __forceinline__ void tile_softmax(f32x4 (&s)[2][NQ], int valid, float sc, WaveState<D, NQ>& st, u32x4 (&pf)[NQ], u32x4* rest = nullptr) {
  if (valid < kTileTokens) {  // wave uniform
    asm volatile("" ::: "memory");  // keeps this a branch: as selects it would run on every tile
    const int c = lane_here() >> 4;
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) s[tb][qb][j] = (16 * tb + 4 * c + j >= valid) ? -INFINITY : s[tb][qb][j];
  }
  float mx[NQ];
  bool grow = false;
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb) {
    mx[qb] = max3(s[0][qb][0], s[0][qb][1], s[0][qb][2]);
    mx[qb] = max3(mx[qb], s[0][qb][3], s[1][qb][0]);
    mx[qb] = max3(mx[qb], s[1][qb][1], s[1][qb][2]);
    mx[qb] = fmaxf(mx[qb], s[1][qb][3]);
    grow |= mx[qb] * sc > st.m[qb] + kSlack;   // sc > 0; true on a run's first tile (m = -inf)
  }
  if (__builtin_amdgcn_ballot_w64(grow)) {
#pragma unroll
    for (int qb = 0; qb < NQ; ++qb) {
      const float top = xor32_max(xor16_max(mx[qb])) * sc;   // finite: the tile holds at least one token
      const float m_new = top > st.m[qb] + kSlack ? top : st.m[qb];
      const float alpha = __builtin_amdgcn_exp2f(st.m[qb] - m_new);
      st.l[qb] *= alpha;
#pragma unroll
      for (int db = 0; db < D / 16; ++db) st.o[qb][db] *= alpha;
      st.m[qb] = m_new;
    }
  }
#pragma unroll
  for (int qb = 0; qb < NQ; ++qb) {
    const float neg_m = -st.m[qb];
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j >> 2][qb][j & 3], sc, neg_m));
    st.l[qb] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    pf[qb] = u32x4{E::pack2(x[0], x[1]), E::pack2(x[2], x[3]), E::pack2(x[4], x[5]), E::pack2(x[6], x[7])};
    if constexpr (REST)
#pragma unroll
      for (int j = 0; j < 4; ++j) rest[qb][j] = E::pack2_rest(x[2 * j], x[2 * j + 1], pf[qb][j]);
  }
}

// O^T += V^T P^T; `v` holds the operands of the first dim blocks.  read_all(): as in tile_scores; rest: as in tile_softmax.
template <typename E, int D, int NQ, bool REST = false, typename F = Nothing>
__device__ __forceinline__ void tile_pv(unsigned vb, VOperands<D>& v, const u32x4 (&pf)[NQ], WaveState<D, NQ>& st, F read_all = F(), const u32x4* rest = nullptr) {
  constexpr int DB = D / 16, VB = VOperands<D>::kBatch;
#pragma unroll
  for (int d0 = 0; d0 < DB; d0 += VB) {
    if (d0 > 0) v.request(vb, d0);
    if (d0 + VB == DB) read_all();
#pragma unroll
    for (int db = 0; db < VB; ++db)
#pragma unroll
      for (int qb = 0; qb < NQ; ++qb) st.o[qb][d0 + db] = E::mfma(v.f[db], pf[qb], st.o[qb][d0 + db]);
    if constexpr (REST)
#pragma unroll
      for (int db = 0; db < VB; ++db)
#pragma unroll
        for (int qb = 0; qb < NQ; ++qb) st.o[qb][d0 + db] = E::mfma(v.f[db], rest[qb], st.o[qb][d0 + db]);
  }
}

// Token groups of a pass at most (see wide_block).
template <int D> struct WideGroups { static constexpr int kMost = D <= 128 ? WideGeom<D>::kSub : kWideWaves; };

// What the waves of a block share in one pass over a KV run, and what a wave does in it.
struct WidePass {
  int kvh;
  int row0;            // the wave's first query row
  int groups;          // its 16-row groups (0: it only loads)
  int set, tg, tgroups;  // its row set, its token group, token groups of the pass
};

// A wave's state in LDS for another wave to merge: its accumulators as 16-byte words, then m and l.
// kFloats: per lane.  (16-byte accesses: a quarter of the instructions of 4-byte ones, on a path that every
// vnode takes once, with cold code.)
template <int D, int NG> struct SharedState {
  static constexpr int DB = D / 16;
  static constexpr int kFloats = NG * (4 * DB + 2);
  static __device__ __forceinline__ void put(float* at, const WaveState<D, NG>& st) {
    const int lane = lane_here();
    f32x4* o = reinterpret_cast<f32x4*>(at) + lane;
    float* ml = at + NG * DB * 4 * kWave + lane;
#pragma unroll
    for (int qb = 0; qb < NG; ++qb) {
      ml[2 * qb * kWave] = st.m[qb];
      ml[(2 * qb + 1) * kWave] = st.l[qb];
#pragma unroll
      for (int db = 0; db < DB; ++db) o[(qb * DB + db) * kWave] = st.o[qb][db];
    }
  }
  static __device__ __forceinline__ void merge(const float* at, WaveState<D, NG>& st) {
    const int lane = lane_here();
    const f32x4* o = reinterpret_cast<const f32x4*>(at) + lane;
    const float* ml = at + NG * DB * 4 * kWave + lane;
#pragma unroll
    for (int qb = 0; qb < NG; ++qb) {
      const float m2 = ml[2 * qb * kWave], l2 = ml[(2 * qb + 1) * kWave];
      const float m = fmaxf(st.m[qb], m2);
      const float a1 = scale_from(st.m[qb], m), a2 = scale_from(m2, m);
      st.l[qb] = st.l[qb] * a1 + l2 * a2;
      st.m[qb] = m;
#pragma unroll
      for (int db = 0; db < DB; ++db) st.o[qb][db] = st.o[qb][db] * a1 + o[(qb * DB + db) * kWave] * a2;
    }
  }
};

// Merge of the waves that hold the same rows (the token groups of a row set) into token group 0,
// pairwise through LDS.  Every wave of the block must call this.
template <int D, int NG>
__device__ __forceinline__ void merge_token_groups(float* xchg, WaveState<D, NG>& st, const WidePass& p) {
  constexpr int kArea = WideRows<D>::kGroups * SharedState<D, 1>::kFloats * kWave;   // (waves of other sets may hold fewer groups)
#pragma unroll 1
  for (int half = p.tgroups >> 1; half >= 1; half >>= 1) {
    __syncthreads();
    if (p.tg >= half && p.tg < 2 * half) SharedState<D, NG>::put(xchg + (size_t)(p.set * half + p.tg - half) * kArea, st);
    __syncthreads();
    if (p.tg < half) SharedState<D, NG>::merge(xchg + (size_t)(p.set * half + p.tg) * kArea, st);
  }
}

// The rows of a wave that holds all of its tokens, written through its area `at` of LDS (16 rows of 4 * D bytes), whole rows
// at a time: straight from the accumulators an instruction writes 64 bytes to each of 16 rows, and four waves' 128 rows of
// 512 bytes leave a unit in 1.7 us, in whole rows in 1.3 (.7 where other units don't write; the 400-request tree, whole
// calls, 60.4 -> 59.8 us; at 512-byte K/V rows, where a block is alone on its unit, nothing is gained).
template <int D, int NG>
__device__ __forceinline__ void write_rows(const Stage1Args& a, unsigned at, const VnodeView& vn, const WidePass& p, const WaveState<D, NG>& st) {
  constexpr int kChunks = D / 4;                             // 16-byte pieces of a row
  constexpr int kRows = kWave / kChunks;                     // rows an instruction writes
  static_assert(16 * 16 * kChunks <= WideGeom<D>::kBytes / kWideWaves, "the rows fit a wave's part of a buffer");
  const int lane = lane_here(), r16 = lane & 15, c = lane >> 4;
  const int rows_total = vn.q_len * a.g;
  // piece k of row r lies in place k ^ (r & 7) of the row: 8 lanes that follow each other write one piece of 8 rows, and read 8
  // pieces of one row, in 8 places of different banks (with k ^ 4 * (r & 7) the 400-request tree lost 479 thousand cycles of a
  // launch to bank conflicts, and 128 requests on an 8192-token prefix took 40.9 us, 40.5 so)
  auto place = [&](int r, int k) { return at + (unsigned)(r * (16 * kChunks) + 16 * (k ^ (r & 7))); };
#pragma unroll
  for (int qb = 0; qb < NG; ++qb) {
    if (qb >= p.groups) break;                               // (a wave without rows writes none)
    const int r = min(p.row0 + 16 * qb + r16, rows_total - 1), there = rows_total - (p.row0 + 16 * qb);
    const int ri = a.by_g(r), head = p.kvh * a.g + r - ri * a.g;
    const int64_t row = vn.q_off + ri;
    const float l = st.l[qb], inv = l > 0.f ? 1.f / l : 0.f;
    const uint64_t dst = (uint64_t)(uintptr_t)(a.mid_o + row * a.so0 + (int64_t)head * a.so1);
    wave_lds_fence();
#pragma unroll
    for (int db = 0; db < D / 16; ++db)
      *reinterpret_cast<__attribute__((address_space(3))) f32x4*>((uintptr_t)place(r16, 4 * db + c)) = st.o[qb][db] * inv;
    if (c == 0 && r16 < there) a.mid_lse[row * a.sl0 + head] = l > 0.f ? (__builtin_amdgcn_logf(l) + st.m[qb]) * kLn2 : -INFINITY;
    wave_lds_fence();
    const int k = lane % kChunks, first = lane / kChunks;
#pragma unroll
    for (int i = 0; i < 16; i += kRows) {
      const f32x4 x = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>((uintptr_t)place(i + first, k));
      const unsigned lo = (unsigned)lane_value((int)(unsigned)dst, i + first), hi = (unsigned)lane_value((int)(unsigned)(dst >> 32), i + first);
      if (i + first < there)
        *reinterpret_cast<__attribute__((address_space(1))) f32x4*>((uintptr_t)(((uint64_t)hi << 32) | lo) + 16 * k) = x;
    }
  }
}

// The two token groups of a row set merged, and the merged rows written, in one exchange through LDS at xchg: this wave,
// of token group HALF, hands the other wave of its set the other half of the dims and merges and writes its own half.  Merged
// into one wave that then writes, a vnode of 64 rows spent 2.1 us here (64 requests on a shared prefix, whole calls, 24.9 ->
// 24.35 us; 111 ragged requests of 64-dim heads 12.45 -> 12.25; not at head_dim 256, where there are no registers for it: 17.2
// -> 20.4).  Every wave of the block must call this, one half or the other.
template <int D, int NG, int HALF>
__device__ __forceinline__ void merge_and_write_half(const Stage1Args& a, float* xchg, const VnodeView& vn, const WidePass& p, const WaveState<D, NG>& st) {
  constexpr int HB = D / 32;                                 // dim blocks of a half
  constexpr int kArea = WideRows<D>::kGroups * (4 * HB + 2) * kWave;   // floats (the other set's waves may hold fewer groups)
  static_assert(WideGroups<D>::kMost == 2 && kWideWaves * kArea * 4 <= WideGeom<D>::kLds, "the waves' halves fit the block's LDS");
  const int lane = lane_here(), r16 = lane & 15, c = lane >> 4;
  float* mine = xchg + (size_t)(2 * p.set + HALF) * kArea;
  const float* other = xchg + (size_t)(2 * p.set + 1 - HALF) * kArea;
  __syncthreads();
#pragma unroll
  for (int qb = 0; qb < NG; ++qb) {
    mine[(4 * HB * NG + 2 * qb) * kWave + lane] = st.m[qb];
    mine[(4 * HB * NG + 2 * qb + 1) * kWave + lane] = st.l[qb];
#pragma unroll
    for (int db = 0; db < HB; ++db) reinterpret_cast<f32x4*>(mine)[(qb * HB + db) * kWave + lane] = st.o[qb][(1 - HALF) * HB + db];
  }
  __syncthreads();
  const int rows_total = vn.q_len * a.g;
#pragma unroll
  for (int qb = 0; qb < NG; ++qb) {
    const float m2 = other[(4 * HB * NG + 2 * qb) * kWave + lane], l2 = other[(4 * HB * NG + 2 * qb + 1) * kWave + lane];
    const float m = fmaxf(st.m[qb], m2);
    const float a1 = scale_from(st.m[qb], m), a2 = scale_from(m2, m);
    const float l = st.l[qb] * a1 + l2 * a2;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    f32x4 o[HB];
#pragma unroll
    for (int db = 0; db < HB; ++db)
      o[db] = (st.o[qb][HALF * HB + db] * a1 + reinterpret_cast<const f32x4*>(other)[(qb * HB + db) * kWave + lane] * a2) * inv;
    const int r = p.row0 + 16 * qb + r16;
    if (qb >= p.groups || r >= rows_total) continue;
    const int ri = a.by_g(r), head = p.kvh * a.g + r - ri * a.g;
    const int64_t row = vn.q_off + ri;
    float* dst = a.mid_o + row * a.so0 + (int64_t)head * a.so1 + 4 * c + 16 * HALF * HB;
#pragma unroll
    for (int db = 0; db < HB; ++db) *reinterpret_cast<f32x4*>(dst + 16 * db) = o[db];
    if (HALF == 0 && c == 0) a.mid_lse[row * a.sl0 + head] = l > 0.f ? (__builtin_amdgcn_logf(l) + m) * kLn2 : -INFINITY;
  }
}

// What a wave does to stream a KV run into the block's ring: it requests slot indices (into a ring of its own, so
// that nothing the compiler tracks is in flight in the loop and no register holds an index longer than one super
// tile), reads back those of the rows it loads, and requests the rows.  Tokens past the run repeat its last
// token: the scores of such rows are masked and their V rows are finite.
template <int D, bool GATHERED> struct RowStream {
  using W = WideGeom<D>;
  const char *kbase, *vbase;
  unsigned k_stride, v_stride;   // bytes, < 2^32 (checked by the host)
  const int32_t* entries;
  int64_t kv_base;
  int kv_len, nsuper;
  unsigned ring, idx_ring;       // idx_ring: four super tiles of indices
  int wave, lane;
  unsigned srow[W::kSlots];

  // (loader role of a lane: 16-byte slot `pos` of row `row(u)` in each 1 KB group it fills)
  __device__ __forceinline__ int group(int u) const { return W::kGroups >= kWideWaves ? u * kWideWaves + wave : wave % W::kGroups; }
  __device__ __forceinline__ int row(int u) const { return group(u) * W::kGroupRows + lane / W::kChunks; }

  __device__ __forceinline__ RowStream(const Stage1Args& a, char* smem, int kvh) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = lane_here();
    kbase = a.k + 2 * ((int64_t)kvh * a.sk1);
    vbase = a.v + 2 * ((int64_t)kvh * a.sv1);
    k_stride = (unsigned)(2 * a.sk0);
    v_stride = (unsigned)(2 * a.sv0);
    ring = lds_offset(smem);
    idx_ring = ring + W::kRing + wave * (4 * 4 * W::kTokens);
  }
  __device__ __forceinline__ void open(const Stage1Args& a, const VnodeView& vn) {
    kv_len = vn.kv_len;
    kv_base = vn.kv_base;
    nsuper = (kv_len + W::kTokens - 1) / W::kTokens;
    entries = GATHERED ? nullptr : a.kv_entries + vn.kv_base;
  }
  __device__ __forceinline__ void issue_indices(int j) const {
    if constexpr (!GATHERED) {
      if (j < nsuper) load_direct4(entries, 4u * (unsigned)min(j * W::kTokens + lane, kv_len - 1), idx_ring + (j & 3) * (4 * W::kTokens));
    }
  }
  __device__ __forceinline__ void read_rows(int j) {
    if (j >= nsuper) return;
#pragma unroll
    for (int u = 0; u < W::kSlots; ++u) {
      if constexpr (GATHERED) srow[u] = (unsigned)(kv_base + min(j * W::kTokens + row(u), kv_len - 1));
      else srow[u] = lds_read4(idx_ring + (j & 3) * (4 * W::kTokens) + 4 * row(u));
    }
  }
  // rows of super tile j -> ring buffer j % 2
  __device__ __forceinline__ void issue_rows(int j) const {
    if (j >= nsuper) return;
    const unsigned buf = ring + (unsigned)(j & 1) * W::kBytes;
    const int pos = lane % W::kChunks;
#pragma unroll
    for (int u = 0; u < W::kUnits; ++u) {
      // unit u of this wave: K groups first, then V groups
      const bool is_v = W::kGroups >= kWideWaves ? u >= W::kSlots : wave >= W::kGroups;
      const int sl = u % W::kSlots;
      const char* src = (is_v ? vbase : kbase) + (uint64_t)srow[sl] * (is_v ? v_stride : k_stride);
      load_direct16(src + 16 * (pos ^ W::swz(row(sl))), buf + (is_v ? W::kBytesK : 0) + group(sl) * 1024);
    }
  }
};

// What a wave reads of a program's record, all of it in one memory round trip: the slots of the rows it loads
// first (straight into RowStream::srow), and the requests of the scratch rows, two per lane.
struct RecordRequests {
  int even, odd;
  __device__ __forceinline__ RecordRequests() : even(0), odd(0) {}
  __device__ __forceinline__ void load(const int32_t* record) {
    const int lane = lane_here();
    even = record[kProgRecRequests + 2 * lane];
    odd = record[kProgRecRequests + 2 * lane + 1];
  }
  // (i differs from lane to lane; every lane of the wave takes part)
  __device__ __forceinline__ int of(int i) const {
    const int e = lane_value(even, i >> 1), o = lane_value(odd, i >> 1);
    return i & 1 ? o : e;
  }
};

// One wave's pass over a vnode's KV run for NG row groups (p.groups <= NG of them exist).  The block
// streams the run through a ring of two 64-token LDS buffers with direct global->LDS loads, one
// super tile ahead of the one being consumed; the slot indices travel the same way, two super tiles further
// ahead.  The caller has opened the run and requested the indices of its first super tiles, and its first rows
// too if `started`; `requests`: those of the vnode's scratch rows, if `started`.
template <typename E, int D, int NG, bool GATHERED>
__device__ __forceinline__ void wide_pass(const Stage1Args& a, char* smem, const VnodeView& vn, const WidePass& p, RowStream<D, GATHERED>& rows,
                                          bool started, const RecordRequests& requests) {
  using W = WideGeom<D>;
  // Rows past the vnode (and those of a wave that only loads) compute its last row again: nothing of theirs
  // is written, and no lane waits on a branch.
  int req[NG], head[NG];
#pragma unroll
  for (int qb = 0; qb < NG; ++qb) {
    const int r = min(p.row0 + 16 * qb + (rows.lane & 15), vn.q_len * a.g - 1);
    req[qb] = a.by_g(r);
    head[qb] = p.kvh * a.g + r - req[qb] * a.g;
  }
  if (started) {
#pragma unroll
    for (int qb = 0; qb < NG; ++qb) req[qb] = requests.of(req[qb]);
  } else {
    if constexpr (GATHERED) {
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) req[qb] = vn.q_off / a.nsplit;
    } else {
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) req[qb] = a.q_entries[vn.q_off + req[qb]];
      // (awaited here: a wait for them where the two branches meet would be a wait for all direct loads in both)
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) asm volatile("" : "+v"(req[qb]));
    }
    if (rows.nsuper > 0) {
      wait_direct_loads<0>();
      rows.read_rows(0);
      rows.issue_rows(0);
    }
  }
  const char* src[NG];
#pragma unroll
  for (int qb = 0; qb < NG; ++qb) src[qb] = a.q + 2 * ((int64_t)req[qb] * a.sq0 + (int64_t)head[qb] * a.sq1 + 8 * (rows.lane >> 4));
  // (the fragments after the rows: ahead of them they would be a round trip of their own)
  u32x4 qf[NG][D / 32];
#pragma unroll
  for (int qb = 0; qb < NG; ++qb)
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) qf[qb][ks] = *reinterpret_cast<const u32x4*>(src[qb] + 64 * ks);
  // nothing the compiler itself tracks (the Q fragments) may still be in flight in the loop:
  // a wait for it there would also wait for every direct load
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  wait_direct_loads<0>();              // (no access to LDS moves above it either)
  // (and the compiler must see the fragments as complete, or it keeps a wait for them in the loop)
#pragma unroll
  for (int qb = 0; qb < NG; ++qb)
#pragma unroll
    for (int ks = 0; ks < D / 32; ++ks) asm volatile("" : "+v"(qf[qb][ks]));
  WaveState<D, NG> st;
  reset_state<D, NG>(st);
  const WideLane16 la = init_lane16<D>(rows.ring, rows.ring + W::kBytesK);
  rows.read_rows(1);

  for (int super = 0; super < rows.nsuper; ++super) {
    wait_direct_loads<0>();
    __syncthreads();   // publishes super tile `super` to the block; the buffer consumed before it is free
    rows.issue_rows(super + 1);
    rows.issue_indices(super + 3);
    rows.read_rows(super + 2);
#pragma unroll 1
    for (int sub = 0; sub < W::kSub; ++sub) {
      const int tile = super * W::kSub + sub;
      const int valid = vn.kv_len - tile * kTileTokens;
      if ((tile & (p.tgroups - 1)) != p.tg || valid <= 0 || p.groups == 0) continue;
      const unsigned off = (super & 1) * W::kBytes + sub * W::kTileBytes;
      f32x4 sc[2][NG];
      u32x4 pf[NG];
      VOperands<D> v;
      tile_scores<E, D, NG>(la.k + off, qf, sc);
      // the V operands do not depend on the probabilities: requested now, they arrive under the soft-max
      // arithmetic (and take the registers the K operands just left)
      v.request(la.v + off, 0);
      tile_softmax<E, D, NG>(sc, valid, a.scale_log2, st, pf);
      tile_pv<E, D, NG>(la.v + off, v, pf, st);
    }
  }
  finish_state<D, NG>(st);
  if constexpr (D <= 128) {
    // (the buffer that the run's last super tile does not lie in: read out before the barrier of that super tile)
    if (p.tgroups == 1) write_rows<D, NG>(a, rows.ring + (unsigned)(rows.nsuper & 1) * W::kBytes + (unsigned)rows.wave * (W::kBytes / kWideWaves), vn, p, st);
    else if (p.tg == 0) merge_and_write_half<D, NG, 0>(a, reinterpret_cast<float*>(smem), vn, p, st);
    else merge_and_write_half<D, NG, 1>(a, reinterpret_cast<float*>(smem), vn, p, st);
  } else {
    if (p.tgroups > 1) merge_token_groups<D, NG>(reinterpret_cast<float*>(smem), st, p);
    if (p.tg == 0) write_partials<D, NG>(a, vn, p.kvh, p.row0, st, p.groups);
  }
  __syncthreads();  // the ring is reused by the next pass
}

// One block (kWideWaves waves) serves the row pieces chunk, chunk + chunks, ... (WideRows<D>::kBlock
// query rows each) of a vnode for one kv head.  Per pass over the run the waves form row sets x
// token groups: a wave consumes the 32-token tiles t with t % tgroups == tg for its row set's 16-row
// groups, and the states of the token groups of a row set are merged at the end.  `listed`: `rows` holds the slots
// of the run's first super tile and `requests` the vnode's requests (a program's record).
template <typename E, int D, bool GATHERED>
__device__ __forceinline__ void wide_block(const Stage1Args& a, char* smem, const VnodeView& vn, int kvh, int chunk, int chunks,
                                           RowStream<D, GATHERED>& rows, bool listed, const RecordRequests& requests) {
  constexpr int NQ = WideRows<D>::kGroups, kRows = WideRows<D>::kBlock;
  const int rows_total = vn.q_len * a.g;
  for (int piece = chunk; piece * kRows < rows_total; piece += chunks) {
    // (one copy of this for every number of row groups, ahead of what differs between them: the first rows are on
    // their way before the code that consumes them is fetched)
    const bool started = listed && piece == 0;      // (the record covers the vnode's first kRows rows)
    rows.open(a, vn);
    if (rows.nsuper > 0) {
      if (started) rows.issue_rows(0);
      else rows.issue_indices(0);
      rows.issue_indices(1);
      rows.issue_indices(2);
    }
    const int row0 = piece * kRows;
    const int groups = (min(row0 + kRows, rows_total) - row0 + 15) >> 4;
    // As many token groups as leave every wave at most NQ row groups: fewer waves then read the same K/V
    // operands from LDS.  No more than a super tile has tiles: between two barriers a wave of a third group
    // would have none (one vnode of 48 rows and 1024 tokens per block, a step of 32 tokens: four groups .52 us, two
    // .43; of 32 rows .43 and .37; a 111-request tree of 16/1 heads with four such vnodes 32.9 -> 27.9 us).  At 512-byte
    // rows, where a block has its unit to itself and merging a row group moves 16 KB, as leave every wave one (64
    // requests of 16/1 heads of 256: 23.0 -> 20.0 us; a step takes the same with two groups or four).
    // One token group from 33 rows on spares most passes the merge, but each group's first maximum has the probability
    // 1, which the storage type holds exactly, and one group so rounds more of P than two: it costs precision (shared
    // prefixes of fp16 against 64 bits, relative RMS over ten inputs 2.88e-4 with two groups, 2.90e-4 with one).
    constexpr int kGroupsWanted = D <= 128 ? NQ * kWideWaves : kWideWaves;
    int log_tgroups = 0;
    while ((1 << log_tgroups) < WideGroups<D>::kMost && groups * (2 << log_tgroups) <= kGroupsWanted) ++log_tgroups;
    static_assert(kWideWaves == 4, "row sets are 4 >> log_tgroups");
    const int log_sets = 2 - log_tgroups;
    WidePass p;
    p.kvh = kvh;
    p.set = rows.wave >> log_tgroups;
    p.tgroups = 1 << log_tgroups;
    p.tg = rows.wave & (p.tgroups - 1);
    const int share = groups >> log_sets, extra = groups - (share << log_sets);     // row groups per set: share, one more in the first `extra`
    p.groups = share + (p.set < extra ? 1 : 0);
    p.row0 = row0 + 16 * (p.set * share + min(p.set, extra));
    // (wave uniform; every path has the same block barriers.  One request's rows, at most 64, leave a wave two groups.)
    if (NQ >= 3 && !GATHERED && p.groups == 3) wide_pass<E, D, NQ, GATHERED>(a, smem, vn, p, rows, started, requests);
    else if (p.groups == 2) wide_pass<E, D, 2, GATHERED>(a, smem, vn, p, rows, started, requests);
    else wide_pass<E, D, 1, GATHERED>(a, smem, vn, p, rows, started, requests);
  }
}

// ---------------------------------------------------------------------------------------
// Narrow vnodes: one wave per (vnode, kv head) streams the run through a wave-private LDS tile of 32
// tokens with direct global->LDS loads, in the same unpadded XOR layout as the wide kernel, and serves up
// to NarrowGeom<D>::kGroups 16-row groups on it per pass.  K and V have one tile each: the K rows of
// the next tile are requested as soon as the scores of the current one are out of LDS, its V rows
// as soon as the current P.V is, so eight waves of a compute unit keep up to 128 KB of rows in flight
// and no barrier holds one wave's loads back for another's arithmetic.  A leaf vnode of a few dozen
// tokens costs little more than its two memory round trips (record, rows).  Slot indices travel the
// same way, two tiles ahead.
//
// What bounds a leaf is that chain of round trips, so nothing the compiler tracks may be awaited between the first
// rows' requests and the query fragments': the request ids and the record were, and a vnode's queries were asked for
// when its rows had landed (1423 leaves of 135 tokens and 64-dim heads: 112.4 us so, 99.9 now; 380 of 86 tokens
// 22.9 and 21.3; 6 waves' worth of leaves 9.7 and 9.2).
// ---------------------------------------------------------------------------------------
template <int D> struct NarrowGeom {
  static constexpr int kRowBytes = 2 * D;
  static constexpr int kChunks = D / 8;
  static constexpr int kBytesK = kTileTokens * kRowBytes;
  static constexpr int kBytes = 2 * kBytesK;
  static constexpr int kGroupRows = kWave / kChunks;            // rows per 1 KB load
  static constexpr int kLoads = kTileTokens / kGroupRows;       // loads per matrix and tile
  static constexpr int kIdxSlot = 4 * kWave;                    // bytes of one tile's indices (32, and the 32 after them)
  static constexpr int kLds = kBytes + 4 * kIdxSlot;            // per wave; a multiple of the row size
  static constexpr int kGroups = 2;                             // 16-row groups per pass (three spill beside the wide path's code)
  static __device__ __forceinline__ int swz(int row) { return chunk_swizzle<D>(row); }
};

// Layout of a narrow vnode's record in Stage1Args::narrow_table (ints): kv_off, kv_len, q_off,
// q_len; then the requests of the vnode's first kNarrowRecRequests scratch rows; then the pool slots
// of its first kTileTokens tokens (the last one repeated past the end of a shorter run).
constexpr int kNarrowRecord = 64;
constexpr int kNarrowRecRequests = 16;
constexpr int kNarrowRecSlots = 4 + kNarrowRecRequests;

// What a wave does to stream its tiles of a narrow vnode's run into its own LDS area.  It asks for slot indices (into a
// ring in LDS), reads back those of the rows it loads, and asks for the rows.  A wave that walks every tile asks for
// two tiles' indices at a time, one that shares its run for one tile's.  Tokens past the run repeat its last token
// (their scores are masked, their V rows are finite).
template <int D, bool GATHERED> struct NarrowStream {
  using N = NarrowGeom<D>;
  const char *kbase, *vbase;
  unsigned k_stride, v_stride;   // bytes, < 2^32 (checked by the host)
  unsigned tile_addr, idx_ring;  // the wave's K tile (its V tile follows), its index ring
  const int32_t* entries;
  int64_t kv_base;
  int kv_len, ntiles, tile0, stride;   // the wave serves the tiles tile0, tile0 + stride, ...
  int lane;
  unsigned srow[N::kLoads];

  __device__ __forceinline__ NarrowStream(const Stage1Args& a, char* smem, unsigned lds0, int kvh, int w, int share) {
    kbase = a.k + 2 * ((int64_t)kvh * a.sk1);
    vbase = a.v + 2 * ((int64_t)kvh * a.sv1);
    k_stride = (unsigned)(2 * a.sk0);
    v_stride = (unsigned)(2 * a.sv0);
    tile_addr = lds_offset(smem) + lds0;
    tile0 = w;
    stride = share;
  }
  // (lane and tile_addr made opaque: the addresses made from them stay in the pass, or the compiler computes some
  // 100 of them ahead of the loop over passes, which nearly always makes one)
  __device__ __forceinline__ void open(const Stage1Args& a, const VnodeView& vn) {
    lane = lane_here();
    asm volatile("" : "+s"(tile_addr));
    idx_ring = tile_addr + N::kBytes;
    kv_len = vn.kv_len;
    kv_base = vn.kv_base;
    ntiles = (kv_len + kTileTokens - 1) / kTileTokens;
    entries = GATHERED ? nullptr : a.kv_entries + vn.kv_base;
  }
  __device__ __forceinline__ bool pairs() const { return stride == 1; }   // wave uniform
  // (loader role of a lane: 16-byte slot `pos` of row `row(g)` in each 1 KB group)
  __device__ __forceinline__ int row(int g) const { return g * N::kGroupRows + lane / N::kChunks; }
  // the slot indices of 64 tokens from the wave's i-th tile on
  __device__ __forceinline__ void issue_indices(int i, int tile) const {
    if constexpr (!GATHERED)
      load_direct4(entries, 4u * (unsigned)min(tile * kTileTokens + lane, kv_len - 1), idx_ring + ((pairs() ? i >> 1 : i) & 3) * N::kIdxSlot);
  }
  // the cache rows this lane loads of the wave's i-th tile
  __device__ __forceinline__ void read_rows(int i, int tile) {
    const unsigned at = idx_ring + (pairs() ? (i & 7) * (N::kIdxSlot / 2) : (i & 3) * N::kIdxSlot);
#pragma unroll
    for (int g = 0; g < N::kLoads; ++g) {
      if constexpr (GATHERED) srow[g] = (unsigned)(kv_base + min(tile * kTileTokens + row(g), kv_len - 1));
      else srow[g] = lds_read4(at + 4 * row(g));
    }
  }
  // the same of the run's first tile, from the vnode's record (a lane's int of it)
  __device__ __forceinline__ void rows_of_record(int rec) {
#pragma unroll
    for (int g = 0; g < N::kLoads; ++g) srow[g] = (unsigned)lane_value(rec, kNarrowRecSlots + row(g));
  }
  // those rows of K (or V) -> the wave's K (V) tile
  __device__ __forceinline__ void issue(bool is_v) const {
    const int pos = lane % N::kChunks;
#pragma unroll
    for (int g = 0; g < N::kLoads; ++g) {
      const char* src = (is_v ? vbase : kbase) + (uint64_t)srow[g] * (is_v ? v_stride : k_stride) + 16 * (pos ^ N::swz(row(g)));
      load_direct16(src, tile_addr + (is_v ? N::kBytesK : 0) + g * 1024);
    }
  }
};

// One wave's share of a narrow vnode for the NG 16-row groups from row0.  The caller has opened the run and asked for
// the wave's first indices, and for its first rows too if `started`.  `rec` is the lane's int of the vnode's record when
// `inlined` (else unused).
//
// REST: what rounding the probabilities leaves over is contracted as well.  Such a remainder is 0, or below it, where its
// probability is not, and an infinite V value then makes NaN of the infinity that the sum is.  So a caller that finds NaN takes the
// sums again without REST (in code that is never fetched otherwise).
template <typename E, int D, int NG, bool GATHERED, bool REST>
__device__ __forceinline__ void narrow_attend(const Stage1Args& a, const VnodeView& vn, NarrowStream<D, GATHERED>& rows, bool started,
                                              int kvh, int row0, WaveState<D, NG>& st, int rec, bool inlined) {
  using N = NarrowGeom<D>;
  constexpr int KS = D / 32;
  const int p = rows.lane & 15, c = rows.lane >> 4;
  const int ntiles = rows.ntiles, tile0 = rows.tile0, tstride = rows.stride;
  const bool pairs = rows.pairs();

  if (tile0 < ntiles) {
    // Fragment ks of a lane: row row0 + 16*qb + p, dims 32*ks + 8*c .. +7.  (Rows past the vnode compute its last
    // row again: nothing of theirs is written, and no lane waits on a branch.)
    int req[NG], head[NG];
#pragma unroll
    for (int qb = 0; qb < NG; ++qb) {
      const int r = min(row0 + 16 * qb + p, vn.q_len * a.g - 1);
      req[qb] = a.by_g(r);
      head[qb] = kvh * a.g + r - req[qb] * a.g;
    }
    if constexpr (GATHERED) {
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) req[qb] = vn.q_off / a.nsplit;
    } else if (inlined && vn.q_len <= kNarrowRecRequests) {   // wave uniform: they are in the record
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) req[qb] = lane_value(rec, 4 + req[qb]);
    } else {
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) req[qb] = a.q_entries[vn.q_off + req[qb]];
      // (awaited here: a wait for them where the two branches meet would be a wait for all direct loads in both)
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
#pragma unroll
      for (int qb = 0; qb < NG; ++qb) asm volatile("" : "+v"(req[qb]));
    }
    const char* src[NG];
#pragma unroll
    for (int qb = 0; qb < NG; ++qb) src[qb] = a.q + 2 * ((int64_t)req[qb] * a.sq0 + (int64_t)head[qb] * a.sq1 + 8 * c);
    if (!started) {
      wait_direct_loads<0>();
      rows.read_rows(0, tile0);
      rows.issue(false);
      rows.issue(true);
    }
    // (the fragments after the rows: ahead of them they would be a round trip of their own)
    u32x4 qf[NG][KS];
#pragma unroll
    for (int qb = 0; qb < NG; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[qb][ks] = *reinterpret_cast<const u32x4*>(src[qb] + 64 * ks);
    reset_state<D, NG>(st);
    const WideLane16 la = init_lane16<D>(rows.tile_addr, rows.tile_addr + N::kBytesK);
    // nothing the compiler itself tracks may still be in flight below: a wait for it would
    // also wait for every direct load
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    wait_direct_loads<0>();              // (no access to LDS moves above it either)
    // (and the compiler must see the fragments as complete, or it keeps a wait for them in the loop)
#pragma unroll
    for (int qb = 0; qb < NG; ++qb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[qb][ks]));
    // The next rows are asked for as soon as a tile's operands are in registers, ahead of the arithmetic on
    // them; at 512-byte rows there are no registers for that, and they follow it.
    constexpr bool kEarly = D <= 128;
    for (int i = 0, tile = tile0; tile < ntiles; ++i, tile += tstride) {
      const int next = tile + tstride;
      const bool more = next < ntiles;
      f32x4 sc[2][NG];
      u32x4 pf[NG];
      VOperands<D> v;
      const bool indices = !GATHERED && more && (!pairs || (i & 1) == 0);   // wave uniform
      wait_direct_loads<N::kLoads>();  // K (and the next tile's indices) landed; V may still be in flight
      if (kEarly && more) rows.read_rows(i + 1, next);
      auto next_k = [&] {
        if (!more) return;
        if constexpr (!kEarly) rows.read_rows(i + 1, next);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the K tile has been read
        rows.issue(false);
        if (indices) rows.issue_indices(i + 2, next + tstride);
      };
      auto next_v = [&] {
        if (!more) return;
        if constexpr (!kEarly) rows.read_rows(i + 1, next);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the V tile has been read
        rows.issue(true);
      };
      if constexpr (kEarly) {
        tile_scores<E, D, NG>(la.k, qf, sc, next_k);
      } else {
        tile_scores<E, D, NG>(la.k, qf, sc);
        next_k();
      }
      u32x4 rest[NG];
      tile_softmax<E, D, NG, REST>(sc, vn.kv_len - tile * kTileTokens, a.scale_log2, st, pf, rest);
      // V landed; the next K and indices may be in flight
      if (indices) wait_direct_loads<N::kLoads + 1>();
      else if (more) wait_direct_loads<N::kLoads>();
      else wait_direct_loads<0>();
      v.request(la.v, 0);
      if constexpr (kEarly) {
        tile_pv<E, D, NG, REST>(la.v, v, pf, st, next_v, rest);
      } else {
        tile_pv<E, D, NG, REST>(la.v, v, pf, st, Nothing(), rest);
        next_v();
      }
    }
  } else {
    reset_state<D, NG>(st);
  }
  finish_state<D, NG>(st);
}

// Whether there is NaN in what the wave holds (a maximum of three numbers is an instruction, and NaN where one of them is).
template <int D, int NG> __device__ __forceinline__ bool holds_nan(const WaveState<D, NG>& st) {
  f32x4 most = st.o[0][0];
#pragma unroll
  for (int i = 1; i < NG * (D / 16); ++i) most = __builtin_elementwise_maximum(most, st.o[i / (D / 16)][i % (D / 16)]);
  const float all = __builtin_elementwise_maximum(__builtin_elementwise_maximum(most[0], most[1]), __builtin_elementwise_maximum(most[2], most[3]));
  return __builtin_amdgcn_ballot_w64(!(all == all)) != 0;
}
template <typename E, int D, int NG, bool GATHERED>
__device__ __forceinline__ void walk_again(const Stage1Args& a, const VnodeView& vn, NarrowStream<D, GATHERED>& rows, int kvh, int row0,
                                           WaveState<D, NG>& st, int rec, bool inlined) {
  wave_lds_fence();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): what the wave has written to its area lies there before rows land on it
  rows.issue_indices(0, rows.tile0);
  if (!rows.pairs()) rows.issue_indices(1, rows.tile0 + rows.stride);
  narrow_attend<E, D, NG, GATHERED, false>(a, vn, rows, false, kvh, row0, st, rec, inlined);
}

// Merge of the `share` waves of one narrow vnode (same rows, interleaved tiles) into the first of
// them, pairwise through LDS at xchg.  Every wave of the block calls this (block barriers).
template <int D, int NG>
__device__ __forceinline__ void merge_shares(float* xchg, WaveState<D, NG>& st, int w, int share) {
  constexpr int kArea = SharedState<D, NG>::kFloats * kWave;
  static_assert(2 * kArea * 4 <= 4 * NarrowGeom<D>::kLds && kArea * 4 <= 2 * NarrowGeom<D>::kLds,
                "half of the waves' states fit the LDS areas of all of them");
#pragma unroll 1
  for (int half = share >> 1; half >= 1; half >>= 1) {
    __syncthreads();
    if (w >= half && w < 2 * half) SharedState<D, NG>::put(xchg + (size_t)(w - half) * kArea, st);
    __syncthreads();
    if (w < half) SharedState<D, NG>::merge(xchg + (size_t)w * kArea, st);
  }
}

// The merged rows of a narrow vnode from the states of the SHARE waves that served it, in LDS at xchg: this wave, the
// w-th, merges and writes its part of the dims of every row.  `more` is given the rows
// too: request(ri), called by every lane of the wave, names the vnode's ri-th request; write(req, head, dim, x) has in x the
// dims dim .. dim + 3 of that request's row; sum_again(), where kSumsAgain, is given what a lane merged of a dim block that holds NaN.
struct WriteNoMore {
  static constexpr bool kSumsAgain = false;
  __device__ __forceinline__ int request(int) const { return 0; }
  __device__ __forceinline__ void write(int, int, int, const f32x4&) const {}
};
template <int D, int NG, int SHARE, typename F = WriteNoMore>
__device__ __forceinline__ void write_merged_shares(const Stage1Args& a, const float* xchg, const VnodeView& vn, int kvh, int row0, int w, const F& more = F()) {
  constexpr int DB = D / 16, kML = NG * DB * 4 * kWave;
  constexpr int kStep = NarrowGeom<D>::kLds / 4;           // floats from one wave's area to the next one's
  constexpr int kParts = DB >= SHARE ? DB / SHARE : 1;     // dim blocks of a wave
  if (DB < SHARE && w >= DB) return;
  const int lane = lane_here(), p = lane & 15, c = lane >> 4;
#pragma unroll 1
  for (int qb = 0; qb < NG; ++qb) {
    const float* ml = xchg + kML + 2 * qb * kWave + lane;
    const f32x4* o = reinterpret_cast<const f32x4*>(xchg) + (qb * DB + w * kParts) * kWave + lane;
    float m_of[SHARE], l_of[SHARE];
    f32x4 o_of[SHARE][kParts];
#pragma unroll
    for (int i = 0; i < SHARE; ++i) {
      m_of[i] = ml[i * kStep];
      l_of[i] = ml[i * kStep + kWave];
#pragma unroll
      for (int db = 0; db < kParts; ++db) o_of[i][db] = o[i * (kStep / 4) + db * kWave];
    }
    float m = m_of[0], l = 0.f;
#pragma unroll
    for (int i = 1; i < SHARE; ++i) m = fmaxf(m, m_of[i]);
    f32x4 sum[kParts];
#pragma unroll
    for (int db = 0; db < kParts; ++db) sum[db] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SHARE; ++i) {
      const float weight = scale_from(m_of[i], m);
      l += l_of[i] * weight;
#pragma unroll
      for (int db = 0; db < kParts; ++db) sum[db] += o_of[i][db] * weight;
    }
    const int r = min(row0 + 16 * qb + p, vn.q_len * a.g - 1), ri = a.by_g(r), head = kvh * a.g + r - ri * a.g;
    const int req = more.request(ri);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    auto write = [&] {
      if (row0 + 16 * qb + p > r) return;
      const int64_t row = vn.q_off + ri;
      float* dst = a.mid_o + row * a.so0 + (int64_t)head * a.so1 + 4 * c + 16 * w * kParts;
#pragma unroll
      for (int db = 0; db < kParts; ++db) {
        *reinterpret_cast<f32x4*>(dst + 16 * db) = sum[db] * inv;
        more.write(req, head, 4 * c + 16 * (w * kParts + db), sum[db] * inv);
      }
      if (w == 0 && c == 0) a.mid_lse[row * a.sl0 + head] = l > 0.f ? (__builtin_amdgcn_logf(l) + m) * kLn2 : -INFINITY;
    };
    write();
    if constexpr (F::kSumsAgain) {
      f32x4 all = sum[0];
#pragma unroll
      for (int db = 1; db < kParts; ++db) all += sum[db];
      const float one = (all[0] + all[1]) + (all[2] + all[3]);
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(one == one)) != 0, 0)) {
#pragma unroll
        for (int db = 0; db < kParts; ++db) more.sum_again(kvh, req, head, 16 * (w * kParts + db), m, sum[db]);
        write();
      }
    }
  }
}
// Merge of the states of the `share` waves (2 or 4) of one narrow vnode through LDS at xchg, and the write of the merged
// rows, in one exchange in which every wave merges its part: pairwise, into one wave that then writes them, a launch of
// few vnodes spends 1.4 us here, in code it fetches cold (4 requests of a short prompt 8.45 us, 8.0 so; 30 of 16/1 heads
// 9.35 and 8.85; serving 1.2 % shorter).  Every wave of the block calls this (a block barrier); `rows`: whether the vnode
// has rows in this pass.
template <int D, int NG>
__device__ __forceinline__ void merge_and_write_shares(const Stage1Args& a, float* xchg, const VnodeView& vn, int kvh, int row0, bool rows,
                                                       const WaveState<D, NG>& st, int w, int share) {
  static_assert(SharedState<D, NG>::kFloats * kWave * 4 <= NarrowGeom<D>::kLds, "a wave's state fits its LDS area");
  asm volatile("" : "+s"(w), "+s"(share), "+s"(kvh));      // (what is made from them stays here)
  if (rows) SharedState<D, NG>::put(xchg + w * (NarrowGeom<D>::kLds / 4), st);
  __syncthreads();
  if (!rows) return;
  if (share == 2) write_merged_shares<D, NG, 2>(a, xchg, vn, kvh, row0, w);
  else write_merged_shares<D, NG, 4>(a, xchg, vn, kvh, row0, w);
}

// What one wave does for a narrow vnode in one pass (NG row groups from row0; none if row0 is past
// its rows, and then the wave only keeps the block's barriers company).
struct NarrowPass {
  int kvh, row0, w, share, rec;
  bool inlined, started;
  unsigned xchg;      // byte offset of the areas of the waves that share the vnode in the block's LDS segment
};
template <typename E, int D, int NG, bool GATHERED, bool REST>
__device__ __forceinline__ void narrow_pass(const Stage1Args& a, char* smem, const VnodeView& vn, NarrowStream<D, GATHERED>& stream, const NarrowPass& p) {
  WaveState<D, NG> st;
  const bool rows = p.row0 < vn.q_len * a.g;
  if (rows) {
    narrow_attend<E, D, NG, GATHERED, REST>(a, vn, stream, p.started, p.kvh, p.row0, st, p.rec, p.inlined);
    if constexpr (REST)
      if (__builtin_expect(holds_nan<D, NG>(st), 0)) walk_again<E, D, NG, GATHERED>(a, vn, stream, p.kvh, p.row0, st, p.rec, p.inlined);
  } else {
    reset_state<D, NG>(st);
  }
  float* xchg = reinterpret_cast<float*>(smem + p.xchg);
  // (rows of less than 256 bytes keep the pairwise merge: with the other one the kernel for narrow vnodes alone takes 131
  // registers instead of 126, three waves per SIMD instead of four, and 269 requests of 64/8 heads of 64 83.1 us instead
  // of 81.9)
  if constexpr (D >= 128) {
    if (p.share > 1) {
      merge_and_write_shares<D, NG>(a, xchg, vn, p.kvh, p.row0, rows, st, p.w, p.share);
      return;
    }
  }
  if (p.share > 1) merge_shares<D, NG>(xchg, st, p.w, p.share);
  if (rows && p.w == 0) write_partials<D, NG>(a, vn, p.kvh, p.row0, st);
}

// A narrow vnode served by `share` consecutive waves of a block (share = 1, 2 or 4, the same
// for the whole launch; the host picks more than one when there are fewer vnodes than wave
// slots): wave w of the vnode takes the tiles w, w + share, ..., and the shares are merged
// through LDS.  `slot` is the wave's index in the block; a wave without a vnode (exists ==
// false) only keeps the block's barriers company.  More rows than a pass holds take several passes.
// ALONE: the block serves no other vnode.  `index`: the vnode's in the narrow range; `records`: Stage1Args::narrow_table.
template <typename E, int D, bool GATHERED, bool ALONE, bool REST = false>
__device__ __forceinline__ void narrow_item(const Stage1Args& a, const int32_t* records, char* smem, int slot, int share, bool exists,
                                            int index, int kvh) {
  using N = NarrowGeom<D>;
  static_assert(N::kGroups == 2, "passes of two row groups, then of one");
  VnodeView vn{0, 0, 0, 0};
  NarrowPass p;
  p.kvh = kvh;
  p.share = share;
  p.w = slot & (share - 1);
  p.xchg = (unsigned)(slot - p.w) * N::kLds;
  p.rec = 0;
  p.inlined = !GATHERED && records != nullptr;   // launch uniform
  if (p.inlined && exists) p.rec = records[(int64_t)index * kNarrowRecord + lane_here()];
  // (what does not depend on the record, while it is on its way)
  NarrowStream<D, GATHERED> rows(a, smem, (unsigned)slot * N::kLds, kvh, p.w, share);
  asm volatile("" : "+s"(rows.kbase), "+s"(rows.vbase), "+s"(rows.k_stride), "+s"(rows.v_stride));
  if (p.inlined) {
    vn.kv_base = __builtin_amdgcn_readlane(p.rec, 0);
    vn.kv_len = __builtin_amdgcn_readlane(p.rec, 1);
    vn.q_off = __builtin_amdgcn_readlane(p.rec, 2);
    vn.q_len = __builtin_amdgcn_readlane(p.rec, 3);
  } else if (exists) {
    vn = uniform(load_vnode<GATHERED>(a, a.narrow_begin + index));
  }
  // (complete for the compiler on every path: a wait for it behind the first direct loads would be a wait for those)
  asm volatile("" : "+v"(p.rec));
  int groups = (vn.q_len * a.g + 15) >> 4;
  if (!ALONE && share > 1 && share < kWideWaves) {
    // every wave of the block makes the same passes (block barriers inside): the most row groups any of
    // its vnodes has, agreed on through one word of each wave's LDS area
    const unsigned word = lds_offset(smem);
    *reinterpret_cast<__attribute__((address_space(3))) int*>((uintptr_t)(word + (unsigned)slot * N::kLds)) = groups;
    __syncthreads();
    for (int i = 0; i < kWideWaves; ++i) groups = max(groups, (int)lds_read4(word + (unsigned)i * N::kLds));
    groups = __builtin_amdgcn_readfirstlane(groups);
    __syncthreads();
  }
  for (int done = 0; done < groups; done += N::kGroups) {
    p.row0 = 16 * done;
    // With the vnode's record at hand and the run's first tile to serve, the first 32 slot indices are already
    // here: the rows are requested at once, ahead of the code that differs between the numbers of row groups.
    rows.open(a, vn);
    p.started = !GATHERED && p.inlined && rows.tile0 == 0;
    if (p.row0 < vn.q_len * a.g && rows.tile0 < rows.ntiles) {
      if (p.started) {
        rows.rows_of_record(p.rec);
        rows.issue(false);
        rows.issue(true);
      }
      if (!p.started || rows.pairs()) rows.issue_indices(0, rows.tile0);   // (the second tile's indices too)
      if (!rows.pairs()) rows.issue_indices(1, rows.tile0 + rows.stride);
    }
    if (groups - done >= 2) narrow_pass<E, D, 2, GATHERED, REST>(a, smem, vn, rows, p);
    else narrow_pass<E, D, 1, GATHERED, REST>(a, smem, vn, rows, p);
    if (share > 1) __syncthreads();  // the exchange area is the staging area of the next pass
  }
}

// Narrow vnodes alone (a launch without wide vnodes), one vnode per block of `narrow_share`
// waves: the footprint of one LDS tile per wave instead of a wide block's ring, so that more of
// these latency-bound waves share a compute unit.
template <typename E, int D, bool GATHERED>
__global__ void __launch_bounds__(kWideBlock, D > 128 ? 1 : 2) stage1_narrow_kernel(const int32_t* records, int hkv, unsigned hkv_mul, unsigned hkv_shift, Stage1Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int index = Divisor{hkv_mul, hkv_shift}(blockIdx.x);
  narrow_item<E, D, GATHERED, true>(a, records, smem, wave, a.narrow_share, true, index, blockIdx.x - index * hkv);
}

// Whole paths (small launches; see ft_decode_programs): every request is in one vnode, whose run is the request's whole path,
// so a vnode's merged rows are the requests' outputs and there is no second launch.  One block per (vnode, kv head), whose
// waves take every kPathWaves-th tile of the run; each starts from a record of its own, with the slots of its first tile.
//
// Bound by the chain of a launch's start, two memory round trips (record, rows) and one more per tile of the same wave, and the
// merge, in few blocks: as many waves as the unit's LDS holds tiles for, 8 of 17 KB or 4 of 33 KB.  (4 requests of a short
// prompt, whole calls: 7.5 us in two launches, 6.4 so, and a launch less for the host: 8.3 and 6.2 back to back.)
//
// A path in so few parts has fewer soft-max references than one in pieces, each the maximum of its part, whose probability is
// 1 and not rounded: the parts of a path would round more of P (408 tokens, against 64 bits 2.67e-4 and 2.71e-4, fp16).  So what
// the rounding leaves over is contracted too, a third of a microsecond, and only the output's rounding is left (2.08e-4).
template <int D> constexpr int kPathWaves = FT_PATH_WAVES(D);
struct PathArgs {
  Stage1Args s;
  char* o;
  int64_t oo0, oo1;
};
constexpr int kPathFirstBytes = 24;      // of stage1_paths_kernel's arguments ahead of PathArgs
__device__ __forceinline__ const PathArgs& path_args_again() {   // (see args_again)
  auto p = (const __attribute__((address_space(4))) PathArgs*)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + kPathFirstBytes);
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+s"(p));
#endif
  return *(const PathArgs*)p;
}
template <typename E, int D> struct WriteOutput {
  const PathArgs& d;
  int q_off, rec;
  bool recorded;                 // wave uniform: the vnode's requests are in the record
  __device__ __forceinline__ int request(int ri) const {
    int req = lane_value(rec, 4 + (ri & (kNarrowRecRequests - 1)));
    if (!recorded) req = d.s.q_entries[q_off + ri];
    return req;
  }
  // A wave that finds NaN in the 16 dims from `dim` on (see narrow_attend) sums them again from the rows in memory, relative to the
  // merged maximum m: slow, but small, and of no concern to the block's other waves (looking at the states ahead of the merge takes
  // .1 us a call, so does letting the block's waves agree on walking the tiles again).
  // Lane (r16, c) takes every fourth token for row r16; `sum` is of the dims dim + 4 c .. + 3.
  static constexpr bool kSumsAgain = true;
  __device__ __forceinline__ void sum_again(int kvh, int req, int head, int dim, float m, f32x4& sum) const {
    const PathArgs& d = path_args_again();
    int again = rec;
    asm volatile("" : "+v"(again));
    const int c = lane_here() >> 4, kv_len = __builtin_amdgcn_readlane(again, 1);
    const int32_t* slots = d.s.kv_entries + __builtin_amdgcn_readlane(again, 0);
    const u32x4* q = reinterpret_cast<const u32x4*>(d.s.q + 2 * ((int64_t)req * d.s.sq0 + (int64_t)head * d.s.sq1));
    float acc[16] = {};
#pragma unroll 1
    for (int t = c; t < kv_len; t += 4) {
      const int64_t slot = slots[t];
      const u32x4* k = reinterpret_cast<const u32x4*>(d.s.k + 2 * (slot * d.s.sk0 + (int64_t)kvh * d.s.sk1));
      const u32x4* v = reinterpret_cast<const u32x4*>(d.s.v + 2 * (slot * d.s.sv0 + (int64_t)kvh * d.s.sv1 + dim));
      float s = 0.f;
#pragma unroll 4
      for (int i = 0; i < D / 8; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) s = __builtin_fmaf(E::of_pair(q[i][e >> 1], e & 1), E::of_pair(k[i][e >> 1], e & 1), s);
      const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s, d.s.scale_log2, -m));
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = __builtin_fmaf(x, E::of_pair(v[e >> 3][(e >> 1) & 3], e & 1), acc[e]);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float of_all = xor32_sum(xor16_sum(acc[e]));
      sum[e & 3] = c == e >> 2 ? of_all : sum[e & 3];
    }
  }
  __device__ __forceinline__ void write(int req, int head, int dim, const f32x4& x) const {
    *reinterpret_cast<u32x2*>(d.o + 2 * ((int64_t)req * d.oo0 + (int64_t)head * d.oo1 + dim)) = u32x2{E::pack2(x[0], x[1]), E::pack2(x[2], x[3])};
  }
};
template <typename E, int D, int NG>
__device__ __forceinline__ void path_pass(const PathArgs& d, char* smem, const VnodeView& vn, NarrowStream<D, false>& rows, int kvh, int row0, int rec) {
  const Stage1Args& a = d.s;
  static_assert(SharedState<D, NG>::kFloats * kWave * 4 <= NarrowGeom<D>::kLds, "a wave's state fits its LDS area");
  WaveState<D, NG> st;
  narrow_attend<E, D, NG, false, true>(a, vn, rows, true, kvh, row0, st, rec, true);
  float* xchg = reinterpret_cast<float*>(smem);
  SharedState<D, NG>::put(xchg + rows.tile0 * (NarrowGeom<D>::kLds / 4), st);
  __syncthreads();
  const WriteOutput<E, D> out{d, vn.q_off, rec, vn.q_len <= kNarrowRecRequests};
  write_merged_shares<D, NG, kPathWaves<D>>(a, xchg, vn, kvh, row0, rows.tile0, out);
}
template <typename E, int D>
__global__ void __launch_bounds__(kWave * kPathWaves<D>, D <= 128 ? 2 : 1) stage1_paths_kernel(const int32_t* wave_records, int hkv, unsigned hkv_mul, unsigned hkv_shift, PathArgs d) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const Stage1Args& a = d.s;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vnode = Divisor{hkv_mul, hkv_shift}(blockIdx.x), kvh = (int)blockIdx.x - vnode * hkv;
  int rec = wave_records[((int64_t)vnode * kPathWaves<D> + wave) * kNarrowRecord + lane_here()];
  NarrowStream<D, false> rows(a, smem, (unsigned)wave * NarrowGeom<D>::kLds, kvh, wave, kPathWaves<D>);
  asm volatile("" : "+s"(rows.kbase), "+s"(rows.vbase), "+s"(rows.k_stride), "+s"(rows.v_stride));
  VnodeView vn;
  vn.kv_base = __builtin_amdgcn_readlane(rec, 0);
  vn.kv_len = __builtin_amdgcn_readlane(rec, 1);
  vn.q_off = __builtin_amdgcn_readlane(rec, 2);
  vn.q_len = __builtin_amdgcn_readlane(rec, 3);
  // (complete for the compiler: a wait for it behind the first direct loads would be a wait for those)
  asm volatile("" : "+v"(rec));
  const int groups = (vn.q_len * a.g + 15) >> 4;
  for (int done = 0; done < groups; done += NarrowGeom<D>::kGroups) {
    rows.open(a, vn);
    if (rows.tile0 < rows.ntiles) {
      rows.rows_of_record(rec);
      rows.issue(false);
      rows.issue(true);
      rows.issue_indices(1, rows.tile0 + rows.stride);
    }
    if (groups - done >= 2) path_pass<E, D, 2>(d, smem, vn, rows, kvh, 16 * done, rec);
    else path_pass<E, D, 1>(d, smem, vn, rows, kvh, 16 * done, rec);
    __syncthreads();  // the exchange area is the staging area of the next pass
  }
}

// Blocks are handed to compute units in index order as units become free, so serving the wide
// vnodes in order of decreasing work (query rows x tokens) is longest-job-first list scheduling:
// the machine does not end on a late start of a long block.  Every block ranks the wide vnodes
// itself (they are few) and takes the one whose rank is `target`.  Block uniform.
//
// On the way, neighbours in the vnode list that attend the same KV run with adjoining scratch
// rows -- the query tiles the planner cut one node into -- are joined into one work item of at
// most `cap` query rows (what the blocks of one vnode serve in a single pass): a tile of 16
// requests x 4 heads fills only half of a block's rows, and two such tiles would stage the same
// run twice.  The first vnode of a group carries the group; the others become empty items.
//
// Every block does this before its first load, with cold code: 3.4 us of a block's start with 64-bit divisions, five
// barriers and the vnodes' entries through LDS; the 400-request tree 60.6 -> 59.9 us with the form below.
constexpr int kMaxRanked = kWideBlock;
// a / b for whole 0 <= a < 2048 and 1 <= b < 2^24: (a + 1/2) / b is at least 1 / 2b from a whole number, which the error
// of the reciprocal, less than 2^-20 of the quotient, does not reach.
__device__ __forceinline__ int small_quotient(int a, int b) { return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b)); }
template <bool GATHERED>
__device__ __forceinline__ void wide_vnode_of_rank(const Stage1Args& a, char* smem, int target, VnodeView& view) {
  const int n = a.vnode_count;
  if (n < 2 || n > kMaxRanked) {
    view = load_vnode<GATHERED>(a, a.vnode_begin + target);
    return;
  }
  // keys[u]: work of vnode u in 23 bits (a float's exponent and leading mantissa bits), then
  // 256 - u: larger key = earlier, no two equal; 0 for a vnode that is not the head of a group
  unsigned* keys = reinterpret_cast<unsigned*>(smem);
  int* q_len_of = reinterpret_cast<int*>(keys + kMaxRanked);
  int* q_end_of = q_len_of + kMaxRanked;                               // scratch rows end, per vnode
  unsigned long long* joined = reinterpret_cast<unsigned long long*>(q_end_of + kMaxRanked);  // one bit per vnode
  VnodeView* found = reinterpret_cast<VnodeView*>(joined + kMaxRanked / 64);
  const int tid = threadIdx.x;
  VnodeView mine{0, 0, 0, 0};
  // bit u: vnode u continues vnode u - 1 (same run, adjoining scratch rows; both read here, in one round trip).
  // Nothing is joined while there are no more blocks than compute units: two half-filled blocks side by side
  // finish sooner than one full block.
  bool joins = false;
  if (tid < n) {
    mine = load_vnode<GATHERED>(a, a.vnode_begin + tid);  // the block's own vnode is among them
    const VnodeView p = load_vnode<GATHERED>(a, a.vnode_begin + max(tid - 1, 0));
    joins = tid > 0 && 2LL * n * a.hkv * a.wide_chunks > a.block_slots && p.kv_base == mine.kv_base && p.kv_len == mine.kv_len &&
            p.q_off + p.q_len == mine.q_off;
    q_len_of[tid] = mine.q_len;
    q_end_of[tid] = mine.q_off + mine.q_len;
  }
  const unsigned long long wave_bits = __ballot(joins);
  if ((tid & 63) == 0) joined[tid >> 6] = wave_bits;
  if (tid == 0) *found = VnodeView{0, 0, 0, 0};    // (stays where there are more ranks than groups: an empty item)
  __syncthreads();
  unsigned key = 0;
  if (tid < n) {
    // first and last vnode of the chain of joined vnodes that holds this one
    int first = tid;
    for (int w = tid >> 6, hi = tid & 63; w >= 0; --w, hi = 63) {
      const unsigned long long stops = ~joined[w] & (hi == 63 ? ~0ull : ((2ull << hi) - 1));
      if (stops) {
        first = 64 * w + 63 - __builtin_clzll(stops);
        break;
      }
    }
    int last = n - 1;
    for (int u = tid + 1, w = u >> 6; w < (n + 63) / 64; ++w, u = 64 * w) {
      const unsigned long long stops = ~joined[w] & (~0ull << (u & 63));
      if (stops) {
        last = min(n, 64 * w + __builtin_ctzll(stops)) - 1;
        break;
      }
    }
    // groups of m vnodes from the start of the chain; the chain's first vnode is a full query tile (a cap of at most
    // 8 chunks of 192 rows; g at most 64)
    const int m = max(1, small_quotient(a.join_rows * a.wide_chunks, max(1, min(q_len_of[first], 4096) * a.g)));
    const int head = first + small_quotient(tid - first, m) * m;
    if (head == tid) {
      mine.q_len = q_end_of[min(last, head + m - 1)] - mine.q_off;
      const float work = (float)mine.q_len * (float)a.g * (float)mine.kv_len;
      // (256 - tid is never 0: the key of a vnode without work must not be the 0 of "no group")
      static_assert(kMaxRanked <= 256, "the low nine bits of a key hold 256 - tid");
      key = ((__builtin_bit_cast(unsigned, work) >> 8) << 9) | (unsigned)(256 - tid);
    }
  }
  keys[tid] = key;  // all kMaxRanked entries: the vector reads below run over the padding
  __syncthreads();
  if (key != 0) {
    int rank = 0;
    for (int j0 = 0; j0 < n; j0 += 16) {  // (keys past n are 0 and count for nothing)
      u32x4 k[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) k[i] = *reinterpret_cast<const u32x4*>(keys + j0 + 4 * i);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) rank += k[i][e] > key ? 1 : 0;
    }
    if (rank == target) *found = mine;
  }
  __syncthreads();
  view = *found;
  __syncthreads();  // the ranking area is reused as the staging ring
}

// The wide vnodes of one block program for one kv head (kv head fastest among the blocks: the eight blocks of a program
// land on the eight XCDs, and a head's K/V only ever enters one XCD's L2), one after the other.
template <typename E, int D, bool AGAIN>
__device__ __forceinline__ void program_block(const Stage1Args& a, const First& f, char* smem, int program, int kvh) {
  const PlanInts table = plan_ints(f.prog_table) + 4 * (int64_t)program;
  const int first = table[0], end = table[1];
  RowStream<D, false> rows(a, smem, kvh);
  RecordRequests requests;
  VnodeView vn{0, 0, 0, 0};
  bool listed = false;
  const bool record = f.prog_records != nullptr;   // launch uniform
  if (record) {
    // table entry and record in one round trip
    const int32_t* at = f.prog_records + (int64_t)program * kProgRecord;
    const PlanInts head = plan_ints(at);
    vn = VnodeView{head[2], head[3], head[1], (int64_t)head[0]};
    listed = head[4] != 0;
#pragma unroll
    for (int u = 0; u < WideGeom<D>::kSlots; ++u) rows.srow[u] = (unsigned)at[kProgRecSlots + rows.row(u)];
    requests.load(at);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+s"(vn.q_off), "+s"(vn.q_len), "+s"(vn.kv_len), "+s"(vn.kv_base));
    // (awaited together: a wait for the last of them behind the first direct loads would be a wait for those too)
    asm volatile("" : "+v"(requests.even), "+v"(requests.odd));
#pragma unroll
    for (int u = 0; u < WideGeom<D>::kSlots; ++u) asm volatile("" : "+v"(rows.srow[u]));
  }
  for (int v = first; v < end; ++v) {
    if (v > first || !record) vn = load_vnode<false>(a, a.vnode_begin + v);
    wide_block<E, D, false>(AGAIN ? args_again() : a, smem, vn, kvh, 0, 1, rows, listed, requests);
    listed = false;
  }
}

// The item of a wave of the fused kernel's trailing blocks: `index` counts them behind the `in_programs`
// items of the programs.  The waves of the last block that have none get `end`: up to three lie past it,
// which is past 2^31 for a launch of the most items the host allows, hence the sum without sign.
__host__ __device__ constexpr int trailing_item(int index, int in_programs, int end) {
  return (unsigned)index + (unsigned)in_programs < (unsigned)end ? index + in_programs : end;
}
static_assert(trailing_item(5, 7, 20) == 12 && trailing_item(12, 7, 20) == 19 && trailing_item(13, 7, 20) == 20);
static_assert(trailing_item(INT32_MAX - 10, 9, INT32_MAX) == INT32_MAX - 1 && trailing_item(INT32_MAX - 10, 13, INT32_MAX) == INT32_MAX);

// How a fused launch gets its wide vnodes: as the planner's list; as block programs (Stage1Args::prog_table); as
// block programs that also serve narrow vnodes (Stage1Args::narrow_in_programs).  A kernel for each: one holds no code
// that its launches do not run.
constexpr int kLists = 0, kPrograms = 1, kEmbedding = 2, kServing = 3;

// What bounds the start of a block is the fetch of its instructions, which every launch begins with an empty
// cache for: with one loop over both kinds of work, compiler-made divisions and the program's record handed round
// through LDS, 232 blocks of a 33 thousand token run asked for their first rows 3.9 us after they had their record, and
// 1.6 us when the same code ran a second time.  So each kind of work is a straight line from here, each wave reads
// what it needs of a record straight into registers, and the rows are on their way before the code that consumes
// them is fetched (whole calls: 6 waves' worth of leaves 10.4 -> 9.7 us, 111 ragged requests 14.5 -> 13.6, the
// 400-request tree in the planner's lists 66.3 -> 64.0).
// Launch order of the fused kernel.  Wide blocks come first: programs in index order, kv head fastest, or
// rank-major, then row chunk, kv head fastest (blocks that stream the same KV run are launched together and share it
// in L2); the narrow blocks follow and fill the machine while the wide blocks drain.
// Waves per SIMD that the registers must leave room for: as many blocks per compute unit as its LDS holds of
// 512-byte rows (one) and 256-byte rows (two).  Below that three have 168 registers each, and the
// kernels take 155 to 160: for the planner's lists they are kept to that (534 requests of 32/8 heads of 64: 102.6 us with
// 168, 110.4 with the 171 that an earlier form took by itself); programs came out slower under the limit.
constexpr int fused_waves(int D, int mode) { return D > 128 ? 1 : D == 128 || mode != kLists ? 2 : 3; }
template <typename E, int D, bool GATHERED, int MODE>
__device__ __forceinline__ void fused_block(const Stage1Args& a, const First& f, char* smem) {
  const int narrow_index = (int)blockIdx.x - f.wide_blocks;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (512-byte rows: most trees gain 1 to 3 % by it, but 32 requests of 64/8 heads of 256 on 15 thousand tokens lose,
  // 121.1 -> 123.3 us.)
  constexpr bool kAgain = D <= 128;
  if (narrow_index < 0) {
    if constexpr (MODE == kLists) {
      const int slot_of_all = f.by_hkv(blockIdx.x), kvh = (int)blockIdx.x - slot_of_all * f.hkv;
      const int rank = a.by_chunks(slot_of_all);
      // Launch slot s of a rank serves chunk (s + rank / 2) % chunks.  Consecutive
      // blocks of one kv head go round robin to the four shader engines of an XCD, strictly in
      // order (a block waits for its engine even when others have room); without the rotation an
      // engine would only ever get first chunks, which run longer than last ones.
      const int chunks = a.wide_chunks, turned = slot_of_all - rank * chunks + (rank >> 1), chunk = turned - a.by_chunks(turned) * chunks;
      VnodeView vn{0, 0, 0, 0};
      wide_vnode_of_rank<GATHERED>(a, smem, rank, vn);
      vn = uniform(vn);
      const Stage1Args& b = kAgain ? args_again() : a;
      RowStream<D, GATHERED> rows(b, smem, kvh);
      wide_block<E, D, GATHERED>(b, smem, vn, kvh, chunk, chunks, rows, false, RecordRequests());
    } else if constexpr (MODE != kEmbedding) {
      const int program = f.by_hkv(blockIdx.x);
      program_block<E, D, kAgain>(a, f, smem, program, (int)blockIdx.x - program * f.hkv);
    } else {
      // A program's narrow vnodes, one wave each, before its wide ones (a negative count) or after them: of the
      // two blocks that share a compute unit one starts with its narrow vnodes and the other ends with them, so that
      // the memory-bound narrow vnodes of one run under the arithmetic-bound wide vnodes of the other.
      const int program = f.by_hkv(blockIdx.x), kvh = (int)blockIdx.x - program * f.hkv;
      const PlanInts table = plan_ints(f.prog_table) + 4 * (int64_t)program;
      const int first = table[2], count = table[3];
      // (one call each, in either order, so that the kernel holds one copy of the code)
#pragma unroll 1
      for (int turn = 0; turn < 2; ++turn) {
        if ((turn == 0) == (count < 0)) {
          for (int v = first + wave; v < first + abs(count); v += kWideWaves)
            narrow_item<E, D, GATHERED, false>(kAgain ? args_again() : a, f.narrow_table, smem, wave, 1, true, v, kvh);
          __syncthreads();  // the waves' tiles become the ring of the next wide vnode
        } else {
          program_block<E, D, kAgain>(a, f, smem, program, kvh);
        }
      }
    }
  } else {
    // trailing blocks: an item per wave, or per `share` waves; a wave that shares no vnode and has none is done
    const int share = f.narrow_share, log_share = share >> 1;   // 1, 2, 4 -> 0, 1, 2
    const int end = f.narrow_items;
    const int item = trailing_item((narrow_index * kWideWaves + wave) >> log_share, MODE == kEmbedding ? a.narrow_in_programs * f.hkv : 0, end);
    if (item < end || share > 1) {
      const int index = f.by_hkv(item);
      // (Vnodes without records beside programs are a serving plan's, where a request's prompt and generated tokens may be one
      // vnode: a maximum, whose probability is 1, the fewer, and more rounded.  128 requests of 2746 tokens, against 64 bits:
      // 2.890e-4 apart, 2.895e-4 as one, 2.842e-4 with what rounding leaves over (fp16); 120 of 1242 2.275e-3, 2.282e-3 and
      // 2.173e-3 (bf16); 0 to .1 us.)
      narrow_item<E, D, GATHERED, false, MODE == kServing>(kAgain ? args_again() : a, f.narrow_table, smem, wave, share, item < end, index, item - index * f.hkv);
    }
  }
}

template <typename E, int D, bool GATHERED, bool PROGRAMS>
__global__ void __launch_bounds__(kWideBlock, fused_waves(D, PROGRAMS ? kPrograms : kLists)) stage1_fused_kernel(FT_FIRST_PARAMETERS, Stage1Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  fused_block<E, D, GATHERED, PROGRAMS ? kPrograms : kLists>(a, FT_FIRST, smem);
}

template <typename E, int D>
__global__ void __launch_bounds__(kWideBlock, fused_waves(D, kEmbedding)) stage1_embedding_kernel(FT_FIRST_PARAMETERS, Stage1Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  fused_block<E, D, false, kEmbedding>(a, FT_FIRST, smem);
}

// Programs, and narrow vnodes without records, whose remainders are contracted: a kernel of its own, for that code beside every launch
// of programs costs the others up to 2 % (with it and the second walk 16.4 -> 16.8 us for 64 of 16/1 heads of 256, the
// 400-request tree 58.7 -> 59.1; without either 57.8).
template <typename E, int D>
__global__ void __launch_bounds__(kWideBlock, fused_waves(D, kServing)) stage1_serving_kernel(FT_FIRST_PARAMETERS, Stage1Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  fused_block<E, D, false, kServing>(a, FT_FIRST, smem);
}

// ---------------------------------------------------------------------------------------
// DeFT-Flatten's first stage (the comparison engine of the reference's benchmark,
// kernel_bench/DeFT.py:194-340): one block per (subtree, kv head).  A subtree is a run of
// consecutive tokens of the depth-first token order (128 in the benchmark) that may span
// several tree nodes; its query set holds every request that attends any of its tokens, and a
// 64-bit word per (group of mask_len requests, token) says which requests of the group attend the
// token.  The block keeps up to 128 tokens of the subtree in LDS (the two super-tile buffers of
// the wide kernel, same layout, same direct loads) and passes its query rows over them 128 at a
// time, 32 per wave, with the scores of tokens a row does not attend set to a large negative
// value before the soft-max (DeFT.py:283-306).  The partial output is rounded to fp16 on its
// way to the fp32 scratch, as the reference kernel does (DeFT.py:391).
// ---------------------------------------------------------------------------------------
struct DeftArgs {
  Stage1Args s;                    // tensors, strides, the six vnode lists (vnode = subtree), scale, scratch
  const int64_t* causalmask;       // per subtree: [groups of mask_len requests][kv_len] words
  const int32_t* causalmask_offset;
  int mask_len;                    // requests per mask word: a power of two, at most 64
  int num_subtrees;
};

constexpr int kDeftChunk = 2 * 64;       // tokens held in LDS at a time (both ring buffers)
// Raw score of a token a row does not attend (the reference writes -1e6 over the scaled score,
// DeFT.py:306).  Finite and moderate on purpose: a tile in which a row attends nothing makes this
// value the row's soft-max reference, and the probabilities of that tile come out as exp2 of the
// rounding error of (score * scale) -- about 1 for this magnitude, infinite for a huge one.  They
// are garbage either way and are wiped out (factor exp2(-1e5) = 0) by the first attended token.
constexpr float kDeftMasked = -1.0e6f;
constexpr int kDeftMaskGroups = 5;       // mask groups 128 consecutive query rows can touch (g = 1, mask_len 32: 4 + 1)

template <typename E, int D>
__global__ void __launch_bounds__(kWideBlock, D > 128 ? 1 : 2) deft_stage1_kernel(DeftArgs d) {
  using W = WideGeom<D>;
  const Stage1Args& a = d.s;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int subtree = blockIdx.x / a.hkv;
  const int kvh = blockIdx.x - subtree * a.hkv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const VnodeView vn = load_vnode<false>(a, subtree);
  const int rows_total = vn.q_len * a.g;
  const int64_t* masks = d.causalmask + d.causalmask_offset[subtree];
  const int grp_row = lane / W::kChunks, pos = lane % W::kChunks;
  const char* kbase = a.k + 2 * ((int64_t)kvh * a.sk1);
  const char* vbase = a.v + 2 * ((int64_t)kvh * a.sv1);
  const unsigned k_stride = (unsigned)(2 * a.sk0), v_stride = (unsigned)(2 * a.sv0);
  const unsigned ring = lds_offset(smem);
  // the mask words of the chunk in LDS, after the ring: [kDeftMaskGroups][kDeftChunk] 64-bit words
  uint32_t* mask_lds = reinterpret_cast<uint32_t*>(smem + W::kRing);
  const unsigned mask_lds_addr = ring + W::kRing;
  WideLane la0;
  init_lane<D>(la0, ring);
  const int nchunks = (vn.kv_len + kDeftChunk - 1) / kDeftChunk;
  const int h = lane >> 5;

  for (int row0 = 0; row0 < rows_total; row0 += kDeftRows) {
    const int my_row0 = row0 + 32 * wave;
    const bool active = my_row0 < rows_total;
    const char* q_src = q_row_address32(a, vn, kvh, active ? my_row0 : rows_total);
    u32x4 qf[D / 16];
    load_q_frags32<D>(q_src, qf);
    WideState<D> st;
    reset_state<D>(st);
    // the lane's request within the subtree's query set, its mask group and its bit in the group's words
    const int my_req = min(my_row0 + (lane & 31), rows_total - 1) / a.g;
    const int first_group = (row0 / a.g) / d.mask_len;
    const int groups_here = min((min(row0 + kDeftRows, rows_total) - 1) / a.g / d.mask_len - first_group + 1, kDeftMaskGroups);
    const int my_group = min(my_req / d.mask_len - first_group, kDeftMaskGroups - 1);
    const int my_bit = my_req & (d.mask_len - 1);
    const bool upper = my_bit >= 32;
    const unsigned bit = 1u << (my_bit & 31);
    for (int chunk = 0; chunk < nchunks; ++chunk) {
      const int c0 = chunk * kDeftChunk;
      const int here = min(kDeftChunk, vn.kv_len - c0);
      __syncthreads();   // the previous pass (or chunk) is out of LDS
      if (row0 == 0 || nchunks > 1) {
        // K and V rows of the chunk: 2 x 16 groups of 1 KB per super tile, dealt to the four waves
        // (tokens past the end repeat the last one: their scores are masked)
#pragma unroll
        for (int sup = 0; sup < 2; ++sup)
#pragma unroll
          for (int u = 0; u < W::kUnits; ++u) {
            const bool is_v = W::kGroups >= kWideWaves ? u >= W::kSlots : wave >= W::kGroups;
            const int sl = u % W::kSlots;
            const int grp = W::kGroups >= kWideWaves ? sl * kWideWaves + wave : wave % W::kGroups;
            const int row = grp * W::kGroupRows + grp_row;
            const int t = min(c0 + sup * W::kTokens + row, vn.kv_len - 1);
            const unsigned slot = (unsigned)a.kv_entries[vn.kv_base + t];
            const char* src = (is_v ? vbase : kbase) + (uint64_t)slot * (is_v ? v_stride : k_stride);
            load_direct16(src + 16 * (pos ^ W::swz(row)), ring + sup * W::kBytes + (is_v ? W::kBytesK : 0) + grp * 1024);
          }
      }
      // the mask words of this pass's groups for the chunk's tokens (zero past the subtree)
      for (int i = threadIdx.x; i < groups_here * kDeftChunk; i += kWideBlock) {
        const int gsel = i / kDeftChunk, t = i - gsel * kDeftChunk;
        const int64_t word = t < here ? masks[(int64_t)(first_group + gsel) * vn.kv_len + c0 + t] : 0;
        mask_lds[2 * i] = (uint32_t)(uint64_t)word;
        mask_lds[2 * i + 1] = (uint32_t)((uint64_t)word >> 32);
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): rows landed (and the Q fragments)
      __syncthreads();
      if (active) {
        const int tiles = (here + kTileTokens - 1) / kTileTokens;
        for (int tile = 0; tile < tiles; ++tile) {
          // the lane's 16 tokens of the tile are four runs of four consecutive ones: 32 bytes of mask words each
          const unsigned words = mask_lds_addr + 8u * (unsigned)(my_group * kDeftChunk + tile * kTileTokens + 4 * h);
          auto mask = [&](f32x16& sc) {
#pragma unroll
            for (int quad = 0; quad < 4; ++quad) {
              const u32x4 w0 = lds_read16(words + 64u * quad), w1 = lds_read16(words + 64u * quad + 16u);
              const unsigned m4[4] = {upper ? w0[1] : w0[0], upper ? w0[3] : w0[2], upper ? w1[1] : w1[0], upper ? w1[3] : w1[2]};
#pragma unroll
              for (int jj = 0; jj < 4; ++jj) sc[4 * quad + jj] = (m4[jj] & bit) ? sc[4 * quad + jj] : kDeftMasked;
            }
          };
          const WideLane la = at_buffer(la0, (unsigned)(tile >> 1) * W::kBytes);
          tile_step32<E, D>(la, (tile & 1) * W::kTileBytes, here - tile * kTileTokens, a.scale_log2, qf, st, mask);
        }
      }
    }
    finish_state<D>(st);
    // (the reference rounds the normalised partial output to fp16 before it stores it, DeFT.py:391)
    if (active) write_partials32<D, true>(a, vn, kvh, my_row0, st);
  }
}

// ---------------------------------------------------------------------------------------
// Stage 2
// ---------------------------------------------------------------------------------------
struct Stage2Args {
  const int32_t* req_entries;
  const int32_t* req_offs;
  const int32_t* req_lens;
  const float* mid_o;
  int64_t so0, so1;
  const float* mid_lse;
  int64_t sl0;
  char* o;
  int64_t oo0, oo1;
  int batch, hq;
  int longest; // no request has more partials than this (the number of vnodes, or more)
  int log_splits;  // 1 << this many waves share a request's list, set by the launcher
  int log_groups;  // and in kLongLists at most 1 << this many groups of D/4 lanes one of more than kLongList entries
  int nsplit;  // > 0: gathered mode, request r owns rows [r*nsplit, (r+1)*nsplit)
  // (or null) one record of kReqRecord int32 per request, written by the host: req_lens[r],
  // req_offs[r], then the request's first kReqRecord - 2 entries -- what the block needs before
  // it can ask for the partial rows, in one memory round trip instead of two
  const int32_t* req_table;
};
constexpr int kReqRecord = 16;
constexpr int kReqRecEntries = kReqRecord - 2;
// How a launch reads its lists: each by one wave; each of more than kReqRecEntries entries by several waves; as that,
// but those of more than kLongList entries by groups of lanes.
constexpr int kWholeLists = 0, kSplitLists = 1, kLongLists = 2;
constexpr int kLongList = 64;
// Rows a wave asks for at once.  A list of more is cut where the machine has room for the waves: the second batch is a memory
// round trip, the merge through LDS less (16 requests of 32/32 heads with 9 rows each, whole calls: 14.2 us in two batches, 13.8
// by four waves).
constexpr int kOneWave = 8;

// The merge of a list of more than kLongList entries, n of them, from `list` on (or the rows from row0 on).  Four waves
// would read it in many batches, one round trip after the other, so it is cut finer: a group of D/4 lanes takes a part for
// one head.  Its lanes hold an entry each, with the entry's weight, fetch the next ones ahead and hand them round.
template <typename E, int D>
__device__ __forceinline__ void merge_long_list(const Stage2Args& a, int req, int n, int row0, PlanInts list) {
  constexpr int LPH = D / 4, kGroups = kBlock / LPH, kBatch = LPH < 8 ? LPH : 8;
  const int group = threadIdx.x / LPH, gl = threadIdx.x % LPH;
  const int log_parts = min(a.log_groups, 31 - __builtin_clz((unsigned)n / kBatch));   // (parts of kBatch entries and more)
  if (((int)blockIdx.y * kGroups) >> log_parts >= a.hq) return;     // block uniform
  const int parts = 1 << log_parts, part_of_group = group & (parts - 1);
  const int head = ((int)blockIdx.y * kGroups + group) >> log_parts;
  const bool exists = head < a.hq;
  const int head_in = exists ? head : a.hq - 1;             // (lanes past the last head read that one's rows and store nothing)
  const int size = (n + parts - 1) >> log_parts, first = part_of_group * size, mine = min(n - first, size);

  const char* o_lane = reinterpret_cast<const char*>(a.mid_o + (int64_t)head_in * a.so1 + 4 * gl);
  auto entry = [&](int i0) {                                // (past the part its last entry again, or the list's: not counted)
    const int i = min(first + i0 + gl, min(first + size, n) - 1);
    return a.nsplit > 0 ? row0 + i : list[i];
  };
  // x of the group's lane j (a constant after unrolling)
  auto of_lane = [](int x, int j) { return LPH == kWave ? __builtin_amdgcn_readlane(x, j) : __shfl(x, j, LPH); };
  float m_run = -INFINITY, l_run = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int row = entry(0);
  for (int base = 0; base < mine; base += LPH) {
    const int held = min(LPH, mine - base);
    float lse = a.mid_lse[(int64_t)row * a.sl0 + head_in];
    const int row_here = row;
    if (base + LPH < mine) row = entry(base + LPH);
    lse = gl < held ? lse : -INFINITY;
    f32x4 part[kBatch];
    auto request = [&](int i0) {
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        part[j] = *reinterpret_cast<const f32x4*>(o_lane + 4 * (int64_t)of_lane(row_here, i0 + j) * a.so0);
    };
    request(0);
    float m_new = lse;
#pragma unroll
    for (int d = LPH / 2; d >= 1; d >>= 1) m_new = fmaxf(m_new, __shfl_xor(m_new, d, LPH));
    m_new = fmaxf(m_run, m_new);
    const float keep = (m_run == -INFINITY) ? 0.f : __expf(m_run - m_new);
    const float w = (lse == -INFINITY) ? 0.f : __expf(lse - m_new);
    l_run *= keep;
    acc *= keep;
    m_run = m_new;
    for (int i0 = 0; i0 < held; i0 += kBatch) {
      if (i0 > 0) request(i0);
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const float w_j = __builtin_bit_cast(float, of_lane(__builtin_bit_cast(int, w), i0 + j));
        l_run += w_j;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += (w_j != 0.f) ? part[j][e] * w_j : 0.f;
      }
    }
  }
  // the groups' states to the first of them
  __shared__ f32x4 acc_of[kBlock];
  __shared__ float m_of[kGroups], l_of[kGroups];
  acc_of[threadIdx.x] = acc;
  if (gl == 0) {
    m_of[group] = m_run;
    l_of[group] = l_run;
  }
  __syncthreads();
  if (part_of_group > 0 || !exists) return;
  float m_all = m_run;
  for (int i = 1; i < parts; ++i) m_all = fmaxf(m_all, m_of[group + i]);
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
  l_run = 0.f;
  for (int i = 0; i < parts; ++i) {
    const float m_i = m_of[group + i];
    const float w = (m_i == -INFINITY) ? 0.f : __expf(m_i - m_all);
    l_run += l_of[group + i] * w;
    acc += acc_of[threadIdx.x + i * LPH] * w;
  }
  acc *= l_run > 0.f ? 1.f / l_run : 0.f;
  const u32x2 out = {E::pack2(acc[0], acc[1]), E::pack2(acc[2], acc[3])};
  *reinterpret_cast<u32x2*>(a.o + 2 * ((int64_t)req * a.oo0 + (int64_t)head * a.oo1 + 4 * gl)) = out;
}

// How the merge kernel spreads a request's heads: a lane holds kVec output dims of one head, and a head has whole rows of
// 16 lanes, so that what such a row's lanes hold of a list can be handed round inside it.
template <int D> struct MergeGeom {
  static constexpr int kVec = D >= 64 ? 4 : D / 16;
  static constexpr int kLanes = D / kVec;                   // lanes of a head: 16, 32 or 64
  static constexpr int kHeads = kWave / kLanes;             // heads of a wave
  typedef float Vec __attribute__((ext_vector_type(kVec)));
};
constexpr int kListRow = 16;                                // entries of a list that a row of lanes holds at a time

// x of lane J of this lane's row of 16 lanes.
template <int J> __device__ __forceinline__ int row_lane(int x) { return __builtin_amdgcn_mov_dpp(x, 0x150 + J, 0xf, 0xf, true); }
// x of the lane N places on in this lane's row of 16, around its end.
template <int N> __device__ __forceinline__ float row_turned(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x120 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_max(float x) {
  x = fmaxf(x, row_turned<8>(x));
  x = fmaxf(x, row_turned<4>(x));
  x = fmaxf(x, row_turned<2>(x));
  return fmaxf(x, row_turned<1>(x));
}
__device__ __forceinline__ float row_sum(float x) {
  x += row_turned<8>(x);
  x += row_turned<4>(x);
  x += row_turned<2>(x);
  return x + row_turned<1>(x);
}

// The N entries from J0 on of the 16 that the rows of lanes hold: their partial rows are asked for, all of them before
// the first is used, and added with their weights.
template <int D, int J0, int N> struct MergeBatch {
  using G = MergeGeom<D>;
  typedef typename G::Vec Vec;
  Vec part[N];

  // (`off`: of the row of the lane's entry, in bytes)
  template <int J = 0> __device__ __forceinline__ void request(const char* o_lane, uint64_t off) {
    const uint64_t base = (uint64_t)(uintptr_t)o_lane;
    unsigned carry, none;
    const unsigned lo = __builtin_addc((unsigned)base, (unsigned)row_lane<J0 + J>((int)(unsigned)off), 0u, &carry);
    const unsigned hi = __builtin_addc((unsigned)(base >> 32), (unsigned)row_lane<J0 + J>((int)(unsigned)(off >> 32)), carry, &none);
    part[J] = *reinterpret_cast<const __attribute__((address_space(1))) Vec*>((uintptr_t)(((uint64_t)hi << 32) | lo));
    if constexpr (J + 1 < N) request<J + 1>(o_lane, off);
  }
  // What the row of an entry of no weight holds is not looked at: it may have attended no token.
  template <int J = 0> __device__ __forceinline__ void forget_weightless(float w) {
    const bool none = __builtin_bit_cast(float, row_lane<J0 + J>(__builtin_bit_cast(int, w))) == 0.f;
#pragma unroll
    for (int e = 0; e < G::kVec; ++e) part[J][e] = none ? 0.f : part[J][e];
    if constexpr (J + 1 < N) forget_weightless<J + 1>(w);
  }
  template <int J = 0> __device__ __forceinline__ void add(float w, Vec& acc) const {
    const float w_j = __builtin_bit_cast(float, row_lane<J0 + J>(__builtin_bit_cast(int, w)));
#pragma unroll
    for (int e = 0; e < G::kVec; ++e) acc[e] = __builtin_fmaf(w_j, part[J][e], acc[e]);
    if constexpr (J + 1 < N) add<J + 1>(w, acc);
  }
};

// f with n, 1 to 8, as a constant.  (Code for each: a branch per entry and row takes as many instructions as the entry.)
template <typename F> __device__ __forceinline__ void with_count(int n, F f) {
#define FT_COUNT(k) f(std::integral_constant<int, k>())
  if (n <= 4) {
    if (n <= 2) { if (n == 1) FT_COUNT(1); else FT_COUNT(2); }
    else { if (n == 3) FT_COUNT(3); else FT_COUNT(4); }
  } else {
    if (n <= 6) { if (n == 5) FT_COUNT(5); else FT_COUNT(6); }
    else { if (n == 7) FT_COUNT(7); else FT_COUNT(8); }
  }
#undef FT_COUNT
}

// `splits` waves of a block (1, 2 or 4) take parts of the request's list and are merged through LDS.  Lane i of every row
// of 16 lanes holds entry i of (16 entries of) the wave's part: its row's offset, its log-sum-exp for the row's head, its
// weight.  A lane then asks for its output dims of every entry's row with the offset of the lane that holds it.
//
// Bound by the partial rows it reads in large launches (33 MB of the 400-request tree in 6.9 us), and in small ones by
// the instructions a wave issues one after the other, some 4.6 cycles each, and by how many rows are in flight.  With a
// list's entries as scalars, each with its own 64-bit address arithmetic, exponential and weight for the whole wave, and
// batches of eight rows whatever the list's length, a wave took 453 instructions for lists of three; 230 so (whole calls: 4 requests
// of a short prompt 7.96 -> 7.62 us, 16 of 32/32 heads 14.17 -> 13.54, 64 on a shared prefix 25.4 -> 24.6, 111 ragged requests
// of 64-dim heads 12.55 -> 12.4, 64 of 16/1 heads of 256 17.44 -> 17.18).
template <typename E, int D, int LISTS>
__global__ void __launch_bounds__(kBlock) stage2_kernel(const int32_t* records, Stage2Args a) {
  using G = MergeGeom<D>;
  typedef typename G::Vec Vec;
  constexpr bool SPLIT = LISTS != kWholeLists;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int gl = lane % G::kLanes, c = lane % kListRow;
  const int req = blockIdx.x;
  const int log_splits = SPLIT ? a.log_splits : 0;          // launch uniform
  const int head = ((((int)blockIdx.y * kWavesPerBlock) + wave) >> log_splits) * G::kHeads + lane / G::kLanes;
  const bool exists = head < a.hq;
  const int head_in = exists ? head : a.hq - 1;             // (lanes past the last head read that one's rows and store nothing)
  // this wave's part [first, first + n) of the request's list, from `list` on
  int n, first = 0, row0 = 0, recorded = 0;
  bool in_record = false;                                   // block uniform: the list is in the request's record
  const int32_t* list = nullptr;
  if (records) {                                            // launch uniform
    const int32_t* rec = records + (int64_t)req * kReqRecord;
    recorded = rec[2 + min(c, kReqRecEntries - 1)];         // (in one round trip with the length)
    n = plan_ints(rec)[0];
    list = a.req_entries + plan_ints(rec)[1];
    in_record = n <= kReqRecEntries;
  } else if (a.nsplit > 0) {
    n = a.nsplit;
    row0 = req * a.nsplit;
  } else {
    n = plan_ints(a.req_lens)[req];
    list = a.req_entries + plan_ints(a.req_offs)[req];
  }
  if constexpr (LISTS == kLongLists) {
    if (n > kLongList) return merge_long_list<E, D>(a, req, n, row0, plan_ints(list));
    // (the grid has the blocks that the one way or the other needs)
    if ((((int)blockIdx.y * kWavesPerBlock) >> log_splits) * G::kHeads >= a.hq) return;
  }
  int split = 0, splits = 1;
  if constexpr (SPLIT) {
    split = wave & ((1 << log_splits) - 1);
    if (n <= kOneWave) {
      if (split > 0) return;
    } else {
      splits = 1 << log_splits;
      const int part = (n + splits - 1) >> log_splits;
      first = split * part;
      n = max(0, min(n - first, part));
    }
  }

  // (rows and heads as numbers without sign: a product with a 64-bit stride is two instructions)
  const char* o_lane = reinterpret_cast<const char*>(a.mid_o) + ((uint64_t)(unsigned)head_in * (uint64_t)(4 * a.so1) + 4 * G::kVec * gl);
  const char* lse_lane = reinterpret_cast<const char*>(a.mid_lse + head_in);
  float m_run = -INFINITY, l_run = 0.f;
  Vec acc = {};
  for (int i0 = 0; i0 < n; i0 += kListRow) {
    int held = n - i0;
    asm volatile("" : "+s"(held));     // (or what every count below makes of it is computed ahead of the loop)
    // (lanes past the part hold an entry of it that has no weight there)
    int row;
    if (in_record) {
      row = SPLIT && first > 0 ? lane_value(recorded, lane - c + ((first + c) & (kListRow - 1))) : recorded;
      const int first_row = row_lane<0>(row);          // (moved by all lanes: in an arm of the choice the source lane would be off)
      row = c < held ? row : first_row;
    } else {
      const int i = first + i0 + min(c, held - 1);
      row = a.nsplit > 0 ? row0 + i : list[i];
    }
    float lse = *reinterpret_cast<const float*>(lse_lane + (uint64_t)(unsigned)row * (uint64_t)(4 * a.sl0));
    const uint64_t off = (uint64_t)(unsigned)row * (uint64_t)(4 * a.so0);
    float w;
    bool zeros;
    with_count(min(held, 8), [&](auto count) {
      MergeBatch<D, 0, count()> rows;
      rows.request(o_lane, off);
      lse = c < held ? lse : -INFINITY;
      const float m_new = fmaxf(m_run, row_max(lse));
      const float m_from = m_new == -INFINITY ? 0.f : m_new;  // (every log-sum-exp so far is -inf: every weight is 0)
      w = __expf(lse - m_from);
      zeros = __builtin_amdgcn_ballot_w64(c < held && w == 0.f) != 0;
      if (i0 > 0) {
        const float keep = __expf(m_run - m_from);
        l_run *= keep;
        acc = keep == 0.f ? Vec{} : acc * keep;
      }
      l_run += row_sum(w);
      m_run = m_new;
      if (zeros) rows.forget_weightless(w);
      rows.add(w, acc);
    });
    if (held > 8)
      with_count(min(held - 8, 8), [&](auto count) {
        MergeBatch<D, 8, count()> rows;
        rows.request(o_lane, off);
        if (zeros) rows.forget_weightless(w);
        rows.add(w, acc);
      });
  }
  if (SPLIT && splits > 1) {
    // the waves' states to the first of them
    __shared__ Vec acc_of[kBlock];
    __shared__ float m_of[kBlock], l_of[kBlock];
    acc_of[threadIdx.x] = acc;
    m_of[threadIdx.x] = m_run;
    l_of[threadIdx.x] = l_run;
    __syncthreads();
    if (split > 0) return;
    float m_all = m_run;
    for (int i = 1; i < splits; ++i) m_all = fmaxf(m_all, m_of[threadIdx.x + i * kWave]);
    acc = Vec{};
    l_run = 0.f;
    for (int i = 0; i < splits; ++i) {
      const float m_i = m_of[threadIdx.x + i * kWave];
      const float w = (m_i == -INFINITY) ? 0.f : __expf(m_i - m_all);
      l_run += l_of[threadIdx.x + i * kWave] * w;
      acc = w == 0.f ? acc : acc + acc_of[threadIdx.x + i * kWave] * w;
    }
  }
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  acc *= inv;
  if (!exists) return;
  char* out = a.o + 2 * ((int64_t)req * a.oo0 + (int64_t)head * a.oo1 + G::kVec * gl);
  if constexpr (G::kVec == 4) *reinterpret_cast<u32x2*>(out) = u32x2{E::pack2(acc[0], acc[1]), E::pack2(acc[2], acc[3])};
  else if constexpr (G::kVec == 2) *reinterpret_cast<unsigned*>(out) = E::pack2(acc[0], acc[1]);
  else *reinterpret_cast<unsigned short*>(out) = (unsigned short)E::pack2(acc[0], 0.f);
}

// ---------------------------------------------------------------------------------------
// The step's new K and V rows into the pools (one launch for both)
// ---------------------------------------------------------------------------------------
struct StoreArgs {
  const char* k_new;
  const char* v_new;
  int64_t kn0, kn1, vn0, vn1;  // element strides of the new rows [tokens, Hkv, D]
  const void* loc;             // pool slot per token, int32 or int64
  int loc_is_int64;
  char* k_pool;
  char* v_pool;
  int64_t sk0, sk1, sv0, sv1;
  int64_t num_slots;
  int hkv, chunks;             // chunks = 16-byte pieces per (token, head) row
  Divisor by_chunks;
  int tokens, per_block;       // of launches whose blocks serve several tokens
  Divisor by_pieces;           // of a token
};

// A thread moves 16 bytes of a K row and the same 16 bytes of the V row.  A token whose slot lies outside the pool is skipped.
// A block serves one token (or, of many heads, a part of it); of tokens that are less than a wave's pieces each (SEVERAL) it
// serves as many as it has threads for, or most lanes of the launch move nothing: 65536 tokens of one 64-dim head 5.3 us so,
// 16.8 by a wave each, 8192 tokens 2.7 and 3.5, of one 128-dim head 8.8 and 17.0.
// Bound by the launch and by memory round trips, and so the
// rows are asked for beside the slot (128 tokens into pools that nothing has touched since the last forward 4 to 4.7 us; touching
// their pages ahead of the slots changes nothing).
constexpr int kStoreBlock = 256;
template <bool SEVERAL> __global__ void __launch_bounds__(kStoreBlock) store_kv_kernel(StoreArgs a) {
  int64_t token = blockIdx.x;
  int i = blockIdx.y * blockDim.x + threadIdx.x;
  if constexpr (SEVERAL) {
    const int at = a.by_pieces(i);
    token = token * a.per_block + at;
    i -= at * a.hkv * a.chunks;
    if (at >= a.per_block || token >= a.tokens) return;
  } else {
    if (i >= a.hkv * a.chunks) return;
  }
  const int head = a.by_chunks(i), chunk = i - head * a.chunks;
  const u32x4 kx = *reinterpret_cast<const u32x4*>(a.k_new + 2 * (token * a.kn0 + head * a.kn1) + 16 * chunk);
  const u32x4 vx = *reinterpret_cast<const u32x4*>(a.v_new + 2 * (token * a.vn0 + head * a.vn1) + 16 * chunk);
  int64_t slot;
  if constexpr (SEVERAL) {
    slot = a.loc_is_int64 ? static_cast<const int64_t*>(a.loc)[token] : (int64_t) static_cast<const int32_t*>(a.loc)[token];
  } else {
    const PlanInts loc = plan_ints(static_cast<const int32_t*>(a.loc));
    slot = a.loc_is_int64 ? (int64_t)(((uint64_t)(unsigned)loc[2 * token + 1] << 32) | (unsigned)loc[2 * token]) : (int64_t)loc[token];
  }
  if (slot < 0 || slot >= a.num_slots) return;
  *reinterpret_cast<u32x4*>(a.k_pool + 2 * (slot * a.sk0 + head * a.sk1) + 16 * chunk) = kx;
  *reinterpret_cast<u32x4*>(a.v_pool + 2 * (slot * a.sv0 + head * a.sv1) + 16 * chunk) = vx;
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------
constexpr int kMaxDevices = 64;
inline int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) (void)hipGetLastError();
  return dev >= 0 && dev < kMaxDevices ? dev : 0;
}
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <typename E, int D, int NQB, bool SPLIT, bool GATHERED>
int launch_stage1_inst(const Stage1Args& a, int hkv, hipStream_t stream) {
  const size_t lds = (size_t)kWavesPerBlock * TileGeom<D>::kBytes;
  auto kern = stage1_kernel<E, D, NQB, SPLIT, GATHERED>;
  // (raising the dynamic LDS limit is idempotent: two threads that both find the flag clear both raise it)
  static std::atomic<bool> configured_on[kMaxDevices];
  std::atomic<bool>& configured = configured_on[current_device()];
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    configured.store(true, std::memory_order_release);
  }
  const unsigned gx = SPLIT ? (unsigned)a.vnode_count : (unsigned)((a.vnode_count + kWavesPerBlock - 1) / kWavesPerBlock);
  hipLaunchKernelGGL(kern, dim3(gx, (unsigned)hkv, 1), dim3(kBlock, 1, 1), lds, stream, a);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

// Waves that share one narrow vnode: the largest power of two (at most a block's four) that
// fills at most three quarters of the wave slots (8 per compute unit).  With far fewer vnodes than slots the
// waves would each walk a long run alone, one memory round trip per tile; with the slots nearly
// full the runs are limited by memory bandwidth already and sharing only adds barriers.
inline int wave_slots() {
  // per device; threads that race on the first call compute and store the same value
  static std::atomic<int> slots_on[kMaxDevices];
  std::atomic<int>& slots = slots_on[current_device()];
  int n = slots.load(std::memory_order_relaxed);
  if (n == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) {
      (void)hipGetLastError();
      cus = 256;
    }
    n = cus * kWaveSlotsPerCu;
    slots.store(n, std::memory_order_relaxed);
  }
  return n;
}
inline int narrow_share_for(int64_t items, int head_dim) {
  const int slots = head_dim > 128 ? wave_slots() / 2 : wave_slots();   // (one block per compute unit at 512-byte rows)
  int share = 1;
  while (share < kWideWaves && 4 * items * (2 * share) <= 3 * (int64_t)slots) share *= 2;
  return share;
}

template <typename E, int D, bool GATHERED, int MODE>
int launch_stage1_fused(const Stage1Args& a0, hipStream_t stream) {
  constexpr size_t kWideLds = (size_t)WideGeom<D>::kLds;
  constexpr size_t kNarrowLds = (size_t)kWideWaves * NarrowGeom<D>::kLds;
  constexpr size_t lds = kWideLds > kNarrowLds ? kWideLds : kNarrowLds;
  void (*kern)(FT_FIRST_PARAMETERS, Stage1Args) = nullptr;
  if constexpr (MODE == kEmbedding) kern = stage1_embedding_kernel<E, D>;
  else if constexpr (MODE == kServing) kern = stage1_serving_kernel<E, D>;
  else kern = stage1_fused_kernel<E, D, GATHERED, MODE == kPrograms>;
  // (raising the dynamic LDS limit is idempotent: two threads that both find the flag clear both raise it)
  static std::atomic<bool> configured_on[kMaxDevices];
  std::atomic<bool>& configured = configured_on[current_device()];
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    configured.store(true, std::memory_order_release);
  }
  Stage1Args a = a0;
  const int64_t narrow_items = (int64_t)(a.narrow_count - a.narrow_in_programs) * a.hkv;  // those of the trailing blocks
  a.narrow_share = narrow_share_for(narrow_items, D);
  const int per_block = kWideWaves / a.narrow_share;
  const int64_t narrow_blocks = (narrow_items + per_block - 1) / per_block;
  a.wide_chunks = std::max(1, std::min(8, (a.wide_rows + WideRows<D>::kBlock - 1) / WideRows<D>::kBlock));
  a.by_chunks = divisor(a.wide_chunks);
  a.block_slots = (D > 128 ? wave_slots() / 2 : wave_slots()) / kWideWaves;
  // Vnodes of one run are joined to full blocks only where that leaves a block per compute unit: 11 query
  // tiles of 64 rows over three 1024-token splits and 8 KV heads take 46.7 us as 96 blocks of 192 rows and
  // 38.4 as 144 of 128.
  a.join_rows = WideRows<D>::kBlock;
  if (a.wide_chunks == 1 && (int64_t)a.vnode_count * a.hkv * a.wide_rows < (int64_t)a.join_rows * (wave_slots() / kWaveSlotsPerCu))
    a.join_rows = std::min(a.join_rows, 128);
  const int64_t wide_blocks = MODE != kLists ? (int64_t)a.num_programs * a.hkv : (int64_t)a.vnode_count * a.wide_chunks * a.hkv;
  const int64_t blocks = wide_blocks + narrow_blocks;
  if (blocks == 0) return FT_OK;
  if (blocks > INT32_MAX) return FT_ERR_ARGUMENT;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, 1), dim3(kWideBlock, 1, 1), lds, stream, a.prog_table, a.prog_records, a.narrow_table,
                     (int)wide_blocks, a.hkv, a.by_hkv.mul, a.by_hkv.shift, a.narrow_share, a.narrow_count * a.hkv, a);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

template <typename E, int D, bool GATHERED>
int launch_stage1_narrow(const Stage1Args& a0, hipStream_t stream) {
  Stage1Args a = a0;
  const int64_t blocks = (int64_t)a.narrow_count * a.hkv;
  if (blocks == 0) return FT_OK;
  if (blocks > INT32_MAX) return FT_ERR_ARGUMENT;
  a.narrow_share = narrow_share_for(blocks, D);
  auto kern = stage1_narrow_kernel<E, D, GATHERED>;
  const size_t lds = (size_t)a.narrow_share * NarrowGeom<D>::kLds;
  // (raising the dynamic LDS limit is idempotent: two threads that both find the flag clear both raise it)
  static std::atomic<bool> configured_on[kMaxDevices];
  std::atomic<bool>& configured = configured_on[current_device()];
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            kWideWaves * NarrowGeom<D>::kLds) != hipSuccess) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    configured.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, 1), dim3(kWave * a.narrow_share, 1, 1), lds, stream, a.narrow_table, a.hkv, a.by_hkv.mul,
                     a.by_hkv.shift, a);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

template <typename E, int D>
int launch_stage1_paths_d(const PathArgs& d, const int32_t* wave_records, hipStream_t stream) {
  const int64_t blocks = (int64_t)d.s.narrow_count * d.s.hkv;
  if (blocks == 0) return FT_OK;
  if (blocks > INT32_MAX) return FT_ERR_ARGUMENT;
  auto kern = stage1_paths_kernel<E, D>;
  constexpr size_t lds = (size_t)kPathWaves<D> * NarrowGeom<D>::kLds;
  // (raising the dynamic LDS limit is idempotent: two threads that both find the flag clear both raise it)
  static std::atomic<bool> configured_on[kMaxDevices];
  std::atomic<bool>& configured = configured_on[current_device()];
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    configured.store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, 1), dim3(kWave * kPathWaves<D>, 1, 1), lds, stream, wave_records, d.s.hkv,
                     d.s.by_hkv.mul, d.s.by_hkv.shift, d);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}
int launch_stage1_paths(const PathArgs& a, const int32_t* wave_records, int head_dim, int dtype, hipStream_t stream) {
#define FT_DISPATCH_D(E)                                         \
  switch (head_dim) {                                            \
    case 32: return launch_stage1_paths_d<E, 32>(a, wave_records, stream);     \
    case 64: return launch_stage1_paths_d<E, 64>(a, wave_records, stream);     \
    case 128: return launch_stage1_paths_d<E, 128>(a, wave_records, stream);   \
    case 256: return launch_stage1_paths_d<E, 256>(a, wave_records, stream);   \
    default: return FT_ERR_HEAD_DIM;                             \
  }
  if (dtype == FT_DTYPE_F16) { FT_DISPATCH_D(F16) }
  if (dtype == FT_DTYPE_BF16) { FT_DISPATCH_D(BF16) }
#undef FT_DISPATCH_D
  return FT_ERR_DTYPE;
}

// `a` names two vnode ranges: [vnode_begin, +vnode_count) of wide vnodes (more than 16 query
// rows) and [narrow_begin, +narrow_count) of narrow ones.
template <typename E, int D, bool GATHERED, bool STAGED = false>
int launch_stage1_d(const Stage1Args& a, hipStream_t stream) {
  if constexpr (STAGED) {
    // head_dim 16: rows half as long as a 32-dim contraction's, padded with zeros on their way through registers
    if (a.vnode_count > 0)
      if (int rc = launch_stage1_inst<E, D, 2, true, GATHERED>(a, a.hkv, stream)) return rc;
    if (a.narrow_count > 0) {
      Stage1Args n = a;
      n.vnode_begin = a.narrow_begin;
      n.vnode_count = a.narrow_count;
      return launch_stage1_inst<E, D, 1, false, GATHERED>(n, a.hkv, stream);
    }
    return FT_OK;
  } else {
    if (a.vnode_count == 0 && !a.prog_table) return launch_stage1_narrow<E, D, GATHERED>(a, stream);
    if constexpr (!GATHERED) {
      if (a.prog_table && a.narrow_in_programs > 0) return launch_stage1_fused<E, D, false, kEmbedding>(a, stream);
      if (a.prog_table && !a.narrow_table) return launch_stage1_fused<E, D, false, kServing>(a, stream);
      if (a.prog_table) return launch_stage1_fused<E, D, false, kPrograms>(a, stream);
    }
    return launch_stage1_fused<E, D, GATHERED, kLists>(a, stream);
  }
}

template <bool GATHERED>
int launch_stage1(const Stage1Args& a, int d, int dtype, hipStream_t stream) {
#define FT_DISPATCH_D(E)                                              \
  switch (d) {                                                        \
    case 16: return launch_stage1_d<E, 32, GATHERED, true>(a, stream);\
    case 32: return launch_stage1_d<E, 32, GATHERED>(a, stream);      \
    case 64: return launch_stage1_d<E, 64, GATHERED>(a, stream);      \
    case 128: return launch_stage1_d<E, 128, GATHERED>(a, stream);    \
    case 256: return launch_stage1_d<E, 256, GATHERED>(a, stream);    \
    default: return FT_ERR_HEAD_DIM;                                  \
  }
  if (dtype == FT_DTYPE_F16) { FT_DISPATCH_D(F16) }
  if (dtype == FT_DTYPE_BF16) { FT_DISPATCH_D(BF16) }
#undef FT_DISPATCH_D
  return FT_ERR_DTYPE;
}

// Waves per list: as many as leave the launch at most two blocks per compute unit (wave_slots() / 4): more blocks than
// that hide each other's round trips anyway.  One wave, and the kernel without the merge, where every list is short or
// the batch fills the machine by itself.
// Lane groups per list of more than kLongList entries by the same rule, where that makes more parts than four waves do (warm, the
// merge alone, four waves and lane groups; 512 entries: one request of 32 heads of 128 16.5 and 7.3 us, of 64 heads of 64 16.6 and
// 6.8, of 16 heads of 256 18.6 and 10.9; 128 entries 5.8 and 4.1, 5.8 and 4.1, 6.2 and 4.7; 65 entries 4.9 and 4.2, 4.9 and 4.7,
// 5.2 and 4.2).  In four parts, or eight of 32 dims, waves read more of a row at once (64 requests of 24 heads of 64 with 512
// entries: 38.6 and 41.5; of 32 heads of 32: 28.4 and 30.2); 512-byte rows are a wave's in either case.
template <typename E, int D>
int launch_stage2_inst(const Stage2Args& a0, hipStream_t stream) {
  constexpr int kHeads = kWavesPerBlock * MergeGeom<D>::kHeads;   // of a block whose waves share no list
  constexpr int kLaneGroups = kBlock / (D / 4);                   // of a block, for long lists
  Stage2Args a = a0;
  auto blocks_per_request = [&](int per_block, int log_parts) { return ((int64_t)(a.hq << log_parts) + per_block - 1) / per_block; };
  auto room = [&](int per_block, int log_parts) { return a.batch * blocks_per_request(per_block, log_parts) <= wave_slots() / 4; };
  a.log_splits = 0;
  while (a.longest > kOneWave && (1 << a.log_splits) < kWavesPerBlock && room(kHeads, a.log_splits + 1)) ++a.log_splits;
  a.log_groups = 0;
  while (a.longest > kLongList && (1 << a.log_groups) < kLaneGroups && room(kLaneGroups, a.log_groups + 1)) ++a.log_groups;
  constexpr int kLeast = D <= 32 ? 16 : D <= 128 ? 8 : 4;
  if ((1 << a.log_groups) < kLeast) a.log_groups = 0;
  const dim3 grid((unsigned)a.batch, (unsigned)std::max(blocks_per_request(kHeads, a.log_splits), a.log_groups ? blocks_per_request(kLaneGroups, a.log_groups) : 0), 1);
  const int32_t* records = a.nsplit > 0 ? nullptr : a.req_table;
  if (a.log_groups > 0) hipLaunchKernelGGL((stage2_kernel<E, D, kLongLists>), grid, dim3(kBlock, 1, 1), 0, stream, records, a);
  else if (a.log_splits > 0) hipLaunchKernelGGL((stage2_kernel<E, D, kSplitLists>), grid, dim3(kBlock, 1, 1), 0, stream, records, a);
  else hipLaunchKernelGGL((stage2_kernel<E, D, kWholeLists>), grid, dim3(kBlock, 1, 1), 0, stream, records, a);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

int launch_stage2(const Stage2Args& a, int d, int dtype, hipStream_t stream) {
#define FT_DISPATCH_D(E)                                       \
  switch (d) {                                                 \
    case 16: return launch_stage2_inst<E, 16>(a, stream);      \
    case 32: return launch_stage2_inst<E, 32>(a, stream);      \
    case 64: return launch_stage2_inst<E, 64>(a, stream);      \
    case 128: return launch_stage2_inst<E, 128>(a, stream);    \
    case 256: return launch_stage2_inst<E, 256>(a, stream);    \
    default: return FT_ERR_HEAD_DIM;                           \
  }
  if (dtype == FT_DTYPE_F16) { FT_DISPATCH_D(F16) }
  if (dtype == FT_DTYPE_BF16) { FT_DISPATCH_D(BF16) }
#undef FT_DISPATCH_D
  return FT_ERR_DTYPE;
}

template <typename E, int D>
int launch_deft_inst(const DeftArgs& d, hipStream_t stream) {
  constexpr size_t lds = (size_t)WideGeom<D>::kRing + kDeftMaskGroups * kDeftChunk * 8;   // two super tiles and the mask words
  auto kern = deft_stage1_kernel<E, D>;
  static std::atomic<bool> configured_on[kMaxDevices];
  std::atomic<bool>& configured = configured_on[current_device()];
  if (!configured.load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    configured.store(true, std::memory_order_release);
  }
  const int64_t blocks = (int64_t)d.num_subtrees * d.s.hkv;
  if (blocks == 0) return FT_OK;
  if (blocks > INT32_MAX) return FT_ERR_ARGUMENT;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks, 1, 1), dim3(kWideBlock, 1, 1), lds, stream, d);
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

int launch_deft(const DeftArgs& d, int head_dim, int dtype, hipStream_t stream) {
#define FT_DISPATCH_D(E)                                         \
  switch (head_dim) {                                            \
    case 32: return launch_deft_inst<E, 32>(d, stream);          \
    case 64: return launch_deft_inst<E, 64>(d, stream);          \
    case 128: return launch_deft_inst<E, 128>(d, stream);        \
    case 256: return launch_deft_inst<E, 256>(d, stream);        \
    default: return FT_ERR_HEAD_DIM;                             \
  }
  if (dtype == FT_DTYPE_F16) { FT_DISPATCH_D(F16) }
  if (dtype == FT_DTYPE_BF16) { FT_DISPATCH_D(BF16) }
#undef FT_DISPATCH_D
  return FT_ERR_DTYPE;
}

int check_common(int d, int g, int dtype) {
  if (dtype != FT_DTYPE_F16 && dtype != FT_DTYPE_BF16) return FT_ERR_DTYPE;
  if (d != 16 && d != 32 && d != 64 && d != 128 && d != 256) return FT_ERR_HEAD_DIM;
  if (g < 1 || g > 64) return FT_ERR_GROUP;
  return FT_OK;
}

}  // namespace

// ---------------------------------------------------------------------------------------
// Scratch of ft_decode_static: the partial results of one decode call (mid_o, then mid_lse) in
// a device array of the library, for callers that cannot allocate.  Every device the library
// runs on holds its own copy until the process ends.  In host code the array's name is a
// stand-in, not a device address: the address on the current device is asked for once per
// device and kept, and only that pointer is handed to kernels.
// ---------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[FT_STATIC_SCRATCH_BYTES];

static int static_scratch_of_current_device(char** out) {
  constexpr int kMaxDevices = 64;
  // No lock: the lookup gives every thread the same address for a device, so threads that race on
  // a device's first call store the same pointer, and later calls are one atomic load.
  static std::atomic<char*> address[kMaxDevices];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return FT_ERR_LAUNCH;
  }
  char* ptr = address[dev].load(std::memory_order_acquire);
  if (!ptr) {
    if (hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
      (void)hipGetLastError();
      return FT_ERR_LAUNCH;
    }
    address[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return FT_OK;
}

extern "C" {

const char* ft_version(void) { return "fasttree_hip 0.1 (gfx950)"; }

int64_t ft_static_scratch_bytes(void) { return (int64_t)FT_STATIC_SCRATCH_BYTES; }

const char* ft_error_string(int code) {
  switch (code) {
    case FT_OK: return "ok";
    case FT_ERR_NULL_POINTER: return "null pointer argument";
    case FT_ERR_DTYPE: return "unsupported dtype (fp16 and bf16 only)";
    case FT_ERR_HEAD_DIM: return "unsupported head dimension (16, 32, 64, 128, 256)";
    case FT_ERR_GROUP: return "unsupported query/KV head ratio";
    case FT_ERR_ALIGNMENT: return "pointer or stride not aligned as required";
    case FT_ERR_ARGUMENT: return "argument out of range";
    case FT_ERR_LAUNCH: return "kernel launch failed";
    case FT_ERR_SCRATCH: return "partial results do not fit the library's static scratch (FT_STATIC_SCRATCH_BYTES)";
    default: return "unknown error";
  }
}

// Validates the stage-1 arguments shared by ft_stage1 and ft_decode and fills everything of
// `a` but the vnode ranges.
static int stage1_setup(Stage1Args& a, const void* q, const void* k, const void* v,
                        int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                        const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                        const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                        const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                        int num_kv_heads, int kv_group_num, int head_dim, float sm_scale,
                        float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0, int dtype) {
  if (int rc = check_common(head_dim, kv_group_num, dtype)) return rc;
  if (!q || !k || !v || !vnode_to_kv_entries || !vnode_to_kv_offs || !vnode_to_kv_lens || !vnode_to_q_entries ||
      !vnode_to_q_offs || !vnode_to_q_lens || !mid_o || !mid_lse)
    return FT_ERR_NULL_POINTER;
  if (num_kv_heads < 1 || num_kv_heads > 65535 || !(sm_scale > 0.f)) return FT_ERR_ARGUMENT;
  // the kernels form row addresses as slot * (32-bit byte stride)
  if (sk0 < 0 || sv0 < 0 || sk0 >= (int64_t(1) << 31) || sv0 >= (int64_t(1) << 31)) return FT_ERR_ARGUMENT;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(mid_o) || (sq0 | sq1 | sk0 | sk1 | sv0 | sv1) % 8 != 0 ||
      (so0 | so1) % 4 != 0)
    return FT_ERR_ALIGNMENT;
  a = Stage1Args{};
  a.q = static_cast<const char*>(q);
  a.k = static_cast<const char*>(k);
  a.v = static_cast<const char*>(v);
  a.sq0 = sq0; a.sq1 = sq1; a.sk0 = sk0; a.sk1 = sk1; a.sv0 = sv0; a.sv1 = sv1;
  a.kv_entries = vnode_to_kv_entries; a.kv_offs = vnode_to_kv_offs; a.kv_lens = vnode_to_kv_lens;
  a.q_entries = vnode_to_q_entries; a.q_offs = vnode_to_q_offs; a.q_lens = vnode_to_q_lens;
  a.g = kv_group_num;
  a.hkv = num_kv_heads;
  a.by_g = divisor(a.g);
  a.by_hkv = divisor(a.hkv);
  a.real_dim = head_dim;
  a.scale_log2 = sm_scale * kLog2e;
  a.mid_o = mid_o; a.so0 = so0; a.so1 = so1; a.mid_lse = mid_lse; a.sl0 = sl0;
  return FT_OK;
}

// A phase whose tile holds at most 16 query rows is served one wave per (vnode, KV head).
static bool is_narrow(int q_tile, int kv_group_num) { return (int64_t)q_tile * kv_group_num <= 16; }

static bool range_ok(int begin, int count, int num_kv_heads) {
  return begin >= 0 && count >= 0 && (int64_t)count * num_kv_heads <= INT32_MAX;
}

int ft_stage1(const void* q, const void* k, const void* v,
              int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
              const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
              const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
              const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
              int vnode_begin, int vnode_count, int num_kv_heads, int kv_group_num, int head_dim,
              int q_tile, int kv_tile, float sm_scale,
              float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
              int dtype, ft_stream_t stream) {
  (void)kv_tile;
  if (int rc = check_common(head_dim, kv_group_num, dtype)) return rc;
  if (vnode_count == 0) return FT_OK;
  Stage1Args a;
  if (int rc = stage1_setup(a, q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                            vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, num_kv_heads,
                            kv_group_num, head_dim, sm_scale, mid_o, so0, so1, mid_lse, sl0, dtype))
    return rc;
  if (q_tile < 1 || !range_ok(vnode_begin, vnode_count, num_kv_heads)) return FT_ERR_ARGUMENT;
  if (is_narrow(q_tile, kv_group_num)) {
    a.narrow_begin = vnode_begin; a.narrow_count = vnode_count;
  } else {
    a.vnode_begin = vnode_begin; a.vnode_count = vnode_count;
    a.wide_rows = (int)std::min<int64_t>((int64_t)q_tile * kv_group_num, 1 << 20);
  }
  return launch_stage1<false>(a, head_dim, dtype, stream);
}

static int stage2_with_table(const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
                             const int32_t* req_to_vnode_lens, const int32_t* req_table,
                             const float* mid_o, int64_t so0, int64_t so1, const float* mid_lse, int64_t sl0,
                             void* o, int64_t oo0, int64_t oo1,
                             int64_t num_vnodes, int batch_size, int num_qo_heads, int head_dim, int dtype, ft_stream_t stream) {
  if (int rc = check_common(head_dim, 1, dtype)) return rc;
  if (batch_size == 0) return FT_OK;
  if (!req_to_vnode_entries || !req_to_vnode_offs || !req_to_vnode_lens || !mid_o || !mid_lse || !o)
    return FT_ERR_NULL_POINTER;
  if (batch_size < 0 || num_qo_heads < 1) return FT_ERR_ARGUMENT;
  if (!aligned16(mid_o) || !aligned16(o) || (so0 | so1) % 4 != 0 || (oo0 | oo1) % 4 != 0) return FT_ERR_ALIGNMENT;
  Stage2Args a{};
  a.req_entries = req_to_vnode_entries; a.req_offs = req_to_vnode_offs; a.req_lens = req_to_vnode_lens;
  a.mid_o = mid_o; a.so0 = so0; a.so1 = so1; a.mid_lse = mid_lse; a.sl0 = sl0;
  a.o = static_cast<char*>(o); a.oo0 = oo0; a.oo1 = oo1;
  a.batch = batch_size; a.hq = num_qo_heads; a.nsplit = 0;
  a.longest = (int)std::min<int64_t>(num_vnodes, INT32_MAX);
  a.req_table = req_table;
  return launch_stage2(a, head_dim, dtype, stream);
}

int ft_stage2(const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
              const int32_t* req_to_vnode_lens,
              const float* mid_o, int64_t so0, int64_t so1, const float* mid_lse, int64_t sl0,
              void* o, int64_t oo0, int64_t oo1,
              int batch_size, int num_qo_heads, int head_dim, int dtype, ft_stream_t stream) {
  return stage2_with_table(req_to_vnode_entries, req_to_vnode_offs, req_to_vnode_lens, nullptr, mid_o, so0, so1, mid_lse,
                           sl0, o, oo0, oo1, INT32_MAX, batch_size, num_qo_heads, head_dim, dtype, stream);
}

int ft_stage1_phases(const void* q, const void* k, const void* v,
                     int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                     const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                     const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                     const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                     float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
                     const int32_t phase_node_nums[2], const int32_t phase_node_offsets[2],
                     const int32_t phase_q_tile_sizes[2], const int32_t phase_kv_tile_sizes[2],
                     int num_qo_heads, int num_kv_heads, int head_dim,
                     float sm_scale, int dtype, ft_stream_t stream) {
  if (!phase_node_nums || !phase_node_offsets || !phase_q_tile_sizes || !phase_kv_tile_sizes) return FT_ERR_NULL_POINTER;
  if (num_kv_heads < 1 || num_qo_heads % num_kv_heads != 0) return FT_ERR_GROUP;
  const int g = num_qo_heads / num_kv_heads;
  if (int rc = check_common(head_dim, g, dtype)) return rc;
  if (phase_node_nums[0] == 0 && phase_node_nums[1] == 0) return FT_OK;
  Stage1Args a;
  if (int rc = stage1_setup(a, q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                            vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, num_kv_heads, g,
                            head_dim, sm_scale, mid_o, so0, so1, mid_lse, sl0, dtype))
    return rc;
  const bool pending[2] = {phase_node_nums[0] != 0, phase_node_nums[1] != 0};
  for (int phase = 0; phase < 2; ++phase)
    if (pending[phase] && (phase_q_tile_sizes[phase] < 1 ||
                           !range_ok(phase_node_offsets[phase], phase_node_nums[phase], num_kv_heads)))
      return FT_ERR_ARGUMENT;
  const bool narrow[2] = {is_narrow(phase_q_tile_sizes[0], g), is_narrow(phase_q_tile_sizes[1], g)};
  auto assign = [](Stage1Args& t, bool is_narrow_range, int begin, int count) {
    if (is_narrow_range) { t.narrow_begin = begin; t.narrow_count = count; }
    else { t.vnode_begin = begin; t.vnode_count = count; }
  };
  const int64_t widest_tile = std::max(narrow[0] ? 0 : phase_q_tile_sizes[0], narrow[1] ? 0 : phase_q_tile_sizes[1]);
  a.wide_rows = (int)std::min<int64_t>(widest_tile * g, 1 << 20);
  // Both phases go into one launch when one is wide and the other narrow, or when they are of
  // the same kind and adjacent in the vnode list (the planner's lists always are).
  if (pending[0] && pending[1] && narrow[0] == narrow[1]) {
    if (phase_node_offsets[0] + phase_node_nums[0] == phase_node_offsets[1] &&
        range_ok(phase_node_offsets[0], phase_node_nums[0] + phase_node_nums[1], num_kv_heads)) {
      assign(a, narrow[0], phase_node_offsets[0], phase_node_nums[0] + phase_node_nums[1]);
      return launch_stage1<false>(a, head_dim, dtype, stream);
    }
    for (int phase = 0; phase < 2; ++phase) {
      Stage1Args b = a;
      assign(b, narrow[phase], phase_node_offsets[phase], phase_node_nums[phase]);
      if (int rc = launch_stage1<false>(b, head_dim, dtype, stream)) return rc;
    }
    return FT_OK;
  }
  for (int phase = 0; phase < 2; ++phase)
    if (pending[phase]) assign(a, narrow[phase], phase_node_offsets[phase], phase_node_nums[phase]);
  return launch_stage1<false>(a, head_dim, dtype, stream);
}

int ft_stage1_programs(const void* q, const void* k, const void* v,
                       int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                       const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                       const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                       const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                       float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
                       const int32_t phase_node_nums[2], const int32_t phase_node_offsets[2],
                       const int32_t* prog_table, int num_programs, int narrow_in_programs,
                       const int32_t* narrow_table, const int32_t* prog_records,
                       int num_qo_heads, int num_kv_heads, int head_dim,
                       float sm_scale, int dtype, ft_stream_t stream) {
  if (!phase_node_nums || !phase_node_offsets) return FT_ERR_NULL_POINTER;
  if (num_kv_heads < 1 || num_qo_heads % num_kv_heads != 0) return FT_ERR_GROUP;
  const int g = num_qo_heads / num_kv_heads;
  if (int rc = check_common(head_dim, g, dtype)) return rc;
  if (head_dim < 32) return FT_ERR_HEAD_DIM;  // the program table is for the direct-load kernels
  if (phase_node_nums[0] == 0 && phase_node_nums[1] == 0) return FT_OK;
  Stage1Args a;
  if (int rc = stage1_setup(a, q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                            vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, num_kv_heads, g,
                            head_dim, sm_scale, mid_o, so0, so1, mid_lse, sl0, dtype))
    return rc;
  for (int phase = 0; phase < 2; ++phase)
    if (!range_ok(phase_node_offsets[phase], phase_node_nums[phase], num_kv_heads)) return FT_ERR_ARGUMENT;
  if (num_programs < 0 || (int64_t)num_programs * num_kv_heads > INT32_MAX) return FT_ERR_ARGUMENT;
  if (num_programs > 0 && !prog_table) return FT_ERR_NULL_POINTER;
  if (narrow_in_programs < 0 || narrow_in_programs > phase_node_nums[1]) return FT_ERR_ARGUMENT;
  if (num_programs == 0 && (phase_node_nums[0] > 0 || narrow_in_programs > 0)) return FT_ERR_ARGUMENT;
  a.vnode_begin = phase_node_offsets[0]; a.vnode_count = phase_node_nums[0];
  a.narrow_begin = phase_node_offsets[1]; a.narrow_count = phase_node_nums[1];
  if (num_programs > 0) { a.prog_table = prog_table; a.num_programs = num_programs; a.narrow_in_programs = narrow_in_programs; }
  a.narrow_table = narrow_table;
  a.prog_records = num_programs > 0 ? prog_records : nullptr;
  a.wide_rows = 1;   // (a program's block serves all row pieces of its vnodes)
  return launch_stage1<false>(a, head_dim, dtype, stream);
}

int ft_decode_programs(const void* q, const void* k, const void* v, void* o,
                       int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                       int64_t oo0, int64_t oo1,
                       const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                       const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                       const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                       const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
                       const int32_t* req_to_vnode_lens,
                       float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
                       const int32_t phase_node_nums[2], const int32_t phase_node_offsets[2],
                       const int32_t* prog_table, int num_programs, int narrow_in_programs,
                       const int32_t* narrow_table, const int32_t* prog_records, const int32_t* req_table,
                       int batch_size, int num_qo_heads, int num_kv_heads, int head_dim,
                       float sm_scale, int dtype, ft_stream_t stream) {
  if (narrow_in_programs == FT_WHOLE_PATHS) {
    // (checked as the two launches would be)
    if (!phase_node_nums || !phase_node_offsets) return FT_ERR_NULL_POINTER;
    if (num_kv_heads < 1 || num_qo_heads % num_kv_heads != 0) return FT_ERR_GROUP;
    const int g = num_qo_heads / num_kv_heads;
    if (int rc = check_common(head_dim, g, dtype)) return rc;
    if (head_dim < 32) return FT_ERR_HEAD_DIM;
    if (phase_node_nums[0] != 0 || num_programs != 0 || batch_size < 0 || num_qo_heads < 1) return FT_ERR_ARGUMENT;
    if (phase_node_nums[1] == 0 || batch_size == 0) return FT_OK;
    PathArgs d{};
    if (int rc = stage1_setup(d.s, q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                              vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, num_kv_heads, g,
                              head_dim, sm_scale, mid_o, so0, so1, mid_lse, sl0, dtype))
      return rc;
    if (!prog_records || !req_to_vnode_entries || !req_to_vnode_offs || !req_to_vnode_lens || !o) return FT_ERR_NULL_POINTER;
    if (!range_ok(phase_node_offsets[1], phase_node_nums[1], num_kv_heads)) return FT_ERR_ARGUMENT;
    if (!aligned16(o) || (oo0 | oo1) % 4 != 0) return FT_ERR_ALIGNMENT;
    d.s.narrow_begin = phase_node_offsets[1]; d.s.narrow_count = phase_node_nums[1];
    d.o = static_cast<char*>(o); d.oo0 = oo0; d.oo1 = oo1;
    return launch_stage1_paths(d, prog_records, head_dim, dtype, stream);
  }
  if (int rc = ft_stage1_programs(q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                                  vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, mid_o, so0,
                                  so1, mid_lse, sl0, phase_node_nums, phase_node_offsets, prog_table, num_programs,
                                  narrow_in_programs, narrow_table, prog_records, num_qo_heads, num_kv_heads, head_dim,
                                  sm_scale, dtype, stream))
    return rc;
  return stage2_with_table(req_to_vnode_entries, req_to_vnode_offs, req_to_vnode_lens, req_table, mid_o, so0, so1,
                           mid_lse, sl0, o, oo0, oo1, (int64_t)phase_node_nums[0] + phase_node_nums[1], batch_size, num_qo_heads, head_dim, dtype,
                           stream);
}

int ft_decode_static(const void* q, const void* k, const void* v, void* o,
                     int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                     int64_t oo0, int64_t oo1,
                     const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                     const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                     const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                     const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
                     const int32_t* req_to_vnode_lens, int64_t num_rows,
                     const int32_t phase_node_nums[2], const int32_t phase_node_offsets[2],
                     const int32_t* prog_table, int num_programs, int narrow_in_programs,
                     const int32_t* narrow_table, const int32_t* prog_records, const int32_t* req_table,
                     int batch_size, int num_qo_heads, int num_kv_heads, int head_dim,
                     float sm_scale, int dtype, ft_stream_t stream) {
  if (num_rows < 0 || num_qo_heads < 1 || head_dim < 1) return FT_ERR_ARGUMENT;
  // mid_o: num_rows x num_qo_heads x head_dim floats, then (256-byte aligned) mid_lse: num_rows x num_qo_heads
  const unsigned __int128 o_bytes = (unsigned __int128)num_rows * (unsigned)num_qo_heads * (unsigned)head_dim * 4u;
  const unsigned __int128 lse_at = (o_bytes + 255u) / 256u * 256u;
  const unsigned __int128 need = lse_at + (unsigned __int128)num_rows * (unsigned)num_qo_heads * 4u;
  if (need > (unsigned __int128)FT_STATIC_SCRATCH_BYTES) return FT_ERR_SCRATCH;
  char* base = nullptr;
  if (int rc = static_scratch_of_current_device(&base)) return rc;
  float* mid_o = reinterpret_cast<float*>(base);
  float* mid_lse = reinterpret_cast<float*>(base + (size_t)lse_at);
  return ft_decode_programs(q, k, v, o, sq0, sq1, sk0, sk1, sv0, sv1, oo0, oo1, vnode_to_kv_entries, vnode_to_kv_offs,
                            vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, req_to_vnode_entries,
                            req_to_vnode_offs, req_to_vnode_lens, mid_o, (int64_t)num_qo_heads * head_dim, head_dim,
                            mid_lse, num_qo_heads, phase_node_nums, phase_node_offsets, prog_table, num_programs,
                            narrow_in_programs, narrow_table, prog_records, req_table, batch_size, num_qo_heads, num_kv_heads, head_dim,
                            sm_scale, dtype, stream);
}

int ft_decode(const void* q, const void* k, const void* v, void* o,
              int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
              int64_t oo0, int64_t oo1,
              const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
              const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
              const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
              const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
              const int32_t* req_to_vnode_lens,
              float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
              const int32_t phase_node_nums[2], const int32_t phase_node_offsets[2],
              const int32_t phase_q_tile_sizes[2], const int32_t phase_kv_tile_sizes[2],
              int batch_size, int num_qo_heads, int num_kv_heads, int head_dim,
              float sm_scale, int dtype, ft_stream_t stream) {
  if (int rc = ft_stage1_phases(q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                                vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, mid_o, so0, so1,
                                mid_lse, sl0, phase_node_nums, phase_node_offsets, phase_q_tile_sizes,
                                phase_kv_tile_sizes, num_qo_heads, num_kv_heads, head_dim, sm_scale, dtype, stream))
    return rc;
  return stage2_with_table(req_to_vnode_entries, req_to_vnode_offs, req_to_vnode_lens, nullptr, mid_o, so0, so1, mid_lse, sl0, o,
                           oo0, oo1, (int64_t)phase_node_nums[0] + phase_node_nums[1], batch_size, num_qo_heads, head_dim, dtype, stream);
}

int ft_deft_stage1(const void* q, const void* k, const void* v,
                   int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                   const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                   const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                   const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                   const int64_t* causalmask, const int32_t* causalmask_offset,
                   int subtree_num, int num_qo_heads, int num_kv_heads, int head_dim, int mask_len, float sm_scale,
                   float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
                   int dtype, ft_stream_t stream) {
  if (num_kv_heads < 1 || num_qo_heads % num_kv_heads != 0) return FT_ERR_GROUP;
  const int g = num_qo_heads / num_kv_heads;
  if (int rc = check_common(head_dim, g, dtype)) return rc;
  if (head_dim < 32) return FT_ERR_HEAD_DIM;
  if (subtree_num == 0) return FT_OK;
  DeftArgs d{};
  if (int rc = stage1_setup(d.s, q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                            vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, num_kv_heads, g,
                            head_dim, sm_scale, mid_o, so0, so1, mid_lse, sl0, dtype))
    return rc;
  if (!causalmask || !causalmask_offset) return FT_ERR_NULL_POINTER;
  if (subtree_num < 0 || !range_ok(0, subtree_num, num_kv_heads)) return FT_ERR_ARGUMENT;
  // a power of two of at most 64 requests per mask word, and few enough words per token for the
  // 128 query rows a block serves at a time
  if (mask_len < 1 || mask_len > 64 || (mask_len & (mask_len - 1)) != 0) return FT_ERR_ARGUMENT;
  const int requests_per_pass = (kDeftRows + g - 1) / g + 1;
  if ((requests_per_pass + mask_len - 1) / mask_len + 1 > kDeftMaskGroups) return FT_ERR_ARGUMENT;
  d.causalmask = causalmask;
  d.causalmask_offset = causalmask_offset;
  d.mask_len = mask_len;
  d.num_subtrees = subtree_num;
  return launch_deft(d, head_dim, dtype, stream);
}

int ft_deft_decode(const void* q, const void* k, const void* v, void* o,
                   int64_t sq0, int64_t sq1, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                   int64_t oo0, int64_t oo1,
                   const int32_t* vnode_to_kv_entries, const int32_t* vnode_to_kv_offs,
                   const int32_t* vnode_to_kv_lens, const int32_t* vnode_to_q_entries,
                   const int32_t* vnode_to_q_offs, const int32_t* vnode_to_q_lens,
                   const int64_t* causalmask, const int32_t* causalmask_offset,
                   const int32_t* req_to_vnode_entries, const int32_t* req_to_vnode_offs,
                   const int32_t* req_to_vnode_lens,
                   float* mid_o, int64_t so0, int64_t so1, float* mid_lse, int64_t sl0,
                   int subtree_num, int batch_size, int num_qo_heads, int num_kv_heads, int head_dim,
                   int mask_len, float sm_scale, int dtype, ft_stream_t stream) {
  if (int rc = ft_deft_stage1(q, k, v, sq0, sq1, sk0, sk1, sv0, sv1, vnode_to_kv_entries, vnode_to_kv_offs,
                              vnode_to_kv_lens, vnode_to_q_entries, vnode_to_q_offs, vnode_to_q_lens, causalmask,
                              causalmask_offset, subtree_num, num_qo_heads, num_kv_heads, head_dim, mask_len, sm_scale,
                              mid_o, so0, so1, mid_lse, sl0, dtype, stream))
    return rc;
  return ft_stage2(req_to_vnode_entries, req_to_vnode_offs, req_to_vnode_lens, mid_o, so0, so1, mid_lse, sl0, o, oo0,
                   oo1, batch_size, num_qo_heads, head_dim, dtype, stream);
}

int ft_gathered_decode(const void* q, const void* k_cache, const void* v_cache,
                       const int32_t* cache_seqlens, void* o,
                       int64_t sq0, int64_t sq1, int64_t oo0, int64_t oo1,
                       int batch_size, int max_seqlen, int num_qo_heads, int num_kv_heads,
                       int head_dim, int kv_split, float sm_scale,
                       float* mid_o, float* mid_lse, int dtype, ft_stream_t stream) {
  if (num_kv_heads < 1 || num_qo_heads % num_kv_heads != 0) return FT_ERR_GROUP;
  const int g = num_qo_heads / num_kv_heads;
  if (int rc = check_common(head_dim, g, dtype)) return rc;
  if (batch_size == 0) return FT_OK;
  if (!q || !k_cache || !v_cache || !cache_seqlens || !o || !mid_o || !mid_lse) return FT_ERR_NULL_POINTER;
  if (batch_size < 0 || max_seqlen < 1 || kv_split < 1 || num_kv_heads > 65535 || !(sm_scale > 0.f)) return FT_ERR_ARGUMENT;
  if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(mid_o) || !aligned16(o) ||
      (sq0 | sq1) % 8 != 0 || (oo0 | oo1) % 4 != 0)
    return FT_ERR_ALIGNMENT;
  const int nsplit = (max_seqlen + kv_split - 1) / kv_split;
  if ((int64_t)batch_size * nsplit > INT32_MAX) return FT_ERR_ARGUMENT;
  Stage1Args a{};
  a.q = static_cast<const char*>(q);
  a.k = static_cast<const char*>(k_cache);
  a.v = static_cast<const char*>(v_cache);
  a.sq0 = sq0; a.sq1 = sq1;
  a.sk0 = a.sv0 = (int64_t)num_kv_heads * head_dim;
  a.sk1 = a.sv1 = head_dim;
  if (is_narrow(1, g)) { a.narrow_begin = 0; a.narrow_count = batch_size * nsplit; }
  else { a.vnode_begin = 0; a.vnode_count = batch_size * nsplit; a.wide_rows = g; }
  a.g = g;
  a.hkv = num_kv_heads;
  a.by_g = divisor(a.g);
  a.by_hkv = divisor(a.hkv);
  a.real_dim = head_dim;
  a.scale_log2 = sm_scale * kLog2e;
  a.mid_o = mid_o; a.so0 = (int64_t)num_qo_heads * head_dim; a.so1 = head_dim;
  a.mid_lse = mid_lse; a.sl0 = num_qo_heads;
  a.cache_seqlens = cache_seqlens; a.max_seqlen = max_seqlen; a.kv_split = kv_split; a.nsplit = nsplit;
  if (int rc = launch_stage1<true>(a, head_dim, dtype, stream)) return rc;
  Stage2Args b{};
  b.mid_o = mid_o; b.so0 = a.so0; b.so1 = a.so1; b.mid_lse = mid_lse; b.sl0 = a.sl0;
  b.o = static_cast<char*>(o); b.oo0 = oo0; b.oo1 = oo1;
  b.batch = batch_size; b.hq = num_qo_heads; b.nsplit = nsplit; b.longest = nsplit;
  return launch_stage2(b, head_dim, dtype, stream);
}

int ft_store_kv(const void* k_new, const void* v_new, int64_t kn0, int64_t kn1, int64_t vn0, int64_t vn1,
                const void* out_cache_loc, int loc_is_int64, int num_tokens,
                void* k_pool, void* v_pool, int64_t sk0, int64_t sk1, int64_t sv0, int64_t sv1,
                int64_t num_slots, int num_kv_heads, int head_dim, int dtype, ft_stream_t stream) {
  if (dtype != FT_DTYPE_F16 && dtype != FT_DTYPE_BF16) return FT_ERR_DTYPE;
  if (head_dim < 8 || head_dim % 8 != 0 || head_dim > 1024) return FT_ERR_HEAD_DIM;
  if (num_tokens == 0) return FT_OK;
  if (!k_new || !v_new || !out_cache_loc || !k_pool || !v_pool) return FT_ERR_NULL_POINTER;
  if (num_tokens < 0 || num_kv_heads < 1 || num_kv_heads > 65535 || num_slots < 0) return FT_ERR_ARGUMENT;
  if (!aligned16(k_new) || !aligned16(v_new) || !aligned16(k_pool) || !aligned16(v_pool) ||
      (kn0 | kn1 | vn0 | vn1 | sk0 | sk1 | sv0 | sv1) % 8 != 0)
    return FT_ERR_ALIGNMENT;
  if (kn0 < 0 || kn1 < 0 || vn0 < 0 || vn1 < 0 || sk0 < 0 || sk1 < 0 || sv0 < 0 || sv1 < 0) return FT_ERR_ARGUMENT;
  StoreArgs a{};
  a.k_new = static_cast<const char*>(k_new); a.v_new = static_cast<const char*>(v_new);
  a.kn0 = kn0; a.kn1 = kn1; a.vn0 = vn0; a.vn1 = vn1;
  a.loc = out_cache_loc; a.loc_is_int64 = loc_is_int64 ? 1 : 0;
  a.k_pool = static_cast<char*>(k_pool); a.v_pool = static_cast<char*>(v_pool);
  a.sk0 = sk0; a.sk1 = sk1; a.sv0 = sv0; a.sv1 = sv1;
  a.num_slots = num_slots; a.hkv = num_kv_heads; a.chunks = head_dim / 8;
  a.by_chunks = divisor(a.chunks);
  const int pieces = num_kv_heads * a.chunks, threads = std::min(kStoreBlock, (pieces + kWave - 1) / kWave * kWave);
  if (pieces < kWave) {
    a.tokens = num_tokens;
    a.per_block = kStoreBlock / pieces;
    a.by_pieces = divisor(pieces);
    const int64_t blocks = ((int64_t)num_tokens + a.per_block - 1) / a.per_block;
    hipLaunchKernelGGL((store_kv_kernel<true>), dim3((unsigned)blocks, 1, 1), dim3(kStoreBlock, 1, 1), 0, stream, a);
  } else {
    hipLaunchKernelGGL((store_kv_kernel<false>), dim3((unsigned)num_tokens, (unsigned)((pieces + threads - 1) / threads), 1),
                       dim3((unsigned)threads, 1, 1), 0, stream, a);
  }
  return hipGetLastError() == hipSuccess ? FT_OK : FT_ERR_LAUNCH;
}

}  // extern "C"
