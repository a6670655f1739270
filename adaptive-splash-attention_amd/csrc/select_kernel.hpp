// Score pass: scores, exact per-row top-k and block mask (tau follows in
// tau_kernel, from the sorted top-k values this pass writes, or in
// tau_compact_kernel, which builds the CSR lists in the same launch).
//
// Reference: build_mask_kernel + insert_topk + entmax_threshold
// (adasplashattention.cu:35-217), one thread per query that scans every key
// and keeps a sorted top-k by insertion.  Here one block of 4 or 8 waves
// owns one 64-row query block of one (batch, head).  During the sweeps the
// waves split the keys, not the rows: a wave takes 16 keys of each of its
// visible key tiles, from per-wave LDS rings filled by global_load_lds
// (16-bit inputs at hd = D) or straight from L2 into MFMA operand registers
// (KQuarter, two tiles in flight), without a barrier per tile, and scores
// them against all 64 rows.  The top-k is found in two sweeps over the
// visible key blocks instead of by insertion:
//
//   sweep 1  every score updates one of 128 or 256 running "class maxima" of
//            its row (one v_med3 per score; class = key offset in the wave's
//            tile x tile ordinal mod R).  Distinct classes hold distinct
//            keys, so if at least k class maxima are >= x, at least k keys
//            score >= x, and every top-k key scores >= x.  The class maxima
//            meet in LDS and a bisection per row finds such an x close to
//            the k-th largest.
//   sweep 2  the scores are recomputed and every key scoring >= x is
//            appended, as (index, score bits), to the row's list in LDS
//            (about 1.05-1.15 k keys per row on random data).  If a row
//            overflows its list, the k-th best stored key becomes an exact
//            key threshold and the block sweeps again for those rows; each
//            round drops at least cap - k keys, so the rounds are bounded
//            (select_round_bound) and the status word reports them.
//   select   each row's candidates are sorted (segmented bitonic sort across
//            lanes, descending key order = score desc, index asc) when the
//            caller asked for top-k indices; otherwise only the values are
//            sorted and the top-k key set is the candidates above the k-th
//            value plus its lowest-index ties.  The first k values go to the
//            workspace for tau_kernel, padded with the empty slot (-1e6).
//   finish   the rows' top-k key blocks are OR-ed into a bitmap per 32-row
//            half of the block: the 64-row mask is their union, and with
//            32-row mask blocks each half's row is written as well.
//
// Sweep filters compare raw dot products (scale > 0) against a threshold
// widened by a relative margin, so that no key whose clamped, scaled score
// reaches the bound is missed; the exact score is only formed for the keys
// that pass.  With caller-given scores (asa_select_from_scores) or a
// non-positive scale the sweeps work on the exact scores directly.
//
// This header holds the score-pass kernel and its launch templates; each
// storage type is instantiated in a translation unit of its own
// (select_bf16.hip, select_f16.hip, select_f32.hip).
#pragma once

#include <climits>
#include <type_traits>

#include "asa_device.hpp"
#include "asa_launch.hpp"
#include "asa_stage.hpp"
#include "asa_tiles.hpp"

namespace asa {
namespace {


__device__ __forceinline__ int wave_min(int v) { return wave_reduce_minmax<false>(v); }
__device__ __forceinline__ int wave_max(int v) { return wave_reduce_minmax<true>(v); }
// Reductions over the NW lanes (4 or 8, equal modulo 64 / NW) that share a
// row of the floor search.
template <int NW, typename F>
__device__ __forceinline__ uint32_t row_reduce(uint32_t v, F op) {
  if constexpr (NW == 8) v = op(v, lane_xor<8>(v));
  return group_reduce_bits(v, op);
}
template <int NW>
__device__ __forceinline__ int row_sum(int v) {
  return int(row_reduce<NW>(uint32_t(v), [](uint32_t x, uint32_t y) { return x + y; }));
}
template <int NW>
__device__ __forceinline__ float row_min(float v) {
  return __uint_as_float(row_reduce<NW>(__float_as_uint(v), [](uint32_t x, uint32_t y) {
    return __float_as_uint(fminf(__uint_as_float(x), __uint_as_float(y)));
  }));
}
template <int NW>
__device__ __forceinline__ float row_max(float v) {
  return __uint_as_float(row_reduce<NW>(__float_as_uint(v), [](uint32_t x, uint32_t y) {
    return __float_as_uint(fmaxf(__uint_as_float(x), __uint_as_float(y)));
  }));
}
// max(m, x) for a running maximum m (never NaN) and an MFMA result x, in
// one v_med3_f32: med3(x, m, +inf) is the larger of x and m, and m when x
// is NaN (NaN loses).  `pinf` is +inf held in a register the compiler
// cannot see into (with a constant +inf it rewrites the med3 as fmaxf(),
// which canonicalises both operands first).  The MFMA results are only
// ever read by compiler-visible instructions, never by inline asm, so the
// compiler keeps the MFMA-to-VALU wait states it owes those reads.
__device__ __forceinline__ float vmax(float m, float x, float pinf) {
  return __builtin_amdgcn_fmed3f(x, m, pinf);
}
__device__ __forceinline__ float opaque_inf() {
  float v = __builtin_inff();
  asm("" : "+v"(v));
  return v;
}
// Smallest / largest of a 32-bit unsigned value over the wave.
template <bool kMax>
__device__ __forceinline__ uint32_t wave_minmax_u32(uint32_t v) {
  return uint32_t(wave_reduce_minmax<kMax>(int(v ^ 0x80000000u))) ^ 0x80000000u;
}
// c + (x >= t).
__device__ __forceinline__ uint32_t count_ge(uint32_t c, float x, float t) {
  return c + (x >= t ? 1u : 0u);
}
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x / 2); }

// Descending bitonic sort of independent segments of 8*LS keys: lanes
// [s*LS, (s+1)*LS) hold segment s, element e = (lane % LS) * 8 + p in v[p].
// Keys are distinct except for the padding value 0.  Exchanges between
// lanes use DPP moves for lane distances below 16.
template <int LS>
__device__ __forceinline__ void segment_sort_desc(uint64_t (&v)[8], int lane) {
  const int i = lane & (LS - 1);
  static_for<1, ilog2(8 * LS) + 1>([&](auto sc) {
    constexpr int size = 1 << decltype(sc)::value;
    static_for<0, decltype(sc)::value>([&](auto jc) {
      constexpr int j = (size >> 1) >> decltype(jc)::value;
      if constexpr (j >= 8) {
        const bool lower = (i & (j >> 3)) == 0;  // e & j depends on the lane only
        for (int p = 0; p < 8; ++p) {
          const int e = i * 8 + p;
          const uint64_t o = lane_xor64<(j >> 3)>(v[p]);
          const bool keep_max = ((e & size) == 0) == lower;
          const bool gt = v[p] > o;
          v[p] = (keep_max == gt) ? v[p] : o;
        }
      } else {
        for (int p = 0; p < 8; ++p) {
          const int pp = p ^ j;
          if (pp > p) {
            const bool desc = ((i * 8 + p) & size) == 0;
            const uint64_t a = v[p], b = v[pp];
            const bool sw = desc ? (a < b) : (a > b);
            v[p] = sw ? b : a;
            v[pp] = sw ? a : b;
          }
        }
      }
    });
  });
}

// Descending sort of independent segments of 8*LS 32-bit values, no
// payload: lanes [s*LS, (s+1)*LS) hold segment s, element e = (lane % LS) * 8
// + p in v[p].  Bitonic network in the form where every comparator puts the
// larger value first: the first step of each merge compares e with its
// mirror e ^ (size - 1), the later steps e with e ^ j.  One max and one min
// per in-lane pair; a lane move, max or min and a select per element across
// lanes.
template <int LS>
__device__ __forceinline__ void segment_sort_desc32(uint32_t (&v)[8], int lane) {
  const int i = lane & (LS - 1);
  static_for<1, ilog2(8 * LS) + 1>([&](auto sc) {
    constexpr int size = 1 << decltype(sc)::value;
    static_for<0, decltype(sc)::value>([&](auto jc) {
      constexpr int j = (size >> 1) >> decltype(jc)::value;
      constexpr bool mirror = j == (size >> 1);
      if constexpr (j >= 8) {
        // partner lane i ^ M, element 7 - p (mirror) or p
        constexpr int M = mirror ? (size - 1) >> 3 : j >> 3;
        const bool lower = (i & (mirror ? (size >> 4) : (j >> 3))) == 0;
        uint32_t o[8];
        for (int p = 0; p < 8; ++p) o[p] = lane_xor<M>(v[mirror ? 7 - p : p]);
        for (int p = 0; p < 8; ++p) v[p] = lower ? max(v[p], o[p]) : min(v[p], o[p]);
      } else {
        for (int p = 0; p < 8; ++p) {
          const int pp = mirror ? (p ^ (size - 1)) : (p ^ j);
          if (pp > p) {
            const uint32_t a = v[p], b = v[pp];
            v[p] = max(a, b);
            v[pp] = min(a, b);
          }
        }
      }
    });
  });
}

// Lowest sweep value that a key scoring >= `th` can have.  `exact`: the
// sweep sees exact scores.  Otherwise it sees raw dot products r with
// score = clamp(fl(r * scale)), scale > 0, and the bound is widened by a
// relative margin far above the rounding error of that product.
__device__ __forceinline__ float sweep_floor(float th, bool exact, float scale) {
  if (exact) return th;
  if (!(th > -10.0f)) return -__builtin_inff();
  const double x = (static_cast<double>(th) - fabs(static_cast<double>(th)) * 0x1p-18 - 1e-30) /
                   static_cast<double>(scale);
  float f = static_cast<float>(x);
  if (static_cast<double>(f) > x) f = nextafterf(f, -__builtin_inff());
  return f;
}


// 16 bytes per lane from `src` to LDS at dst + 16 * lane (global_load_lds).
// Outside the kernel template: with a template-dependent pointer the host
// pass drops the kernel's launch stub.
__device__ __forceinline__ void lds_dma16(const unsigned char* src, unsigned char* dst) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)(dst), 16, 0, 0);
}

enum SweepMode : int {
  kRawDots = 0,     // MFMA dot products, scale > 0: filters on raw dots
  kExactScores = 1, // MFMA dot products converted to exact scores (scale <= 0)
  kGivenScores = 2  // caller-given scores
};

// How the score pass addresses K: rows of exactly D elements at hd = D
// (compile-time strides), rows at a run-time stride with hd = D, or any
// stride and hd (column tests).
enum KLayout : int { kKDense = 0, kKRows = 1, kKGeneral = 2 };

// One wave's quarter of a 64-key tile (keys 16 w .. 16 w + 15) as MFMA A
// operands, loaded straight from global memory (L2) into registers: lane
// (c, g) holds key 16 w + c at the head-dimension slots that rows_x_frag
// gives lane group g.  product() forms, for each of the four 16-row groups
// cb of the query block, the scores of the quarter's keys against rows
// 16 cb + c with the same operands in the same accumulation order as
// rows_x_frag, so every score is bit-identical to those of the passes that use
// it: the forward (but for fp32 at d <= 64, whose split products round
// otherwise; kSplitLeastU) and the tile backward.
// acc[cb][r] is the score of key 16 w + 4 g + r and row 16 cb + c.
template <typename T, int D> struct KQuarter;
template <typename T, int D> struct KQuarter16 {
  using V8 = typename Half<T>::v8;
  V8 a[D / 32];
  // `src`: the tile's first row plus the lane's byte offset (its key's row,
  // 16 g bytes in).  This register path loads 16 half rows per instruction,
  // a third of the L2 rate of whole-row loads; the rings (sweep_ring) read
  // whole rows where hd = D.  KL (KLayout): with kKGeneral columns >= hd read
  // as zero.
  template <int KL>
  __device__ __forceinline__ void load(const unsigned char* tile, uint32_t off, int hd, int g) {
    for (int s = 0; s < D / 32; ++s)
      a[s] = KL != kKGeneral || 32 * s + 8 * g < hd ? *reinterpret_cast<const V8*>(tile + (off + 64u * s)) : V8{};
  }
  __device__ __forceinline__ void product(f32x4 (&acc)[4], const RowFrag<T, D> (&qf)[4]) const {
    for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < D / 32; ++s)
      for (int cb = 0; cb < 4; ++cb) acc[cb] = mfma(a[s], qf[cb].v[s], acc[cb]);
  }
};
template <int D> struct KQuarter<u16, D> : KQuarter16<u16, D> {};
template <int D> struct KQuarter<h16, D> : KQuarter16<h16, D> {};
template <int D> struct KQuarter<float, D> {
  f32x4 a[D / 16];
  template <int KL>
  __device__ __forceinline__ void load(const unsigned char* tile, uint32_t off, int hd, int g) {
    for (int j = 0; j < D / 16; ++j)
      a[j] = KL != kKGeneral || 16 * j + 4 * g < hd ? *reinterpret_cast<const f32x4*>(tile + (off + 64u * j)) : f32x4{};
  }
  __device__ __forceinline__ void product(f32x4 (&acc)[4], const RowFrag<float, D> (&qf)[4]) const {
    for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < D / 16; ++j)
      for (int cb = 0; cb < 4; ++cb)
        for (int r = 0; r < 4; ++r) acc[cb] = mfma(a[j][r], qf[cb].v[j][r], acc[cb]);
  }
};

// The sweeps' LDS rings (16-bit inputs, hd = D): slots of 16 keys x 64
// dimensions (2 KiB) per wave.  Sweep 1 has the whole area below tkey to
// itself (four tiles in flight); the later sweeps' ring lies beside the
// candidate lists: two slots at d = 64, where a third would cost a resident
// block, three at 128.
constexpr int kSlotBytes = 2048;
constexpr int ring1_slots(int D) { return 4 * D / 64; }
constexpr int ring2_slots(int D) { return D == 64 ? 2 : 3; }

// LDS layout, shared by the kernel and the host-side size query.  The class
// maxima exchanged between the sweeps share their bytes with the candidate
// lists (they are read before the first candidate is written).
struct SelLayout {
  int cand, cm, scm, ring, tk, tkey, drop, fl, cnt, ctl, bits, vlist, total;
};
__host__ __device__ inline int align_up(int x, int a) { return (x + a - 1) / a * a; }
// Class sets per (row, position) of sweep 1, over NW waves: 64 of 16 NW R
// classes.  256 classes tighten the sweep-2 floor (fewer candidates) but
// double the class-maxima exchange in LDS; up to k = 64 the exchange at 128
// keeps two select blocks per compute unit (at d = 128, k = 64: 68 KB of
// LDS and 199 VGPRs against 86 KB and 257, measured 11.8 against 17.4 ms
// over 1x32x16384).
__host__ __device__ inline int classes_per_lane(int k, int NW) { return (k <= 64 ? 8 : 16) / NW; }
// ringD: the rings' D, or 0 for the variants without rings.
__host__ __device__ inline SelLayout sel_layout(int k, int cap, int nKB, int NW, int ringD) {
  SelLayout l;
  l.scm = 16 * NW * classes_per_lane(k, NW) + 4;  // floats per row of the class-maxima exchange (+4: rows 4 banks apart)
  const int cand_bytes = kBlock * (cap + 1) * 8;  // rows of cap + 1 slots (see cslot)
  const int cm_bytes = kBlock * l.scm * 4;
  const int ring_bytes = ringD ? NW * ring2_slots(ringD) * kSlotBytes : 0;
  const int tk_bytes = k * kBlock * 4;
  l.cand = 0;
  l.cm = 0;
  // the later sweeps' ring and the sorted top-k values (emission) share bytes
  l.ring = align_up(cand_bytes > cm_bytes ? cand_bytes : cm_bytes, 16);
  l.tk = l.ring;
  l.tkey = l.ring + align_up(ring_bytes > tk_bytes ? ring_bytes : tk_bytes, 16);
  const int ring1_bytes = ringD ? NW * ring1_slots(ringD) * kSlotBytes : 0;
  if (l.tkey < ring1_bytes) l.tkey = ring1_bytes;
  l.drop = l.tkey + kBlock * 8;
  l.fl = l.drop + kBlock * 8;
  l.cnt = l.fl + kBlock * 4;
  l.ctl = l.cnt + kBlock * 4;
  l.bits = l.ctl + 16;
  l.vlist = l.bits + align_up(2 * ((nKB + 31) / 32) * 4, 16);  // one bitmap per 32-row half
  l.total = l.vlist + align_up(nKB * 4, 16);
  return l;
}

// Overflow rounds a row can need.  Round 0 stores the first `cap` of its c_0
// candidates; the k-th best stored key T_1 then excludes at least the cap - k
// stored keys below it, so round 1 finds c_1 <= c_0 - (cap - k) keys >= T_1,
// and so on: with c_0 <= NK, at most 2 + (NK - cap) / (cap - k) rounds end
// with every candidate stored.
__host__ __device__ inline int select_round_bound(int NK, int k, int cap) {
  return 2 + (NK > cap ? (NK - cap) / (cap - k) + 1 : 0);
}

// Score pass of one (batch, head) and 64-row query block; NW = 4 or 8
// waves.  Wave w multiplies quarter w % 4 of the visible key tiles it takes
// (every tile of the list with 4 waves, every other one, from w / 4, with
// 8) with all 64 rows (no LDS staging, no barrier inside a sweep); lane
// (c, g) sees rows 16 cb + c and keys 16 (w % 4) + 4 g + r of each tile.  R
// class maxima per (lane, row, r) give 16 NW R classes per row.
//
// Waves per SIMD: three for the headline variant (bf16, d = 64, two classes
// per lane), whose ~50 KB of LDS let three blocks into a compute unit, and
// 168 VGPRs three waves onto a SIMD (one more VGPR would drop it to two);
// two for the 8-wave block.
template <typename T, int D, int R, int NW>
constexpr int select_waves_per_simd() { return NW == 8 ? 2 : sizeof(T) == 2 && D == 64 && R == 2 ? 3 : 1; }

// KL: the K layout (KLayout).  With hd = D (kKDense, kKRows) there are no
// column tests, and with 16-bit inputs sweep 1 reads K through the LDS ring
// (whose loads read whole rows).
template <typename T, int D, int MODE, int R, int KL, int NW>
__global__ __launch_bounds__(NW * kWave, (select_waves_per_simd<T, D, R, NW>())) void select_kernel(SelectParams p) {
  static_assert(NW == 4 || NW == 8, "waves per block");
  constexpr int kThreads = NW * kWave;
  constexpr int kPhases = NW / 4;     // tiles of the list taken side by side
  constexpr int kRows = kBlock / NW;  // rows per wave outside the sweeps
  constexpr bool kExact = MODE != kRawDots;
  constexpr bool kTiles = MODE != kGivenScores;
  constexpr int UR = R > 2 ? R : 2;  // sweep-1 unroll: class of a tile = ordinal % R
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int k = p.d.k, NQ = p.d.NQ, NK = p.d.NK, nKB = p.d.nKB, nQB = p.d.nQB;
  const int cap = p.cap;
  const int nbw = (nKB + 31) >> 5;
  const SelLayout lay = sel_layout(k, cap, nKB, NW, is_half<T> && KL != kKGeneral ? D : 0);
  uint64_t* s_cand = reinterpret_cast<uint64_t*>(smem + lay.cand);
  float* s_cm = reinterpret_cast<float*>(smem + lay.cm);
  float* s_tk = reinterpret_cast<float*>(smem + lay.tk);
  uint64_t* s_tkey = reinterpret_cast<uint64_t*>(smem + lay.tkey);
  unsigned long long* s_drop = reinterpret_cast<unsigned long long*>(smem + lay.drop);
  float* s_fl = reinterpret_cast<float*>(smem + lay.fl);
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(smem + lay.cnt);
  uint32_t* s_ctl = reinterpret_cast<uint32_t*>(smem + lay.ctl);
  uint32_t* s_bits = reinterpret_cast<uint32_t*>(smem + lay.bits);
  int32_t* s_vlist = reinterpret_cast<int32_t*>(smem + lay.vlist);
  // Slot of candidate e of row r, rows cap + 1 slots apart: an append's
  // address is one multiply-add (XOR-ing row bits into a slot-major layout
  // spread the sort's reads over more banks but cost every append four
  // more instructions).
  const int cstride = cap + 1;
  auto cslot = [&](int e, int r) { return r * cstride + e; };

  const int t = threadIdx.x, w = t >> 6, L = t & 63, g = L >> 4, c = L & 15;
  int brank, bh;
  xcd_rank_order(blockIdx.x, nQB, p.d.BH, brank, bh);
  const int qb = nQB - 1 - brank, q0 = qb * kBlock;  // heaviest first
  const size_t grow0 = size_t(bh) * NQ + q0;  // global index of the block's row 0
  const float scale = p.d.scale;

  // The lane's rows 16 cb + c.
  bool rowok[4];
  int qpos[4];
  for (int cb = 0; cb < 4; ++cb) {
    rowok[cb] = q0 + 16 * cb + c < NQ;
    qpos[cb] = rowok[cb] ? p.q_idx[grow0 + 16 * cb + c] : 0;
  }
  // Position range of the valid rows of the whole block (lane L <-> row L).
  const bool lv = q0 + L < NQ;
  const int lpos = lv ? p.q_idx[grow0 + L] : 0;
  const int qmax_blk = wave_max(lv ? lpos : INT_MIN);
  const int qmin_blk = wave_min(lv ? lpos : INT_MAX);

  if (t < kBlock) {
    s_cnt[t] = 0u;
    s_drop[t] = 0ull;
  }
  if (t < 4) s_ctl[t] = 0u;
  for (int i = t; i < 2 * nbw; i += kThreads) s_bits[i] = 0u;

  const int32_t* kidx = p.k_idx + size_t(bh) * NK;
  // Visible key blocks in ascending order, entry = block | class << 24, with
  // class 1 (partially visible: per-key tests needed) or 2 (every key
  // visible to every row), from the blocks' position bounds.
  if (w == 0) {
    const int2* kbnd = p.kbounds + size_t(bh) * nKB;
    int n = 0;
    for (int base = 0; base < nKB; base += kWave) {
      const int kt = base + L;
      int v = 0;
      if (kt < nKB) {
        const int2 kb = kbnd[kt];
        v = kb.x > qmax_blk ? 0 : ((kb.y > qmin_blk || (kt + 1) * kBlock > NK) ? 1 : 2);
      }
      const uint64_t m = __ballot(v != 0);
      const int before = __builtin_popcountll(m & ((uint64_t(1) << L) - 1));
      if (v != 0) s_vlist[n + before] = kt | (v << 24);
      n += __builtin_popcountll(m);
    }
    if (L == 0) s_ctl[1] = uint32_t(n);
  }
  __syncthreads();
  // this wave's tiles of the list: entries phase, phase + kPhases, ...
  const int phase = kPhases == 1 ? 0 : __builtin_amdgcn_readfirstlane(w >> 2);
  const int nvis = (int(s_ctl[1]) + kPhases - 1 - phase) / kPhases;
  const int wq = w & 3;  // and its quarter of them

  RowFrag<T, D> qf[4];  // Q^T operands: row 16 cb + c in column c of the products
  const T* Kb = nullptr;
  if constexpr (kTiles) {
    const T* Qh = static_cast<const T*>(p.q) + head_at(p.lq, bh, p.d.H);
    for (int cb = 0; cb < 4; ++cb)
      qf[cb].load(Qh + size_t(rowok[cb] ? q0 + 16 * cb + c : 0) * p.lq.sn, rowok[cb], L, p.d.hd);
    Kb = static_cast<const T*>(p.k) + head_at(p.lk, bh, p.d.H);
  }
  // K addressing: a tile's first row from scalar registers plus a 32-bit
  // lane offset (one load form for every tile; forming 64-bit lane addresses
  // per step took a quarter of sweep 1's VALU instructions).  Keys >= NK of
  // the last tile read its last valid key instead: they lie in a partially
  // visible tile, where the visibility test discards their scores.
  const uint32_t ksnb = KL == kKDense ? uint32_t(D * sizeof(T)) : uint32_t(p.lk.sn) * uint32_t(sizeof(T));
  const unsigned char* const Kbytes = reinterpret_cast<const unsigned char*>(Kb);
  const int klast = NK - 1 - (nKB - 1) * kBlock;  // last valid key of the last tile
  auto tile_at = [&](int kt) { return Kbytes + size_t(uint32_t(kt)) * (size_t(kBlock) * ksnb); };
  const int kq0 = 16 * wq + c;  // the lane's A-operand key within a tile
  const uint32_t koff = uint32_t(kq0) * ksnb + 16u * g, koff_last = uint32_t(min(kq0, klast)) * ksnb + 16u * g;

  // One pass over the visible key blocks: body(u, kt, visb, acc) for each,
  // u = (ordinal of the block in the wave's list) % U known at compile time.  The K quarters of
  // the next two tiles are in flight while a tile is used.  In partially
  // visible tiles bit 4 cb + r of visb is cleared and acc set to
  // -inf where key 16 wq + 4 g + r is not visible to row 16 cb + c (visb is
  // 0xffff for a whole tile); the body is called once, after the masking,
  // so its code is not repeated per case.  The wave's list entries are held
  // one per lane, 128 at a time: window() before step i0 (a multiple of 64
  // or the first) loads entries i0 .. i0 + 127, and entry(i) reads one of
  // them (reading entries past the first 64 from LDS at each step instead
  // put two LDS round trips into every step of a long list).
  int vl[2], vbase = 0;
  auto list_at = [&](int i) { return i < nvis ? s_vlist[kPhases * i + phase] : 0; };
  auto window = [&](int i0) {
    vl[0] = i0 == 0 ? list_at(L) : vl[1];
    vl[1] = list_at(i0 + kWave + L);
    vbase = i0;
  };
  auto entry = [&](int i) {  // vbase <= i < vbase + 128
    const int at = i - vbase;
    const int a0 = __builtin_amdgcn_readlane(vl[0], at & (kWave - 1));
    const int a1 = __builtin_amdgcn_readlane(vl[1], at & (kWave - 1));
    return at < kWave ? a0 : a1;
  };
  // Per tile, after its scores are formed: the visibility masking, then
  // body(u, kb0, visb, acc).  The padding of the last group of U tiles
  // (i >= nvis: no key visible, key limit INT_MIN) takes the partial
  // tiles' path: a separate path that set acc to constants made the
  // compiler copy acc between register sets on every whole tile.
  auto finish = [&](auto uc, int i, int e, f32x4(&acc)[4], auto&& body) __attribute__((always_inline)) {
    const int kb0 = (e & 0xffffff) * kBlock + 16 * wq + 4 * g;  // the lane's first key
    if constexpr (MODE == kExactScores)
      for (int cb = 0; cb < 4; ++cb)
        for (int r = 0; r < 4; ++r) acc[cb][r] = clamp_score(acc[cb][r] * scale);
    uint32_t visb = 0xffffu;
    if (i >= nvis || (e >> 24) == 1) {  // wave-uniform
      const int klim = i < nvis ? NK : INT_MIN;
      for (int r = 0; r < 4; ++r) {
        const int key = kb0 + r;
        const int kp = key < klim ? kidx[key] : INT_MAX;
        for (int cb = 0; cb < 4; ++cb)
          if (!(key < klim && kp <= qpos[cb])) {
            visb &= ~(1u << (4 * cb + r));
            acc[cb][r] = -__builtin_inff();
          }
      }
    }
    body(uc, kb0, visb, acc);
  };
  auto sweep = [&](auto u_tag, auto&& body) {
    constexpr int U = decltype(u_tag)::value;
    if (nvis == 0) return;  // wave-uniform
    window(0);
    KQuarter<T, D> kq[2];
    auto fetch = [&](KQuarter<T, D>& f, int e) {
      const int kt = e & 0xffffff;
      f.template load<KL>(tile_at(kt), kt == nKB - 1 ? koff_last : koff, p.d.hd, g);
    };
    // The loads are unconditional (past the end of the list they repeat its
    // last tile), so the number in flight is the same on every path and the
    // waits before a tile's products cover that tile's loads only.
    int ent[2] = {entry(0), entry(nvis > 1 ? 1 : 0)};  // the tiles in kq[0], kq[1]
    if constexpr (kTiles) {
      // issued in the loop's order (kq[0]'s loads first), so that the
      // loop head's wait is the same from the prologue and the back edge
      fetch(kq[0], ent[0]);
      __builtin_amdgcn_sched_barrier(0);
      fetch(kq[1], ent[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MODE == kGivenScores) {
      for (int i0 = 0; i0 < nvis; i0 += U) {
        if (i0 - vbase >= kWave) window(vbase + kWave);
        static_for<0, U>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const int i = i0 + u;
          const int e = ent[u & 1];
          f32x4 acc[4];
          const int kb0 = (e & 0xffffff) * kBlock + 16 * wq + 4 * g;
          for (int cb = 0; cb < 4; ++cb)
            for (int r = 0; r < 4; ++r) {
              const int key = kb0 + r;
              acc[cb][r] = rowok[cb] && key < NK
                               ? clamp_score(p.scores[(grow0 + 16 * cb + c) * NK + key])
                               : 0.0f;
            }
          ent[u & 1] = entry(i + 2 < nvis ? i + 2 : nvis - 1);
          finish(uc, i, e, acc, body);
        });
      }
    } else {
      // Software-pipelined by one tile: the products of tile i + 1 are
      // issued before tile i's scores are used, so the matrix unit works
      // under tile i's filter and candidate appends (the appends wait on
      // LDS).  accs[i & 1] holds tile i's scores; kq[j & 1] holds tile j's
      // operands, fetched two steps before its products.  The last step's
      // products (tile nvis, a repeat of the list's last tile) are unused.
      f32x4 accs[2][4];
      kq[0].product(accs[0], qf);
      int ecur = ent[0];
      ent[0] = entry(2 < nvis ? 2 : nvis - 1);
      fetch(kq[0], ent[0]);
      for (int i0 = 0; i0 < nvis; i0 += U) {
        if (i0 - vbase >= kWave) window(vbase + kWave);
        static_for<0, U>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const int i = i0 + u;
          const int enext = ent[(u + 1) & 1];
          kq[(u + 1) & 1].product(accs[(u + 1) & 1], qf);
          ent[(u + 1) & 1] = entry(i + 3 < nvis ? i + 3 : nvis - 1);
          fetch(kq[(u + 1) & 1], ent[(u + 1) & 1]);
          if (u == 0 || i < nvis) finish(uc, i, ecur, accs[u & 1], body);  // wave-uniform
          ecur = enext;
        });
      }
    }
  };
  // With 16-bit inputs and hd = D the sweeps read their K quarters through a
  // ring in LDS filled by global_load_lds (the loads in flight hold no
  // VGPRs).  Each wave owns NS slots of 16 keys x 64 dimensions, row-major;
  // a tile takes D / 64 of them.  Each DMA instruction reads 8 rows of 128
  // contiguous bytes: a load of 16 half rows, the MFMA operand layout,
  // streams from L2 at a third of the rate (measured at the headline shape:
  // 8.5 against 28 TB/s), and with it the second sweep ran at that rate
  // whatever its candidates cost (2150 against 820 clocks per tile and wave
  // for the first one at d = 128, two waves per SIMD).  global_load_lds
  // puts lane L's 16 bytes at the instruction's base + 16 L, so lane L
  // fetches the chunk that belongs at that place: row r's chunk x is stored
  // at chunk x ^ ((r >> 1) & 7), which makes the operand reads (16 rows at
  // one chunk per 16 lanes) fall in distinct banks.  The compiler does not
  // order LDS reads after the DMA that fills them, so the waits are
  // explicit: vmcnt before a slot is read (the (NS - 1) younger slots' loads
  // may stay in flight), lgkmcnt(0) before a slot is refilled.
  constexpr bool kRingSweep = kTiles && is_half<T> && KL != kKGeneral;
  auto sweep_ring = [&](auto ns_tag, int ring_at, auto&& body) {
   if constexpr (kRingSweep) {
    constexpr int NS = decltype(ns_tag)::value;
    constexpr int KH = D / 64;                           // slots per tile
    constexpr int UT = NS % KH == 0 ? NS / KH : NS;      // tiles after which the slots repeat
    if (nvis == 0) return;  // wave-uniform
    window(0);
    unsigned char* ringw = smem + ring_at + __builtin_amdgcn_readfirstlane(w) * NS * kSlotBytes;
    // lane L of instruction j: quarter row r = 8 j + L / 8, stored chunk
    // L % 8, fetched chunk (L % 8) ^ ((r >> 1) & 7)
    uint32_t doff[2], doff_last[2], roff[2];
    for (int j = 0; j < 2; ++j) {
      const int r = 8 * j + L / 8, key = 16 * wq + r;
      const uint32_t ch = 16u * uint32_t((L % 8) ^ ((r >> 1) & 7));
      doff[j] = uint32_t(key) * ksnb + ch;
      doff_last[j] = uint32_t(min(key, klast)) * ksnb + ch;
      // operand j of lane (c, g): quarter row c, chunk 4 j + g
      roff[j] = uint32_t(c * 128 + 16 * ((4 * j + g) ^ ((c >> 1) & 7)));
    }
    auto dma = [&](int slot, int e, int half) __attribute__((always_inline)) {
      const int kt = e & 0xffffff;
      const unsigned char* tile = tile_at(kt) + 128 * half;
      const bool last = kt == nKB - 1;
      for (int j = 0; j < 2; ++j)
        lds_dma16(tile + (last ? doff_last[j] : doff[j]), ringw + slot * kSlotBytes + j * kWave * 16);
    };
    // The Q fragments' loads are waited for here, by an s_waitcnt the
    // compiler sees: otherwise its wait for them before the first product
    // stays in the loop as vmcnt(0) on every tile (encoding: vmcnt 0,
    // expcnt 7, lgkmcnt 15).
    __builtin_amdgcn_s_waitcnt(0x0f70);
    for (int q = 0; q < NS; ++q) dma(q, entry(min(q / KH, nvis - 1)), q % KH);
    for (int i0 = 0; i0 < nvis; i0 += UT) {
      if (i0 - vbase >= kWave) window(vbase + kWave);
      if constexpr (KH == 1) {
        // d = 64: two tiles per step, so that a step's latencies (operand
        // reads, products, their results) are paid once for both
        static_for<0, UT / 2>([&](auto uc) {
          constexpr int u = 2 * decltype(uc)::value;
          const int i = i0 + u;
          if (i >= nvis) return;  // wave-uniform
          using V8 = typename Half<T>::v8;
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * 2) : "memory");
          V8 a[2][2];
          for (int q = 0; q < 2; ++q)
            for (int j = 0; j < 2; ++j)
              a[q][j] = *reinterpret_cast<const V8*>(ringw + (u + q) * kSlotBytes + roff[j]);
          f32x4 acc[2][4];
          for (int q = 0; q < 2; ++q)
            for (int cb = 3; cb >= 0; --cb) acc[q][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
          // KQuarter's products: reduction steps in order
          for (int j = 0; j < 2; ++j)
            for (int q = 0; q < 2; ++q)
              for (int cb = 3; cb >= 0; --cb) acc[q][cb] = mfma(a[q][j], qf[cb].v[j], acc[q][cb]);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          for (int q = 0; q < 2; ++q) dma(u + q, entry(min(i + q + NS, nvis - 1)), 0);
          finish(std::integral_constant<int, u>{}, i, entry(i), acc[0], body);
          if (i + 1 < nvis)  // wave-uniform
            finish(std::integral_constant<int, u + 1>{}, i + 1, entry(i + 1), acc[1], body);
        });
      } else {
        static_for<0, UT>([&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const int i = i0 + u;
          if (i >= nvis) return;  // wave-uniform
          using V8 = typename Half<T>::v8;
          f32x4 acc[4];
          for (int cb = 0; cb < 4; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
          static_for<0, KH>([&](auto hc) {
            constexpr int h = decltype(hc)::value, slot = (u * KH + h) % NS;
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * 2) : "memory");
            V8 a[2];
            for (int j = 0; j < 2; ++j)
              a[j] = *reinterpret_cast<const V8*>(ringw + slot * kSlotBytes + roff[j]);
            // KQuarter's products: reduction steps s = 2 h + j in order
            for (int j = 0; j < 2; ++j)
              for (int cb = 3; cb >= 0; --cb) acc[cb] = mfma(a[j], qf[cb].v[2 * h + j], acc[cb]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            dma(slot, entry(min(i + (h + NS) / KH, nvis - 1)), (h + NS) % KH);
          });
          finish(uc, i, entry(i), acc, body);
        });
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
   }
  };

  // ---------------- sweep 1: class maxima ----------------
  float cm[4][4 * R];
  const float pinf = opaque_inf();
  for (int cb = 0; cb < 4; ++cb)
    for (int j = 0; j < 4 * R; ++j) cm[cb][j] = -__builtin_inff();
  auto maxima = [&](auto uc, int, uint32_t, f32x4 (&acc)[4]) {
    constexpr int j = decltype(uc)::value % R;
    for (int cb = 0; cb < 4; ++cb)
      for (int r = 0; r < 4; ++r) cm[cb][r + 4 * j] = vmax(cm[cb][r + 4 * j], acc[cb][r], pinf);
  };
  if constexpr (kRingSweep) {
    sweep_ring(std::integral_constant<int, ring1_slots(D)>{}, 0, maxima);
    __syncthreads();  // every wave's ring reads are done before the exchange reuses the bytes
  } else {
    sweep(std::integral_constant<int, UR>{}, maxima);
  }

  // Exchange: row 16 cb + c's 16 NW R class maxima, 4 R from each of its
  // 4 NW lanes (NW waves x 4 lane groups), then wave w finds the floors of
  // rows kRows w + L % kRows, the row's lane L / kRows holding classes
  // [16 R (L / kRows), 16 R (L / kRows + 1)).
  for (int cb = 0; cb < 4; ++cb)
    for (int r = 0; r < 4; ++r)
      for (int j = 0; j < R; ++j)
        s_cm[(16 * cb + c) * lay.scm + ((w * 4 + g) * 4 + r) * R + j] = cm[cb][r + 4 * j];
  __syncthreads();
  {
    const int row = kRows * w + L % kRows, part = L / kRows;
    float v[16 * R];
    for (int i = 0; i < 16 * R; i += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(s_cm + row * lay.scm + 16 * R * part + i);
      for (int j = 0; j < 4; ++j) v[i + j] = x[j];
    }
    // a value x with at least k class maxima >= x (bisection between the
    // smallest and largest class maximum), then the sweep-2 floor
    float lo = __builtin_inff(), hi = -__builtin_inff();
    uint32_t nfin = 0;
    for (int i = 0; i < 16 * R; ++i) {
      nfin = count_ge(nfin, v[i], -3.0e38f);
      if (v[i] >= -3.0e38f) {
        lo = fminf(lo, v[i]);
        hi = fmaxf(hi, v[i]);
      }
    }
    const int nf = row_sum<NW>(int(nfin));
    lo = row_min<NW>(lo);
    hi = row_max<NW>(hi);
    float x = -__builtin_inff();
    auto at_least = [&](float m) {  // class maxima of the row >= m
      uint32_t cnt = 0;
      for (int i = 0; i < 16 * R; ++i) cnt = count_ge(cnt, v[i], m);
      return row_sum<NW>(int(cnt));
    };
    for (int it = 0; it < 8; ++it) {
      const float mid = 0.5f * (lo + hi);
      if (at_least(mid) >= k) lo = mid;
      else hi = mid;
    }
    // Eight steps are enough where a row's maxima spread evenly.  Where they
    // fall into clumps (clustered keys) lo can still be below many of them,
    // and lists of 1.75 k then overflow (a third sweep on most blocks at
    // 1x32x16384, k = 64): more steps until k + k / 32 at most reach lo.
    if (k > 42) {  // block-uniform; below, the lists hold k + 32
      int nlo = at_least(lo);
      for (int it = 0; it < 16 && __any(nlo > k + (k >> 5)); ++it) {
        const float mid = 0.5f * (lo + hi);
        const int n = at_least(mid);
        if (n >= k) {
          lo = mid;
          nlo = n;
        } else {
          hi = mid;
        }
      }
    }
    if (nf >= k) x = lo;
    const float th = kExact ? x : (x == -__builtin_inff() ? x : clamp_score(x * scale));
    // NaN marks a row that collects nothing (past NQ)
    if (part == 0) s_fl[row] = q0 + row < NQ ? sweep_floor(th, kExact, scale) : __builtin_nanf("");
  }
  __syncthreads();

  // ---------------- sweep 2 (and overflow rounds): candidates ----------------
  // A key of row 16 cb + c is a candidate when visible and !(v < fl[cb]):
  // with fl[cb] = -inf (the row's threshold is <= -10) every visible key is
  // one.  NaN dots (score -10) always pass; where the threshold is above -10
  // they cannot reach the top-k and only take a slot.  In rounds > 0 the
  // candidate's key must also reach the row's exact threshold s_tkey.
  // selection key of a stored candidate
  auto raw_key = [&](uint64_t raw) {
    const float v = __uint_as_float(uint32_t(raw));
    return make_key(kExact ? v : clamp_score(v * scale), int(raw >> 32));
  };
  float fl[4];
  int max_round = 0;
  const int round_bound = select_round_bound(NK, k, cap);
  for (int round = 0;; ++round) {
    // fl = NaN marks a row that collects nothing this round
    // A zero floor is held as -0, so that v - fl is +0 for both signed
    // zeros v (with +0, -0 - +0 = -0 would read as v < fl).
    // Rows with fl = -inf take every visible key (amask), whatever the sign
    // of a NaN difference.
    uint32_t cmask = 0, amask = 0;
    for (int cb = 0; cb < 4; ++cb) {
      fl[cb] = s_fl[16 * cb + c];
      if (fl[cb] == 0.0f) fl[cb] = -0.0f;
      if (!__builtin_isnan(fl[cb])) cmask |= 0xfu << (4 * cb);  // bit order of collect's m
      if (fl[cb] == -__builtin_inff()) amask |= 0xfu << (4 * cb);
    }
    // Candidates are stored raw, (index << 32) | bits of the sweep value,
    // and turned into selection keys when they are sorted.  Per tile, the
    // lane's candidate bits m (bit 4 cb + r: key kb0 + r of row
    // 16 cb + c) come branch-free, two instructions per score, in the order
    // the MFMA results arrive (cb = 0 first); the few lanes with candidates
    // then append two per trip (LDS atomics on the rows' counts), so the
    // wave runs half as many trips as its busiest lane has candidates.
    auto collect = [&](int kb0, uint32_t visb, f32x4 (&acc)[4], auto later) {
      // bit 4 cb + r <- sign of v - fl: set where v < fl, so that
      // the complement marks !(v < fl) (NaN differences have a clear sign
      // bit)
      uint32_t m = 0;
      for (int cb = 3; cb >= 0; --cb)
        for (int r = 3; r >= 0; --r)
          m = __builtin_amdgcn_alignbit(m, __float_as_uint(acc[cb][r] - fl[cb]), 31);
      m = (~m | amask) & cmask & visb;
      // score b = 4 cb + r by selects (parking the 16 scores in LDS to read
      // one back took the bytes that the later sweeps' ring now has)
      auto pick = [&](int b) {
        float x[4];
        for (int r = 0; r < 4; ++r) {
          const float lo = (b & 4) ? acc[1][r] : acc[0][r], hi = (b & 4) ? acc[3][r] : acc[2][r];
          x[r] = (b & 8) ? hi : lo;
        }
        const float lo = (b & 1) ? x[1] : x[0], hi = (b & 1) ? x[3] : x[2];
        return (b & 2) ? hi : lo;
      };
      auto append = [&](int row, int key, float v, uint32_t pos) {
        if (pos < uint32_t(cap))
          s_cand[cslot(pos, row)] = (uint64_t(uint32_t(key)) << 32) | __float_as_uint(v);
        else  // the best candidate left out
          atomicMax(&s_drop[row], make_key(kExact ? v : clamp_score(v * scale), key));
      };
      while (m != 0u) {
        const int b = __builtin_ctz(m);  // 4 cb + r
        m &= m - 1u;
        const int row = 4 * (b & 12) + c, key = kb0 | (b & 3);
        const float v = pick(b);
        if constexpr (decltype(later)::value) {
          if (make_key(kExact ? v : clamp_score(v * scale), key) < s_tkey[row]) continue;
        }
        append(row, key, v, atomicAdd(&s_cnt[row], 1u));
      }
    };
    auto collect_sweep = [&](auto later) {
      auto body = [&](auto, int kb0, uint32_t visb, f32x4 (&acc)[4]) { collect(kb0, visb, acc, later); };
      if constexpr (kRingSweep) sweep_ring(std::integral_constant<int, ring2_slots(D)>{}, lay.ring, body);
      else sweep(std::integral_constant<int, 2>{}, body);
    };
    if (round == 0) collect_sweep(std::false_type{});
    else collect_sweep(std::true_type{});
    __syncthreads();
    max_round = round;
    // Rows that overflowed: with T the k-th best stored key, every top-k key
    // is >= T.  A row whose best left-out candidate is below T has its whole
    // top-k in the list and is done.  That is the rule where many keys tie
    // at the score clamp: the lists fill in nearly ascending key order, so
    // the left-out ties come after the kept ones.  With the larger lists
    // above k = 42 (select_plan) a block's overflow rounds fell from two
    // to one: clustered keys, 1x32x16384, d = 128, k = 64, 11.3 -> 9.9 ms;
    // 1x8x32768 with 16 heavy keys, d = 128, k = 128, 10.6 -> 4.9 ms.
    // The others take T as an exact threshold, restart their lists, and the
    // block sweeps again for them.
    if (t < kBlock && q0 + t < NQ && s_cnt[t] > uint32_t(cap)) s_ctl[0] = uint32_t(round + 1);
    __syncthreads();
    if (s_ctl[0] != uint32_t(round + 1)) break;  // block-uniform
    for (int j = 0; j < kRows; ++j) {
      const int r = kRows * w + j;
      const bool over = q0 + r < NQ && s_cnt[r] > uint32_t(cap);  // wave-uniform
      if (!over) {
        if (L == 0) s_fl[r] = __builtin_nanf("");
        continue;
      }
      // T by bisection between bounds of the stored keys (their smallest
      // and largest score and index words), four compares and population
      // counts per step; the keys are distinct: some bound is met by exactly
      // k of them
      uint64_t v[4];
      uint32_t hmin = ~0u, hmax = 0u, lmin = ~0u, lmax = 0u;
      for (int e = 0; e < 4; ++e) {
        const bool in = L + kWave * e < cap;
        v[e] = in ? raw_key(s_cand[cslot(L + kWave * e, r)]) : 0ull;
        const uint32_t h = uint32_t(v[e] >> 32), l = uint32_t(v[e]);
        hmin = in ? min(hmin, h) : hmin;
        hmax = in ? max(hmax, h) : hmax;
        lmin = in ? min(lmin, l) : lmin;
        lmax = in ? max(lmax, l) : lmax;
      }
      uint64_t lo = (uint64_t(wave_minmax_u32<false>(hmin)) << 32) | wave_minmax_u32<false>(lmin);
      uint64_t hi = (uint64_t(wave_minmax_u32<true>(hmax)) << 32) | wave_minmax_u32<true>(lmax);
      while (lo < hi) {  // count(>= lo) >= k; T in [lo, hi]
        const uint64_t mid = hi - ((hi - lo) >> 1);
        int n = 0;
        for (int e = 0; e < 4; ++e) n += __builtin_popcountll(__ballot(v[e] >= mid));
        if (n >= k) lo = mid;
        else hi = mid - 1;
        if (n == k) {  // T is the smallest key >= mid
          uint32_t h = ~0u, l = ~0u;
          for (int e = 0; e < 4; ++e) h = v[e] >= mid ? min(h, uint32_t(v[e] >> 32)) : h;
          h = wave_minmax_u32<false>(h);
          for (int e = 0; e < 4; ++e)
            l = v[e] >= mid && uint32_t(v[e] >> 32) == h ? min(l, uint32_t(v[e])) : l;
          lo = hi = (uint64_t(h) << 32) | wave_minmax_u32<false>(l);
        }
      }
      if (L == 0) {
        const bool whole = s_drop[r] < lo;
        if (whole) {
          s_cnt[r] = uint32_t(cap);
          s_fl[r] = __builtin_nanf("");
        } else {
          s_tkey[r] = lo;
          s_fl[r] = sweep_floor(key_score(lo), kExact, scale);
          s_drop[r] = 0ull;
          s_ctl[2] = uint32_t(round + 1);
        }
      }
    }
    __syncthreads();  // all overflow reads of the lists and counts are done
    if (s_ctl[2] != uint32_t(round + 1)) break;  // block-uniform: every list is whole
    if (round + 1 >= round_bound) {
      // cannot happen (select_round_bound); reported, not looped on
      if (t == 0 && p.status) atomicOr(p.status, kStatusSelectRounds);
      break;
    }
    if (t < kBlock && !__builtin_isnan(s_fl[t])) s_cnt[t] = 0u;
    __syncthreads();
  }
  if (max_round > 0 && t == 0 && p.status)
    atomicMax(p.status, (uint32_t(max_round > 255 ? 255 : max_round) << 8));

  // ---------------- select: sort each row's candidates ----------------
  // The top-k key blocks go into the mask bitmap of the row's 32-row half
  // (wave w sorts rows kRows w .. kRows w + kRows - 1): with at most 64 key
  // blocks as one register word per lane, OR-ed over the wave at the end
  // (the per-entry LDS atomics would all hit the same two words).
  const bool kb_word = nKB <= 64;
  uint32_t* s_hbits = s_bits + (kRows * w / 32) * nbw;
  uint64_t kbm = 0;
  auto emit = [&](int r, int e, uint64_t key) {
    if (e >= k || q0 + r >= NQ) return;
    const bool real = key != 0ull;
    const float sv = real ? key_score(key) : kSentinel;
    const int idx = real ? key_index(key) : -1;
    s_tk[e * kWave + r] = sv;
    const size_t gr = size_t(bh) * NQ + q0 + r;
    if (p.topk_idx) {
      p.topk_idx[gr * k + e] = idx;
      p.topk_val[gr * k + e] = sv;
    }
    if (idx >= 0) {
      const int kb = idx / kBlock;
      if (kb_word) kbm |= uint64_t(1) << kb;
      else atomicOr(&s_hbits[kb >> 5], 1u << (kb & 31));
    }
  };
  auto ncand = [&](int r) -> int { return (q0 + r < NQ) ? min(int(s_cnt[r]), cap) : 0; };
  // With top-k outputs requested: segments of LS lanes x 8 keys sort one
  // row's (score, index) keys each; a group of 8 rows runs as one LS=8 pass
  // (<= 64 keys per row), two LS=16 or four LS=32 passes.
  auto sort_rows = [&](auto ls_tag, int row0) {
    constexpr int LS = decltype(ls_tag)::value;
    const int r = row0 + L / LS, i = L & (LS - 1), n = ncand(r);
    uint64_t v[8];
    for (int pp = 0; pp < 8; ++pp) {
      const int e = i * 8 + pp;
      v[pp] = e < n ? raw_key(s_cand[cslot(e, r)]) : 0ull;
    }
    segment_sort_desc<LS>(v, L);
    for (int pp = 0; pp < 8; ++pp) emit(r, i * 8 + pp, v[pp]);
  };
  // Otherwise only the values are sorted (32-bit order codes, no payload):
  // tau needs the top-k values in order, and the block mask needs the set of
  // top-k keys, which is every candidate scoring above the k-th value v_k
  // plus, of those scoring v_k, the ones with the lowest indices.  The
  // candidates are then read once more, unsorted, for the mask bits.
  auto select_rows = [&](auto ls_tag, int row0) {
    constexpr int LS = decltype(ls_tag)::value;
    const int r = row0 + L / LS, i = L & (LS - 1), n = ncand(r);
    const bool rok = q0 + r < NQ;
    auto ord_raw = [&](uint64_t raw) {
      const float x = __uint_as_float(uint32_t(raw));
      return ord_of(kExact ? x : clamp_score(x * scale));
    };
    uint32_t v[8], o8[8];  // o8: the lane's unsorted order codes, kept for the mask bits
    int x8[8];             //     and their key indices
    for (int pp = 0; pp < 8; ++pp) {
      const int e = i * 8 + pp;
      const uint64_t raw = e < n ? s_cand[cslot(e, r)] : 0ull;
      o8[pp] = e < n ? ord_raw(raw) : 0u;  // 0: empty slot
      x8[pp] = int(raw >> 32);
      v[pp] = o8[pp];
    }
    segment_sort_desc32<LS>(v, L);
    for (int pp = 0; pp < 8; ++pp) {
      const int e = i * 8 + pp;
      if (e < k && rok) s_tk[e * kWave + r] = v[pp] ? score_of_ord(v[pp]) : kSentinel;
    }
    // v_k and, over the row's sorted values, how many exceed / equal it
    const int src = (k - 1) >> 3, sp = (k - 1) & 7;
    uint32_t mine = v[0];
    for (int pp = 1; pp < 8; ++pp)
      if (pp == sp) mine = v[pp];
    const uint32_t vk = src < LS ? uint32_t(__shfl(int(mine), (L & ~(LS - 1)) + src, kWave)) : 0u;
    int gt = 0, eq = 0;
    for (int pp = 0; pp < 8; ++pp) {
      gt += v[pp] > vk ? 1 : 0;
      eq += v[pp] == vk ? 1 : 0;
    }
    for (int d = 1; d < LS; d <<= 1) {
      gt += __shfl_xor(gt, d, kWave);
      eq += __shfl_xor(eq, d, kWave);
    }
    // vk == 0: fewer than k candidates, all selected; else take the ties'
    // lowest indices when not all of them fit
    const int need = k - gt;
    const bool split = vk != 0u && eq > need;
    // the ties taken are those with index <= tlim: the need-th lowest index
    // among them, by bisection in every row of the wave at once (counting
    // each tie's lower-indexed ones instead took a quarter of the pass where
    // many keys tie at the score clamp: 400 of 1632 k clocks per block on
    // clustered keys, 1x32x16384, d = 128, k = 64)
    int tlim = INT_MAX;
    if (__any(split)) {  // wave-uniform
      int lo = 0, hi = split ? NK - 1 : 0;
      while (__any(lo < hi)) {
        const int mid = lo + ((hi - lo) >> 1);
        int cnt = 0;
        for (int pp = 0; pp < 8; ++pp) cnt += (o8[pp] == vk && x8[pp] <= mid) ? 1 : 0;
        static_for<0, ilog2(LS)>([&](auto dc) {
          cnt += int(lane_xor<(1 << decltype(dc)::value)>(uint32_t(cnt)));
        });
        if (cnt >= need) hi = mid;
        else lo = min(mid + 1, hi);
      }
      if (split) tlim = lo;
    }
    for (int pp = 0; pp < 8; ++pp) {
      const int e = i * 8 + pp;
      if (e >= n) continue;
      const uint32_t o = o8[pp];
      const int idx = x8[pp];
      if (vk == 0u || o > vk || (o == vk && idx <= tlim)) {
        const int kb = idx / kBlock;
        if (kb_word) kbm |= uint64_t(1) << kb;
        else atomicOr(&s_hbits[kb >> 5], 1u << (kb & 31));
      }
    }
  };
  const bool want_topk = p.topk_idx != nullptr;
  for (int base = kRows * w; base < kRows * (w + 1); base += 8) {
    int need = k;
    for (int j = 0; j < 8; ++j) need = max(need, ncand(base + j));
    if (want_topk) {
      if (need <= 64) {
        sort_rows(std::integral_constant<int, 8>{}, base);
      } else if (need <= 128) {
        sort_rows(std::integral_constant<int, 16>{}, base);
        sort_rows(std::integral_constant<int, 16>{}, base + 4);
      } else {
        for (int h = 0; h < 4; ++h) sort_rows(std::integral_constant<int, 32>{}, base + 2 * h);
      }
    } else {
      if (need <= 64) {
        select_rows(std::integral_constant<int, 8>{}, base);
      } else if (need <= 128) {
        select_rows(std::integral_constant<int, 16>{}, base);
        select_rows(std::integral_constant<int, 16>{}, base + 4);
      } else {
        for (int h = 0; h < 4; ++h) select_rows(std::integral_constant<int, 32>{}, base + 2 * h);
      }
    }
  }
  if (kb_word) {  // block-uniform
    kbm |= lane_xor64<1>(kbm);
    kbm |= lane_xor64<2>(kbm);
    kbm |= lane_xor64<4>(kbm);
    kbm |= lane_xor64<8>(kbm);
    auto bor = [](uint32_t x, uint32_t y) { return x | y; };
    const uint32_t lo = group_reduce_bits(uint32_t(kbm), bor);
    const uint32_t hi = group_reduce_bits(uint32_t(kbm >> 32), bor);
    if (L == 0) {
      if (lo) atomicOr(&s_hbits[0], lo);
      if (hi) atomicOr(&s_hbits[1], hi);  // nonzero only when nKB > 32 (nbw = 2)
    }
  }
  __syncthreads();

  // ---------------- mask row; sorted values for the tau kernel ----------------
  // the 64-row mask is the union of the halves; with 32-row blocks each
  // half's row is written too (the second only when the block has one)
  uint8_t* mrow = p.mask + (size_t(bh) * nQB + qb) * nKB;
  const int nQH = half_blocks(NQ);
  uint8_t* hrow = p.half ? p.half + (size_t(bh) * nQH + 2 * qb) * nKB : nullptr;
  const bool second = 2 * qb + 1 < nQH;
  for (int kb = t; kb < nKB; kb += kThreads) {
    const uint32_t b0 = (s_bits[kb >> 5] >> (kb & 31)) & 1u;
    const uint32_t b1 = (s_bits[nbw + (kb >> 5)] >> (kb & 31)) & 1u;
    mrow[kb] = uint8_t(b0 | b1);
    if (hrow) {
      hrow[kb] = uint8_t(b0);
      if (second) hrow[nKB + kb] = uint8_t(b1);
    }
  }
  const size_t rows = size_t(p.d.BH) * NQ;
  for (int i = t; i < k * kBlock; i += kThreads) {
    const int e = i >> 6, r = i & 63;
    if (q0 + r < NQ) p.tkv[size_t(e) * rows + size_t(bh) * NQ + q0 + r] = s_tk[e * kWave + r];
  }
}

template <typename T, int D, int MODE, int R, int KL, int NW>
hipError_t launch_one(const SelectParams& p, hipStream_t s) {
  const SelLayout l =
      sel_layout(p.d.k, p.cap, p.d.nKB, NW, is_half<T> && KL != kKGeneral ? D : 0);
  auto kern = select_kernel<T, D, MODE, R, KL, NW>;
  if (l.total > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, l.total);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(p.d.nQB * p.d.BH), dim3(NW * kWave), l.total, s, p);
  return hipGetLastError();
}

// The hd = D variants (kKDense, kKRows) for the 16-bit MFMA sweeps with raw
// dots (the usual scale > 0) that read K through the LDS rings; the others
// take the general loads into registers.
template <typename T, int D, int MODE, int R, int NW>
hipError_t launch_ring(const SelectParams& p, hipStream_t s) {
  if constexpr (is_half<T> && MODE == kRawDots)
    if (p.ring) {
      if (p.lk.sn == D) return launch_one<T, D, MODE, R, kKDense, NW>(p, s);
      return launch_one<T, D, MODE, R, kKRows, NW>(p, s);
    }
  return launch_one<T, D, MODE, R, kKGeneral, NW>(p, s);
}

// Class sets per (row, position): classes_per_lane; waves: select_plan.
template <typename T, int D, int MODE>
hipError_t launch_r(const SelectParams& p, hipStream_t s) {
  if constexpr (MODE == kRawDots && (is_half<T> || D == 64))
    if (p.waves == 8) {
      if (p.d.k <= 64) return launch_ring<T, D, MODE, 1, 8>(p, s);
      return launch_ring<T, D, MODE, 2, 8>(p, s);
    }
  if (p.d.k <= 64) return launch_ring<T, D, MODE, 2, 4>(p, s);
  return launch_ring<T, D, MODE, 4, 4>(p, s);
}

template <typename T, int D>
hipError_t launch_mode(const SelectParams& p, hipStream_t s) {
  if (p.d.scale > 0.0f) return launch_r<T, D, kRawDots>(p, s);
  return launch_r<T, D, kExactScores>(p, s);
}

template <typename T>
hipError_t launch_type(const SelectParams& p, hipStream_t s) {
  if (p.d.D == 64) return launch_mode<T, 64>(p, s);
  if (p.d.D == 128) return launch_mode<T, 128>(p, s);
  return hipErrorInvalidValue;
}

}  // namespace

}  // namespace asa
