// Supplied-noise target sampling and the exact_target acceptance walk.
//
// Replaces sample_from_logits / exact_accept_paths_batch
// (flashgrpo/decoding/acceptance.py:34-130, 179-260; correction tokens as in
// flashgrpo_b200/decoding/acceptance.py:184-267). torch.multinomial cannot take
// caller noise, so the draw follows one integer inverse-CDF rule that the CPU
// oracle reproduces bit for bit:
//   m = max x (NaN ignored), q_i = weight_q40(m, x_i, kt): 2^40 * 2^-(a_i / 2^20) for the
//   fixed-point exponent a_i = trunc((m - x_i) * fp32(2^20 / ln 2) / T) (fg_common.h)
//   candidate order (key(x) desc, index asc); top_k keeps the first k; top_p
//   keeps position j while the preceding kept mass <= floor(total * tp32 / 2^32)
//   target = floor(total_kept * u32 / 2^32); token = first kept index (vocab
//   order) whose inclusive q prefix exceeds target.
// Integer sums make every result independent of reduction order.
//
// draw_path chooses where a draw runs:
//  * rows of up to 65,536 logits (32,768 with a cut), unless greedy: one launch of one workgroup per row
//    that holds the row in registers (resident_sample);
//  * longer rows with a workspace: over 16 chunks per row, unrestricted draws in three launches (two in a
//    walk step whose row maxima come from the LM head's epilogue), greedy draws in two (one; see "split
//    sampling"), top-k and top-p draws in four or two (see "split top-k / top-p");
//  * otherwise (block_sample): one 1024-thread workgroup per row, the row split into 16 contiguous wave
//    segments; a wave walks its segment 512 elements (8 per lane, 16-byte loads) per step. Top-k / top-p
//    use an MSB-first 4 x 8-bit radix select over the keys with count or q-weighted histograms in LDS.
#include <mutex>
#include <type_traits>

#include "fg_common.h"

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kStep = 512;  // elements per wave step

// Histogram copies: lane l adds to copy l % kCopies of a bin, the copies of a bin side by side on
// banks of their own, so that logits close to each other wait less for one word (the q-mass
// pass of 64 x 152,064: 13.4 -> 12.2 us with 8 copies instead of one per wave).
constexpr int kCopies = 8;

struct Shared {
  uint64_t exp2[1024];  // kExp2Table
  uint64_t wsum[kWaves];
  uint64_t hist[256][kCopies];
  uint64_t wkey[kWaves];
  float wmax[kWaves];
  uint64_t u64b[2];
  int32_t i32b[2];
};

template <int DT>
struct Row {
  const char* p;
  int V;
  int seg;
  float kt;             // weight scale: fp32(2^20 / ln 2) / T
  const uint64_t* tbl;  // kExp2Table in LDS
  float m;              // row maximum (NaN ignored)

  FG_DEVICE int load(int i0, float (&x)[8]) const {
    if (i0 + 8 <= V) {
      fg::load8<DT>(p, i0, x);
      return 8;
    }
    int n = V - i0;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = j < n ? fg::load_elem<DT>(p, i0 + j) : 0.0f;
    return n < 0 ? 0 : n;
  }
  // candidates are ranked by the logits themselves (the temperature scales the weight)
  FG_DEVICE float scaled(float x) const { return x; }
  FG_DEVICE uint64_t weight(float s) const { return fg::weight_q40(m, s, kt, tbl); }
};

// Candidate-set predicate: key > kappa, or key == kappa and index <= last.
struct KeyCut {
  uint32_t kappa;
  uint32_t last;
  FG_DEVICE bool operator()(uint32_t key, uint32_t i) const { return key > kappa || (key == kappa && i <= last); }
};
constexpr KeyCut kAll{0u, 0xffffffffu};

// Calls f(i, s, key) for each element of this wave's segment, 8 per lane per step.
template <int DT, class F>
FG_DEVICE void for_wave_segment(const Row<DT>& r, F&& f) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lo = wave * r.seg;
  const int hi = min(r.V, lo + r.seg);
  for (int base = lo; base < hi; base += kStep) {
    int i0 = base + lane * 8;
    float x[8];
    int n = r.load(i0, x);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < n) {
        float s = r.scaled(x[j]);
        f(i0 + j, s, fg::sort_key32(s));
      }
  }
}

// Elements equal to kappa inside a candidate cut.
struct TiePred {
  KeyCut within;
  uint32_t kappa;
  FG_DEVICE bool operator()(uint32_t key, uint32_t i) const { return key == kappa && within(key, i); }
};

// Block sum over pred-elements of w (1 or q); per-wave partials land in sh.wsum.
template <bool WEIGHTED, int DT, class Pred>
FG_DEVICE uint64_t block_sum(const Row<DT>& r, Pred pred, Shared& sh) {
  __syncthreads();
  uint64_t acc = 0;
  for_wave_segment(r, [&](int i, float s, uint32_t key) {
    if (pred(key, (uint32_t)i)) acc += WEIGHTED ? r.weight(s) : 1ull;
  });
  acc = fg::wave_sum_u64(acc);
  if ((threadIdx.x & 63) == 0) sh.wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  uint64_t tot = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) tot += sh.wsum[w];
  return tot;
}

// First index (vocabulary order) among pred-elements whose inclusive running
// sum of w exceeds target (-1 if none). sh.wsum must hold the per-wave sums of
// the same (pred, w), as left by block_sum.
template <bool WEIGHTED, int DT, class Pred>
FG_DEVICE int block_locate(const Row<DT>& r, Pred pred, uint64_t target, Shared& sh) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint64_t before = 0;
  int win = -1;
  for (int w = 0; w < kWaves; ++w) {
    if (before + sh.wsum[w] > target) {
      win = w;
      break;
    }
    before += sh.wsum[w];
  }
  __syncthreads();
  if (threadIdx.x == 0) sh.i32b[0] = -1;
  __syncthreads();
  if (wave == win) {
    uint64_t run = before;
    const int lo = wave * r.seg;
    const int hi = min(r.V, lo + r.seg);
    for (int base = lo; base < hi; base += kStep) {
      int i0 = base + lane * 8;
      float x[8];
      int n = r.load(i0, x);
      uint64_t w8[8];
      uint64_t mine = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w8[j] = 0;
        if (j < n) {
          float s = r.scaled(x[j]);
          if (pred(fg::sort_key32(s), (uint32_t)(i0 + j))) w8[j] = WEIGHTED ? r.weight(s) : 1ull;
        }
        mine += w8[j];
      }
      uint64_t incl = fg::wave_incl_scan_u64(mine);
      uint64_t step_total = fg::shfl_u64(incl, 63);
      if (run + step_total > target) {
        uint64_t excl = run + incl - mine;
        if (excl <= target && target < run + incl) {
          uint64_t c = excl;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            c += w8[j];
            if (c > target) {
              sh.i32b[0] = i0 + j;
              break;
            }
          }
        }
        break;
      }
      run += step_total;
    }
  }
  __syncthreads();
  return sh.i32b[0];
}

// MSB-first radix select over `within`-elements in candidate order
// (key desc, index asc): returns the cut that keeps every position up to and
// including the first one where the running count / q-mass exceeds target.
template <bool WEIGHTED, int DT>
FG_DEVICE KeyCut radix_select(const Row<DT>& r, KeyCut within, uint64_t target, Shared& sh) {
  uint32_t prefix = 0, pmask = 0;
  uint64_t above = 0;  // mass of within-elements whose key is above the current range
  const int lane = threadIdx.x & 63;
  for (int level = 0; level < 4; ++level) {
    const int shift = 24 - 8 * level;
    __syncthreads();
    for (int d = threadIdx.x; d < 256 * kCopies; d += kThreads) (&sh.hist[0][0])[d] = 0;
    __syncthreads();
    for_wave_segment(r, [&](int i, float s, uint32_t key) {
      if (within(key, (uint32_t)i) && (key & pmask) == prefix)
        atomicAdd((unsigned long long*)&sh.hist[(key >> shift) & 255u][lane % kCopies],
                  (unsigned long long)(WEIGHTED ? r.weight(s) : 1ull));
    });
    __syncthreads();
    if (threadIdx.x < 64) {
      // lane l owns digits 255-4l .. 252-4l, scanned from the largest digit down
      uint64_t h[4], mine = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[j] = 0;
#pragma unroll 1
        for (int q = 0; q < kCopies; ++q) h[j] += sh.hist[255 - 4 * lane - j][q];
        mine += h[j];
      }
      uint64_t incl = fg::wave_incl_scan_u64(mine);
      uint64_t excl = incl - mine;
      if (above + excl <= target && target < above + incl) {
        uint64_t c = above + excl;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (c + h[j] > target) {
            sh.i32b[1] = 255 - 4 * lane - j;
            sh.u64b[1] = c;
            break;
          }
          c += h[j];
        }
      }
    }
    __syncthreads();
    prefix |= (uint32_t)sh.i32b[1] << shift;
    above = sh.u64b[1];
    pmask |= 255u << shift;
  }
  // Ties on the selected key resolve in index order.
  TiePred tie{within, prefix};
  block_sum<WEIGHTED, DT>(r, tie, sh);
  int last = block_locate<WEIGHTED, DT>(r, tie, target - above, sh);
  return KeyCut{prefix, (uint32_t)last};
}

// First maximum of the raw logits (rank keys: value desc, index asc).
template <int DT>
FG_DEVICE int block_argmax(const Row<DT>& raw, Shared& sh) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  uint64_t best = 0;
  for_wave_segment(raw, [&](int i, float, uint32_t key) {
    uint64_t k = ((uint64_t)key << 32) | (uint64_t)(0xffffffffu - (uint32_t)i);
    best = k > best ? k : best;
  });
  best = fg::wave_max_u64(best);
  __syncthreads();
  if (lane == 0) sh.wkey[wave] = best;
  __syncthreads();
  uint64_t b = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) b = sh.wkey[w] > b ? sh.wkey[w] : b;
  return (int)fg::rank_key_index(b);
}

template <int DT>
FG_DEVICE Row<DT> make_row(const void* rowp, int V) {
  Row<DT> r;
  r.p = (const char*)rowp;
  r.V = V;
  r.seg = (((V + kWaves - 1) / kWaves) + kStep - 1) / kStep * kStep;
  r.kt = 0.0f;
  r.tbl = nullptr;
  r.m = 0.0f;
  return r;
}

struct SampleParams {
  float temperature;
  int greedy;
  int top_k;      // 0 = off
  uint32_t tp32;  // 0 = off
  bool cut() const { return !greedy && (top_k > 0 || tp32 != 0); }
};

// One draw from one row by the whole block. Returns the token (all threads).
template <int DT>
FG_DEVICE int block_sample(const void* rowp, int V, const SampleParams& sp, uint32_t u, Shared& sh) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  Row<DT> r = make_row<DT>(rowp, V);
  r.kt = fg::weight_kt(sp.temperature > 0.0f && sp.temperature != 1.0f, sp.temperature);
  r.tbl = sh.exp2;
  if (sp.greedy) return block_argmax<DT>(r, sh);
  fg::exp2_table_to_lds(sh.exp2);  // visible after the barriers of the max below
  float mx = -INFINITY;
  for_wave_segment(r, [&](int, float s, uint32_t) { mx = fmaxf(mx, s); });
  mx = fg::wave_max(mx);
  __syncthreads();
  if (lane == 0) sh.wmax[wave] = mx;
  __syncthreads();
  mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sh.wmax[w]);
  r.m = mx;

  KeyCut keep = kAll;
  if (sp.top_k > 0) keep = radix_select<false, DT>(r, kAll, (uint64_t)(sp.top_k - 1), sh);
  if (sp.tp32) {
    uint64_t tot = block_sum<true, DT>(r, keep, sh);
    keep = radix_select<true, DT>(r, keep, fg::mulhi_u64_u32(tot, sp.tp32), sh);
  }
  uint64_t total = block_sum<true, DT>(r, keep, sh);
  if (total == 0) return block_argmax<DT>(r, sh);
  return block_locate<true, DT>(r, keep, fg::mulhi_u64_u32(total, u), sh);
}

// ------------------------------------------------------------------ selection by the fixed-point exponent
// Bins of the exponent a (fg_common.h), 8 per octave below the row maximum, or 256 (128 at least) over
// the row's own range where that is narrower, so that a flat row's bins hold no more elements than
// another's: a never grows with x, so the bins are runs of the candidate order. Elements of weight 0
// are in no bin: they cannot be drawn, and in the candidate order only NaN comes before one with weight.
constexpr int kSelBins = 256;
constexpr int kSelBinShift = 17;             // 2^17 steps of a: 8 bins per octave
constexpr uint32_t kSelAMax = 40u << 20;     // larger a weigh 0
constexpr int kSelList = 8192;               // list entries per row
constexpr int kSelTopK = 4096;               // largest top_k the list path takes

FG_DEVICE uint32_t fixed_exponent(float m, float x, float kt) {
#pragma clang fp contract(off)
  return (uint32_t)fminf((m - x) * kt, fg::kWeightZmax);
}
// The weight of weight_q40 from its exponent.
FG_DEVICE uint64_t exponent_weight(uint32_t a, const uint64_t* tbl) {
  const uint64_t e = tbl[(a >> 10) & 1023u];
  const uint32_t w = (uint32_t)e - (__umul24((uint32_t)(e >> 32), a & 1023u) >> 10);
  return ((uint64_t)w << 32) >> ((a >> 20) + 23u);
}
// Steps of a (log2) of a bin in a row from `low` to m.
FG_DEVICE int bin_shift(float m, float low, float kt) {
  const uint32_t range = low <= m ? fixed_exponent(m, low, kt) : 0u;
  return min(kSelBinShift, max(0, 24 - (int)__clz((int)(range | 1u))));
}
FG_DEVICE int sel_bin(uint32_t a, int shift) { return min((int)(a >> shift), kSelBins - 1); }
FG_DEVICE float above_inf(float x) { return x > -INFINITY ? x : INFINITY; }  // for the least logit
FG_DEVICE float wave_min(float v) { return -fg::wave_max(-v); }

// Largest-first selection over the keys ck[0, n) >= cut (whole block of kThreads; the keys are
// distinct): the key at which the running count, or the running q-mass of the logit that a key
// holds, first exceeds target. LOW orders by the low word alone (index ascending). The caller
// guarantees that the total exceeds target. Radix select from the highest differing bit, 8
// bits a level, ending early where one key is left.
struct SelectShared {
  uint64_t hist[256];
  uint32_t cnt[256];
  uint64_t wred[kWaves];
  uint64_t above, found;
  int digit;
};

template <bool MASS, bool LOW>
FG_DEVICE uint64_t list_select(const uint64_t* ck, int n, uint64_t cut, uint64_t target, float m, float kt,
                               const uint64_t* tbl, SelectShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63;
  const auto value = [](uint64_t k) { return LOW ? (k & 0xffffffffull) : k; };
  // bits in which the considered keys differ
  uint64_t ones = 0, zeros = 0;
#pragma unroll 1
  for (int i = tid; i < n; i += kThreads)
    if (ck[i] >= cut) {
      ones |= value(ck[i]);
      zeros |= ~value(ck[i]);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ones |= fg::shfl_xor_u64(ones, o);
    zeros |= fg::shfl_xor_u64(zeros, o);
  }
  __syncthreads();  // sh is free
  if (lane == 0) {
    sh.wred[tid >> 6] = ones;
    sh.hist[tid >> 6] = zeros;
  }
  __syncthreads();
#pragma unroll 2
  for (int w = 0; w < kWaves; ++w) {
    ones |= sh.wred[w];
    zeros |= sh.hist[w];
  }
  const uint64_t diff = ones & zeros;
  if (diff == 0) return value(ones);  // one key
  int shift = max(0, 56 - __builtin_clzll(diff));
  // the chosen bits so far: the ones above the highest differing bit are common to all
  uint64_t fixed = shift + 8 >= 64 ? 0ull : ~0ull << (shift + 8);
  uint64_t prefix = ones & fixed, above = 0;
  for (;;) {
    __syncthreads();
    if (tid < 256) {
      sh.hist[tid] = 0;
      sh.cnt[tid] = 0;
    }
    __syncthreads();
#pragma unroll 1
    for (int i = tid; i < n; i += kThreads) {
      const uint64_t k = ck[i], v = value(k);
      if (k >= cut && (v & fixed) == prefix) {
        const int d = (int)(v >> shift) & 255;
        atomicAdd(&sh.cnt[d], 1u);
        if constexpr (MASS)
          atomicAdd((unsigned long long*)&sh.hist[d],
                    (unsigned long long)fg::weight_q40(m, fg::rank_key_value(k), kt, tbl));
      }
    }
    __syncthreads();
    if (tid < 64) {  // lane l owns digits 255 - 4 l .. 252 - 4 l
      uint64_t h[4], mine = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 255 - 4 * lane - j;
        h[j] = MASS ? sh.hist[d] : (uint64_t)sh.cnt[d];
        mine += h[j];
      }
      const uint64_t incl = fg::wave_incl_scan_u64(mine), excl = incl - mine;
      if (above + excl <= target && target < above + incl) {
        uint64_t c = above + excl;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (c + h[j] > target) {
            sh.digit = 255 - 4 * lane - j;
            sh.above = c;
            break;
          }
          c += h[j];
        }
      }
    }
    __syncthreads();
    above = sh.above;
    prefix |= (uint64_t)sh.digit << shift;
    fixed |= 255ull << shift;
    if (sh.cnt[sh.digit] == 1) {
#pragma unroll 1
      for (int i = tid; i < n; i += kThreads)
        if (ck[i] >= cut && (value(ck[i]) & fixed) == prefix) sh.found = value(ck[i]);
      __syncthreads();
      return sh.found;
    }
    if (shift == 0) return prefix;
    shift = max(0, shift - 8);
  }
}

// At most kSmallList keys are ranked by comparing each with every other, kSmallPer threads a
// key: one pass instead of the four barriers a level of the radix select.
constexpr int kSmallList = 256;
constexpr int kSmallPer = kThreads / kSmallList;

struct SmallShared {
  uint64_t w[kSmallList];     // q-mass
  uint64_t mass[kSmallList];  // q-mass of the keys before it in candidate order
  uint64_t at[kSmallList];    // kept q-mass of the keys before it in index order
  int rank[kSmallList];       // keys before it in candidate order
  uint64_t key;
  int tok;
};

FG_DEVICE void small_rank(const uint64_t* ck, int n, float m, float kt, const uint64_t* tbl, SmallShared& sh) {
  const int tid = threadIdx.x, i = tid & (kSmallList - 1);
  if (tid < kSmallList) {
    sh.w[i] = i < n ? fg::weight_q40(m, fg::rank_key_value(ck[i]), kt, tbl) : 0ull;
    sh.mass[i] = 0;
    sh.at[i] = 0;
    sh.rank[i] = 0;
    if (tid == 0) sh.tok = -1;
  }
  __syncthreads();
  if (i < n) {
    const uint64_t key = ck[i];
    int rank = 0;
    uint64_t mass = 0;
#pragma unroll 2
    for (int j = tid / kSmallList; j < n; j += kSmallPer)
      if (ck[j] > key) {
        ++rank;
        mass += sh.w[j];
      }
    if (rank) {
      atomicAdd(&sh.rank[i], rank);
      atomicAdd((unsigned long long*)&sh.mass[i], (unsigned long long)mass);
    }
  }
  __syncthreads();
}

// The key at which the running q-mass of the n <= kSmallList keys first exceeds target.
FG_DEVICE uint64_t small_cut(const uint64_t* ck, int n, uint64_t target, float m, float kt, const uint64_t* tbl,
                             SmallShared& sh) {
  small_rank(ck, n, m, kt, tbl, sh);
  const int i = threadIdx.x;
  if (i < n && sh.mass[i] <= target && target < sh.mass[i] + sh.w[i]) sh.key = ck[i];
  __syncthreads();
  return sh.key;
}

// list_draw of n <= kSmallList keys.
FG_DEVICE int small_draw(const uint64_t* ck, int n, int64_t slots, uint32_t tp32, uint32_t u, float m, float kt,
                         const uint64_t* tbl, SmallShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, i = tid & (kSmallList - 1);
  small_rank(ck, n, m, kt, tbl, sh);
  // every wave sums the kept mass: keys lane, lane + 64, ...
  constexpr int P = kSmallList / 64;
  uint64_t kw[P], total = 0;
#pragma unroll
  for (int h = 0; h < P; ++h) {
    kw[h] = sh.rank[lane + 64 * h] < slots ? sh.w[lane + 64 * h] : 0ull;
    total += kw[h];
  }
  total = fg::wave_sum_u64(total);
  if (tp32) {
    const uint64_t thr = fg::mulhi_u64_u32(total, tp32);
    total = 0;
#pragma unroll
    for (int h = 0; h < P; ++h) {
      if (sh.mass[lane + 64 * h] > thr) kw[h] = 0;
      total += kw[h];
    }
    total = fg::wave_sum_u64(total);
  }
  __syncthreads();
  if (tid < 64) {
#pragma unroll
    for (int h = 0; h < P; ++h) sh.w[lane + 64 * h] = kw[h];
  }
  __syncthreads();
  if (total == 0) return -1;
  const uint64_t target = fg::mulhi_u64_u32(total, u);
  if (i < n) {
    const uint32_t low = (uint32_t)ck[i];  // falls with the index
    uint64_t before = 0;
#pragma unroll 2
    for (int j = tid / kSmallList; j < n; j += kSmallPer)
      if ((uint32_t)ck[j] > low) before += sh.w[j];
    if (before) atomicAdd((unsigned long long*)&sh.at[i], (unsigned long long)before);
  }
  __syncthreads();
  if (tid < n && sh.at[tid] <= target && target < sh.at[tid] + sh.w[tid])
    sh.tok = (int)fg::rank_key_index(ck[tid]);
  __syncthreads();
  return sh.tok;
}

// Sum over the block (kThreads) of v.
FG_DEVICE uint64_t select_block_sum(uint64_t v, SelectShared& sh) {
  v = fg::wave_sum_u64(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.wred[threadIdx.x >> 6] = v;
  __syncthreads();
  uint64_t t = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) t += sh.wred[w];
  return t;
}

// The draw among n listed candidates (whole block): the first `slots` of them in candidate order,
// then the top-p cut (tp32 != 0), then the noise u. -1 when nothing has weight.
FG_DEVICE int list_draw(const uint64_t* ck, int n, int64_t slots, uint32_t tp32, uint32_t u, float m, float kt,
                        const uint64_t* tbl, SelectShared& sel, SmallShared& small) {
  if (n <= kSmallList) return small_draw(ck, n, slots, tp32, u, m, kt, tbl, small);
  uint64_t cut = 0;
  const auto kept_sum = [&]() {
    uint64_t k = 0;
#pragma unroll 1
    for (int i = threadIdx.x; i < n; i += kThreads)
      if (ck[i] >= cut) k += fg::weight_q40(m, fg::rank_key_value(ck[i]), kt, tbl);
    return select_block_sum(k, sel);
  };
  if (slots < n) cut = list_select<false, false>(ck, n, 0, (uint64_t)(slots - 1), m, kt, tbl, sel);
  uint64_t total = kept_sum();
  if (total == 0) return -1;
  if (tp32) {
    cut = list_select<true, false>(ck, n, cut, fg::mulhi_u64_u32(total, tp32), m, kt, tbl, sel);
    total = kept_sum();
  }
  return (int)fg::rank_key_index(list_select<true, true>(ck, n, cut, fg::mulhi_u64_u32(total, u), m, kt, tbl, sel));
}

// Loads elements i0 .. i0 + 7 of a chunk ending at hi; past hi come -inf, whose weight is
// 0 against any row maximum, so the weights need no per-element test.
template <int DT>
FG_DEVICE void split_load8(const char* p, int i0, int hi, float (&x)[8]) {
  if (i0 + 8 <= hi) {
    fg::load8<DT>(p, i0, x);
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = i0 + j < hi ? fg::load_elem<DT>(p, i0 + j) : -INFINITY;
}

// First index in [lo, hi) whose inclusive running mass w(x, index) exceeds target (the whole
// block of THREADS; -1 if none), scanned in index order one group of THREADS x 8 elements at a
// time (thread t holds 8 consecutive elements of a group), stopping at the group that holds
// the target. The LOADS groups of a pass are loaded together. wsum: THREADS / 64 words.
template <int DT, int THREADS, int LOADS, class W>
FG_DEVICE int split_locate(const char* p, int lo, int hi, W&& weight, uint64_t target, uint64_t* wsum, int* found) {
  constexpr int WAVES = THREADS / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) *found = -1;
  uint64_t run = 0;  // block-uniform
  bool done = false;
  for (int base = lo; base < hi && !done; base += THREADS * 8 * LOADS) {
    float x[LOADS][8];
#pragma unroll
    for (int u = 0; u < LOADS; ++u)
      if (base + u * THREADS * 8 < hi) split_load8<DT>(p, base + (u * THREADS + tid) * 8, hi, x[u]);
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      if (base + u * THREADS * 8 >= hi) break;  // uniform
      const int i0 = base + (u * THREADS + tid) * 8;
      uint64_t mine = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) mine += weight(x[u][j], i0 + j);
      const uint64_t incl = fg::wave_incl_scan_u64(mine);
      __syncthreads();  // wsum of the previous group has been read
      if (lane == 63) wsum[wave] = incl;
      __syncthreads();
      uint64_t woff = 0, stot = 0;
#pragma unroll 4
      for (int w = 0; w < WAVES; ++w) {
        if (w < wave) woff += wsum[w];
        stot += wsum[w];
      }
      if (run + stot > target) {  // uniform: this group holds the target
        uint64_t cum = run + woff + incl - mine;
        if (cum <= target && target < cum + mine) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            cum += weight(x[u][j], i0 + j);
            if (cum > target) {
              *found = i0 + j;
              break;
            }
          }
        }
        done = true;
        break;
      }
      run += stot;
    }
  }
  __syncthreads();
  return *found;
}

// Where a cut lies: kept are the exponents below lo, and those in [lo, hi) whose rank key is at least cut.
struct RowCut {
  uint32_t lo, hi;
  uint64_t cut;
  uint64_t rest;  // q-mass (top-p) or count (top-k) before the cut within [lo, hi)
  int n, nan;     // top-k: listed elements (all kept ones among them), NaN logits (they take slots)
};
FG_DEVICE RowCut bin_cut(int bin, int shift, uint64_t rest) {
  return RowCut{(uint32_t)bin << shift, bin < kSelBins - 1 ? (uint32_t)(bin + 1) << shift : kSelAMax + 1, 0, rest, 0, 0};
}

struct NarrowShared {
  uint64_t wred[kWaves];
  uint32_t ones[kWaves], zeros[kWaves];
  uint64_t before;
  int digit, n, nan, found;
};

// f(x, i0) for every 8 elements from i0 on of a row, over the whole block; past V the logits are -inf.
template <int DT, class F>
FG_DEVICE void for_row8(const char* p, int V, F&& f) {
  for (int base = 0; base < V; base += kThreads * 16) {
    float x[2][8];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (base + u * kThreads * 8 < V) split_load8<DT>(p, base + (u * kThreads + threadIdx.x) * 8, V, x[u]);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (base + u * kThreads * 8 < V) f(x[u], base + (u * kThreads + (int)threadIdx.x) * 8);
  }
}

// The cut of a row whose class [c.lo, c.hi) holds more elements than a list (flat rows, long ties), by one
// workgroup: the class is cut into at most 256 parts by exponent and replaced by the one that holds the
// cut, until its elements fit the list; a class of one value is cut by index. Top-k starts from all
// exponents with c.rest = top_k. False where the row has no weight, NaN takes every slot, or more
// distinct logits than a list share one exponent (2^-20 octaves).
// Two passes over the row a step, as a rule one step. In place of block_sample, whose radix over the key
// bits makes four passes a cut: top-k 50 of 64 equal rows of 152,064 bf16 logits 590 -> 170 us, top-k 1,000 of
// rows with a standard deviation of 0.05 in units of the temperature 236 -> 48 (bins of the row's range too).
template <int DT, bool COUNT>
FG_DEVICE bool narrow_cut(const char* p, int V, float m, float kt, const uint64_t* tbl, uint64_t* ck, RowCut& c,
                          NarrowShared& sh, SelectShared& sel, SmallShared& small) {
  const int tid = threadIdx.x, lane = tid & 63;
  uint64_t* hist = ck;  // [kSelBins][kCopies], until the list takes its place
  static_assert(kSelBins * kCopies <= kSelList, "the histogram fits the list");
  const auto list = [&](auto&& take) {  // elements x at i with take(a, x, i) into ck; sh.n is 0
    for_row8<DT>(p, V, [&](const float(&x)[8], int i0) {
      uint32_t hit = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (take(fixed_exponent(m, x[j], kt), x[j], i0 + j)) hit |= 1u << j;
      if (!hit) return;
      int at = atomicAdd(&sh.n, (int)__popc(hit));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (hit >> j & 1u) {
          if (at < kSelList) ck[at] = fg::rank_key(x[j], (uint32_t)(i0 + j));
          ++at;
        }
    });
    __syncthreads();
  };
  for (bool first = COUNT;; first = false) {
    const uint32_t width = c.hi - c.lo;
    const int shift = max(0, 24 - (int)__clz((int)(width - 1)));
    __syncthreads();  // ck and sh are free
    if (width == 1) {  // one exponent already
      if (tid == 0) sh.n = 0;
      __syncthreads();
    } else {
      for (int i = tid; i < kSelBins * kCopies; i += kThreads) hist[i] = 0;
      if (tid == 0) {
        sh.digit = -1;
        sh.n = 0;
        sh.nan = 0;
      }
      __syncthreads();
      int nan = 0;
      for_row8<DT>(p, V, [&](const float(&x)[8], int) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t a = fixed_exponent(m, x[j], kt);
          if constexpr (COUNT) nan += x[j] != x[j];
          if (a - c.lo < width)
            atomicAdd((unsigned long long*)&hist[((a - c.lo) >> shift) * kCopies + lane % kCopies],
                      (unsigned long long)(COUNT ? 1ull : exponent_weight(a, tbl)));
        }
      });
      if (COUNT && first && nan) atomicAdd(&sh.nan, nan);
      __syncthreads();
      if (tid < 64) {  // the part of the cut: lane l owns parts 4 l .. 4 l + 3
        uint64_t b[4], mine = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          b[j] = 0;
#pragma unroll
          for (int q = 0; q < kCopies; ++q) b[j] += hist[(4 * lane + j) * kCopies + q];
          mine += b[j];
        }
        const uint64_t incl = fg::wave_incl_scan_u64(mine), total = fg::shfl_u64(incl, 63);
        bool ok = total > 0;
        uint64_t target = c.rest;
        if (first) {
          const uint64_t slots = (uint64_t)max((int)c.rest - sh.nan, 0);
          ok &= slots > 0;
          target = (total <= slots ? total : slots) - 1;
        }
        if (ok && incl - mine <= target && target < incl) {
          uint64_t before = incl - mine;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (before + b[j] > target) {
              sh.digit = 4 * lane + j;
              sh.before = target - before;
              break;
            }
            before += b[j];
          }
        }
      }
      __syncthreads();
      if (sh.digit < 0) return false;
      if (first) c.nan = sh.nan;
      c.rest = sh.before;
      c.lo += (uint32_t)sh.digit << shift;
      c.hi = min(c.hi, c.lo + (1u << shift));
    }
    uint32_t ones = 0, zeros = 0;  // bits in which the keys of the class differ
    list([&](uint32_t a, float x, int) {
      const bool in = a - c.lo < c.hi - c.lo;
      const uint32_t key = fg::sort_key32(x);
      ones |= in ? key : 0u;
      zeros |= in ? ~key : 0u;
      return in || (COUNT && a < c.lo);
    });
    c.n = sh.n;
    if (c.n <= kSelList) {
      if constexpr (!COUNT)
        c.cut = c.n <= kSmallList ? small_cut(ck, c.n, c.rest, m, kt, tbl, small)
                                  : list_select<true, false>(ck, c.n, 0, c.rest, m, kt, tbl, sel);
      return true;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ones |= (uint32_t)__shfl_xor((int)ones, o, 64);
      zeros |= (uint32_t)__shfl_xor((int)zeros, o, 64);
    }
    if (lane == 0) {
      sh.ones[tid >> 6] = ones;
      sh.zeros[tid >> 6] = zeros;
    }
    __syncthreads();
#pragma unroll 4
    for (int w = 0; w < kWaves; ++w) {
      ones |= sh.ones[w];
      zeros |= sh.zeros[w];
    }
    if ((ones & zeros) == 0) {  // one value: its first elements are kept, as many as rest reaches
      const uint32_t key = ones;
      const float v = fg::rank_key_value((uint64_t)key << 32);
      const uint64_t w = COUNT ? 1ull : exponent_weight(fixed_exponent(m, v, kt), tbl);  // > 0: the class has mass
      const int idx = split_locate<DT, kThreads, 2>(
          p, 0, V, [&](float x, int) { return fg::sort_key32(x) == key ? 1ull : 0ull; }, c.rest / w, sh.wred, &sh.found);
      c.cut = ((uint64_t)key << 32) | (uint64_t)(0xffffffffu - (uint32_t)idx);
      if constexpr (COUNT) {  // at most top_k elements
        if (tid == 0) sh.n = 0;
        __syncthreads();
        list([&](uint32_t a, float x, int i) {
          return a < c.lo || (a < c.hi && fg::rank_key(x, (uint32_t)i) >= c.cut);
        });
        c.n = sh.n;
      }
      return true;
    }
    if (c.hi - c.lo == 1) return false;
  }
}

// ------------------------------------------------------------------ one workgroup, the row in registers
// A row of up to 8,192 G logits held by one workgroup, 8 G per thread (element 8 (1024 u + t) + j
// of thread t): one memory pass and one launch for every draw but a greedy one, by the rule of block_sample.
//  * the maximum;
//  * top-k / top-p: a histogram over the bins above (counts / q-mass), the bin of the cut, a
//    list of its elements (top-k: and of those above), the exact cut among them;
//  * the draw: q-mass sums per (group, wave) in vocabulary order, then the one wave that holds the
//    target scans its lanes. Top-k draws among its list.
// Bound by latency: one memory round trip and about 32 G weights per thread between some ten
// barriers. Against the launches it replaces (three for an unrestricted draw, seven for top-p),
// a draw of 8 x 32,000 bf16 rows took, us: unrestricted 16.6 -> 10.9, top-p 48.8 -> 30.4, top-k 50
// 49.0 -> 14.7; of 512 rows 43.2 -> 19.9, 220.7 -> 63.4, 102.0 -> 32.0.
enum Cut : int { kNoCut, kTopP, kTopK };  // kTopK: with a top-p cut after it or not

template <int CUT>
struct ResidentShared {
  uint64_t hist[CUT ? kSelBins : 1][kCopies];
  uint64_t ck[CUT ? kSelList : 1];
  uint64_t wsum[kWaves * 8];   // [group][wave]
  SelectShared sel;
  SmallShared small;
  uint64_t before;
  uint32_t least, most;
  int bin, n, nan, tok;
};

template <int DT, int G, int CUT>
FG_DEVICE int resident_sample(const void* rowp, int V, const SampleParams& sp, uint32_t u, Shared& sh,
                              ResidentShared<CUT>& rs) {
  constexpr bool CUTS = CUT != kNoCut, count = CUT == kTopK;
  static_assert(G * kWaves <= kWaves * 8, "group sums");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const auto load_group = [&](int g, float(&v)[8]) {
    const int i0 = (g * kThreads + tid) * 8;
    if (i0 + 8 <= V) {
      fg::load8<DT>(rowp, i0, v);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = i0 + j < V ? fg::load_elem<DT>(rowp, i0 + j) : -INFINITY;
    }
  };
  float x[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) load_group(g, x[g]);
  // Each pass computes from the logits alone, one group at a time: values kept from one pass to
  // the next, or several groups in flight, would not fit the 128 registers of 1,024 threads.
  [[maybe_unused]] const auto fresh = [&](int g) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(x[g][j]));
  };
  fg::exp2_table_to_lds(sh.exp2);
  const float kt = fg::weight_kt(sp.temperature > 0.0f && sp.temperature != 1.0f, sp.temperature);
  if constexpr (CUTS) {
    for (int i = tid; i < kCopies * kSelBins; i += kThreads) (&rs.hist[0][0])[i] = 0;
    if (tid == 0) {
      rs.bin = kSelBins;
      rs.n = 0;
      rs.nan = 0;
    }
  }
  float m = -INFINITY;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, x[g][j]);
  m = fg::wave_max(m);
  if (lane == 0) sh.wmax[wave] = m;
  __syncthreads();
  m = sh.wmax[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, sh.wmax[w]);
  const auto weight = [&](float v) { return fg::weight_q40(m, v, kt, sh.exp2); };
  RowCut rc{};
  uint64_t hit = 0;  // bit 8 g + j: this thread's element j of group g is listed, later: is kept
  uint32_t e[CUTS ? G : 1][8];  // the exponents stand for the logits from here on
  if constexpr (CUTS) {
    uint64_t* h = &rs.hist[0][lane % kCopies];
    int nan = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      fresh(g);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        e[g][j] = fixed_exponent(m, x[g][j], kt);
        nan += x[g][j] != x[g][j];
      }
    }
    if (nan) atomicAdd(&rs.nan, nan);
    const auto fresh_e = [&](int g) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(e[g][j]));
    };
    const auto index_of = [&](int bit) { return ((bit >> 3) * kThreads + tid) * 8 + (bit & 7); };
    // all exponents in 8 bins an octave, then, while the cut's bin overflows the list, that bin's range in 256
    uint32_t lo = 0, hi = kSelAMax + 1;
    int shift = kSelBinShift, n;
    for (bool first = true;; first = false) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        fresh_e(g);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (e[g][j] - lo < hi - lo)
            atomicAdd((unsigned long long*)&h[sel_bin(e[g][j] - lo, shift) * kCopies],
                      (unsigned long long)(count ? 1ull : exponent_weight(e[g][j], sh.exp2)));
      }
      __syncthreads();
      if (wave == 0) {  // the bin of the cut: lane l owns bins 4 l .. 4 l + 3
        uint64_t b[4], mine = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          b[j] = 0;
#pragma unroll
          for (int q = 0; q < kCopies; ++q) b[j] += rs.hist[4 * lane + j][q];
          mine += b[j];
        }
        const uint64_t incl = fg::wave_incl_scan_u64(mine), total = fg::shfl_u64(incl, 63);
        const uint64_t slots = (uint64_t)max(sp.top_k - rs.nan, 0);  // NaN ranks first and takes slots
        // block_sample (bin stays kSelBins): no weight, or every slot taken by NaN
        const bool ok = total > 0 && (!count || slots > 0);
        const uint64_t target = !first  ? rc.rest
                                : count ? (total <= slots ? total : slots) - 1
                                        : fg::mulhi_u64_u32(total, sp.tp32);
        if (ok && incl - mine <= target && target < incl) {
          uint64_t c = incl - mine;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (c + b[j] > target) {
              rs.bin = 4 * lane + j;
              rs.before = target - c;  // position of the cut within the bin
              break;
            }
            c += b[j];
          }
        }
      }
      __syncthreads();
      n = -1;
      if (rs.bin == kSelBins) break;
      rc.lo = lo + ((uint32_t)rs.bin << shift);
      rc.hi = rs.bin == kSelBins - 1 ? hi : min(hi, rc.lo + (1u << shift));
      rc.rest = rs.before;
      hit = 0;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        fresh_e(g);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (e[g][j] < rc.hi && (count || e[g][j] >= rc.lo)) hit |= 1ull << (8 * g + j);
      }
      if (hit) {
        int at = atomicAdd(&rs.n, (int)__popcll(hit));
        for (uint64_t rest = hit; rest; rest &= rest - 1) {
          const int i = index_of(__builtin_ctzll(rest));
          if (at < kSelList) rs.ck[at] = fg::rank_key(fg::load_elem<DT>(rowp, i), (uint32_t)i);
          ++at;
        }
      }
      __syncthreads();
      n = rs.n;
      if (G * 8 * kThreads <= kSelList || n <= kSelList) break;
      uint32_t least = 0xffffffffu, most = 0;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        fresh_e(g);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const bool in = e[g][j] >= rc.lo && e[g][j] < rc.hi;
          least = min(least, in ? e[g][j] : 0xffffffffu);
          most = max(most, in ? e[g][j] : 0u);
        }
      }
      for (int i = tid; i < kCopies * kSelBins; i += kThreads) (&rs.hist[0][0])[i] = 0;
      if (tid == 0) {
        rs.least = 0xffffffffu;
        rs.most = 0;
      }
      __syncthreads();  // rs.n and rs.bin have been read
      atomicMin(&rs.least, least);
      atomicMax(&rs.most, most);
      if (tid == 0) rs.n = 0;
      __syncthreads();
      lo = rs.least;
      hi = rs.most + 1;
      n = -1;
      if (hi - lo == 1) break;  // long ties
      shift = max(0, 24 - (int)__clz((int)(hi - 1 - lo)));
    }
    if (n < 0) {
      __syncthreads();
      return block_sample<DT>(rowp, V, sp, u, sh);
    }
    if constexpr (count) {
      const int tok = list_draw(rs.ck, n, (int64_t)sp.top_k - rs.nan, sp.tp32, u, m, kt, sh.exp2, rs.sel, rs.small);
      __syncthreads();
      return tok;
    }
    rc.cut = n <= kSmallList ? small_cut(rs.ck, n, rc.rest, m, kt, sh.exp2, rs.small)
                             : list_select<true, false>(rs.ck, n, 0, rc.rest, m, kt, sh.exp2, rs.sel);
    for (uint64_t rest = hit; rest; rest &= rest - 1) {
      const int i = index_of(__builtin_ctzll(rest));
      if (fg::rank_key(fg::load_elem<DT>(rowp, i), (uint32_t)i) < rc.cut) hit &= ~(rest & -rest);
    }
  }
  // the draw among the kept elements, in vocabulary order: q-mass of each (group, wave)
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if constexpr (CUTS) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(e[g][j]));
    } else {
      fresh(g);
    }
    uint64_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (CUTS) {
        if (e[g][j] < rc.lo || ((hit >> (8 * g + j)) & 1)) w += exponent_weight(e[g][j], sh.exp2);
      } else {
        w += weight(x[g][j]);
      }
    }
    w = fg::wave_sum_u64(w);
    if (lane == 0) rs.wsum[g * kWaves + wave] = w;
  }
  if (tid == 0) rs.tok = -1;
  __syncthreads();
  // every wave finds the (group, wave) run that holds the target: lane l owns runs PL l ..
  constexpr int PL = (G * kWaves + 63) / 64;
  uint64_t run[PL], mine = 0;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    run[j] = lane * PL + j < G * kWaves ? rs.wsum[lane * PL + j] : 0ull;
    mine += run[j];
  }
  const uint64_t incl = fg::wave_incl_scan_u64(mine), total = fg::shfl_u64(incl, 63);
  if (total == 0) {
    __syncthreads();
    return block_argmax<DT>(make_row<DT>(rowp, V), sh);
  }
  const uint64_t target = fg::mulhi_u64_u32(total, u);
  uint64_t c = incl - mine, at = 0;
  int sel = -1;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    if (sel < 0 && c <= target && target < c + run[j]) {
      sel = lane * PL + j;
      at = c;
    }
    c += run[j];
  }
  const int src = (int)__builtin_ctzll(__ballot(sel >= 0));  // exactly one lane holds it
  sel = __shfl(sel, src, 64);
  at = fg::shfl_u64(at, src);
  if (sel % kWaves == wave) {  // this wave weighs its elements of the group again
    const int g = sel / kWaves;
    float v[8];
    load_group(g, v);
    uint64_t w[8], sum = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = (g * kThreads + tid) * 8 + j;
      w[j] = weight(v[j]);
      if constexpr (CUTS) {
        const uint32_t a = fixed_exponent(m, v[j], kt);
        if (a >= rc.hi || (a >= rc.lo && fg::rank_key(v[j], (uint32_t)i) < rc.cut)) w[j] = 0;
      }
      sum += w[j];
    }
    uint64_t cum = at + fg::wave_incl_scan_u64(sum) - sum;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (cum <= target && target < cum + w[j]) rs.tok = (g * kThreads + tid) * 8 + j;
      cum += w[j];
    }
  }
  __syncthreads();
  return rs.tok;
}

template <int DT, int G, int CUT>
FG_DEVICE int row_sample(const void* rowp, int V, const SampleParams& sp, uint32_t u, Shared& sh) {
  if constexpr (G > 0) {
    __shared__ ResidentShared<CUT> rs;
    return resident_sample<DT, G, CUT>(rowp, V, sp, u, sh, rs);
  } else {
    return block_sample<DT>(rowp, V, sp, u, sh);
  }
}

FG_DEVICE uint32_t noise_value(const uint32_t* noise, int64_t noise_index, uint64_t seed, uint64_t step,
                               uint32_t seq, uint32_t draw) {
  if (noise) return noise[noise_index];
  return fg::counter_noise(seed, step, seq, draw);
}

template <int DT, int G, int CUT>
__global__ void __launch_bounds__(kThreads) sample_rows_kernel(
    const void* __restrict__ logits, int64_t row_stride, int vocab, const int32_t* __restrict__ row_index,
    const int32_t* __restrict__ forced, const uint32_t* __restrict__ noise, int noise_stride, int noise_col,
    uint64_t seed, uint64_t step, const int32_t* __restrict__ seq_ids, int draw, SampleParams sp,
    int32_t* __restrict__ out) {
  __shared__ Shared sh;
  const int rrow = blockIdx.x;
  if (forced && forced[rrow] >= 0) {
    if (threadIdx.x == 0) out[rrow] = forced[rrow];
    return;
  }
  const int src = row_index ? row_index[rrow] : rrow;
  const char* rowp = (const char*)logits + (int64_t)src * row_stride * (DT == fg::kBF16 ? 2 : 4);
  uint32_t seq = seq_ids ? (uint32_t)seq_ids[rrow] : (uint32_t)rrow;
  uint32_t u = noise_value(noise, (int64_t)rrow * noise_stride + noise_col, seed, step, seq, (uint32_t)draw);
  int tok = row_sample<DT, G, CUT>(rowp, vocab, sp, u, sh);
  if (threadIdx.x == 0) out[rrow] = tok;
}

// Walk state lives in the caller's workspace: parent[B], active[B], and the
// walk step at which each row last sampled (-1 before its first draw) [B].
__global__ void walk_init_kernel(const int32_t* __restrict__ tree_tokens, const int32_t* __restrict__ parents,
                                 const int32_t* __restrict__ n_nodes, int nmax, int batch, int32_t* acc_tokens,
                                 int32_t* acc_nodes, int acc_stride, int32_t* acc_len, int32_t* last_node,
                                 int32_t* correction, int32_t* state) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  acc_tokens[(int64_t)b * acc_stride] = tree_tokens[(int64_t)b * nmax];
  acc_nodes[(int64_t)b * acc_stride] = 0;
  for (int j = 1; j < acc_stride; ++j) {  // the rest of the rows start at 0
    acc_tokens[(int64_t)b * acc_stride + j] = 0;
    acc_nodes[(int64_t)b * acc_stride + j] = 0;
  }
  acc_len[b] = 1;
  last_node[b] = 0;
  correction[b] = -1;
  int has_child = 0;
  for (int c = 1; c < n_nodes[b]; ++c) has_child |= parents[(int64_t)b * nmax + c] == 0;
  state[b] = 0;                  // parent
  state[batch + b] = has_child;  // active
  state[2 * batch + b] = -1;     // last sampling step
}

// Lazy LM-head rows of a walk step: row b samples from hidden row b*nmax + parent[b].
__global__ void walk_rows_kernel(const int32_t* __restrict__ state, int batch, int nmax, int32_t* row_index,
                                 int32_t* row_active) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  row_index[b] = b * nmax + state[b];
  row_active[b] = state[batch + b];
}

// Walk update of tree b after its draw `tok` at `parent`, by the 64 lanes of one wave
// (nmax <= 64, host-checked): lane c loads node c's parent and token, one ballot finds the
// first child of `parent` drawing `tok` (the lowest such node index) and a second whether
// that child has children; lane 0 writes the results. A serial scan by one thread would
// wait for up to 2 nmax dependent loads. tok and parent are taken from lane 0.
// next_rows / next_active (optional): the LM-head rows of the next walk step of tree b,
// as walk_rows_kernel would write them.
FG_DEVICE void walk_apply(int b, int tok, int parent, const int32_t* tree_tokens, const int32_t* parents,
                          const int32_t* n_nodes, int nmax, int batch, int walk_step, int32_t* acc_tokens,
                          int32_t* acc_nodes, int acc_stride, int32_t* acc_len, int32_t* last_node,
                          int32_t* correction, int32_t* state, int32_t* err_flag, int32_t* next_rows = nullptr,
                          int32_t* next_active = nullptr) {
  const int lane = threadIdx.x & 63;
  tok = __builtin_amdgcn_readfirstlane(tok);
  parent = __builtin_amdgcn_readfirstlane(parent);
  const int nn = n_nodes[b];
  const bool in = lane >= 1 && lane < nn;
  const int pc = in ? parents[(int64_t)b * nmax + lane] : -2;
  const int tc = in ? tree_tokens[(int64_t)b * nmax + lane] : 0;
  const uint64_t hit = __ballot(in && pc == parent && tc == tok);
  const int match = hit ? (int)__builtin_ctzll(hit) : -1;
  const uint64_t kids = __ballot(in && match >= 0 && lane > match && pc == match);
  if (lane != 0) return;
  state[2 * batch + b] = walk_step;
  if (match < 0) {
    correction[b] = tok;
    state[batch + b] = 0;
  } else {
    int len = acc_len[b];
    if (len < acc_stride) {
      acc_tokens[(int64_t)b * acc_stride + len] = tok;
      acc_nodes[(int64_t)b * acc_stride + len] = match;
      acc_len[b] = len + 1;
    } else if (err_flag) {
      atomicOr(err_flag, 4);
    }
    last_node[b] = match;
    state[b] = match;
    state[batch + b] = kids != 0ull;
  }
  if (next_rows) {
    next_rows[b] = b * nmax + state[b];
    next_active[b] = state[batch + b];
  }
}

template <int DT, int G, int CUT>
__global__ void __launch_bounds__(kThreads) walk_step_kernel(
    const void* __restrict__ logits, int64_t row_stride, int vocab, const int32_t* __restrict__ slot_map,
    const int32_t* __restrict__ tree_tokens, const int32_t* __restrict__ parents, const int32_t* __restrict__ n_nodes,
    int nmax, int batch, int walk_step, int rows_by_batch, const uint32_t* __restrict__ noise, int noise_stride,
    int noise_col0, uint64_t seed, uint64_t step, const int32_t* __restrict__ seq_ids, int draw0, SampleParams sp,
    int32_t* acc_tokens, int32_t* acc_nodes, int acc_stride, int32_t* acc_len, int32_t* last_node,
    int32_t* correction, int32_t* state, int32_t* err_flag, int32_t* next_rows, int32_t* next_active) {
  __shared__ Shared sh;
  const int b = blockIdx.x;
  if (!state[batch + b]) return;
  const int parent = state[b];
  const int64_t slot = rows_by_batch ? (int64_t)b
                       : slot_map    ? (int64_t)slot_map[(int64_t)b * nmax + parent]
                                     : (int64_t)b * nmax + parent;
  if (slot < 0) {
    if (threadIdx.x == 0) {
      if (err_flag) atomicOr(err_flag, 2);
      state[batch + b] = 0;
      if (next_active) next_active[b] = 0;
    }
    return;
  }
  const char* rowp = (const char*)logits + slot * row_stride * (DT == fg::kBF16 ? 2 : 4);
  uint32_t seq = seq_ids ? (uint32_t)seq_ids[b] : (uint32_t)b;
  uint32_t u = noise_value(noise, (int64_t)b * noise_stride + noise_col0 + walk_step, seed, step, seq,
                           (uint32_t)(draw0 + walk_step));
  int tok = row_sample<DT, G, CUT>(rowp, vocab, sp, u, sh);
  if (threadIdx.x < 64)
    walk_apply(b, tok, parent, tree_tokens, parents, n_nodes, nmax, batch, walk_step, acc_tokens, acc_nodes, acc_stride,
               acc_len, last_node, correction, state, err_flag, next_rows, next_active);
}

// ------------------------------------------------------------------ split sampling
// Unrestricted draws (no top-k / top-p) and greedy draws spread one row over
// kSplitChunks workgroups instead of one. The row maximum and its first maximum
// come as parts: per-chunk parts of split_max_kernel, or the per-workgroup parts
// the LM head writes with the logits (fg_lm_head_topk's row maxima). Then (1) per
// chunk, the q-mass against the row maximum (split_sum_kernel); (2) per row, the
// chunk whose running mass crosses the target and the index inside it
// (split_pick_kernel) -- the same integer rule as block_sample, so the token is
// identical. Greedy draws need only the parts and the pick. The chunk sums are
// handed over at a launch boundary: a device-scope fence per workgroup to hand
// them over inside one launch measured slower than the second launch.
constexpr int kSplitChunks = 16;
constexpr int kSplitThreads = 256;
constexpr int kSplitWaves = kSplitThreads / 64;

struct SplitArgs {
  const void* logits;
  int64_t row_stride;
  int vocab;
  int chunk;                 // elements per chunk (multiple of 8)
  const int32_t* row_index;  // logits row of sampled row r (NULL: r)
  const int32_t* forced;     // rows with forced[r] >= 0 are not sampled
  const int32_t* active;     // rows with active[r] == 0 are not sampled (NULL: all)
  float temperature;
  int scale;
  int greedy;
  float* part_max;           // [rows, kSplitChunks]
  uint64_t* part_key;
  uint64_t* part_sum;
  uint64_t* part_gsum;       // [rows, kSplitChunks, kSplitMaxGroups] q-mass per group of kSplitGroup (top-p: SelState)
  int groups;                // groups per chunk (group sums kept only up to kSplitMaxGroups)
  float* row_m;              // [rows] row maximum (sum launch -> pick launch)
  uint64_t* row_best;        // [rows] first maximum's rank key; restricted draws: bin_shift
  // row maxima parts read by the draw launch: [rows, src_stride], src_parts used
  const float* src_max;
  const uint64_t* src_key;
  int src_parts;
  int64_t src_stride;
  // restricted draws (see "split top-k / top-p")
  int top_k;
  uint32_t tp32;
  uint64_t* hist;            // [rows, kSplitChunks, 256] chunk histograms (q-mass or counts)
  struct SelState* sel;      // [rows]
  uint64_t* part_a;          // [rows, kSplitChunks] q-mass above the cut's bin
  int32_t* part_nan;         // [rows, kSplitChunks] NaN count
  int32_t* part_n;           // the same words: listed candidates (short top-k)
  uint32_t* list;            // [rows, kSelList] indices of the elements around the cut
  int32_t* list_n;           // [rows] listed elements (may exceed kSelList: then not all are there)
};

template <int DT>
FG_DEVICE const char* split_row(const SplitArgs& a, int r) {
  const int64_t src = a.row_index ? a.row_index[r] : r;
  return (const char*)a.logits + src * a.row_stride * (DT == fg::kBF16 ? 2 : 4);
}

FG_DEVICE bool split_skip(const SplitArgs& a, int r) {
  return (a.forced && a.forced[r] >= 0) || (a.active && !a.active[r]);
}

// Elements per workgroup pass: kSplitLoads groups of 8 per thread, all loads in flight
// before the weights are computed (5 groups: a 152,064-logit row's 9,504-element chunk is
// one pass, so a chunk costs one memory round trip).
constexpr int kSplitLoads = 5;
constexpr int kSplitGroup = kSplitThreads * 8;
constexpr int kSplitPass = kSplitGroup * kSplitLoads;
// Per-group q-mass is kept for chunks of up to kSplitMaxGroups groups (vocabularies up to
// 16 x 16 x 2,048 = 524,288): the pick then weighs one group instead of the whole chunk.
constexpr int kSplitMaxGroups = 16;

// Load group u of a pass starting at base (elements base + (u * kSplitThreads + t) * 8 ..
// + 7 of thread t) holds an element before hi. Uniform over the workgroup: a group wholly
// past the chunk end is neither loaded nor weighed (the chunk of a 128,256-logit row, 8,016
// elements, reads four of the kSplitLoads groups).
FG_DEVICE bool split_group_live(int base, int u, int hi) { return base + u * kSplitThreads * 8 < hi; }

// Chunk maxima (raw maximum, NaN ignored, with KEY the first-maximum rank key, without it the least
// logit of each pass's first load group beside it, which bounds bin_shift's range). Per pass a thread
// takes the maximum of its elements (NaN ignored) and then the first index holding it (the
// first NaN when there is one, which ranks highest), and forms one rank key per pass instead
// of one per element.
template <int DT, bool KEY>
__global__ void __launch_bounds__(kSplitThreads) split_max_kernel(SplitArgs a) {
  const int c = blockIdx.x, r = blockIdx.y;
  if (split_skip(a, r)) return;
  __shared__ float smax[kSplitWaves];
  __shared__ uint64_t skey[kSplitWaves];
  const char* p = split_row<DT>(a, r);
  const int lo = c * a.chunk, hi = min(a.vocab, lo + a.chunk);
  float mx = -INFINITY, low = INFINITY;
  uint64_t best = 0;
  for (int base = lo; base < hi; base += kSplitPass) {
    float x[kSplitLoads][8];
#pragma unroll
    for (int u = 0; u < kSplitLoads; ++u)
      if (split_group_live(base, u, hi)) split_load8<DT>(p, base + (u * kSplitThreads + threadIdx.x) * 8, hi, x[u]);
    // the -inf padding past hi never wins: real elements come first and the first index holding
    // the maximum is taken
    float pm = -INFINITY;
    bool nan = false;
#pragma unroll
    for (int u = 0; u < kSplitLoads; ++u) {
      if (!split_group_live(base, u, hi)) continue;
      float low8 = INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pm = fmaxf(pm, x[u][j]);
        if constexpr (KEY) nan |= x[u][j] != x[u][j];
        else if (u == 0) low8 = fminf(low8, x[u][j]);
      }
      if (!KEY && u == 0 && base + (int)threadIdx.x * 8 + 8 <= hi) low = fminf(low, low8);
    }
    if constexpr (!KEY) {
      mx = fmaxf(mx, pm);
      continue;
    }
    int first = -1;
    float kv = pm;
#pragma unroll
    for (int u = kSplitLoads - 1; u >= 0; --u) {
      if (!split_group_live(base, u, hi)) continue;
      const int i0 = base + (u * kSplitThreads + threadIdx.x) * 8;
#pragma unroll
      for (int j = 7; j >= 0; --j) first = (nan ? x[u][j] != x[u][j] : x[u][j] == pm) ? i0 + j : first;
    }
    if (nan) kv = __uint_as_float(0x7fc00000u);
    mx = fmaxf(mx, pm);
    if (first >= 0) {
      const uint64_t k = fg::rank_key(kv, (uint32_t)first);
      best = k > best ? k : best;
    }
  }
  mx = fg::wave_max(mx);
  if constexpr (KEY) best = fg::wave_max_u64(best);
  else best = __float_as_uint(wave_min(low));
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    smax[wave] = mx;
    skey[wave] = best;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kSplitWaves; ++w) {
      mx = fmaxf(mx, smax[w]);
      if constexpr (KEY) best = skey[w] > best ? skey[w] : best;
      else best = __float_as_uint(fminf(__uint_as_float((uint32_t)best), __uint_as_float((uint32_t)skey[w])));
    }
    mx = fmaxf(smax[0], mx);
    if constexpr (KEY) {
      a.part_max[r * kSplitChunks + c] = mx;
      a.part_key[r * kSplitChunks + c] = skey[0] > best ? skey[0] : best;
    } else {
      a.part_key[r * kSplitChunks + c] = (uint64_t)__float_as_uint(mx) << 32 | (uint32_t)best;
    }
  }
}

FG_DEVICE float split_kt(const SplitArgs& a) { return fg::weight_kt(a.scale != 0, a.temperature); }

FG_DEVICE uint64_t split_weight8(const float (&x)[8], float kt, float m, const uint64_t* tbl) {
  uint64_t acc = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) acc += fg::weight_q40(m, x[j], kt, tbl);
  return acc;
}

// Per row: the raw maximum and first maximum from the row's parts (whole block).
FG_DEVICE void split_parts_max(const SplitArgs& a, int r, float* smax, uint64_t* skey, float& mx, uint64_t& best) {
  const int tid = threadIdx.x;
  mx = -INFINITY;
  best = 0;
  for (int q = tid; q < a.src_parts; q += kSplitThreads) {
    mx = fmaxf(mx, a.src_max[r * a.src_stride + q]);
    const uint64_t k = a.src_key[r * a.src_stride + q];
    best = k > best ? k : best;
  }
  mx = fg::wave_max(mx);
  best = fg::wave_max_u64(best);
  if ((tid & 63) == 0) {
    smax[tid >> 6] = mx;
    skey[tid >> 6] = best;
  }
  __syncthreads();
  mx = smax[0];
  best = skey[0];
#pragma unroll
  for (int w = 1; w < kSplitWaves; ++w) {
    mx = fmaxf(mx, smax[w]);
    best = skey[w] > best ? skey[w] : best;
  }
}

// q-mass of each chunk against the row maximum taken from the row's parts; chunk 0 also
// keeps the scaled maximum and the first maximum for the pick launch.
template <int DT>
__global__ void __launch_bounds__(kSplitThreads) split_sum_kernel(SplitArgs a) {
  const int c = blockIdx.x, r = blockIdx.y, tid = threadIdx.x;
  if (split_skip(a, r)) return;
  __shared__ uint64_t tbl[1024];
  __shared__ float smax[kSplitWaves];
  __shared__ uint64_t skey[kSplitWaves];
  __shared__ uint64_t gsum[kSplitMaxGroups];
  const char* p = split_row<DT>(a, r);
  const int lo = c * a.chunk, hi = min(a.vocab, lo + a.chunk);
  // the first pass's logits are in flight while the row maximum is gathered from the parts
  float x[kSplitLoads][8];
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u)
    if (split_group_live(lo, u, hi)) split_load8<DT>(p, lo + (u * kSplitThreads + tid) * 8, hi, x[u]);
  fg::exp2_table_to_lds(tbl);  // visible after the barrier in split_parts_max
  if (tid < kSplitMaxGroups) gsum[tid] = 0;
  float mx;
  uint64_t best;
  split_parts_max(a, r, smax, skey, mx, best);
  const float m = mx, kt = split_kt(a);
  // each group's q-mass: wave sums added into LDS (group g of the chunk = elements
  // [lo + 2048 g, lo + 2048 (g + 1)) = load group g % kSplitLoads of pass g / kSplitLoads)
  const bool keep_groups = a.groups <= kSplitMaxGroups;
  int g = 0;
  for (int base = lo; base < hi; base += kSplitPass) {
    if (base != lo) {
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u)
        if (split_group_live(base, u, hi)) split_load8<DT>(p, base + (u * kSplitThreads + tid) * 8, hi, x[u]);
    }
#pragma unroll
    for (int u = 0; u < kSplitLoads; ++u) {
      if (!split_group_live(base, u, hi)) continue;
      const uint64_t w = fg::wave_sum_u64(split_weight8(x[u], kt, m, tbl));
      if ((tid & 63) == 0) atomicAdd((unsigned long long*)&gsum[keep_groups ? g + u : 0], (unsigned long long)w);
    }
    g += kSplitLoads;
  }
  __syncthreads();
  if (tid == 0) {
    uint64_t t = 0;
    const int ng = keep_groups ? a.groups : 1;
    for (int q = 0; q < ng; ++q) {
      t += gsum[q];
      if (keep_groups) a.part_gsum[((size_t)r * kSplitChunks + c) * kSplitMaxGroups + q] = gsum[q];
    }
    a.part_sum[r * kSplitChunks + c] = t;
    if (c == 0) {
      a.row_m[r] = m;
      a.row_best[r] = best;
    }
  }
}

// Outputs of a draw: a token per row, or one step of the acceptance walk.
struct DrawOut {
  const uint32_t* noise;
  int noise_stride;
  int noise_col;   // walk: noise column noise_col + walk_step
  uint64_t seed, step;
  const int32_t* seq_ids;
  int draw;        // walk: counter draw draw + walk_step
  int32_t* out;    // [rows] (sample mode)
  // walk mode
  const int32_t* tree_tokens;
  const int32_t* parents;
  const int32_t* n_nodes;
  int nmax, batch, walk_step;
  int32_t* acc_tokens;
  int32_t* acc_nodes;
  int acc_stride;
  int32_t* acc_len;
  int32_t* last_node;
  int32_t* correction;
  int32_t* state;
  int32_t* err_flag;
  int32_t* next_rows;    // optional: the next walk step's LM-head rows
  int32_t* next_active;
};

// The draw of each row (one workgroup per row) from the chunk sums of split_sum_kernel
// (greedy draws: from the row's parts alone): the chunk whose running mass crosses the
// target, then the index inside it.
template <int DT, bool WALK>
__global__ void __launch_bounds__(kSplitThreads) split_pick_kernel(SplitArgs a, DrawOut d) {
  const int r = blockIdx.x, tid = threadIdx.x;
  __shared__ uint64_t tbl[1024];
  __shared__ float smax[kSplitWaves];
  __shared__ uint64_t skey[kSplitWaves];
  __shared__ uint64_t wsum[kSplitWaves];
  __shared__ int s_found;
  if constexpr (WALK) {
    if (!d.state[d.batch + r]) return;
  } else {
    if (a.forced && a.forced[r] >= 0) {
      if (tid == 0) d.out[r] = a.forced[r];
      return;
    }
  }
  int tok;
  if (a.greedy) {
    float mx;
    uint64_t best;
    split_parts_max(a, r, smax, skey, mx, best);
    tok = (int)fg::rank_key_index(best);
  } else {
    tok = (int)fg::rank_key_index(a.row_best[r]);
    uint64_t sums[kSplitChunks], total = 0;
#pragma unroll
    for (int q = 0; q < kSplitChunks; ++q) {
      sums[q] = a.part_sum[r * kSplitChunks + q];
      total += sums[q];
    }
    if (total > 0) {
      fg::exp2_table_to_lds(tbl);  // visible after split_locate's first barrier
      const uint32_t seq = d.seq_ids ? (uint32_t)d.seq_ids[r] : (uint32_t)r;
      const int ws = WALK ? d.walk_step : 0;
      const uint32_t u = noise_value(d.noise, (int64_t)r * d.noise_stride + d.noise_col + ws, d.seed, d.step, seq,
                                     (uint32_t)(d.draw + ws));
      const uint64_t target = fg::mulhi_u64_u32(total, u);
      uint64_t before = 0;
      int cs = kSplitChunks - 1;
      for (int q = 0; q < kSplitChunks; ++q) {
        if (before + sums[q] > target) {
          cs = q;
          break;
        }
        before += sums[q];
      }
      int clo = cs * a.chunk, chi = min(a.vocab, clo + a.chunk);
      if (a.groups <= kSplitMaxGroups) {
        // the group of 2,048 whose running mass crosses the target: one group is weighed
        const uint64_t* gs = a.part_gsum + ((size_t)r * kSplitChunks + cs) * kSplitMaxGroups;
        const int ng = (chi - clo + kSplitGroup - 1) / kSplitGroup;
        int q = ng - 1;
        for (int k = 0; k < ng; ++k) {
          if (before + gs[k] > target) {
            q = k;
            break;
          }
          before += gs[k];
        }
        clo += q * kSplitGroup;
        chi = min(chi, clo + kSplitGroup);
      }
      const float m = a.row_m[r], kt = split_kt(a);
      const int idx = split_locate<DT, kSplitThreads, kSplitLoads>(
          split_row<DT>(a, r), clo, chi, [&](float x, int) { return fg::weight_q40(m, x, kt, tbl); }, target - before,
          wsum, &s_found);
      if (idx >= 0) tok = idx;  // always: the chunk holds the target
    }
  }
  if constexpr (WALK) {
    if (tid < 64)
      walk_apply(r, tok, d.state[r], d.tree_tokens, d.parents, d.n_nodes, d.nmax, d.batch, d.walk_step, d.acc_tokens,
                 d.acc_nodes, d.acc_stride, d.acc_len, d.last_node, d.correction, d.state, d.err_flag, d.next_rows,
                 d.next_active);
  } else {
    if (tid == 0) d.out[r] = tok;
  }
}

// ------------------------------------------------------------------ split top-k / top-p
// Restricted draws over kSplitChunks workgroups per row, four launches (two for a short top-k, see
// split_topk_kernel), the same integer rule as block_sample:
//  (1) chunk maxima (split_max_kernel), unless the row's maxima parts are given;
//  (2) per chunk, a histogram over the bins of the fixed-point exponent: q-mass for top-p,
//      counts for top-k;
//  (3) each chunk merges the row's 16 histograms, finds the bin that holds the cut and appends
//      the indices of its own elements of that bin (top-k: of that bin and the ones above) to
//      the row's list;
//  (4) one workgroup per row selects the cut exactly among the list (64-bit rank keys, so ties
//      resolve in index order) and locates the draw: top-k among the list, top-p in the one
//      chunk whose running kept mass crosses the target.
// A row whose list overflows (flat rows) is narrowed further in launch (4) (narrow_cut); one whose total
// is 0 or whose top-k slots are all taken by NaN is drawn by block_sample there.
//
// Bound by VALU and LDS issue of the two weighing passes. An 8-bit radix select over the key
// bits needed four histogram launches instead of one: the first level's 256 bins are the sign
// and exponent bits, so nearly every LDS atomic hit the same few words (17 us per level at
// 64 x 152,064), and a bf16 row's last two levels had nothing left to separate. Measured, a draw:
// top-p 0.95 at 64 x 152,064 bf16 114 -> 50 us (seven launches before).
static_assert(kSelBins == kSplitThreads, "one histogram bin per thread");

// Where the cut of one row lies (written by chunk 0 of launch 3).
struct SelState {
  uint64_t rest;  // position of the cut within the list: q-mass (top-p) or count (top-k) before it
  int32_t slow;   // the row has no weight, or NaN takes every slot: block_sample draws it
  int32_t all;    // every listed element is kept (top-k with no more candidates than slots)
  int32_t bin;    // the cut's bin
  int32_t form;   // bin_shift << 1 | whether part_gsum holds each chunk's least and largest listed key and their count
};

template <int DT, bool COUNT>
__global__ void __launch_bounds__(kSplitThreads) split_hist_kernel(SplitArgs a) {
  const int c = blockIdx.x, r = blockIdx.y, tid = threadIdx.x;
  if (split_skip(a, r)) return;
  using Bin = std::conditional_t<COUNT, uint32_t, uint64_t>;
  using AtomicBin = std::conditional_t<COUNT, unsigned int, unsigned long long>;
  __shared__ uint64_t tbl[COUNT ? 1 : 1024];
  __shared__ Bin h[kSelBins][kCopies];
  __shared__ float smax[kSplitWaves];
  __shared__ int s_nan;
  const char* p = split_row<DT>(a, r);
  const int lo = c * a.chunk, hi = min(a.vocab, lo + a.chunk);
  float x[kSplitLoads][8];
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u)
    if (split_group_live(lo, u, hi)) split_load8<DT>(p, lo + (u * kSplitThreads + tid) * 8, hi, x[u]);
  if constexpr (!COUNT) fg::exp2_table_to_lds(tbl);
#pragma unroll
  for (int q = 0; q < kCopies; ++q) (&h[0][0])[q * kSplitThreads + tid] = 0;
  if (tid == 0) s_nan = 0;
  // row maximum and least logit: this path's own parts hold both, given maxima come without the least
  static_assert(kSplitChunks == 16, "a part per lane of 16");
  float m;
  int shift = kSelBinShift;
  const float kt = split_kt(a);
  if (a.src_max == a.part_max) {
    const uint64_t both = a.part_key[r * kSplitChunks + (tid & (kSplitChunks - 1))];
    m = __uint_as_float((uint32_t)(both >> 32));
    float low = __uint_as_float((uint32_t)both);
#pragma unroll
    for (int o = kSplitChunks / 2; o > 0; o >>= 1) {
      m = fmaxf(m, __shfl_xor(m, o, 64));
      low = fminf(low, __shfl_xor(low, o, 64));
    }
    shift = __builtin_amdgcn_readfirstlane(bin_shift(m, low, kt));
    __syncthreads();
  } else {
    m = -INFINITY;
    for (int q = tid; q < a.src_parts; q += kSplitThreads) m = fmaxf(m, a.src_max[r * a.src_stride + q]);
    m = fg::wave_max(m);
    if ((tid & 63) == 0) smax[tid >> 6] = m;
    __syncthreads();
    m = smax[0];
#pragma unroll
    for (int w = 1; w < kSplitWaves; ++w) m = fmaxf(m, smax[w]);
  }
  Bin* mine = &h[0][tid % kCopies];
  int nan = 0;
  for (int base = lo; base < hi; base += kSplitPass) {
    if (base != lo) {
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u)
        if (split_group_live(base, u, hi)) split_load8<DT>(p, base + (u * kSplitThreads + tid) * 8, hi, x[u]);
    }
#pragma unroll
    for (int u = 0; u < kSplitLoads; ++u) {
      if (!split_group_live(base, u, hi)) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t e = fixed_exponent(m, x[u][j], kt);
        if constexpr (COUNT) nan += x[u][j] != x[u][j];
        if (e <= kSelAMax) {
          const Bin w = COUNT ? (Bin)1 : (Bin)fg::weight_q40(m, x[u][j], kt, tbl);
          atomicAdd((AtomicBin*)&mine[sel_bin(e, shift) * kCopies], (AtomicBin)w);
        }
      }
    }
  }
  if constexpr (COUNT) {
    if (nan) atomicAdd(&s_nan, nan);
  }
  __syncthreads();
  Bin t = 0;
#pragma unroll
  for (int q = 0; q < kCopies; ++q) t += h[tid][q];
  a.hist[((size_t)r * kSplitChunks + c) * kSelBins + tid] = t;
  if (tid == 0) {
    if constexpr (COUNT) a.part_nan[r * kSplitChunks + c] = s_nan;
    if (c == 0) {
      a.list_n[r] = 0;
      a.row_m[r] = m;
      a.row_best[r] = (uint64_t)shift;
    }
  }
}

// Inclusive sum of v over the workgroup's threads in order, and its total.
FG_DEVICE uint64_t split_incl_scan(uint64_t v, uint64_t* wsum, uint64_t& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t incl = fg::wave_incl_scan_u64(v);
  __syncthreads();  // wsum of an earlier scan has been read
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  uint64_t off = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kSplitWaves; ++w) {
    if (w < wave) off += wsum[w];
    total += wsum[w];
  }
  return off + incl;
}

template <int DT, bool COUNT>
__global__ void __launch_bounds__(kSplitThreads) split_gather_kernel(SplitArgs a) {
  const int c = blockIdx.x, r = blockIdx.y, tid = threadIdx.x;
  if (split_skip(a, r)) return;
  __shared__ uint64_t wsum[kSplitWaves];
  __shared__ int s_bin, s_base;
  __shared__ uint64_t s_before, s_mass;
  __shared__ uint32_t s_least, s_most;
  const char* p = split_row<DT>(a, r);
  const int lo = c * a.chunk, hi = min(a.vocab, lo + a.chunk);
  float x[kSplitLoads][8];
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u)
    if (split_group_live(lo, u, hi)) split_load8<DT>(p, lo + (u * kSplitThreads + tid) * 8, hi, x[u]);
  const int shift = (int)a.row_best[r];
  const uint64_t* hp = a.hist + (size_t)r * kSplitChunks * kSelBins;
  uint64_t v = 0, own = 0;
#pragma unroll
  for (int q = 0; q < kSplitChunks; ++q) {
    const uint64_t w = hp[q * kSelBins + tid];
    v += w;
    own = q == c ? w : own;
  }
  uint64_t total;
  const uint64_t incl = split_incl_scan(v, wsum, total);
  // the cut is the candidate position whose running sum first exceeds target
  uint64_t target = 0;
  bool slow = total == 0, all = false;
  if constexpr (COUNT) {
    uint64_t nan = 0;  // NaN ranks first and takes slots
    for (int q = 0; q < kSplitChunks; ++q) nan += (uint64_t)a.part_nan[r * kSplitChunks + q];
    slow |= (uint64_t)a.top_k <= nan;
    const uint64_t slots = slow ? 1 : (uint64_t)a.top_k - nan;
    all = total <= slots;
    target = all ? (total ? total - 1 : 0) : slots - 1;
  } else {
    target = fg::mulhi_u64_u32(total, a.tp32);
  }
  if (tid == 0) s_bin = kSelBins - 1;
  __syncthreads();
  if (incl - v <= target && target < incl) {  // one thread, unless the total is 0
    s_bin = tid;
    s_before = incl - v;
    s_mass = v;
  }
  if (tid == 0) {
    s_least = 0xffffffffu;
    s_most = 0;
  }
  __syncthreads();
  const int bin = s_bin;
  const RowCut rc = bin_cut(bin, shift, 0);
  // top-p: half a list or more in the bin, by its q-mass: is it one value?
  const bool crowded = !COUNT && !slow &&
                       (float)s_mass > (float)(kSelList / 2) * __builtin_amdgcn_exp2f(40.0f - (float)rc.lo * 0x1p-20f);
  if (c == 0 && tid == 0)
    a.sel[r] = SelState{slow ? 0 : COUNT ? target : target - s_before, slow, all, bin, shift << 1 | (int)crowded};
  if (slow) return;
  if constexpr (!COUNT) {  // this chunk's q-mass above the cut's bin
    uint64_t above;
    split_incl_scan(tid < bin ? own : 0, wsum, above);
    if (tid == 0) a.part_a[r * kSplitChunks + c] = above;
  }
  const float m = a.row_m[r], kt = split_kt(a);
  uint32_t* list = a.list + (size_t)r * kSelList;
  uint32_t least = 0xffffffffu, most = 0;  // keys listed here (crowded)
  int listed_here = 0;
  const auto listed = [&](float xv) {
    const uint32_t e = fixed_exponent(m, xv, kt);
    return e < rc.hi && (COUNT || e >= rc.lo);
  };
  for (int base = lo; base < hi; base += kSplitPass) {
    if (base != lo) {
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u)
        if (split_group_live(base, u, hi)) split_load8<DT>(p, base + (u * kSplitThreads + tid) * 8, hi, x[u]);
    }
    uint64_t hit = 0;  // bit 8 u + j: element j of group u is listed
#pragma unroll
    for (int u = 0; u < kSplitLoads; ++u) {
      if (!split_group_live(base, u, hi)) continue;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (listed(x[u][j])) hit |= 1ull << (8 * u + j);
    }
    if (crowded) {
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (hit >> (8 * u + j) & 1) {
            const uint32_t key = fg::sort_key32(x[u][j]);
            least = min(least, key);
            most = max(most, key);
          }
    }
    uint64_t count;
    const int at = (int)split_incl_scan((uint64_t)__popcll(hit), wsum, count) - __popcll(hit);
    listed_here += (int)count;
    if (tid == 0 && count) s_base = atomicAdd(&a.list_n[r], (int)count);
    __syncthreads();
    int o = s_base + at;
    while (hit) {
      const int bit = __builtin_ctzll(hit);
      hit &= hit - 1;
      if (o < kSelList) list[o] = (uint32_t)(base + ((bit >> 3) * kSplitThreads + tid) * 8 + (bit & 7));
      ++o;
    }
  }
  if (crowded) {
    atomicMin(&s_least, least);
    atomicMax(&s_most, most);
    __syncthreads();
    if (tid == 0) {
      uint64_t* info = a.part_gsum + ((size_t)r * kSplitChunks + c) * kSplitMaxGroups;
      info[0] = (uint64_t)s_least << 32 | s_most;
      info[1] = (uint64_t)listed_here;
    }
  }
}

template <int DT, bool COUNT, bool WALK>
__global__ void __launch_bounds__(kThreads) split_select_kernel(SplitArgs a, DrawOut d, SampleParams sp) {
  __shared__ Shared sh;
  __shared__ SelectShared sel;
  __shared__ SmallShared small;
  __shared__ NarrowShared narrow;
  __shared__ uint64_t ck[kSelList];
  __shared__ uint64_t s_kept[kSplitChunks][kCopies];  // kept q-mass per chunk
  const int r = blockIdx.x, tid = threadIdx.x;
  if constexpr (WALK) {
    if (!d.state[d.batch + r]) return;
  } else {
    if (a.forced && a.forced[r] >= 0) {
      if (tid == 0) d.out[r] = a.forced[r];
      return;
    }
  }
  const uint32_t seq = d.seq_ids ? (uint32_t)d.seq_ids[r] : (uint32_t)r;
  const int ws = WALK ? d.walk_step : 0;
  const uint32_t u = noise_value(d.noise, (int64_t)r * d.noise_stride + d.noise_col + ws, d.seed, d.step, seq,
                                 (uint32_t)(d.draw + ws));
  const SelState st = a.sel[r];
  const int n = a.list_n[r];
  const char* rowp = split_row<DT>(a, r);
  const float m = a.row_m[r], kt = split_kt(a);
  const bool flat = n > kSelList;
  bool ok = !st.slow;
  int tok = -1;
  if (ok) {
    fg::exp2_table_to_lds(sh.exp2);
    if (!COUNT && tid < kSplitChunks * kCopies)
      s_kept[tid / kCopies][tid % kCopies] = tid % kCopies || flat ? 0ull : a.part_a[r * kSplitChunks + tid / kCopies];
  }
  if constexpr (COUNT) {
    int64_t slots = st.all ? (int64_t)n : (int64_t)st.rest + 1;
    int listed = n;
    if (ok && flat) {
      RowCut c{0, kSelAMax + 1, 0, (uint64_t)a.top_k, 0, 0};
      ok = narrow_cut<DT, true>(rowp, a.vocab, m, kt, sh.exp2, ck, c, narrow, sel, small);
      slots = (int64_t)a.top_k - c.nan;
      listed = c.n;
    } else if (ok) {
      for (int i = tid; i < n; i += kThreads) {
        const uint32_t idx = a.list[(size_t)r * kSelList + i];
        ck[i] = fg::rank_key(fg::load_elem<DT>(rowp, idx), idx);
      }
    }
    __syncthreads();
    if (ok) tok = list_draw(ck, listed, slots, sp.tp32, u, m, kt, sh.exp2, sel, small);
  } else if (ok) {
    RowCut c = bin_cut(st.bin, st.form >> 1, st.rest);
    const auto kept_weight = [&](float x, int i) -> uint64_t {
      const uint32_t e = fixed_exponent(m, x, kt);
      return e < c.lo || (e < c.hi && fg::rank_key(x, (uint32_t)i) >= c.cut) ? exponent_weight(e, sh.exp2) : 0ull;
    };
    // a flat row whose bin holds one value is cut by index, from the chunks' counts of it
    uint32_t least = 0xffffffffu, most = 0;
    int ties = 0;  // lane l: chunk l's
    if (flat && (st.form & 1)) {
      if ((tid & 63) < kSplitChunks) {
        const uint64_t* info = a.part_gsum + ((size_t)r * kSplitChunks + (tid & 63)) * kSplitMaxGroups;
        ties = (int)info[1];
        if (ties) {
          least = (uint32_t)(info[0] >> 32);
          most = (uint32_t)info[0];
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        least = min(least, (uint32_t)__shfl_xor((int)least, o, 64));
        most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
      }
    }
    if (least == most) {
      __syncthreads();  // sh.exp2
      const float v = fg::rank_key_value((uint64_t)least << 32);
      const uint64_t w = exponent_weight(fixed_exponent(m, v, kt), sh.exp2), last = c.rest / w;
      const uint64_t upto = fg::wave_incl_scan_u64((uint64_t)ties);
      const int c1 = (int)__builtin_ctzll(__ballot(last < upto));  // the chunk of the last kept one
      const uint64_t in1 = last - fg::shfl_u64(upto - (uint64_t)ties, c1);
      const int idx = split_locate<DT, kThreads, 2>(
          rowp, c1 * a.chunk, min(a.vocab, (c1 + 1) * a.chunk),
          [&](float x, int) { return fg::sort_key32(x) == least ? 1ull : 0ull; }, in1, sh.wsum, &sh.i32b[0]);
      c.cut = ((uint64_t)least << 32) | (uint64_t)(0xffffffffu - (uint32_t)idx);
      if (tid < kSplitChunks)
        s_kept[tid][0] = a.part_a[r * kSplitChunks + tid] + w * (tid < c1 ? (uint64_t)ties : tid == c1 ? in1 + 1 : 0ull);
    } else if (flat) {
      ok = narrow_cut<DT, false>(rowp, a.vocab, m, kt, sh.exp2, ck, c, narrow, sel, small);
      if (ok)
        for_row8<DT>(rowp, a.vocab, [&](const float(&x)[8], int i0) {
          uint64_t w = 0;
#pragma unroll
          for (int j = 0; j < 8; ++j) w += kept_weight(x[j], i0 + j);
          if (w) atomicAdd((unsigned long long*)&s_kept[i0 / a.chunk][tid % kCopies], (unsigned long long)w);
        });
    } else {
      for (int i = tid; i < n; i += kThreads) {
        const uint32_t idx = a.list[(size_t)r * kSelList + i];
        ck[i] = fg::rank_key(fg::load_elem<DT>(rowp, idx), idx);
      }
      __syncthreads();
      c.cut = n <= kSmallList ? small_cut(ck, n, c.rest, m, kt, sh.exp2, small)
                              : list_select<true, false>(ck, n, 0, c.rest, m, kt, sh.exp2, sel);
      for (int i = tid; i < n; i += kThreads)
        if (ck[i] >= c.cut)
          atomicAdd((unsigned long long*)&s_kept[fg::rank_key_index(ck[i]) / (uint32_t)a.chunk][tid % kCopies],
                    (unsigned long long)fg::weight_q40(m, fg::rank_key_value(ck[i]), kt, sh.exp2));
    }
    __syncthreads();
    if (ok) {
      // every wave: lane l holds chunk l's kept mass
      uint64_t kept = 0;
      if ((tid & 63) < kSplitChunks)
#pragma unroll
        for (int q = 0; q < kCopies; ++q) kept += s_kept[tid & 63][q];
      const uint64_t incl = fg::wave_incl_scan_u64(kept), target = fg::mulhi_u64_u32(fg::shfl_u64(incl, 63), u);
      const int c2 = (int)__builtin_ctzll(__ballot(target < incl));  // the total exceeds the target
      const uint64_t before = fg::shfl_u64(incl - kept, c2);
      tok = split_locate<DT, kThreads, 2>(rowp, c2 * a.chunk, min(a.vocab, (c2 + 1) * a.chunk), kept_weight,
                                          target - before, sh.wsum, &sh.i32b[0]);
    }
  }
  if (!ok) {
    __syncthreads();
    tok = block_sample<DT>(rowp, a.vocab, sp, u, sh);
  }
  if constexpr (WALK) {
    if (tid < 64)
      walk_apply(r, tok, d.state[r], d.tree_tokens, d.parents, d.n_nodes, d.nmax, d.batch, d.walk_step, d.acc_tokens,
                 d.acc_nodes, d.acc_stride, d.acc_len, d.last_node, d.correction, d.state, d.err_flag, d.next_rows,
                 d.next_active);
  } else {
    if (tid == 0) d.out[r] = tok;
  }
}

// Short top-k (top_k <= kTopkMax, rows of one pass per chunk) in two launches and without the row
// maximum. Each chunk takes the maxima of 512 disjoint sets of its elements (two per thread): the
// top_k-th largest of them bounds the chunk's own top_k-th element from below, and listing the
// elements from there on lists little more than top_k. One workgroup per row draws among the
// lists, dropping first what lies below (a) some chunk's bound or (b) the least of the
// chunks' bounds on their ceil(top_k / 16)-th elements: at least top_k elements of the row lie at
// or above either. Elements 40 octaves below the chunk's maximum and -inf weigh 0 against any
// row maximum and are not listed; NaN, which ranks first, always is. A row with a chunk of more
// than kTopkList candidates (flat rows, long ties) is cut by narrow_cut over the whole row.
// Bound by launch and memory latency: top-k 50 at 32 x 151,936 bf16 took 207 us in one workgroup per
// row, 47 with the four launches above, 25 with these two.
constexpr int kTopkMax = 256;
constexpr int kTopkList = kSelList / kSplitChunks;  // list entries per chunk

template <int DT>
__global__ void __launch_bounds__(kSplitThreads) split_topk_kernel(SplitArgs a) {
  const int c = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, wave = tid >> 6;
  if (split_skip(a, r)) return;
  __shared__ uint32_t h[kSelBins];
  __shared__ float smax[kSplitWaves], smin[kSplitWaves], slow[2][kSplitWaves];
  __shared__ uint64_t wsum[kSplitWaves];
  __shared__ int s_bin[2];
  const char* p = split_row<DT>(a, r);
  const int lo = c * a.chunk, hi = min(a.vocab, lo + a.chunk);
  float x[kSplitLoads][8];
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u)
    if (split_group_live(lo, u, hi)) split_load8<DT>(p, lo + (u * kSplitThreads + tid) * 8, hi, x[u]);
  h[tid] = 0;
  if (tid < 2) s_bin[tid] = kSelBins;
  float sm[2] = {-INFINITY, -INFINITY};  // maxima of this thread's two sets
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u) {
    if (!split_group_live(lo, u, hi)) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) sm[j >> 2] = fmaxf(sm[j >> 2], x[u][j]);
  }
  float m = fg::wave_max(fmaxf(sm[0], sm[1])), low = wave_min(fminf(above_inf(sm[0]), above_inf(sm[1])));
  if ((tid & 63) == 0) {
    smax[wave] = m;
    smin[wave] = low;
  }
  __syncthreads();
  m = smax[0];
  low = smin[0];
#pragma unroll
  for (int w = 1; w < kSplitWaves; ++w) {
    m = fmaxf(m, smax[w]);
    low = fminf(low, smin[w]);
  }
  const float kt = split_kt(a);
  const int shift = bin_shift(m, low, kt);
  // bin of a set's maximum, kSelBins for one that weighs 0 against any maximum from m on
  int sb[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t e = fixed_exponent(m, sm[q], kt);
    sb[q] = e <= kSelAMax ? sel_bin(e, shift) : kSelBins;
    if (sb[q] < kSelBins) atomicAdd(&h[sb[q]], 1u);
  }
  __syncthreads();
  const uint64_t v = h[tid];
  uint64_t total;
  const uint64_t incl = split_incl_scan(v, wsum, total);
  const uint64_t want[2] = {(uint64_t)a.top_k, (uint64_t)((a.top_k + kSplitChunks - 1) / kSplitChunks)};
#pragma unroll
  for (int q = 0; q < 2; ++q)
    if (incl - v < want[q] && want[q] <= incl) s_bin[q] = tid;  // none when there are fewer sets with weight
  __syncthreads();
  // the least set maximum in the bins up to that one: at least want[q] elements reach it
  float t[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float l = INFINITY;
#pragma unroll
    for (int k = 0; k < 2; ++k) l = sb[k] <= s_bin[q] && sb[k] < kSelBins ? fminf(l, sm[k]) : l;
    l = -fg::wave_max(-l);
    if ((tid & 63) == 0) slow[q][wave] = l;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    t[q] = slow[q][0];
#pragma unroll
    for (int w = 1; w < kSplitWaves; ++w) t[q] = fminf(t[q], slow[q][w]);
    if (s_bin[q] == kSelBins) t[q] = -INFINITY;
  }
  uint64_t hit = 0;  // listed elements
#pragma unroll
  for (int u = 0; u < kSplitLoads; ++u) {
    if (!split_group_live(lo, u, hi)) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float xv = x[u][j];
      if (xv != xv || (xv >= t[0] && fixed_exponent(m, xv, kt) <= kSelAMax)) hit |= 1ull << (8 * u + j);
    }
  }
  uint64_t count;
  int o = (int)split_incl_scan((uint64_t)__popcll(hit), wsum, count) - __popcll(hit);
  const size_t at = ((size_t)r * kSplitChunks + c) * kTopkList;
  for (; hit; hit &= hit - 1, ++o) {
    const int bit = __builtin_ctzll(hit);
    const int i = lo + ((bit >> 3) * kSplitThreads + tid) * 8 + (bit & 7);
    if (o < kTopkList) a.list[at + o] = (uint32_t)i;
  }
  if (tid == 0) {
    a.part_n[r * kSplitChunks + c] = (int32_t)count;
    a.part_key[r * kSplitChunks + c] = ((uint64_t)fg::sort_key32(t[0]) << 32) | fg::sort_key32(t[1]);
    a.part_max[r * kSplitChunks + c] = m;
  }
}

template <int DT, bool WALK>
__global__ void __launch_bounds__(kThreads) split_topk_draw_kernel(SplitArgs a, DrawOut d, SampleParams sp) {
  static_assert(kWaves == kSplitChunks, "one wave per chunk list");
  __shared__ Shared sh;
  __shared__ SelectShared sel;
  __shared__ SmallShared small;
  __shared__ NarrowShared narrow;
  __shared__ uint64_t ck[kSelList];
  __shared__ int s_n;
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, c = tid >> 6;
  if constexpr (WALK) {
    if (!d.state[d.batch + r]) return;
  } else {
    if (a.forced && a.forced[r] >= 0) {
      if (tid == 0) d.out[r] = a.forced[r];
      return;
    }
  }
  const char* rowp = split_row<DT>(a, r);
  const size_t at = ((size_t)r * kSplitChunks + c) * kTopkList;
  uint32_t idx = a.list[at + lane];  // the first entries, before their count is known
  const int mine = a.part_n[r * kSplitChunks + c];
  const uint32_t seq = d.seq_ids ? (uint32_t)d.seq_ids[r] : (uint32_t)r;
  const int ws = WALK ? d.walk_step : 0;
  const uint32_t u = noise_value(d.noise, (int64_t)r * d.noise_stride + d.noise_col + ws, d.seed, d.step, seq,
                                 (uint32_t)(d.draw + ws));
  float m = lane < kSplitChunks ? a.part_max[r * kSplitChunks + lane] : -INFINITY;
  const uint64_t bounds = a.part_key[r * kSplitChunks + (lane & (kSplitChunks - 1))];
  m = fg::wave_max(m);
  uint32_t hi_key = (uint32_t)(bounds >> 32), lo_key = (uint32_t)bounds;
#pragma unroll
  for (int q = kSplitChunks / 2; q > 0; q >>= 1) {
    hi_key = max(hi_key, (uint32_t)__shfl_xor((int)hi_key, q, 64));
    lo_key = min(lo_key, (uint32_t)__shfl_xor((int)lo_key, q, 64));
  }
  const uint64_t floor = (uint64_t)max(hi_key, lo_key) << 32;
  fg::exp2_table_to_lds(sh.exp2);
  if (tid == 0) s_n = 0;
  const bool full = __syncthreads_or(mine > kTopkList) != 0;
  if (!full)
    for (int o = lane;;) {
      const uint64_t key = o < mine ? fg::rank_key(fg::load_elem<DT>(rowp, idx), idx) : 0ull;
      const bool in = o < mine && key >= floor;
      const uint64_t mask = __ballot(in);
      int base = 0;
      if (lane == 0 && mask) base = atomicAdd(&s_n, (int)__popcll(mask));
      base = __shfl(base, 0, 64);
      if (in) ck[base + (int)__popcll(mask & ((1ull << lane) - 1))] = key;
      o += 64;
      if (o - lane >= mine) break;  // wave-uniform
      idx = a.list[at + min(o, kTopkList - 1)];
    }
  __syncthreads();
  int tok = -1;
  int n = s_n;
  int64_t slots = sp.top_k;
  if (full) {
    RowCut c2{0, kSelAMax + 1, 0, (uint64_t)sp.top_k, 0, 0};
    n = narrow_cut<DT, true>(rowp, a.vocab, m, split_kt(a), sh.exp2, ck, c2, narrow, sel, small) ? c2.n : 0;
    slots -= c2.nan;
  }
  if (n > 0) tok = list_draw(ck, n, slots, sp.tp32, u, m, split_kt(a), sh.exp2, sel, small);
  __syncthreads();
  if (tok < 0) tok = block_sample<DT>(rowp, a.vocab, sp, u, sh);
  if constexpr (WALK) {
    if (tid < 64)
      walk_apply(r, tok, d.state[r], d.tree_tokens, d.parents, d.n_nodes, d.nmax, d.batch, d.walk_step, d.acc_tokens,
                 d.acc_nodes, d.acc_stride, d.acc_len, d.last_node, d.correction, d.state, d.err_flag, d.next_rows,
                 d.next_active);
  } else {
    if (tid == 0) d.out[r] = tok;
  }
}

template <int DT, bool COUNT, bool WALK>
void split_select_launch(const SplitArgs& a, const DrawOut& d, const SampleParams& sp, int rows, bool with_max,
                         hipStream_t s) {
  const dim3 grid(kSplitChunks, rows), block(kSplitThreads);
  if (COUNT && sp.top_k <= kTopkMax && a.chunk <= kSplitPass) {
    hipLaunchKernelGGL(split_topk_kernel<DT>, grid, block, 0, s, a);
    hipLaunchKernelGGL((split_topk_draw_kernel<DT, WALK>), dim3(rows), dim3(kThreads), 0, s, a, d, sp);
    return;
  }
  if (with_max) hipLaunchKernelGGL((split_max_kernel<DT, false>), grid, block, 0, s, a);
  hipLaunchKernelGGL((split_hist_kernel<DT, COUNT>), grid, block, 0, s, a);
  hipLaunchKernelGGL((split_gather_kernel<DT, COUNT>), grid, block, 0, s, a);
  hipLaunchKernelGGL((split_select_kernel<DT, COUNT, WALK>), dim3(rows), dim3(kThreads), 0, s, a, d, sp);
}

// A draw with a top-k and / or top-p cut.
template <bool WALK>
void split_select(int dtype, const SplitArgs& a, const DrawOut& d, const SampleParams& sp, int rows, bool with_max,
                  hipStream_t s) {
  if (dtype == fg::kBF16) {
    if (sp.top_k) split_select_launch<fg::kBF16, true, WALK>(a, d, sp, rows, with_max, s);
    else split_select_launch<fg::kBF16, false, WALK>(a, d, sp, rows, with_max, s);
  } else {
    if (sp.top_k) split_select_launch<fg::kF32, true, WALK>(a, d, sp, rows, with_max, s);
    else split_select_launch<fg::kF32, false, WALK>(a, d, sp, rows, with_max, s);
  }
}

// A split draw: the chunk maxima unless a.src_* already hold row maxima parts, the
// chunk sums (not for greedy draws), the pick (1 to 3 launches).
template <int DT, bool WALK>
void split_draw(const SplitArgs& a, const DrawOut& d, int rows, bool with_max, hipStream_t s) {
  if (with_max)
    hipLaunchKernelGGL((split_max_kernel<DT, true>), dim3(kSplitChunks, rows), dim3(kSplitThreads), 0, s, a);
  if (!a.greedy) hipLaunchKernelGGL(split_sum_kernel<DT>, dim3(kSplitChunks, rows), dim3(kSplitThreads), 0, s, a);
  hipLaunchKernelGGL((split_pick_kernel<DT, WALK>), dim3(rows), dim3(kSplitThreads), 0, s, a, d);
}

// Scratch of unrestricted and greedy draws, and of restricted ones on top of it.
constexpr size_t split_base_bytes(int rows) {
  return (size_t)rows * (kSplitChunks * (4 + 8 + 8) + (8 + 4) + kSplitChunks * kSplitMaxGroups * 8) + 256;
}
constexpr size_t split_workspace_bytes(int rows) {
  return split_base_bytes(rows) + (size_t)rows * (kSplitChunks * (kSelBins * 8 + 8 + 4) + sizeof(SelState) +
                                                  kSelList * 4 + 4) + 64;
}

// Scratch of fg_sample_tokens_noalloc: the split partials of up to
// kNoAllocMaxRows rows (17.5 MB per device, held until the process ends). Each
// kernel of the split paths writes every partial it owns before a later launch
// reads it, so nothing in it has to start at zero. Host code never hands
// `scratch` itself to a kernel (in host code the name is only a stand-in): it
// passes the per-device address that hipGetSymbolAddress returns.
constexpr int kNoAllocMaxRows = 256;
constexpr size_t kScratchBytes = split_workspace_bytes(kNoAllocMaxRows);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per device.
int scratch_for_current_device(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fg::fail("fg_sample_tokens_noalloc: no current HIP device");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fg::fail(std::string("fg_sample_tokens_noalloc: hipGetSymbolAddress(scratch) failed: ") +
                      hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

// Carves the split partials out of a caller workspace; false when it is too small (restricted
// draws need more than the others).
bool split_setup(SplitArgs& a, void* workspace, size_t bytes, int rows, const void* logits, int64_t row_stride,
                 int vocab, float temperature, const SampleParams& sp) {
  const bool cut = sp.cut();
  if (sp.top_k > kSelTopK && cut) return false;
  if (!workspace || bytes < (cut ? split_workspace_bytes(rows) : split_base_bytes(rows))) return false;
  char* w = (char*)(((uintptr_t)workspace + 15) & ~(uintptr_t)15);
  const size_t chunks = (size_t)rows * kSplitChunks;
  a.part_key = (uint64_t*)w;
  a.part_sum = a.part_key + chunks;
  a.row_best = a.part_sum + chunks;
  a.part_gsum = a.row_best + rows;
  a.part_max = (float*)(a.part_gsum + chunks * kSplitMaxGroups);
  a.row_m = a.part_max + chunks;
  w = (char*)(((uintptr_t)(a.row_m + rows) + 15) & ~(uintptr_t)15);
  a.hist = cut ? (uint64_t*)w : nullptr;
  a.part_a = cut ? a.hist + chunks * kSelBins : nullptr;
  a.sel = cut ? (SelState*)(a.part_a + chunks) : nullptr;
  a.part_nan = cut ? (int32_t*)(a.sel + rows) : nullptr;
  a.part_n = a.part_nan;
  a.list = cut ? (uint32_t*)(a.part_nan + chunks) : nullptr;
  a.list_n = cut ? (int32_t*)(a.list + (size_t)rows * kSelList) : nullptr;
  a.src_max = a.part_max;
  a.src_key = a.part_key;
  a.src_parts = kSplitChunks;
  a.src_stride = kSplitChunks;
  a.top_k = sp.top_k;
  a.tp32 = sp.tp32;
  a.logits = logits;
  a.row_stride = row_stride;
  a.vocab = vocab;
  a.chunk = ((vocab + kSplitChunks - 1) / kSplitChunks + 7) / 8 * 8;
  a.groups = (a.chunk + kSplitGroup - 1) / kSplitGroup;
  a.temperature = temperature;
  a.greedy = sp.greedy;
  a.scale = !a.greedy && temperature > 0.0f && temperature != 1.0f;
  a.row_index = nullptr;
  a.forced = nullptr;
  a.active = nullptr;
  return true;
}

// Length clamp, EOS cut, finished flag and the b200 pending root.
// Follows flashgrpo/decoding/flash_medusa_decoder.py:899-922 and
// flashgrpo_b200/decoding/flash_medusa_decoder.py:2303-2319.
__global__ void accept_finalize_kernel(const int32_t* __restrict__ acc_tokens, const int32_t* __restrict__ acc_nodes,
                                       int acc_stride, int32_t* acc_len, int32_t* last_node,
                                       const int32_t* __restrict__ correction, const int32_t* __restrict__ old_len,
                                       int max_length, int eos_token_id, int32_t* finished, int32_t* pending_root,
                                       int batch) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  const int raw = acc_len[b];
  int keep = max(1, max_length - old_len[b]);
  int len = min(raw, keep);
  int eos = 0;
  if (eos_token_id >= 0) {
    for (int j = 0; j < len; ++j)
      if (acc_tokens[(int64_t)b * acc_stride + j] == eos_token_id) {
        len = j + 1;
        eos = 1;
        break;
      }
  }
  acc_len[b] = len;
  last_node[b] = acc_nodes[(int64_t)b * acc_stride + len - 1];
  int fin = eos || old_len[b] + len >= max_length;
  finished[b] = fin;
  if (pending_root) pending_root[b] = (correction[b] >= 0 && len == raw && !fin) ? correction[b] : -1;
}

SampleParams make_params(float temperature, int greedy, int top_k, int vocab, uint32_t tp32) {
  SampleParams sp;
  sp.temperature = temperature;
  sp.greedy = greedy || temperature == 0.0f;
  sp.top_k = (top_k > 0 && top_k < vocab) ? top_k : 0;
  sp.tp32 = tp32;
  return sp;
}

// Where a draw runs, the one rule: in one workgroup per row that holds `groups` x 8,192 logits in registers
// (resident_sample), else over the split launches, which need the workspace, else in block_sample. `maxima`:
// the row maxima parts are given. us on bf16 rows at each line:
//  * greedy draws read each logit once and weigh none. Given maxima make them one launch that reads no logit
//    (64 x 32,000: 2.5, resident 7.5). Otherwise split from 8,193 logits (8 x 32,000: 6.3, resident 8.1, block 8.7;
//    64 x 512: split 7.0, block 5.2), up to 32,768 of them for at most 128 rows (256 x 32,000: 10.9 and 9.0).
//  * a top_k over kSelTopK overfills the list: block_sample alone (8 x 32,000, top_k 5,000: 55, 70 after a
//    resident histogram).
//  * up to 8,192 logits one group, up to 16,384 two, up to 32,768 four: the padding is weighed too (64 x 512: one
//    group 6.3, four 9.8, block_sample 7.6; top-p 11.4 and 16.1).
//  * up to 65,536 without a cut eight from kLongRows rows on, or from kLongRowsMaxima with given maxima, when the
//    split draw is two launches (65,536: 8 rows split 13.9 and resident 14.1, 64 rows 17.0 and 14.6, 512 59 and
//    34; with maxima 64 rows 11.3 and 14.0, 256 25.8 and 16.5). With a cut the weighing passes are two and the
//    split launches win (64 x 65,536, top-p: 59.7 and 41.6).
struct DrawPath {
  int groups;
  bool split;
};
constexpr int kLongRows = 16, kLongRowsMaxima = 128;
DrawPath draw_path(int vocab, const SampleParams& sp, int rows, bool workspace, bool maxima) {
  if (sp.greedy) return {0, workspace && (maxima || vocab > 8192 * 4 || (vocab > 8192 && rows <= 128))};
  if (sp.top_k > kSelTopK) return {0, false};
  if (vocab <= 8192 * 4) return {vocab <= 8192 ? 1 : vocab <= 8192 * 2 ? 2 : 4, false};
  const bool whole = vocab <= 8192 * 8 && !sp.cut() && (!workspace || rows >= (maxima ? kLongRowsMaxima : kLongRows));
  return {whole ? 8 : 0, workspace && !whole};
}

// f(dtype, groups, Cut), each an integral constant, for the one-workgroup-per-row kernels.
template <class F>
void for_row_kernel(int dtype, int path_groups, const SampleParams& sp, F&& f) {
  const auto types = [&](auto dt) {
    const auto cuts = [&](auto g) {
      if (!sp.cut()) f(dt, g, std::integral_constant<int, kNoCut>{});
      else if (sp.top_k) f(dt, g, std::integral_constant<int, kTopK>{});
      else f(dt, g, std::integral_constant<int, kTopP>{});
    };
    switch (path_groups) {
      case 1: cuts(std::integral_constant<int, 1>{}); break;
      case 2: cuts(std::integral_constant<int, 2>{}); break;
      case 4: cuts(std::integral_constant<int, 4>{}); break;
      case 8: f(dt, std::integral_constant<int, 8>{}, std::integral_constant<int, kNoCut>{}); break;
      default: f(dt, std::integral_constant<int, 0>{}, std::integral_constant<int, kNoCut>{}); break;
    }
  };
  if (dtype == fg::kBF16) types(std::integral_constant<int, fg::kBF16>{});
  else types(std::integral_constant<int, fg::kF32>{});
}

int sample_tokens_impl(const char* who, const void* logits, int dtype, int64_t row_stride, int rows, int vocab,
                       const int32_t* row_index, const int32_t* forced, const uint32_t* noise,
                       int noise_stride, int noise_col, uint64_t seed, uint64_t step,
                       const int32_t* seq_ids, int draw, float temperature, int greedy, int top_k,
                       uint32_t top_p_fixed, int32_t* out_tokens, void* workspace,
                       size_t workspace_bytes, void* stream) {
  FG_REQUIRE(logits && out_tokens, std::string(who) + ": null pointer");
  FG_REQUIRE(rows > 0 && vocab > 0 && vocab < (1 << 23), std::string(who) + ": vocab must be in [1, 2^23)");
  FG_REQUIRE(dtype == fg::kF32 || dtype == fg::kBF16, std::string(who) + ": dtype");
  FG_REQUIRE(row_stride >= vocab && row_stride % 8 == 0 && ((uintptr_t)logits & 31) == 0,
             std::string(who) + ": rows must be 32-byte aligned (row_stride % 8 == 0)");
  SampleParams sp = make_params(temperature, greedy, top_k, vocab, top_p_fixed);
  hipStream_t s = (hipStream_t)stream;
  SplitArgs a;
  const bool scratch = split_setup(a, workspace, workspace_bytes, rows, logits, row_stride, vocab, temperature, sp);
  const DrawPath path = draw_path(vocab, sp, rows, scratch, false);
  if (path.split) {
    a.row_index = row_index;
    a.forced = forced;
    DrawOut d{};
    d.noise = noise; d.noise_stride = noise_stride; d.noise_col = noise_col;
    d.seed = seed; d.step = step; d.seq_ids = seq_ids; d.draw = draw; d.out = out_tokens;
    if (sp.cut()) split_select<false>(dtype, a, d, sp, rows, true, s);
    else if (dtype == fg::kBF16) split_draw<fg::kBF16, false>(a, d, rows, true, s);
    else split_draw<fg::kF32, false>(a, d, rows, true, s);
    return fg::check_launch(who);
  }
  for_row_kernel(dtype, path.groups, sp, [&](auto dt, auto g, auto cut) {
    hipLaunchKernelGGL((sample_rows_kernel<decltype(dt)::value, decltype(g)::value, decltype(cut)::value>),
                       dim3(rows), dim3(kThreads), 0, s,
                       logits, row_stride, vocab, row_index, forced, noise, noise_stride, noise_col, seed, step,
                       seq_ids, draw, sp, out_tokens);
  });
  return fg::check_launch(who);
}

}  // namespace

extern "C" {

size_t fg_sample_workspace(int rows) { return rows > 0 ? split_workspace_bytes(rows) : 0; }

int fg_sample_tokens(const void* logits, int dtype, int64_t row_stride, int rows, int vocab,
                     const int32_t* row_index, const int32_t* forced, const uint32_t* noise, int noise_stride,
                     int noise_col, uint64_t seed, uint64_t step, const int32_t* seq_ids, int draw,
                     float temperature, int greedy, int top_k, uint32_t top_p_fixed, int32_t* out_tokens,
                     void* workspace, size_t workspace_bytes, void* stream) {
  return sample_tokens_impl("fg_sample_tokens", logits, dtype, row_stride, rows, vocab, row_index, forced, noise,
                            noise_stride, noise_col, seed, step, seq_ids, draw, temperature, greedy, top_k,
                            top_p_fixed, out_tokens, workspace, workspace_bytes, stream);
}

size_t fg_sample_tokens_noalloc_max_rows(void) { return kNoAllocMaxRows; }

int fg_sample_tokens_noalloc(const void* logits, int dtype, int64_t row_stride, int rows, int vocab,
                             const int32_t* row_index, const int32_t* forced, const uint32_t* noise,
                             int noise_stride, int noise_col, uint64_t seed, uint64_t step, const int32_t* seq_ids,
                             int draw, float temperature, int greedy, int top_k, uint32_t top_p_fixed,
                             int32_t* out_tokens, void* stream) {
  FG_REQUIRE(rows > 0 && rows <= kNoAllocMaxRows,
             "fg_sample_tokens_noalloc: rows must be in [1, " + std::to_string(kNoAllocMaxRows) + "] (got " +
                 std::to_string(rows) + ")");
  void* ws = nullptr;
  if (int rc = scratch_for_current_device(&ws)) return rc;
  return sample_tokens_impl("fg_sample_tokens_noalloc", logits, dtype, row_stride, rows, vocab, row_index, forced,
                            noise, noise_stride, noise_col, seed, step, seq_ids, draw, temperature, greedy, top_k,
                            top_p_fixed, out_tokens, ws, kScratchBytes, stream);
}

int fg_accept_walk(const void* tree_logits, int dtype, int64_t row_stride, int vocab, const int32_t* slot_map,
                   const int32_t* tree_tokens, const int32_t* parents, const int32_t* n_nodes, int nmax, int batch,
                   int max_walk_steps, const uint32_t* noise, int noise_stride, int noise_col0, uint64_t seed,
                   uint64_t step, const int32_t* seq_ids, int draw0, float temperature, int greedy, int top_k,
                   uint32_t top_p_fixed, int32_t* acc_tokens, int32_t* acc_nodes, int acc_stride, int32_t* acc_len,
                   int32_t* last_node, int32_t* correction, int32_t* workspace, int32_t* err_flag, void* stream) {
  FG_REQUIRE(tree_logits && tree_tokens && parents && n_nodes && acc_tokens && acc_nodes && acc_len && last_node &&
                 correction && workspace,
             "fg_accept_walk: null pointer");
  FG_REQUIRE(batch > 0 && nmax > 0 && nmax <= 64 && vocab > 0 && vocab < (1 << 23), "fg_accept_walk: bad shape");
  FG_REQUIRE(acc_stride >= 1 && max_walk_steps >= 0, "fg_accept_walk: bad acc_stride / steps");
  FG_REQUIRE(dtype == fg::kF32 || dtype == fg::kBF16, "fg_accept_walk: dtype");
  FG_REQUIRE(row_stride >= vocab && row_stride % 8 == 0 && ((uintptr_t)tree_logits & 31) == 0,
             "fg_accept_walk: rows must be 32-byte aligned (row_stride % 8 == 0)");
  SampleParams sp = make_params(temperature, greedy, top_k, vocab, top_p_fixed);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(walk_init_kernel, dim3((batch + 63) / 64), dim3(64), 0, s, tree_tokens, parents, n_nodes, nmax,
                     batch, acc_tokens, acc_nodes, acc_stride, acc_len, last_node, correction, workspace);
  for (int t = 0; t < max_walk_steps; ++t) {
    for_row_kernel(dtype, draw_path(vocab, sp, batch, false, false).groups, sp, [&](auto dt, auto g, auto cut) {
      hipLaunchKernelGGL((walk_step_kernel<decltype(dt)::value, decltype(g)::value, decltype(cut)::value>),
                         dim3(batch), dim3(kThreads), 0, s,
                         tree_logits, row_stride, vocab, slot_map, tree_tokens, parents, n_nodes, nmax, batch, t, 0,
                         noise, noise_stride, noise_col0, seed, step, seq_ids, draw0, sp, acc_tokens, acc_nodes,
                         acc_stride, acc_len, last_node, correction, workspace, err_flag, nullptr, nullptr);
    });
  }
  return fg::check_launch("fg_accept_walk");
}

int fg_walk_begin(const int32_t* tree_tokens, const int32_t* parents, const int32_t* n_nodes, int nmax, int batch,
                  int32_t* acc_tokens, int32_t* acc_nodes, int acc_stride, int32_t* acc_len, int32_t* last_node,
                  int32_t* correction, int32_t* state, void* stream) {
  FG_REQUIRE(tree_tokens && parents && n_nodes && acc_tokens && acc_nodes && acc_len && last_node && correction &&
                 state,
             "fg_walk_begin: null pointer");
  FG_REQUIRE(batch > 0 && nmax > 0 && nmax <= 64 && acc_stride >= 1, "fg_walk_begin: bad shape");
  hipLaunchKernelGGL(walk_init_kernel, dim3((batch + 63) / 64), dim3(64), 0, (hipStream_t)stream, tree_tokens,
                     parents, n_nodes, nmax, batch, acc_tokens, acc_nodes, acc_stride, acc_len, last_node, correction,
                     state);
  return fg::check_launch("fg_walk_begin");
}

int fg_walk_rows(const int32_t* state, int batch, int nmax, int32_t* row_index, int32_t* row_active, void* stream) {
  FG_REQUIRE(state && row_index && row_active && batch > 0 && nmax > 0, "fg_walk_rows: bad arguments");
  hipLaunchKernelGGL(walk_rows_kernel, dim3((batch + 63) / 64), dim3(64), 0, (hipStream_t)stream, state, batch, nmax,
                     row_index, row_active);
  return fg::check_launch("fg_walk_rows");
}

int fg_walk_step(const void* step_logits, int dtype, int64_t row_stride, int vocab, const int32_t* tree_tokens,
                 const int32_t* parents, const int32_t* n_nodes, int nmax, int batch, int walk_step,
                 const uint32_t* noise, int noise_stride, int noise_col0, uint64_t seed, uint64_t step,
                 const int32_t* seq_ids, int draw0, float temperature, int greedy, int top_k, uint32_t top_p_fixed,
                 int32_t* acc_tokens, int32_t* acc_nodes, int acc_stride, int32_t* acc_len, int32_t* last_node,
                 int32_t* correction, int32_t* state, int32_t* err_flag, const float* part_max,
                 const uint64_t* part_key, int nparts, int32_t* next_row_index, int32_t* next_row_active,
                 void* workspace, size_t workspace_bytes, void* stream) {
  FG_REQUIRE(step_logits && tree_tokens && parents && n_nodes && acc_tokens && acc_nodes && acc_len && last_node &&
                 correction && state,
             "fg_walk_step: null pointer");
  FG_REQUIRE(batch > 0 && nmax > 0 && nmax <= 64 && vocab > 0 && vocab < (1 << 23) && walk_step >= 0,
             "fg_walk_step: bad shape");
  FG_REQUIRE(dtype == fg::kF32 || dtype == fg::kBF16, "fg_walk_step: dtype");
  FG_REQUIRE(row_stride >= vocab && row_stride % 8 == 0 && ((uintptr_t)step_logits & 31) == 0,
             "fg_walk_step: rows must be 32-byte aligned (row_stride % 8 == 0)");
  FG_REQUIRE(!part_max == !part_key && (!part_max || nparts > 0), "fg_walk_step: part_max / part_key / nparts");
  FG_REQUIRE(!next_row_index == !next_row_active, "fg_walk_step: next_row_index and next_row_active go together");
  SampleParams sp = make_params(temperature, greedy, top_k, vocab, top_p_fixed);
  hipStream_t s = (hipStream_t)stream;
  SplitArgs a;
  const bool scratch = split_setup(a, workspace, workspace_bytes, batch, step_logits, row_stride, vocab, temperature, sp);
  const DrawPath path = draw_path(vocab, sp, batch, scratch, part_max != nullptr);
  if (path.split) {
    a.active = state + batch;
    const bool with_max = part_max == nullptr;
    if (!with_max) {
      a.src_max = part_max;
      a.src_key = part_key;
      a.src_parts = nparts;
      a.src_stride = nparts;
    }
    DrawOut d{};
    d.noise = noise; d.noise_stride = noise_stride; d.noise_col = noise_col0;
    d.seed = seed; d.step = step; d.seq_ids = seq_ids; d.draw = draw0;
    d.tree_tokens = tree_tokens; d.parents = parents; d.n_nodes = n_nodes;
    d.nmax = nmax; d.batch = batch; d.walk_step = walk_step;
    d.acc_tokens = acc_tokens; d.acc_nodes = acc_nodes; d.acc_stride = acc_stride; d.acc_len = acc_len;
    d.last_node = last_node; d.correction = correction; d.state = state; d.err_flag = err_flag;
    d.next_rows = next_row_index; d.next_active = next_row_active;
    if (sp.cut()) split_select<true>(dtype, a, d, sp, batch, with_max, s);
    else if (dtype == fg::kBF16) split_draw<fg::kBF16, true>(a, d, batch, with_max, s);
    else split_draw<fg::kF32, true>(a, d, batch, with_max, s);
    return fg::check_launch("fg_walk_step");
  }
  for_row_kernel(dtype, path.groups, sp, [&](auto dt, auto g, auto cut) {
    hipLaunchKernelGGL((walk_step_kernel<decltype(dt)::value, decltype(g)::value, decltype(cut)::value>),
                       dim3(batch), dim3(kThreads), 0, s,
                       step_logits, row_stride, vocab, nullptr, tree_tokens, parents, n_nodes, nmax, batch, walk_step, 1,
                       noise, noise_stride, noise_col0, seed, step, seq_ids, draw0, sp, acc_tokens, acc_nodes,
                       acc_stride, acc_len, last_node, correction, state, err_flag, next_row_index, next_row_active);
  });
  return fg::check_launch("fg_walk_step");
}

int fg_accept_finalize(const int32_t* acc_tokens, const int32_t* acc_nodes, int acc_stride, int32_t* acc_len,
                       int32_t* last_node, const int32_t* correction, const int32_t* old_len, int max_length,
                       int eos_token_id, int32_t* finished, int32_t* pending_root, int batch, void* stream) {
  FG_REQUIRE(acc_tokens && acc_nodes && acc_len && last_node && correction && old_len && finished,
             "fg_accept_finalize: null pointer");
  FG_REQUIRE(batch > 0 && acc_stride >= 1, "fg_accept_finalize: bad shape");
  hipLaunchKernelGGL(accept_finalize_kernel, dim3((batch + 63) / 64), dim3(64), 0, (hipStream_t)stream, acc_tokens,
                     acc_nodes, acc_stride, acc_len, last_node, correction, old_len, max_length, eos_token_id,
                     finished, pending_root, batch);
  return fg::check_launch("fg_accept_finalize");
}

}  // extern "C"
