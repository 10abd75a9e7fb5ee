// vs_sample.h - what the sampling kernels share (vs_sample.hip, vs_batch.hip): the workspace layout of a row, the
// kernel arguments, LDS histograms and sorts, the draw of Sampler.sample on a sorted list, and the readers of the
// penalty counts.
#pragma once
#include "vs_common.h"
#include "vs_host.h"

#pragma clang fp contract(off)

namespace vs {

constexpr int SNT = 512;         // threads per workgroup
constexpr int SNW = SNT / WAVE;  // waves per workgroup
constexpr int NRED = 16;         // entries of each LDS reduction/broadcast array (>= SNW and >= 6)
static_assert(NRED >= 2 * SNW, "one reduction slot per wave, and the TOPK wave heads at 8 ..");
constexpr int EPT_MAX = 24;      // logits per lane in flight during the load
constexpr int NBIN = 256;        // radix digit = 8 bits
constexpr int MAX_ROUNDS = 32;   // histogram slots per row (8 count + 1 coarse + 4 fine + 1 + 7 + 7 radix rounds)
constexpr int GMAX = 64;         // workgroups per row
constexpr int GCAP = 1024;       // gather area of the FULL path (keys)
constexpr int GSMALL = 128;      // kept sets up to this size are finished in one workgroup
constexpr int GCAP2 = 512;       // elements gathered from the located value bins (<= SNT: one per thread in the final scans)
static_assert(GCAP2 <= SNT, "the final in-bin scans hold one gathered element per thread");
constexpr int NSET = 4;          // coarse value bins refined in the second histogram round
constexpr int BIGCAP = 5120;     // kept logits of the selected coarse bins that one workgroup resolves after a gather
constexpr int RANK_MAX = 512;    // largest set ranked by counting
constexpr int KEYS_CAP = 8192;   // LDS key area (64 KB): the merged candidate lists of a row
constexpr int KCAP = 256;        // largest top_k of the TOPK class
constexpr int RPL_MAX = 64;      // rows per launch (workspace is sized for this many)
constexpr int PAIRS_ALL = 2048;  // (id, count) tables up to this many entries are loaded whole by every workgroup
// Row-barrier time bounds in ticks of the 100 MHz real-time counter. A row's workgroups arrive within ~10 us of one
// another on an idle device; under a plain launch a wait that outlasts 200 us means some workgroup of the row is not
// resident (other streams hold the CUs), and the row gives up so that the host can repeat the call cooperatively.
// Under a cooperative launch every workgroup is resident, so only slowed waves can delay a barrier: 5 ms.
constexpr uint64_t WAIT_TICKS = 20000;        // 200 us
constexpr uint64_t WAIT_TICKS_COOP = 500000;  // 5 ms
// LDS scalar slots (misc): 0-17 single counters and flags, then arrays
constexpr int M_SEGC = 24;                         // [SNW] candidates per wave (TOPK)
constexpr int M_CNTS = M_SEGC + SNW;               // [GMAX] kept count per workgroup (FULL, small kept set)
constexpr int M_OFFS = M_CNTS + GMAX;              // [GMAX] their offsets
constexpr int M_XCH = (M_OFFS + GMAX + 1) & ~1;    // 2 x u64 exchange slots (8-byte aligned)
constexpr int M_STAT1 = M_XCH + 4;                 // [SNW] block_stats maxima
constexpr int M_STAT2 = M_STAT1 + SNW;             // [SNW]
constexpr int M_WB = M_STAT2 + SNW;                // [SNW] lane_max_bound per-wave bounds
constexpr int M_NZ = M_WB + SNW;                   // [SNW] lane_max_bound lanes with a finite logit
constexpr int NMISC = M_NZ + SNW;

enum RowClass { CLS_GREEDY = 0, CLS_TOPK = 1, CLS_FULL = 2 };

// Per-row control block; all zero between calls.
struct RowCtl {
  uint32_t bar;     // spin-barrier arrivals
  uint32_t done;    // workgroups finished (bits 0-15), of them the one that wrote the row's result (bits
                    // 16-23) and those that timed out at a row barrier (bits 24-31)
  uint32_t nfin;    // finite count of the row
  uint32_t mkey;    // ord32 of the largest finite logit
  u64 amkey;        // np.argmax key of the row
  uint32_t gcount;  // gather reservations
  uint32_t mcnt;    // min-p kept count
  u64 mfix;         // min-p kept fixed-point mass
  double mf64;      // min-p kept float64 mass
  uint32_t epoch;   // calls of this row so far (the XL row-barrier flags carry it); cleanup advances it
  uint32_t nminkey; // ~ord32 of the smallest finite logit (max-reduced)
  uint32_t g2count; // second gather reservations
  uint32_t gmax;    // largest per-workgroup kept count
};
static_assert(sizeof(RowCtl) == 64, "RowCtl layout");

struct Part {  // one per workgroup, written with device-coherent stores
  u64 amkey;
  uint32_t nfin;
  uint32_t kc;
  float mf;
  uint32_t pad;
  double se;
  u64 heads[8];  // TOPK lists of the unsorted format: eight of the list's largest keys (0 = none)
};
static_assert(sizeof(Part) == 96, "Part layout");

struct HistSlot {
  uint32_t cnt[NBIN];
  u64 fix[NBIN];
  double f64[NBIN];
  u64 mk[NBIN];
};

// Areas written with workgroup-scope stores (parts, lists, gathers, flags) start on their own 128-byte lines,
// apart from the lines that device-scope atomics update (the control block, the histogram slots).
constexpr size_t OFF_PART = 128;
constexpr size_t OFF_CAND = OFF_PART + sizeof(Part) * GMAX;
constexpr size_t OFF_GATHER = OFF_CAND + sizeof(u64) * KEYS_CAP;
constexpr size_t OFF_HIST = OFF_GATHER + sizeof(u64) * GCAP;
constexpr size_t OFF_BIG = OFF_HIST + sizeof(HistSlot) * MAX_ROUNDS;
constexpr size_t OFF_FLAGS = OFF_BIG + sizeof(u64) * BIGCAP;  // [GMAX] XL row-barrier flags
constexpr size_t ROW_WS = OFF_FLAGS + sizeof(u64) * GMAX;
static_assert(OFF_CAND % 128 == 0 && OFF_GATHER % 128 == 0 && OFF_HIST % 128 == 0 && OFF_BIG % 128 == 0 &&
                  OFF_FLAGS % 128 == 0 && ROW_WS % 128 == 0,
              "row workspace areas on 128-byte lines");

struct SampleArgs {
  const void* logits;
  int64_t ld;
  int B;     // rows in this launch
  int row0;  // first batch row of this launch
  int V;
  int G;
  int CH;
  int NV;      // vector loads per lane (vs_batch.hip: candidates a workgroup keeps of a row without a top-k cut)
  int vec_ok;  // 16-byte loads allowed
  int has_hist;
  int lds_ch;  // chunk length the LDS areas are sized for
  int kcap;    // candidate-list capacity per workgroup (a power of two; vs_batch.hip: a multiple of 64)
  int kmax;    // largest top_k of the TOPK class for this launch
  uint32_t spin_limit;  // polls before a row barrier gives up (testing hook; 0xFFFFFFFF: unbounded by polls)
  uint32_t debug;  // VS_DEBUG_* testing flags (vs_set_debug)
  uint64_t spin_ticks;  // real-time ticks (10 ns) before a row barrier gives up
  double fix_scale;  // probability -> fixed point (2^fix_shift)
  int fix_shift;
  double zspan_max;     // ln(fix_scale) - ln(1e6): the kept-value span up to which z comes from fixed point
  const vs_row_params* params;
  vs_row_state* state;  // device-resident request state, or null
  int list_k;           // > 0: top-list mode (vs_topk_batch): every row publishes its list_k largest logits, sorted
  int32_t* list_ids;    // [B, list_k]
  float* list_vals;     // [B, list_k]
  int32_t* pool;        // history pool of the state entry point
  const int32_t* slots;  // state entry point: row r uses params[slots[r]] and state[slots[r]] (null: r)
  const int32_t* tabs;   // state entry point: the (id, count) tables the states point into
  const int32_t* hist;
  const int32_t* bias_ids;
  const float* bias_vals;
  const int32_t* mask_ids;
  int32_t* out_ids;
  float* out_lp;
  uint32_t* out_flags;
  int32_t* out_keep;
  char* ws;
  unsigned long long* trace;  // development builds only (VS_TRACE); null otherwise
};

// LDS layout (dynamic): [xv: CH floats] [keys: max(KEYS_CAP u64, CH u32), the penalty counts during the edits]
// [tk: 2*KCAP u64] [hist] [scratch] [fine bins]. Every class reads its chunk from xv; keys holds candidate lists.
struct Smem {
  uint32_t* cnt;  // penalty counts (during the edits)
  float* xv;      // the processed chunk
  u64* fkeys;     // gathered keys (= keys)
  u64* keys;      // candidate lists
  u64* tk;
  uint32_t* hc;
  u64* hfix;
  double* hf64;
  u64* hmk;
  u64* red64;
  double* redf;
  int* redi;
  int* misc;     // NMISC ints
  uint32_t* fc;  // NSET*256 fine-bin counts
  u64* ffix;     // NSET*256 fine-bin fixed-point masses
  double* ff64;  // NSET*256 fine-bin float64 masses
  uint32_t* rc;  // 256-bin histogram of a workgroup-local radix select (count, fixed-point and float64 mass,
  u64* rfix;     // largest key), used while the other histograms must keep their contents
  double* rf64;
  u64* rmk;
};

__host__ __device__ inline size_t xv_bytes(int CH) { return ((size_t)CH * 4 + 15) & ~(size_t)15; }
__host__ __device__ inline size_t keys_bytes(int CH) {
  const size_t a = (size_t)KEYS_CAP * 8, b = xv_bytes(CH);
  return a > b ? a : b;
}
__host__ __device__ inline size_t region0(int CH) { return xv_bytes(CH) + keys_bytes(CH); }
__device__ __forceinline__ Smem carve(char* base, int CH) {
  Smem s;
  s.xv = (float*)base;
  s.keys = (u64*)(base + xv_bytes(CH));
  s.fkeys = s.keys;
  s.cnt = (uint32_t*)s.keys;  // the penalty counts use the key area before any class needs it
  char* p = base + region0(CH);
  s.tk = (u64*)p;
  p += 2 * KCAP * 8;
  s.hfix = (u64*)p;
  p += NBIN * 8;
  s.hf64 = (double*)p;
  p += NBIN * 8;
  s.hmk = (u64*)p;
  p += NBIN * 8;
  s.hc = (uint32_t*)p;
  p += NBIN * 4;
  s.red64 = (u64*)p;
  p += NRED * 8;
  s.redf = (double*)p;
  p += NRED * 8;
  s.redi = (int*)p;
  p += NRED * 4;
  s.misc = (int*)p;
  p += NMISC * 4;
  s.ffix = (u64*)p;
  p += NSET * NBIN * 8;
  s.ff64 = (double*)p;
  p += NSET * NBIN * 8;
  s.fc = (uint32_t*)p;
  p += NSET * NBIN * 4;
  s.rfix = (u64*)p;
  p += NBIN * 8;
  s.rf64 = (double*)p;
  p += NBIN * 8;
  s.rmk = (u64*)p;
  p += NBIN * 8;
  s.rc = (uint32_t*)p;
  return s;
}
static size_t smem_bytes(int CH) {
  return region0(CH) + 2 * KCAP * 8 + NBIN * (8 + 8 + 8 + 4) + NRED * (8 + 8 + 4) + NMISC * 4 + NSET * NBIN * (8 + 8 + 4) +
         NBIN * (8 + 8 + 8 + 4);
}

// ---------------------------------------------------------------------------------------------------------------
// Histogram scan. One wave walks the 256 bins: lane L owns digits 255-4L .. 252-4L (descending key order), so the
// bins are visited in rank order with one wave-wide scan and a ballot. Finds the first digit whose bin is non-empty
// and whose inclusive cumulative weight reaches `target`; when none does (a target above the total by rounding) the
// lowest non-empty digit, i.e. the last element. Weight = count (count mode) or fixed-point mass. Also returns the
// cumulative sums of all higher digits. The caller has synchronised after filling the bins.
// ---------------------------------------------------------------------------------------------------------------
struct ScanOut {
  int digit;
  u64 cnt_before, fix_before;
  double f64_before;
  u64 cnt, fix;
  double f64;
  u64 mk;
};

__device__ __forceinline__ ScanOut scan256(const Smem& s, const uint32_t* hc, const u64* hfix, const double* hf64,
                                           const u64* hmk, bool count_mode, double target) {
  if (threadIdx.x < WAVE) {
    const int L = threadIdx.x;
    u64 c[4], w[4];
    double f[4];
    u64 lc = 0, lw = 0;
    double lf = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = NBIN - 1 - (4 * L + i);
      c[i] = hc[d];
      w[i] = count_mode ? c[i] : hfix[d];
      f[i] = hf64[d];
      lc += c[i];
      lw += w[i];
      lf += f[i];
    }
    const u64 iw = wave_scan(lw), ic = wave_scan(lc);
    const double iff = wave_scan(lf);
    u64 cw = iw - lw, cc = ic - lc;
    double cf = iff - lf;
    int hit = -1, last = -1;
    u64 hw = 0, hc2 = 0;
    double hf = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (c[i] > 0) last = i;
      if (hit < 0 && c[i] > 0 && (double)(cw + w[i]) >= target) {
        hit = i;
        hw = cw;
        hc2 = cc;
        hf = cf;
      }
      cw += w[i];
      cc += c[i];
      cf += f[i];
    }
    const unsigned long long hb = __ballot(hit >= 0);
    int lane_sel, i_sel;
    if (hb) {
      lane_sel = __ffsll((long long)hb) - 1;
      i_sel = lane_bcast(hit, lane_sel);
    } else {
      const unsigned long long lb = __ballot(last >= 0);
      lane_sel = lb ? 63 - __clzll((long long)lb) : 0;
      i_sel = lb ? lane_bcast(last, lane_sel) : 0;
      if (i_sel < 0) i_sel = 0;
    }
    if (L == lane_sel) {
      if (!hb) {
        hw = iw - lw;
        hc2 = ic - lc;
        hf = iff - lf;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (i < i_sel) {
            hw += w[i];
            hc2 += c[i];
            hf += f[i];
          }
        }
      }
      const int d = NBIN - 1 - (4 * L + i_sel);
      s.misc[0] = d;
      s.red64[0] = hc2;
      s.red64[1] = hw;
      s.redf[0] = hf;
      s.red64[2] = hc[d];
      s.red64[3] = hfix[d];
      s.redf[1] = hf64[d];
      s.red64[4] = hmk ? hmk[d] : 0;
    }
  }
  __syncthreads();
  ScanOut o;
  o.digit = s.misc[0];
  o.cnt_before = s.red64[0];
  o.fix_before = count_mode ? 0 : s.red64[1];
  o.f64_before = s.redf[0];
  o.cnt = s.red64[2];
  o.fix = s.red64[3];
  o.f64 = s.redf[1];
  o.mk = s.red64[4];
  __syncthreads();
  return o;
}

__device__ __forceinline__ ScanOut hist_scan(const Smem& s, bool count_mode, double target) {
  return scan256(s, s.hc, s.hfix, s.hf64, s.hmk, count_mode, target);
}

// Prefix sums of a 256-bin histogram in scan order (digit 255 first, the order scan256 walks): pc[d] and pw[d] hold
// the count and fixed-point sums over digits 255 .. d (inclusive), pf[d] the float64 sum over digits 255 .. d+1
// (exclusive). Called by one whole wave.
__device__ __forceinline__ void hist_prefix(const uint32_t* hc, const u64* hw, const double* hf, u64* pc, u64* pw,
                                            double* pf) {
  const int L = lane_id();
  u64 c[4], w[4];
  double f[4];
  u64 lc = 0, lw = 0;
  double lf = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = NBIN - 1 - (4 * L + i);
    c[i] = hc[d];
    w[i] = hw[d];
    f[i] = hf[d];
    lc += c[i];
    lw += w[i];
    lf += f[i];
  }
  u64 cc = wave_scan(lc) - lc, cw = wave_scan(lw) - lw;
  double cf = wave_scan(lf) - lf;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = NBIN - 1 - (4 * L + i);
    pf[d] = cf;
    cc += c[i];
    cw += w[i];
    cf += f[i];
    pc[d] = cc;
    pw[d] = cw;
  }
}

// The smallest integer >= t (0 for t <= 0, the largest u64 from 2^64 up).
__device__ __forceinline__ u64 ceil_u64(double t) {
  return t <= 0.0 ? (u64)0 : (t >= 18446744073709551616.0 ? ~(u64)0 : (u64)__builtin_ceil(t));
}

// scan256's answer from prefix arrays (hist_prefix): the first digit in scan order whose bin is non-empty and whose
// inclusive weight reaches `target` (the last non-empty digit when none does, which only rounding can cause), with
// the sums before it. Every wave computes it on its own, so no barrier is needed; the caller has synchronised after
// hist_prefix.
__device__ __forceinline__ ScanOut hist_find(const uint32_t* hc, const u64* hw, const double* hf, const u64* pc,
                                             const u64* pw, const double* pf, double target) {
  const int L = lane_id();
  uint32_t c[4];
  u64 w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = NBIN - 1 - (4 * L + i);
    c[i] = hc[d];
    w[i] = pw[d];
  }
  const u64 tg = ceil_u64(target);  // an integer sum reaches target iff it reaches ceil(target)
  int hit = 4, last = -1;
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    hit = (c[i] > 0 && w[i] >= tg) ? i : hit;
    last = (last < 0 && c[i] > 0) ? i : last;
  }
  const unsigned long long hb = __ballot(hit < 4);
  int lane_sel, i_sel;
  if (hb) {
    lane_sel = __ffsll((long long)hb) - 1;
    i_sel = lane_bcast(hit, lane_sel);
  } else {
    const unsigned long long lb = __ballot(last >= 0);
    lane_sel = lb ? 63 - __clzll((long long)lb) : 0;
    i_sel = lb ? lane_bcast(last, lane_sel) : 0;
  }
  const int d = NBIN - 1 - (4 * lane_sel + i_sel);
  ScanOut o;
  o.digit = d;
  o.cnt = hc[d];
  o.fix = hw[d];
  o.f64 = hf[d];
  o.cnt_before = pc[d] - o.cnt;
  o.fix_before = pw[d] - o.fix;
  o.f64_before = pf[d];
  o.mk = 0;
  return o;
}

__device__ __forceinline__ void hist_clear(const Smem& s) {
  const int t = threadIdx.x;
  if (t < NBIN) {
    s.hc[t] = 0;
    s.hfix[t] = 0;
    s.hf64[t] = 0.0;
    s.hmk[t] = 0;
  }
  __syncthreads();
}

__device__ __forceinline__ void hist_add(const Smem& s, u64 key, int shift, u64 fx, double f) {
  const int d = (int)((key >> shift) & 0xFF);
  atomicAdd(&s.hc[d], 1u);
  if (fx) atomicAdd(&s.hfix[d], fx);
  if (f != 0.0) unsafeAtomicAdd(&s.hf64[d], f);
  atomicMax(&s.hmk[d], key);
}

__device__ __forceinline__ bool prefix_match(u64 key, int shift, u64 prefix) {
  return shift >= 56 ? true : ((key >> (shift + 8)) == prefix);
}

// k-th largest of n unique keys in LDS (1 <= k <= n): returns T with |{keys >= T}| == k. Radix select, 8-bit
// digits from the top, stopping as soon as a bin is taken whole.
__device__ __forceinline__ u64 block_kth(const Smem& s, const u64* keys, int n, int k) {
  u64 prefix = 0;
  int shift = 56;
  int krem = k;
  for (;;) {
    hist_clear(s);
    for (int i = threadIdx.x; i < n; i += SNT) {
      const u64 key = keys[i];
      if (prefix_match(key, shift, prefix)) atomicAdd(&s.hc[(key >> shift) & 0xFF], 1u);
    }
    __syncthreads();
    const ScanOut o = hist_scan(s, true, (double)krem);
    const int need = krem - (int)o.cnt_before;
    const u64 np = (prefix << 8) | (u64)o.digit;
    if ((int)o.cnt == need || shift == 0) return np << shift;
    krem = need;
    prefix = np;
    shift -= 8;
  }
}

// Logarithms of the logprob formulas in float32 (the result is a float32 logprob; float log and log1p are
// accurate to a few float ulps, far inside its tolerance), in the forms that keep relative accuracy:
// log(z) for z >= 1 as log1p(z - 1), and log(p / z) for 0 < p <= z as log1p((p - z) / z) when p >= z / 2 (the
// difference is exact) or log(p / z) below.
__device__ __forceinline__ double log_ge1(double z) { return (double)log1pf((float)(z - 1.0)); }
__device__ __forceinline__ double log_ratio(double p, double z) {
  return p >= 0.5 * z ? (double)log1pf((float)((p - z) / z)) : (double)logf((float)(p / z));
}

struct Final {
  int32_t token;
  float lp;
  uint32_t flags;
  int32_t keep;
};

// sampler.py:141-156 on n <= 64 * EM keys sorted descending in LDS (a[0] is the row maximum), in one wave: lane
// L owns positions [L*E, L*E+E), E = ceil(n / 64) <= EM, so every sum and prefix is a lane-sequential loop plus one
// wave scan. Lane 0 leaves the result in LDS for wave_sample.
template <int EM>  // n <= 64 * EM
__device__ __forceinline__ void wave_sample_em(const Smem& s, const u64* a, int n, const vs_row_params& P) {
  {
    const int L = threadIdx.x;
    const int E = EM == 1 ? 1 : (n + WAVE - 1) / WAVE;
    const int i0 = L * E;
    const float tt = P.temperature;
    const float xs0 = key_value(a[0]) / tt;  // sampler.py:141 xs[0]
    double pr[EM];
    double ls = 0.0;
#pragma unroll
    for (int q = 0; q < EM; ++q) {
      pr[q] = 0.0;
      if (q < E && i0 + q < n) {
        const float xs = key_value(a[i0 + q]) / tt;
        const float d = xs - xs0;  // float32 subtraction (:142)
        // exp in float32, widened: relative error <= 2^-23 per mass (the reference's float64 exp of the same d
        // differs by less; sums and cumulative sums inherit that bound, far inside the 1e-6 boundary band and the
        // 1e-5 logprob tolerance; pr[0] = exp(0) = 1 exactly, so a dominant first token's logprob stays exact)
        pr[q] = (double)expf(d);
        ls += pr[q];
      }
    }
    // one scan gives both the total (:143) and each lane's cumulative mass before its first position
    const double incl = wave_scan(ls);
    const double S = lane_bcast(incl, WAVE - 1);
    VS_TRX(40);
#pragma unroll
    for (int q = 0; q < EM; ++q) pr[q] = pr[q] / S;
    const double base = (incl - ls) / S;
    VS_TRX(41);
    int keep = n;
    uint32_t flags = 0;
    if (P.top_p < 1.0) {  // :145-148 first position with cumsum >= top_p
      const double tp = P.top_p;
      double c = base;
      int hit = -1;
      int fb = 0;
#pragma unroll
      for (int q = 0; q < EM; ++q) {
        if (q < E && i0 + q < n) {
          const double prev = c;
          c += pr[q];
          if (hit < 0 && c >= tp) {
            hit = i0 + q;
            fb = fabs(c - tp) < 1e-6 || fabs(prev - tp) < 1e-6;
          }
        }
      }
      const unsigned long long hb = __ballot(hit >= 0);
      if (hb) {
        const int ls2 = __ffsll((long long)hb) - 1;
        keep = lane_bcast(hit, ls2) + 1;
        if (lane_bcast(fb, ls2)) flags |= VS_OUT_TOPP_BOUNDARY;
      }
    }
    if (P.min_p > 0.0) {  // :149-152 first position with pr < pr[0] * min_p
      const double thr = lane_bcast(pr[0], 0) * P.min_p;
      int hit = -1;
#pragma unroll
      for (int q = 0; q < EM; ++q)
        if (hit < 0 && q < E && i0 + q < n && pr[q] < thr) hit = i0 + q;
      const unsigned long long hb = __ballot(hit >= 0);
      int cnt = hb ? lane_bcast(hit, __ffsll((long long)hb) - 1) : n;
      cnt = cnt > 1 ? cnt : 1;
      keep = keep < cnt ? keep : cnt;
    }
    VS_TRX(42);
    double z;  // :153, the cumulative mass through the last kept position (read from the lane that holds it)
    {
      const int owner = (keep - 1) / E, qq = keep - 1 - owner * E;
      double cz = base;
#pragma unroll
      for (int q = 0; q < EM; ++q)
        if (q <= qq && q < E) cz += pr[q];
      z = lane_bcast(cz, owner);
    }
    const double uz = P.u * z;      // :154
    double c = base;
    int hit = -1;
    double hp = 0.0, hc = 0.0;
#pragma unroll
    for (int q = 0; q < EM; ++q) {
      if (q < E && i0 + q < keep) {
        c += pr[q];
        if (hit < 0 && c >= uz) {
          hit = i0 + q;
          hp = pr[q];
          hc = c;
        }
      }
    }
    const unsigned long long hb = __ballot(hit >= 0);
    int j;
    if (hb) {  // :155 searchsorted(cumsum, u*z, 'left')
      const int ls2 = __ffsll((long long)hb) - 1;
      j = lane_bcast(hit, ls2);
      hp = lane_bcast(hp, ls2);
      hc = lane_bcast(hc, ls2);
    } else {  // :156 min(j, keep-1): the last kept position
      j = keep - 1;
      const int owner = j / E, qq = j - owner * E;
      double cc = base, pp = 0.0;
#pragma unroll
      for (int q = 0; q < EM; ++q)
        if (q <= qq && q < E) {
          cc += pr[q];
          pp = pr[q];
        }
      hp = lane_bcast(pp, owner);
      hc = lane_bcast(cc, owner);
    }
    VS_TRX(43);
    if (L == 0) {
      const double tol = 1e-6 * z;
      if (fabs(hc - uz) < tol || (j >= 1 && fabs(hc - hp - uz) < tol)) flags |= VS_OUT_DRAW_BOUNDARY;
      s.misc[1] = (int)key_index(a[j]);
      s.misc[2] = keep;
      s.misc[3] = (int)flags;
      s.redf[0] = log_ratio(hp, z);
    }
  }
}
// sampler.py:141-156 on n <= 256 keys sorted descending in LDS (see wave_sample_em); all threads call it.
__device__ __forceinline__ Final wave_sample(const Smem& s, const u64* a, int n, const vs_row_params& P) {
  if (threadIdx.x < WAVE) {
    if (n <= WAVE) wave_sample_em<1>(s, a, n, P);
    else if (n <= 2 * WAVE) wave_sample_em<2>(s, a, n, P);
    else wave_sample_em<4>(s, a, n, P);
  }
  __syncthreads();
  Final f;
  f.token = s.misc[1];
  f.keep = s.misc[2];
  f.flags = (uint32_t)s.misc[3];
  f.lp = (float)s.redf[0];
  __syncthreads();
  return f;
}


__device__ __forceinline__ int pow2_ceil(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// Descending order by rank: out[#{j : in[j] > in[i]}] = in[i] for ranks below kout (distinct keys get distinct
// ranks). T lanes of one wave share each key's comparisons (T = the largest power of two <= 64 with T * n <= SNT,
// at least 1); each lane reads 8 keys per step, so 8 LDS reads are in flight instead of one per loop trip.
// The caller has synchronised after writing `in`; ends with a barrier.
__device__ __forceinline__ void rank_sort(const u64* in, int n, u64* out, int kout) {
  // T = SNT / 2^ceil(log2 n), clamped to [1, 64]
  const int lg = n > 1 ? 32 - __builtin_clz((unsigned)(n - 1)) : 0;
  int T = lg >= 9 ? 1 : (SNT >> lg);
  T = T > 64 ? 64 : T;
  const int t = threadIdx.x;
  const int sub = t & (T - 1);
  const int step = 8 * T;
  for (int i0 = 0; i0 < n; i0 += SNT / T) {  // uniform trip count
    const int i = i0 + t / T;
    const u64 ki = in[i < n ? i : 0];
    int r = 0;
    for (int j0 = 0; j0 < n; j0 += step) {  // uniform trip count
      u64 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = j0 + u * T + sub;
        v[u] = in[j < n ? j : 0];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) r += (j0 + u * T + sub < n && v[u] > ki) ? 1 : 0;
    }
    if (T > 1) r += lane_xor<1>(r);
    if (T > 2) r += lane_xor<2>(r);
    if (T > 4) r += lane_xor<4>(r);
    if (T > 8) r += lane_xor<8>(r);
    if (T > 16) r += lane_xor<16>(r);
    if (T > 32) r += lane_xor<32>(r);
    if (sub == 0 && i < n && r < kout) out[r] = ki;
  }
  __syncthreads();
}

constexpr int SEGW = KEYS_CAP / SNW;  // per-wave candidate segment
// Bits of an ord32 value resolved by the ballot bisections that bound the k-th largest logit from below (sign,
// exponent and 7 mantissa bits).
constexpr int BOUND_BITS = 16;
// Key-area offset (u64 words) of the value-bin prefix sums: above what the final in-bin resolution uses
// (4352 words), 3 * 256 coarse + 3 * NSET * 256 fine words.
constexpr int PFX_OFF = 4352;
static_assert(PFX_OFF + 3 * NBIN * (1 + NSET) <= KEYS_CAP, "prefix sums fit the key area");
// Key-area layout of the value-bin path below the prefix sums: words 0-511 gathered keys, then from word 512 the
// fine-bin id of every chunk position (u16; 0xFFFF = not in the kept set).
constexpr int FID_OFF = 512;
static_assert(FID_OFF * 8 + EPT_MAX * SNT * 2 <= PFX_OFF * 8, "fine-bin ids fit below the prefix sums");

// Sort 64*E keys held by one wave descending (lane L holds positions L + 64*i in e[i]); the bitonic network is
// fully unrolled: partners at distance < 64 are exchanged across lanes (DPP / permlane), the others in-lane.
template <int E>
__device__ __forceinline__ void wave_sort_desc(u64 (&e)[E]) {
  const int L = lane_id();
#pragma unroll
  for (int k = 2; k <= 64 * E; k <<= 1) {
#pragma unroll
    for (int j = k >> 1; j > 0; j >>= 1) {
      if (j >= 64) {
        const int d = j / 64;
#pragma unroll
        for (int i = 0; i < E; ++i) {
          if ((i & d) == 0) {
            const int pos = L + 64 * i;
            const bool desc = (pos & k) == 0;
            const u64 a = e[i], b = e[i + d];
            const u64 mx = a > b ? a : b, mn = a > b ? b : a;
            e[i] = desc ? mx : mn;
            e[i + d] = desc ? mn : mx;
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const u64 o = lane_xor_rt(e[i], j);
          const int pos = L + 64 * i;
          const bool take_max = ((pos & k) == 0) == ((pos & j) == 0);
          e[i] = ((e[i] > o) == take_max) ? e[i] : o;
        }
      }
    }
  }
}

// Sorted copy of n <= 256 keys: out[r] = key of rank r for r < kout. One wave sorts (the others wait at the final
// barrier); larger n falls back to rank counting over the whole workgroup.
__device__ __forceinline__ void small_sort(const u64* in, int n, u64* out, int kout) {
  if (n > 256) {
    rank_sort(in, n, out, kout);
    return;
  }
  if (threadIdx.x < WAVE) {
    const int L = threadIdx.x;
    if (n <= 64) {
      u64 e[1] = {L < n ? in[L] : (u64)0};
      wave_sort_desc<1>(e);
      if (L < kout) out[L] = e[0];
    } else if (n <= 128) {
      u64 e[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) e[i] = L + 64 * i < n ? in[L + 64 * i] : (u64)0;
      wave_sort_desc<2>(e);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (L + 64 * i < kout) out[L + 64 * i] = e[i];
    } else {
      u64 e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = L + 64 * i < n ? in[L + 64 * i] : (u64)0;
      wave_sort_desc<4>(e);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (L + 64 * i < kout) out[L + 64 * i] = e[i];
    }
  }
  __syncthreads();
}

// Lower bound for the k-th largest logit of the workgroup, from the lane maxima (ord32 values, 0 for a lane with no
// finite logit): each wave finds its q-th largest lane maximum, q = min(ceil(k/8), its non-zero lanes), by a
// most-significant-bit-first radix select on ballots. Those q lanes of every wave hold values >= the smallest wave's
// result, so when the waves' q add up to >= k the workgroup has >= k logits >= L. L = 0 otherwise (no bound).
// nlanes = lanes holding a finite logit.
struct LaneBound {
  uint32_t L;
  int nlanes;
};
__device__ __forceinline__ LaneBound lane_max_bound(uint32_t tmax, int k, const Smem& s) {
  const int q = (k + SNW - 1) / SNW;
  const int nz = __popcll(__ballot(tmax != 0));
  const int got = nz < q ? nz : q;
  uint32_t wb = 0;
  if (got > 0) {
    // the top BOUND_BITS bits only: the result (low bits zero) is still a valid lower bound, within a factor of
    // 1 + 2^-7 of the exact q-th largest value, for half the dependent ballot steps
    for (int b = 31; b >= 32 - BOUND_BITS; --b) {
      const uint32_t c = wb | (1u << b);
      if ((int)__popcll(__ballot(tmax >= c)) >= got) wb = c;
    }
  }
  VS_TRX(37);
  const int w = threadIdx.x / WAVE;
  uint32_t* wbs = (uint32_t*)(s.misc + M_WB);
  if (lane_id() == 0) {
    wbs[w] = wb;
    s.redi[w] = got;
    s.misc[M_NZ + w] = nz;
  }
  __syncthreads();
  VS_TRX(38);
  LaneBound r;
  uint32_t L = ~0u;
  int tot = 0, nl = 0;
  int gw[SNW], nw[SNW];
  uint32_t bw[SNW];
#pragma unroll
  for (int i = 0; i < SNW; ++i) {  // all reads first, then selects (a guarded read becomes a branch per wave)
    gw[i] = s.redi[i];
    nw[i] = s.misc[M_NZ + i];
    bw[i] = wbs[i];
  }
#pragma unroll
  for (int i = 0; i < SNW; ++i) {
    tot += gw[i];
    nl += nw[i];
    const uint32_t b = gw[i] > 0 ? bw[i] : ~0u;
    L = b < L ? b : L;
  }
  __syncthreads();
  r.L = tot >= k ? L : 0u;
  r.nlanes = nl;
  return r;
}

// One LDS exchange for the per-workgroup statistics: a sum, two 32-bit maxima and a 64-bit maximum.
struct Stats {
  int n;
  uint32_t mx1, mx2;
  u64 am;
};
__device__ __forceinline__ Stats block_stats(int n, uint32_t mx1, uint32_t mx2, const Smem& s) {
  n = wave_sum(n);
  mx1 = wave_max(mx1);
  mx2 = wave_max(mx2);
  const int w = threadIdx.x / WAVE;
  uint32_t* m1 = (uint32_t*)(s.misc + M_STAT1);
  uint32_t* m2 = (uint32_t*)(s.misc + M_STAT2);
  __syncthreads();
  if (lane_id() == 0) {
    s.redi[w] = n;
    m1[w] = mx1;
    m2[w] = mx2;
  }
  __syncthreads();
  Stats r = {0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < SNW; ++i) {
    r.n += s.redi[i];
    r.mx1 = m1[i] > r.mx1 ? m1[i] : r.mx1;
    r.mx2 = m2[i] > r.mx2 ? m2[i] : r.mx2;
  }
  __syncthreads();
  return r;
}

// The state entry point's Sampler.accept (sampler.py:75-79) and the draw's state advance, by the one thread that
// writes the row's result; the launch boundary orders it before the next call's reads.
__device__ __forceinline__ uint32_t commit_state(const SampleArgs& A, int r, int32_t token, uint32_t flags,
                                                 const vs_row_state& st, uint64_t rng_next) {
  if (!A.state || (flags & VS_OUT_TIMEOUT)) return flags;
  vs_row_state* S = A.state + (A.slots ? A.slots[r] : r);
  if (!(flags & (VS_OUT_GREEDY | VS_OUT_NOFINITE | VS_OUT_FORCED))) S->rng = rng_next;
  if (st.hist_len < st.hist_cap) {
    A.pool[st.hist_off + st.hist_len] = token;
    S->hist_len = st.hist_len + 1;
  } else {
    flags |= VS_OUT_HIST_FULL;
  }
  S->produced = st.produced + 1;
  return flags;
}

__device__ __forceinline__ void write_out(const SampleArgs& A, int row, const Final& f, const vs_row_state& st,
                                          uint64_t rng_next) {
  if (threadIdx.x == 0) {
    const int r = A.row0 + row;
    const uint32_t flags = commit_state(A, r, f.token, f.flags, st, rng_next);
    A.out_ids[r] = f.token;
    A.out_lp[r] = f.lp;
    if (A.out_flags) A.out_flags[r] = flags;
    if (A.out_keep) A.out_keep[r] = f.keep;
  }
}

// round(e * 2^S) to the nearest integer, ties to even, for a float 0 <= e <= 1 and 0 < S <= 63, in float
// arithmetic (sh = 2^(S - 32), sc = 2^S): h = trunc(e * sh) is the part of e * 2^S at and above 2^32 (an integral
// float, exact), and e * sc - h * 2^32 is the rest, exact because it is e's mantissa without its top bits. A rest
// with a fraction is below 2^24, so its rounding cannot carry into h. Equal to rint((double)e * 2^S).
__device__ __forceinline__ u64 fixed_mass(float e, float sh, float sc) {
  const float h = __builtin_truncf(e * sh);
  const float r = __builtin_fmaf(-h, 4294967296.0f, e * sc);
  return ((u64)(uint32_t)h << 32) | (u64)(uint32_t)__builtin_rintf(r);
}

// e^d for d <= 0 with about 2 ulp relative error: 2^(d log2 e) from the hardware base-2 exponential, with the
// rounding error of the product d * log2(e) (exact through an fma, plus the constant's own tail) applied as a
// first-order correction: e^d = 2^y * 2^(lo) ~ 2^y (1 + lo ln 2) for the tiny lo.
// `corr` is ln 2 for that correction (0 drops it: plain 2^(d L)).
__device__ __forceinline__ float exp_nonpos(float d, float corr = 0.693147180559945309f) {
  const float L = 1.44269502162933349609375f;  // log2(e) rounded to float
  const float Llo = 1.9259629891e-8f;          // log2(e) - L
  const float y = d * L;
  const float lo = fmaf(d, L, -y) + d * Llo;
  const float e = __builtin_amdgcn_exp2f(y);
  return fmaf(e, lo * corr, e);
}

// Sorted-id range search: first position in ids[b, e) with ids[p] >= x.
__device__ __forceinline__ int lower_bound_ids(const int32_t* ids, int b, int e, int32_t x) {
  while (b < e) {
    const int m = (b + e) >> 1;
    if (ids[m] < x)
      b = m + 1;
    else
      e = m;
  }
  return b;
}

template <int DT>
struct DTraits;
template <>
struct DTraits<VS_F32> {
  typedef float LT;
  static constexpr int VEC = 4;
  __device__ static float cv(LT v) { return v; }
};
template <>
struct DTraits<VS_BF16> {
  typedef uint16_t LT;
  static constexpr int VEC = 8;
  __device__ static float cv(LT v) { return bf16_to_f32(v); }
};
template <>
struct DTraits<VS_F16> {
  typedef uint16_t LT;
  static constexpr int VEC = 8;
  __device__ static float cv(LT v) { return f16_to_f32(v); }
};

// ---------------------------------------------------------------------------------------------------------------
// History counts (the counts Sampler.accept keeps, sampler.py:77-78) for the tokens in [lo, hi): cnt[tok - lo] += 1
// for every occurrence. The history is read as 16-byte vectors, HB per lane per batch, HD batches in flight; the
// first HD batches are loaded before the logits arrive.
// ---------------------------------------------------------------------------------------------------------------
constexpr int HB = 2;  // 16-byte vectors per lane per batch (8 ids)
struct HistWin {
  int64_t b, e, a, nv;  // [b, e): the ids; a: first 16-byte aligned position; nv: whole vectors from a
};
__device__ __forceinline__ HistWin hist_window(int64_t b, int64_t e) {
  HistWin w;
  w.b = b;
  w.e = e;
  w.a = (b + 3) & ~(int64_t)3;
  if (w.a > e) w.a = e;
  w.nv = (e - w.a) >> 2;
  return w;
}
// Loads vectors v0 + u * SNT (u < HB), the index clamped to the last vector so that every load is unconditional
// (conditional loads make the compiler wait for all loads at the loop latch); the consumer masks by position.
// Requires w.nv >= 1.
__device__ __forceinline__ void hist_load(const int32_t* h, const HistWin& w, int64_t v0, int4 (&r)[HB]) {
  const int4* hv = (const int4*)(h + w.a);
#pragma unroll
  for (int u = 0; u < HB; ++u) {
    const int64_t vi = v0 + (int64_t)u * SNT;
    r[u] = hv[vi < w.nv ? vi : w.nv - 1];
  }
}
// Count N ids per lane into cnt[id - lo] for the ids in [lo, hi).
template <int N>
__device__ __forceinline__ void hist_add_ids(const int32_t (&tk)[N], int lo, int hi, uint32_t* cnt) {
#pragma unroll
  for (int q = 0; q < N; ++q) {
    const uint32_t o = (uint32_t)(tk[q] - lo);
    if (o < (uint32_t)(hi - lo)) atomicAdd(&cnt[o], 1u);
  }
}
constexpr int HD = 4;  // batches in flight
// cnt[tok - lo] += 1 for every history id in [lo, hi).
__device__ __forceinline__ void hist_count(const int32_t* h, const HistWin& w, int4 (&r)[HD][HB], int lo, int hi,
                                           uint32_t* cnt) {
  const int t = threadIdx.x;
  {  // the unaligned head (< 4 ids) and tail (< 4 ids), one id per lane
    const int nh = (int)(w.a - w.b);
    const int64_t tb = w.a + w.nv * 4;
    const int nt = (int)(w.e - tb);
    int32_t one[1] = {-1};
    if (t < nh) one[0] = h[w.b + t];
    else if (t - nh < nt) one[0] = h[tb + (t - nh)];
    hist_add_ids(one, lo, hi, cnt);
  }
  constexpr int64_t BATCH = (int64_t)SNT * HB;  // vectors per batch
  // One group = HD batches: the first was loaded ahead of time; every later group issues all its loads before
  // counting (no registers carried across iterations, so the loads of a group are in flight together).
  auto take = [&](int64_t v0, int4 (&r)[HD][HB]) {
#pragma unroll
    for (int d = 0; d < HD; ++d) {
      const int64_t vb = v0 + d * BATCH;
      if (vb >= w.nv) break;  // uniform
      int32_t tk[4 * HB];
#pragma unroll
      for (int u = 0; u < HB; ++u) {
        const bool ok = vb + (int64_t)u * SNT + t < w.nv;
        tk[4 * u] = ok ? r[d][u].x : -1;
        tk[4 * u + 1] = ok ? r[d][u].y : -1;
        tk[4 * u + 2] = ok ? r[d][u].z : -1;
        tk[4 * u + 3] = ok ? r[d][u].w : -1;
      }
      hist_add_ids(tk, lo, hi, cnt);
    }
  };
  if (w.nv > 0) take(0, r);
  for (int64_t v0 = BATCH * HD; v0 < w.nv; v0 += BATCH * HD) {
    int4 q[HD][HB];
#pragma unroll
    for (int d = 0; d < HD; ++d) hist_load(h, w, v0 + d * BATCH + t, q[d]);
    take(v0, q);
  }
}

// fn(id) for every id of a history window whose whole vectors are all in the prefetched batches r (w.nv <= HD *
// SNT * HB); the unaligned head and tail ids are loaded again. Ids outside the window are not visited.
template <typename Fn>
__device__ __forceinline__ void hist_visit_prefetched(const int32_t* h, const HistWin& w, const int4 (&r)[HD][HB],
                                                      Fn fn) {
  const int t = threadIdx.x;
  {
    const int nh = (int)(w.a - w.b);
    const int64_t tb = w.a + w.nv * 4;
    const int nt = (int)(w.e - tb);
    if (t < nh) fn(h[w.b + t]);
    else if (t - nh < nt) fn(h[tb + (t - nh)]);
  }
  constexpr int64_t BATCH = (int64_t)SNT * HB;
#pragma unroll
  for (int d = 0; d < HD; ++d) {
    const int64_t vb = d * BATCH;
    if (vb >= w.nv) break;  // uniform
#pragma unroll
    for (int u = 0; u < HB; ++u) {
      if (vb + (int64_t)u * SNT + t < w.nv) {
        fn(r[d][u].x);
        fn(r[d][u].y);
        fn(r[d][u].z);
        fn(r[d][u].w);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Penalty counts given as a table (VS_ROW_HIST_PAIRS): n (id, count) pairs sorted by id with unique ids, the form of
// Sampler.counts (sampler.py:77-78, iterated at :113-122). A workgroup needs the entries with ids in [lo, hi) only.
// Thread t loads the id at entry pos(t) = t * n / SNT ahead (with the logits); the block counts the probes below lo
// (c0) and below hi (c1). Every entry with an id in [lo, hi) then lies in [pos(c0 - 1) + 1, pos(c1)) (pos(-1) = -1,
// pos(SNT) = n): at most 2 n / SNT entries beyond the wanted ones, which the range test of the edit skips.
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ int64_t probe_at(int64_t n, int j) { return ((int64_t)j * n) / SNT; }

__device__ __forceinline__ void pair_range(int64_t n, int32_t probe, int lo, int hi, int* red, int64_t* r0,
                                           int64_t* r1) {
  const int w = threadIdx.x / WAVE;
  const int n0 = __popcll(__ballot(probe < lo)), n1 = __popcll(__ballot(probe < hi));
  if (lane_id() == 0) {
    red[w] = n0;
    red[SNW + w] = n1;
  }
  __syncthreads();
  int c0 = 0, c1 = 0;
#pragma unroll
  for (int i = 0; i < SNW; ++i) {
    c0 += red[i];
    c1 += red[SNW + i];
  }
  *r0 = c0 == 0 ? 0 : probe_at(n, c0 - 1) + 1;
  *r1 = c1 == SNT ? n : probe_at(n, c1);
}

// vs_batch.hip: the launches for a batch of B rows (a: every field that does not depend on the split of a row);
// ws_rows: workspace rows there are.
int batch_path(SampleArgs a, int dtype, int B, size_t ws_rows, const DevInfo* dv, hipStream_t stream);

}  // namespace vs
