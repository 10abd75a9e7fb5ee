// vs_batch.hip - Sampler.sample (volundr-mlx/sampler.py:100-156) for batches of more rows than one launch of
// vs_sample_kernel holds, in three launches.
//
// vs_sample_kernel keeps a row's chunks in LDS (one workgroup per CU) because rows without a top-k cut meet at row
// barriers, so a launch holds only the rows that are resident together and a large batch runs as a chain of such
// launches, each as long as its slowest row. Here
//   vs_batch_kernel    streams the logits once, a chunk per workgroup in registers, and leaves per chunk a short list:
//     GREEDY  the first-max key and the log-sum-exp partial;
//     TOPK    at least its k largest logits, so the row's k largest are in the lists (a list that overflows is cut to them);
//     FULL    its logits down to a bound of its own, and the mass exp(x/t - max/t) of the rest. The row's logits above
//             the largest such bound are then all listed, and the row's whole mass is known.
//   vs_finish_kernel   finishes each row from its lists, one workgroup per row. A FULL row is finished here if its
//     top-p cut, min-p cut and draw fall among the logits that are known to be listed (a language model's usual row).
//   vs_resolve_kernel  takes the rows left open with as many workgroups per row as there are: flat distributions by one
//     histogram pass and one gather pass over the row, a top-k above the lists' reach likewise, everything else (long
//     runs of tied values, a top-k of thousands, no finite logit) by a radix select over passes. It ends at once when no
//     row is open. Only here do workgroups wait for one another (a cluster's barrier, bounded in time); GREEDY rows and
//     TOPK rows with a finite logit are never left open.
#include "vs_sample.h"


#pragma clang fp contract(off)

namespace vs {

constexpr int BATCH_ROWS = 2 * RPL_MAX;  // rows per launch
constexpr int BATCH_NK = 16;             // listed keys a thread of the finish kernel holds
constexpr int BSEL = RANK_MAX;           // keys it ranks at most
constexpr uint32_t L_NONE = ~0u;         // a chunk of a FULL row whose list does not hold what it should
constexpr int SEG_CAP = 256;             // candidates a wave stages at most
constexpr int RNB = 2048;                // value bins of the resolve kernel
constexpr int RCAP = 2048;               // keys it gathers
constexpr int RRING = 3;                 // radix histograms in use at a time
constexpr int CMAX = 32;                 // workgroups per open row at most

// Workspace of a launch's row r: workspace rows hold two each. Row r < RPL_MAX uses the part and cand areas of
// workspace row r, row r >= RPL_MAX the gather and big areas of workspace row r - RPL_MAX (areas whose contents no call
// relies on; of a partial all but the word `pad`, by whose tags vs_sample_kernel tells this call's partials from what
// earlier ones left). The open flags sit in the control blocks' lines, after RowCtl: those of rows [56 k, 56 k + 56) in
// workspace row k. Nothing here has to be zero when a call starts.
// open flag: finished, left to the flat, the top-k or the general method
enum { ROW_DONE = 0, ROW_FLAT = 1, ROW_ANY = 2, ROW_TOPK = 3 };
constexpr size_t OFF_OPEN = 64;
constexpr int OPEN_PER = 56;
static_assert(OFF_OPEN >= sizeof(RowCtl) && OFF_OPEN + OPEN_PER <= OFF_PART, "after RowCtl, before the partials");
static_assert(sizeof(Part) * GMAX <= sizeof(u64) * GCAP, "the second row's partials fit the gather area");
__device__ __forceinline__ uint8_t* open_flag(char* ws, int r) {
  return (uint8_t*)(ws + (size_t)(r / OPEN_PER) * ROW_WS + OFF_OPEN) + r % OPEN_PER;
}
__device__ __forceinline__ char* part_area(char* ws, int r) {
  return ws + (size_t)(r % RPL_MAX) * ROW_WS + (r < RPL_MAX ? OFF_PART : OFF_GATHER);
}
__device__ __forceinline__ char* list_area(char* ws, int r) {
  return ws + (size_t)(r % RPL_MAX) * ROW_WS + (r < RPL_MAX ? OFF_CAND : OFF_BIG);
}
// What the finish kernel leaves of an open row (over its partials), and the row's counters in the resolve kernel.
struct OpenRow {
  int n;             // finite logits
  float xmax, xmin;  // the largest and smallest of them (ROW_TOPK: a value that the top-k cut hardly lies below)
  uint32_t bar;      // arrivals at the cluster's barriers
  uint32_t gcnt;     // gathered keys
  uint32_t tag;      // the first partial's tag word, left alone
  uint32_t cnt[4];   // sums over the cluster: counts
  int shift;         // masses are summed in fixed point at 2^shift: the whole row's stay below 2^63
  u64 fix[3];        // and masses
  u64 amkey;
};
static_assert(offsetof(OpenRow, tag) == offsetof(Part, pad) && sizeof(OpenRow) <= sizeof(Part), "the tag words stay");
// An open row's list area: the mass histogram of the flat method (or the ring of radix histograms), then the keys.
struct RadixSlot {
  uint32_t cnt[NBIN];
  u64 fix[NBIN];
  u64 mk[NBIN];
};
constexpr size_t HIST_BYTES = RNB * 8;
static_assert(RRING * sizeof(RadixSlot) <= HIST_BYTES, "the ring fits");
static_assert(HIST_BYTES + RCAP * 8 <= BIGCAP * 8 && BIGCAP <= KEYS_CAP, "an open row's areas fit the smaller list area");

// The edits of one logit gathered in one LDS word: bits 0-28 its count among the generated tokens, 29 an entry of the
// (id, count) table, 30 suppressed (before the penalties), 31 stop-masked (after them).
constexpr uint32_t EW_STOP = 1u << 31, EW_SUPP = 1u << 30, EW_TAB = 1u << 29, EW_COUNT = EW_TAB - 1;
constexpr uint32_t EW_MAX = EW_COUNT / 2;  // counts above it do not go through the words

template <int DT>
struct BTraits;
template <>
struct BTraits<VS_F32> {
  static constexpr uint32_t NEG_INF_WORD = 0xFF800000u;
  __device__ static float get(const uint4& r, int q) {
    return __uint_as_float(q == 0 ? r.x : q == 1 ? r.y : q == 2 ? r.z : r.w);
  }
};
template <>
struct BTraits<VS_BF16> {
  static constexpr uint32_t NEG_INF_WORD = 0xFF80FF80u;
  __device__ static float get(const uint4& r, int q) {
    const uint32_t w = q < 2 ? r.x : q < 4 ? r.y : q < 6 ? r.z : r.w;
    return __uint_as_float((q & 1) ? (w & 0xFFFF0000u) : (w << 16));
  }
};
template <>
struct BTraits<VS_F16> {
  static constexpr uint32_t NEG_INF_WORD = 0xFC00FC00u;
  __device__ static float get(const uint4& r, int q) {
    const uint32_t w = q < 2 ? r.x : q < 4 ? r.y : q < 6 ? r.z : r.w;
    return f16_to_f32((uint16_t)((q & 1) ? (w >> 16) : (w & 0xFFFFu)));
  }
};

// A row's parameters and where its logits lie.
struct RowIn {
  vs_row_params P;
  vs_row_state st;
  uint64_t rng_next;
  const char* line;  // the 16-byte line the row's first logit lies in, mis logits before it
  int mis, vlim;
  bool argmax_vv, pen, has_tab, has_raw, edits;
  int64_t tabn;
  const int2* tab;
};

template <int DT>
__device__ __forceinline__ void row_place(const SampleArgs& A, int grow, RowIn& R) {
  constexpr int ES = 16 / DTraits<DT>::VEC;
  const char* rowb = (const char*)A.logits + (int64_t)grow * A.ld * ES;
  R.mis = (int)((uintptr_t)rowb & 15) / ES;
  R.line = rowb - R.mis * ES;
}

// The row's parameters, the draw and history of the state entry point (see vs_sample_kernel).
__device__ __forceinline__ void row_params(const SampleArgs& A, int grow, RowIn& R) {
  const int srow = A.slots ? A.slots[grow] : grow;
  if (A.params) {
    R.P = A.params[srow];
  } else {  // top-list mode: plain logits, top_k = list_k, no edits
    R.P = vs_row_params{1.0f, 1.0f, 0.0f, 0.0f, A.list_k, 0u, 1.0, 0.0, 0.0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  }
  R.st = vs_row_state{};
  R.rng_next = 0;
  vs_row_params& P = R.P;
  if (A.state) {
    R.st = A.state[srow];
    R.rng_next = xorshift64s_step(R.st.rng);
    P.u = xorshift64s_uniform(R.rng_next);
    P.hist_begin = R.st.hist_off + R.st.hist_base;
    P.hist_end = R.st.hist_off + R.st.hist_len;
    if (R.st.produced >= R.st.min_new_tokens) P.stop_end = P.stop_begin;
  }
  R.argmax_vv = (P.flags & VS_ROW_ARGMAX_VV) && (P.flags & VS_ROW_GREEDY) && P.stop_end == P.stop_begin;
  R.vlim = R.argmax_vv ? min(A.V, P.vocab_valid) : A.V;
  if (R.argmax_vv) P.bias_end = P.bias_begin, P.supp_end = P.supp_begin, P.hist_end = P.hist_begin;
  const bool pairs = (P.flags & VS_ROW_HIST_PAIRS) && !A.state;
  R.tabn = pairs ? (P.hist_end - P.hist_begin) >> 1 : ((A.state && A.tabs) ? (int64_t)R.st.tab_len : 0);
  R.tab = (const int2*)(pairs ? A.hist + P.hist_begin : (A.tabs ? A.tabs + R.st.tab_off : nullptr));
  R.pen = A.has_hist && !R.argmax_vv &&
          (P.repetition_penalty != 1.0f || P.frequency_penalty != 0.0f || P.presence_penalty != 0.0f);
  R.has_tab = R.pen && R.tabn > 0;
  R.has_raw = R.pen && !pairs && P.hist_end > P.hist_begin;
  R.edits = R.has_tab || R.has_raw || P.supp_end > P.supp_begin || P.stop_end > P.stop_begin;
}

// A tile of a row: positions [p0, p1), counted from R.line, so that every load is aligned whatever the row stride;
// position p is logit p - mis. Lane t holds positions p0 + (j SNT + t) VEC + q in v[j VEC + q]. All loads in flight.
template <int DT, int NVL>
__device__ __forceinline__ void tile_load(const RowIn& R, int p0, int p1, uint4 (&raw)[NVL]) {
  typedef typename DTraits<DT>::LT LT;
  constexpr int VEC = DTraits<DT>::VEC;
  constexpr uint32_t NI = BTraits<DT>::NEG_INF_WORD;
#pragma unroll
  for (int j = 0; j < NVL; ++j) {
    const int p = p0 + (j * SNT + (int)threadIdx.x) * VEC;
    raw[j] = make_uint4(NI, NI, NI, NI);
    if (p >= R.mis && p + VEC <= p1) raw[j] = *(const uint4*)((const LT*)R.line + p);
  }
}

// What a row's edits need from memory, loaded together as soon as the row's parameters are there: one latency instead of
// one for each kind of edit, which come one after another in tile_edit (128 mixed requests at V = 163840 fp32: 46.8 us a
// call with each list read where it is used, 45.5 with all of them read here). A field is meaningful where its kind has entries.
constexpr int AHEAD_TAB = 4;  // table entries per lane; a longer table is probed first
struct EditAhead {
  int supp, stop, bias, bias_before;  // ids
  int2 tab[AHEAD_TAB];
  int32_t one;   // of the raw history's unaligned head and tail
  int4 raw[HB];  // its first batch
};
__device__ __forceinline__ void edit_ahead(const SampleArgs& A, const RowIn& R, EditAhead& H) {
  const int t = threadIdx.x;
  const vs_row_params& P = R.P;
  if (P.bias_end > P.bias_begin) {
    const int p = min(P.bias_begin + t, P.bias_end - 1);
    H.bias = A.bias_ids[p];
    H.bias_before = A.bias_ids[max(p - 1, P.bias_begin)];
  }
  if (P.supp_end > P.supp_begin) H.supp = A.mask_ids[min(P.supp_begin + t, P.supp_end - 1)];
  if (P.stop_end > P.stop_begin) H.stop = A.mask_ids[min(P.stop_begin + t, P.stop_end - 1)];
  if (R.has_tab) {
    const bool probe = R.tabn > AHEAD_TAB * SNT;
    H.tab[0] = R.tab[probe ? probe_at(R.tabn, t) : min((int64_t)t, R.tabn - 1)];
#pragma unroll
    for (int u = 1; u < AHEAD_TAB; ++u)
      if (!probe && u * SNT < R.tabn) H.tab[u] = R.tab[min((int64_t)(u * SNT + t), R.tabn - 1)];
  }
  if (R.has_raw) {
    const HistWin w = hist_window(P.hist_begin, P.hist_end);
    const int nh = (int)(w.a - w.b), nt = (int)(w.e - (w.a + w.nv * 4));
    H.one = -1;
    if (t < nh + nt) H.one = A.hist[t < nh ? w.b + t : w.a + w.nv * 4 + (t - nh)];
    if (w.nv > 0) hist_load(A.hist, w, t, H.raw);
  }
}

// The tile as float32 with the logit edits and penalties (sampler.py:104-126; float32 throughout) applied; positions
// that hold no logit of the row read -inf. X: SNT * NVL * VEC words of LDS, free again on return; red: NRED ints.
template <int DT, int NVL>
__device__ __forceinline__ void tile_edit(const SampleArgs& A, const RowIn& R, const EditAhead& H, int p0, int p1,
                                          const uint4 (&raw)[NVL], float (&v)[NVL * DTraits<DT>::VEC], uint32_t* X, int* red) {
  typedef DTraits<DT> TR;
  typedef typename TR::LT LT;
  constexpr int VEC = TR::VEC, E = NVL * VEC;
  const int t = threadIdx.x, mis = R.mis;
  const vs_row_params& P = R.P;
#pragma unroll
  for (int j = 0; j < NVL; ++j)
#pragma unroll
    for (int q = 0; q < VEC; ++q) v[j * VEC + q] = BTraits<DT>::get(raw[j], q);
  // the row's first and last line, where a 16-byte word is not all the row's
  if (p0 < mis || ((p1 & (VEC - 1)) != 0 && p1 == A.V + mis)) {
#pragma unroll
    for (int j = 0; j < NVL; ++j) {
      const int p = p0 + (j * SNT + t) * VEC;
      if (p < p1 && !(p >= mis && p + VEC <= p1)) {
#pragma unroll
        for (int q = 0; q < VEC; ++q)
          if (p + q >= mis && p + q < p1) v[j * VEC + q] = TR::cv(((const LT*)R.line)[p + q]);
      }
    }
  }
  if (p1 - mis > R.vlim) {
#pragma unroll
    for (int i = 0; i < E; ++i)
      if (p0 + ((i / VEC) * SNT + t) * VEC + i % VEC - mis >= R.vlim) v[i] = -__builtin_inff();
  }
  const float rep = P.repetition_penalty, fpen = P.frequency_penalty, ppen = P.presence_penalty;
  const int l0 = p0 - mis;  // the logit of the tile's first position
  const int lo = max(l0, 0), hi = p1 - mis;
  float* F = (float*)X;
  auto put = [&]() {
#pragma unroll
    for (int i = 0; i < E; ++i) F[((i / VEC) * SNT + t) * VEC + i % VEC] = v[i];
    __syncthreads();
  };
  auto take = [&]() {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = F[((i / VEC) * SNT + t) * VEC + i % VEC];
    __syncthreads();
  };
  if (P.bias_end > P.bias_begin) {  // :104-109; ids sorted, equal ids in application order: one lane per run
    put();
    for (int p = P.bias_begin + t; p < P.bias_end; p += SNT) {
      const bool first = p < P.bias_begin + SNT;
      const int id = first ? H.bias : A.bias_ids[p];
      if (id >= lo && id < hi && (p == P.bias_begin || (first ? H.bias_before : A.bias_ids[p - 1]) != id)) {
        float y = F[id - l0];
        for (int q = p; q < P.bias_end && A.bias_ids[q] == id; ++q) y = y + A.bias_vals[q];
        F[id - l0] = y;
      }
    }
    take();
  }
  if (!R.edits) return;
#pragma unroll
  for (int j = 0; j < E / 4; ++j) ((uint4*)X)[j * SNT + t] = make_uint4(0, 0, 0, 0);
  uint32_t* W = X + (lo - l0);  // W[id - lo]
  const uint32_t len = (uint32_t)max(hi - lo, 0);
  int64_t q0 = 0, q1 = R.has_tab ? R.tabn : 0;
  bool huge = false;
  __syncthreads();
  for (int p = P.supp_begin + t; p < P.supp_end; p += SNT) {  // :110-112
    const uint32_t o = (uint32_t)((p < P.supp_begin + SNT ? H.supp : A.mask_ids[p]) - lo);
    if (o < len) atomicOr(&W[o], EW_SUPP);
  }
  for (int p = P.stop_begin + t; p < P.stop_end; p += SNT) {  // :123-126
    const uint32_t o = (uint32_t)((p < P.stop_begin + SNT ? H.stop : A.mask_ids[p]) - lo);
    if (o < len) atomicOr(&W[o], EW_STOP);
  }
  if (R.has_tab) {  // :113-122, the counts of a table (ids ascending and unique)
    auto count = [&](int2 e) {
      const uint32_t o = (uint32_t)(e.x - lo);
      if (o < len) {
        if ((uint32_t)e.y > EW_MAX) huge = true;
        else atomicAdd(&W[o], EW_TAB + (uint32_t)e.y);
      }
    };
    if (R.tabn <= AHEAD_TAB * SNT) {  // every workgroup looks at all of them: cheaper than the probes' second latency
#pragma unroll
      for (int u = 0; u < AHEAD_TAB; ++u)
        if (u * SNT + t < R.tabn) count(H.tab[u]);
    } else {  // the entries of [lo, hi) lie between two probes
      pair_range(R.tabn, H.tab[0].x, lo, hi, red, &q0, &q1);
      for (int64_t p = q0 + t; p < q1; p += SNT) count(R.tab[p]);
    }
  }
  if (R.has_raw) {  // :113-122, the tokens themselves
    const HistWin w = hist_window(P.hist_begin, P.hist_end);
    const int32_t one[1] = {H.one};
    hist_add_ids(one, lo, hi, W);
    auto count = [&](const int4 (&r)[HB], int64_t v0) {
      int32_t tk[4 * HB];
#pragma unroll
      for (int u = 0; u < HB; ++u) {
        const bool ok = v0 + (int64_t)u * SNT + t < w.nv;
        tk[4 * u] = ok ? r[u].x : -1;
        tk[4 * u + 1] = ok ? r[u].y : -1;
        tk[4 * u + 2] = ok ? r[u].z : -1;
        tk[4 * u + 3] = ok ? r[u].w : -1;
      }
      hist_add_ids(tk, lo, hi, W);
    };
    constexpr int64_t BATCH = (int64_t)SNT * HB;
    if (w.nv > 0) count(H.raw, 0);
    for (int64_t v0 = BATCH; v0 < w.nv; v0 += (HD - 1) * BATCH) {  // the loads of a round are in flight together
      int4 r[HD - 1][HB];
#pragma unroll
      for (int d = 0; d < HD - 1; ++d) hist_load(A.hist, w, v0 + d * BATCH + t, r[d]);
#pragma unroll
      for (int d = 0; d < HD - 1; ++d)
        if (v0 + d * BATCH < w.nv) count(r[d], v0 + d * BATCH);
    }
  }
  const bool anyhuge = __syncthreads_or(huge);
#pragma unroll
  for (int j = 0; j < NVL; ++j) {
#pragma unroll
    for (int h = 0; h < VEC / 4; ++h) {
      const uint4 w4 = ((const uint4*)X)[(j * SNT + t) * (VEC / 4) + h];
      const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
      if ((w4.x | w4.y | w4.z | w4.w) != 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (w[q] != 0) {
            float y = (w[q] & EW_SUPP) ? -__builtin_inff() : v[j * VEC + h * 4 + q];
            if (w[q] & (EW_TAB | EW_COUNT)) {
              const uint32_t c = w[q] & EW_COUNT;
              if (rep != 1.0f) {
                const float dv = y / rep, ml = y * rep;
                y = y > 0.0f ? dv : ml;
              }
              const float fc = fpen * (float)c;
              const float sub = fc + (c > 0 ? ppen : 0.0f);
              y = y - sub;
            }
            v[j * VEC + h * 4 + q] = (w[q] & EW_STOP) ? -__builtin_inff() : y;
          }
        }
      }
    }
  }
  __syncthreads();  // the words are read: the area is free
  if (__builtin_expect(anyhuge, 0)) {  // table entries whose counts do not fit the words: edited one by one
    put();
    for (int64_t p = q0 + t; p < q1; p += SNT) {
      const int2 e = R.tab[p];
      const uint32_t o = (uint32_t)(e.x - lo);
      if (o < len && (uint32_t)e.y > EW_MAX) {
        float y = F[e.x - l0];
        if (rep != 1.0f) {
          const float dv = y / rep, ml = y * rep;
          y = y > 0.0f ? dv : ml;
        }
        const float fc = fpen * (float)e.y;
        F[e.x - l0] = y - (fc + (e.y > 0 ? ppen : 0.0f));
      }
    }
    take();
  }
}

// exp(x/t - max/t), sampler.py:141-142 (below e^-150, a float zero, the argument would only overflow in exp_nonpos)
__device__ __forceinline__ float mass_at(float d) { return exp_nonpos(fmaxf(d, -150.0f)); }

// sampler.py:144-156 on the n largest keys of a row, sorted descending in LDS, where S is the mass of the row's whole
// kept set (n <= 64 * EM keys reach past every cut: see the merge). `total` is the size of the kept set, -1 where it is
// not known (then top-p or min-p cuts it); `mend`: every key of the row past these n fails min-p. Lane layout and order
// of sums as in wave_sample_em. Lane 0 leaves token, keep, flags and logprob in LDS, misc[0] = 0 if a cut or the draw was
// not found among the keys after all.
template <int EM>
__device__ __forceinline__ void wave_sample_tail(const u64* a, int n, double S, int total, bool mend,
                                                 const vs_row_params& P, int* misc, double* lp) {
  const int L = threadIdx.x;
  const int E = (n + WAVE - 1) / WAVE;
  const int i0 = L * E;
  const float tt = P.temperature;
  const float xs0 = key_value(a[0]) / tt;
  double pr[EM];
  double ls = 0.0;
#pragma unroll
  for (int q = 0; q < EM; ++q) {
    pr[q] = 0.0;
    if (q < E && i0 + q < n) {
      pr[q] = (double)mass_at(key_value(a[i0 + q]) / tt - xs0) / S;
      ls += pr[q];
    }
  }
  const double base = wave_scan(ls) - ls;
  uint32_t flags = 0;
  bool ok = true;
  int keep = total;
  if (P.top_p < 1.0) {  // :145-148 first position with cumsum >= top_p
    const double tp = P.top_p;
    double c = base;
    int hit = -1, fb = 0;
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
      const int ln = __ffsll((long long)hb) - 1;
      keep = lane_bcast(hit, ln) + 1;
      if (lane_bcast(fb, ln)) flags |= VS_OUT_TOPP_BOUNDARY;
    } else {
      keep = -1;
    }
  }
  if (P.min_p > 0.0) {  // :149-152 first position with pr < pr[0] * min_p
    const double thr = lane_bcast(pr[0], 0) * P.min_p;
    int hit = -1;
#pragma unroll
    for (int q = 0; q < EM; ++q)
      if (hit < 0 && q < E && i0 + q < n && pr[q] < thr) hit = i0 + q;
    const unsigned long long hb = __ballot(hit >= 0);
    if (hb || mend) {
      int cnt = hb ? lane_bcast(hit, __ffsll((long long)hb) - 1) : n;
      cnt = cnt > 1 ? cnt : 1;
      keep = keep < 0 || cnt < keep ? cnt : keep;
    } else if (keep < 0 || keep > n) {
      ok = false;
    }
  }
  ok = ok && keep > 0;
  double z = 1.0;  // :153: the mass through the last kept position, all of S when nothing cuts the kept set
  if (P.top_p < 1.0 || P.min_p > 0.0) {
    const int last = keep > 0 ? (keep <= n ? keep - 1 : n - 1) : 0;
    ok = ok && keep <= n;
    const int owner = last / E, qq = last - owner * E;
    double cz = base;
#pragma unroll
    for (int q = 0; q < EM; ++q)
      if (q <= qq && q < E) cz += pr[q];
    z = lane_bcast(cz, owner);
  }
  const double uz = P.u * z;  // :154
  const int nd = keep < n ? keep : n;
  double c = base;
  int hit = -1;
  double hp = 0.0, hc = 0.0;
#pragma unroll
  for (int q = 0; q < EM; ++q) {
    if (q < E && i0 + q < nd) {
      c += pr[q];
      if (hit < 0 && c >= uz) {
        hit = i0 + q;
        hp = pr[q];
        hc = c;
      }
    }
  }
  const unsigned long long hb = __ballot(hit >= 0);
  int j = 0;
  if (hb) {  // :155
    const int ln = __ffsll((long long)hb) - 1;
    j = lane_bcast(hit, ln);
    hp = lane_bcast(hp, ln);
    hc = lane_bcast(hc, ln);
  } else if (ok && nd == keep) {  // :156 min(j, keep - 1): the last kept position
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
  } else {
    ok = false;
  }
  if (L == 0) {
    const double tol = 1e-6 * z;
    if (fabs(hc - uz) < tol || (j >= 1 && fabs(hc - hp - uz) < tol)) flags |= VS_OUT_DRAW_BOUNDARY;
    misc[0] = ok ? 1 : 0;
    misc[1] = (int)key_index(a[j]);
    misc[2] = keep;
    misc[3] = (int)flags;
    // from the difference itself and the kept mass, not from the token's rounded mass: a mean error of 1e-7 less
    *lp = ok ? (double)(key_value(a[j]) / tt - xs0) - log_ge1(z * S) : 0.0;
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Pass over the logits. What bounds it: the chain load - edits - bound - list of each workgroup with two or three of
// them per CU (128 mixed requests at V = 163840 fp32: 32.8 us for 84 MB, 2.6 TB/s; the vector instructions alone would
// take 12 us). Nothing waits on anything outside the workgroup, and the lists travel by plain stores: with the merge in
// the row's last workgroup instead of a launch of its own this kernel took 52 us (arrivals, 128 merges of 11 us each in
// workgroups that hold stream slots, and an XCD a little behind the others arriving last in every row and so getting
// most of the merges).
// ---------------------------------------------------------------------------------------------------------------
struct StreamLds {
  u64 key[SNW];
  double sum[SNW];
  float wmax[SNW], wmin[SNW];
  uint32_t wb[SNW];
  int got[SNW], nf[SNW], segc[SNW];
  int red[NRED];
};
__host__ __device__ constexpr size_t stream_lds(int tile) {  // the edit words, later the waves' staged candidates
  return (size_t)tile * 4 > SNW * SEG_CAP * 8 ? (size_t)tile * 4 : SNW * SEG_CAP * 8;
}

template <int DT, int NVL>
__global__ __launch_bounds__(SNT, 4) void vs_batch_kernel(SampleArgs A) {
  constexpr int VEC = DTraits<DT>::VEC;
  constexpr int E = NVL * VEC;  // logits per lane
  extern __shared__ __align__(16) char smem_raw[];
  __shared__ StreamLds s;
  const int t = threadIdx.x, wv = t / WAVE, ln = lane_id();
  const int row = (int)blockIdx.x / A.G, g = (int)blockIdx.x - row * A.G;
  const int grow = A.row0 + row;
  VS_TR_DECL(A);
  VS_TR(A, 0);
  RowIn R;
  row_place<DT>(A, grow, R);
  const int p0 = g * A.CH;
  const int p1 = max(p0, min(A.V + R.mis, p0 + A.CH));  // an empty chunk where the last one holds only padding
  uint4 raw[NVL];
  tile_load<DT, NVL>(R, p0, p1, raw);
  row_params(A, grow, R);
  const vs_row_params& P = R.P;
  if (__builtin_expect((P.flags & VS_ROW_FORCE) != 0, 0)) return;  // the logits are not read
  EditAhead H;
  edit_ahead(A, R, H);
  VS_TR(A, 1);
  float v[E];
  tile_edit<DT, NVL>(A, R, H, p0, p1, raw, v, (uint32_t*)smem_raw, s.red);
  VS_TR(A, 2);

  const int top_k = P.top_k;
  const int cls = (P.flags & VS_ROW_GREEDY) ? CLS_GREEDY : ((top_k >= 1 && top_k <= A.kmax) ? CLS_TOPK : CLS_FULL);
  Part* part = (Part*)part_area(A.ws, row) + g;
  u64* list = (u64*)list_area(A.ws, row) + (size_t)g * A.kcap;
  const int l0 = p0 - R.mis;
  constexpr float L2E = 1.44269504088896340736f;
  // the lane's largest value, and whether it holds a NaN or an infinity (x * 0 is NaN then)
  float best = -__builtin_inff(), zero[2] = {0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < E; i += 2) {
    best = max3f(best, v[i], v[i + 1]);
    zero[0] = __builtin_fmaf(v[i], 0.0f, zero[0]);
    zero[1] = __builtin_fmaf(v[i + 1], 0.0f, zero[1]);
  }
  const bool odd = !(zero[0] + zero[1] == 0.0f);

  if (cls == CLS_GREEDY) {
    // ---- sampler.py:127-128: np.argmax(x), first maximum; logprob = log-softmax of the processed row ----
    // The largest finite logit first; the key only in the waves that hold the chunk's maximum (or a NaN or an infinity,
    // where the key's order decides element by element).
    const bool wodd = __any(odd);
    float mf = best;
    if (wodd) {
      mf = -__builtin_inff();
#pragma unroll
      for (int i = 0; i < E; ++i) mf = fmaxf(mf, is_finite(v[i]) ? v[i] : -__builtin_inff());
    }
    mf = wave_max_dpp(mf);
    if (ln == 0) s.wmax[wv] = mf;
    __syncthreads();
    float m = s.wmax[0];
#pragma unroll
    for (int i = 1; i < SNW; ++i) m = fmaxf(m, s.wmax[i]);
    u64 am = 0;
    if (wodd) {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int id = l0 + ((i / VEC) * SNT + t) * VEC + i % VEC;
        if (id >= 0 && id < R.vlim && id < p1 - R.mis) {
          const u64 k = amkey64(v[i], (uint32_t)id);
          am = k > am ? k : am;
        }
      }
      am = wave_max(am);
    } else if (mf == m) {
      int bi = 1 << 30;
#pragma unroll
      for (int i = E - 1; i >= 0; --i) bi = v[i] == m ? (i / VEC) * SNT * VEC + i % VEC : bi;
      bi = wave_min(bi + t * VEC);
      am = amkey64(m, (uint32_t)(l0 + bi));
    }
    double se = 0.0;
    if (is_finite(m)) {
      float a4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (wodd) {
#pragma unroll
        for (int i = 0; i < E; ++i)
          a4[i % 4] += __builtin_amdgcn_exp2f(is_finite(v[i]) ? (v[i] - m) * L2E : -__builtin_inff());
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) a4[i % 4] += __builtin_amdgcn_exp2f((v[i] - m) * L2E);
      }
      se = wave_sum_dpp(((double)a4[0] + (double)a4[1]) + ((double)a4[2] + (double)a4[3]));
    }
    if (ln == 0) {
      s.key[wv] = am;
      s.sum[wv] = se;
    }
    __syncthreads();
    if (t == 0) {
      u64 k = 0;
      double e = 0.0;
#pragma unroll
      for (int i = 0; i < SNW; ++i) {
        k = s.key[i] > k ? s.key[i] : k;
        e += s.sum[i];
      }
      part->amkey = k;
      part->mf = m;
      part->se = e;
    }
    VS_TR(A, 7);
    VS_TR_FLUSH(A);
    return;
  }

  // ---- TOPK and FULL rows: finite logits only (sampler.py:130), anything else becomes -inf ----
  const bool full = cls == CLS_FULL;
  const int k = full ? A.NV : top_k;
  int nf = E;
  if (__builtin_expect(odd, 0)) {
    nf = 0;
    best = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const bool f = is_finite(v[i]);
      nf += f ? 1 : 0;
      v[i] = f ? v[i] : -__builtin_inff();
      best = fmaxf(best, v[i]);
    }
  }
  VS_TR(A, 3);
  // Lower bound of the chunk's k-th largest logit from the lane maxima: see lane_max_bound (here with the waves' maxima
  // and finite counts in the same exchange).
  uint32_t L;
  float wm, mn = 0.0f;  // the chunk's largest (-inf: none) and smallest finite logit
  {
    const uint32_t tmax = nf ? ord32(best) : 0u;
    const int q = (k + SNW - 1) / SNW;
    const int nz = __popcll(__ballot(tmax != 0));
    const int got = nz < q ? nz : q;
    uint32_t wb = 0;
    if (got > 0) {
      for (int b = 31; b >= 32 - BOUND_BITS; --b) {
        const uint32_t c = wb | (1u << b);
        if ((int)__popcll(__ballot(tmax >= c)) >= got) wb = c;
      }
    }
    const float wmx = wave_max_dpp(best);
    const int wnf = __any(odd) ? wave_sum_dpp(nf) : WAVE * E;
    if (full) {  // the smallest finite logit, which tells whether the exp(-40) filter drops any
      mn = __builtin_inff();
#pragma unroll
      for (int i = 0; i < E; i += 2) mn = min3f(mn, v[i], v[i + 1]);
      if (nf < E) {
        mn = __builtin_inff();
#pragma unroll
        for (int i = 0; i < E; ++i) mn = is_finite(v[i]) && v[i] < mn ? v[i] : mn;
      }
      mn = wave_min_dpp(mn);
    }
    if (ln == 0) {
      s.wb[wv] = wb;
      s.got[wv] = got;
      s.nf[wv] = wnf;
      s.wmax[wv] = wmx;
      s.wmin[wv] = mn;
    }
    __syncthreads();
    L = ~0u;
    wm = -__builtin_inff();
    int tot = 0;
    nf = 0;
#pragma unroll
    for (int i = 0; i < SNW; ++i) {
      const uint32_t bi = s.got[i] > 0 ? s.wb[i] : ~0u;
      L = bi < L ? bi : L;
      tot += s.got[i];
      nf += s.nf[i];
      wm = fmaxf(wm, s.wmax[i]);
      mn = i == 0 ? s.wmin[0] : fminf(mn, s.wmin[i]);
    }
    L = tot >= k ? L : 0u;
  }
  VS_TR(A, 4);
  // Candidates: finite logits >= the bound (every finite one without a bound). Each wave appends its own to its
  // segment by ballots (no atomics); a FULL row adds up the mass of the others, relative to the chunk's maximum.
  // (A staged candidate is its bits and its place; the key is made on the way out.)
  const float Lf = L ? inv_ord32(L) : -__FLT_MAX__;
  uint2* seg = (uint2*)smem_raw + wv * SEG_CAP;
  int cw = 0;
  auto stage = [&](int i, bool c) {
    const unsigned long long m = __ballot(c);
    if (m) {
      const int pos =
          (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)cw));
      if (c && pos < SEG_CAP) seg[pos] = make_uint2(__float_as_uint(v[i]), (uint32_t)(((i / VEC) * SNT + t) * VEC + i % VEC));
      cw += (int)__popcll(m);
    }
  };
  double rest = 0.0;
  if (full && nf > 0) {
    // x/t rounded as in sampler.py:141, by the rounded reciprocal and the quotient's remainder; its exponential to 2 ulp
    // (as exp_nonpos); four of them at a time added as a tree, then float64. With (x - max) (log2 e / t) in the exponent and
    // sums of eight the mass was off by up to 1e-6 for tied values 15 to 20 nats down, and all to one side for some t.
    const float tt = P.temperature, rt = 1.0f / tt, xw = wm / tt, low = -150.0f;
    constexpr float L2E_LO = 1.9259629891e-8f;  // log2(e) less L2E
#pragma unroll
    for (int i0 = 0; i0 < E; i0 += 4) {
      float e[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = v[i0 + j], q = x * rt;
        const bool in = x >= Lf;
        // (a NaN, from an x of -inf, becomes the lower limit, whose mass is a float zero)
        const float d = max3f(__builtin_fmaf(__builtin_fmaf(-q, tt, x), rt, q) - xw, low, low);
        const float y = d * L2E, yl = __builtin_fmaf(d, L2E_LO, __builtin_fmaf(d, L2E, -y));
        const float m = __builtin_amdgcn_exp2f(y);
        e[j] = in ? 0.0f : __builtin_fmaf(m, yl * 0.693147180559945309f, m);
        stage(i0 + j, in);
      }
      rest += (double)((e[0] + e[1]) + (e[2] + e[3]));
    }
    rest = wave_sum_dpp(rest);
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) stage(i, v[i] >= Lf);
  }
  VS_TR(A, 5);
  if (ln == 0) {
    s.segc[wv] = cw;
    s.sum[wv] = rest;
  }
  __syncthreads();
  {
    int C, off;
    bool bad;
    auto total = [&]() {
      C = off = 0;
      bad = false;
#pragma unroll
      for (int i = 0; i < SNW; ++i) {
        off += i < wv ? s.segc[i] : 0;
        C += s.segc[i];
        bad = bad || s.segc[i] > SEG_CAP;
      }
      bad = bad || C > A.kcap;
    };
    total();
    if (__builtin_expect(bad && !full, 0)) {
      // The bound lets about 1.7 k logits through, runs of tied values all of them. A TOPK list needs its k largest keys:
      // a bisection for a bound that leaves at least k and no more than fit, on the value, then, where one value is left
      // and still too many hold it, on the place. It ends at the first bound that does, exactly at k otherwise. Without
      // it such a row was resolved by a radix select over passes (top_k 200, 20 rows of V = 248320 bf16: 243 us a call
      // against 83 in launches of vs_sample_kernel).
      int step = 0, cnt;
      bool fits;
      auto count = [&](auto pred) {  // two sets of words in turn: one barrier a step
        int c = 0;
#pragma unroll
        for (int i = 0; i < E; ++i) c += (int)__popcll(__ballot(pred(i)));
        int* x = s.red + (step++ & 1) * SNW;
        if (ln == 0) x[wv] = c;
        __syncthreads();
        cnt = 0;
        fits = true;
#pragma unroll
        for (int i = 0; i < SNW; ++i) {
          cnt += x[i];
          fits = fits && x[i] <= SEG_CAP;
        }
        fits = fits && cnt <= A.kcap;
      };
      auto place = [&](int i) -> int { return ((i / VEC) * SNT + t) * VEC + i % VEC; };  // of v[i], in the order of the ids
      uint32_t lo = L ? L : ord32(-__FLT_MAX__), hi = ord32(wm) + 1;  // too many from lo up, fewer than k from hi up
      fits = false;
      while (!fits && hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        const float f = inv_ord32(mid);
        count([&](int i) { return v[i] >= f; });
        if (cnt < k) {
          hi = mid;
          fits = false;
        } else {
          lo = mid;
        }
      }
      const float f = inv_ord32(lo);
      int pl = -1, ph = SNT * E;  // f's places up to pl are too few, up to ph enough
      while (!fits && ph - pl > 1) {
        const int mid = (pl + ph) / 2;
        count([&](int i) { return v[i] > f || (v[i] == f && place(i) <= mid); });
        if (cnt < k) {
          pl = mid;
          fits = false;
        } else {
          ph = mid;
        }
      }
      L = lo;
      cw = 0;
#pragma unroll
      for (int i = 0; i < E; ++i) stage(i, v[i] > f || (v[i] == f && place(i) <= ph));
      if (ln == 0) s.segc[wv] = cw;
      __syncthreads();
      total();
    }
    if (!bad)
      for (int j = ln; j < cw; j += WAVE) list[off + j] = key64(__uint_as_float(seg[j].x), (uint32_t)l0 + seg[j].y);
    if (t == 0) {
      double r = 0.0;
#pragma unroll
      for (int i = 0; i < SNW; ++i) r += s.sum[i];
      part->nfin = (uint32_t)nf;
      part->kc = (uint32_t)C;
      part->heads[1] = bad ? L_NONE : L;  // (the tag word `pad` is vs_sample_kernel's alone)
      part->heads[0] = ((u64)__float_as_uint(wm) << 32) | __float_as_uint(mn);
      part->se = r;
    }
  }
  VS_TR(A, 6);
  VS_TR_FLUSH(A);
}

// ---------------------------------------------------------------------------------------------------------------
// One workgroup per row finishes it from the lists, or leaves it open. A chain of small steps (8 us for top-k rows, 12.6
// us with FULL rows among 128 mixed ones): the loads, value bins over the keys, the cut bin, the keys down to it ranked, the
// draw in one wave.
// ---------------------------------------------------------------------------------------------------------------
struct FinishLds {
  uint32_t hc[NBIN];  // counts by value bin
  uint32_t at[NBIN];  // the next place of each bin
  u64 hf[NBIN];       // masses, in fixed point (at 2^50): the same sums in any order
  u64 sel[BSEL];      // the keys to rank
  u64 tk[BSEL];       // ranked
  double sum[NRED];
  int nz[SNW];
  int cnt[2 * SNW];
  int misc[8];
};

__global__ __launch_bounds__(SNT, 4) void vs_finish_kernel(SampleArgs A) {
  __shared__ FinishLds s;
  const int t = threadIdx.x, wv = t / WAVE, ln = lane_id();
  const int G = A.G, row = blockIdx.x, grow = A.row0 + row;
  const Part* parts = (const Part*)part_area(A.ws, row);
  const u64* lists = (const u64*)list_area(A.ws, row);
  uint8_t* flag = open_flag(A.ws, row);
  VS_TR_DECL(A);
  VS_TR(A, 0);
  // every list's summary, in every wave (a greedy row's: its key, maximum and sum)
  const Part pp = parts[ln < G ? ln : 0];
  if (t < NBIN) {
    s.hc[t] = 0;
    s.hf[t] = 0;
  }
  if (t == 0) s.misc[4] = 0;
  RowIn R;
  row_params(A, grow, R);
  const vs_row_params& P = R.P;
  if (__builtin_expect((P.flags & VS_ROW_FORCE) != 0, 0)) {  // sampler.py:88-90
    if (t == 0) *flag = ROW_DONE;
    Final f;
    f.token = P.force_token;
    f.lp = 0.0f;
    f.flags = VS_OUT_FORCED;
    f.keep = 0;
    write_out(A, row, f, R.st, 0);
    return;
  }
  const int top_k = P.top_k;
  const int cls = (P.flags & VS_ROW_GREEDY) ? CLS_GREEDY : ((top_k >= 1 && top_k <= A.kmax) ? CLS_TOPK : CLS_FULL);
  if (cls == CLS_GREEDY) {
    if (t < WAVE) {
      const float L2E = 1.44269504088896340736f;
      const u64 bam = wave_max(ln < G ? pp.amkey : (u64)0);
      const float M = wave_max(ln < G ? pp.mf : -__builtin_inff());
      const double S = wave_sum((ln < G && pp.se > 0.0 && is_finite(M))
                                    ? pp.se * (double)__builtin_amdgcn_exp2f((pp.mf - M) * L2E)
                                    : 0.0);
      const float xj = am_is_nan(bam) ? __builtin_nanf("") : key_value(bam);
      Final f;
      f.token = (int32_t)key_index(bam);
      // log(S) = log1p(S - 1): S >= 1 holds the maximum's own term
      f.lp = (is_finite(xj) && S > 0.0) ? (float)((double)xj - ((double)M + (double)log1pf((float)(S - 1.0)))) : 0.0f;
      f.flags = VS_OUT_GREEDY;
      f.keep = 0;
      if (t == 0) *flag = ROW_DONE;
      write_out(A, row, f, R.st, R.rng_next);
    }
    return;
  }
  const bool full = cls == CLS_FULL;
  const int k = full ? A.NV : top_k;
  const int cg = ln < G ? (int)pp.kc : 0;           // list ln's length
  const uint32_t pl = ln < G ? (uint32_t)pp.heads[1] : 0u;  // its bound
  const int pn = ln < G ? (int)pp.nfin : 0;
  const float pm = pn ? __uint_as_float((uint32_t)(pp.heads[0] >> 32)) : -__builtin_inff();
  const float pmn = pn ? __uint_as_float((uint32_t)pp.heads[0]) : __builtin_inff();
  const int n = wave_sum(pn);                       // finite logits of the row
  const uint32_t Lmax = wave_max(pl);
  const float xmax = wave_max(pm), xmin = wave_min(pmn);
  const float tt = P.temperature;
  const float xs0 = xmax / tt;
  // a top-k cut above the lists' reach: the chunks' bounds lie around the 64 G-th logit; sixteen times as far below the
  // maximum, and 40, lies hardly any cut, and the bins from there up are still fine (the smallest value of a row masked
  // with finite numbers says nothing)
  const uint32_t lmin = wave_min(pl != 0 ? pl : L_NONE);
  const float xcut = lmin != L_NONE ? fmaxf(xmin, xmax - fmaxf(16.0f * (xmax - inv_ord32(lmin)), 40.0f)) : xmin;
  auto leave_open = [&](int how) {
    // 63 bits for the row's mass: at most each chunk's unlisted mass and 1 for every listed logit, times the chunk's maximum
    const double most = wave_sum(pn ? (pp.se + (double)cg) * (double)expf(pm / tt - xs0) : 0.0) * 1.001;
    const int fits = most >= 1.0 && most < 1e9 ? 62 - ilogb(most) : A.fix_shift;
    const int shift = fits > A.fix_shift ? fits : A.fix_shift;
    __syncthreads();  // the partials and lists are read
    OpenRow* o = (OpenRow*)part_area(A.ws, row);
    if (t == 0) {
      *flag = (uint8_t)how;
      o->n = n;
      o->xmax = xmax;
      o->xmin = how == ROW_TOPK ? xcut : xmin;
      o->bar = o->gcnt = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o->cnt[i] = 0;
        if (i < 3) o->fix[i] = 0;
      }
      o->amkey = 0;
      o->shift = shift;
    }
    u64* h = (u64*)list_area(A.ws, row);
    for (int i = t; i < (int)(HIST_BYTES / 8); i += SNT) h[i] = 0;
  };
  if (A.list_k > 0 && n == 0) {  // top-list mode: a row without a finite logit has no entries
    for (int i = t; i < A.list_k; i += SNT) {
      A.list_ids[(size_t)grow * A.list_k + i] = -1;
      A.list_vals[(size_t)grow * A.list_k + i] = -__builtin_inff();
    }
    return;
  }
  // incomplete lists; no finite logit (sampler.py:131-132); a top-k above the lists' reach; quotients that overflow
  const bool cutk = full && top_k > 0 && top_k < n;
  if (Lmax == L_NONE || n == 0 || cutk || (full && (!(tt > 0.0f) || !is_finite(xs0) || !is_finite(xmin / tt)))) {
    const bool plain = full && n > 0 && tt > 0.0f && is_finite(xs0) && is_finite(xmin / tt);
    leave_open(!plain ? ROW_ANY : cutk ? ROW_TOPK : ROW_FLAT);
    return;
  }
  // Keys below M are not needed: of a FULL row every key from the largest bound up is listed; a chunk of a TOPK row that
  // lists k keys above its bound bounds the row's k-th key.
  const u64 M = (u64)(full ? Lmax : wave_max(cg >= k ? pl : 0u)) << 32;
  const float xlow = M ? inv_ord32((uint32_t)(M >> 32)) : xmin;
  // every key that can pass pr >= min_p pr[0] lies at or above xq
  const bool has_mp = full && P.min_p > 0.0;
  float xq = -__builtin_inff();
  if (has_mp) xq = P.min_p < 1.0 ? xmax + tt * (logf((float)P.min_p) - 1e-4f - 1e-5f * fabsf(xs0)) : xmax;
  // FULL: the mass of the unlisted logits, relative to the row's maximum
  // (the chunk's scale e^(pm/tt - xs0) with the difference's rounding made good: it is common to all of the chunk)
  const double dm = (double)(pm / tt) - (double)xs0;
  const float dmf = (float)dm;
  const double rsum =
      full ? wave_sum(pn && pp.se > 0.0 ? pp.se * ((double)mass_at(dmf) * (1.0 + (dm - (double)dmf))) : 0.0) : 0.0;
  if (full && !(has_mp && xq > xlow)) {
    // a flat row shows here: no listed logit's mass is above 1, so the lists cannot hold the share that is asked for
    const double p = P.top_p < 1.0 ? P.top_p : (has_mp ? 1.0 : P.u);
    if (p * rsum > (1.0 - p) * (double)wave_sum(cg)) {
      leave_open(ROW_FLAT);
      return;
    }
  }
  // The listed keys, in registers: wave w takes lists w, w + 8, .., each in rounds of 64 (the host keeps
  // ceil(G / 8) * ceil(kcap / 64) <= BATCH_NK).
  u64 kk[BATCH_NK];
  const int pr = max((wave_max(cg) + WAVE - 1) / WAVE, 1);
  const int nu = (G + SNW - 1) / SNW * pr;
  {
    int li = __builtin_amdgcn_readfirstlane(wv), j = 0;
#pragma unroll
    for (int u = 0; u < BATCH_NK; ++u) {
      kk[u] = 0;
      if (u < nu) {
        if (li < G && j + ln < lane_bcast(cg, li)) kk[u] = lists[(size_t)li * A.kcap + j + ln];
        j += WAVE;
        if (j >= pr * WAVE) {
          j = 0;
          li += SNW;
        }
      }
    }
  }
  const int keff = full ? 0 : (k < n ? k : n);  // sampler.py:133-134
  VS_TR(A, 8);
  __syncthreads();
  double sx = 0.0;  // FULL: the mass of the listed keys
  int ck = 0;       // FULL: listed keys that pass the exp(-40) filter
  const float thr = full && n > 4096 ? xs0 - 40.0f : -__builtin_inff();  // sampler.py:137-139
  // Value bins between the maximum and M's value, largest first: bin numbers never fall as the value falls.
  const float bsc = xmax > xlow ? 255.0f / (xmax - xlow) : 0.0f;
  auto bin_of = [&](float x) -> int { return (int)fminf((xmax - x) * bsc, 255.0f); };
#pragma unroll
  for (int u = 0; u < BATCH_NK; ++u) {
    if (u >= nu) break;
    if (kk[u] != 0) {
      const float x = key_value(kk[u]);
      float e = 0.0f;
      if (full) {
        const float xs = x / tt;
        e = mass_at(xs - xs0);
        sx += (double)e;
        ck += xs >= thr ? 1 : 0;
      }
      if (kk[u] >= M) {
        const int b = bin_of(x);
        atomicAdd(&s.hc[b], 1u);
        if (full) atomicAdd(&s.hf[b], fixed_mass(e, 0x1p18f, 0x1p50f));
      } else {
        kk[u] = 0;
      }
    }
  }
  if (full) {
    sx = wave_sum(sx);
    ck = wave_sum(ck);
    if (ln == 0) {
      s.sum[wv] = sx;
      s.nz[wv] = ck;
    }
  }
  __syncthreads();
  VS_TR(A, 9);
  double S = rsum;
  int total = -1;  // FULL: the size of the kept set, where it is known
  if (full) {
    ck = 0;
#pragma unroll
    for (int i = 0; i < SNW; ++i) {
      S += s.sum[i];
      ck += s.nz[i];
    }
    if (xmin / tt >= thr) total = n;       // nothing is filtered
    else if (xlow / tt < thr) total = ck;  // what passes is listed (an unlisted logit is below a bound <= xlow)
    if (total < 0 && !(P.top_p < 1.0) && !has_mp) {  // no cut: the kept set is all of it, which has to be counted
      leave_open(ROW_FLAT);
      return;
    }
  }
  // The last bin needed (every wave computes it): lane ln holds bins 4 ln .. 4 ln + 3.
  int cut, nsel = 0;
  bool mend = false;  // every key past the cut bin fails min-p
  {
    int c4[4];
    u64 f4[4];
    int lc = 0;
    u64 lf = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      c4[i] = (int)s.hc[4 * ln + i];
      f4[i] = s.hf[4 * ln + i];
      lc += c4[i];
      lf += f4[i];
    }
    const int ic = wave_scan(lc);
    const u64 iff = wave_scan(lf);
    int cc = ic - lc;
    u64 cf = iff - lf;
    // the bin where the count reaches keff (TOPK), or the mass reaches the top-p cut, else the draw (FULL)
    const bool cuts = P.top_p < 1.0 || P.min_p > 0.0;
    const double tgt = P.top_p < 1.0 ? P.top_p * S : (cuts ? 1e300 : P.u * S * (1.0 + 1e-12));
    int hit = 1 << 20, cum[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cc += c4[i];
      cf += f4[i];
      cum[i] = cc;
      if (hit == 1 << 20 && c4[i] > 0 && (full ? (double)cf * 0x1p-50 >= tgt : cc >= keff)) hit = 4 * ln + i;
      if (t < WAVE) s.at[4 * ln + i] = (uint32_t)(cc - c4[i]);
    }
    cut = wave_min(hit);
    if (has_mp && xq > xlow) {  // every key from xq up is listed
      const int b = bin_of(xq);
      mend = b <= cut;
      cut = mend ? b : cut;
    }
    if (cut < (1 << 20))
      nsel = lane_bcast(cut % 4 == 0 ? cum[0] : cut % 4 == 1 ? cum[1] : cut % 4 == 2 ? cum[2] : cum[3], cut / 4);
  }
  if (!full && M == 0) {  // no bound: every listed key
    cut = NBIN - 1;
    nsel = wave_sum(cg);
  }
  if (full && (cut >= (1 << 20) || nsel > BSEL || nsel < 1)) {
    leave_open(ROW_FLAT);
    return;
  }
  VS_TR(A, 10);
  int mine = 0;
#pragma unroll
  for (int u = 0; u < BATCH_NK; ++u) {
    if (u >= nu) break;
    if (kk[u] != 0 && bin_of(key_value(kk[u])) > cut) kk[u] = 0;
    mine += kk[u] != 0 ? 1 : 0;
  }
  // More than 128 keys are put in order bin by bin; rank_sort's comparisons grow with the square of their number (128
  // requests without cuts, V = 32768 f32: this kernel 21 us with it alone, 12 now).
  const bool by_bin = nsel > 2 * WAVE && nsel <= BSEL;
  if (__builtin_expect(nsel > BSEL, 0)) {
    // A TOPK row whose cut bin holds more keys than are ranked (tied values): a bisection on the keys, as in the stream
    // kernel, until at least keff and at most BSEL are left. There are keff from lo up, fewer from hi up.
    u64 lo = M, hi = ((u64)ord32(xmax) + 1) << 32;
    for (int step = 0; nsel > BSEL && hi - lo > 1; ++step) {
      const u64 mid = lo + (hi - lo) / 2;
      int c = 0;
#pragma unroll
      for (int u = 0; u < BATCH_NK; ++u) {
        if (u >= nu) break;
        c += (int)__popcll(__ballot(kk[u] >= mid));
      }
      int* x = s.cnt + (step & 1) * SNW;
      if (ln == 0) x[wv] = c;
      __syncthreads();
      c = 0;
#pragma unroll
      for (int i = 0; i < SNW; ++i) c += x[i];
      if (c < keff) {
        hi = mid;
      } else {
        lo = mid;
        nsel = c;
      }
    }
    mine = 0;
#pragma unroll
    for (int u = 0; u < BATCH_NK; ++u) {
      if (u >= nu) break;
      if (kk[u] < lo) kk[u] = 0;
      mine += kk[u] != 0 ? 1 : 0;
    }
  }
  if (by_bin) {  // sampler.py:140
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BATCH_NK; ++u) {
      if (u >= nu) break;
      if (kk[u] != 0) s.sel[atomicAdd(&s.at[bin_of(key_value(kk[u]))], 1u)] = kk[u];
    }
    __syncthreads();
    VS_TR(A, 11);
    if (t < nsel) {
      const u64 key = s.sel[t];
      const int bin = bin_of(key_value(key)), end = (int)s.at[bin], begin = end - (int)s.hc[bin];
      int r = begin;
      for (int j = begin; j < end; ++j) r += s.sel[j] > key ? 1 : 0;
      if (full || r < keff) s.tk[r] = key;
    }
    __syncthreads();
  } else {
    int at = wave_alloc(mine, &s.misc[4]);
    if (mine) {
#pragma unroll
      for (int u = 0; u < BATCH_NK; ++u) {
        if (u >= nu) break;
        if (kk[u] != 0) {
          if (at < BSEL) s.sel[at] = kk[u];
          ++at;
        }
      }
    }
    __syncthreads();
    VS_TR(A, 11);
    rank_sort(s.sel, nsel, s.tk, full ? nsel : keff);  // sampler.py:140
  }
  VS_TR(A, 12);
  if (A.list_k > 0) {  // top-list mode (vs_topk_batch)
    for (int i = t; i < A.list_k; i += SNT) {
      A.list_ids[(size_t)grow * A.list_k + i] = i < keff ? (int32_t)key_index(s.tk[i]) : -1;
      A.list_vals[(size_t)grow * A.list_k + i] = i < keff ? key_value(s.tk[i]) : -__builtin_inff();
    }
  } else if (!full) {
    Smem w = {};
    w.misc = s.misc;
    w.redf = s.sum;
    const Final f = wave_sample(w, s.tk, keff, P);
    write_out(A, row, f, R.st, R.rng_next);
    if (t == 0) *flag = ROW_DONE;
  } else {
    if (t < WAVE) {
      if (nsel <= 2 * WAVE) wave_sample_tail<2>(s.tk, nsel, S, total, mend, P, s.misc, s.sum);
      else wave_sample_tail<BSEL / WAVE>(s.tk, nsel, S, total, mend, P, s.misc, s.sum);
      if (t == 0 && s.misc[0]) {
        Final f;
        f.token = s.misc[1];
        f.keep = s.misc[2];
        f.lp = (float)s.sum[0];
        // the route bits the general kernel reports for such a row
        const bool small = total >= 0 && total <= GSMALL;
        f.flags = (uint32_t)s.misc[3] | (small || !(P.min_p > 0.0) ? (uint32_t)VS_OUT_GATHER : 0u) |
                  (small ? 0u : (uint32_t)VS_OUT_COOP);
        *flag = ROW_DONE;
        write_out(A, row, f, R.st, R.rng_next);
      }
    }
    __syncthreads();
    if (!s.misc[0]) leave_open(ROW_FLAT);
  }
  VS_TR(A, 13);
  VS_TR_FLUSH(A);
}

// ---------------------------------------------------------------------------------------------------------------
// The open rows, a cluster of workgroups each. Every pass streams the row again (the logits, then in a nearby cache) with
// its edits; the workgroups of a cluster add their histograms up in the row's list area and meet at a barrier after each
// pass. All of them see the same sums and take the same decisions; workgroup 0 writes the result. A wait that reaches its
// bound ends the workgroup; workgroup 0 then reports VS_OUT_TIMEOUT (it passes a barrier only when every workgroup has
// contributed to everything before it). Where a workgroup's share of the row fits LDS the second pass of the flat method
// reads it there (24576 logits; 20 near-flat rows of V = 163840: 39 us per call, 56 in two launches of vs_sample_kernel).
// ---------------------------------------------------------------------------------------------------------------
constexpr int RE = 16;                          // logits per lane and tile
constexpr int RTILE = RE * SNT;                 // positions per tile at most
constexpr uint64_t WAIT_TICKS_OPEN = 100000;    // 1 ms
constexpr int RKEEP = 3;                        // tiles whose edited logits stay in LDS between the passes
constexpr size_t RESOLVE_LDS = (size_t)RKEEP * RTILE * 4;  // the tiles: their edit words, then their logits

struct ResolveLds {
  u64 hist[RNB];      // flat method: masses by value bin, then their inclusive sums
  u64 keys[RCAP];     // gathered keys
  uint32_t hc[NBIN];  // radix: counts, masses, largest keys by digit
  u64 hm[NBIN];
  u64 hk[NBIN];
  double redd[NRED];
  double at[2];       // a position's mass and the sum through it
  u64 red64[NRED];
  int red[NRED];
  int misc[16];
  int list[BATCH_ROWS];
};

// The digit of a 256-bin histogram, walked from digit 255 down, where the weight (count or mass) reaches `target`: the
// first non-empty one whose inclusive sum does, else the last non-empty one. Every wave computes it.
struct Digit {
  int d;
  uint32_t cnt_before, cnt;
  u64 mass_before, mass;  // in fixed point
  u64 mk;
};
__device__ __forceinline__ Digit find_digit(const uint32_t* hc, const u64* hm, const u64* hk, bool by_count, u64 target) {
  const int L = lane_id();
  uint32_t c[4], lc = 0;
  u64 f[4], lf = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int d = NBIN - 1 - (4 * L + i);
    c[i] = hc[d];
    f[i] = hm[d];
    lc += c[i];
    lf += f[i];
  }
  uint32_t cc = wave_scan(lc) - lc;
  u64 cf = wave_scan(lf) - lf;
  int hit = -1, last = -1;
  uint32_t cb = 0, lcb = 0;
  u64 fb = 0, lfb = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (c[i] > 0) {
      last = i;
      lcb = cc;
      lfb = cf;
      if (hit < 0 && (by_count ? (u64)(cc + c[i]) : cf + f[i]) >= target) {
        hit = i;
        cb = cc;
        fb = cf;
      }
    }
    cc += c[i];
    cf += f[i];
  }
  const unsigned long long hb = __ballot(hit >= 0), lb = __ballot(last >= 0);
  const int ls = hb ? __ffsll((long long)hb) - 1 : (lb ? 63 - __clzll((long long)lb) : 0);
  const int is = hb ? lane_bcast(hit, ls) : (lb ? lane_bcast(last, ls) : 0);
  Digit r;
  r.d = NBIN - 1 - (4 * ls + is);
  r.cnt_before = lane_bcast(hb ? cb : lcb, ls);
  r.mass_before = lane_bcast(hb ? fb : lfb, ls);
  r.cnt = hc[r.d];
  r.mass = hm[r.d];
  r.mk = hk[r.d];
  return r;
}

template <int DT>
__global__ __launch_bounds__(SNT, 2) void vs_resolve_kernel(SampleArgs A) {
  constexpr int VEC = DTraits<DT>::VEC, NVL = RE / VEC;
  extern __shared__ __align__(16) char smem_raw[];
  __shared__ ResolveLds s;
  const int t = threadIdx.x;
  VS_TR_DECL(A);
  VS_TR(A, 0);
  // the open rows of the launch
  static_assert(BATCH_ROWS == 2 * WAVE, "one wave lists the open rows, two per lane");
  if (t < WAVE) {
    bool op[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = t + i * WAVE;
      op[i] = r < A.B && *open_flag(A.ws, r < A.B ? r : 0) != ROW_DONE;
    }
    int n = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const unsigned long long m = __ballot(op[i]);
      if (op[i]) s.list[n + __popcll(m & ((1ull << t) - 1ull))] = t + i * WAVE;
      n += __popcll(m);
    }
    if (t == 0) s.misc[0] = n;
  }
  __syncthreads();
  const int nitems = s.misc[0];
  if (nitems == 0) return;
  // workgroups per row: as many as leave a cluster for every row; no more rows than workgroups (batch_plan)
  const int C = max(1, min(CMAX, (int)gridDim.x / nitems));
  const int nb = gridDim.x, b = blockIdx.x;
  const int l = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;  // a cluster's workgroups on one XCD where they fit
  const int cl = l / C, w = l % C;
  if (cl >= nitems) return;
  const int row = s.list[cl], grow = A.row0 + row;
  const int how = *open_flag(A.ws, row);
  OpenRow* o = (OpenRow*)part_area(A.ws, row);
  char* area = list_area(A.ws, row);
  u64* gkeys = (u64*)(area + HIST_BYTES);
  RowIn R;
  row_place<DT>(A, grow, R);
  row_params(A, grow, R);
  const vs_row_params& P = R.P;
  const int n = o->n;
  const float xmax = o->xmax, xmin = o->xmin, tt = P.temperature;
  const float xs0 = xmax / tt;
  // this workgroup's tiles: m of them, from tile w m on
  const int span = A.V + R.mis;
  const int m = (span + C * RTILE - 1) / (C * RTILE);
  const int tile = ((span + C * m - 1) / (C * m) + VEC - 1) / VEC * VEC;
  const bool resident = m <= RKEEP;
  auto tiles = [&](auto fn) {
    uint4 raw[NVL];
    tile_load<DT, NVL>(R, w * m * tile, max(w * m * tile, min(span, w * m * tile + tile)), raw);
    for (int i = 0; i < m; ++i) {
      const int p0 = (w * m + i) * tile, p1 = max(p0, min(span, p0 + tile));
      float v[RE];
      float4* slot = (float4*)smem_raw + (resident ? i : 0) * (RTILE / 4);
      EditAhead H;
      edit_ahead(A, R, H);
      tile_edit<DT, NVL>(A, R, H, p0, p1, raw, v, (uint32_t*)slot, s.red);
      if (resident) {
#pragma unroll
        for (int j = 0; j < RE / 4; ++j) slot[j * SNT + t] = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
      }
      const int p2 = p0 + tile;
      if (i + 1 < m) tile_load<DT, NVL>(R, p2, max(p2, min(span, p2 + tile)), raw);
      const int l0 = p0 - R.mis;
#pragma unroll
      for (int e = 0; e < RE; ++e) fn(v[e], l0 + ((e / VEC) * SNT + t) * VEC + e % VEC);
    }
  };
  // a pass that may be a later one: from LDS where every tile is held there (each lane reads what it wrote)
  bool held = false;
  auto tiles_again = [&](auto fn) {
    if (!(resident && held)) {
      tiles(fn);
      held = true;
      return;
    }
    for (int i = 0; i < m; ++i) {
      const float4* slot = (const float4*)smem_raw + i * (RTILE / 4);
      const int l0 = (w * m + i) * tile - R.mis;
#pragma unroll
      for (int j = 0; j < RE / 4; ++j) {
        const float4 q = slot[j * SNT + t];
        const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) fn(v[e], l0 + (((4 * j + e) / VEC) * SNT + t) * VEC + (4 * j + e) % VEC);
      }
    }
  };
  uint32_t nbar = 0;
  bool ok = true;
  auto barrier = [&]() -> bool {  // every store and atomic of the cluster before it is seen after it
    ++nbar;
    ok = row_barrier(&o->bar, nbar * (uint32_t)C, A.spin_limit, WAIT_TICKS_OPEN, &s.misc[1]);
    return ok;
  };
  Final fin;
  fin.token = -1;
  fin.lp = 0.0f;
  fin.flags = VS_OUT_TIMEOUT;
  fin.keep = 0;
  auto finish = [&]() {
    if (w == 0) write_out(A, row, fin, R.st, R.rng_next);
  };
  const bool filt = n > 4096;
  const float thr = filt ? xs0 - 40.0f : -__builtin_inff();  // sampler.py:137-139
  const bool has_tp = P.top_p < 1.0, has_mp = P.min_p > 0.0;
  // Masses are summed in fixed point: the sums do not depend on the order of the additions, so a call's cuts, draws and
  // logprobs are the same every time. A mass is rounded by 2^-63 of the row's at most, no more than float64 sums of as
  // many terms lose. (64 near-flat rows of V = 163840 f32 take 65.2 us a call, 63.6 with float64 sums.)
  const float fsc = __builtin_amdgcn_ldexpf(1.0f, o->shift), fsh = __builtin_amdgcn_ldexpf(1.0f, o->shift - 32);
  const double inv_scale = 1.0 / (double)fsc;
  auto fix_of = [&](float e) -> u64 { return fixed_mass(e, fsh, fsc); };

  u64 Tk = 0, Tfix = 0;  // the smallest key kept by the top-k cut and the mass kept by it (0: not known yet)

  VS_TR(A, 1);
  if (how == ROW_FLAT) {
    // ---- one histogram of masses over value bins, one gather of the bins the cuts and the draw can lie in ----
    // Bins run from the maximum to the smallest value that can be kept; bin numbers never fall as the value falls.
    const float xl = filt ? fmaxf(xmin, xmax - 40.0f * tt * 1.00001f - 1e-30f) : xmin;
    const float bsc = xmax > xl && xmax - xl < 3.0e38f ? ((float)RNB - 0.5f) / (xmax - xl) : 0.0f;
    auto bin_of = [&](float x) -> int { return (int)fminf((xmax - x) * bsc, (float)(RNB - 1)); };
    for (int i = t; i < RNB; i += SNT) s.hist[i] = 0;
    if (t == 0) s.misc[2] = 0;
    __syncthreads();
    const bool unit = tt == 1.0f;  // x / 1 == x: no division
    auto add_mass = [&](float x, float xs) {
      if (is_finite(x) & (xs >= thr)) atomicAdd(&s.hist[bin_of(x)], fix_of(mass_at(xs - xs0)));
    };
    if (unit) tiles([&](float x, int) { add_mass(x, x); });
    else tiles([&](float x, int) { add_mass(x, x / tt); });
    held = true;
    __syncthreads();
    VS_TR(A, 2);
    u64* gh = (u64*)area;
    if (C > 1) {
#pragma unroll
      for (int i = 0; i < RNB / SNT; ++i) {
        const u64 f = s.hist[t + i * SNT];
        if (f != 0) atomicAdd(&gh[t + i * SNT], f);
      }
      if (!barrier()) {
        finish();
        return;
      }
    }
    VS_TR(A, 3);
    // inclusive sums, in place: thread t owns bins 4 t .. 4 t + 3
    static_assert(RNB == 4 * SNT, "four bins per thread");
    u64 c4[4], cprev, Sfix;
    {
      u64 f[4], lf = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[i] = C > 1 ? ld_relaxed64(&gh[4 * t + i]) : s.hist[4 * t + i];
        lf += f[i];
      }
      u64 c = block_scan<SNT>(lf, s.red64, &Sfix) - lf;
      cprev = c;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        c += f[i];
        c4[i] = c;
        s.hist[4 * t + i] = c;
      }
    }
    if (t == 0) s.misc[5] = s.misc[6] = s.misc[7] = RNB - 1;
    __syncthreads();
    const double S = (double)Sfix * inv_scale;
    // the first bin whose inclusive sum reaches target (fixed point), into misc[at] by its owner
    auto find = [&](double target, int at) {
      u64 tg = ceil_u64(target), prev = cprev;
      tg = tg < 1 ? 1 : (tg > Sfix ? Sfix : tg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (c4[i] >= tg && prev < tg) s.misc[at] = 4 * t + i;
        prev = c4[i];
      }
    };
    auto before = [&](int bin) -> u64 { return bin > 0 ? s.hist[bin - 1] : 0; };
    const double tgt_p = P.top_p * (double)Sfix;
    u64 zlo = Sfix, zhi = Sfix;
    int T = -1;
    if (has_tp) {
      find(tgt_p, 5);
      __syncthreads();
      T = s.misc[5];
      zlo = before(T);
      zhi = s.hist[T];
    }
    const double pthr = (1.0 / S) * P.min_p;  // sampler.py:149-152
    if (has_mp) {
      // the kept prefix ends between the values log(min_p) -+ 1e-4 below the maximum (in units of the temperature)
      const float lg = logf((float)P.min_p), sl = 1e-4f + 1e-5f * fabsf(xs0);
      const float xa = xmax + tt * fminf(lg + sl, 0.0f), xb = xmax + tt * fminf(lg - sl, 0.0f);
      zlo = min(zlo, before(bin_of(fmaxf(xa, xl))));
      zhi = min(zhi, s.hist[bin_of(fmaxf(xb, xl))]);
      zlo = min(zlo, zhi);
    }
    find(P.u * (double)zlo * (1.0 - 1e-9), 6);
    find(P.u * (double)zhi * (1.0 + 1e-9), 7);
    __syncthreads();
    const int D0 = s.misc[6], D1 = s.misc[7];
    VS_TR(A, 4);
    int cT = 0, cM = 0, kc = 0;
    u64 fM = 0;
    auto take = [&](float x, float xs, int id) {
      if (is_finite(x) & (xs >= thr)) {
        const int bin = bin_of(x);
        ++kc;
        cT += bin < T ? 1 : 0;
        if (has_mp) {
          const float e = mass_at(xs - xs0);
          if (!((double)e / S < pthr)) {
            ++cM;
            fM += fix_of(e);
          }
        }
        if ((bin == T) | ((bin >= D0) & (bin <= D1))) {
          const int p = atomicAdd(&s.misc[2], 1);
          if (p < RCAP) s.keys[p] = key64(x, (uint32_t)id);
        }
      }
    };
    if (unit) tiles_again([&](float x, int id) { take(x, x, id); });
    else tiles_again([&](float x, int id) { take(x, x / tt, id); });
    VS_TR(A, 5);
    cT = block_sum<SNT>(cT, s.red);
    kc = block_sum<SNT>(kc, s.red);
    cM = has_mp ? block_sum<SNT>(cM, s.red) : 0;
    fM = has_mp ? block_sum<SNT>(fM, s.red64) : 0;
    const int nloc = s.misc[2];
    if (t == 0) {
      if (cT) atomicAdd(&o->cnt[0], (uint32_t)cT);
      if (kc) atomicAdd(&o->cnt[2], (uint32_t)kc);
      if (has_mp) {
        atomicAdd(&o->cnt[1], (uint32_t)cM);
        atomicAdd(&o->fix[0], fM);
      }
      s.misc[3] = (int)atomicAdd(&o->gcnt, (uint32_t)nloc);
    }
    __syncthreads();
    const int g0 = s.misc[3];
    for (int i = t; i < nloc && i < RCAP; i += SNT)
      if (g0 + i < RCAP) st_dev(&gkeys[g0 + i], s.keys[i]);
    if (!barrier()) {
      finish();
      return;
    }
    VS_TR(A, 6);
    const int ng = (int)ld_relaxed(&o->gcnt);
    if (ng <= RCAP) {
      if (w != 0) {
        VS_TR_FLUSH(A);
        return;
      }
      const int cnt_t = (int)ld_relaxed(&o->cnt[0]), cnt_m = (int)ld_relaxed(&o->cnt[1]);
      const int total = (int)ld_relaxed(&o->cnt[2]);
      const u64 fix_m = ld_relaxed64(&o->fix[0]);
      u64* mem = (u64*)smem_raw;  // [RCAP] members
      static_assert(RCAP * 8 <= RESOLVE_LDS, "the members fit the tile area");
      u64 kr[RCAP / SNT];
#pragma unroll
      for (int i = 0; i < RCAP / SNT; ++i) kr[i] = t + i * SNT < ng ? ld_dev(&gkeys[t + i * SNT]) : (u64)0;
      struct Pick {
        u64 key;
        int rank;         // members above it
        u64 below, mass;  // the mass above it, its own
      };
      auto mass_of = [&](u64 key) -> u64 { return fix_of(mass_at(key_value(key) / tt - xs0)); };
      auto clear = [&]() {
        __syncthreads();
        if (t < NBIN) {
          s.hc[t] = 0;
          s.hm[t] = 0;
          s.hk[t] = 0;
        }
        __syncthreads();
      };
      // The first member of `bin`, in descending order, at which the bin's mass reaches tgt (the last if none): by
      // 256 parts of the bin, then among the few members of the part.
      auto pick = [&](int bin, u64 tgt) -> Pick {
        Pick r = {0, 0, 0, 0};
        auto part_of = [&](u64 key) -> int {  // 255 .. 0 as the value falls, -1: another bin
          const float p = fminf((xmax - key_value(key)) * bsc, (float)(RNB - 1)), f = p - (float)(int)p;
          return key != 0 && (int)p == bin ? NBIN - 1 - (int)(f * 255.99f) : -1;
        };
        if (t == 0) s.misc[4] = 0;
        clear();
#pragma unroll
        for (int i = 0; i < RCAP / SNT; ++i) {
          const int d = part_of(kr[i]);
          if (d >= 0) {
            atomicAdd(&s.hc[d], 1u);
            atomicAdd(&s.hm[d], mass_of(kr[i]));
          }
        }
        __syncthreads();
        const Digit q0 = find_digit(s.hc, s.hm, s.hk, false, tgt);
        if (q0.cnt == 0) return r;
        r.rank = (int)q0.cnt_before;
        r.below = q0.mass_before;
#pragma unroll
        for (int i = 0; i < RCAP / SNT; ++i)
          if (part_of(kr[i]) == q0.d) mem[atomicAdd(&s.misc[4], 1)] = kr[i];
        __syncthreads();
        const int nm = (int)q0.cnt;
        if (nm <= WAVE) {  // every wave: lane L holds member L and sums the members above it
          const int L = lane_id();
          const u64 ki = L < nm ? mem[L] : (u64)0;
          const u64 me = ki ? mass_of(ki) : 0;
          int rk = 0;
          u64 ab = 0;
          for (int j = 0; j < nm; ++j) {
            const bool gt = lane_bcast(ki, j) > ki;
            const u64 mj = lane_bcast(me, j);
            rk += gt ? 1 : 0;
            ab += gt ? mj : (u64)0;
          }
          const int hit = wave_min(ki && r.below + ab + me >= tgt ? rk : nm - 1);
          const int ln = __ffsll((long long)__ballot(ki != 0 && rk == hit)) - 1;
          r.key = lane_bcast(ki, ln);
          r.rank += hit;
          r.below += lane_bcast(ab, ln);
          r.mass = lane_bcast(me, ln);
          return r;
        }
        u64 prefix = 0;
        for (int shift = 56;; shift -= 8) {  // many members (tied values): a radix select by mass
          clear();
          for (int i = t; i < nm; i += SNT) {
            const u64 key = mem[i];
            if (prefix_match(key, shift, prefix)) {
              const int d = (int)((key >> shift) & 0xFF);
              atomicAdd(&s.hc[d], 1u);
              atomicAdd(&s.hm[d], mass_of(key));
              atomicMax(&s.hk[d], key);
            }
          }
          __syncthreads();
          const Digit q = find_digit(s.hc, s.hm, s.hk, false, tgt > r.below ? tgt - r.below : 0);
          r.rank += (int)q.cnt_before;
          r.below += q.mass_before;
          prefix = (prefix << 8) | (u64)q.d;
          if (q.cnt <= 1 || shift == 0) {
            r.key = q.mk;
            r.mass = q.mass;
            return r;
          }
        }
      };
      uint32_t flags = VS_OUT_COOP | (has_mp ? 0u : (uint32_t)VS_OUT_GATHER);
      int keep = total;
      u64 zfix = Sfix;
      bool good = true;
#pragma nounroll
      for (int draw = has_tp ? 0 : 1; draw < 2; ++draw) {  // the top-p cut, then the draw: one instance of the pick
        double tgt = tgt_p;
        int bin = T;
        if (draw) {
          if (has_mp) {  // sampler.py:149-152
            const int km = cnt_m > 1 ? cnt_m : 1;
            if (km < keep) {
              keep = km;
              zfix = cnt_m >= 1 ? fix_m : (u64)fsc;
            }
          }
          tgt = P.u * (double)zfix;  // :153-156
          bin = D0;
          while (bin < D1 && s.hist[bin] < ceil_u64(tgt)) ++bin;
        }
        const u64 bb = before(bin), tg = ceil_u64(tgt);
        const Pick pk = pick(bin, tg > bb ? tg - bb : 0);
        good = good && pk.key != 0;
        const double bef = (double)(bb + pk.below), tol = 1e-6 * (double)(draw ? zfix : Sfix);
        if (fabs(bef - tgt) < tol || fabs(bef + (double)pk.mass - tgt) < tol)
          flags |= draw ? VS_OUT_DRAW_BOUNDARY : VS_OUT_TOPP_BOUNDARY;
        if (!draw) {  // :145-148
          keep = cnt_t + pk.rank + 1;
          zfix = bb + pk.below + pk.mass;
        } else if (good) {
          fin.token = (int32_t)key_index(pk.key);
          fin.lp = (float)((double)(key_value(pk.key) / tt - xs0) - log_ge1((double)zfix * inv_scale));
          fin.keep = keep;
          fin.flags = flags;
        }
        VS_TR(A, 7);
      }
      finish();
      VS_TR(A, 8);
      VS_TR_FLUSH(A);
      return;
    }
    // too many keys in those bins (long runs of tied values): the general method
  } else if (how == ROW_TOPK) {
    // ---- a top-k cut above the lists' reach: one histogram of counts over value bins, then one gather. Where the bins
    // down to the one the cut lies in hold few keys, they are gathered and workgroup 0 orders them by bin and finishes on
    // the k largest. Otherwise that one bin is gathered and the mass above it summed, and the general method goes on from
    // the cut's key. The radix selects of the general method took nine and more passes for all of it (36 rows of
    // V = 163840 f32, top_k 1000: 148 us a call against 109 in launches of vs_sample_kernel, now 41; top_k 5000: 120, 96 and
    // 82). ----
    const int k = P.top_k;
    const float bsc = xmax > xmin && xmax - xmin < 3.0e38f ? ((float)RNB - 0.5f) / (xmax - xmin) : 0.0f;
    auto bin_of = [&](float x) -> int { return (int)fminf((xmax - x) * bsc, (float)(RNB - 1)); };
    uint32_t* hc = (uint32_t*)s.hist;  // [RNB] counts, then their inclusive sums
    uint32_t* cur = hc + RNB;          // [RNB] the next place of each bin
    for (int i = t; i < RNB; i += SNT) hc[i] = 0;
    if (t == 0) {
      s.misc[2] = 0;
      s.misc[5] = -1;
    }
    __syncthreads();
    tiles_again([&](float x, int) {
      if (is_finite(x) & (x >= xmin)) atomicAdd(&hc[bin_of(x)], 1u);
    });
    __syncthreads();
    uint32_t* gh = (uint32_t*)area;
    if (C > 1) {
#pragma unroll
      for (int i = 0; i < RNB / SNT; ++i) {
        const uint32_t c = hc[t + i * SNT];
        if (c) atomicAdd(&gh[t + i * SNT], c);
      }
      if (!barrier()) {
        finish();
        return;
      }
    }
    {  // inclusive sums, in place: thread t owns bins 4 t .. 4 t + 3
      int c[4], lc = 0, tot;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        c[i] = (int)(C > 1 ? ld_relaxed(&gh[4 * t + i]) : hc[4 * t + i]);
        lc += c[i];
      }
      int cc = block_scan<SNT>(lc, s.red, &tot) - lc;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int before = cc;
        cc += c[i];
        hc[4 * t + i] = (uint32_t)cc;
        cur[4 * t + i] = (uint32_t)before;
        if (cc >= k && before < k) {
          s.misc[5] = 4 * t + i;
          s.misc[6] = cc;
        }
      }
    }
    __syncthreads();
    const int kb = s.misc[5], above = kb > 0 ? (int)hc[kb - 1] : 0;
    const bool all = kb >= 0 && s.misc[6] <= RCAP;
    const int ng = all ? s.misc[6] : kb >= 0 ? s.misc[6] - above : RCAP + 1;
    if (ng <= RCAP) {
      const int b0 = all ? 0 : kb;
      u64 fa = 0;
      tiles_again([&](float x, int id) {
        const int bin = is_finite(x) & (x >= xmin) ? bin_of(x) : RNB;
        if (bin <= kb) {
          if (bin >= b0) {
            const int p = atomicAdd(&s.misc[2], 1);
            if (p < RCAP) s.keys[p] = key64(x, (uint32_t)id);
          } else {
            fa += fix_of(mass_at(x / tt - xs0));
          }
        }
      });
      if (!all) {
        fa = block_sum<SNT>(fa, s.red64);
        if (t == 0) atomicAdd(&o->fix[1], fa);
      }
      __syncthreads();
      const int nloc = s.misc[2];
      if (t == 0) s.misc[3] = (int)atomicAdd(&o->gcnt, (uint32_t)nloc);
      __syncthreads();
      const int g0 = s.misc[3];
      for (int i = t; i < nloc && i < RCAP; i += SNT)
        if (g0 + i < RCAP) st_dev(&gkeys[g0 + i], s.keys[i]);
      if (!barrier()) {
        finish();
        return;
      }
      if (all && w != 0) return;
      u64* mem = (u64*)smem_raw;  // [RCAP] the keys, bin by bin
      u64* srt = mem + RCAP;      // [RCAP] the k largest, in order
      static_assert(2 * RCAP * 8 <= RESOLVE_LDS && RCAP <= 4 * SNT, "both fit the tile area, four keys per thread");
      u64 kr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) kr[i] = t + i * SNT < ng ? ld_dev(&gkeys[t + i * SNT]) : (u64)0;
      if (!all) {  // every workgroup: the cut's key, and the mass of the bin's keys from it up
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kr[i]) s.keys[t + i * SNT] = kr[i];
        __syncthreads();
        u64 f = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (kr[i]) {
            int r = above;
            for (int j = 0; j < ng; ++j) r += s.keys[j] > kr[i] ? 1 : 0;
            if (r < k) f += fix_of(mass_at(key_value(kr[i]) / tt - xs0));
            if (r == k - 1) s.hk[0] = kr[i];
          }
        }
        Tfix = block_sum<SNT>(f, s.red64) + ld_relaxed64(&o->fix[1]);
        Tk = s.hk[0];
      }
      if (all) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (kr[i]) mem[atomicAdd(&cur[bin_of(key_value(kr[i]))], 1u)] = kr[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (kr[i]) {
            const int bin = bin_of(key_value(kr[i])), end = (int)hc[bin];
            int r = bin > 0 ? (int)hc[bin - 1] : 0;
            for (int j = r; j < end; ++j) r += mem[j] > kr[i] ? 1 : 0;
            if (r < k) srt[r] = kr[i];
          }
        }
        __syncthreads();
        // sampler.py:141-156 on srt[0, k): thread t owns positions E t .. E t + E - 1
        const int E = (k + SNT - 1) / SNT, i0 = E * t;
        double pr[4], ls = 0.0, S;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          pr[q] = q < E && i0 + q < k ? (double)mass_at(key_value(srt[i0 + q]) / tt - xs0) : 0.0;
          ls += pr[q];
        }
        const double base0 = block_scan<SNT>(ls, s.redd, &S) - ls;
        const double base = base0 / S;
#pragma unroll
        for (int q = 0; q < 4; ++q) pr[q] = pr[q] / S;
        constexpr int NOWHERE = 1 << 30;
        int keep = k;
        uint32_t flags = VS_OUT_COOP;
        // the first position below `end` whose cumulative mass reaches tgt (NOWHERE: none), its mass and the sum through it
        // in s.at[0] and s.at[1]
        auto reach = [&](double tgt, int end) -> int {
          double c = base, hp = 0.0, hc2 = 0.0;
          int hit = NOWHERE;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (q < E && i0 + q < end) {
              c += pr[q];
              if (hit == NOWHERE && c >= tgt) {
                hit = i0 + q;
                hp = pr[q];
                hc2 = c;
              }
            }
          }
          const int at = block_min<SNT>(hit, s.red);
          if (at != NOWHERE && at == hit) {
            s.at[0] = hp;
            s.at[1] = hc2;
          }
          __syncthreads();
          return at;
        };
        // the position `at` itself: its mass and the sum through it, likewise
        auto look = [&](int at) {
          if (at / E == t) {
            double c = base, hp = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (q < E && i0 + q <= at) {
                c += pr[q];
                hp = pr[q];
              }
            }
            s.at[0] = hp;
            s.at[1] = c;
          }
          __syncthreads();
        };
        if (has_tp) {  // :145-148
          const int at = reach(P.top_p, k);
          if (at != NOWHERE) {
            keep = at + 1;
            if (fabs(s.at[1] - P.top_p) < 1e-6 || fabs(s.at[1] - s.at[0] - P.top_p) < 1e-6)
              flags |= VS_OUT_TOPP_BOUNDARY;
          }
        }
        if (has_mp) {  // :149-152 (the largest key's mass is 1 before the division by S)
          const double pthr = (1.0 / S) * P.min_p;
          int hit = NOWHERE;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (hit == NOWHERE && q < E && i0 + q < k && pr[q] < pthr) hit = i0 + q;
          const int at = block_min<SNT>(hit, s.red);
          const int cnt = at == NOWHERE ? k : max(at, 1);
          keep = cnt < keep ? cnt : keep;
        }
        __syncthreads();
        look(keep - 1);
        const double z = s.at[1], uz = P.u * z;  // :153-154
        __syncthreads();
        int j = reach(uz, keep);
        if (j == NOWHERE) look(j = keep - 1);  // :155-156
        const double hp = s.at[0], hs = s.at[1], tol = 1e-6 * z;
        if (fabs(hs - uz) < tol || (j >= 1 && fabs(hs - hp - uz) < tol)) flags |= VS_OUT_DRAW_BOUNDARY;
        fin.token = (int32_t)key_index(srt[j]);
        fin.lp = (float)((double)(key_value(srt[j]) / tt - xs0) - log_ge1(z * S));
        fin.keep = keep;
        fin.flags = flags;
        finish();
        return;
      }
    }
    // the general method, once everyone has read the sums
    if (!barrier()) {
      finish();
      return;
    }
  }
  if (how != ROW_ANY) {  // on cleared histograms
    if (w == 0)
      for (int i = t; i < (int)(HIST_BYTES / 8); i += SNT) st_dev((u64*)area + i, (u64)0);
    if (t == 0 && w == 0) {  // (the flat method's sums)
      st_dev(&o->cnt[2], 0u);
      st_dev(&o->fix[0], (u64)0);
    }
    if (!barrier()) {
      finish();
      return;
    }
  }

  // ---- the general method: exact selections by radix passes on the 64-bit keys ----
  if (n == 0) {  // sampler.py:131-132
    u64 am = 0;
    tiles_again([&](float x, int id) {
      if (id >= 0 && id < R.vlim) {
        const u64 k = amkey64(x, (uint32_t)id);
        am = k > am ? k : am;
      }
    });
    am = block_max<SNT>(am, s.red64);
    if (t == 0) atomicMax(&o->amkey, am);
    if (barrier()) {
      fin.token = (int32_t)key_index(ld_relaxed64(&o->amkey));
      fin.flags = VS_OUT_NOFINITE;
    }
    finish();
    return;
  }
  int k = P.top_k > 0 ? (P.top_k < n ? P.top_k : n) : n;  // sampler.py:133-134
  if (k < 1) k = 1;
  const bool cutk = k < n;
  const float kthr = cutk ? -__builtin_inff() : thr;
  auto kept = [&](float x, int id, u64& key, float& xs) -> bool {
    key = key64(x, (uint32_t)id);
    xs = x / tt;
    return is_finite(x) & (key >= Tk) & !(xs < kthr);
  };
  RadixSlot* ring = (RadixSlot*)area;
  int round = 0;
  // The kept key at which the weight (count or mass, in descending order) reaches target, with the sums above it.
  struct Sel {
    u64 key;
    uint32_t cnt_before;
    u64 mass_before, mass;
  };
  auto select = [&](bool by_count, u64 target) -> Sel {
    Sel r = {0, 0, 0, 0};
    u64 prefix = 0;
    for (int shift = 56;; shift -= 8) {
      if (t < NBIN) {
        s.hc[t] = 0;
        s.hm[t] = 0;
        s.hk[t] = 0;
      }
      __syncthreads();
      tiles_again([&](float x, int id) {
        u64 key;
        float xs;
        if (kept(x, id, key, xs) && prefix_match(key, shift, prefix)) {
          const int d = (int)((key >> shift) & 0xFF);
          atomicAdd(&s.hc[d], 1u);
          if (!by_count) atomicAdd(&s.hm[d], fix_of(mass_at(xs - xs0)));
          atomicMax(&s.hk[d], key);
        }
      });
      __syncthreads();
      RadixSlot* h = ring + round % RRING;
      if (t < NBIN && s.hc[t]) {
        atomicAdd(&h->cnt[t], s.hc[t]);
        if (!by_count) atomicAdd(&h->fix[t], s.hm[t]);
        atomicMax(&h->mk[t], s.hk[t]);
      }
      // the next round's slot was last read after the barrier before the last one, which every workgroup has left
      if (w == 0 && round >= RRING - 1 && t < NBIN) {
        RadixSlot* z = ring + (round + 1) % RRING;
        st_dev(&z->cnt[t], 0u);
        st_dev(&z->fix[t], (u64)0);
        st_dev(&z->mk[t], (u64)0);
      }
      ++round;
      if (!barrier()) return r;
      if (t < NBIN) {
        s.hc[t] = ld_relaxed(&h->cnt[t]);
        s.hm[t] = ld_relaxed64(&h->fix[t]);
        s.hk[t] = ld_relaxed64(&h->mk[t]);
      }
      __syncthreads();
      const u64 above = by_count ? (u64)r.cnt_before : r.mass_before;
      const Digit q = find_digit(s.hc, s.hm, s.hk, by_count, target > above ? target - above : 0);
      r.cnt_before += q.cnt_before;
      r.mass_before += q.mass_before;
      prefix = (prefix << 8) | (u64)q.d;
      __syncthreads();
      if (by_count && (u64)(r.cnt_before + q.cnt) == target) {  // the digit is kept whole: its lowest key bounds the cut
        r.key = prefix << shift;
        return r;
      }
      if (q.cnt <= 1 || shift == 0) {
        r.key = q.mk;
        r.mass = q.mass;
        return r;
      }
    }
  };
  if (cutk && Tk == 0) {
    const Sel sk = select(true, (u64)k);
    if (!ok) {
      finish();
      return;
    }
    Tk = sk.key;
  }
  // sums over the kept set: its size and mass, or (with the mass known) those of what min-p keeps of it
  auto sums = [&](double S, double pthr, int at) -> bool {
    int c = 0;
    u64 f = 0;
    tiles_again([&](float x, int id) {
      u64 key;
      float xs;
      if (kept(x, id, key, xs)) {
        const float e = mass_at(xs - xs0);
        if (S == 0.0 || !((double)e / S < pthr)) {
          ++c;
          f += fix_of(e);
        }
      }
    });
    c = block_sum<SNT>(c, s.red);
    f = block_sum<SNT>(f, s.red64);
    if (t == 0) {
      atomicAdd(&o->cnt[at + 1], (uint32_t)c);
      atomicAdd(&o->fix[at], f);
    }
    return barrier();
  };
  if (Tfix == 0 && !sums(0.0, 0.0, 1)) {
    finish();
    return;
  }
  const u64 Sfix = Tfix ? Tfix : ld_relaxed64(&o->fix[1]);
  int keep = Tfix ? k : (int)ld_relaxed(&o->cnt[2]);
  u64 zfix = Sfix;
  uint32_t flags = VS_OUT_COOP;  // the general kernel's route bit
  if (has_tp) {  // sampler.py:145-148
    const double tgt = P.top_p * (double)Sfix;
    const Sel a = select(false, ceil_u64(tgt));
    if (!ok) {
      finish();
      return;
    }
    keep = (int)a.cnt_before + 1;
    zfix = a.mass_before + a.mass;
    const double tol = 1e-6 * (double)Sfix;
    if (fabs((double)a.mass_before - tgt) < tol || fabs((double)zfix - tgt) < tol) flags |= VS_OUT_TOPP_BOUNDARY;
  }
  if (has_mp) {  // :149-152
    const double S = (double)Sfix * inv_scale;
    if (!sums(S, (1.0 / S) * P.min_p, 2)) {
      finish();
      return;
    }
    const int cm = (int)ld_relaxed(&o->cnt[3]), km = cm > 1 ? cm : 1;
    if (km < keep) {
      keep = km;
      zfix = cm >= 1 ? ld_relaxed64(&o->fix[2]) : (u64)fsc;
    }
  }
  const double uz = P.u * (double)zfix;  // :153-156
  const Sel d = select(false, ceil_u64(uz));
  if (ok && d.key != 0) {
    const double tol = 1e-6 * (double)zfix;
    if (fabs((double)d.mass_before - uz) < tol || fabs((double)(d.mass_before + d.mass) - uz) < tol)
      flags |= VS_OUT_DRAW_BOUNDARY;
    fin.token = (int32_t)key_index(d.key);
    fin.lp = (float)((double)(key_value(d.key) / tt - xs0) - log_ge1((double)zfix * inv_scale));
    fin.keep = keep;
    fin.flags = flags;
  }
  finish();
}

template <int DT>
static const void* stream_fn(int E) {
  constexpr int VEC = DTraits<DT>::VEC;
  return E == 16 ? (const void*)vs_batch_kernel<DT, 16 / VEC> : (const void*)vs_batch_kernel<DT, 32 / VEC>;
}

// How a batch of B rows is launched on a device of `cus` CUs; mis: logits between the 16-byte line and the first logit.
struct BatchPlan {
  int rows;  // rows per launch
  int E;     // logits per lane of the stream kernel
  int G;     // its workgroups per row
  int CH;    // positions per workgroup
  int kcap;  // keys of a chunk's list at most
  int kmax;  // largest top_k finished from the lists
  int nv;    // candidates per chunk of a row without a top-k cut
};
static BatchPlan batch_plan(int V, int64_t ld, int dtype, int mis, int B, size_t ws_rows, int cus) {
  const int VEC = dtype == VS_F32 ? 4 : 8;
  BatchPlan p;
  // The resolve kernel has a workgroup per CU and gives every open row at least one: no more rows than CUs (a device
  // partition can have fewer than BATCH_ROWS).
  int nmax = ws_rows >= (size_t)RPL_MAX ? BATCH_ROWS : (int)ws_rows;
  if (nmax > cus) nmax = cus;
  p.rows = B < nmax ? B : nmax;
  // positions of a row, counted from the 16-byte line of its first logit (the rows' places in their lines differ
  // unless the stride is a multiple of 16 bytes)
  const int span = V + (ld % VEC == 0 ? mis : VEC - 1);
  // Logits per lane. 32 spend fewer instructions per logit and leave the finish kernel half the lists, 16 keep three
  // workgroups on a CU instead of two and give a small batch enough of them. V = 163840 fp32, mixed requests, us per
  // call with 16 / 32: B = 24 26.8 / 27.7, 48 34.3 / 31.7, 96 42.6 / 41.0; the line lies where 32 still fill the CUs
  // one and a half times.
  const int g32 = (span + 32 * SNT - 1) / (32 * SNT), g16 = (span + 16 * SNT - 1) / (16 * SNT);
  p.E = 2 * p.rows * g32 >= 3 * cus || g16 > GMAX ? 32 : 16;
  p.G = p.E == 32 ? g32 : g16;
  p.CH = ((span + p.G - 1) / p.G + VEC - 1) / VEC * VEC;
  p.G = (span + p.CH - 1) / p.CH;
  const int per_wave = (p.G + SNW - 1) / SNW;  // lists a wave of the finish kernel takes, BATCH_NK rounds of 64 keys together
  p.kcap = (p.rows > RPL_MAX ? BIGCAP : KEYS_CAP) / p.G / WAVE * WAVE;
  if (p.kcap > BATCH_NK / per_wave * WAVE) p.kcap = BATCH_NK / per_wave * WAVE;
  p.kmax = p.kcap < KCAP ? p.kcap : KCAP;
  // candidates per chunk of a row without a top-k cut (a chunk lists about 1.5 times as many): the nucleus of a language
  // model's row is a few hundred logits; 48, 64 and 96 measured within 2% of one another
  p.nv = p.kcap / 3 / 8 * 8 < 64 ? p.kcap / 3 / 8 * 8 : 64;
  return p;
}

int batch_path(SampleArgs a, int dtype, int B, size_t ws_rows, const DevInfo* dv, hipStream_t stream) {
  const int es = dtype == VS_F32 ? 4 : 2;
  const BatchPlan p = batch_plan(a.V, a.ld, dtype, (int)((uintptr_t)a.logits % 16) / es, B, ws_rows, dv->cus);
  a.G = p.G;
  a.CH = p.CH;
  a.kcap = p.kcap;
  a.kmax = p.kmax;
  a.NV = p.nv;
  const void* sfn =
      dtype == VS_F32 ? stream_fn<VS_F32>(p.E) : dtype == VS_BF16 ? stream_fn<VS_BF16>(p.E) : stream_fn<VS_F16>(p.E);
  const void* rfn = dtype == VS_F32    ? (const void*)vs_resolve_kernel<VS_F32>
                    : dtype == VS_BF16 ? (const void*)vs_resolve_kernel<VS_BF16>
                                       : (const void*)vs_resolve_kernel<VS_F16>;
  const void* ffn = (const void*)vs_finish_kernel;
  for (int r0 = 0; r0 < B; r0 += p.rows) {
    a.row0 = r0;
    a.B = (B - r0) < p.rows ? (B - r0) : p.rows;
    void* kargs[] = {&a};
    hipError_t e = hipLaunchKernel(sfn, dim3((unsigned)(a.B * p.G)), dim3(SNT), kargs, stream_lds(p.E * SNT), stream);
    if (e == hipSuccess) e = hipLaunchKernel(ffn, dim3((unsigned)a.B), dim3(SNT), kargs, 0, stream);
    // one workgroup per CU: all resident, so that a cluster's waits end (top lists leave no row open)
    if (e == hipSuccess && a.list_k == 0)
      e = hipLaunchKernel(rfn, dim3((unsigned)dv->cus), dim3(SNT), kargs, RESOLVE_LDS, stream);
    if (e != hipSuccess) return hip_fail(e, "vs_sample_batch: launch");
  }
  return VS_OK;
}

}  // namespace vs

extern "C" int vs_batch_plan(int dtype, int V, int64_t ld, int mis, int B, size_t ws_bytes, int cus, int* out) {
  if (!out || V < 1 || ld < V || mis < 0 || B < 1 || cus < 1 || ws_bytes < vs::ROW_WS ||
      (dtype != VS_F32 && dtype != VS_BF16 && dtype != VS_F16))
    return vs::fail(VS_EINVAL, "vs_batch_plan: bad arguments");
  const vs::BatchPlan p = vs::batch_plan(V, ld, dtype, mis, B, ws_bytes / vs::ROW_WS, cus);
  const int v[] = {p.rows, p.E, p.G, p.CH, p.kcap, p.kmax, p.nv};
  for (int i = 0; i < 7; ++i) out[i] = v[i];
  return VS_OK;
}
