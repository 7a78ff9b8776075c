// gfx950 kernel for the processed distributions of rows (probs(),
// src/pagellm/engine/sampling.py:65-91), the draw from them, and the draw alone
// for rows of a middling vocabulary: one workgroup of 1024 threads per row.
//
// The row's output is its scratch: once top-k is settled, one pass writes each
// token's exp to its place in out_probs, and every later pass reads it back
// instead of computing it again.  The general
// pipeline (plh_pipeline.h) reads the logits five to nine times, a thread's 32
// tokens in one 128-byte run, and computes each token's exp in up to five of
// its passes.  The k-th logit and the top-p cut are found on order keys: levels
// of 2048 bins of 2^sh consecutive keys from the largest down (counts, and
// fixed-point masses for the cut), until one wave can order what is left.
//
// Layout: block j of thread t holds the kVW consecutive tokens from
// (j * 1024 + t) * kVW, one 16-byte load of logits; the last V % kVW tokens are
// one more block of a token per thread.  The tokens of a wave's part of a
// block are consecutive, and these pieces (j, wave) are in vocabulary order.
// A thread reads back only exps it wrote itself.
//
// Bound by instruction issue on a row's CU: 15 to 25 instructions per token and
// pass, four to nine passes.  320 x 32 000 float32 (five kinds of rows): 204 us
// -> 108 us; one row of 32 000 with top-p 120 -> 51 us, temperature only 78 ->
// 28 us, of 128 256 399 -> 161 us.  Measured and not taken: eight loads in
// flight (same), two workgroups a CU at 64 registers (32 000 tokens: 256 rows
// 5% slower, 320 rows 2%), exps in 2-token vectors (p 0.9: 8% slower).
#include "plh_device.h"
#include "plh_fast.h"
#include "plh_kernels.h"
#include "plh_pipeline.h"

namespace plh {

namespace {

constexpr int kPT = 1024;           // threads per row
constexpr int kPW = kPT / kWave;    // waves
constexpr int kPU = 4;              // 16-byte loads in flight per thread
constexpr int kLevBins = 2048;      // bins of a selection level
constexpr int kMaxPieces = (kProbsV / (2 * kPT) + 1) * kPW;

struct ProbsSmem {
  union {
    struct {
      uint64_t mass[kLevBins];
      uint32_t cnt[kLevBins];
    };
    uint64_t piece[kMaxPieces];  // masses of the pieces
  };
  double exp_tab[64];
  uint64_t lkey[kWave], lw[kWave];  // the last bin's elements
  int lidx[kWave];
  uint64_t redu[kPW], redc[kPW];
  double redd[kPW];
  int redi[kPW];
  uint64_t out_u[1];
  int out_i[4];
  uint32_t bitmap[kProbsV / 32];
};

// Workgroup reductions over 16 waves: each wave's value to LDS, one barrier,
// every thread combines them pairwise in one order; a second barrier frees the
// slots.  Pairwise, because the last additions carry most of the rounding of a
// float64 sum: the normaliser of 32 000 tokens is 7e-17 from exact (rms), 1.1e-16
// with the waves added one after another.
template <typename T, class Op>
__device__ __forceinline__ T all_waves(T v, T* red, const Op& op) {
  if (lane() == 0) red[wave()] = v;
  __syncthreads();
  T r[kPW];
#pragma unroll
  for (int w = 0; w < kPW; ++w) r[w] = red[w];
#pragma unroll
  for (int h = kPW / 2; h > 0; h >>= 1)
#pragma unroll
    for (int w = 0; w < h; ++w) r[w] = op(r[w], r[w + h]);
  __syncthreads();
  return r[0];
}

// Exclusive scan of one value per thread.
template <typename T>
__device__ __forceinline__ T excl_scan(T v, T* red) {
  const T x = wave_scan_incl(v, T(0), OpAdd{});
  if (lane() == kWave - 1) red[wave()] = x;
  __syncthreads();
  T pre = 0;
#pragma unroll
  for (int w = 0; w < kPW; ++w) pre += w < wave() ? red[w] : T(0);
  __syncthreads();
  return pre + (x - v);
}

struct Cut {
  bool found;
  uint64_t key;   // the selected element's key
  int equals;     // how many elements share it ...
  int rank;       // ... and how many of those come up to the selected one (at least 1)
};

// Walking keys from the largest down, the element at which the running count
// (MASS: weight) first reaches target.  each(fn) calls fn(key, w, idx) for the
// calling thread's elements, w being the weight (1 for counts).  top: no key
// is larger; the first level's bins are 2^sh keys wide.
template <bool MASS, class Each>
__device__ __forceinline__ Cut select_key(const Each& each, uint64_t top, int sh, uint64_t target, ProbsSmem& sm) {
  uint64_t klo = top >= ((uint64_t)kLevBins << sh) ? top - ((uint64_t)kLevBins << sh) + 1 : 0;
  uint64_t from = 0, to = ~0ull;  // keys still in play; those below klo count as bin 0
  uint64_t above = 0;
  for (;;) {
    for (int b = threadIdx.x; b < kLevBins; b += kPT) {
      sm.cnt[b] = 0u;
      if (MASS) sm.mass[b] = 0ull;
    }
    if (threadIdx.x == 0) sm.out_i[0] = -1;
    __syncthreads();
    each([&](uint64_t key, uint64_t w, int) {
      if (key < from || key > to) return;
      const uint64_t d = key < klo ? 0 : (key - klo) >> sh;
      const int b = (int)(d < kLevBins ? d : kLevBins - 1);
      lds_add(&sm.cnt[b], 1u);
      if (MASS) lds_add(&sm.mass[b], w);
    });
    __syncthreads();
    // thread t holds the t-th run of bins from the top
    constexpr int per = kLevBins / kPT;
    uint64_t v[per], sum = 0;
#pragma unroll
    for (int i = 0; i < per; ++i) {
      const int b = kLevBins - 1 - (per * (int)threadIdx.x + i);
      v[i] = MASS ? sm.mass[b] : sm.cnt[b];
      sum += v[i];
    }
    uint64_t run = above + excl_scan<uint64_t>(sum, sm.redu);
#pragma unroll
    for (int i = 0; i < per; ++i) {
      if (run < target && run + v[i] >= target) {  // one bin
        sm.out_i[0] = kLevBins - 1 - (per * (int)threadIdx.x + i);
        sm.out_u[0] = run;
      }
      run += v[i];
    }
    __syncthreads();
    const int b = sm.out_i[0];
    if (b < 0) return Cut{false, 0, 0, 0};
    above = sm.out_u[0];
    const int n = (int)sm.cnt[b];
    const uint64_t nlo = b == 0 ? from : klo + ((uint64_t)b << sh);
    const uint64_t nhi = b == kLevBins - 1 ? to : klo + ((uint64_t)b << sh) + ((1ull << sh) - 1);
    from = nlo;
    to = nhi < to ? nhi : to;
    __syncthreads();
    if (n <= kWave) {
      if (threadIdx.x == 0) sm.out_i[1] = 0;
      __syncthreads();
      each([&](uint64_t key, uint64_t w, int idx) {
        if (key < from || key > to) return;
        const int i = lds_fetch_add(&sm.out_i[1], 1);
        sm.lkey[i] = key;
        sm.lw[i] = w;
        sm.lidx[i] = idx;
      });
      __syncthreads();
      if (wave() == 0) {
        const int l = lane();
        const uint64_t key = l < n ? sm.lkey[l] : 0, w = l < n ? sm.lw[l] : 0;
        const int idx = l < n ? sm.lidx[l] : INT_MAX;
        uint64_t run2 = above;
        int rank = 1, equals = 0;
        for (int i = 0; i < n; ++i) {
          const uint64_t ki = lane_value(key, i), wi = lane_value(w, i);
          const int xi = lane_value(idx, i);
          const bool ahead = ki > key || (ki == key && xi < idx);
          run2 += ahead ? wi : 0;
          rank += ki == key && xi < idx ? 1 : 0;
          equals += ki == key ? 1 : 0;
        }
        if (l < n && run2 < target && run2 + w >= target) {  // one lane
          sm.out_u[0] = key;
          sm.out_i[2] = rank;
          sm.out_i[3] = equals;
        }
      }
      __syncthreads();
      const Cut c{true, sm.out_u[0], sm.out_i[3], sm.out_i[2]};
      __syncthreads();
      return c;
    }
    // the elements' own range
    uint64_t lo = ~0ull, hi = 0, wt = 0;
    each([&](uint64_t key, uint64_t w, int) {
      if (key < from || key > to) return;
      lo = key < lo ? key : lo;
      hi = key > hi ? key : hi;
      wt = w;
    });
    from = all_waves(wave_min(lo), sm.redu, OpMin{});
    to = all_waves(wave_max(hi), sm.redc, OpMax{});
    if (from == to) {  // all equal: as many of them as reach the target
      wt = all_waves(wave_max(wt), sm.redu, OpMax{});
      const uint64_t need = wt > 0 ? (target - above - 1) / wt + 1 : (uint64_t)n;
      return Cut{true, from, n, (int)(need < (uint64_t)n ? need : (uint64_t)n)};
    }
    klo = from;
    const uint64_t span = to - from;
    sh = span < (uint64_t)kLevBins ? 0 : 64 - __builtin_clzll(span) - 11;
  }
}

// EXPORT: the row's distribution is wanted, and its place holds the exps.
// Otherwise (ids only) they are held in LDS, and before them the penalised
// logits, for rows of at most kRowV tokens.
template <typename TIn, bool EXPORT>
__global__ __launch_bounds__(kPT) void k_probs_row(SampleArgs a) {
  constexpr int kVW = 16 / (int)sizeof(TIn);
  typedef TIn VI __attribute__((ext_vector_type(kVW))) __attribute__((aligned(sizeof(TIn))));
  typedef double VO __attribute__((ext_vector_type(kVW))) __attribute__((aligned(8)));
  __shared__ ProbsSmem sm;
  __shared__ alignas(16) double row_e[EXPORT ? 1 : kRowV];
  const int row = blockIdx.x, V = a.V, tid = threadIdx.x;
  const TIn* x = reinterpret_cast<const TIn*>(a.logits) + (int64_t)row * a.ld;
  double* const po = EXPORT ? a.out_probs + (int64_t)row * V : nullptr;
  const RowParams rp = load_row_params(a, row);
  if (tid < 64) sm.exp_tab[tid] = kExp2Frac64[tid];
  if (rp.pen_active) {
    for (int w = tid; w < (V + 31) / 32; w += kPT) sm.bitmap[w] = 0u;
    __syncthreads();
    for (int64_t h = rp.h0 + tid; h < rp.h1; h += kPT) {
      const int id = a.hist_ids[h];
      if ((unsigned)id < (unsigned)V) lds_or(&sm.bitmap[id >> 5], 1u << (id & 31));
    }
  }
  __syncthreads();

  const int nvec = V / kVW, rem = V - nvec * kVW;   // whole vectors, tokens past them
  const int nb = (nvec + kPT - 1) / kPT;            // blocks, without the last one
  // A pass over the thread's tokens: f(j, t, n, v) with v[0 .. n-1] the values
  // of tokens t .. t+n-1 (n is kVW, or 0 where the row ends before the thread;
  // in the block of the last V % kVW tokens, j = nb, 1 or 0).  Every thread
  // makes the same calls.
  auto pass = [&](auto vec, auto one, auto f) {
    for (int j0 = 0; j0 < nb; j0 += kPU) {
      decltype(vec(0)) v[kPU];
#pragma unroll
      for (int u = 0; u < kPU; ++u) v[u] = vec(min((j0 + u) * kPT + tid, nvec - 1) * kVW);
#pragma unroll
      for (int u = 0; u < kPU; ++u) {
        if (j0 + u >= nb) break;  // uniform
        const int i = (j0 + u) * kPT + tid;
        double d[kVW];
#pragma unroll
        for (int e = 0; e < kVW; ++e) d[e] = (double)v[u][e];
        f(j0 + u, i * kVW, i < nvec ? kVW : 0, d);
      }
    }
    if (rem > 0) {
      const int t = nvec * kVW + tid;
      double d[kVW] = {};
      if (tid < rem) d[0] = (double)one(t);
      f(nb, t, tid < rem ? 1 : 0, d);
    }
  };
  // the penalised logits
  auto pass_z = [&](auto f) {
    pass([&](int t) { return *reinterpret_cast<const VI*>(x + t); }, [&](int t) { return x[t]; },
         [&](int j, int t, int n, double (&d)[kVW]) {
           if (rp.pen_active && n > 0) {
             // kVW divides 32: one word (the last block: its first bit)
             const uint32_t pb = sm.bitmap[t >> 5] >> (t & 31);
#pragma unroll
             for (int e = 0; e < kVW; ++e)
               if ((pb >> e) & 1u && e < n) d[e] = penalize(d[e], rp.pen);
           }
           f(j, t, n, d);
         });
  };
  // the exps, once written
  auto pass_e = [&](auto f) {
    if constexpr (EXPORT)
      pass([&](int t) { return *reinterpret_cast<const VO*>(po + t); }, [&](int t) { return po[t]; }, f);
    else
      pass([&](int t) { return *reinterpret_cast<const VO*>(row_e + t); }, [&](int t) { return row_e[t]; }, f);
  };
  auto store = [&](int t, int n, const double (&p)[kVW]) {
    if (n == kVW) {
      VO v;
#pragma unroll
      for (int e = 0; e < kVW; ++e) v[e] = p[e];
      if constexpr (EXPORT) *reinterpret_cast<VO*>(po + t) = v;
      else *reinterpret_cast<VO*>(row_e + t) = v;
    } else if (n > 0) {
      if constexpr (EXPORT) po[t] = p[0];
      else row_e[t] = p[0];
    }
  };

  // ---- the maximum, and its lowest index (:73, :79)
  ArgMax best{-INFINITY, INT_MAX};
  pass_z([&](int, int t, int n, double (&z)[kVW]) {
#pragma unroll
    for (int e = 0; e < kVW; ++e)
      if (e < n) best = argmax_merge(best, ArgMax{z[e], t + e});
    if constexpr (!EXPORT) store(t, n, z);  // the later passes over the logits
  });
  auto pass_y = [&](auto f) {
    if constexpr (EXPORT) pass_z(f);
    else pass_e(f);
  };
  best = wave_argmax(best);
  const double zmax = all_waves(best.v, sm.redd, [](double p, double q) { return p > q ? p : q; });
  if (rp.greedy) {  // :71-74
    const int id = min(all_waves(best.v == zmax ? best.i : INT_MAX, sm.redi, OpMin{}), V - 1);
    if (tid == 0) a.out_ids[row] = id;
    if constexpr (!EXPORT) return;
    typedef double V2 __attribute__((ext_vector_type(2))) __attribute__((aligned(8)));
    for (int i = 2 * tid; i < V; i += 2 * kPT) {  // a kilobyte per store of a wave
      if (i + 1 < V) *reinterpret_cast<V2*>(po + i) = V2{i == id ? 1.0 : 0.0, i + 1 == id ? 1.0 : 0.0};
      else po[i] = i == id ? 1.0 : 0.0;
    }
    return;
  }
  const double T = rp.T, invT = 1.0 / T;

  // ---- top-k: keep y >= kth_y (:76-78)
  double z_lo = -INFINITY;
  if (rp.topk) {
    auto each = [&](auto fn) {
      pass_y([&](int, int t, int n, double (&z)[kVW]) {
#pragma unroll
        for (int e = 0; e < kVW; ++e)
          if (e < n) fn(key_of(z[e]), (uint64_t)1, t + e);
      });
    };
    // bins of 1/256 octave of the logit
    const Cut c = select_key<false>(each, key_of(zmax), 44, (uint64_t)rp.top_k, sm);
    if (c.found) z_lo = topk_floor(val_of_key(c.key), T);
  }

  // ---- softmax over the survivors (:79-81): the exps to the row's output
  const PCalc pc{invT, zmax * invT, 1.0, z_lo, sm.exp_tab};
  double s = 0.0;
  pass_y([&](int, int t, int n, double (&z)[kVW]) {
    double v[kVW];
#pragma unroll
    for (int e = 0; e < kVW; ++e) {
      v[e] = p_of(pc, z[e]);
      if (e < n) s += v[e];
    }
    store(t, n, v);
  });
  const double S = all_waves(wave_sum(s), sm.redd, OpAdd{}), invS = 1.0 / S;

  // ---- top-p (:82-90): the cut in (p descending, index ascending) order
  bool have_cut = false;
  double cut = 0.0;   // every p above it is kept ...
  int equals = 0, rank = 0;  // ... and of those equal to it the first `rank`
  if (rp.topp) {
    auto each = [&](auto fn) {
      pass_e([&](int, int t, int n, double (&d)[kVW]) {
#pragma unroll
        for (int e = 0; e < kVW; ++e) {
          const double p = d[e] * invS;
          if (e < n && p > 0.0) fn(pkey_of(p), to_fx(p), t + e);
        }
      });
    };
    // bins of 1/64 octave of the probability; the largest is at most invS
    const Cut c = select_key<true>(each, pkey_of(invS), 46, topp_target(rp.top_p), sm);
    have_cut = c.found;
    cut = __longlong_as_double((long long)c.key);
    equals = c.equals;
    rank = c.rank;
  }
  const bool ties = have_cut && rank < equals;
  // the probability a token keeps, or 0 (without top-p: p itself)
  auto keep = [&](double p) { return !have_cut || p >= cut ? p : 0.0; };

  // ---- the kept masses of the pieces, in vocabulary order (:94-98)
  double kept = 0.0;
  int before = 0;  // tokens equal to the cut in earlier blocks
  pass_e([&](int j, int t, int n, double (&d)[kVW]) {
    double p[kVW];
#pragma unroll
    for (int e = 0; e < kVW; ++e) p[e] = e < n ? keep(d[e] * invS) : 0.0;
    if (ties) {  // uniform
      int m = 0;
#pragma unroll
      for (int e = 0; e < kVW; ++e) m += p[e] == cut ? 1 : 0;
      int k = before + excl_scan<int>(m, sm.redi);
      before += all_waves(wave_sum(m), sm.redi, OpAdd{});
#pragma unroll
      for (int e = 0; e < kVW; ++e) {
        const bool eq = p[e] == cut;
        if (eq && k >= rank) d[e] = p[e] = 0.0;
        k += eq ? 1 : 0;
      }
      store(t, n, d);  // the tokens after the cut weigh nothing from here on
    }
    uint64_t m = 0;
#pragma unroll
    for (int e = 0; e < kVW; ++e) {
      m += to_fx(p[e]);
      kept += p[e];
    }
    m = wave_sum(m);
    if (lane() == 0) sm.piece[j * kPW + wave()] = m;
  });
  const double s2 = all_waves(wave_sum(kept), sm.redd, OpAdd{});  // its barriers also publish the pieces

  // ---- inverse-CDF draw: the crossing piece, then its token, by the wave
  // that holds it
  {
    const int pieces = (nb + (rem > 0 ? 1 : 0)) * kPW;
    uint64_t tot = 0;
    for (int i = 0; i < pieces; i += kWave) tot += wave_sum(i + lane() < pieces ? sm.piece[i + lane()] : 0);
    const uint64_t t_fx = (uint64_t)__double2ull_rd(rp.u * (double)tot);
    uint64_t run = 0, start = 0;
    int at = -1;
    for (int i = 0; i < pieces && at < 0; i += kWave) {
      const uint64_t v = i + lane() < pieces ? sm.piece[i + lane()] : 0;
      const uint64_t incl = run + wave_scan_incl(v, (uint64_t)0, OpAdd{});
      const uint64_t over = __ballot(incl > t_fx);
      if (over != 0) {
        const int k = __builtin_ctzll(over);
        at = i + k;
        start = lane_value(incl - v, k);
      }
      run = lane_value(incl, kWave - 1);
    }
    if (at < 0) {
      if (tid == 0) a.out_ids[row] = V - 1;
    } else if (at % kPW == wave()) {
      const int j = at / kPW, i = j * kPT + tid;
      const int t = j < nb ? i * kVW : nvec * kVW + tid, n = j < nb ? (i < nvec ? kVW : 0) : (tid < rem ? 1 : 0);
      uint64_t w[kVW], ts = 0;
#pragma unroll
      for (int e = 0; e < kVW; ++e) {
        w[e] = e < n ? to_fx(keep((EXPORT ? po[t + e] : row_e[t + e]) * invS)) : 0;
        ts += w[e];
      }
      uint64_t c = start + wave_scan_incl(ts, (uint64_t)0, OpAdd{}) - ts;
      int hit = INT_MAX;
#pragma unroll
      for (int e = 0; e < kVW; ++e) {
        c += w[e];
        if (hit == INT_MAX && c > t_fx) hit = t + e;
      }
      hit = wave_min(hit);
      if (lane() == 0) a.out_ids[row] = min(hit, V - 1);
    }
  }

  if constexpr (!EXPORT) return;
  // ---- the distribution: top-p renormalises the kept mass (:89-90)
  pass_e([&](int, int t, int n, double (&d)[kVW]) {
    double p[kVW];
#pragma unroll
    for (int e = 0; e < kVW; ++e) {
      p[e] = keep(d[e] * invS);
      if (have_cut) p[e] = p[e] / s2;
    }
    store(t, n, p);
  });
}

}  // namespace

// Ids of rows of kSmallV + 1 to kRowV tokens.  Microseconds, the chunked path /
// here, 16 rows: 4096 tokens top-k 20.1 / 13.2, top-p 49 / 12.8, top-k + top-p +
// penalty 63 / 17.7, Zipf rows with top-p and penalty 27.8 / 12.6; 8192 tokens
// 18.1 / 16.6, 53 / 16.6, 23.8 / 21.9, 27.4 / 15.6.  One workgroup fills a CU, so
// past one row a CU the long rows with a top-k take longer (1024 x 8192: top-k
// 56 / 64, top-k + top-p + penalty 73 / 88; 1024 x 4096: 62 / 49, 226 / 68).
bool one_launch_ids(int B, int V, int num_cu) { return V <= kRowV / 2 || (V <= kRowV && B <= num_cu); }

hipError_t launch_probs_rows(const SampleArgs& a, bool f64, hipStream_t s, hipEvent_t between) {
  const bool e = a.out_probs != nullptr;
  auto k = f64 ? (e ? k_probs_row<double, true> : k_probs_row<double, false>)
               : (e ? k_probs_row<float, true> : k_probs_row<float, false>);
  hipLaunchKernelGGL(k, dim3(a.B), dim3(kPT), 0, s, a);
  if (between != nullptr) {
    const hipError_t r = hipEventRecord(between, s);
    if (r != hipSuccess) return r;
  }
  return hipGetLastError();
}

}  // namespace plh
