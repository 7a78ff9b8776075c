// gfx950 kernel for rows of a small vocabulary (character and byte models):
// the whole of sample() / probs() (src/pagellm/engine/sampling.py:65-107) in
// one launch, one workgroup per row, with the row in registers.
//
// The chunked path's two launches are two latency chains (parameters, logits,
// candidate slots, the merge's loads) whatever the row's length.  Here thread
// t holds tokens t*E .. t*E+E-1; the row's logits are sorted (bitonic, in
// registers, over lanes and, for the widest strides, through LDS), after which
// top-k is one position of the sorted row and the top-p cut one prefix sum of
// its fixed-point masses.  Only values are sorted: which of the tokens that
// share the cut's probability are kept is a count in vocabulary order.
//
// Bound by its chain of steps: one load round trip (two with a history), a
// handful of workgroup reductions, and (log2 N)(log2 N + 1) / 2 exchange steps
// of a row padded to N = 2^n tokens.
//
// 16 rows, microseconds per call, the chunked path / here: 65 tokens 23.6 / 8.3
// (top-k, top-p and penalty), 512 tokens 68 / 9.7, 1024 tokens 69 / 13.1; greedy
// rows 10.5 / 8.  Past 1024 tokens the sort grows longer than the selection of
// k_probs_row (2048 tokens: 20 here, 12.5 to 17.5 there).  probs() of 16 rows:
// 65 tokens 66 / 8.4 against the general pipeline, 1000 tokens 67 / 13.5.
#include "plh_device.h"
#include "plh_fast.h"
#include "plh_kernels.h"
#include "plh_pipeline.h"

namespace plh {

namespace {

template <int E>
struct SmallSmem {
  double sort[kThreads * E];
  double redd[kWaves];
  uint64_t redu[kWaves];
  int redi[kWaves];
  double exp_tab[kWaves][64];
  uint32_t bitmap[kThreads * E / 32];
  double kth;
  double cut_p;
  uint64_t cut_above;
  int cut_count;
};

__device__ __forceinline__ double lane_xor(double v, int m) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const int addr = (lane() ^ m) * 4;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)u);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Sorts the first N (a power of two, uniform) of the workgroup's values in
// descending order; thread t holds values t*E .. t*E+E-1.
template <int E>
__device__ __forceinline__ void sort_desc(double (&v)[E], int N, double* lds) {
  const int i0 = (int)threadIdx.x * E;
  for (int k = 2; k <= N; k <<= 1) {
    int j = k >> 1;
    for (; j >= kWave * E; j >>= 1) {  // partners in other waves
      wg_barrier();
#pragma unroll
      for (int e = 0; e < E; ++e) lds[i0 + e] = v[e];
      wg_barrier();
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = i0 + e;
        const double o = lds[i ^ j];
        v[e] = (((i & j) == 0) == ((i & k) == 0)) ? fmax(v[e], o) : fmin(v[e], o);
      }
    }
    for (; j >= E; j >>= 1) {  // partners in other lanes
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = i0 + e;
        const double o = lane_xor(v[e], j / E);
        v[e] = (((i & j) == 0) == ((i & k) == 0)) ? fmax(v[e], o) : fmin(v[e], o);
      }
    }
#pragma unroll
    for (int js = E / 2; js > 0; js >>= 1) {  // partners in the same thread
      if (js > j) continue;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if ((e & js) != 0) continue;
        const bool up = ((i0 + e) & k) == 0;
        const double a = fmax(v[e], v[e + js]), b = fmin(v[e], v[e + js]);
        v[e] = up ? a : b;
        v[e + js] = up ? b : a;
      }
    }
  }
}

template <typename TIn, int E>
__global__ __launch_bounds__(kThreads) void k_sample_small(SampleArgs a) {
  __shared__ SmallSmem<E> sm;
  const int row = blockIdx.x, V = a.V, tid = threadIdx.x, i0 = tid * E;
  const TIn* x = reinterpret_cast<const TIn*>(a.logits) + (int64_t)row * a.ld;
  RowLoad rl;
  issue_row_params(a, row, rl);
  TIn raw[E];
#pragma unroll
  for (int e = 0; e < E; ++e) raw[e] = x[min(i0 + e, V - 1)];
  double* tab = sm.exp_tab[wave()];
  init_exp_table_wave(tab);
  const RowParams rp = row_params_of(a, rl);

  double z[E];
#pragma unroll
  for (int e = 0; e < E; ++e) z[e] = i0 + e < V ? (double)raw[e] : -INFINITY;
  if (rp.pen_active) {
    for (int w = tid; w < kThreads * E / 32; w += kThreads) sm.bitmap[w] = 0u;
    wg_barrier();
    constexpr int kBatch = 4;
    for (int64_t h0 = rp.h0; h0 < rp.h1; h0 += kBatch * kThreads) {
      int id[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        const int64_t h = h0 + j * kThreads + tid;
        id[j] = h < rp.h1 ? a.hist_ids[h] : -1;
      }
#pragma unroll
      for (int j = 0; j < kBatch; ++j)
        if ((unsigned)id[j] < (unsigned)V) lds_or(&sm.bitmap[id[j] >> 5], 1u << (id[j] & 31));
    }
    wg_barrier();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = i0 + e;
      if ((sm.bitmap[i >> 5] >> (i & 31)) & 1u) z[e] = penalize(z[e], rp.pen);
    }
  }

  double* po = a.out_probs != nullptr ? a.out_probs + (int64_t)row * V : nullptr;
  if (rp.greedy) {  // sampling.py:71-74 / :102-106
    ArgMax best{-INFINITY, INT_MAX};
#pragma unroll
    for (int e = 0; e < E; ++e) best = argmax_merge(best, ArgMax{z[e], i0 + e});
    best = block_argmax(best, sm.redd, sm.redi);
    const int id = min(best.i, V - 1);
    if (po != nullptr) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (i0 + e < V) po[i0 + e] = i0 + e == id ? 1.0 : 0.0;
    }
    if (tid == 0) a.out_ids[row] = id;
    return;
  }
  const double T = rp.T, invT = 1.0 / T;

  // the logits in descending order (only a mask needs it), and the maximum
  double s[E], zmax;
  const bool sorted = rp.topk || rp.topp;
  if (sorted) {
#pragma unroll
    for (int e = 0; e < E; ++e) s[e] = z[e];
    int N = 2;
    while (N < V) N <<= 1;
    sort_desc<E>(s, N, sm.sort);
    if (tid == 0) sm.redd[0] = s[0];
    if (rp.topk && (rp.top_k - 1) / E == tid) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        if ((rp.top_k - 1) % E == e) sm.kth = s[e];
    }
    wg_barrier();
    zmax = sm.redd[0];
    wg_barrier();
  } else {
    zmax = z[0];
#pragma unroll
    for (int e = 1; e < E; ++e) zmax = fmax(zmax, z[e]);
    zmax = block_max(zmax, sm.redd);
  }

  // ---- top-k: keep y >= kth_y (:76-78)
  double z_lo = -INFINITY;
  if (rp.topk) z_lo = topk_floor(sm.kth, T);

  // ---- softmax over the survivors (:79-81)
  const double ymax = zmax * invT;
  const PCalc pc0{invT, ymax, 1.0, z_lo, tab};
  double p[E], sum = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    p[e] = i0 + e < V ? p_of(pc0, z[e]) : 0.0;
    sum += p[e];
  }
  const double S = block_sum(sum, sm.redd), invS = 1.0 / S;
#pragma unroll
  for (int e = 0; e < E; ++e) p[e] *= invS;

  // ---- top-p (:82-90): in descending order, the first token whose inclusive
  // mass reaches top_p is the cut.  Tokens of a larger p are kept, and as many
  // of those that share the cut's p (lowest index first) as reach it.
  bool have_cut = false;
  double cut_p = 0.0;
  int cut_count = 0;
  if (rp.topp) {
    const uint64_t target = topp_target(rp.top_p);
    const PCalc pc{invT, ymax, invS, z_lo, tab};
    double q[E];
    uint64_t w = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      q[e] = i0 + e < V ? p_of(pc, s[e]) : 0.0;
      w += to_fx(q[e]);
    }
    uint64_t tot;
    uint64_t run = block_excl_scan<uint64_t>(w, sm.redu, &tot);
    have_cut = tot >= target;
    if (have_cut) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint64_t we = to_fx(q[e]);
        if (run < target && run + we >= target) {  // one token of the row
          sm.cut_p = q[e];
          sm.cut_above = run + we;
        }
        run += we;
      }
      wg_barrier();
      cut_p = sm.cut_p;
      // how many of the cut's equals come up to the cut
      const uint64_t above = sm.cut_above;
      run -= w;
      int n = 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        run += to_fx(q[e]);
        n += q[e] == cut_p && run <= above && i0 + e < V ? 1 : 0;
      }
      cut_count = block_sum<int>(n, sm.redi);
    }
  }
  // ---- the kept tokens' masses, in vocabulary order
  int equal = 0;
  if (have_cut) {
    int mine = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) mine += i0 + e < V && p[e] == cut_p ? 1 : 0;
    int tot;
    equal = block_excl_scan<int>(mine, sm.redi, &tot);
  }
  uint64_t w[E], mass = 0;
  double kept = 0.0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (have_cut) {
      const bool eq = i0 + e < V && p[e] == cut_p;
      if (!(p[e] > cut_p || (eq && equal < cut_count))) p[e] = 0.0;
      equal += eq ? 1 : 0;
    }
    w[e] = to_fx(p[e]);
    mass += w[e];
    kept += p[e];
  }

  // ---- inverse-CDF draw (:94-98)
  uint64_t tot;
  uint64_t run = block_excl_scan<uint64_t>(mass, sm.redu, &tot);
  const uint64_t t_fx = (uint64_t)__double2ull_rd(rp.u * (double)tot);
  int hit = INT_MAX;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    run += w[e];
    if (hit == INT_MAX && run > t_fx) hit = i0 + e;
  }
  hit = block_min<int>(hit, sm.redi);
  if (tid == 0) a.out_ids[row] = min(hit, V - 1);

  if (po != nullptr) {  // top-p renormalises the kept mass (:89-90)
    const double s2 = have_cut ? block_sum(kept, sm.redd) : 1.0;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (i0 + e < V) po[i0 + e] = have_cut ? p[e] / s2 : p[e];
  }
}

static_assert(kSmallV == 2 * kThreads, "the widest instantiation below");

template <typename TIn>
void launch_small_t(const SampleArgs& a, hipStream_t s) {
  const dim3 grid(a.B), block(kThreads);
  if (a.V <= kThreads) hipLaunchKernelGGL((k_sample_small<TIn, 1>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_sample_small<TIn, 2>), grid, block, 0, s, a);
}

}  // namespace

hipError_t launch_sample_small(const SampleArgs& a, bool f64, hipStream_t s, hipEvent_t between) {
  if (f64) launch_small_t<double>(a, s);
  else launch_small_t<float>(a, s);
  if (between != nullptr) {
    const hipError_t e = hipEventRecord(between, s);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

}  // namespace plh
