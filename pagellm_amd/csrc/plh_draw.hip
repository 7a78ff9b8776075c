// gfx950 kernels for draw() (src/pagellm/engine/sampling.py:94-98): the
// inverse-CDF draw from rows of non-negative weights.
//
// A row is cut into pieces of 512 tokens.  One pass over the row sums each
// piece in float64 (a wave's piece is whole 16-byte loads of consecutive
// tokens); the running piece totals, added in one fixed order, give W and the
// first piece whose total exceeds u * W, and only that piece is read again for
// the token.  float32 rows are widened exactly.
//
//   k_draw_row    one workgroup per row, the piece sums in LDS: one launch;
//   k_draw_parts  a workgroup per 16 384 tokens of a row, the piece sums in
//   k_draw_pick   the workspace, then a wave per row: for long rows that are
//                 too few to fill the chip one workgroup each.
//
// The float64 sums run in another order than numpy's cumsum, so the token
// differs from the reference's only when u lies within ~1e-15 (relative) of a
// CDF boundary.  Where rounding leaves the crossing just past the piece's end,
// the piece's last token of positive weight is taken (a neighbour of the
// boundary either way).
//
// Bound by the read of the rows and, for a few dozen rows, by one workgroup's
// latency chain (a load round trip, the piece sums, the reread).
// 64 x 32 000 float64: 39.9 -> 6.4 us against three passes over the row with a
// float64 division per token; 512 x 152 064: 108 us, 5.8 TB/s.
#include "plh_device.h"
#include "plh_kernels.h"

namespace plh {

namespace {

constexpr int kPiece = 512;         // tokens per piece
constexpr int kDrawChunk = 32;   // pieces per workgroup of k_draw_parts
constexpr int kMaxPieces = 2048;  // pieces whose sums k_draw_row holds (V <= 1 048 576)

template <typename TIn>
struct DrawGeo {
  static constexpr int kVW = 16 / (int)sizeof(TIn);
  static constexpr int kLoads = kPiece / (kVW * kWave);  // 16-byte loads per lane and piece
  typedef TIn V __attribute__((ext_vector_type(kVW))) __attribute__((aligned(sizeof(TIn))));
};

__device__ __forceinline__ double weight_of(double v) { return v > 0.0 ? v : 0.0; }

// The calling lane's tokens of piece s: load j holds tokens
// s * 512 + (j * 64 + lane) * kVW onwards.  Tokens past the row weigh nothing.
template <typename TIn>
__device__ __forceinline__ void load_piece(const TIn* p, int V, int s, typename DrawGeo<TIn>::V (&x)[DrawGeo<TIn>::kLoads]) {
  using G = DrawGeo<TIn>;
  const int i0 = s * kPiece + lane() * G::kVW;
  if (V - s * kPiece >= kPiece) {
#pragma unroll
    for (int j = 0; j < G::kLoads; ++j)
      x[j] = *reinterpret_cast<const typename G::V*>(p + i0 + j * G::kVW * kWave);
  } else {
#pragma unroll
    for (int j = 0; j < G::kLoads; ++j)
#pragma unroll
      for (int e = 0; e < G::kVW; ++e) {
        const int i = i0 + j * G::kVW * kWave + e;
        x[j][e] = i < V ? p[i] : TIn(0);
      }
  }
}

template <typename TIn>
__device__ __forceinline__ double lane_sum(const typename DrawGeo<TIn>::V (&x)[DrawGeo<TIn>::kLoads]) {
  using G = DrawGeo<TIn>;
  double t = 0.0;
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j)
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) t += weight_of((double)x[j][e]);
  return t;
}

// The sums of pieces s .. s+U-1 into out[0 ..], all loads in flight together;
// pieces past the last (all up to it lie inside the row) read as the last and
// are dropped, so that no branch parts the loads.
template <int U, typename TIn>
__device__ __forceinline__ void sum_batch(const TIn* p, int s, int last, double* out) {
  typename DrawGeo<TIn>::V x[U][DrawGeo<TIn>::kLoads];
#pragma unroll
  for (int i = 0; i < U; ++i) load_piece(p, INT_MAX, min(s + i, last), x[i]);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const double t = wave_sum(lane_sum<TIn>(x[i]));
    if (lane() == 0 && s + i <= last) out[i] = t;
  }
}

// Sums pieces s0 .. s1-1 of a row into out[0 ..], by one wave.
template <typename TIn>
__device__ __forceinline__ void sum_pieces(const TIn* p, int V, int s0, int s1, double* out) {
  typename DrawGeo<TIn>::V tail[DrawGeo<TIn>::kLoads];
  const bool ragged = s0 < s1 && (int64_t)s1 * kPiece > V;  // the row's last piece, cut short
  const int last = ragged ? s1 - 2 : s1 - 1;
  if (ragged) load_piece(p, V, s1 - 1, tail);
  int s = s0;
  for (; s + 4 <= last; s += 8) sum_batch<8>(p, s, last, out + (s - s0));
  if (s + 2 <= last) sum_batch<4>(p, s, last, out + (s - s0));
  else if (s + 1 <= last) sum_batch<2>(p, s, last, out + (s - s0));
  else if (s <= last) sum_batch<1>(p, s, last, out + (s - s0));
  if (ragged) {
    const double t = wave_sum(lane_sum<TIn>(tail));
    if (lane() == 0) out[s1 - 1 - s0] = t;
  }
}

// The drawn token of a row whose n piece sums are sum(i); by one wave, every
// lane alike.
template <typename TIn, class Sum>
__device__ __forceinline__ int pick_token(const TIn* p, int V, double u, const Sum& sum, int n) {
  using G = DrawGeo<TIn>;
  double run = 0.0;
  for (int base = 0; base < n; base += kWave)
    run = lane_value(run + wave_scan_incl(sum(base + lane()), 0.0, OpAdd{}), kWave - 1);
  const double W = run;
  // no mass, or more than a double holds, or u past the end: the last id
  // (sampling.py:98 clamps to V - 1)
  if (!(W > 0.0) || W > 1.7976931348623157e308 || u >= 1.0) return V - 1;
  const double t = fmax(u * W, 0.0);
  // the first piece whose running total exceeds t, else the last with mass
  int f = -1, last = -1;
  double before = 0.0, blast = 0.0;
  run = 0.0;
  for (int base = 0; base < n && f < 0; base += kWave) {
    const double v = sum(base + lane());
    const double incl = run + wave_scan_incl(v, 0.0, OpAdd{});
    const uint64_t pos = __ballot(v > 0.0), over = __ballot(v > 0.0 && incl > t);
    if (over != 0) {
      const int k = __builtin_ctzll(over);
      f = base + k;
      before = lane_value(incl - v, k);
    } else if (pos != 0) {
      const int k = 63 - __builtin_clzll(pos);
      last = base + k;
      blast = lane_value(incl - v, k);
    }
    run = lane_value(incl, kWave - 1);
  }
  const bool crossed = f >= 0;
  if (!crossed) {
    f = last;
    before = blast;
  }
  typename G::V x[G::kLoads];
  load_piece(p, V, f, x);
  int tok = -1, tail = -1;
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j) {
    double w[G::kVW], ts = 0.0;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) {
      w[e] = weight_of((double)x[j][e]);
      ts += w[e];
    }
    const double incl = wave_scan_incl(ts, 0.0, OpAdd{});
    double cum = before + (incl - ts);
    const int i0 = f * kPiece + (j * kWave + lane()) * G::kVW;
    int hit = INT_MAX, pos = -1;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) {
      cum += w[e];
      if (w[e] > 0.0) {
        pos = i0 + e;
        if (hit == INT_MAX && cum > t) hit = i0 + e;
      }
    }
    tail = max(tail, wave_max(pos));
    const int h = wave_min(hit);
    if (crossed && tok < 0 && h != INT_MAX) tok = h;
    before += lane_value(incl, kWave - 1);
  }
  return tok >= 0 ? tok : tail;
}

template <typename TIn>
__global__ __launch_bounds__(kThreads) void k_draw_row(DrawArgs a) {
  __shared__ double sums[kMaxPieces];
  const int row = blockIdx.x, n = (a.V - 1) / kPiece + 1, w = uniform(wave());
  const TIn* p = reinterpret_cast<const TIn*>(a.p) + (int64_t)row * a.ld;
  const double u = a.uniforms[row];
  int id;
  if (n <= kMaxPieces) {
    const int per = (n + kWaves - 1) / kWaves, s0 = min(w * per, n), s1 = min(s0 + per, n);
    sum_pieces(p, a.V, s0, s1, sums + s0);
    wg_barrier();
    if (w != 0) return;
    id = pick_token(p, a.V, u, [&](int i) { return i < n ? sums[i] : 0.0; }, n);
  } else {
    // longer than any vocabulary, and no workspace to hold the sums: one wave
    // forms each piece's sum where it is needed
    if (w != 0) return;
    id = pick_token(p, a.V, u, [&](int i) {
      double mine = 0.0;
      const int first = i - lane();
      for (int k = 0; k < kWave && first + k < n; ++k) {
        typename DrawGeo<TIn>::V x[DrawGeo<TIn>::kLoads];
        load_piece(p, a.V, first + k, x);
        const double t = wave_sum(lane_sum<TIn>(x));
        if (lane() == k) mine = t;
      }
      return mine;
    }, n);
  }
  if (lane() == 0) a.out_ids[row] = id;
}

template <typename TIn>
__global__ __launch_bounds__(kThreads) void k_draw_parts(DrawArgs a) {
  const int n = (a.V - 1) / kPiece + 1, C = (n + kDrawChunk - 1) / kDrawChunk;
  const int row = blockIdx.x / C, c = blockIdx.x % C, w = uniform(wave());
  const TIn* p = reinterpret_cast<const TIn*>(a.p) + (int64_t)row * a.ld;
  constexpr int per = kDrawChunk / kWaves;
  const int s0 = min(c * kDrawChunk + w * per, n), s1 = min(s0 + per, n);
  sum_pieces(p, a.V, s0, s1, a.sums + (size_t)row * n + s0);
}

template <typename TIn>
__global__ __launch_bounds__(kWave) void k_draw_pick(DrawArgs a) {
  const int row = blockIdx.x, n = (a.V - 1) / kPiece + 1;
  const TIn* p = reinterpret_cast<const TIn*>(a.p) + (int64_t)row * a.ld;
  const double* sums = a.sums + (size_t)row * n;
  const int id = pick_token(p, a.V, a.uniforms[row], [&](int i) { return i < n ? sums[i] : 0.0; }, n);
  if (lane() == 0) a.out_ids[row] = id;
}

}  // namespace

// Two launches where one workgroup per row leaves most of the chip idle and
// the row is long enough to pay for the second launch: measured (float64, one
// launch / two) 64 rows x 32 000 6.4 / 6.7 us, 8 x 50 257 8.0 / 6.8, 64 x 50 257
// 8.3 / 8.0, 16 x 152 064 16.5 / 8.5, 64 x 152 064 19.2 / 18.3, 128 x 152 064
// 28.5 / 28.6; float32 alike.  And for rows whose sums do not fit in LDS.
size_t draw_ws_bytes(int B, int V, int num_cu) {
  const size_t n = (size_t)(V - 1) / kPiece + 1;
  const bool two = (V > 40000 && 4 * (int64_t)B <= num_cu) || n > kMaxPieces;
  return two ? (size_t)B * n * sizeof(double) : 0;
}

template <typename TIn>
void launch_draw_t(const DrawArgs& a, hipStream_t s) {
  if (a.sums == nullptr) {
    hipLaunchKernelGGL(k_draw_row<TIn>, dim3(a.B), dim3(kThreads), 0, s, a);
    return;
  }
  const int n = (a.V - 1) / kPiece + 1, C = (n + kDrawChunk - 1) / kDrawChunk;
  hipLaunchKernelGGL(k_draw_parts<TIn>, dim3((unsigned)((size_t)a.B * C)), dim3(kThreads), 0, s, a);
  hipLaunchKernelGGL(k_draw_pick<TIn>, dim3(a.B), dim3(kWave), 0, s, a);
}

hipError_t launch_draw(const DrawArgs& a, bool f64, hipStream_t s) {
  if (f64) launch_draw_t<double>(a, s);
  else launch_draw_t<float>(a, s);
  return hipGetLastError();
}

}  // namespace plh
