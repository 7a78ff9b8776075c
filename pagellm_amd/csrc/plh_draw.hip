// gfx950 kernels for draw() (src/pagellm/engine/sampling.py:94-98): the
// inverse-CDF draw from rows of non-negative weights.
//
// A row is cut into pieces of 512 tokens.  One pass over the row sums each
// piece (a wave's piece is whole 16-byte loads of consecutive tokens); the
// running piece totals give the total W and the first piece whose total exceeds
// u * W, and only that piece is read again for the token.  float32 rows are
// widened exactly.
//
// Masses are added in fixed point, in units of 2^-62 of the power of two above
// W (a scaling, exact, where a division by W rounds), so a total does not depend
// on the order of its sum, and u times the total is exact; a piece's own mass is
// summed in float64 first, but in a row of at most 8 pieces, which a wave each
// keeps in registers.  How far a boundary between tokens lies from its exact
// place (rms, in W; logits N(0, 2); masses divided by W in units of 2^-62 and a
// rounded u * W / float64 throughout / here): 512 tokens 3.9e-17 / 7.4e-17 /
// 1.1e-18, 4096 3.6e-17 / 7.6e-17 / 2.5e-18, 32 000 4.1e-17 / 7.1e-17 / 2.5e-17,
// 152 064 3.9e-17 / 7.5e-17 / 2.4e-17.
//
// The token differs from the reference's (numpy's float64 cumsum) only when u
// lies within ~1e-15 (relative) of a CDF boundary.  Where rounding leaves the
// crossing just past the piece's end, the piece's last token of positive weight is
// taken (a neighbour of the boundary either way).
//
// Bound by the read of the rows and, for a few dozen rows, by one workgroup's
// latency chain (a load round trip, the piece sums, the reread).
// 64 x 32 000 float64: 39.9 -> 6.3 us against three passes over the row with a
// float64 division per token; 512 x 152 064: 106 us, 5.9 TB/s.
#include "plh_device.h"
#include "plh_kernels.h"
#include "plh_pieces.h"

namespace plh {

namespace {

constexpr int kDrawChunk = 32;   // pieces per workgroup of k_draw_parts
constexpr int kMaxPieces = 2048;  // pieces whose sums k_draw_row holds (V <= 1 048 576)

__device__ __forceinline__ double weight_of(double v) { return v > 0.0 ? v : 0.0; }

template <typename TIn>
__device__ __forceinline__ double lane_sum(const typename PieceGeo<TIn>::V (&x)[PieceGeo<TIn>::kLoads]) {
  using G = PieceGeo<TIn>;
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
  typename PieceGeo<TIn>::V x[U][PieceGeo<TIn>::kLoads];
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
  typename PieceGeo<TIn>::V tail[PieceGeo<TIn>::kLoads];
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

// Whether a row of total mass W is drawn from: not without mass, or with more
// than a double holds, or for a u past the end: the last id (sampling.py:98
// clamps to V - 1).
__device__ __forceinline__ bool drawable(double W, double u) {
  return W > 0.0 && W <= 1.7976931348623157e308 && !(u >= 1.0);
}

// Fixed-point masses in units of 2^-62 of the power of two above W.
struct FxScale {
  int shift;
  __device__ __forceinline__ explicit FxScale(double W) : shift(62 - __builtin_amdgcn_frexp_exp(W)) {}
  __device__ __forceinline__ uint64_t operator()(double w) const { return __double2ull_rn(ldexp(w, shift)); }
};

// floor(u * tot) for u < 1 (0 for u <= 0 and NaN), exact: below tot.
__device__ __forceinline__ uint64_t fx_target(double u, uint64_t tot) {
  if (!(u > 0.0)) return 0;
  const uint64_t m = (uint64_t)ldexp(__builtin_amdgcn_frexp_mant(u), 53);  // u = m 2^-s
  const int s = 53 - __builtin_amdgcn_frexp_exp(u);                        // at least 53
  const uint64_t hi = __umul64hi(m, tot), lo = m * tot;
  if (s < 64) return (hi << (64 - s)) | (lo >> s);
  return s < 128 ? hi >> (s - 64) : 0;
}

// The first token of piece s whose running mass exceeds t, INT_MAX where none
// does; before: the running mass at the piece's start; x: the lane's tokens, as
// load_piece lays them out.  last: the piece's last token of positive weight.
template <typename TIn>
__device__ __forceinline__ int pick_fx(const typename PieceGeo<TIn>::V (&x)[PieceGeo<TIn>::kLoads], int s,
                                       const FxScale& fx, uint64_t before, uint64_t t, int* last) {
  using G = PieceGeo<TIn>;
  int hit = INT_MAX, pos = -1;
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j) {
    uint64_t w[G::kVW], ts = 0;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) ts += w[e] = fx(weight_of((double)x[j][e]));
    const uint64_t incl = wave_scan_incl(ts, (uint64_t)0, OpAdd{});
    uint64_t c = before + (incl - ts);
    const int i0 = s * kPiece + (j * kWave + lane()) * G::kVW;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) {
      c += w[e];
      if (hit == INT_MAX && c > t) hit = i0 + e;
      if (x[j][e] > TIn(0)) pos = i0 + e;
    }
    before += lane_value(incl, kWave - 1);
  }
  *last = wave_max(pos);
  return wave_min(hit);
}

// The drawn token of a row whose n piece sums are sum(i); by one wave, every
// lane alike.
template <typename TIn, class Sum>
__device__ __forceinline__ int pick_token(const TIn* p, int V, double u, const Sum& sum, int n) {
  using G = PieceGeo<TIn>;
  double W = 0.0;  // sets the scale only: any order will do
  for (int base = 0; base < n; base += kWave) W += sum(base + lane());
  W = wave_sum(W);
  if (!drawable(W, u)) return V - 1;
  const FxScale fx(W);
  uint64_t tot = 0;
  for (int base = 0; base < n; base += kWave) tot += fx(sum(base + lane()));
  tot = wave_sum(tot);
  const uint64_t t = fx_target(u, tot);
  uint64_t run = 0, before = 0;
  int piece = -1;
  for (int base = 0; base < n && piece < 0; base += kWave) {
    const uint64_t v = fx(sum(base + lane())), incl = run + wave_scan_incl(v, (uint64_t)0, OpAdd{});
    const uint64_t over = __ballot(incl > t);
    if (over != 0) {
      const int k = __builtin_ctzll(over);
      piece = base + k;
      before = lane_value(incl - v, k);
    }
    run = lane_value(incl, kWave - 1);
  }
  typename G::V x[G::kLoads];
  load_piece(p, V, piece, x);
  int last;
  const int hit = pick_fx<TIn>(x, piece, fx, before, t, &last);
  return hit != INT_MAX ? hit : last;
}

// The same for a row of at most kWaves pieces, one a wave, kept in registers;
// by the whole workgroup.
template <typename TIn>
__device__ __forceinline__ void draw_short_row(const TIn* p, int V, double u, int32_t* out) {
  using G = PieceGeo<TIn>;
  __shared__ double sums[kWaves];
  __shared__ uint64_t mass[kWaves];
  const int w = uniform(wave());
  typename G::V x[G::kLoads];
  load_piece(p, V, w, x);  // zeros past the row
  const double mine = wave_sum(lane_sum<TIn>(x));
  if (lane() == 0) sums[w] = mine;
  wg_barrier();
  double W = 0.0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) W += sums[i];
  if (!drawable(W, u)) {
    if (threadIdx.x == 0) *out = V - 1;
    return;
  }
  const FxScale fx(W);
  uint64_t m = 0;
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j)
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) m += fx(weight_of((double)x[j][e]));
  m = wave_sum(m);
  if (lane() == 0) mass[w] = m;
  wg_barrier();
  uint64_t before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    if (i == w) before = tot;
    tot += mass[i];
  }
  const uint64_t t = fx_target(u, tot);
  if (t < before || t - before >= m) return;  // uniform: one wave goes on
  int last;
  const int hit = pick_fx<TIn>(x, w, fx, before, t, &last);
  if (lane() == 0) *out = hit;
}

template <typename TIn>
__global__ __launch_bounds__(kThreads) void k_draw_row(DrawArgs a) {
  __shared__ double sums[kMaxPieces];
  const int row = blockIdx.x, n = (a.V - 1) / kPiece + 1, w = uniform(wave());
  const TIn* p = reinterpret_cast<const TIn*>(a.p) + (int64_t)row * a.ld;
  const double u = a.uniforms[row];
  if (n <= kWaves) {  // the kernel's rows are all of V tokens: uniform
    draw_short_row(p, a.V, u, a.out_ids + row);
    return;
  }
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
        typename PieceGeo<TIn>::V x[PieceGeo<TIn>::kLoads];
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
