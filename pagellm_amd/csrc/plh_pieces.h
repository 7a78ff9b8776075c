// Rows cut into pieces of 512 tokens for float64 inverse-CDF draws: a piece is
// whole 16-byte loads of a wave, its weights are summed in one fixed order, and
// a draw reads again only the piece where the running total crosses.
#pragma once

#include "plh_device.h"

namespace plh {

constexpr int kPiece = 512;  // tokens per piece

template <typename TIn>
struct PieceGeo {
  static constexpr int kVW = 16 / (int)sizeof(TIn);
  static constexpr int kLoads = kPiece / (kVW * kWave);  // 16-byte loads per lane and piece
  typedef TIn V __attribute__((ext_vector_type(kVW))) __attribute__((aligned(sizeof(TIn))));
};

// The calling lane's tokens of piece s: load j holds tokens
// s * 512 + (j * 64 + lane) * kVW onwards.  Tokens past the row read as 0.
template <typename TIn>
__device__ __forceinline__ void load_piece(const TIn* p, int V, int s,
                                           typename PieceGeo<TIn>::V (&x)[PieceGeo<TIn>::kLoads]) {
  using G = PieceGeo<TIn>;
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

// The total of n piece sums sum(0) .. sum(n-1) (sum(i) is 0 from n on), added
// in one fixed order; by one wave, every lane alike.
template <class Sum>
__device__ __forceinline__ double pieces_total(const Sum& sum, int n) {
  double run = 0.0;
  for (int base = 0; base < n; base += kWave)
    run = lane_value(run + wave_scan_incl(sum(base + lane()), 0.0, OpAdd{}), kWave - 1);
  return run;
}

// The first piece whose running total exceeds t (crossed), else the last one
// with mass (-1: none), and the total before it.
struct Crossing {
  int piece;
  bool crossed;
  double before;
};

template <class Sum>
__device__ __forceinline__ Crossing cross_pieces(const Sum& sum, int n, double t) {
  Crossing c{-1, false, 0.0};
  double run = 0.0;
  for (int base = 0; base < n && !c.crossed; base += kWave) {
    const double v = sum(base + lane());
    const double incl = run + wave_scan_incl(v, 0.0, OpAdd{});
    const uint64_t pos = __ballot(v > 0.0), over = __ballot(v > 0.0 && incl > t);
    if (pos != 0) {
      const int k = over != 0 ? __builtin_ctzll(over) : 63 - __builtin_clzll(pos);
      c = Crossing{base + k, over != 0, lane_value(incl - v, k)};
    }
    run = lane_value(incl, kWave - 1);
  }
  return c;
}

// The token of the crossing piece, whose weights are w (the lane's, as
// load_piece lays them out): the first whose running total exceeds t; where
// none does (rounding, or the piece was not crossed), its last of positive
// weight.  -1: no positive weight.
template <typename TIn>
__device__ __forceinline__ int pick_in_piece(const Crossing& c, double t,
                                             const double (&w)[PieceGeo<TIn>::kLoads][PieceGeo<TIn>::kVW]) {
  using G = PieceGeo<TIn>;
  int tok = -1, tail = -1;
  double before = c.before;
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j) {
    double ts = 0.0;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) ts += w[j][e];
    const double incl = wave_scan_incl(ts, 0.0, OpAdd{});
    double cum = before + (incl - ts);
    const int i0 = c.piece * kPiece + (j * kWave + lane()) * G::kVW;
    int hit = INT_MAX, pos = -1;
#pragma unroll
    for (int e = 0; e < G::kVW; ++e) {
      cum += w[j][e];
      if (w[j][e] > 0.0) {
        pos = i0 + e;
        if (hit == INT_MAX && cum > t) hit = i0 + e;
      }
    }
    tail = max(tail, wave_max(pos));
    const int h = wave_min(hit);
    if (c.crossed && tok < 0 && h != INT_MAX) tok = h;
    before += lane_value(incl, kWave - 1);
  }
  return tok >= 0 ? tok : tail;
}

}  // namespace plh
