// gfx950 kernels for the logits producer: the model's final RMSNorm and
// lm_head product, logits = rms_norm(h, norm, eps) @ lm_head
// (src/pagellm/model/transformer.py:79-82, :271), in float32 as the
// reference computes it, written straight into the sampler's logits buffer.
//
// Two launches, or three: a prep kernel (one workgroup per row: RMSNorm with
// numpy's float32 steps, and act = (h * r) * norm in the layout the product
// reads), the product, and where k is cut into slices their sum:
//
//   k_head_skinny   at most 32 rows, or sums of a few products: one read of W,
//                   fp32 matrix cores
//   k_head_split    more rows: float32 products on the bf16 matrix cores,
//                   each operand split exactly into three bf16 parts
//   k_head_sum      the slices' partial sums
//
// The order of a sum depends on N, D, V, ldw and the number of CUs (head_plan),
// not on the data: equal calls give equal bits, but a row's last bits may change
// with the number of rows beside it.
#include "plh_device.h"
#include "plh_kernels.h"

#include <algorithm>
#include <cmath>

namespace plh {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// r = 1 / sqrt(mean(x * x) + eps) of a row of h, the same bits in every thread
// of the workgroup.
__device__ __forceinline__ float row_rinv(const HeadArgs& a, const float* x) {
  __shared__ double red[kWaves];
  double s = 0.0;
  for (int d = threadIdx.x; d < a.D; d += kThreads) {
    const float v = x[d];
    s += (double)(v * v);  // the float32 square, as numpy forms x * x
  }
  s = block_sum(s, red);
  // np.mean in float32, + eps as a float32 (a Python float is a weak
  // scalar), float32 sqrt and reciprocal (transformer.py:81)
  return 1.0f / sqrtf((float)s / (float)a.D + a.eps);
}

// Where a product kernel's sums go: out, or with several slices of k
// (gridDim.z) the slice's own [N, V] partial sums, which k_head_sum adds up.
struct HeadOut {
  float* p;
  size_t ld;
};

__device__ __forceinline__ HeadOut head_out(const HeadArgs& a) {
  if (gridDim.z == 1) return HeadOut{a.out, (size_t)a.ldo};
  return HeadOut{a.part + (size_t)blockIdx.z * a.N * a.V, (size_t)a.V};
}

// ------------------------------------------------------------- few rows
//
// Up to 32 rows (a decode step of a few sequences) the product is bound by
// one read of W from HBM, and a 256-row tile spends its time multiplying
// padding.  These rows take two launches of their own: k_head_prep (RMSNorm
// and the operand layout, one workgroup per row) and k_head_skinny.
//
// k_head_skinny<R>: R = 16 or 32 rows x 128 columns per workgroup on
// v_mfma_f32_16x16x4 / 32x32x2_f32.  The 8 waves share the columns and split
// k, so that a workgroup has 8 independent streams of W in flight; W goes
// from HBM straight into the MFMA operand registers (a lane's 16-byte load is
// one k row's value for each of four column tiles whose columns interleave by
// 4), with no LDS on the way, and the waves' sums meet in LDS once at the
// end, in a fixed order.  A lane's columns 4c .. 4c+3 are the same lane's of
// four accumulators, so the logits leave in 16-byte stores.
//
// 8 x 4096 x 128 256: 370 us, W read at 5.7 TB/s (a large copy moves 5.2 TB/s
// here); 2 000 us in the 256-row tile.

// k values per operand group: one 16-byte load of act per lane
template <int R>
struct Skinny {
  static constexpr int kQ = 64 / R;          // k values side by side in one MFMA
  static constexpr int kG = 4 * kQ;          // k values per group (4 MFMA steps)
  static constexpr int kCG = 128 / (4 * R);  // column groups of 4 R columns
};
constexpr int kSkinnyCols = 128;

__host__ __device__ constexpr int skinny_rows(int N) { return N <= 16 ? 16 : 32; }
__host__ __device__ constexpr int skinny_groups(int D, int R) { return (D + 256 / R - 1) / (256 / R); }

// act for k_head_skinny: group g holds k = g*kG .. +kG; lane (q, row) of an
// MFMA step t reads k = g*kG + kQ*t + q, so its four steps are 16 bytes at
// ((g*kQ + q)*R + row)*4.  Zero outside d < D; rows N .. R-1 are not written
// (an accumulator row depends on its own act row only, and those rows of the
// accumulators are never stored).
template <int R>
__global__ __launch_bounds__(kThreads) void k_head_prep(HeadArgs a) {
  using S = Skinny<R>;
  const int n = blockIdx.x, D = a.D;
  const float* x = a.h + (size_t)n * a.ldh;
  const float r = row_rinv(a, x);
  const int groups = skinny_groups(D, R);
  float* o = static_cast<float*>(a.act) + (size_t)(n / R) * groups * S::kG * R;
  for (int d = threadIdx.x; d < groups * S::kG; d += kThreads) {
    const int g = d / S::kG, e = d % S::kG;
    o[((size_t)(g * S::kQ + e % S::kQ) * R + n % R) * 4 + e / S::kQ] = d < D ? (x[d] * r) * a.norm[d] : 0.0f;
  }
}

typedef float f32x4u __attribute__((ext_vector_type(4))) __attribute__((aligned(4)));

template <int R>
struct SkinnyAcc;
template <>
struct SkinnyAcc<16> {
  typedef f32x4 T;
  static __device__ __forceinline__ T mma(float x, float y, T c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
  }
  // accumulator register r of lane l holds this row
  static __device__ __forceinline__ int row(int r, int l) { return 4 * (l >> 4) + r; }
};
template <>
struct SkinnyAcc<32> {
  typedef f32x16 T;
  static __device__ __forceinline__ T mma(float x, float y, T c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int r, int l) { return 8 * (r >> 2) + 4 * (l >> 5) + (r & 3); }
};

// ANY: V < 128, or rows of W more than 64 MB apart: columns are read one by
// one and clamped.  Otherwise the last workgroup's columns are the last 128,
// so every 16-byte load lies inside its row (columns of two workgroups are
// computed alike by both), and the loads are buffer loads whose row offsets
// are scalars.
template <int R, bool ANY>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_head_skinny(HeadArgs a) {
  using S = Skinny<R>;
  using A = SkinnyAcc<R>;
  constexpr int kRegs = R * R / 64;
  // half of the waves' accumulators at a time
  __shared__ f32x4 sm[kWaves / 2][S::kCG * kRegs][64];
  const int D = a.D, V = a.V, l = lane(), w = uniform(wave());
  // the row tiles of one column tile side by side (more than one: rows of W far
  // apart, or short sums)
  const int rt = (a.N + R - 1) / R, tile = (int)(blockIdx.x % (unsigned)rt);
  const int vx = (int)(blockIdx.x / (unsigned)rt) * kSkinnyCols, v0 = ANY ? vx : min(vx, V - kSkinnyCols);
  const int c = l % R, q = l / R;
  const int n0 = tile * R;
  const float* act =
      static_cast<const float*>(a.act) + (size_t)tile * skinny_groups(D, R) * S::kG * R + (size_t)(q * R + c) * 4;

  typename A::T acc[S::kCG][4];
#pragma unroll
  for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < kRegs; ++r) acc[cg][j][r] = 0.0f;

  struct Regs {
    f32x4 x;
    f32x4 y[4][S::kCG];
  };
  auto mma = [&](const Regs& o) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[cg][j] = A::mma(o.x[t], o.y[t][cg][j], acc[cg][j]);
  };
  // a group whose columns or k may lie outside the matrix: rows of W past D
  // read as 0
  auto load_any = [&](int g, Regs& o) {
    o.x = *reinterpret_cast<const f32x4*>(act + (size_t)g * S::kG * R);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int k = g * S::kG + S::kQ * t + q;
      const float* p = a.w + (size_t)min(k, D - 1) * a.ldw;
#pragma unroll
      for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = p[min(v0 + 4 * c + 4 * R * cg + e, V - 1)];
          o.y[t][cg][e] = k < D ? y : 0.0f;
        }
    }
  };

  // groups whose k all lie inside D; with several slices of k (blockIdx.z)
  // wave w of slice z takes w + 8 z, w + 8 (z + slices), ...
  const int full = D / S::kG, step = kWaves * (int)gridDim.z, g0 = w + kWaves * (int)blockIdx.z;
  if constexpr (ANY) {
    for (int g = g0; g * S::kG < D; g += step) {
      Regs o;
      load_any(g, o);
      mma(o);
    }
  } else {
    if (full * S::kG < D && g0 == full % step) {
      Regs o;
      load_any(full, o);
      mma(o);
    }
    const int voff = (int)(q * a.ldw + 4 * c) * 4, row = (int)(S::kQ * a.ldw) * 4;
    auto load = [&](int g, Regs& o) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(a.w + (size_t)g * S::kG * a.ldw + v0), (short)0, 0x7fffffff, 0x00020000);
      o.x = *reinterpret_cast<const f32x4*>(act + (size_t)g * S::kG * R);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int cg = 0; cg < S::kCG; ++cg)
          o.y[t][cg] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff + 16 * R * cg, row * t, 0));
    };
    // the next group's loads are in flight while this one is multiplied
    Regs r0, r1;
    if (g0 < full) load(g0, r0);
    for (int g = g0; g < full; g += 2 * step) {
      if (g + step < full) load(g + step, r1);
      __builtin_amdgcn_sched_barrier(0);
      mma(r0);
      __builtin_amdgcn_sched_barrier(0);
      if (g + step < full) {
        if (g + 2 * step < full) load(g + 2 * step, r0);
        __builtin_amdgcn_sched_barrier(0);
        mma(r1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // the waves' sums, in the order ((0+4)+(2+6)) + ((1+5)+(3+7)); each lane's
  // four column tiles travel as one 16-byte value
#pragma unroll
  for (int half = kWaves / 2; half >= 1; half >>= 1) {
    if (w >= half && w < 2 * half) {
#pragma unroll
      for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
        for (int r = 0; r < kRegs; ++r)
          sm[w - half][cg * kRegs + r][l] = f32x4{acc[cg][0][r], acc[cg][1][r], acc[cg][2][r], acc[cg][3][r]};
    }
    wg_barrier();
    if (w < half) {
#pragma unroll
      for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
          const f32x4 o = sm[w][cg * kRegs + r][l];
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[cg][j][r] += o[j];
        }
    }
    wg_barrier();
  }
  if (w != 0) return;
  const HeadOut to = head_out(a);
#pragma unroll
  for (int cg = 0; cg < S::kCG; ++cg)
#pragma unroll
    for (int r = 0; r < kRegs; ++r) {
      const int n = n0 + A::row(r, l);
      const int v = v0 + 4 * c + 4 * R * cg;
      if (n >= a.N) continue;
      float* o = to.p + (size_t)n * to.ld + v;
      const f32x4 y{acc[cg][0][r], acc[cg][1][r], acc[cg][2][r], acc[cg][3][r]};
      if constexpr (ANY) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (v + j < V) o[j] = y[j];
      } else {
        *reinterpret_cast<f32x4u*>(o) = y;
      }
    }
}

// ------------------------------------------------------------ many rows
//
// float32 products on the bf16 matrix cores.  A float32 x is exactly
// hi + mid + lo, three bf16 values (both operands are first scaled by 2^47, so
// that the parts of the smallest float32, 2^-149, are normal bf16 numbers), so
//   a * w = ah*wh + (ah*wm + am*wh) + (ah*wl + am*wm + al*wh) + rest,
// each product exact and summed in float32 by v_mfma_f32_32x32x16_bf16.  With
// parts rounded to nearest |rest| <= 1.01 * 2^-24 of the operands' powers of two
// (am*wl and al*wm, 2^-8 * 2^-17 each), of either sign: half the last bit of a
// float32 product.  (Truncated parts are 2^-7 and 2^-15 and all of x's sign: rest
// was up to 2^-21 and one-sided, and sums of like signs dropped their low
// products on the way, 1.2e-5 of the sum at D = 4096.)  Six bf16 products cost
// 6/16 of one on the fp32 matrix cores (2.5 PFLOP/s against 157 TFLOP/s), and a
// sum over k is rounded 6 times per 16 k instead of 8.  2-norm error against
// float64 in units of 2^-24, the fp32 matrix product / here (one slice):
//   D                          1     2     4     8    64   256   1000   4096
//   N(0,1) x 0.02 N(0,1)    0.42  0.56  0.65  0.84  2.35  4.77   9.55  19.2
//                           0.61  0.58  0.54  0.52  1.77  3.94   8.16  16.8
//   U(1,2) x U(1,2)         0.45  0.51  0.60  0.75  2.03  3.88   7.79  15.9
//                           0.60  0.48  0.48  0.50  1.41  2.89   5.30   9.9
// and less with several slices of k.  Sums of fewer than kSplitMinD products take
// the fp32 kernel.
//
// k_head_split<BM>: a BM-row x 256-column tile per workgroup, 8 waves of 64
// rows x (BM / 2) columns (at least 32), k in stages of 16.  act comes split
// from the prep kernel.  A thread holds one column's 8 k values of W (read
// coalesced over the lanes, so rows of any alignment are read alike), splits
// them and stores the three parts for the whole workgroup in LDS,
// double-buffered; LDS is read and written 16 bytes a lane, consecutive lanes
// consecutive pieces.  Both operands' loads run kPF stages ahead in registers.
// They are issued together: loads return in order, and an operand loaded one
// stage ahead on its own made every stage wait for the other's newest loads
// (4096 x 128 256: 64 rows 690 us, 256 rows 1 420 us).  The stage loop has no
// branch and no predicated load for the same reason: at a join the loads'
// registers were copied, which waits for them.  Nor does it lean on a range
// check, which covers the lanes' offsets of a buffer load but not its scalar
// offset: every address is clamped into W (a last row or column read twice
// instead), and act is 0 for k >= D, up to whole units of 4 stages.  (A
// descriptor per row of W, exact in its range, costs 40 scalar instructions
// a stage: 4096 x 128 256, 256 rows 1 240 -> 1 320 us, 64 rows 460 -> 520 us.)
// What the parts cannot carry leaves no finite sum (infinities, operands of
// 2^81 on, sums that reach 2^34 on the way); those 32 x 32 tiles are formed again
// on the fp32 matrix cores, from the rows in float32.  Not for a row of act that
// holds a NaN: its sums are NaN already, and one broken request in a batch would
// have every column tile formed again (256 x 4096 x 128 256: 3 010 us against
// 1 220).  What is left of that is broken weights: an infinite lm_head value 1 450 us,
// an infinite norm value 5 100 us.
//
// Against the fp32 matrix product in 256-row tiles, 4096 x 128 256: 256 rows
// 2 010 -> 1 220-1 270 us (1.27-1.33 PFLOP/s of bf16 products, the rate of a large
// bf16 matrix product here), 128 rows 2 005 -> 735-770 us, 64 rows 2 000 -> 470-485
// us, bound by W's way through a CU; 45 x 1000 x 50 257: 290 -> 55-57 us.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplitCols = 256;  // columns per workgroup
constexpr int kSplitK = 16;      // k per stage: one MFMA step
constexpr int kSplitMaxLdw = 1 << 24;  // a thread's eight rows of W lie within 2^29 bytes
constexpr int kSplitMinD = 4;    // products a sum has at least
constexpr int kRedoK = 32;       // k per step of the float32 product
constexpr float kSplitScale = 0x1p47f, kSplitUnscale = 0x1p-94f;

__host__ __device__ constexpr int split_stages(int D) { return (D + kSplitK - 1) / kSplitK; }
// k groups of act: whole units of the 4 stages that a thread holds at most
__host__ __device__ constexpr int split_groups(int D) { return (split_stages(D) + 3) / 4 * 8; }

struct Split8 {
  u32x4 part[3];  // hi, mid, lo: 8 bf16 each
};

// 2^47 x = hi + mid + lo, each the bf16 nearest to what is left: each remainder
// is exact, and the last a bf16 itself (|mid| <= 2^-8 and |lo| <= 2^-17 of the
// power of two below x, both signs).
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x2 r{x[2 * i] * kSplitScale, x[2 * i + 1] * kSplitScale};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
      s.part[p][i] = u;
      if (p < 2) {
        r[0] -= __uint_as_float(u << 16);
        r[1] -= __uint_as_float(u & 0xffff0000u);
      }
    }
  }
  return s;
}

// act for k_head_split: part p, k group kg (8 k), row n at
// ((p * groups + kg) * lda + n) * 8; zero for k >= D and for the rows N .. lda-1
// that fill the last tile.  Also each row in float32 (act32, zero for k >= D), and
// whether it holds a NaN (the rows past N count as such).
__global__ __launch_bounds__(kThreads) void k_head_prep_split(HeadArgs a) {
  const int n = blockIdx.x, D = a.D;
  const int groups = split_groups(D);
  u32x4* o = static_cast<u32x4*>(a.act);
  if (n >= a.N) {
    for (int i = threadIdx.x; i < 3 * groups; i += kThreads) o[(size_t)i * a.lda + n] = u32x4{0u, 0u, 0u, 0u};
    if (threadIdx.x == 0) a.nan_rows[n] = 1;
    return;
  }
  const float* x = a.h + (size_t)n * a.ldh;
  const float r = row_rinv(a, x);
  __shared__ int red[kWaves];
  int nan = 0;
  for (int kg = threadIdx.x; kg < groups; kg += kThreads) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int d = 8 * kg + e;
      v[e] = d < D ? (x[d] * r) * a.norm[d] : 0.0f;
      nan |= v[e] != v[e];
    }
    f32x4* row = reinterpret_cast<f32x4*>(a.act32 + ((size_t)n * groups + kg) * 8);
    row[0] = f32x4{v[0], v[1], v[2], v[3]};
    row[1] = f32x4{v[4], v[5], v[6], v[7]};
    const Split8 s = split8(v);
#pragma unroll
    for (int p = 0; p < 3; ++p) o[((size_t)p * groups + kg) * a.lda + n] = s.part[p];
  }
  nan = block_max(nan, red);
  if (threadIdx.x == 0) a.nan_rows[n] = nan;
}

__device__ __forceinline__ bool not_finite(float x) { return !(fabsf(x) <= 3.4028234663852886e38f); }

// One 32 x 32 tile of out, rows n.. and columns v.., on the fp32 matrix cores:
// half-wave h takes k 4h .. 4h+3 of every eight.
__device__ __forceinline__ f32x16 head_tile_f32(const HeadArgs& a, int n, int v) {
  constexpr int kStep = kRedoK / 8;
  const int l = lane(), D = a.D, half = 4 * (l >> 5);
  const int row = min(n + (l & 31), a.N - 1), col = min(v + (l & 31), a.V - 1);
  const float* x = a.act32 + (size_t)row * split_groups(D) * 8 + half;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  for (int kb = 0; kb < D; kb += kRedoK, x += kRedoK) {
    const int k0 = kb + half;
    f32x4 xs[kStep];
    float ys[kStep][4];
#pragma unroll
    for (int i = 0; i < kStep; ++i) {
      xs[i] = *reinterpret_cast<const f32x4*>(x + 8 * i);
#pragma unroll
      for (int t = 0; t < 4; ++t) ys[i][t] = a.w[(size_t)min(k0 + 8 * i + t, D - 1) * a.ldw + col];
    }
#pragma unroll
    for (int i = 0; i < kStep; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xs[i][t], k0 + 8 * i + t < D ? ys[i][t] : 0.0f, acc, 0, 0, 0);
  }
  return acc;
}

template <int BM>
struct SplitGeo {
  static constexpr int kWR = BM / 64;                         // waves along the rows
  static constexpr int kNT = kSplitCols / 32 * kWR / kWaves;  // 32-column tiles per wave
  static constexpr int kA = (6 * BM + kThreads - 1) / kThreads;  // 16-byte pieces of act per thread and stage
  static constexpr int kPF = BM <= 128 ? 4 : 2;               // stages in registers
  static constexpr int kEu = BM == 64 ? 4 : 2;                // waves per SIMD
};

template <int BM>
struct SplitSmem {
  u32x4 a[2][SplitGeo<BM>::kA * kThreads];  // [buffer][(part * 2 + k group) * BM + row], and a thread's unused pieces
  u32x4 b[2][3][2][kSplitCols];    // [buffer][part][k group][column]
};

template <int BM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(SplitGeo<BM>::kEu, SplitGeo<BM>::kEu))) void
k_head_split(HeadArgs a) {
  using G = SplitGeo<BM>;
  constexpr int kNT = G::kNT, kPF = G::kPF;
  __shared__ SplitSmem<BM> sm;
  const int D = a.D, V = a.V, l = lane(), w = uniform(wave());
  // the row tiles of one column tile run side by side, so that all but the
  // first find W in the caches
  const int rt = (int)a.lda / BM;
  const int v0 = (int)(blockIdx.x / rt) * kSplitCols, n0 = (int)(blockIdx.x % rt) * BM;
  const int wr = w % G::kWR, wc = w / G::kWR;
  // this slice's stages, a multiple of kPF
  const int groups = split_groups(D), units = (split_stages(D) + kPF - 1) / kPF;
  const int sb = (int)((int64_t)units * blockIdx.z / gridDim.z) * kPF;
  const int se = (int)((int64_t)units * (blockIdx.z + 1) / gridDim.z) * kPF;

  // W: this thread's column and k group (uniform over the wave); act: 16-byte
  // pieces tid, tid + 512, ... of the stage's 6 BM
  const int col = (int)threadIdx.x & (kSplitCols - 1), kg = w >> 2;
  const int pitch = (int)a.ldw * 4, voff = min(col, V - 1 - v0) * 4;
  float wreg[kPF][8];
  u32x4 areg[kPF][G::kA];
  auto load = [&](int s, float (&o)[8], u32x4 (&x)[G::kA]) {
    const int k0 = min(s * kSplitK + kg * 8, D - 1), last = min(D - 1 - k0, 7) * pitch;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.w + (size_t)k0 * a.ldw + v0), (short)0, 0x7fffffff, 0x00020000);
    const u32x4* ap = static_cast<const u32x4*>(a.act) + (size_t)min(2 * s, groups - 2) * a.lda + n0;
#pragma unroll
    for (int i = 0; i < G::kA; ++i) {
      const int q = min((int)threadIdx.x + kThreads * i, 6 * BM - 1);
      x[i] = ap[((size_t)(q / (2 * BM)) * groups + (q / BM) % 2) * a.lda + q % BM];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, voff, min(j * pitch, last), 0));
  };
  auto store = [&](int buf, const float (&o)[8], const u32x4 (&x)[G::kA]) {
    const Split8 s = split8(o);
#pragma unroll
    for (int p = 0; p < 3; ++p) sm.b[buf][p][kg][col] = s.part[p];
#pragma unroll
    for (int i = 0; i < G::kA; ++i) sm.a[buf][(int)threadIdx.x + kThreads * i] = x[i];
  };

  f32x16 acc[2][kNT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

#pragma unroll
  for (int i = 0; i < kPF; ++i) load(sb + i, wreg[i], areg[i]);
  store(0, wreg[0], areg[0]);
  wg_barrier();
  // lane l of an operand holds row (column) l % 32 and k group l / 32
  const int c0 = wc * 32 * kNT + (l & 31), r0 = (l >> 5) * BM + wr * 64 + (l & 31);
  for (int s0 = sb; s0 < se; s0 += kPF) {
#pragma unroll
    for (int i = 0; i < kPF; ++i) {
      const int buf = i & 1;  // kPF is even
      load(s0 + i + kPF, wreg[i], areg[i]);  // these registers went to LDS one stage ago
      u32x4 fa[2][3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) fa[mt][p] = sm.a[buf][2 * BM * p + r0 + 32 * mt];
      // small products first
      constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        u32x4 fb[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) fb[p] = sm.b[buf][p][l >> 5][c0 + 32 * nt];
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[mt][pa[t]]),
                                                                  __builtin_bit_cast(bf16x8, fb[pb[t]]), acc[mt][nt],
                                                                  0, 0, 0);
      }
      store(buf ^ 1, wreg[(i + 1) % kPF], areg[(i + 1) % kPF]);
      // the split's 60 vector instructions among the products, not behind them
      // (64 rows x 4096 x 128 256: 505 -> 483 us, 45 x 1000 x 50 257: 64 -> 57 us)
#pragma unroll
      for (int q = 0; q < 12 * kNT; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                             // an MFMA ...
        __builtin_amdgcn_sched_group_barrier(0x002, (60 + 12 * kNT) / (12 * kNT), 0);  // ... and its share
      }
      wg_barrier();
    }
  }

  // accumulator r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32
  const int nb = n0 + wr * 64 + 4 * (l >> 5), vb = v0 + c0;
  auto row_of = [&](int mt, int r) { return nb + 32 * mt + 8 * (r >> 2) + (r & 3); };
  const HeadOut to = head_out(a);
  const float scale = gridDim.z == 1 ? kSplitUnscale : 1.0f;  // slices: where they are added up
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = row_of(mt, r), v = vb + 32 * nt;
        if (n < a.N && v < V) to.p[(size_t)n * to.ld + v] = acc[mt][nt][r] * scale;
      }
  if (gridDim.z > 1) return;
  uint32_t redo = 0;  // bit 2 nt + mt: that tile of this wave
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      bool bad = false;
#pragma unroll
      for (int r = 0; r < 16; ++r) bad |= not_finite(acc[mt][nt][r]);
      if (__ballot(bad) == 0) continue;
      uint32_t left = 0;  // bit r: not finite, and its row holds no NaN
#pragma unroll
      for (int r = 0; r < 16; ++r) left |= not_finite(acc[mt][nt][r]) ? 1u << r : 0u;
      for (int r = 0; r < 16; ++r) left &= ~((uint32_t)a.nan_rows[row_of(mt, r)] << r);
      if (__ballot(left != 0) != 0) redo |= 1u << (2 * nt + mt);
    }
  for (; redo != 0; redo &= redo - 1) {
    const int mt = __builtin_ctz(redo) & 1, nt = __builtin_ctz(redo) >> 1, v = vb + 32 * nt;
    const f32x16 y = head_tile_f32(a, n0 + wr * 64 + 32 * mt, v0 + wc * 32 * kNT + 32 * nt);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (row_of(mt, r) < a.N && v < V) to.p[(size_t)row_of(mt, r) * to.ld + v] = y[r];
  }
}

// ------------------------------------------------------------ slices of k
//
// out = the slices' partial sums added in order.  SPLIT: they are scaled, and an
// element that the bf16 parts cannot carry is formed again in float32.
template <bool SPLIT>
__global__ __launch_bounds__(256) void k_head_sum(HeadArgs a, int slices) {
  const int v = blockIdx.x * 256 + threadIdx.x, n = blockIdx.y;
  if (v >= a.V) return;
  const float* p = a.part + (size_t)n * a.V + v;
  const size_t pitch = (size_t)a.N * a.V;
  float s = 0.0f;
#pragma unroll 8
  for (int z = 0; z < slices; ++z) s += p[z * pitch];
  if constexpr (SPLIT) {
    if (not_finite(s) && a.nan_rows[n] != 0) {
      s = NAN;
    } else if (not_finite(s)) {
      const float* x = a.act32 + (size_t)n * split_groups(a.D) * 8;
      s = 0.0f;
#pragma unroll 8
      for (int k = 0; k < a.D; ++k) s = fmaf(x[k], a.w[(size_t)k * a.ldw + v], s);
    } else {
      s *= kSplitUnscale;
    }
  }
  a.out[(size_t)n * a.ldo + v] = s;
}

// ---------------------------------------------------------------- launch

struct HeadPlan {
  int rows;    // rows per workgroup: 16, 32 (k_head_skinny), 64, 128, 256 (k_head_split)
  int slices;  // slices of k, each a workgroup of its own
};

// Microseconds a plan takes, to choose between plans: rounds of workgroups
// times k steps times one step, but at least the read of W, plus the partial
// sums' way through the caches.  The steps were measured at N 8 to 256 over
// 4096 x 1000 (4 to 16 workgroups: a step's latency) and 4096 x 128 256 (every
// CU at work: its throughput).
double plan_us(const HeadPlan& p, int N, int D, int V, int num_cu) {
  const double w_bytes = 4.0 * D * V, rows = (N + p.rows - 1) / p.rows;
  double us;
  if (p.rows <= 32) {
    const int kg = 256 / p.rows;  // k per group
    const double steps = std::ceil((double)((D + kg - 1) / kg) / (kWaves * p.slices));
    const double wgs = (double)((V + kSkinnyCols - 1) / kSkinnyCols) * rows * p.slices;
    us = std::ceil(wgs / (2.0 * num_cu)) * steps * 1.1;  // two workgroups per CU
    us = std::max(us, w_bytes / 5.4e6);
  } else {
    const int unit = p.rows == 256 ? 2 : 4;  // a slice is whole units of stages
    const double steps = unit * std::ceil((double)((split_stages(D) + unit - 1) / unit) / p.slices);
    const double wgs = (double)((V + kSplitCols - 1) / kSplitCols) * rows * p.slices;
    if (p.rows == 64)  // one workgroup on a CU, or rounds of two
      us = steps * (wgs <= num_cu ? 0.7 : 1.55 * std::ceil(wgs / (2.0 * num_cu)));
    else
      us = steps * (p.rows == 128 ? 1.4 : 2.3) * std::ceil(wgs / num_cu);
    us = std::max(us, w_bytes / 4.4e6);
  }
  return p.slices > 1 ? us + 3.0 + 8.0 * p.slices * N * V / 5e6 : us;
}

// Rows per workgroup and slices of k.  Up to 32 rows the product is bound by
// the read of W, not by the matrix cores (at 157 TFLOP/s 32 rows take half of
// W's time in HBM), and k_head_skinny reads W at the rate of a copy; 33 rows
// on would read it twice there (4096 x 128 256: 720 us for 17 rows in two tiles
// of 16, 410 us in one of 32).  Sums of fewer than kSplitMinD products go there for
// their precision (the table at k_head_split).  Slices fill the chip where the columns alone
// do not (4096 x 1000, 8 rows: 44 us in one slice, 15 us in 16).
HeadPlan head_plan(int N, int D, int V, int64_t ldw, int num_cu) {
  const bool skinny = N <= 32 || D < kSplitMinD || ldw > kSplitMaxLdw;
  const int lo = skinny ? (N <= 16 ? 16 : 32) : 64, hi = skinny ? lo : 256;
  HeadPlan best{lo, 1};
  double best_us = plan_us(best, N, D, V, num_cu);
  for (int rows = lo; rows <= hi; rows *= 2)
    for (int slices = 1; slices <= (N <= 4096 ? 32 : 1); slices *= 2) {  // k_head_sum's grid holds N in y
      const HeadPlan p{rows, slices};
      const double us = plan_us(p, N, D, V, num_cu);
      if (us < best_us) {
        best = p;
        best_us = us;
      }
    }
  return best;
}

// The workspace: act in the product's layout; for k_head_split also in float32,
// and the rows that hold a NaN; the partial sums.  Offsets in bytes.
struct HeadWs {
  size_t act32, nan_rows, part, bytes;
};

HeadWs head_ws(const HeadPlan& p, int N, int D, int V) {
  const size_t rows = ((size_t)N + p.rows - 1) / p.rows * p.rows, K = (size_t)split_groups(D) * 8;
  const bool split = p.rows > 32;
  size_t at = K * rows * (split ? 6 : 4);
  auto take = [&](size_t bytes) {
    const size_t o = (at + 255) / 256 * 256;
    at = o + bytes;
    return o;
  };
  HeadWs w{};
  w.act32 = take(split ? K * N * sizeof(float) : 0);
  w.nan_rows = take(split ? rows * sizeof(int) : 0);
  w.part = take(p.slices > 1 ? (size_t)p.slices * N * V * sizeof(float) : 0);
  w.bytes = at;
  return w;
}

size_t head_ws_bytes(int N, int D, int V, int64_t ldw, int num_cu) {
  return head_ws(head_plan(N, D, V, ldw, num_cu), N, D, V).bytes;
}

template <int R>
void launch_skinny(const HeadArgs& a, int slices, hipStream_t s) {
  hipLaunchKernelGGL(k_head_prep<R>, dim3(a.N), dim3(kThreads), 0, s, a);
  const dim3 grid((unsigned)((a.V + kSkinnyCols - 1) / kSkinnyCols) * (unsigned)((a.N + R - 1) / R), 1, (unsigned)slices);
  if (a.V < kSkinnyCols || a.ldw > kSplitMaxLdw) hipLaunchKernelGGL((k_head_skinny<R, true>), grid, dim3(kThreads), 0, s, a);
  else hipLaunchKernelGGL((k_head_skinny<R, false>), grid, dim3(kThreads), 0, s, a);
}

template <int BM>
void launch_split(HeadArgs a, int slices, hipStream_t s) {
  const unsigned rt = (unsigned)((a.N + BM - 1) / BM);
  a.lda = (int64_t)rt * BM;
  hipLaunchKernelGGL(k_head_prep_split, dim3((unsigned)a.lda), dim3(kThreads), 0, s, a);
  hipLaunchKernelGGL(k_head_split<BM>, dim3((unsigned)((a.V + kSplitCols - 1) / kSplitCols) * rt, 1, (unsigned)slices),
                     dim3(kThreads), 0, s, a);
}

hipError_t launch_head(HeadArgs a, int num_cu, hipStream_t s) {
  const HeadPlan p = head_plan(a.N, a.D, a.V, a.ldw, num_cu);
  const HeadWs ws = head_ws(p, a.N, a.D, a.V);
  char* base = static_cast<char*>(a.act);
  a.act32 = reinterpret_cast<float*>(base + ws.act32);
  a.nan_rows = reinterpret_cast<int*>(base + ws.nan_rows);
  a.part = reinterpret_cast<float*>(base + ws.part);
  a.lda = (int64_t)((a.N + p.rows - 1) / p.rows) * p.rows;
  switch (p.rows) {
    case 16: launch_skinny<16>(a, p.slices, s); break;
    case 32: launch_skinny<32>(a, p.slices, s); break;
    case 64: launch_split<64>(a, p.slices, s); break;
    case 128: launch_split<128>(a, p.slices, s); break;
    default: launch_split<256>(a, p.slices, s); break;
  }
  if (p.slices > 1) {
    const dim3 grid((unsigned)((a.V + 255) / 256), (unsigned)a.N);
    if (p.rows <= 32) hipLaunchKernelGGL(k_head_sum<false>, grid, dim3(256), 0, s, a, p.slices);
    else hipLaunchKernelGGL(k_head_sum<true>, grid, dim3(256), 0, s, a, p.slices);
  }
  return hipGetLastError();
}

}  // namespace plh
