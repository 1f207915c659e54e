// The chunked gated delta-rule scan at feature widths the D = 512 kernels do not cover (gfx950).
//
// Used for D = 1024 over pre-lifted features: the factored d_k = 128 path of the reference
// (kernels/factored_kernel_deltanet.py:42-183: two 64 -> 512 lifts concatenated and renormalised, then
// the same chunk algebra with 1024 features and d_v = 128).  The rule and readout are those of the
// D = 512 scan: y_t = S_{t-1} phi_q(t), S_t = lambda_t S_{t-1} (I - beta_t phi_k phi_k^T) + beta_t v_t phi_k^T.
//
// Three launches per call, with one fp32 record per (batch, head, 64-token chunk):
//   prep   (parallel)   Grams K K^T and Q K^T from the feature rows, A, T = (I + A)^-1 (column-oriented
//                       substitution), Tp = T diag(beta g), P, U~ = T (beta o V); K packed in MFMA fragment
//                       order (with fp32 features transposed too)
//   carry  (sequential) S^T at every chunk start; X_K = K S^T, W = U~ - Tp X_K,
//                       S^T <- g_C S^T + K^T (kappa o W); the final state
//   output (parallel)   Y = diag(a) Q S_c^T + P W
// Notation as the D = 512 scan: l_i = sum_{t <= i} log clamp(lambda_t, 1e-5, 1), g = e^l, g_C = g_63,
// a_i = g_{i-1}, kappa_j = g_C / g_j; A_ij = beta_i (g_i/g_j) k_i.k_j, P_ij = (g_{i-1}/g_j) q_i.k_j, j < i.
// Products over the D features use the precision policy P (bf16 operands for bf16 inputs), the 64 x 64
// chunk algebra fp32 MFMA.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <type_traits>
#include "kdn_frag.hpp"
#include "kdn_internal.hpp"
#include "kdn_io.hpp"
#include "kdn_tile.hpp"

namespace kdn {
namespace gen {

constexpr int C = 64;
constexpr int LD = 68;

// Record fields that hold operands in the precision policy's type are sized for fp32.
//
// Feature order.  A fragment read straight from a feature row takes eight consecutive features per lane (one
// 16- or 32-byte load): lane (g = l >> 4) slot s holds feature 8g + s of a 32-feature block.  A pair of
// accumulator tiles (2j, 2j + 1) over the block's features then holds feature 8g + 4a + i in row 4g + i of
// tile 2j + a, so that a lane's eight values of the pair are again eight consecutive features.
__device__ __forceinline__ int feature_of(int tile, int row) { return 32 * (tile >> 1) + 8 * (row >> 2) + 4 * (tile & 1) + (row & 3); }

template <int D, int DV>
struct Rec {
  static constexpr int NV = DV / 16;
  static constexpr size_t KXF = 0;            // K-row fragments [m 4][jb D/32][lane]; backward with bf16 fragments: Q's
                                              // likewise in the second half (QXF)
  static constexpr size_t KTF = KXF + C * D;  // fp32: K^T-row fragments [tile D/16][jb 2][lane]
  static constexpr size_t S = KTF + C * D;    // S^T at the chunk start as output fragments [jb D/32][n NV][lane]
  static constexpr size_t TPF = S + D * DV;   // Tp = T diag(beta g) as A fragments [row tile 4][jb 2][lane] f32x8
  static constexpr size_t P = TPF + C * C;    // forward: as A fragments, likewise; backward: rows [64][64]
  static constexpr size_t U = P + C * C;      // U~ as tiles [m 4][n NV][lane] f32x4
  static constexpr size_t W = U + C * DV;     // forward: tiles, likewise; backward: rows [64][DV]
  static constexpr size_t VEC = W + C * DV;   // 64-vectors: l, kappa
  static constexpr size_t V_L = VEC, V_KAP = VEC + 64;
  static constexpr size_t floats = VEC + 128;
};

// The backward's record (kdn_delta_scan_bwd at D = 1024): the forward's record (its S field holding fp32 tiles) followed
// by the fields of the gradient (offsets in floats).  D x DV matrices in accumulator tiles [n NV][tile D/16][lane]
// f32x4: lane (g, v = l & 15) holds features feature_of(tile, 4g + i) of value 16n + v.
template <int D, int DV>
struct BRec {
  static constexpr size_t SR = Rec<D, DV>::S;       // S^T at the chunk start, fp32 tiles
  static constexpr size_t T = Rec<D, DV>::floats;   // [64][64] (I + A)^-1
  static constexpr size_t G = T + C * C;            // [64][64] K K^T (on and below the diagonal tiles)
  static constexpr size_t TPT = G + C * C;          // Tp^T as A fragments, as TPF
  static constexpr size_t XK = TPT + C * C;         // [64][DV] K S^T
  static constexpr size_t QTF = XK + C * DV;        // fp32: Q^T-row fragments, as KTF
  static constexpr size_t RR = QTF + C * D;         // P^T dY, tiles as U~
  static constexpr size_t GR = RR + C * DV;         // dL/dS^T at the chunk end, fp32 tiles
  static constexpr size_t X = GR + D * DV;          // [64][DV] K Gamma
  static constexpr size_t DW = X + C * DV;          // [64][DV] dL/dW
  static constexpr size_t DWT = DW + C * DV;        // the same as tiles, as U~
  static constexpr size_t ZN = DWT + C * DV;        // [64][DV] -Tp^T dW (= dL/dX_K)
  static constexpr size_t AY = ZN + C * DV;         // [64][DV] a o dY
  static constexpr size_t AYF = AY + C * DV;        // a o dY as B fragments over tokens [n NV][jb 2][lane]
  static constexpr size_t OPS = AYF + C * DV;       // right operands of the feature gradients (bop_*), fragments
  static constexpr size_t PART = OPS + 3 * C * DV + 3 * C * C;  // [D/32][64] a o dY . Q S^T by 32-feature block, then
                                                                // [D/32] <Gamma, S> likewise
  static constexpr size_t V_BETA = PART + (D / 32 * 65 + 63) / 64 * 64;  // 64-vectors: beta, dl without the terms of S
  static constexpr size_t V_DL = V_BETA + 64;
  // The record's size as it was with more fields (workspace queries and the segment rule go by it): a quarter is unused.
  static constexpr size_t floats = T + 3 * D * DV + 7 * C * DV + 4 * C * C;
  static_assert(V_DL + 64 <= floats, "the fields fit the record");
};
// Fragment index in OPS: token tile m, 32-deep block of the value columns (AY, KW, ZN) or of the tokens
// (N, M + M^T, N^T).
template <int DV> __host__ __device__ constexpr int bop_v(int o, int m, int kb) { return (o * 4 + m) * (DV / 32) + kb; }
template <int DV> __host__ __device__ constexpr int bop_t(int o, int m, int jb) { return 3 * 4 * (DV / 32) + (o * 4 + m) * 2 + jb; }
template <int DV> __host__ __device__ constexpr int bop_count() { return 3 * 4 * (DV / 32) + 3 * 4 * 2; }

struct Params {
  int64_t B, T, H, nch;
  const void* q; int64_t qs0, qs1, qs2;
  const void* k; int64_t ks0, ks1, ks2;
  const void* v; int64_t vs0, vs1, vs2;
  const float* beta; int64_t bs0, bs1, bs2;
  const float* decay; int64_t ds0, ds1, ds2;
  const float* init; int64_t is0, is1, is2, is3;
  float* fin; int64_t fs0, fs1, fs2, fs3;
  void* y; int64_t ys0, ys1, ys2;
  float* ws;
  int qkvec, vvec, yvec;  // rows of q and k / of v / of y start on 16 bytes (4 elements for y), whatever the token
};

struct BwdP {
  const float* dy; int64_t ys0, ys1, ys2;         // NULL in the checkpoint pass
  const float* dfin; int64_t fs0, fs1, fs2, fs3;  // dL/dS^T at the end (NULL: zero)
  float* dq; int64_t dqs0, dqs1, dqs2;
  float* dk; int64_t dks0, dks1, dks2;
  float* dv; int64_t dvs0, dvs1, dvs2;
  float* dbeta; int64_t dbs0, dbs1, dbs2;
  float* ddecay; int64_t dds0, dds1, dds2;        // NULL: not wanted
  float* dinit; int64_t gis0, gis1, gis2, gis3;   // dL/dS^T at the start (NULL: not wanted)
  int yvec, gvec;                                 // rows of dy / of dq and dk start on 16 bytes
};

// Record of (b, h, c): the forward's layout, or the backward's longer one.
template <int D, int DV, bool BWD = false>
__device__ __forceinline__ float* record(const Params& p, int64_t b, int64_t h, int64_t c) {
  constexpr int64_t F = BWD ? (int64_t)BRec<D, DV>::floats : (int64_t)Rec<D, DV>::floats;
  return p.ws + ((b * p.H + h) * p.nch + c) * F;
}

// Eight consecutive elements as a fragment of policy PB.
template <class PB, typename InT, bool VEC>
__device__ __forceinline__ typename PB::frag load8(const InT* x) {
  typedef __attribute__((ext_vector_type(8))) InT in8;
  if constexpr (VEC) {
    const in8 t = *reinterpret_cast<const in8*>(x);
    if constexpr (std::is_same<typename PB::frag, in8>::value) {
      return t;
    } else {
      f32x8 r;
#pragma unroll
      for (int s = 0; s < 8; ++s) r[s] = (float)t[s];
      return PB::from_f32(r);
    }
  } else {
    f32x8 r;
#pragma unroll
    for (int s = 0; s < 8; ++s) r[s] = ldx(x + s);
    return PB::from_f32(r);
  }
}
template <class PB>
__device__ __forceinline__ typename PB::frag zero_frag() {
  f32x8 z;
#pragma unroll
  for (int s = 0; s < 8; ++s) z[s] = 0.f;
  return PB::from_f32(z);
}
// Fragment of the input's rows r0 .. r0 + 15, features k0 .. k0 + 31 (rows at or past `nrows` read as zero;
// their loads go to the last row).
template <class PB, typename InT, bool VEC>
__device__ __forceinline__ typename PB::frag row_frag(const InT* base, int64_t rs, int r0, int k0, int lane, int nrows) {
  const int row = r0 + (lane & 15);
  const typename PB::frag f = load8<PB, InT, VEC>(base + (row < nrows ? row : nrows - 1) * rs + k0 + 8 * (lane >> 4));
  return row < nrows ? f : zero_frag<PB>();
}
// Row tile `tile`, tokens k0 + kappa of the transposed input (fp32 fragments).
template <typename InT>
__device__ __forceinline__ f32x8 col_frag(const InT* base, int64_t rs, int tile, int k0, int lane, int nrows) {
  f32x8 r;
  const int f = feature_of(tile, lane & 15);
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int row = k0 + kappa(lane, s);
    r[s] = row < nrows ? ldx(base + row * rs + f) : 0.f;
  }
  return r;
}
// B fragments that pick row tile a of a 32-feature block: a row fragment times selector(a) has the
// accumulator layout of that tile's transpose (the values exactly: one product with 1, the rest with 0).
template <class PB>
__device__ __forceinline__ typename PB::frag selector(int a, int lane) {
  f32x8 e;
#pragma unroll
  for (int s = 0; s < 8; ++s) e[s] = ((lane & 15) >> 2) == (lane >> 4) && s == 4 * a + (lane & 3) ? 1.f : 0.f;
  return PB::from_f32(e);
}

// ---------------------------------------------------------------------------------------------- prep
// grid (nch, H, B), 256 threads.  The features are split over the waves: wave w reads blocks [w D/128,
// (w+1) D/128) of every row of K and Q once, multiplies what it read (the tiles on and below the
// diagonal), packs it, and the four waves' partial Grams are added in LDS; reading rows 16w .. instead,
// every wave read all of K, element by element.  The bound is the traffic: 256 KB in and 128 KB (backward
// 256 KB) of fragments out per chunk.  2016 chunks, bf16, d_v = 128: 668 -> 284 us, backward 676 -> 442 us (which now
// also forms R and packs a o dY and Q).
template <class PB, typename InT, int D, int DV, bool BWD, bool VEC>
__device__ __forceinline__ void prep_grams(const Params& p, float* rec, const InT* Kin, const InT* Qin, int w, int lane,
                                           int nrows, f32x4 (&gkk)[10], f32x4 (&gqk)[10]) {
  using R = Rec<D, DV>;
  using frag = typename PB::frag;
  frag* kxf = reinterpret_cast<frag*>(rec + R::KXF);
  frag* qxf = kxf + 4 * (D / 32) * 64;
  constexpr int NJ = D / 128;
  constexpr bool PACKQ = BWD && std::is_same<PB, PrecBF16>::value;
#pragma unroll
  for (int t = 0; t < 10; ++t) gkk[t] = gqk[t] = zero4();
  const InT* kr[4];
  const InT* qr[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int row = 16 * m + (lane & 15), rc = row < nrows ? row : nrows - 1;
    kr[m] = Kin + rc * p.ks1 + 32 * NJ * w + 8 * (lane >> 4);
    qr[m] = Qin + rc * p.qs1 + 32 * NJ * w + 8 * (lane >> 4);
  }
  frag kn[4], qn[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    kn[m] = load8<PB, InT, VEC>(kr[m]);
    qn[m] = load8<PB, InT, VEC>(qr[m]);
  }
#pragma unroll
  for (int jj = 0; jj < NJ; ++jj) {
    frag kf[4], qf[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      kf[m] = kn[m];
      qf[m] = qn[m];
      if (16 * m + (lane & 15) >= nrows) kf[m] = qf[m] = zero_frag<PB>();
      if (jj + 1 < NJ) {
        kn[m] = load8<PB, InT, VEC>(kr[m] + 32 * (jj + 1));
        qn[m] = load8<PB, InT, VEC>(qr[m] + 32 * (jj + 1));
      }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      kxf[(m * (D / 32) + NJ * w + jj) * 64 + lane] = kf[m];
      if constexpr (PACKQ) qxf[(m * (D / 32) + NJ * w + jj) * 64 + lane] = qf[m];
#pragma unroll
      for (int n = 0; n <= m; ++n) {
        gkk[m * (m + 1) / 2 + n] = PB::mma(gkk[m * (m + 1) / 2 + n], kf[m], kf[n]);
        gqk[m * (m + 1) / 2 + n] = PB::mma(gqk[m * (m + 1) / 2 + n], qf[m], kf[n]);
      }
    }
  }
}

template <class PB, typename InT, int D, int DV, bool BWD = false>
__global__ void __launch_bounds__(256) gen_prep_kernel(Params p, BwdP g) {
  using R = Rec<D, DV>;
  using BR = BRec<D, DV>;
  using frag = typename PB::frag;
  constexpr int LDV = DV + 4, NV = R::NV;
  constexpr int BUF = C * LD + C * LDV > 40 * 256 ? C * LD + C * LDV : 40 * 256;
  __shared__ __attribute__((aligned(16))) float bA[C * LD];  // A (as the inverse reads it), then P
  __shared__ __attribute__((aligned(16))) float buf[BUF];    // partial Grams [wave][tile][lane], then T and the value rows
  __shared__ float s_ell[C], s_beta[C];
  float* bT = buf;
  float* bV = buf + C * LD;

  const int64_t c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = c * C;
  float* rec = record<D, DV, BWD>(p, b, h, c);
  const int nrows = (int)(p.T - t0 < C ? p.T - t0 : C);

  if (w == 0) {
    const int64_t t = t0 + lane;
    const bool valid = t < p.T;
    const float be = valid ? p.beta[b * p.bs0 + t * p.bs1 + h * p.bs2] : 0.f;
    const float la = (valid && p.decay) ? p.decay[b * p.ds0 + t * p.ds1 + h * p.ds2] : 1.f;
    float l = logf(fminf(fmaxf(la, 1e-5f), 1.f));
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float u = __shfl_up(l, o);
      if (lane >= o) l += u;
    }
    s_ell[lane] = l;
    s_beta[lane] = be;
    rec[R::V_L + lane] = l;
    rec[R::V_KAP + lane] = expf(__shfl(l, 63) - l);
    if constexpr (BWD) rec[BR::V_BETA + lane] = be;
  }
  // the chunk's feature rows, read in place (rows past T read as zero)
  const InT* Kin = reinterpret_cast<const InT*>(p.k) + b * p.ks0 + t0 * p.ks1 + h * p.ks2;
  const InT* Qin = reinterpret_cast<const InT*>(p.q) + b * p.qs0 + t0 * p.qs1 + h * p.qs2;
  f32x4 pt[3];  // this wave's tiles of P (tiles w, w + 4, w + 8 of the ten)
  {
    f32x4 gkk[10], gqk[10];
    if (p.qkvec) prep_grams<PB, InT, D, DV, BWD, true>(p, rec, Kin, Qin, w, lane, nrows, gkk, gqk);
    else prep_grams<PB, InT, D, DV, BWD, false>(p, rec, Kin, Qin, w, lane, nrows, gkk, gqk);
    f32x4* part = reinterpret_cast<f32x4*>(buf);
#pragma unroll
    for (int t = 0; t < 10; ++t) part[(w * 10 + t) * 64 + lane] = gkk[t];
    for (int idx = tid; idx < C * C; idx += 256) bA[idx] = 0.f;
    __syncthreads();
    auto reduced = [&](int t) {
      return ((part[t * 64 + lane] + part[(10 + t) * 64 + lane]) + part[(20 + t) * 64 + lane]) + part[(30 + t) * 64 + lane];
    };
    for (int t = w; t < 10; t += 4) {
      const int m = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3, n = t - m * (m + 1) / 2;
      const f32x4 s = reduced(t);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * m + 4 * (lane >> 4) + i, cj = 16 * n + (lane & 15);
        // A transposed for the column-oriented inverse: [j][p][s] = A[4s+p][j]
        if (cj < ri) bA[(cj * 4 + (ri & 3)) * 16 + (ri >> 2)] = s_beta[ri] * expf(fminf(s_ell[ri] - s_ell[cj], 0.f)) * s[i];
        if constexpr (BWD) rec[BR::G + ri * C + cj] = s[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 10; ++t) part[(w * 10 + t) * 64 + lane] = gqk[t];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; ++k) pt[k] = w + 4 * k < 10 ? reduced(w + 4 * k) : zero4();
    __syncthreads();
  }
  if constexpr (!std::is_same<PB, PrecBF16>::value) {
    // fp32 fragments: the transposed operands packed too (wave w the feature tiles [w D/64, (w+1) D/64))
    frag* ktf = reinterpret_cast<frag*>(rec + R::KTF);
    for (int tt = 0; tt < D / 64; ++tt) {
      const int ft = w * (D / 64) + tt;
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        ktf[(ft * 2 + jb) * 64 + lane] = PB::from_f32(col_frag(Kin, p.ks1, ft, 32 * jb, lane, nrows));
        if constexpr (BWD)
          reinterpret_cast<frag*>(rec + BR::QTF)[(ft * 2 + jb) * 64 + lane] = PB::from_f32(col_frag(Qin, p.qs1, ft, 32 * jb, lane, nrows));
      }
    }
  }
  // beta o V in LDS; T = (I + A)^-1 (column-oriented substitution over lane quads)
  {
    const InT* Vin = reinterpret_cast<const InT*>(p.v) + b * p.vs0 + t0 * p.vs1 + h * p.vs2;
#pragma unroll 8
    for (int idx = tid; idx < C * DV; idx += 256) {
      const int r = idx / DV, e = idx % DV;
      bV[r * LDV + e] = r < nrows ? s_beta[r] * ldx(Vin + r * p.vs1 + e) : 0.f;
    }
  }
  unit_lower_inverse(bA, bT, LD, w, lane);
  __syncthreads();
  // P to LDS (A is used up), zero above its diagonal
  for (int idx = tid; idx < C * LD; idx += 256) bA[idx] = 0.f;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int t = w + 4 * k;
    const int m = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3, n = t - m * (m + 1) / 2;
    if (t < 10) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * m + 4 * (lane >> 4) + i, cj = 16 * n + (lane & 15);
        if (cj < ri) bA[ri * LD + cj] = expf(fminf((ri > 0 ? s_ell[ri - 1] : 0.f) - s_ell[cj], 0.f)) * pt[k][i];
      }
    }
  }
  // Tp (and its transpose) as fragments, T
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
    f32x8 f = frag_rows(bT, LD, 16 * w, 32 * jb, lane);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int j = 32 * jb + kappa(lane, s);
      f[s] = f[s] * s_beta[j] * expf(s_ell[j]);
    }
    reinterpret_cast<f32x8*>(rec + R::TPF)[(w * 2 + jb) * 64 + lane] = f;
    if constexpr (BWD) {
      const int j = 16 * w + (lane & 15);
      f32x8 ft = frag_cols(bT, LD, 16 * w, 32 * jb, lane);
#pragma unroll
      for (int s = 0; s < 8; ++s) ft[s] = ft[s] * s_beta[j] * expf(s_ell[j]);
      reinterpret_cast<f32x8*>(rec + BR::TPT)[(w * 2 + jb) * 64 + lane] = ft;
    }
  }
  if constexpr (BWD) {
    for (int idx = tid; idx < C * C; idx += 256) rec[BR::T + idx] = bT[(idx >> 6) * LD + (idx & 63)];
  }
  // U~ = T (beta o V), row tile w
  {
    const f32x8 ta0 = frag_rows(bT, LD, 16 * w, 0, lane), ta1 = frag_rows(bT, LD, 16 * w, 32, lane);
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const f32x4 u = mm<PrecF32>(mm<PrecF32>(zero4(), ta0, frag_cols(bV, LDV, 16 * n, 0, lane)), ta1,
                                  frag_cols(bV, LDV, 16 * n, 32, lane));
      reinterpret_cast<f32x4*>(rec + R::U)[(w * NV + n) * 64 + lane] = u;
    }
  }
  __syncthreads();
  if constexpr (!BWD) {
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) reinterpret_cast<f32x8*>(rec + R::P)[(w * 2 + jb) * 64 + lane] = frag_rows(bA, LD, 16 * w, 32 * jb, lane);
  } else {
    for (int idx = tid; idx < C * C; idx += 256) rec[R::P + idx] = bA[(idx >> 6) * LD + (idx & 63)];
    if (!g.dy) return;  // the checkpoint pass
    // R = P^T dY; a o dY as rows and as fragments over tokens and over values
    const float* Yin = g.dy + b * g.ys0 + t0 * g.ys1 + h * g.ys2;
#pragma unroll 8
    for (int idx = tid; idx < C * DV; idx += 256) {
      const int r = idx / DV, e = idx % DV;
      bV[r * LDV + e] = r < nrows ? Yin[r * g.ys1 + e] : 0.f;
    }
    __syncthreads();
    const f32x8 pa0 = frag_cols(bA, LD, 16 * w, 0, lane), pa1 = frag_cols(bA, LD, 16 * w, 32, lane);
#pragma unroll
    for (int n = 0; n < NV; ++n)
      reinterpret_cast<f32x4*>(rec + BR::RR)[(w * NV + n) * 64 + lane] =
          mm<PrecF32>(mm<PrecF32>(zero4(), pa0, frag_cols(bV, LDV, 16 * n, 0, lane)), pa1, frag_cols(bV, LDV, 16 * n, 32, lane));
    __syncthreads();
    for (int idx = tid; idx < C * DV; idx += 256) {
      const int r = idx / DV, e = idx % DV;
      const float ay = (r > 0 ? expf(s_ell[r - 1]) : 1.f) * bV[r * LDV + e];
      bV[r * LDV + e] = ay;
      rec[BR::AY + idx] = ay;
    }
    __syncthreads();
    frag* ayf = reinterpret_cast<frag*>(rec + BR::AYF);
    frag* ops = reinterpret_cast<frag*>(rec + BR::OPS);
#pragma unroll
    for (int k = 0; k < NV / 2; ++k) {  // NV 2 fragments over tokens: four waves
      const int f = w * (NV / 2) + k;
      ayf[f * 64 + lane] = PB::from_f32(frag_cols(bV, LDV, 16 * (f >> 1), 32 * (f & 1), lane));
    }
#pragma unroll
    for (int kb = 0; kb < DV / 32; ++kb) ops[bop_v<DV>(0, w, kb) * 64 + lane] = PB::from_f32(frag_rows(bV, LDV, 16 * w, 32 * kb, lane));
  }
}

// --------------------------------------------------------------------------------------------- carry
// grid: 8 * ceil(B*H / 8) * NV workgroups of CARRY_WAVES waves; workgroup (head-batch hb, value tile n), the
// NV value tiles of a head on one XCD.  Wave w keeps features [w D/8, (w+1) D/8) of its D x 16 slice of the
// carried matrix in registers: S^T forward, Gamma = dL/dS^T in reverse (REV, chunks last to first).
//
// Per chunk: store the slice; X = K Sigma (partial over the wave's features, reduced through LDS by waves 0..3,
// one token tile each); forward W = U~ - Tp X and Z = kappa o W, reverse dW = R + kappa o X and Z = -Tp^T dW;
// Sigma <- g_C Sigma (+ H = Q^T (a o dY)) + K^T Z.
//
// What bounds a step: the lines the CU takes from L2 (K 128 KB, in reverse Q likewise) and its three barriers with
// the 64-deep fp32 product of Tp between them.  With bf16 fragments K^T and Q^T are formed from the rows on
// the matrix cores, the next chunk's rows are loaded as soon as their registers come free, and waves 4..7 pull
// later chunks into L2 (as the D = 512 backward's carries do); fp32 fragments, twice the registers, are read
// where they are used.  32 heads, 63 chunks, bf16, d_v = 128, us per carry: forward 669 -> 280, in the backward
// (fp32 tiles of S written) 750 -> 359, reverse 1233 -> 534 against four waves that loaded K and K^T where they
// used them, K^T from memory and, in reverse, H (512 KB a chunk, another 502 us to form) in fp32.
constexpr int CARRY_WAVES = 8;
constexpr int CARRY_AHEAD = 3;  // chunks between a step and the operands it pulls into L2
struct CarryShared {
  f32x4 xp[CARRY_WAVES][4][64];
  f32x4 x[4][64];
  f32x4 z[4][64];
};

template <class PB, int D, int DV, bool BWD, bool REV>
struct CarryOps {
  using R = Rec<D, DV>;
  using BR = BRec<D, DV>;
  using frag = typename PB::frag;
  static constexpr int NV = DV / 16, JPW = D / 32 / CARRY_WAVES, TPW = 2 * JPW;
  static constexpr bool KEEP = std::is_same<PB, PrecBF16>::value;
  frag kx[4][KEEP ? JPW : 1];    // K rows 16m .., features of block JPW w + jj; in reverse then Q's
  frag kt[KEEP ? TPW : 1][2];    // K^T tile TPW w + t, tokens 32jb ..
  frag y[2];                     // a o dY (reverse)
  f32x8 tp[2];                   // waves 0..3: row tile w of Tp or Tp^T
  f32x4 ur, kap;                 // U~ or R, kappa
  float l63;

  __device__ __forceinline__ static frag k_frag(const float* rec, int w, int m, int jj, int lane) {
    return uni(reinterpret_cast<const frag*>(rec + R::KXF) + (m * (D / 32) + JPW * w + jj) * 64)[lane];
  }
  __device__ __forceinline__ void load_rows(const float* rec, bool q, int w, int lane) {
    const frag* f = reinterpret_cast<const frag*>(rec + R::KXF) + (q ? 4 * (D / 32) * 64 : 0);
#pragma unroll
    for (int jj = 0; jj < JPW; ++jj)
#pragma unroll
      for (int m = 0; m < 4; ++m) kx[m][jj] = uni(f + (m * (D / 32) + JPW * w + jj) * 64)[lane];
  }
  // Tile t of the transpose of the rows in kx, tokens 32jb ..
  __device__ __forceinline__ frag transposed(int t, int jb, const frag (&sel)[2]) const {
    return PB::from_f32(pair_to8(PB::mma(zero4(), kx[2 * jb][t >> 1], sel[t & 1]), PB::mma(zero4(), kx[2 * jb + 1][t >> 1], sel[t & 1])));
  }
  __device__ __forceinline__ void transpose_k(const frag (&sel)[2]) {
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      __builtin_amdgcn_sched_barrier(0);  // four products' results at a time
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        kt[t][jb] = transposed(t, jb, sel);
        asm volatile("" : "+v"(kt[t][jb]));  // packed here, not at its use
      }
    }
  }
  __device__ __forceinline__ void load_y(const float* rec, int n, int lane) {
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) y[jb] = uni(reinterpret_cast<const frag*>(rec + BR::AYF) + (n * 2 + jb) * 64)[lane];
  }
  __device__ __forceinline__ void load_lead(const float* rec, int w, int n, int lane) {
    const f32x8* f = reinterpret_cast<const f32x8*>(rec + (REV ? BR::TPT : R::TPF));
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) tp[jb] = uni(f + (w * 2 + jb) * 64)[lane];
    ur = uni(reinterpret_cast<const f32x4*>(rec + (REV ? BR::RR : R::U)) + (w * NV + n) * 64)[lane];
    kap = reinterpret_cast<const f32x4*>(uni(rec + R::V_KAP + 16 * w))[lane >> 4];
  }
  __device__ __forceinline__ void load_l63(const float* rec) { l63 = uni(rec + R::V_L + 63)[0]; }
};

// One dword of each 128-byte line of a later chunk's operands, shared out over waves 4..7 of the head's NV
// workgroups: pulls them into the XCD's L2.
template <class PB, int D, int DV, bool REV>
struct CarryPrefetch {
  using R = Rec<D, DV>;
  using BR = BRec<D, DV>;
  static constexpr int LANES = 256 * (DV / 16);
  static constexpr int AREA = C * D * (int)sizeof(typename PB::frag) / 8 / 128;  // lines of K
  static constexpr bool BF = std::is_same<PB, PrecBF16>::value;
  // K rows (bf16, reverse: and Q's behind them; fp32: K^T and in reverse Q^T), Tp, U~ or R, the vectors, a o dY
  static constexpr int E0 = BF && REV ? 2 * AREA : AREA, E1 = E0 + (BF ? 0 : AREA), E2 = E1 + (!BF && REV ? AREA : 0);
  static constexpr int E3 = E2 + 128, E4 = E3 + 2 * DV, E5 = E4 + 4;
  static constexpr int LINES = E5 + (REV ? C * DV * (int)sizeof(typename PB::frag) / 8 / 128 : 0);
  static constexpr int PER = (LINES + LANES - 1) / LANES;
  unsigned v[PER];  // the loaded words: used, and so waited for, only where the next step replaces them
  __device__ __forceinline__ void load(const float* rec, int n, int w, int lane) {
    const unsigned* r = reinterpret_cast<const unsigned*>(uni(rec));
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = (n * 4 + (w - 4)) * 64 + lane + LANES * k;
      unsigned at = R::VEC;
      if (i < E0) at = R::KXF + 32 * i;
      else if (i < E1) at = R::KTF + 32 * (i - E0);
      else if (i < E2) at = BR::QTF + 32 * (i - E1);
      else if (i < E3) at = (REV ? BR::TPT : R::TPF) + 32 * (i - E2);
      else if (i < E4) at = (REV ? BR::RR : R::U) + 32 * (i - E3);
      else if (i < E5) at = R::VEC + 32 * (i - E4);
      else if (REV && i < LINES) at = BR::AYF + 32 * (i - E5);
      v[k] = r[at];
    }
  }
};

// `lead`: waves 0..3, which reduce X and take the Tp product, and so transpose K before the first barrier; the others
// transpose it while those work.  The two run their own loops (one loop with both paths does not fit the registers).
template <class PB, int D, int DV, bool BWD, bool REV, bool lead>
__device__ __forceinline__ void carry_step(CarryShared& sh, float* rec, const float* nrec, const float* frec,
                                           CarryOps<PB, D, DV, BWD, REV>& o, CarryPrefetch<PB, D, DV, REV>& pf, unsigned& sink,
                                           f32x4 (&Sg)[D / 16 / CARRY_WAVES], const typename PB::frag (&sel)[2], int w,
                                           int lane, int n) {
  using O = CarryOps<PB, D, DV, BWD, REV>;
  using R = Rec<D, DV>;
  using BR = BRec<D, DV>;
  using frag = typename PB::frag;
  constexpr int NV = O::NV, JPW = O::JPW, TPW = O::TPW;
  constexpr bool KEEP = O::KEEP;
  const int row0 = 16 * w + 4 * (lane >> 4), vc = 16 * n + (lane & 15);  // a lead wave's rows and column
  // K times the carried slice, partial over this wave's features
  f32x4 xp[4];
  frag sb[JPW];
#pragma unroll
  for (int jj = 0; jj < JPW; ++jj) {
    sb[jj] = PB::from_f32(pair_to8(Sg[2 * jj], Sg[2 * jj + 1]));
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      if constexpr (KEEP) xp[m] = PB::mma(jj ? xp[m] : zero4(), o.kx[m][jj], sb[jj]);
      else xp[m] = PB::mma(jj ? xp[m] : zero4(), O::k_frag(rec, w, m, jj, lane), sb[jj]);
    }
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) sh.xp[w][m][lane] = xp[m];
  __builtin_amdgcn_sched_barrier(0);
  // the slice to the record: fp32 tiles (backward), output fragments (forward)
  if constexpr (BWD) {
    f32x4* dst = reinterpret_cast<f32x4*>(rec + (REV ? BR::GR : BR::SR));
#pragma unroll
    for (int t = 0; t < TPW; ++t) uni(dst + (n * (D / 16) + TPW * w + t) * 64)[lane] = Sg[t];
  } else {
    frag* sf = reinterpret_cast<frag*>(rec + R::S);
#pragma unroll
    for (int jj = 0; jj < JPW; ++jj) uni(sf + ((JPW * w + jj) * NV + n) * 64)[lane] = sb[jj];
  }
  const float gC = expf(o.l63);
#pragma unroll
  for (int t = 0; t < TPW; ++t) Sg[t] = Sg[t] * gC;
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (KEEP && lead) {
    o.transpose_k(sel);
    __builtin_amdgcn_sched_barrier(0);
    o.load_rows(REV ? rec : nrec, REV, w, lane);
  }
  o.load_l63(nrec);
  lds_barrier();
  if constexpr (lead) {
    f32x4 X = sh.xp[0][w][lane];
#pragma unroll
    for (int v = 1; v < CARRY_WAVES; ++v) X += sh.xp[v][w][lane];
    if constexpr (!REV) {
      sh.x[w][lane] = X;
      if constexpr (BWD) {
        float* d = uni(rec + BR::XK);
#pragma unroll
        for (int i = 0; i < 4; ++i) d[(row0 + i) * DV + vc] = X[i];
      }
    } else {
      const f32x4 dW = o.ur + o.kap * X;
      sh.x[w][lane] = dW;
      float* dx = uni(rec + BR::X);
      float* dd = uni(rec + BR::DW);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dx[(row0 + i) * DV + vc] = X[i];
        dd[(row0 + i) * DV + vc] = dW[i];
      }
      uni(reinterpret_cast<f32x4*>(rec + BR::DWT) + (w * NV + n) * 64)[lane] = dW;
    }
  } else if constexpr (KEEP) {
    o.transpose_k(sel);
    __builtin_amdgcn_sched_barrier(0);
    o.load_rows(REV ? rec : nrec, REV, w, lane);
  }
  lds_barrier();
  if constexpr (lead) {
    const f32x4 t = mm<PrecF32>(mm<PrecF32>(zero4(), o.tp[0], pair_to8(sh.x[0][lane], sh.x[1][lane])), o.tp[1],
                                pair_to8(sh.x[2][lane], sh.x[3][lane]));
    if constexpr (!REV) {
      const f32x4 Wt = o.ur - t;
      sh.z[w][lane] = o.kap * Wt;
      if constexpr (BWD) {
        float* d = uni(rec + R::W);
#pragma unroll
        for (int i = 0; i < 4; ++i) d[(row0 + i) * DV + vc] = Wt[i];
      } else {
        uni(reinterpret_cast<f32x4*>(rec + R::W) + (w * NV + n) * 64)[lane] = Wt;
      }
    } else {
      sh.z[w][lane] = -t;
      float* d = uni(rec + BR::ZN);
#pragma unroll
      for (int i = 0; i < 4; ++i) d[(row0 + i) * DV + vc] = -t[i];
    }
    __builtin_amdgcn_sched_barrier(0);
    o.load_lead(nrec, w, n, lane);
  } else if (frec) {
#pragma unroll
    for (int k = 0; k < CarryPrefetch<PB, D, DV, REV>::PER; ++k) sink ^= pf.v[k];
    pf.load(frec, n, w, lane);
  }
  if constexpr (REV) {
    // this wave's rows of H = Q^T (a o dY) for value tile n
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      if constexpr (KEEP) {
        __builtin_amdgcn_sched_barrier(0);
        Sg[t] = PB::mma(PB::mma(Sg[t], o.transposed(t, 0, sel), o.y[0]), o.transposed(t, 1, sel), o.y[1]);
      } else {
        const frag* qtf = reinterpret_cast<const frag*>(rec + BR::QTF) + (TPW * w + t) * 2 * 64;
        Sg[t] = PB::mma(PB::mma(Sg[t], uni(qtf)[lane], o.y[0]), uni(qtf + 64)[lane], o.y[1]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    o.load_y(nrec, n, lane);
    if constexpr (KEEP) o.load_rows(nrec, false, w, lane);
  }
  lds_barrier();
  const frag zb0 = PB::from_f32(pair_to8(sh.z[0][lane], sh.z[1][lane]));
  const frag zb1 = PB::from_f32(pair_to8(sh.z[2][lane], sh.z[3][lane]));
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    if constexpr (KEEP) {
      Sg[t] = PB::mma(PB::mma(Sg[t], o.kt[t][0], zb0), o.kt[t][1], zb1);
    } else {
      const frag* ktf = reinterpret_cast<const frag*>(rec + R::KTF) + (TPW * w + t) * 2 * 64;
      Sg[t] = PB::mma(PB::mma(Sg[t], uni(ktf)[lane], zb0), uni(ktf + 64)[lane], zb1);
    }
  }
}

template <class PB, int D, int DV, bool BWD, bool REV, bool lead>
__device__ __forceinline__ void carry_loop(CarryShared& sh, const Params& p, int b, int h, int nch, f32x4 (&Sg)[D / 16 / CARRY_WAVES],
                                           const typename PB::frag (&sel)[2], int w, int lane, int n, unsigned& sink) {
  using O = CarryOps<PB, D, DV, BWD, REV>;
  O o;
  {
    const float* rec = record<D, DV, BWD>(p, b, h, REV ? nch - 1 : 0);
    if constexpr (O::KEEP) o.load_rows(rec, false, w, lane);
    o.load_l63(rec);
    if constexpr (lead) o.load_lead(rec, w, n, lane);
    if constexpr (REV) o.load_y(rec, n, lane);
  }
  CarryPrefetch<PB, D, DV, REV> pf = {};
  for (int step = 0; step < nch; ++step) {
    const int c = REV ? nch - 1 - step : step;
    const int cn = step + 1 < nch ? (REV ? c - 1 : c + 1) : c;  // the last step loads its own chunk again
    const int cf = REV ? c - CARRY_AHEAD : c + CARRY_AHEAD;
    carry_step<PB, D, DV, BWD, REV, lead>(sh, record<D, DV, BWD>(p, b, h, c), record<D, DV, BWD>(p, b, h, cn),
                                          cf >= 0 && cf < nch ? record<D, DV, BWD>(p, b, h, cf) : nullptr, o, pf, sink, Sg, sel, w,
                                          lane, n);
  }
}

// The carried slice from / to a caller's state (NULL: zero / nothing).  In reverse over segments source and
// destination may be the same buffer: a thread rewrites exactly the elements it read.
template <class PB, int D, int DV, bool BWD, bool REV>
__global__ void __launch_bounds__(64 * CARRY_WAVES) gen_carry_kernel(Params p, const float* src, int64_t s0, int64_t s1, int64_t s2,
                                                                   int64_t s3, float* dst, int64_t o0, int64_t o1, int64_t o2,
                                                                   int64_t o3) {
  using O = CarryOps<PB, D, DV, BWD, REV>;
  constexpr int NV = O::NV, TPW = O::TPW;
  __shared__ CarryShared sh;
  const int64_t id = blockIdx.x;
  const int64_t xcd = id & 7, jdx = id >> 3;
  const int n = (int)(jdx % NV);
  const int64_t hb = (jdx / NV) * 8 + xcd;
  if (hb >= p.B * p.H) return;
  // the division is done in vector registers: back to scalars, so that every record address is one
  const int b = __builtin_amdgcn_readfirstlane((int)(hb / p.H));
  const int h = (int)hb - b * (int)p.H;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vc = 16 * n + (lane & 15);

  f32x4 Sg[TPW];
  // the slice's offsets are formed again at the end where, held through the loop, they would be spilled
  constexpr bool AGAIN = !O::KEEP || (REV && DV == 64);
  const int lb = AGAIN ? fresh(lane) : lane;
#pragma unroll
  for (int t = 0; t < TPW; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      Sg[t][i] = src ? src[b * s0 + h * s1 + feature_of(TPW * w + t, 4 * (lb >> 4) + i) * s2 + (16 * n + (lb & 15)) * s3] : 0.f;
  const typename PB::frag sel[2] = {selector<PB>(0, lane), selector<PB>(1, lane)};
  const int nch = (int)p.nch;
  unsigned sink = 0;  // keeps the prefetch loads alive (never stored: nch is positive)
  if (w < 4) carry_loop<PB, D, DV, BWD, REV, true>(sh, p, b, h, nch, Sg, sel, w, lane, n, sink);
  else carry_loop<PB, D, DV, BWD, REV, false>(sh, p, b, h, nch, Sg, sel, w, lane, n, sink);
  if (p.nch < 0) p.ws[0] = (float)sink;
  if (dst) {
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[b * o0 + h * o1 + feature_of(TPW * w + t, 4 * (lane >> 4) + i) * o2 + vc * o3] = Sg[t][i];
  }
}

// -------------------------------------------------------------------------------------------- output
// grid (nch, H, B), 256 threads; wave w the token tiles 2 (w & 1), 2 (w & 1) + 1 and half the value tiles, so that
// both operands are read twice (token tile w with every value tile: S four times).  Computed transposed
// (values in the rows), which puts four consecutive values of a token in a lane.
template <typename T>
__device__ __forceinline__ void store_el(T* p, float v);
template <>
__device__ __forceinline__ void store_el<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void store_el<__bf16>(__bf16* p, float v) { *p = (__bf16)v; }

template <class PB, typename InT, int D, int DV, bool VEC>
__device__ __forceinline__ void output_qs(const Params& p, const float* rec, const InT* Qin, int m0, int n0, int lane, int nrows,
                                          f32x4 (&acc)[DV / 32][2]) {
  constexpr int NV = DV / 16;
  const typename PB::frag* sf = reinterpret_cast<const typename PB::frag*>(rec + Rec<D, DV>::S);
#pragma unroll 4
  for (int jb = 0; jb < D / 32; ++jb) {
    typename PB::frag q[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) q[k] = row_frag<PB, InT, VEC>(Qin, p.qs1, 16 * (m0 + k), 32 * jb, lane, nrows);
#pragma unroll
    for (int n = 0; n < NV / 2; ++n) {
      const typename PB::frag s = sf[(jb * NV + n0 + n) * 64 + lane];
#pragma unroll
      for (int k = 0; k < 2; ++k) acc[n][k] = PB::mma(acc[n][k], s, q[k]);
    }
  }
}

template <class PB, typename InT, typename OutT, int D, int DV>
__global__ void __launch_bounds__(256) gen_output_kernel(Params p) {
  using R = Rec<D, DV>;
  constexpr int NV = R::NV;
  const int64_t c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = 2 * (w & 1), n0 = (w >> 1) * (NV / 2);
  const int64_t t0 = c * C;
  const float* rec = record<D, DV>(p, b, h, c);
  const int nrows = (int)(p.T - t0 < C ? p.T - t0 : C);
  const InT* Qin = reinterpret_cast<const InT*>(p.q) + b * p.qs0 + t0 * p.qs1 + h * p.qs2;
  f32x4 acc[NV / 2][2];
#pragma unroll
  for (int n = 0; n < NV / 2; ++n) acc[n][0] = acc[n][1] = zero4();
  if (p.qkvec) output_qs<PB, InT, D, DV, true>(p, rec, Qin, m0, n0, lane, nrows, acc);
  else output_qs<PB, InT, D, DV, false>(p, rec, Qin, m0, n0, lane, nrows, acc);
  const f32x8* pf = reinterpret_cast<const f32x8*>(rec + R::P);
  const f32x4* wt = reinterpret_cast<const f32x4*>(rec + R::W);
  OutT* y = reinterpret_cast<OutT*>(p.y) + b * p.ys0 + h * p.ys2;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const f32x8 p0 = pf[((m0 + k) * 2) * 64 + lane], p1 = pf[((m0 + k) * 2 + 1) * 64 + lane];
    const int64_t t = t0 + 16 * (m0 + k) + (lane & 15);
    const int ri = 16 * (m0 + k) + (lane & 15);
    const float a = ri > 0 ? expf(rec[R::V_L + ri - 1]) : 1.f;
#pragma unroll
    for (int n = 0; n < NV / 2; ++n) {
      auto tile = [&](int m) { return wt[(m * NV + n0 + n) * 64 + lane]; };
      const f32x4 pw = mm<PrecF32>(mm<PrecF32>(zero4(), pair_to8(tile(0), tile(1)), p0), pair_to8(tile(2), tile(3)), p1);
      const f32x4 r = a * acc[n][k] + pw;
      if (t < p.T) {
        OutT* d = y + t * p.ys1 + 16 * (n0 + n) + 4 * (lane >> 4);
        if (p.yvec) {
          typedef __attribute__((ext_vector_type(4))) OutT out4;
          out4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = (OutT)r[i];
          *reinterpret_cast<out4*>(d) = o;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) store_el<OutT>(d + i, r[i]);
        }
      }
    }
  }
}

template <class PB, int D, int DV, bool BWD>
static void launch_carry(const Params& p, hipStream_t st) {
  const unsigned wgs = (unsigned)(((p.B * p.H + 7) / 8) * 8 * (DV / 16));
  hipLaunchKernelGGL((gen_carry_kernel<PB, D, DV, BWD, false>), dim3(wgs), dim3(64 * CARRY_WAVES), 0, st, p, p.init, p.is0, p.is1,
                     p.is2, p.is3, p.fin, p.fs0, p.fs1, p.fs2, p.fs3);
}

template <class PB, typename InT, typename OutT, int D, int DV>
static int launch(const Params& p, hipStream_t st) {
  const dim3 chunk_grid((unsigned)p.nch, (unsigned)p.H, (unsigned)p.B);
  hipLaunchKernelGGL((gen_prep_kernel<PB, InT, D, DV>), chunk_grid, dim3(256), 0, st, p, BwdP{});
  launch_carry<PB, D, DV, false>(p, st);
  hipLaunchKernelGGL((gen_output_kernel<PB, InT, OutT, D, DV>), chunk_grid, dim3(256), 0, st, p);
  return launch_status();
}

template <int D, int DV>
static int launch_dtypes(const Params& p, int in_dt, int out_dt, hipStream_t st) {
  if (in_dt == KDN_DTYPE_BF16) {
    if (out_dt == KDN_DTYPE_BF16) return launch<PrecBF16, __bf16, __bf16, D, DV>(p, st);
    return launch<PrecBF16, __bf16, float, D, DV>(p, st);
  }
  if (out_dt == KDN_DTYPE_BF16) return launch<PrecF32, float, __bf16, D, DV>(p, st);
  return launch<PrecF32, float, float, D, DV>(p, st);
}

static size_t record_floats(int D, int DV) {
  if (D == 1024 && DV == 64) return Rec<1024, 64>::floats;
  if (D == 1024 && DV == 128) return Rec<1024, 128>::floats;
  return 0;
}

// ============================================================================================ backward
// Backward of the general-D scan (D = 1024 over pre-lifted features, d_v 64 or 128, the delta rule): the
// gradients of a loss with respect to phi_q, phi_k, v, beta, lambda and the initial state, given dL/dy
// and dL/d(final state).  The closed form per chunk is that of the D = 512 backward (kdn_bwd.hip), with
// one record per (batch, head, chunk) for the whole sequence:
//   prep, carry (the forward's kernels)  T, K K^T, Tp, P, U~, W; S^T at every chunk start, X_K = K S^T; and
//                                        R = P^T dY, a o dY
//   reverse carry (sequential)           Gamma = dL/dS^T at every chunk end, X = K Gamma, H = Q^T (a o dY),
//                                        dW = R + kappa o X, Z = Tp^T dW, Gamma <- g_C Gamma + H - K^T Z
//   grad    (parallel)                   dv, dbeta, the terms of dlambda without S; the right operands of the
//                                        feature gradients
//   dphi    (parallel, 256 features per workgroup)
//                                        dphi_q^T = S^T (a o dY)^T + K^T N^T
//                                        dphi_k^T = Gamma (kappa o W)^T - S^T Z^T + K^T (M + M^T) + Q^T N
//                                        and the terms of dlambda with S, a o dY . Q S^T and <Gamma, S>, in partial sums
//   decay   (parallel)                   dlambda, where it is wanted
// with S the chunk-start state as the recurrence's d_v x D matrix (the carries hold S^T, D x d_v),
// N_ij = dP_ij g_{i-1}/g_j and M_ij = dA_ij beta_i g_i/g_j below the diagonal, dP = dY W^T and
// dA = -T^T dT T^T.  S and Gamma, 512 KB each per chunk in fp32, are most of the backward's traffic: each is
// written once, in the accumulators' own tiles, and read once.
// The contractions that involve the features (the carries, H, Q S^T and the feature gradients) take the
// forward's precision policy (bf16 operands with fp32 accumulation for bf16 inputs, as the D = 512
// backward); the 64 x 64 chunk algebra runs on fp32 MFMA.  Every reduction has a fixed order (no
// atomics).

// ---------------------------------------------------------------------------------------------- grad
// grid (nch, H, B), 256 threads; wave w owns row tile w of the 64 x 64 chunk algebra.  Rows of the
// fixed-order partial-sum tables: dl_i from the kappa term, the column sums of P o dP per row tile (4),
// the row sums of P o dP (at i - 1), beta g (T o dTp) column sums, the column sums of beta o A o dA per row
// tile (4), its row sums; dbeta_i from the V . T^T dW row sums, the Tp column sums and the A o dA row sums.
constexpr int GDL_K = 0, GDL_COLP = 1, GDL_RP = 5, GDL_TS = 6, GDL_DLC = 7, GDL_A = 11, GNDL = 12;
constexpr int GDB_V = 0, GDB_TS = 1, GDB_A = 2, GNDB = 3;

// Sum over the 64 lanes of a wave in a fixed order (the result in every lane).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// The products over the value columns (phase 1 of grad), VV: V's rows and dY's start on 16 bytes.
template <typename InT, int D, int DV, bool VV>
__device__ __forceinline__ void grad_products(const float* rec, const InT* Vin, int64_t vs, const float* Yin, int64_t ys, int rt,
                                              int lane, int nrows, f32x4 (&dtp)[4], f32x4 (&e1)[4], f32x4 (&dp)[4]) {
  using F = Rec<D, DV>;
  using R = BRec<D, DV>;
#pragma unroll
  for (int n4 = 0; n4 < 4; ++n4) dtp[n4] = e1[n4] = dp[n4] = zero4();
#pragma unroll 2
  for (int kb = 0; kb < DV / 32; ++kb) {
    const f32x8 da = frag_rows_plain(rec + R::DW, DV, 16 * rt, 32 * kb, lane);
    const f32x8 ya = row_frag<PrecF32, float, VV>(Yin, ys, 16 * rt, 32 * kb, lane, nrows);
#pragma unroll
    for (int n4 = 0; n4 < 4; ++n4) {
      dtp[n4] = mm<PrecF32>(dtp[n4], da, frag_rows_plain(rec + R::XK, DV, 16 * n4, 32 * kb, lane));
      e1[n4] = mm<PrecF32>(e1[n4], da, row_frag<PrecF32, InT, VV>(Vin, vs, 16 * n4, 32 * kb, lane, nrows));
      dp[n4] = mm<PrecF32>(dp[n4], ya, frag_rows_plain(rec + F::W, DV, 16 * n4, 32 * kb, lane));
    }
  }
}

template <class PB, typename InT, int D, int DV>
__global__ void __launch_bounds__(256) gbwd_grad_kernel(Params p, BwdP g) {
  using F = Rec<D, DV>;
  using R = BRec<D, DV>;
  using frag = typename PB::frag;
  constexpr int NV = DV / 16;
  __shared__ __attribute__((aligned(16))) float bT[C * LD];   // T
  __shared__ __attribute__((aligned(16))) float bD[C * LD];   // dT, then M + M^T
  __shared__ __attribute__((aligned(16))) float bY1[C * LD];  // dT T^T
  __shared__ __attribute__((aligned(16))) float bN[C * LD];   // N
  __shared__ float s_ell[C], s_beta[C], s_kap[C];
  __shared__ float s_dl[GNDL][C], s_db[GNDB][C], s_ts[4][C], s_kt[C], s_63;

  const int64_t c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rt = w;
  const int64_t t0 = c * C;
  float* rec = record<D, DV, true>(p, b, h, c);
  frag* ops = reinterpret_cast<frag*>(rec + R::OPS);
  const int nrows = (int)(p.T - t0 < C ? p.T - t0 : C);
  const InT* Vin = reinterpret_cast<const InT*>(p.v) + b * p.vs0 + t0 * p.vs1 + h * p.vs2;
  const float* Yin = g.dy + b * g.ys0 + t0 * g.ys1 + h * g.ys2;

  if (tid < C) {
    s_ell[tid] = rec[F::V_L + tid];
    s_beta[tid] = rec[R::V_BETA + tid];
    s_kap[tid] = rec[F::V_KAP + tid];
  }
  for (int idx = tid; idx < GNDL * C; idx += 256) (&s_dl[0][0])[idx] = 0.f;
  for (int idx = tid; idx < GNDB * C; idx += 256) (&s_db[0][0])[idx] = 0.f;
  for (int idx = 4 * tid; idx < C * C; idx += 1024)
    *reinterpret_cast<f32x4*>(bT + (idx >> 6) * LD + (idx & 63)) = *reinterpret_cast<const f32x4*>(rec + R::T + idx);
  __syncthreads();

  // ---- phase 1: dTp = -dW X_K^T, dW V^T, dP = dY W^T -> dT, N, the Tp and P o dP sums; T^T dW -> dv, dbeta;
  //      the kappa term; kappa o W and Z as operands of the feature gradients
  {
    f32x4 dtp[4], e1[4], dp[4];
    if (p.vvec && g.yvec) grad_products<InT, D, DV, true>(rec, Vin, p.vs1, Yin, g.ys1, rt, lane, nrows, dtp, e1, dp);
    else grad_products<InT, D, DV, false>(rec, Vin, p.vs1, Yin, g.ys1, rt, lane, nrows, dtp, e1, dp);
    float rowp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n4 = 0; n4 < 4; ++n4) {
      const int cj = 16 * n4 + (lane & 15);
      const float bj = s_beta[cj], gj = expf(s_ell[cj]);
      float ts = 0.f, colp = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * rt + 4 * (lane >> 4) + i;
        const float dtpv = -dtp[n4][i];
        ts += bT[ri * LD + cj] * dtpv;
        bD[ri * LD + cj] = bj * (e1[n4][i] + gj * dtpv);
        float nv = 0.f;
        if (cj < ri) {
          const float pb = dp[n4][i] * rec[F::P + ri * C + cj];
          rowp[i] += pb;
          colp += pb;
          nv = dp[n4][i] * expf(fminf(s_ell[ri - 1] - s_ell[cj], 0.f));
        }
        bN[ri * LD + cj] = nv;
      }
      ts = sum_col4(ts);
      colp = sum_col4(colp);
      if (lane < 16) {
        s_ts[rt][cj] = ts;
        s_dl[GDL_COLP + rt][cj] = -colp;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float rp = sum_row16(rowp[i]);
      if ((lane & 15) == 0 && ri > 0) s_dl[GDL_RP][ri - 1] = rp;
    }
    // T^T dW, rows 16 rt ..: dv and the V . (T^T dW) row sums
    const f32x8 ta0 = frag_cols(bT, LD, 16 * rt, 0, lane), ta1 = frag_cols(bT, LD, 16 * rt, 32, lane);
    const f32x4* dwt = reinterpret_cast<const f32x4*>(rec + R::DWT);
    float dbv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nv = 0; nv < NV; ++nv) {
      auto tile = [&](int m) { return dwt[(m * NV + nv) * 64 + lane]; };
      const f32x4 td = mm<PrecF32>(mm<PrecF32>(zero4(), ta0, pair_to8(tile(0), tile(1))), ta1, pair_to8(tile(2), tile(3)));
      const int vcol = 16 * nv + (lane & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * rt + 4 * (lane >> 4) + i;
        if (ri < nrows) {
          g.dv[b * g.dvs0 + (t0 + ri) * g.dvs1 + h * g.dvs2 + vcol] = s_beta[ri] * td[i];
          dbv[i] += ldx(Vin + ri * p.vs1 + vcol) * td[i];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float s = sum_row16(dbv[i]);
      if ((lane & 15) == 0) s_db[GDB_V][ri] = s;
    }
  }
  {
    // the kappa term: dkappa_i = W_i . X_i (token 16w + (l & 15), a quarter of the columns per lane group, the
    // four partials added in a fixed order); kappa o W and -Z as fragments
    const int r = 16 * w + (lane & 15);
    const float kap = s_kap[r];
    float dk = 0.f;
#pragma unroll
    for (int kb = 0; kb < DV / 32; ++kb) {
      const f32x8 wv = frag_rows(rec + F::W, DV, 16 * w, 32 * kb, lane), xv = frag_rows(rec + R::X, DV, 16 * w, 32 * kb, lane);
#pragma unroll
      for (int s = 0; s < 8; ++s) dk += wv[s] * xv[s];
      ops[bop_v<DV>(1, w, kb) * 64 + lane] = PB::from_f32(kap * wv);
      ops[bop_v<DV>(2, w, kb) * 64 + lane] = PB::from_f32(frag_rows(rec + R::ZN, DV, 16 * w, 32 * kb, lane));
    }
    dk = sum_col4(dk);
    if (lane < 16) {
      s_dl[GDL_K][r] = -dk * kap;
      s_kt[r] = dk * kap;
    }
  }
  __syncthreads();
  if (w == 0) {
    const float tot = wave_sum(s_kt[lane]);
    if (lane == 0) s_63 = tot;
  }
  // ---- phase 2: the Tp sums; Y1 = dT T^T; N and N^T as fragments
  if (tid < C) {
    const float gj = expf(s_ell[tid]), ts = ((s_ts[0][tid] + s_ts[1][tid]) + s_ts[2][tid]) + s_ts[3][tid];
    s_db[GDB_TS][tid] = gj * ts;
    s_dl[GDL_TS][tid] = s_beta[tid] * gj * ts;
  }
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
    ops[bop_t<DV>(0, w, jb) * 64 + lane] = PB::from_f32(frag_rows(bN, LD, 16 * w, 32 * jb, lane));
    ops[bop_t<DV>(2, w, jb) * 64 + lane] = PB::from_f32(frag_cols(bN, LD, 16 * w, 32 * jb, lane));
  }
  {
    const f32x8 a0 = frag_rows(bD, LD, 16 * rt, 0, lane), a1 = frag_rows(bD, LD, 16 * rt, 32, lane);
#pragma unroll
    for (int n4 = 0; n4 < 4; ++n4) {
      const f32x4 y1 = mm<PrecF32>(mm<PrecF32>(zero4(), a0, frag_rows(bT, LD, 16 * n4, 0, lane)), a1,
                                   frag_rows(bT, LD, 16 * n4, 32, lane));
#pragma unroll
      for (int i = 0; i < 4; ++i) bY1[(16 * rt + 4 * (lane >> 4) + i) * LD + 16 * n4 + (lane & 15)] = y1[i];
    }
  }
  __syncthreads();

  // ---- phase 3: dA = -T^T Y1 (strictly lower); M + M^T (over dT); dbeta and dl from A
  {
    const f32x8 ta0 = frag_cols(bT, LD, 16 * rt, 0, lane), ta1 = frag_cols(bT, LD, 16 * rt, 32, lane);
    float dbr[4] = {0.f, 0.f, 0.f, 0.f}, dlr[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n4 = 0; n4 < 4; ++n4) {
      const f32x4 dA = -mm<PrecF32>(mm<PrecF32>(zero4(), ta0, frag_cols(bY1, LD, 16 * n4, 0, lane)), ta1,
                                    frag_cols(bY1, LD, 16 * n4, 32, lane));
      const int cj = 16 * n4 + (lane & 15);
      float dlc = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * rt + 4 * (lane >> 4) + i;
        if (cj < ri) {
          const float ex = expf(fminf(s_ell[ri] - s_ell[cj], 0.f));
          const float e = dA[i] * ex * rec[R::G + ri * C + cj];
          const float ab = s_beta[ri] * e;
          dbr[i] += e;
          dlr[i] += ab;
          dlc += ab;
          const float mv = dA[i] * s_beta[ri] * ex;
          bD[ri * LD + cj] = mv;
          bD[cj * LD + ri] = mv;
        } else if (cj == ri) {
          bD[ri * LD + cj] = 0.f;
        }
      }
      dlc = sum_col4(dlc);
      if (lane < 16) s_dl[GDL_DLC + rt][cj] = -dlc;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float a = sum_row16(dbr[i]), d = sum_row16(dlr[i]);
      if ((lane & 15) == 0) {
        s_db[GDB_A][ri] = a;
        s_dl[GDL_A][ri] = d;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) ops[bop_t<DV>(1, w, jb) * 64 + lane] = PB::from_f32(frag_rows(bD, LD, 16 * w, 32 * jb, lane));

  // ---- phase 4: dbeta, and dl without the terms of S
  if (w == 0) {
    float dl = 0.f;
#pragma unroll
    for (int k = 0; k < GNDL; ++k) dl += s_dl[k][lane];
    if (lane == 63) dl += s_63;
    float dbeta = 0.f;
#pragma unroll
    for (int k = 0; k < GNDB; ++k) dbeta += s_db[k][lane];
    rec[R::V_DL + lane] = dl;
    if (lane < nrows) g.dbeta[b * g.dbs0 + (t0 + lane) * g.dbs1 + h * g.dbs2] = dbeta;
  }
}

// dlambda: one wave per chunk adds the partial sums over the feature blocks in their order, then
// dlog lambda_t = sum_{i >= t} dl_i.
template <int D, int DV>
__global__ void __launch_bounds__(64) gbwd_decay_kernel(Params p, BwdP g) {
  using F = Rec<D, DV>;
  using R = BRec<D, DV>;
  const int64_t c = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x;
  const float* rec = record<D, DV, true>(p, b, h, c);
  const float* part = rec + R::PART;
  float da = 0.f, gs = 0.f;
#pragma unroll 8
  for (int k = 0; k < D / 32; ++k) {
    da += part[k * 64 + lane];
    gs += part[D / 32 * 64 + k];
  }
  // dl_{i-1} takes row i's a o dY . Q S^T, dl_63 takes g_C <Gamma, S>
  const float up = __shfl_down(da, 1);
  float dl = rec[R::V_DL + lane] + (lane < 63 ? up : expf(rec[F::V_L + 63]) * gs);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float u = __shfl_down(dl, o);
    if (lane + o < 64) dl += u;
  }
  const int64_t t = c * C + lane;
  if (t < p.T) {
    const float la = p.decay ? p.decay[b * p.ds0 + t * p.ds1 + h * p.ds2] : 1.f;
    g.ddecay[b * g.dds0 + t * g.dds1 + h * g.dds2] = (la >= 1e-5f && la <= 1.f) ? dl / la : 0.f;
  }
}

// ---------------------------------------------------------------------------------------------- dphi
// grid (nch * D / 256, H, B), DPHI_WAVES waves; workgroup (chunk, block of 256 features), wave w features
// [32 w, 32 w + 32) of the block for all 64 tokens.  The gradients are formed transposed (features in the
// rows): a lane's pair of accumulator tiles is eight consecutive features of a token.  The bound is the
// traffic, 1.9 MB a chunk, of which S and Gamma are 1 MB: both are read once, as coalesced tiles that serve as
// the operand of Q S^T as they are, and of the gradients after an exact transpose on the matrix cores (products
// with selector()).  With bf16 fragments the right operands, the same for every wave, are staged in LDS.
// 2016 chunks, bf16, d_v = 128: 1316 -> 919 us (4.2 TB/s) with the sums over S taken over from the gradient kernel
// (1319 -> 343 us), which read S and Gamma a second time.
constexpr int DPHI_WAVES = 8;
template <class PB, typename InT, int D, int DV>
__global__ void __launch_bounds__(64 * DPHI_WAVES) gbwd_dphi_kernel(Params p, BwdP g) {
  using F = Rec<D, DV>;
  using R = BRec<D, DV>;
  using frag = typename PB::frag;
  constexpr bool BF = std::is_same<PB, PrecBF16>::value;
  constexpr int FB = 32 * DPHI_WAVES, NOP = bop_count<DV>();
  __shared__ frag s_ops[BF ? NOP * 64 : 1];
  const int64_t c = blockIdx.x / (D / FB), h = blockIdx.y, b = blockIdx.z;
  const int fb = (int)(blockIdx.x % (D / FB));
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t0 = c * C;
  float* rec = record<D, DV, true>(p, b, h, c);
  const int nrows = (int)(p.T - t0 < C ? p.T - t0 : C);
  const frag* ops = reinterpret_cast<const frag*>(rec + R::OPS);
  if constexpr (BF) {
#pragma unroll
    for (int k = 0; k < NOP / DPHI_WAVES; ++k) s_ops[(k * DPHI_WAVES + w) * 64 + lane] = ops[(k * DPHI_WAVES + w) * 64 + lane];
  }
  auto op = [&](int i) { return BF ? s_ops[i * 64 + lane] : ops[i * 64 + lane]; };
  const int jf = fb * DPHI_WAVES + w;  // the wave's 32-feature block
  const frag sel[2] = {selector<PB>(0, lane), selector<PB>(1, lane)};
  // token rows of Q and K (fragments [m][jb]): packed by prep with bf16 fragments, else from the input
  frag qf[4];
  if constexpr (BF) {
    const frag* qxf = reinterpret_cast<const frag*>(rec + F::KXF) + 4 * (D / 32) * 64;
#pragma unroll
    for (int m = 0; m < 4; ++m) qf[m] = qxf[(m * (D / 32) + jf) * 64 + lane];
  } else {
    const InT* Qin = reinterpret_cast<const InT*>(p.q) + b * p.qs0 + t0 * p.qs1 + h * p.qs2;
#pragma unroll
    for (int m = 0; m < 4; ++m) qf[m] = row_frag<PB, InT, false>(Qin, p.qs1, 16 * m, 32 * jf, lane, nrows);
  }
  if constexpr (BF) __syncthreads();
  f32x4 aq[4][2], ak[4][2];  // [token tile][feature tile]
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int t = 0; t < 2; ++t) aq[m][t] = ak[m][t] = zero4();
  float dap[4] = {0.f, 0.f, 0.f, 0.f}, gs = 0.f;
  const bool want = g.ddecay != nullptr;
  const f32x4* st = reinterpret_cast<const f32x4*>(rec + R::SR) + 2 * jf * 64 + (BF ? lane : 0);
  const f32x4* gt = reinterpret_cast<const f32x4*>(rec + R::GR) + 2 * jf * 64 + (BF ? lane : 0);
  // contractions over the value columns: S^T (a o dY)^T, Gamma (kappa o W)^T, -S^T Z^T
#pragma unroll 1
  for (int kb = 0; kb < DV / 32; ++kb) {
    frag sb[2], gb[2];
#pragma unroll
    for (int nn = 0; nn < 2; ++nn) {
      const size_t at = (size_t)(2 * kb + nn) * (D / 16) * 64;
      f32x8 sv, gv;
      if constexpr (BF) {
        sv = pair_to8(st[at], st[at + 64]);
        gv = pair_to8(gt[at], gt[at + 64]);
      } else {  // scalar bases: fp32 fragments leave no vector registers for the addresses
        const f32x4 *sp = uni(st + at), *gp = uni(gt + at);
        sv = pair_to8(sp[lane], sp[64 + lane]);
        gv = pair_to8(gp[lane], gp[64 + lane]);
      }
#pragma unroll
      for (int s = 0; s < 8; ++s) gs += sv[s] * gv[s];
      sb[nn] = PB::from_f32(sv);
      gb[nn] = PB::from_f32(gv);
    }
    if (want) {
#pragma unroll
      for (int nn = 0; nn < 2; ++nn)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const f32x4 qs = PB::mma(zero4(), sb[nn], qf[m]);
          const f32x4 ay = *reinterpret_cast<const f32x4*>(rec + R::AY + (16 * m + (lane & 15)) * DV + 32 * kb + 16 * nn + 4 * (lane >> 4));
          dap[m] += ((ay[0] * qs[0] + ay[1] * qs[1]) + ay[2] * qs[2]) + ay[3] * qs[3];
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const frag sf = PB::from_f32(pair_to8(PB::mma(zero4(), sb[0], sel[t]), PB::mma(zero4(), sb[1], sel[t])));
      const frag gf = PB::from_f32(pair_to8(PB::mma(zero4(), gb[0], sel[t]), PB::mma(zero4(), gb[1], sel[t])));
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        aq[m][t] = PB::mma(aq[m][t], sf, op(bop_v<DV>(0, m, kb)));
        ak[m][t] = PB::mma(PB::mma(ak[m][t], gf, op(bop_v<DV>(1, m, kb))), sf, op(bop_v<DV>(2, m, kb)));
      }
    }
  }
  // contractions over the chunk's tokens: K^T N^T, K^T (M + M^T), Q^T N
  {
    frag kf[4];
    const frag* kxf = reinterpret_cast<const frag*>(rec + F::KXF);
#pragma unroll
    for (int m = 0; m < 4; ++m) kf[m] = kxf[(m * (D / 32) + jf) * 64 + lane];
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const frag kt = PB::from_f32(pair_to8(PB::mma(zero4(), kf[2 * jb], sel[t]), PB::mma(zero4(), kf[2 * jb + 1], sel[t])));
        const frag qt = PB::from_f32(pair_to8(PB::mma(zero4(), qf[2 * jb], sel[t]), PB::mma(zero4(), qf[2 * jb + 1], sel[t])));
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          aq[m][t] = PB::mma(aq[m][t], kt, op(bop_t<DV>(0, m, jb)));
          ak[m][t] = PB::mma(PB::mma(ak[m][t], kt, op(bop_t<DV>(1, m, jb))), qt, op(bop_t<DV>(2, m, jb)));
        }
      }
  }
  const int le = BF ? lane : fresh(lane);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int ri = 16 * m + (le & 15);
    if (ri >= nrows) continue;
    const int64_t t = t0 + ri;
    const int f = 32 * jf + 8 * (le >> 4);
    float* dq = g.dq + b * g.dqs0 + t * g.dqs1 + h * g.dqs2 + f;
    float* dk = g.dk + b * g.dks0 + t * g.dks1 + h * g.dks2 + f;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      if (g.gvec) {
        *reinterpret_cast<f32x4*>(dq + 4 * a) = aq[m][a];
        *reinterpret_cast<f32x4*>(dk + 4 * a) = ak[m][a];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          dq[4 * a + i] = aq[m][a][i];
          dk[4 * a + i] = ak[m][a][i];
        }
      }
    }
  }
  if (want) {
    float* part = rec + R::PART;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const float s = sum_col4(dap[m]);
      if (le < 16) part[jf * 64 + 16 * m + le] = s;
    }
    gs = wave_sum(gs);
    if (le == 0) part[D / 32 * 64 + jf] = gs;
  }
}

template <class PB, typename InT, int D, int DV>
static int launch_bwd(const Params& p, const BwdP& g, hipStream_t st) {
  const dim3 chunk_grid((unsigned)p.nch, (unsigned)p.H, (unsigned)p.B);
  const unsigned wgs = (unsigned)(((p.B * p.H + 7) / 8) * 8 * (DV / 16));
  hipLaunchKernelGGL((gen_prep_kernel<PB, InT, D, DV, true>), chunk_grid, dim3(256), 0, st, p, g);
  launch_carry<PB, D, DV, true>(p, st);
  hipLaunchKernelGGL((gen_carry_kernel<PB, D, DV, true, true>), dim3(wgs), dim3(64 * CARRY_WAVES), 0, st, p, g.dfin, g.fs0, g.fs1,
                     g.fs2, g.fs3, g.dinit, g.gis0, g.gis1, g.gis2, g.gis3);
  hipLaunchKernelGGL((gbwd_grad_kernel<PB, InT, D, DV>), chunk_grid, dim3(256), 0, st, p, g);
  hipLaunchKernelGGL((gbwd_dphi_kernel<PB, InT, D, DV>), dim3((unsigned)(p.nch * (D / (32 * DPHI_WAVES))), (unsigned)p.H, (unsigned)p.B),
                     dim3(64 * DPHI_WAVES), 0, st, p, g);
  if (g.ddecay) hipLaunchKernelGGL((gbwd_decay_kernel<D, DV>), chunk_grid, dim3(64), 0, st, p, g);
  return launch_status();
}

// The checkpoint pass of a segmented backward: the recompute and the forward carry of one segment, which
// writes the state at the segment's end to p.fin.
template <class PB, typename InT, int D, int DV>
static int launch_ckpt(const Params& p, hipStream_t st) {
  const dim3 chunk_grid((unsigned)p.nch, (unsigned)p.H, (unsigned)p.B);
  hipLaunchKernelGGL((gen_prep_kernel<PB, InT, D, DV, true>), chunk_grid, dim3(256), 0, st, p, BwdP{});
  launch_carry<PB, D, DV, true>(p, st);
  return launch_status();
}

static size_t bwd_record_floats(int D, int DV) {
  if (D == 1024 && DV == 64) return BRec<1024, 64>::floats;
  if (D == 1024 && DV == 128) return BRec<1024, 128>::floats;
  return 0;
}

// Segments of the backward: fwd->segment_chunks when positive, else the largest power of two from 4 to 256
// chunks whose records fit 24 GiB (one 256-chunk segment at B*H = 32, d_v = 128: 26.7 ms per backward
// against 29.7 in two segments of 128, which 12 GiB gave); at most the sequence's chunks.  Workspace: one segment's records, one
// fp32 [B][H][1024][d_v] state per segment boundary (the checkpoints), the carried dL/dS (with more than
// one segment) and the forward carry's final state (scratch).
constexpr size_t BWD_SEGMENT_BUDGET = (size_t)24 << 30;
struct BwdPlan {
  int64_t nch, seg, nsegs;
  size_t rec_bytes, state_bytes, ckpt_off, carry_off, fin_off, total;
};
static BwdPlan bwd_plan(const kdn_scan_args* f) {
  BwdPlan L;
  L.nch = (f->T + C - 1) / C;
  const int64_t heads = f->B * f->H;
  const size_t per_chunk = (size_t)heads * bwd_record_floats((int)f->D, (int)f->d_v) * sizeof(float);
  int64_t seg = 4;
  if (f->segment_chunks > 0) {
    seg = f->segment_chunks;
  } else {
    const size_t fit = BWD_SEGMENT_BUDGET / per_chunk;
    while (seg < 256 && (size_t)(2 * seg) <= fit) seg *= 2;
  }
  if (seg > L.nch) seg = L.nch;
  L.seg = seg;
  L.nsegs = (L.nch + seg - 1) / seg;
  L.rec_bytes = (size_t)seg * per_chunk;
  L.state_bytes = (size_t)heads * (size_t)f->D * (size_t)f->d_v * sizeof(float);
  L.ckpt_off = L.rec_bytes;
  L.carry_off = L.ckpt_off + (size_t)(L.nsegs - 1) * L.state_bytes;
  L.fin_off = L.carry_off + (L.nsegs > 1 ? L.state_bytes : 0);
  L.total = L.fin_off + L.state_bytes;
  return L;
}

// Whether every row of a (B, T, H, d) view starts on `bytes` (strides of dimensions of one are not used).
static bool rows_aligned(const Params& p, const void* x, int64_t s0, int64_t s1, int64_t s2, size_t elem, size_t bytes) {
  const int64_t n = (int64_t)(bytes / elem);
  return aligned(x, bytes) && (p.B == 1 || s0 % n == 0) && (p.T == 1 || s1 % n == 0) && (p.H == 1 || s2 % n == 0);
}
static void set_row_flags(Params& p, size_t isz) {
  p.qkvec = rows_aligned(p, p.q, p.qs0, p.qs1, p.qs2, isz, 16) && rows_aligned(p, p.k, p.ks0, p.ks1, p.ks2, isz, 16);
  p.vvec = rows_aligned(p, p.v, p.vs0, p.vs1, p.vs2, isz, 16);
}

}  // namespace gen

bool general_scan_applies(const kdn_scan_args* a) { return a && a->D == 1024; }

int general_scan_validate(const kdn_scan_args* a) {
  if (a->feature_mode != 1 || a->d_k != a->D) return KDN_ERR_UNSUPPORTED;  // pre-lifted features only
  if (a->rule != 0 || a->cu_seqlens || a->state_slots) return KDN_ERR_UNSUPPORTED;
  if (a->d_v != 64 && a->d_v != 128) return KDN_ERR_UNSUPPORTED;
  return KDN_OK;
}

size_t general_scan_workspace_bytes(const kdn_scan_args* a) {
  const int64_t nch = (a->T + gen::C - 1) / gen::C;
  return (size_t)(a->B * a->H * nch) * gen::record_floats(a->D, a->d_v) * sizeof(float);
}

int general_scan(const kdn_scan_args* a, void* stream) {
  if (a->workspace_bytes < general_scan_workspace_bytes(a)) return KDN_ERR_WORKSPACE_TOO_SMALL;
  gen::Params p = {};
  p.B = a->B; p.T = a->T; p.H = a->H; p.nch = (a->T + gen::C - 1) / gen::C;
  if (p.nch > 0x7fffffff) return KDN_ERR_UNSUPPORTED;
  p.q = a->q; p.qs0 = a->q_stride[0]; p.qs1 = a->q_stride[1]; p.qs2 = a->q_stride[2];
  p.k = a->k; p.ks0 = a->k_stride[0]; p.ks1 = a->k_stride[1]; p.ks2 = a->k_stride[2];
  p.v = a->v; p.vs0 = a->v_stride[0]; p.vs1 = a->v_stride[1]; p.vs2 = a->v_stride[2];
  p.beta = a->beta; p.bs0 = a->beta_stride[0]; p.bs1 = a->beta_stride[1]; p.bs2 = a->beta_stride[2];
  p.decay = a->decay; p.ds0 = a->decay_stride[0]; p.ds1 = a->decay_stride[1]; p.ds2 = a->decay_stride[2];
  p.init = a->initial_state;
  p.is0 = a->init_stride[0]; p.is1 = a->init_stride[1]; p.is2 = a->init_stride[2]; p.is3 = a->init_stride[3];
  p.fin = a->final_state;
  p.fs0 = a->final_stride[0]; p.fs1 = a->final_stride[1]; p.fs2 = a->final_stride[2]; p.fs3 = a->final_stride[3];
  p.y = a->y; p.ys0 = a->y_stride[0]; p.ys1 = a->y_stride[1]; p.ys2 = a->y_stride[2];
  p.ws = reinterpret_cast<float*>(a->workspace);
  gen::set_row_flags(p, dtype_size(a->in_dtype));
  const size_t osz = dtype_size(a->out_dtype);
  p.yvec = gen::rows_aligned(p, p.y, p.ys0, p.ys1, p.ys2, osz, 4 * osz);
  const hipStream_t st = as_stream(stream);
  if (a->d_v == 64) return gen::launch_dtypes<1024, 64>(p, a->in_dtype, a->out_dtype, st);
  return gen::launch_dtypes<1024, 128>(p, a->in_dtype, a->out_dtype, st);
}

}  // namespace kdn

namespace kdn {

bool general_bwd_applies(const kdn_scan_args* f) { return f && f->D == 1024; }

static int general_bwd_check(const kdn_scan_bwd_args* a) {
  if (!a || !a->fwd) return KDN_ERR_INVALID_ARGUMENT;
  const kdn_scan_args* f = a->fwd;
  if (f->B <= 0 || f->T <= 0 || f->H <= 0 || !valid_dtype(f->in_dtype)) return KDN_ERR_INVALID_ARGUMENT;
  if (f->B > 65535 || f->H > 65535) return KDN_ERR_UNSUPPORTED;  // grid y / z limits of the chunk launches
  const int rc = general_scan_validate(f);
  if (rc != KDN_OK) return rc;
  if (a->dinv_tau) return KDN_ERR_UNSUPPORTED;  // pre-lifted features have no temperature
  if (!f->q || !f->k || !f->v || !f->beta) return KDN_ERR_INVALID_ARGUMENT;
  if (!a->dy || !a->dq || !a->dk || !a->dv || !a->dbeta) return KDN_ERR_INVALID_ARGUMENT;
  if (a->ddecay && !f->decay) return KDN_ERR_INVALID_ARGUMENT;
  for (int i = 0; i < 3; ++i) {
    if (f->q_stride[i] < 0 || f->k_stride[i] < 0 || f->v_stride[i] < 0 || f->beta_stride[i] < 0 ||
        (f->decay && f->decay_stride[i] < 0) || a->dy_stride[i] < 0 || a->dq_stride[i] < 0 || a->dk_stride[i] < 0 ||
        a->dv_stride[i] < 0 || a->dbeta_stride[i] < 0 || (a->ddecay && a->ddecay_stride[i] < 0))
      return KDN_ERR_INVALID_ARGUMENT;
  }
  for (int i = 0; i < 4; ++i) {
    if ((f->initial_state && f->init_stride[i] < 0) || (a->d_final_state && a->dfinal_stride[i] < 0) ||
        (a->d_initial_state && a->dinit_stride[i] < 0))
      return KDN_ERR_INVALID_ARGUMENT;
  }
  const size_t isz = dtype_size(f->in_dtype);
  if (!aligned(f->q, isz) || !aligned(f->k, isz) || !aligned(f->v, isz) || !aligned(f->beta, 4))
    return KDN_ERR_MISALIGNED;
  if (!aligned(a->dy, 4) || !aligned(a->dq, 4) || !aligned(a->dk, 4) || !aligned(a->dv, 4) || !aligned(a->dbeta, 4))
    return KDN_ERR_MISALIGNED;
  return KDN_OK;
}

size_t general_bwd_workspace_bytes(const kdn_scan_bwd_args* a) {
  if (general_bwd_check(a) != KDN_OK) return 0;
  return gen::bwd_plan(a->fwd).total;
}

int64_t general_bwd_segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks) {
  if (general_bwd_check(a) != KDN_OK) return 0;
  const gen::BwdPlan L = gen::bwd_plan(a->fwd);
  if (segment_chunks) *segment_chunks = L.seg;
  return L.nsegs;
}

// Segmented like the D = 512 backward: a checkpoint pass runs the recompute and the forward carry over
// segments 0 .. n-2 and keeps the state at each segment start; then each segment, last first, recomputes
// its chunks from its checkpoint, carries dL/dS back from the next segment (in place in one buffer: every
// workgroup of the reverse carry reads its slice before it writes it) and writes its gradients.  A segment
// is the chunk range [c0, c0 + n) as a sequence of its own (input and gradient pointers advanced by 64 c0
// tokens); the kernels carry the same sums in the same order as over the whole sequence, so the results
// do not depend on the segment length.
template <class PB, typename InT, int D, int DV>
static int general_bwd_run(const gen::Params& p, const gen::BwdP& g, const gen::BwdPlan& L, size_t isz,
                           hipStream_t st) {
  unsigned char* ws = reinterpret_cast<unsigned char*>(p.ws);
  const int64_t ss0 = p.H * D * DV, ss1 = (int64_t)D * DV, ss2 = DV, ss3 = 1;  // checkpoint / carry layout
  auto state_at = [&](size_t off) { return reinterpret_cast<float*>(ws + off); };
  auto segment = [&](int64_t s, gen::Params& ps, gen::BwdP& gs) {
    const int64_t c0 = s * L.seg, n = (L.nch - c0 < L.seg) ? L.nch - c0 : L.seg, t0 = c0 * gen::C;
    ps = p;
    gs = g;
    ps.nch = n;
    ps.T = (p.T - t0 < n * gen::C) ? p.T - t0 : n * gen::C;
    ps.q = static_cast<const unsigned char*>(p.q) + (size_t)(t0 * p.qs1) * isz;
    ps.k = static_cast<const unsigned char*>(p.k) + (size_t)(t0 * p.ks1) * isz;
    ps.v = static_cast<const unsigned char*>(p.v) + (size_t)(t0 * p.vs1) * isz;
    ps.beta = p.beta + t0 * p.bs1;
    if (p.decay) ps.decay = p.decay + t0 * p.ds1;
    gs.dy = g.dy + t0 * g.ys1;
    gs.dq = g.dq + t0 * g.dqs1;
    gs.dk = g.dk + t0 * g.dks1;
    gs.dv = g.dv + t0 * g.dvs1;
    gs.dbeta = g.dbeta + t0 * g.dbs1;
    if (g.ddecay) gs.ddecay = g.ddecay + t0 * g.dds1;
    if (s > 0) {  // the state at the segment start: the checkpoint of segment s - 1's end
      ps.init = state_at(L.ckpt_off + (size_t)(s - 1) * L.state_bytes);
      ps.is0 = ss0; ps.is1 = ss1; ps.is2 = ss2; ps.is3 = ss3;
    }
  };
  for (int64_t s = 0; s + 1 < L.nsegs; ++s) {
    gen::Params ps;
    gen::BwdP gs;
    segment(s, ps, gs);
    ps.fin = state_at(L.ckpt_off + (size_t)s * L.state_bytes);
    ps.fs0 = ss0; ps.fs1 = ss1; ps.fs2 = ss2; ps.fs3 = ss3;
    const int rc = gen::launch_ckpt<PB, InT, D, DV>(ps, st);
    if (rc != KDN_OK) return rc;
  }
  for (int64_t s = L.nsegs - 1; s >= 0; --s) {
    gen::Params ps;
    gen::BwdP gs;
    segment(s, ps, gs);
    ps.fin = state_at(L.fin_off);
    ps.fs0 = ss0; ps.fs1 = ss1; ps.fs2 = ss2; ps.fs3 = ss3;
    if (s + 1 < L.nsegs) {  // dL/dS at the segment end, left by the next segment's reverse carry
      gs.dfin = state_at(L.carry_off);
      gs.fs0 = ss0; gs.fs1 = ss1; gs.fs2 = ss2; gs.fs3 = ss3;
    }
    if (s > 0) {  // dL/dS at the segment start, for the previous segment
      gs.dinit = state_at(L.carry_off);
      gs.gis0 = ss0; gs.gis1 = ss1; gs.gis2 = ss2; gs.gis3 = ss3;
    }
    const int rc = gen::launch_bwd<PB, InT, D, DV>(ps, gs, st);
    if (rc != KDN_OK) return rc;
  }
  return KDN_OK;
}

int general_bwd(const kdn_scan_bwd_args* a, void* stream) {
  const int rc = general_bwd_check(a);
  if (rc != KDN_OK) return rc;
  if (a->workspace_bytes < general_bwd_workspace_bytes(a)) return KDN_ERR_WORKSPACE_TOO_SMALL;
  if (!a->workspace) return KDN_ERR_INVALID_ARGUMENT;
  if (!aligned(a->workspace, 256)) return KDN_ERR_MISALIGNED;
  const kdn_scan_args* f = a->fwd;
  const gen::BwdPlan L = gen::bwd_plan(f);
  gen::Params p = {};
  p.B = f->B; p.T = f->T; p.H = f->H; p.nch = L.nch;
  if (p.nch > 0x7fffffff) return KDN_ERR_UNSUPPORTED;
  p.q = f->q; p.qs0 = f->q_stride[0]; p.qs1 = f->q_stride[1]; p.qs2 = f->q_stride[2];
  p.k = f->k; p.ks0 = f->k_stride[0]; p.ks1 = f->k_stride[1]; p.ks2 = f->k_stride[2];
  p.v = f->v; p.vs0 = f->v_stride[0]; p.vs1 = f->v_stride[1]; p.vs2 = f->v_stride[2];
  p.beta = f->beta; p.bs0 = f->beta_stride[0]; p.bs1 = f->beta_stride[1]; p.bs2 = f->beta_stride[2];
  p.decay = f->decay; p.ds0 = f->decay_stride[0]; p.ds1 = f->decay_stride[1]; p.ds2 = f->decay_stride[2];
  p.init = f->initial_state;
  p.is0 = f->init_stride[0]; p.is1 = f->init_stride[1]; p.is2 = f->init_stride[2]; p.is3 = f->init_stride[3];
  p.ws = reinterpret_cast<float*>(a->workspace);
  const int DV = (int)f->d_v;
  gen::BwdP g = {};
  g.dy = a->dy; g.ys0 = a->dy_stride[0]; g.ys1 = a->dy_stride[1]; g.ys2 = a->dy_stride[2];
  g.dfin = a->d_final_state;
  g.fs0 = a->dfinal_stride[0]; g.fs1 = a->dfinal_stride[1]; g.fs2 = a->dfinal_stride[2]; g.fs3 = a->dfinal_stride[3];
  g.dq = a->dq; g.dqs0 = a->dq_stride[0]; g.dqs1 = a->dq_stride[1]; g.dqs2 = a->dq_stride[2];
  g.dk = a->dk; g.dks0 = a->dk_stride[0]; g.dks1 = a->dk_stride[1]; g.dks2 = a->dk_stride[2];
  g.dv = a->dv; g.dvs0 = a->dv_stride[0]; g.dvs1 = a->dv_stride[1]; g.dvs2 = a->dv_stride[2];
  g.dbeta = a->dbeta; g.dbs0 = a->dbeta_stride[0]; g.dbs1 = a->dbeta_stride[1]; g.dbs2 = a->dbeta_stride[2];
  g.ddecay = a->ddecay; g.dds0 = a->ddecay_stride[0]; g.dds1 = a->ddecay_stride[1]; g.dds2 = a->ddecay_stride[2];
  g.dinit = a->d_initial_state;
  g.gis0 = a->dinit_stride[0]; g.gis1 = a->dinit_stride[1]; g.gis2 = a->dinit_stride[2]; g.gis3 = a->dinit_stride[3];
  const hipStream_t st = as_stream(stream);
  const size_t isz = dtype_size(f->in_dtype);
  gen::set_row_flags(p, isz);
  g.yvec = gen::rows_aligned(p, g.dy, g.ys0, g.ys1, g.ys2, 4, 16);
  g.gvec = gen::rows_aligned(p, g.dq, g.dqs0, g.dqs1, g.dqs2, 4, 16) && gen::rows_aligned(p, g.dk, g.dks0, g.dks1, g.dks2, 4, 16);
  if (DV == 64) {
    if (f->in_dtype == KDN_DTYPE_BF16) return general_bwd_run<PrecBF16, __bf16, 1024, 64>(p, g, L, isz, st);
    return general_bwd_run<PrecF32, float, 1024, 64>(p, g, L, isz, st);
  }
  if (f->in_dtype == KDN_DTYPE_BF16) return general_bwd_run<PrecBF16, __bf16, 1024, 128>(p, g, L, isz, st);
  return general_bwd_run<PrecF32, float, 1024, 128>(p, g, L, isz, st);
}

}  // namespace kdn
