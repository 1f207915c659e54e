// Backward pass of the chunked gated delta rule and of the feature lift (gfx950).
//
// The reference differentiates its chunked torch forward with autograd (FusedKernelDeltaNetFunction,
// kernels/fused_kernel_deltanet.py:158-179: the backward recomputes the forward under autograd).  Here
// the gradient of the same function is computed directly, in closed form per 64-token chunk, by four
// launches that recompute what they need from the inputs:
//
//   prep  (parallel over chunks x heads)  lift q, k; Gram matrices K K^T, Q K^T; A, T = (I + A)^-1,
//                                         Tp = T diag(beta g), U~ = T (beta o V), P; R = P^T dY and
//                                         a o dY (a_i = g_{i-1})
//   chain (sequential over chunks)        forward:  S_c^T at every chunk start, X_K = K S_c^T,
//                                                   W = U~ - Tp X_K, S_{c+1}^T = g_C S_c^T + K^T (kappa o W)
//         (same kernel, reversed)         backward: Gamma = dL/dS^T at every chunk end, X = K Gamma,
//                                                   dW = R + kappa o X, H = Q^T (a o dY),
//                                                   Gamma <- g_C Gamma + H - K^T Tp^T dW
//   grad  (parallel over chunks x heads)  dv, dbeta, dlambda and dphi_q, dphi_k in closed form, then
//                                         the lift backward (cos -> -sin, renormalisation, input
//                                         normalisation) to dq, dk
//
// Notation per chunk (tokens i, j in 0..63): l_i = sum_{t <= i} log clamp(lambda_t, 1e-5, 1), g = e^l,
// g_C = g_63, a_i = g_{i-1} (a_0 = 1), kappa_j = g_C / g_j; A_ij = beta_i (g_i/g_j) k_i.k_j and
// P_ij = (g_{i-1}/g_j) q_i.k_j for j < i; Y = diag(a) Q S^T + P W; S_C^T = g_C S^T + K^T diag(kappa) W.
// The matrices live in a per-(head, chunk) record of the workspace (struct Rec).  Products use the
// MFMA fragment conventions of kdn_frag.hpp: the lift and the 64 x 64 chunk algebra in fp32
// (16x16x4 f32), the contractions over the 512 features in the precision policy P (fp32 for fp32
// inputs, bf16 operands with fp32 accumulation for bf16 inputs).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <type_traits>
#include "kdn_frag.hpp"
#include "kdn_internal.hpp"
#include "kdn_io.hpp"
#include "kdn_tile.hpp"

namespace kdn {
namespace bwd {

constexpr int C = 64, D = 512, DK = 64, DV = 64;
constexpr int LD = 68;  // LDS row stride (floats) of a 64-wide tile: rows stay 16-byte aligned
constexpr size_t OMT_BYTES = (size_t)4 * 16 * 64 * 16;  // the Omega^T fragment table

// The gradient kernel runs eight waves: wave w owns row tile w & 3 and column tiles 2 (w >> 2) .. +1 of
// the 64 x 64 chunk algebra.  Rows of its dl_i contribution table, one per source term: the dkappa term
// (-t_i), the column sums of P o dP per row tile (4 rows), the row sums of P o dP per column half (at
// i - 1; 2 rows), beta g (T o dTp) column sums, the a o dY . Q S^T term per column half (at i - 1; 2
// rows), the column sums of A o dA per row tile (4 rows) and the row sums of A o dA per column half (2).
constexpr int GRAD_WAVES = 8;
constexpr int DL_KAPPA = 0, DL_COLP = 1, DL_RP = 5, DL_TS = 7, DL_DA = 8, DL_DLC = 10, DL_A = 14, NDL = 16;
// Rows of its dbeta table: the T^T dW . V row sums per column half (2), the Tp column sums, the A o dA
// row sums per column half (2).
constexpr int DB_V = 0, DB_TS = 2, DB_A = 3, NDB = 5;

// Fragment slots of the dx kernel's B operands in the record's K-fragment area: token tile m (0..3),
// operand o, 32-token depth block jb; 32 slots for dK^T (4 operands) then 16 for dQ^T (2 operands).
__host__ __device__ constexpr int bop_dk(int m, int o, int jb) { return (m * 4 + o) * 2 + jb; }
__host__ __device__ constexpr int bop_dq(int m, int o, int jb) { return 32 + (m * 2 + o) * 2 + jb; }

// Per (head, chunk) record, offsets in floats.  Areas that hold operands in the policy's type are sized for
// fp32.
struct Rec {
  static constexpr size_t Q = 0;                // SF: S^T as B fragments [n 4][jb 16][lane] for Q S^T (fp32 features:
                                                // first the lifted q rows [64][512], until the Gram matrices)
  static constexpr size_t K = Q + C * D;        // fp32 features: the lifted k rows, then Q in fragment order (QXF);
                                                // bf16: Tp as A fragments [row tile 4][jb 2][lane] f32x8 (TPF)
  static constexpr size_t TPF = K;
  static constexpr size_t AYF = K + C * D;      // a o dY as B fragments [n 4][jb 2][lane] (sized for f32x8)
  static constexpr size_t S = AYF + 4 * 2 * 64 * 8;  // S^T at the chunk start, in 4-value pieces (piece_at)
  static constexpr size_t G = S + D * DV;       // dL/dS^T at the chunk end, likewise
  static constexpr size_t T = G + D * DV;       // [64][64] (I + A)^-1
  static constexpr size_t TPT = T + C * C;      // Tp^T = diag(beta g) T^T as A fragments [row tile 4][jb 2][lane] f32x8
  static constexpr size_t P = TPT + C * C;      // [64][64]
  static constexpr size_t GKK = P + C * C;      // [64][64] K K^T
  static constexpr size_t U = GKK + C * C;      // U~ = T (beta o V) as tiles [m 4][n 4][lane] f32x4
  static constexpr size_t R = U + C * DV;       // P^T dY, tiles as U~
  static constexpr size_t W = R + C * DV;       // W = U~ - Tp X_K, tiles
  static constexpr size_t XK = W + C * DV;      // K S^T, tiles
  static constexpr size_t DW = XK + C * DV;     // dL/dW, tiles
  static constexpr size_t X = DW + C * DV;      // K Gamma, tiles
  // 64-vectors: l, beta, |phi~_q|, |phi~_k|, beta g (0 for the linear rule), phi_q . dphi_q and
  // phi_k . dphi_k (from the gradient kernel), kappa
  static constexpr size_t VEC = X + C * DV;
  static constexpr size_t V_ELL = VEC, V_BETA = VEC + 64, V_NORM = VEC + 128, V_BG = VEC + 256, V_RD = VEC + 320, V_KAP = VEC + 448;
  // K in MFMA fragment order for the chains (one 16- or 32-byte load per lane and fragment), in the
  // precision policy's fragment type (bf16x8 or f32x8; the area is sized for f32x8):
  static constexpr size_t KXF = VEC + 512;      // [m 4][jb 16][lane]: rows 16m.., features 32jb..; with bf16 features Q
                                                // likewise in the second half (QXF)
  static constexpr size_t KTF = KXF + C * D;    // [ft 32][jb 2][lane]: K^T rows 16ft.., tokens 32jb..
  static constexpr size_t QTF = KTF + C * D;    // [ft 32][jb 2][lane]: Q^T rows 16ft.., tokens 32jb..
  static constexpr size_t floats = QTF + C * D;
};
static_assert((Rec::floats * 4) % 256 == 0, "records stay 256-byte aligned");
static_assert(48 * 64 * sizeof(f32x8) <= (Rec::KTF - Rec::KXF) * sizeof(float), "the dx operands fit the K-fragment area");

struct Params {
  int64_t B, T, H, nch;
  int64_t c0, nseg, cap;  // this segment: first global chunk, chunks in it, records per head in its buffer
  const void* q; int64_t qs0, qs1, qs2;
  const void* k; int64_t ks0, ks1, ks2;
  const void* v; int64_t vs0, vs1, vs2;
  const float* beta; int64_t bs0, bs1, bs2;
  const float* decay; int64_t ds0, ds1, ds2;
  const __bf16* omega; const float* phase;
  float inv_tau; int normalize;
  // the feature map beyond one shared structured Omega: low parts of Omega (Omega = hi + lo; NULL when
  // hi is exact), head strides of Omega and the phases in elements (0: shared), per-head 1/tau (NULL:
  // inv_tau), phi = sqrt(2/D) cos(.) without renormalisation; the linear update rule
  const __bf16* omega_lo; int64_t oms, phs;
  const float* inv_tau_head;
  int no_renorm, linear;
  float* dit;       // dL/d(1/tau) of each (batch, head, chunk) [B][H][nch] (NULL: not wanted)
  float* dinv_tau;  // dL/d(1/tau) per head [H], the sum of dit over batches and chunks
  const float* init; int64_t is0, is1, is2, is3;  // S^T at the segment start (NULL: zero)
  const float* dy; int64_t ys0, ys1, ys2;
  const float* dfin; int64_t fs0, fs1, fs2, fs3;  // dL/dS^T at the segment end (NULL: zero)
  float* dq; int64_t dqs0, dqs1, dqs2;
  float* dk; int64_t dks0, dks1, dks2;
  float* dv; int64_t dvs0, dvs1, dvs2;
  float* dbeta; int64_t dbs0, dbs1, dbs2;
  float* ddecay; int64_t dds0, dds1, dds2;
  float* gout; int64_t gos0, gos1, gos2, gos3;    // dL/dS^T at the segment start (NULL: not kept)
  float* ws;                                       // this segment's buffer of records
  const bf16x8* omt;  // Omega^T fragments [part][a 4][jb 16][lane] (workspace tail, written before the gradients)
  int64_t omt_hs;     // entries between heads' tables (0: one table); part 1 (the lo parts) at +OMT_ENTRIES
};
constexpr int OMT_ENTRIES = 4 * 16 * 64;

__device__ __forceinline__ float head_inv_tau(const Params& p, int64_t h) {
  return p.inv_tau_head ? p.inv_tau_head[h] : p.inv_tau;
}

// Record of local chunk c (0 .. nseg - 1) of the segment.
__device__ __forceinline__ float* record(const Params& p, int64_t b, int64_t h, int64_t c) {
  return p.ws + ((b * p.H + h) * p.cap + c) * (int64_t)Rec::floats;
}

// The features and the carried S^T, Gamma are stored in their record areas as bf16 under the bf16 policy
// (every product that reads them rounds its operands to bf16 anyway; <Gamma, S> reads the rounded values)
// and as fp32 under the fp32 policy.
template <class P> struct Feat { typedef float T; };
template <> struct Feat<PrecBF16> { typedef __bf16 T; };
template <class P> struct IsBf16Policy : std::integral_constant<bool, std::is_same<P, PrecBF16>::value> {};
template <class P>
__device__ __forceinline__ typename Feat<P>::T* feat(float* rec, size_t off) {
  return reinterpret_cast<typename Feat<P>::T*>(rec + off);
}
template <class P>
__device__ __forceinline__ const typename Feat<P>::T* feat(const float* rec, size_t off) {
  return reinterpret_cast<const typename Feat<P>::T*>(rec + off);
}
__device__ __forceinline__ f32x4 ld4_t(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 ld4_t(const __bf16* p) {
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  const f32x4 r = {(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  return r;
}

// Operand fragments straight in the policy's type (no fp32 round trip for bf16 data):
//   frag_rows_p: kappa-ordered rows of a record matrix in its storage type (as frag_rows)
//   omega_frag:  rows r0.. of the bf16 Omega [D][64], plain depth order (as frag_rows_plain_bf16)
//   bf16_frag:   a bf16x8 fragment
template <class P>
__device__ __forceinline__ typename P::frag frag_rows_p(const typename Feat<P>::T* b, int ld, int r0, int k0, int lane) {
  if constexpr (IsBf16Policy<P>::value) {
    typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
    const __bf16* q = b + (size_t)(r0 + (lane & 15)) * ld + k0 + 4 * (lane >> 4);
    const bf16x4 lo = *reinterpret_cast<const bf16x4*>(q);
    const bf16x4 hi = *reinterpret_cast<const bf16x4*>(q + 16);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  } else {
    return frag_rows(b, ld, r0, k0, lane);
  }
}
template <class P>
__device__ __forceinline__ typename P::frag omega_frag(const __bf16* omega, int r0, int k0, int lane) {
  if constexpr (IsBf16Policy<P>::value)
    return *reinterpret_cast<const bf16x8*>(omega + (size_t)(r0 + (lane & 15)) * DK + k0 + 8 * (lane >> 4));
  else
    return frag_rows_plain_bf16(omega, DK, r0, k0, lane);
}
// The carried 512 x 64 matrices in 4-value pieces: piece (ft, n, lane) holds values 16n + 4(lane >> 4) + 0..3 of
// feature 16ft + (lane & 15), so that an A fragment of their rows is two pieces and a wave's store or load
// of a piece is one contiguous run.
template <class P>
struct Piece {
  typedef __attribute__((ext_vector_type(4))) typename Feat<P>::T type;
};
template <class P>
__device__ __forceinline__ typename P::frag frag_pieces(const float* rec, size_t off, int ft, int jb, int lane) {
  const auto* pc = uni(reinterpret_cast<const typename Piece<P>::type*>(rec + off) + (ft * 4 + 2 * jb) * 64);
  return __builtin_shufflevector(pc[lane], pc[64 + lane], 0, 1, 2, 3, 4, 5, 6, 7);
}
// Q in fragment order [m 4][jb 16][lane].
template <class P>
__device__ __forceinline__ typename P::frag* qxf_area(float* rec) {
  if constexpr (IsBf16Policy<P>::value) return reinterpret_cast<typename P::frag*>(rec + Rec::KXF) + 64 * 64;
  else return reinterpret_cast<typename P::frag*>(rec + Rec::K);
}
template <class P>
__device__ __forceinline__ typename P::frag bf16_frag(const bf16x8& t) {
  if constexpr (IsBf16Policy<P>::value) {
    return t;
  } else {
    f32x8 r;
#pragma unroll
    for (int s = 0; s < 8; ++s) r[s] = (float)t[s];
    return r;
  }
}


// A fragment of Omega held in registers, converted at its use (held converted, fp32's would take twice as many).
template <class P>
__device__ __forceinline__ typename P::frag omega_reg(const bf16x8& t) {
  bf16x8 u = t;
  if constexpr (!IsBf16Policy<P>::value) asm volatile("" : "+v"(u));
  return bf16_frag<P>(u);
}

// Thread `tid` of 256 holds 16 consecutive features (tid & 3) * 16 .. of token row tid >> 2: loads the
// raw row part of x (zero past T), its L2 norm over the 64 features (shared by the four threads of the
// row), and the normalised part (x / max(|x|, 1e-6), or x itself without normalisation).
template <typename InT>
__device__ __forceinline__ float load_x_part(const InT* x, int64_t base, bool valid, int normalize, float* part) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) part[e] = 0.f;
  if (valid) {  // rows are 16-byte aligned (checked at the call)
    load8<InT>(x + base, part);
    load8<InT>(x + base + 8, part + 8);
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) ss += part[e] * part[e];
  ss += xor_shuffle<1>(ss);
  ss += xor_shuffle<2>(ss);
  const float nrm = sqrtf(ss);
  if (normalize) {
    const float inv = 1.f / fmaxf(nrm, 1e-6f);
#pragma unroll
    for (int e = 0; e < 16; ++e) part[e] *= inv;
  }
  return nrm;
}

// The normalised rows the lift consumes, as the forward lifts them: for bf16 inputs F.normalize keeps the
// dtype, so x^ is rounded to bf16; its products with the bf16-exact Omega are then exact on the bf16
// MFMA, and the pre-activations s equal the forward's.
template <typename InT>
__device__ __forceinline__ void round_like_input(int normalize, float* part) {
  if constexpr (std::is_same<InT, __bf16>::value) {
    if (normalize) {
#pragma unroll
      for (int e = 0; e < 16; ++e) part[e] = (float)(__bf16)part[e];
    }
  }
}

// ---------------------------------------------------------------------------------------------- prep
// grid (nch, H, B), 256 threads.
// LO: Omega has low parts (their products are added in the lift).
template <class P, typename InT, bool LO>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) bwd_prep_kernel(Params p) {
  // Four 64 x 64 tiles (71 KB with the vectors), so that two workgroups share a CU.
  __shared__ __attribute__((aligned(16))) float smem[4 * C * LD];
  float* xs = smem;               // normalised x rows; then beta o V; then dY
  float* bA = smem + C * LD;      // a o dY; later A
  float* bT = smem + 2 * C * LD;  // T
  float* bP = smem + 3 * C * LD;  // P
  // bT and bP are free during the lift: there each wave stages its 128 features of 32 token rows (bf16,
  // rows padded to 272 bytes against bank conflicts) to read them back as fragments
  constexpr int STG_ROW = 272, STG_WAVE = 32 * STG_ROW;
  static_assert(4 * STG_WAVE <= 2 * C * LD * (int)sizeof(float), "the lift's staging fits bT and bP");
  __shared__ float s_ell[C], s_beta[C], s_n[C], s_red[4][C];

  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = (p.c0 + blockIdx.x) * C;
  float* rec = record(p, b, h, blockIdx.x);
  const int r = tid >> 2, c0 = (tid & 3) * 16;
  const bool rvalid = t0 + r < p.T;

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
    rec[Rec::V_ELL + lane] = l;
    rec[Rec::V_BETA + lane] = be;
    rec[Rec::V_BG + lane] = p.linear ? 0.f : be * expf(l);
    rec[Rec::V_KAP + lane] = expf(__shfl(l, 63) - l);
  }
  {
    float dyp[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) dyp[e] = rvalid ? p.dy[b * p.ys0 + (t0 + r) * p.ys1 + h * p.ys2 + c0 + e] : 0.f;
    __syncthreads();
    const float a = r == 0 ? 1.f : expf(s_ell[r - 1]);
#pragma unroll
    for (int e = 0; e < 16; ++e) bA[r * LD + c0 + e] = a * dyp[e];
  }

  const float amp = sqrtf(2.f / D);
  const __bf16* om = p.omega + h * p.oms;
  const __bf16* oml = LO ? p.omega_lo + h * p.oms : nullptr;
  const float* phs = p.phase + h * p.phs;
  const float itau = head_inv_tau(p, h);
  // This wave's 128 rows of Omega and its phases, kept in registers for the four lifts below (q and k, two halves
  // of the tokens), instead of read in each of them, half a line of sixteen rows per load.  With the Grams below:
  // 4096 chunks, bf16, 586 -> 573 us; fp32 with low parts, 1024 chunks, 238 -> 216 us.  What bounds the kernel is the
  // record it writes, 380 KB a chunk in bf16.
  bf16x8 og[8][2];
  float phg[8];
#pragma unroll
  for (int ft = 0; ft < 8; ++ft) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
      og[ft][kb] = *reinterpret_cast<const bf16x8*>(om + (size_t)(128 * w + 16 * ft + (lane & 15)) * DK + 32 * kb + 8 * (lane >> 4));
    phg[ft] = phs[128 * w + 16 * ft + (lane & 15)];
  }
  for (int which = 0; which < 2; ++which) {  // 0: q, 1: k
    const InT* x = reinterpret_cast<const InT*>(which == 0 ? p.q : p.k);
    const int64_t xb = which == 0 ? b * p.qs0 + (t0 + r) * p.qs1 + h * p.qs2 : b * p.ks0 + (t0 + r) * p.ks1 + h * p.ks2;
    float part[16];
    load_x_part<InT>(x, xb + c0, rvalid, p.normalize, part);
    round_like_input<InT>(p.normalize, part);
#pragma unroll
    for (int e = 0; e < 16; ++e) xs[r * LD + c0 + e] = part[e];
    // The barriers of the lift order LDS only: the record stores issued in it drain in the background
    // (once, at the fence after the lift) instead of at every barrier.
    lds_barrier();

    // phi~ (tokens x this wave's 128 features), in two halves of 32 tokens: tile [ft][u] holds rows
    // token 16 (2 hm + u) + .., column feature.
    typename Feat<P>::T* phi = feat<P>(rec, which == 0 ? Rec::Q : Rec::K);
    for (int hm = 0; hm < 2; ++hm) {
      f32x4 acc[8][2];
      typename P::frag xa[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) xa[u][jb] = P::from_f32(frag_rows_plain(xs, LD, 16 * (2 * hm + u), 32 * jb, lane));
      float ss[2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) ss[u][i] = 0.f;
#pragma unroll
      for (int ft = 0; ft < 8; ++ft) {
        const int f0 = 128 * w + 16 * ft;
        const typename P::frag o0 = omega_reg<P>(og[ft][0]), o1 = omega_reg<P>(og[ft][1]);
        const float ph = phg[ft];
        f32x8 l0 = {}, l1 = {};
        if constexpr (LO) {  // the low parts: their products are added like the forward's
          l0 = frag_rows_plain_bf16(oml, DK, f0, 0, lane);
          l1 = frag_rows_plain_bf16(oml, DK, f0, 32, lane);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4 sv = P::mma(P::mma(zero4(), xa[u][0], o0), xa[u][1], o1);
          if constexpr (LO) sv = P::mma(P::mma(sv, xa[u][0], P::from_f32(l0)), xa[u][1], P::from_f32(l1));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = amp * cos_rad(sv[i] * itau + ph);
            sv[i] = v;
            ss[u][i] += v * v;
          }
          acc[ft][u] = sv;
        }
        __builtin_amdgcn_sched_barrier(0);  // one feature tile per scheduling region (no operand hoisting)
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = sum_row16(ss[u][i]);
          if ((lane & 15) == 0) s_red[w][32 * hm + 16 * u + 4 * (lane >> 4) + i] = v;
        }
      lds_barrier();
      if (tid < 32) {
        const int row = 32 * hm + tid;
        const float n = sqrtf(s_red[0][row] + s_red[1][row] + s_red[2][row] + s_red[3][row]);
        s_n[row] = n;
        rec[Rec::V_NORM + 64 * which + row] = n;
      }
      lds_barrier();
      // The normalised tiles: the q^T / k^T fragments of depth block hm straight from the registers (an
      // accumulator tile pair [ft][0..1] is the fragment of feature tile ft, tokens 32 hm + kappa), and
      // the row fragments (fp32 features: the rows, packed below).
      {
        using frag = typename P::frag;
        frag* tf = reinterpret_cast<frag*>(rec + (which == 0 ? Rec::QTF : Rec::KTF));
        f32x4 sc[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = 32 * hm + 16 * u + 4 * (lane >> 4) + i;
            sc[u][i] = (t0 + row < p.T) ? (p.no_renorm ? 1.f : 1.f / (s_n[row] + 1e-8f)) : 0.f;
          }
#pragma unroll
        for (int ft = 0; ft < 8; ++ft) {
          acc[ft][0] = acc[ft][0] * sc[0];
          acc[ft][1] = acc[ft][1] * sc[1];
          tf[((8 * w + ft) * 2 + hm) * 64 + lane] = P::from_f32(pair_to8(acc[ft][0], acc[ft][1]));
        }
        if constexpr (IsBf16Policy<P>::value) {
          // rows through this wave's staging area, read back as fragments
          unsigned char* stg = reinterpret_cast<unsigned char*>(bT) + w * STG_WAVE;
#pragma unroll
          for (int ft = 0; ft < 8; ++ft)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                *reinterpret_cast<__bf16*>(stg + (16 * u + 4 * (lane >> 4) + i) * STG_ROW + 2 * (16 * ft + (lane & 15))) =
                    (__bf16)acc[ft][u][i];
          wave_lds_sync();
          {
            // K packed in fragment order for the chains, from the same staging rows: token tiles
            // 2 hm, 2 hm + 1, feature blocks 4w .. 4w + 3 (lane: row l & 15, features kappa(l, 0..7));
            // Q likewise for the Grams below and the gradient launch (QXF)
            typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
            frag* kxf = which == 0 ? qxf_area<P>(rec) : reinterpret_cast<frag*>(rec + Rec::KXF);
#pragma unroll
            for (int mu = 0; mu < 2; ++mu)
#pragma unroll
              for (int jj = 0; jj < 4; ++jj) {
                const unsigned char* q = stg + (16 * mu + (lane & 15)) * STG_ROW + 2 * (32 * jj + 4 * (lane >> 4));
                const bf16x4 lo = *reinterpret_cast<const bf16x4*>(q);
                const bf16x4 hi = *reinterpret_cast<const bf16x4*>(q + 32);
                kxf[((2 * hm + mu) * 16 + 4 * w + jj) * 64 + lane] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
              }
          }
          wave_lds_sync();
        } else {
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int row = 32 * hm + 16 * u + 4 * (lane >> 4) + i;
#pragma unroll
              for (int ft = 0; ft < 8; ++ft) phi[(size_t)row * D + 128 * w + 16 * ft + (lane & 15)] = acc[ft][u][i];
            }
        }
      }
    }
    lds_barrier();
  }
  // The Grams below read the features this workgroup just wrote to the record: a workgroup-scope release /
  // acquire (__syncthreads) orders them.  A device-scope fence here wrote back and invalidated the whole
  // L2 in every workgroup (recompute 365 -> 213 us per segment launch without it).
  __syncthreads();

  // K packed in fragment order for the chains: wave w the K-row fragments of feature blocks 4w .. 4w+3
  // (the K^T fragments went to the record during the lift; with bf16 features these too, from the
  // lift's staging rows).
  if constexpr (!IsBf16Policy<P>::value) {
    using frag = typename P::frag;
    const typename Feat<P>::T* K = feat<P>(rec, Rec::K);
    frag* kxf = reinterpret_cast<frag*>(rec + Rec::KXF);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) kxf[(m * 16 + 4 * w + jj) * 64 + lane] = frag_rows_p<P>(K, D, 16 * m, 32 * (4 * w + jj), lane);
  }

  // a o dY as the B fragments of H = Q^T (a o dY), which the reverse carry forms per chunk from these and
  // the Q^T fragments (wave w: value tile w)
  {
    using frag = typename P::frag;
    frag* ayf = reinterpret_cast<frag*>(rec + Rec::AYF);
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) ayf[(w * 2 + jb) * 64 + lane] = P::from_f32(frag_cols(bA, LD, 16 * w, 32 * jb, lane));
  }
  __syncthreads();  // a o dY in bA is dead from here on (bA becomes A below)

  // Gram matrices: each wave the products over its 128 features of the tiles on and below the diagonal, from the
  // fragments it has just written (one contiguous 16- or 32-byte piece per lane; Q from its rows with fp32
  // features), the four waves' parts added in LDS; A and P into LDS.  A row tile per wave over all features read
  // every fragment of K in every wave, 384 KB a chunk.
  {
    using frag = typename P::frag;
    const typename Feat<P>::T* Q = feat<P>(rec, Rec::Q);
    const frag* kxf = reinterpret_cast<const frag*>(rec + Rec::KXF);
    f32x4 gkk[10], gqk[10];
#pragma unroll
    for (int t = 0; t < 10; ++t) gkk[t] = gqk[t] = zero4();
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int jb = 4 * w + jj;
      frag kf[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) kf[m] = kxf[(m * 16 + jb) * 64 + lane];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        frag qf, *fq = qxf_area<P>(rec) + (m * 16 + jb) * 64 + lane;
        if constexpr (IsBf16Policy<P>::value) {
          qf = *fq;
        } else {  // Q's rows into fragment order over the k rows, which every wave has packed by now
          qf = frag_rows_p<P>(Q, D, 16 * m, 32 * jb, lane);
          *fq = qf;
        }
#pragma unroll
        for (int n = 0; n <= m; ++n) {
          gkk[m * (m + 1) / 2 + n] = P::mma(gkk[m * (m + 1) / 2 + n], kf[m], kf[n]);
          gqk[m * (m + 1) / 2 + n] = P::mma(gqk[m * (m + 1) / 2 + n], qf, kf[n]);
        }
      }
    }
    // 40 partial tiles of 1 KB: 17 fit xs, the rest bT and bP
    static_assert(17 * 256 <= C * LD && 23 * 256 <= 2 * C * LD, "the partial Grams fit");
    auto part = [&](int t, int v) {
      const int u = v * 10 + t;
      return reinterpret_cast<f32x4*>(u < 17 ? xs + u * 256 : bT + (u - 17) * 256) + lane;
    };
    auto total = [&](int t) { return ((*part(t, 0) + *part(t, 1)) + *part(t, 2)) + *part(t, 3); };
    auto tile_m = [](int t) { return t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3; };
#pragma unroll
    for (int t = 0; t < 10; ++t) *part(t, w) = gkk[t];
    for (int idx = tid; idx < C * C; idx += 256) bA[idx] = 0.f;
    lds_barrier();
    for (int t = w; t < 10; t += 4) {
      const int m = tile_m(t), n = t - m * (m + 1) / 2;
      const f32x4 g = total(t);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * m + 4 * (lane >> 4) + i, cj = 16 * n + (lane & 15);
        rec[Rec::GKK + ri * C + cj] = g[i];
        // A transposed for the column-oriented inverse below: [j][p][s] = A[4s+p][j]
        // (the linear rule has no erasure coupling: A = 0, so T = I and Tp = 0 below)
        if (cj < ri && !p.linear) bA[(cj * 4 + (ri & 3)) * 16 + (ri >> 2)] = s_beta[ri] * expf(fminf(s_ell[ri] - s_ell[cj], 0.f)) * g[i];
      }
    }
    lds_barrier();
#pragma unroll
    for (int t = 0; t < 10; ++t) *part(t, w) = gqk[t];
    lds_barrier();
    f32x4 pt[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) pt[k] = w + 4 * k < 10 ? total(w + 4 * k) : zero4();
    lds_barrier();
    for (int idx = tid; idx < C * LD; idx += 256) bP[idx] = 0.f;
    lds_barrier();
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int t = w + 4 * k, m = tile_m(t), n = t - m * (m + 1) / 2;
      if (t < 10) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ri = 16 * m + 4 * (lane >> 4) + i, cj = 16 * n + (lane & 15);
          if (cj < ri) bP[ri * LD + cj] = expf(fminf((ri > 0 ? s_ell[ri - 1] : 0.f) - s_ell[cj], 0.f)) * pt[k][i];
        }
      }
    }
  }
  __syncthreads();
  // T = (I + A)^-1 (column-oriented substitution over lane quads)
  unit_lower_inverse(bA, bT, LD, w, lane);
  __syncthreads();
  for (int idx = tid; idx < C * C; idx += 256) {
    const int i = idx >> 6, j = idx & 63;
    rec[Rec::T + idx] = bT[i * LD + j];
    rec[Rec::P + idx] = bP[i * LD + j];
  }
  if constexpr (IsBf16Policy<P>::value) {
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      f32x8 tp = frag_rows(bT, LD, 16 * w, 32 * jb, lane);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int j = 32 * jb + kappa(lane, s);
        tp[s] = p.linear ? 0.f : tp[s] * s_beta[j] * expf(s_ell[j]);
      }
      reinterpret_cast<f32x8*>(rec + Rec::TPF)[(w * 2 + jb) * 64 + lane] = tp;
    }
  }
  {
    const int j = 16 * w + (lane & 15);
    const float be = p.linear ? 0.f : s_beta[j], g = expf(s_ell[j]);
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
      reinterpret_cast<f32x8*>(rec + Rec::TPT)[(w * 2 + jb) * 64 + lane] = frag_cols(bT, LD, 16 * w, 32 * jb, lane) * be * g;
  }
  {
    const InT* v = reinterpret_cast<const InT*>(p.v);
    const int64_t vb = b * p.vs0 + (t0 + r) * p.vs1 + h * p.vs2 + c0;
    const float be = s_beta[r];
#pragma unroll
    for (int e = 0; e < 16; ++e) xs[r * LD + c0 + e] = rvalid ? be * ldx(v + vb + e) : 0.f;
  }
  __syncthreads();
  // U~ = T (beta o V) (row tile w)
  {
    const f32x8 ta0 = frag_rows(bT, LD, 16 * w, 0, lane), ta1 = frag_rows(bT, LD, 16 * w, 32, lane);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const f32x4 u = mm<PrecF32>(mm<PrecF32>(zero4(), ta0, frag_cols(xs, LD, 16 * n, 0, lane)), ta1, frag_cols(xs, LD, 16 * n, 32, lane));
      reinterpret_cast<f32x4*>(rec + Rec::U)[(w * 4 + n) * 64 + lane] = u;
    }
  }
  __syncthreads();  // beta o V is dead: dY again (the same fp32 values) in its place
#pragma unroll
  for (int e = 0; e < 16; ++e)
    xs[r * LD + c0 + e] = rvalid ? p.dy[b * p.ys0 + (t0 + r) * p.ys1 + h * p.ys2 + c0 + e] : 0.f;
  __syncthreads();
  // R = P^T dY (row tile w)
  {
    const f32x8 pa0 = frag_cols(bP, LD, 16 * w, 0, lane), pa1 = frag_cols(bP, LD, 16 * w, 32, lane);
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const f32x4 rr = mm<PrecF32>(mm<PrecF32>(zero4(), pa0, frag_cols(xs, LD, 16 * n, 0, lane)), pa1, frag_cols(xs, LD, 16 * n, 32, lane));
      reinterpret_cast<f32x4*>(rec + Rec::R)[(w * 4 + n) * 64 + lane] = rr;
    }
  }
}

// --------------------------------------------------------------------------------------------- chain
// grid: 8 * ceil(B*H / 8) * 4 workgroups of CHAIN_WAVES waves; workgroup (head-batch hb, value tile n) with
// the four value tiles of a head on one XCD.  Wave w keeps features 64w .. 64w+63 of its 512 x 16 slice of
// the carried matrix (S^T forward, Gamma backward) in registers.
//
// Per chunk: store the slice (chunk start S^T / chunk end Gamma); X = K Sigma (partial over the wave's
// features, reduced through LDS by waves 0..3, one token tile each); forward W = U~ - Tp X_K and
// Z = kappa o W, reverse dW = R + kappa o X and Z = -Tp^T dW; Sigma <- g_C Sigma (+ H) + K^T Z.
//
// What bounds a step: the CU takes one 128-byte line from L2 every four to six cycles, so the lines a step
// loads (K 64 KB, in reverse Q^T 64 KB; K^T is formed from K on the matrix cores, 16 products with the
// identity) and the latency of those that miss L2; then the chain of its three barriers with the 64-deep
// fp32 product of Tp (512 cycles) between them.  Loads of a wave complete in issue order, so every operand
// of chunk c + 1 is issued where its registers come free in step c, a step ahead of its use, and waves 4..7,
// which wait for the reduction and the Tp product, pull chunk c + CHAIN_AHEAD's lines into L2.  Eight waves
// of 64 features put two on a SIMD; the slice goes out as 8-byte pieces (transposed exactly, again by
// products with the identity) and whole fragments.  16 heads, 256 chunks, us per carry, forward / reverse:
// 706 / 948; without the prefetch 856 / 1111; K^T loaded 896 / 899; loads at the top of the step 1175 / 1115;
// four waves of 128 features with 32 two-byte stores a lane 1051 / 1351.  With L2 always hit: 644 / 645.
// The barriers order the LDS exchange only (no wave reads another's global writes within a step), so
// the loads issued ahead and the stores of the step stay in flight across them.
constexpr int CHAIN_WAVES = 8;
constexpr int CHAIN_AHEAD = 3;  // chunks between a step and the operands it pulls into L2
struct ChainShared {
  f32x4 xp[CHAIN_WAVES][4][64];
  f32x4 x[4][64];
  f32x4 z[4][64];
};

// A chunk's operands of one wave, in registers.
template <class P, bool REV>
struct ChainOps {
  using frag = typename P::frag;
  // fp32 fragments take twice the registers: K's and Q^T's then share theirs, each loaded where the other is
  // used up, the Q^T of a chunk inside its step
  static constexpr bool SHARE = REV && !IsBf16Policy<P>::value;
  frag kx[4][2];              // K rows 16m .., features 64w + 32jj ..
  frag kt[4][2];              // K^T rows 64w + 16t .., tokens 32jb ..
  frag qt[REV ? 4 : 1][2];    // Q^T likewise, and a o dY (reverse)
  frag y[2];
  // waves 0..3: row tile w of Tp or Tp^T; with fp32 features, whose record has no room for Tp's fragments, the
  // forward carry takes T's rows and scales them by beta g
  static constexpr bool SCALE = !REV && !IsBf16Policy<P>::value;
  f32x8 tp[2];
  f32x4 bg[SCALE ? 4 : 1];    // beta g
  f32x4 ur, kap;              // U~ or R, kappa
  float l63;

  __device__ __forceinline__ void load_kx(const float* rec, int w, int lane) {
    const frag* f = reinterpret_cast<const frag*>(rec + Rec::KXF);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) kx[m][jj] = uni(f + (m * 16 + 2 * w + jj) * 64)[lane];
  }
  __device__ __forceinline__ void load_kt(const float* rec, int w, int lane) {
    const frag* f = reinterpret_cast<const frag*>(rec + Rec::KTF);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) kt[t][jb] = uni(f + ((4 * w + t) * 2 + jb) * 64)[lane];
  }
  // The same from kx with bf16 features: a K fragment times the identity has the accumulator layout of K^T
  // columns, two token tiles of it are a K^T fragment (the values exactly).
  __device__ __forceinline__ void transpose_k(const frag (&eye)[2]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      __builtin_amdgcn_sched_barrier(0);  // four products' results at a time
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        kt[t][jb] = P::from_f32(pair_to8(P::mma(zero4(), kx[2 * jb][t >> 1], eye[t & 1]), P::mma(zero4(), kx[2 * jb + 1][t >> 1], eye[t & 1])));
        asm volatile("" : "+v"(kt[t][jb]));  // packed here, not at its use
      }
    }
  }
  __device__ __forceinline__ void load_q(const float* rec, int w, int n, int lane) {
    if constexpr (REV) {
      const frag* fy = reinterpret_cast<const frag*>(rec + Rec::AYF);
      const frag* f = reinterpret_cast<const frag*>(rec + Rec::QTF);
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) y[jb] = uni(fy + (n * 2 + jb) * 64)[lane];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) qt[t][jb] = uni(f + ((4 * w + t) * 2 + jb) * 64)[lane];
    }
  }
  __device__ __forceinline__ void load_lead(const float* rec, int w, int n, int lane) {
    if constexpr (!SCALE) {
      const f32x8* f = reinterpret_cast<const f32x8*>(rec + (REV ? Rec::TPT : Rec::TPF));
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) tp[jb] = uni(f + (w * 2 + jb) * 64)[lane];
    } else {
      const float* t = uni(rec + Rec::T + 16 * w * C);
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) tp[jb] = frag_rows(t, C, 0, 32 * jb, lane);
      const f32x4* vb = reinterpret_cast<const f32x4*>(uni(rec + Rec::V_BG));
#pragma unroll
      for (int k = 0; k < 4; ++k) bg[k] = vb[4 * k + (lane >> 4)];
    }
    ur = uni(reinterpret_cast<const f32x4*>(rec + (REV ? Rec::R : Rec::U)) + (w * 4 + n) * 64)[lane];
    kap = reinterpret_cast<const f32x4*>(uni(rec + Rec::V_KAP + 16 * w))[lane >> 4];
  }
  __device__ __forceinline__ void load_l63(const float* rec) { l63 = uni(rec + Rec::V_ELL + 63)[0]; }
};

// One dword of each 128-byte line of a later chunk's operands, shared out over waves 4..7 of the head's four
// workgroups (1024 lanes): pulls them into the XCD's L2.
template <class P, bool REV>
struct ChainPrefetch {
  static constexpr int AREA = 4096 * (int)sizeof(typename P::frag) / 128;  // lines of a K, K^T or Q^T area
  static constexpr int KT = IsBf16Policy<P>::value ? 0 : AREA;             // K^T is loaded with fp32 features only
  static constexpr int E0 = AREA, E1 = E0 + KT, E2 = E1 + (REV ? AREA : 0), E3 = E2 + 128, E4 = E3 + 128, E5 = E4 + 16;
  static constexpr int LINES = E5 + (REV ? 4 * (int)sizeof(typename P::frag) : 0);
  static constexpr int PER = (LINES + 1023) / 1024;
  unsigned v[PER];  // the loaded words: used, and so waited for, only where the next step replaces them
  __device__ __forceinline__ void load(const float* rec, int n, int w, int lane) {
    const unsigned* r = reinterpret_cast<const unsigned*>(uni(rec));
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = (n * 4 + (w - 4)) * 64 + lane + 1024 * k;
      unsigned at = Rec::VEC;
      if (i < E0) at = Rec::KXF + 32 * i;
      else if (i < E1) at = Rec::KTF + 32 * (i - E0);
      else if (i < E2) at = Rec::QTF + 32 * (i - E1);
      else if (i < E3) at = (REV ? Rec::TPT : ChainOps<P, REV>::SCALE ? Rec::T : Rec::TPF) + 32 * (i - E2);
      else if (i < E4) at = (REV ? Rec::R : Rec::U) + 32 * (i - E3);
      else if (i < E5) at = Rec::VEC + 32 * (i - E4);
      else if (REV && i < LINES) at = Rec::AYF + 32 * (i - E5);
      v[k] = r[at];
    }
  }
};

template <class P, bool REV>
__device__ __forceinline__ void chain_step(ChainShared& sh, float* rec, const float* nrec, const float* frec, ChainOps<P, REV>& o,
                                           ChainPrefetch<P, REV>& pf, unsigned& sink,
                                           f32x4 (&Sg)[4], const typename P::frag (&eye)[2], int w, int lane, int n) {
  using frag = typename P::frag;
  using piece = typename Piece<P>::type;
  const bool lead = w < 4;
  constexpr bool SHARE = ChainOps<P, REV>::SHARE;
  // K times the carried slice, partial over this wave's features
  frag sb[2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) sb[jj] = P::from_f32(pair_to8(Sg[2 * jj], Sg[2 * jj + 1]));
  f32x4 xp[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) xp[m] = P::mma(zero4(), o.kx[m][0], sb[0]);
#pragma unroll
  for (int m = 0; m < 4; ++m) xp[m] = P::mma(xp[m], o.kx[m][1], sb[1]);
#pragma unroll
  for (int m = 0; m < 4; ++m) sh.xp[w][m][lane] = xp[m];
  // the old slice is dead past the products above (sb holds what is stored): apply g_C now
  const float gC = expf(o.l63);
  f32x4 old[IsBf16Policy<P>::value ? 1 : 4];
  if constexpr (!IsBf16Policy<P>::value) {
#pragma unroll
    for (int t = 0; t < 4; ++t) old[t] = Sg[t];
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) Sg[t] = Sg[t] * gC;
  __builtin_amdgcn_sched_barrier(0);
  if (IsBf16Policy<P>::value && lead) {
    o.transpose_k(eye);
    __builtin_amdgcn_sched_barrier(0);
    o.load_kx(nrec, w, lane);
  }
  if constexpr (!IsBf16Policy<P>::value) {
    if constexpr (SHARE) o.load_q(rec, w, n, lane);
    else o.load_kx(nrec, w, lane);
  }
  o.load_l63(nrec);

  // the slice to the record: pieces of its rows (both carries), B fragments (forward)
  {
    piece* dst = reinterpret_cast<piece*>(rec + (REV ? Rec::G : Rec::S));
    if constexpr (IsBf16Policy<P>::value) {
      // D = Sigma^T-tile x identity: lane (feature l & 15, values 4 (l >> 4) + i), the bf16 values exactly
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f32x4 d = P::mma(zero4(), sb[t >> 1], eye[t & 1]);
        piece v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (typename Feat<P>::T)d[i];
        uni(dst + ((4 * w + t) * 4 + n) * 64)[lane] = v;
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          reinterpret_cast<typename Feat<P>::T*>(uni(dst + ((4 * w + t) * 4 + n) * 64))[(4 * (lane >> 4) + i + 16 * ((lane & 15) >> 2)) * 4 + (lane & 3)] = old[t][i];
    }
    if constexpr (!REV) {
      frag* sf = reinterpret_cast<frag*>(rec + Rec::Q);
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) uni(sf + (n * 16 + 2 * w + jj) * 64)[lane] = sb[jj];
    }
  }
  lds_barrier();
  if (lead) {
    f32x4 X = sh.xp[0][w][lane];
#pragma unroll
    for (int v = 1; v < CHAIN_WAVES; ++v) X += sh.xp[v][w][lane];
    if constexpr (!REV) {
      sh.x[w][lane] = X;
      uni(reinterpret_cast<f32x4*>(rec + Rec::XK) + (w * 4 + n) * 64)[lane] = X;
    } else {
      const f32x4 dW = o.ur + o.kap * X;
      sh.x[w][lane] = dW;
      uni(reinterpret_cast<f32x4*>(rec + Rec::X) + (w * 4 + n) * 64)[lane] = X;
      uni(reinterpret_cast<f32x4*>(rec + Rec::DW) + (w * 4 + n) * 64)[lane] = dW;
    }
  } else if constexpr (IsBf16Policy<P>::value) {
    o.transpose_k(eye);
    __builtin_amdgcn_sched_barrier(0);
    o.load_kx(nrec, w, lane);
  }
  lds_barrier();
  if (lead) {
    const f32x8 x0 = pair_to8(sh.x[0][lane], sh.x[1][lane]), x1 = pair_to8(sh.x[2][lane], sh.x[3][lane]);
    if constexpr (ChainOps<P, REV>::SCALE) {
      o.tp[0] = o.tp[0] * pair_to8(o.bg[0], o.bg[1]);
      o.tp[1] = o.tp[1] * pair_to8(o.bg[2], o.bg[3]);
    }
    const f32x4 t = mm<PrecF32>(mm<PrecF32>(zero4(), o.tp[0], x0), o.tp[1], x1);
    if constexpr (!REV) {
      const f32x4 Wt = o.ur - t;
      sh.z[w][lane] = o.kap * Wt;
      uni(reinterpret_cast<f32x4*>(rec + Rec::W) + (w * 4 + n) * 64)[lane] = Wt;
    } else {
      sh.z[w][lane] = -t;
    }
    __builtin_amdgcn_sched_barrier(0);
    o.load_lead(nrec, w, n, lane);
  } else if (frec) {
#pragma unroll
    for (int k = 0; k < ChainPrefetch<P, REV>::PER; ++k) sink ^= pf.v[k];
    pf.load(frec, n, w, lane);
  }
  if constexpr (REV) {
    // this wave's rows of H = Q^T (a o dY) for value tile n, added to the carry
#pragma unroll
    for (int t = 0; t < 4; ++t) Sg[t] = Sg[t] + P::mma(P::mma(zero4(), o.qt[t][0], o.y[0]), o.qt[t][1], o.y[1]);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SHARE) o.load_kx(nrec, w, lane);
    else o.load_q(nrec, w, n, lane);
  }
  lds_barrier();
  const frag zb0 = P::from_f32(pair_to8(sh.z[0][lane], sh.z[1][lane]));
  const frag zb1 = P::from_f32(pair_to8(sh.z[2][lane], sh.z[3][lane]));
#pragma unroll
  for (int t = 0; t < 4; ++t) Sg[t] = P::mma(P::mma(Sg[t], o.kt[t][0], zb0), o.kt[t][1], zb1);
  if constexpr (!IsBf16Policy<P>::value) {
    __builtin_amdgcn_sched_barrier(0);
    o.load_kt(nrec, w, lane);
  }
}

// The carry of workgroup `id` of a chain grid.
template <class P, bool REV>
__device__ __forceinline__ void chain_body(const Params& p, ChainShared& sh, int64_t id) {
  using frag = typename P::frag;
  const int64_t xcd = id & 7, jdx = id >> 3;
  const int n = (int)(jdx & 3);
  const int64_t hb = (jdx >> 2) * 8 + xcd;
  if (hb >= p.B * p.H) return;
  // the division is done in vector registers: back to scalars, so that every record address is one
  const int b = __builtin_amdgcn_readfirstlane((int)(hb / p.H));
  const int h = (int)hb - b * (int)p.H;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vc = 16 * n + (lane & 15);

  f32x4 Sg[4];
  {
    const float* src = REV ? p.dfin : p.init;
    const int64_t s0 = REV ? p.fs0 : p.is0, s1 = REV ? p.fs1 : p.is1, s2 = REV ? p.fs2 : p.is2, s3 = REV ? p.fs3 : p.is3;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int f = 64 * w + 16 * t + 4 * (lane >> 4) + i;
        Sg[t][i] = src ? src[b * s0 + h * s1 + f * s2 + vc * s3] : 0.f;
      }
  }
  // the two halves of a 32 x 32 identity as B fragments: depth kappa(l, s), column 16 k + (l & 15)
  frag eye[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    f32x8 e;
#pragma unroll
    for (int s = 0; s < 8; ++s) e[s] = kappa(lane, s) == 16 * k + (lane & 15) ? 1.f : 0.f;
    eye[k] = P::from_f32(e);
  }
  const int nseg = (int)p.nseg;
  ChainOps<P, REV> o;
  {
    const float* rec = record(p, b, h, REV ? nseg - 1 : 0);
    o.load_kx(rec, w, lane);
    o.load_l63(rec);
    if (w < 4) o.load_lead(rec, w, n, lane);
    if constexpr (!ChainOps<P, REV>::SHARE) o.load_q(rec, w, n, lane);
    if constexpr (!IsBf16Policy<P>::value) o.load_kt(rec, w, lane);
  }
  ChainPrefetch<P, REV> pf = {};
  unsigned sink = 0;  // keeps the prefetch loads alive (never stored: nseg is positive)
  for (int step = 0; step < nseg; ++step) {
    const int c = REV ? nseg - 1 - step : step;
    const int cn = step + 1 < nseg ? (REV ? c - 1 : c + 1) : c;  // the last step loads its own chunk again
    const int cf = REV ? c - CHAIN_AHEAD : c + CHAIN_AHEAD;
    chain_step<P, REV>(sh, record(p, b, h, c), record(p, b, h, cn), cf >= 0 && cf < nseg ? record(p, b, h, cf) : nullptr, o,
                       pf, sink, Sg, eye, w, lane, n);
  }
  if (p.nseg < 0) p.ws[0] = (float)sink;
  if constexpr (REV) {
    // dL/dS^T at the segment start: the next (earlier) segment's reverse carry starts from it; this
    // thread rewrites exactly the elements it read at the top when both are the segment carry
    if (p.gout) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int f = 64 * w + 16 * t + 4 * (lane >> 4) + i;
          p.gout[b * p.gos0 + h * p.gos1 + f * p.gos2 + vc * p.gos3] = Sg[t][i];
        }
    }
  }
}

template <class P, bool REV>
__global__ void __launch_bounds__(64 * CHAIN_WAVES) bwd_chain_kernel(Params p) {
  __shared__ ChainShared sh;
  chain_body<P, REV>(p, sh, blockIdx.x);
}

// Both carries of a segment in one launch: workgroups below `half` carry S^T forward, the others dL/dS^T
// backward (each reads only what the recompute wrote and they write disjoint fields).  `half` is a
// multiple of 8, so both halves keep the XCD mapping of a single carry.
template <class P>
__global__ void __launch_bounds__(64 * CHAIN_WAVES) bwd_chains_kernel(Params p, unsigned half) {
  __shared__ ChainShared sh;
  if (blockIdx.x < half) chain_body<P, false>(p, sh, blockIdx.x);
  else chain_body<P, true>(p, sh, blockIdx.x - half);
}

// ---------------------------------------------------------------------------------------------- grad
// Thread (row r, features c0 .. c0 + 15): dx = inv_tau * dx^ through the input normalisation, dx^ the sum of
// two partials, written for tokens before T.
template <typename InT>
__device__ __forceinline__ void write_dx(const Params& p, const InT* x, int64_t xbase, float* out, int64_t obase,
                                         const float* dx0, const float* dx1, int r, int c0, bool valid, float itau) {
  float part[16];
  const float nrm = load_x_part<InT>(x, xbase, valid, p.normalize, part);
  float g[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) g[e] = itau * (dx0[r * LD + c0 + e] + dx1[r * LD + c0 + e]);
  if (p.normalize) {
    float dot = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) dot += part[e] * g[e];
    dot += xor_shuffle<1>(dot);
    dot += xor_shuffle<2>(dot);
    if (nrm > 1e-6f) {
      const float inv = 1.f / nrm;
#pragma unroll
      for (int e = 0; e < 16; ++e) g[e] = (g[e] - part[e] * dot) * inv;
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) g[e] *= 1e6f;
    }
  }
  if (valid) {
    float* o = out + obase;
    if ((reinterpret_cast<uintptr_t>(o) & 15) == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4 v = {g[4 * e], g[4 * e + 1], g[4 * e + 2], g[4 * e + 3]};
        reinterpret_cast<f32x4*>(o)[e] = v;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) o[e] = g[e];
    }
  }
}

// grid (nseg, H, B), GRAD_WAVES waves.  Wave w: row tile rt = w & 3, column tiles 2 ch .. 2 ch + 1 with
// ch = w >> 2 (the first four waves also load the tiles and the per-row terms).
template <class P, typename InT>
__global__ void __launch_bounds__(64 * GRAD_WAVES) bwd_grad_kernel(Params p) {
  __shared__ __attribute__((aligned(16))) float bY[C * LD];   // dY, then a o dY
  __shared__ __attribute__((aligned(16))) float bW[C * LD];   // W, then kappa o W
  __shared__ __attribute__((aligned(16))) float bdW[C * LD];  // dW, then Zn = -Tp^T dW
  __shared__ __attribute__((aligned(16))) float bXK[C * LD];  // X_K, then N
  __shared__ __attribute__((aligned(16))) float bX[C * LD];   // X, then dT, then M + M^T
  __shared__ __attribute__((aligned(16))) float bV[C * LD];   // V, then Y1 = dT T^T
  __shared__ __attribute__((aligned(16))) float bT[C * LD];   // T
  __shared__ float s_ell[C], s_beta[C];
  // Fixed-order reductions (the gradients do not depend on the order the waves run in): every partial
  // sum has a slot of its own, written once, and the slots are added in a fixed order; no atomics.
  //   s_dlp: contributions to dl_i = dL/dl_i (rows DL_*); s_dbp: to dbeta_i (rows DB_*);
  //   s_tsp: column sums of T o dTp per row tile;
  //   s_w63: sums that land on dl_63: the dkappa term per row tile [0..3], <Gamma, S> per wave [4..11]
  //   s_da0: the a o dY . Q S^T term of row 0 (a_0 = 1 is no decay: only phi . dphi takes it)
  __shared__ float s_dlp[NDL][C], s_dbp[NDB][C], s_tsp[4][C], s_w63[4 + GRAD_WAVES], s_da0[2];

  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rt = w & 3, ch = w >> 2;
  const int64_t t0 = (p.c0 + blockIdx.x) * C;
  float* rec = record(p, b, h, blockIdx.x);
  const int r = (tid >> 2) & 63, c0 = (tid & 3) * 16;  // loaders (tid < 256): row r, columns c0 .. c0 + 15
  const bool rvalid = t0 + r < p.T;

  if (tid < C) {
    s_ell[tid] = rec[Rec::V_ELL + tid];
    s_beta[tid] = rec[Rec::V_BETA + tid];
  }
  if (tid == 0)  // the only slots no source writes
    s_dlp[DL_RP][63] = s_dlp[DL_RP + 1][63] = s_dlp[DL_DA][63] = s_dlp[DL_DA + 1][63] = 0.f;
  if (tid < 256) {
    const InT* v = reinterpret_cast<const InT*>(p.v);
    const int64_t vb = b * p.vs0 + (t0 + r) * p.vs1 + h * p.vs2 + c0;
    const int64_t yb = b * p.ys0 + (t0 + r) * p.ys1 + h * p.ys2 + c0;
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4)
      *reinterpret_cast<f32x4*>(&bT[r * LD + c0 + 4 * e4]) = *reinterpret_cast<const f32x4*>(rec + Rec::T + r * C + c0 + 4 * e4);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int o = r * LD + c0 + e;
      bY[o] = rvalid ? p.dy[yb + e] : 0.f;
      bV[o] = rvalid ? ldx(v + vb + e) : 0.f;
    }
  }
  // W, dW, X_K, X: tiles of the chains (row tile rt, column tiles 2 ch, 2 ch + 1) into rows
#pragma unroll
  for (int nn = 0; nn < 2; ++nn) {
    const int n = 2 * ch + nn;
    auto tile = [&](size_t off, float* dst) {
      const f32x4 v = reinterpret_cast<const f32x4*>(rec + off)[(rt * 4 + n) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[(16 * rt + 4 * (lane >> 4) + i) * LD + 16 * n + (lane & 15)] = v[i];
    };
    tile(Rec::W, bW);
    tile(Rec::DW, bdW);
    tile(Rec::XK, bXK);
    tile(Rec::X, bX);
  }
  __syncthreads();
  const float l63 = s_ell[63], gC = expf(l63);

  // ---- phase 1: dkappa; T^T dW -> dv, dbeta; dTp, dT; dP -> N
  if (tid < 256) {
    float dkp = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) dkp += bW[r * LD + c0 + e] * bX[r * LD + c0 + e];
    dkp += __shfl_xor(dkp, 1);
    dkp += __shfl_xor(dkp, 2);
    const float t = dkp * expf(l63 - s_ell[r]);  // the same in the four threads of row r
    if ((tid & 3) == 0) s_dlp[DL_KAPPA][r] = -t;
    const float tw = sum_col4(sum_row16((tid & 3) == 0 ? t : 0.f));
    if (lane == 0) s_w63[w] = tw;
  }
  f32x4 dT[2], nN[2];
  {
    const f32x8 ta0 = frag_cols(bT, LD, 16 * rt, 0, lane), ta1 = frag_cols(bT, LD, 16 * rt, 32, lane);
    const f32x8 da0 = frag_rows(bdW, LD, 16 * rt, 0, lane), da1 = frag_rows(bdW, LD, 16 * rt, 32, lane);
    const f32x8 ya0 = frag_rows(bY, LD, 16 * rt, 0, lane), ya1 = frag_rows(bY, LD, 16 * rt, 32, lane);
    float dbp[4] = {0.f, 0.f, 0.f, 0.f}, rowp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nn = 0; nn < 2; ++nn) {
      const int n = 2 * ch + nn;
      const int cj = 16 * n + (lane & 15);
      // T^T dW
      const f32x4 td = mm<PrecF32>(mm<PrecF32>(zero4(), ta0, frag_cols(bdW, LD, 16 * n, 0, lane)), ta1, frag_cols(bdW, LD, 16 * n, 32, lane));
      // -dW X_K^T and dW V^T
      const f32x4 dtp = -mm<PrecF32>(mm<PrecF32>(zero4(), da0, frag_rows(bXK, LD, 16 * n, 0, lane)), da1, frag_rows(bXK, LD, 16 * n, 32, lane));
      const f32x4 e1 = mm<PrecF32>(mm<PrecF32>(zero4(), da0, frag_rows(bV, LD, 16 * n, 0, lane)), da1, frag_rows(bV, LD, 16 * n, 32, lane));
      // dY W^T
      const f32x4 dp = mm<PrecF32>(mm<PrecF32>(zero4(), ya0, frag_rows(bW, LD, 16 * n, 0, lane)), ya1, frag_rows(bW, LD, 16 * n, 32, lane));
      const float bj = s_beta[cj], lj = s_ell[cj], gj = expf(lj);
      float ts = 0.f, colp = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * rt + 4 * (lane >> 4) + i;
        const bool valid = t0 + ri < p.T;
        if (valid) p.dv[b * p.dvs0 + (t0 + ri) * p.dvs1 + h * p.dvs2 + cj] = s_beta[ri] * td[i];
        dbp[i] += bV[ri * LD + cj] * td[i];
        // the linear rule's T = I and Tp = 0 are constants: no gradient flows through them
        ts += p.linear ? 0.f : bT[ri * LD + cj] * dtp[i];
        dT[nn][i] = p.linear ? 0.f : bj * (e1[i] + gj * dtp[i]);
        if (cj < ri) {
          const float pb = dp[i] * rec[Rec::P + ri * C + cj];
          rowp[i] += pb;
          colp += pb;
          const float lim1 = s_ell[ri - 1];
          nN[nn][i] = dp[i] * expf(fminf(lim1 - lj, 0.f));
        } else {
          nN[nn][i] = 0.f;
        }
      }
      ts = sum_col4(ts);
      colp = sum_col4(colp);
      if (lane < 16) {
        s_tsp[rt][cj] = ts;
        s_dlp[DL_COLP + rt][cj] = -colp;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float db = sum_row16(dbp[i]), rp = sum_row16(rowp[i]);
      if ((lane & 15) == 0) {
        s_dbp[DB_V + ch][ri] = db;
        if (ri > 0) s_dlp[DL_RP + ch][ri - 1] = rp;
      }
    }
  }
  __syncthreads();

  // ---- phase 2: dT and N to LDS; Tp sums; Q S^T -> da; a o dY, kappa o W; <Gamma, S>
#pragma unroll
  for (int nn = 0; nn < 2; ++nn)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i, cj = 16 * (2 * ch + nn) + (lane & 15);
      bX[ri * LD + cj] = dT[nn][i];
      bXK[ri * LD + cj] = nN[nn][i];
    }
  if (tid < C) {
    const float g = expf(s_ell[tid]), ts = ((s_tsp[0][tid] + s_tsp[1][tid]) + s_tsp[2][tid]) + s_tsp[3][tid];
    s_dbp[DB_TS][tid] = g * ts;
    s_dlp[DL_TS][tid] = s_beta[tid] * g * ts;
  }
  {
    const typename P::frag* qxf = qxf_area<P>(rec);
    const typename P::frag* sf = reinterpret_cast<const typename P::frag*>(rec + Rec::Q);
    f32x4 qs[2];
#pragma unroll
    for (int nn = 0; nn < 2; ++nn) qs[nn] = zero4();
#pragma unroll 4
    for (int jb = 0; jb < D / 32; ++jb) {
      const typename P::frag qa = qxf[(rt * 16 + jb) * 64 + lane];
#pragma unroll
      for (int nn = 0; nn < 2; ++nn) qs[nn] = P::mma(qs[nn], qa, sf[((2 * ch + nn) * 16 + jb) * 64 + lane]);
    }
    float dap[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nn = 0; nn < 2; ++nn)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dap[i] += bY[(16 * rt + 4 * (lane >> 4) + i) * LD + 16 * (2 * ch + nn) + (lane & 15)] * qs[nn][i];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float da = sum_row16(dap[i]);
      if ((lane & 15) == 0) {
        if (ri > 0) s_dlp[DL_DA + ch][ri - 1] = da * expf(s_ell[ri - 1]);
        else s_da0[ch] = da;
      }
    }
    // scale this wave's block only (no other wave reads it in this phase)
    for (int e = lane; e < 16 * 32; e += 64) {
      const int ri = 16 * rt + (e >> 5), cv = 32 * ch + (e & 31);
      bY[ri * LD + cv] *= ri > 0 ? expf(s_ell[ri - 1]) : 1.f;
      bW[ri * LD + cv] *= expf(l63 - s_ell[ri]);
    }
  }
  {
    float gs = 0.f;
    const typename Feat<P>::T* G4 = feat<P>(rec, Rec::G);
    const typename Feat<P>::T* S4 = feat<P>(rec, Rec::S);
    // 16 iterations per thread, unrolled so that their loads are in flight together
#pragma unroll 8
    for (int e = tid; e < D * DV / 4; e += 64 * GRAD_WAVES) {
      const f32x4 g = ld4_t(G4 + 4 * e), s = ld4_t(S4 + 4 * e);
      gs += g[0] * s[0] + g[1] * s[1] + g[2] * s[2] + g[3] * s[3];
    }
    gs = sum_col4(sum_row16(gs));
    if (lane == 0) s_w63[4 + w] = gs;
  }
  __syncthreads();

  // ---- phase 3: Y1 = dT T^T; Zn = -Tp^T dW
  f32x4 y1[2], zn[2];
  {
    const f32x8 a0 = frag_rows(bX, LD, 16 * rt, 0, lane), a1 = frag_rows(bX, LD, 16 * rt, 32, lane);
    const f32x8* tpt = reinterpret_cast<const f32x8*>(rec + Rec::TPT);
    const f32x8 p0 = tpt[(rt * 2) * 64 + lane], p1 = tpt[(rt * 2 + 1) * 64 + lane];
#pragma unroll
    for (int nn = 0; nn < 2; ++nn) {
      const int n = 2 * ch + nn;
      y1[nn] = mm<PrecF32>(mm<PrecF32>(zero4(), a0, frag_rows(bT, LD, 16 * n, 0, lane)), a1, frag_rows(bT, LD, 16 * n, 32, lane));
      zn[nn] = -mm<PrecF32>(mm<PrecF32>(zero4(), p0, frag_cols(bdW, LD, 16 * n, 0, lane)), p1, frag_cols(bdW, LD, 16 * n, 32, lane));
    }
  }
  __syncthreads();
#pragma unroll
  for (int nn = 0; nn < 2; ++nn)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i, cj = 16 * (2 * ch + nn) + (lane & 15);
      bV[ri * LD + cj] = y1[nn][i];
      bdW[ri * LD + cj] = zn[nn][i];
    }
  __syncthreads();

  // ---- phase 4: dA = -T^T Y1 (strictly lower); M + M^T into bX; dbeta, dl from A
  {
    const f32x8 ta0 = frag_cols(bT, LD, 16 * rt, 0, lane), ta1 = frag_cols(bT, LD, 16 * rt, 32, lane);
    float dbr[4] = {0.f, 0.f, 0.f, 0.f}, dlr[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nn = 0; nn < 2; ++nn) {
      const int n = 2 * ch + nn;
      const f32x4 dA = -mm<PrecF32>(mm<PrecF32>(zero4(), ta0, frag_cols(bV, LD, 16 * n, 0, lane)), ta1, frag_cols(bV, LD, 16 * n, 32, lane));
      const int cj = 16 * n + (lane & 15);
      float dlc = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ri = 16 * rt + 4 * (lane >> 4) + i;
        if (cj < ri) {
          const float ex = expf(fminf(s_ell[ri] - s_ell[cj], 0.f));
          const float e = dA[i] * ex * rec[Rec::GKK + ri * C + cj];
          const float ab = s_beta[ri] * e;
          dbr[i] += e;
          dlr[i] += ab;
          dlc += ab;
          const float mv = dA[i] * s_beta[ri] * ex;
          bX[ri * LD + cj] = mv;
          bX[cj * LD + ri] = mv;
        } else if (cj == ri) {
          bX[ri * LD + cj] = 0.f;
        }
      }
      dlc = sum_col4(dlc);
      if (lane < 16) s_dlp[DL_DLC + rt][cj] = -dlc;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ri = 16 * rt + 4 * (lane >> 4) + i;
      const float a = sum_row16(dbr[i]), d = sum_row16(dlr[i]);
      if ((lane & 15) == 0) {
        s_dbp[DB_A + ch][ri] = a;
        s_dlp[DL_A + ch][ri] = d;
      }
    }
  }
  __syncthreads();

  // ---- phase 5: dbeta and dlambda (dlog lambda_t = sum_{i >= t} dl_i); phi . dphi per token, which the
  // renormalisation's backward needs over all features: every term of dphi is a product with Q, K rows or
  // the carries, so phi . dphi is a sum of terms already here:
  //   phi_q[i] . dphi_q[i] = a_i dY_i . (Q S)_i + sum_j P_ij dP_ij
  //   phi_k[j] . dphi_k[j] = (kappa o W)_j . X_j + sum_i P_ij dP_ij + sum_i Tp_ij dTp_ij (X_K . Zn)
  //                          + row and column sums of A o dA (M + M^T)
  if (w == 1) {
    float rq = lane > 0 ? s_dlp[DL_DA][lane - 1] + s_dlp[DL_DA + 1][lane - 1] : s_da0[0] + s_da0[1];
    if (lane > 0) rq += s_dlp[DL_RP][lane - 1] + s_dlp[DL_RP + 1][lane - 1];
    float rk = s_dlp[DL_TS][lane] - s_dlp[DL_KAPPA][lane];
#pragma unroll
    for (int v = 0; v < 4; ++v) rk -= s_dlp[DL_COLP + v][lane] + s_dlp[DL_DLC + v][lane];
    rk += s_dlp[DL_A][lane] + s_dlp[DL_A + 1][lane];
    rec[Rec::V_RD + lane] = rq;
    rec[Rec::V_RD + 64 + lane] = rk;
  }
  if (w == 0) {
    float dl = 0.f;
#pragma unroll
    for (int k = 0; k < NDL; ++k) dl += s_dlp[k][lane];
    if (lane == 63) {
      float kap = 0.f, gs = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) kap += s_w63[v];
#pragma unroll
      for (int v = 0; v < GRAD_WAVES; ++v) gs += s_w63[4 + v];
      dl += kap + gs * gC;
    }
    float dbeta = 0.f;
#pragma unroll
    for (int k = 0; k < NDB; ++k) dbeta += s_dbp[k][lane];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float u = __shfl_down(dl, o);
      if (lane + o < 64) dl += u;
    }
    const int64_t t = t0 + lane;
    if (t < p.T) {
      p.dbeta[b * p.dbs0 + t * p.dbs1 + h * p.dbs2] = dbeta;
      if (p.ddecay) {
        const float la = p.decay ? p.decay[b * p.ds0 + t * p.ds1 + h * p.ds2] : 1.f;
        p.ddecay[b * p.dds0 + t * p.dds1 + h * p.dds2] = (la >= 1e-5f && la <= 1.f) ? dl / la : 0.f;
      }
    }
  }

  // ---- the B operands of the dx kernel, as P fragments in the record's K-fragment area (dead once both
  // carries are done): token tile m = w & 3, depth block jb = w >> 2, dK^T [kappa o W, Zn, N^T, M + M^T],
  // dQ^T [a o dY, N]
  {
    using frag = typename P::frag;
    frag* bop = reinterpret_cast<frag*>(rec + Rec::KXF);
    const int m = rt, jb = ch;
    bop[bop_dk(m, 0, jb) * 64 + lane] = P::from_f32(frag_rows(bW, LD, 16 * m, 32 * jb, lane));
    bop[bop_dk(m, 1, jb) * 64 + lane] = P::from_f32(frag_rows(bdW, LD, 16 * m, 32 * jb, lane));
    bop[bop_dk(m, 2, jb) * 64 + lane] = P::from_f32(frag_cols(bXK, LD, 16 * m, 32 * jb, lane));
    bop[bop_dk(m, 3, jb) * 64 + lane] = P::from_f32(frag_rows(bX, LD, 16 * m, 32 * jb, lane));
    bop[bop_dq(m, 0, jb) * 64 + lane] = P::from_f32(frag_rows(bY, LD, 16 * m, 32 * jb, lane));
    bop[bop_dq(m, 1, jb) * 64 + lane] = P::from_f32(frag_rows(bXK, LD, 16 * m, 32 * jb, lane));
  }
}

// ---------------------------------------------------------------------------------------------- dx
// grid (nseg, H, B), DX_WAVES waves of 64 features each.
//   dK^T = Gamma (kappa o W)^T + S^T Zn^T + Q^T N + K^T (M + M^T)      dQ^T = S^T (a o dY)^T + K^T N^T
// for all 64 tokens, 32 features at a time, each followed by their lift backward: with theta = inv_tau (Omega x^) + b recomputed,
//   dphi~ = dphi / (n + 1e-8) - phi (phi . dphi) / n,  ds = -sqrt(2/D) sin(theta) dphi~,  dx^ = ds Omega
// (phi . dphi from the gradient kernel, phi from the cosine of the same angle), and the input
// normalisation's backward to dk, dq.  GEN: the general feature map (per-head or hi + lo Omega, per-head
// phases and 1/tau, optional renormalisation, dL/d(1/tau)); LO (with GEN): Omega has low parts.
//
// The kernel is bound by the record's bytes: each A operand (Gamma, S^T, Q^T, K^T rows, 64 KB each with
// bf16 features) is read once, for both gradients and all four token tiles;
// the token-side operands of the gradient kernel (48 fragments) are staged in LDS, one read feeding two
// feature tiles.  Two halves of 32 tokens and k before q, with the rows of phi read again for phi . dphi,
// took 1 MB of HBM reads per chunk and head: 4096 chunks 1328 us, this form 426.
constexpr int DX_WAVES = 8;

template <class P>
struct DxShared {
  static constexpr int NBOP = IsBf16Policy<P>::value ? 48 : 0;  // fp32 operands (96 KB) are read from L2: the fp32
                                                                // products take longer than that
  static constexpr size_t BOP_BYTES = (size_t)NBOP * 64 * sizeof(typename P::frag), RED_BYTES = 4 * C * LD * sizeof(float);
  // the token-side operands (bop_dk, bop_dq), then dx^ partials [wave group 2][q, k][64][LD]
  __attribute__((aligned(16))) unsigned char big[BOP_BYTES > RED_BYTES ? BOP_BYTES : RED_BYTES];
  typename P::frag x[2][4][2][64];  // normalised q, k rows as B fragments (plain depth order)
  // per input and token: 1 / (n + 1e-8) and (phi . dphi) / n (without renormalisation dphi~ = dphi: 1, 0)
  float inv[2][C], rdn[2][C], dit[DX_WAVES];
};

// dx^ of the inputs W0 .. W0 + NWH - 1 (0 q, 1 k) into the shared partials: with bf16 features both at once,
// so that S^T and K^T are read once; with fp32 features, whose fragments take twice the registers, k, then q.
template <class P, bool LO, bool GEN, int W0, int NWH>
__device__ __forceinline__ void dx_features(const Params& p, DxShared<P>& sh, const float* rec, int64_t h, int w, int lane,
                                            float itau, float& dit) {
  using frag = typename P::frag;
  constexpr int NFT = 32 / DX_WAVES;                   // 16-feature tiles per wave
  constexpr int PF = IsBf16Policy<P>::value ? 2 : 1;   // feature tiles whose A operands are held at once
  constexpr bool HASQ = W0 == 0, HASK = W0 + NWH == 2;
  const frag* bop = DxShared<P>::NBOP ? reinterpret_cast<const frag*>(sh.big) : reinterpret_cast<const frag*>(rec + Rec::KXF);
  const int fb = 64 * w;
  const __bf16* omega = GEN ? p.omega + h * p.oms : p.omega;
  const __bf16* omega_lo = LO ? p.omega_lo + h * p.oms : nullptr;
  const float* phase = GEN ? p.phase + h * p.phs : p.phase;
  const bf16x8* omt = GEN ? p.omt + h * p.omt_hs : p.omt;
  const float amp = sqrtf(2.f / D);
  // dL/dtheta by input, 32-feature block, token tile, as the B fragments of dx^^T = Omega^T dtheta^T
  frag bs[NWH][NFT / 2][4];
#pragma unroll
  for (int fp = 0; fp < NFT / 2; ++fp) {
    f32x4 acc[NWH][2][4];  // features 32 fp + 16 f + 4 (lane >> 4) + i, token 16u + (lane & 15)
#pragma unroll
    for (int fs0 = 0; fs0 < 2; fs0 += PF) {
      frag fg[PF][2], fs[PF][2], fq[PF][2], fk[PF][2];
      const frag* qtf = reinterpret_cast<const frag*>(rec + Rec::QTF);
      const frag* ktf = reinterpret_cast<const frag*>(rec + Rec::KTF);
#pragma unroll
      for (int f = 0; f < PF; ++f)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) {
          const int ft = NFT * w + 2 * fp + fs0 + f;
          if constexpr (HASK) {
            fg[f][jb] = frag_pieces<P>(rec, Rec::G, ft, jb, lane);
            fq[f][jb] = uni(qtf + (ft * 2 + jb) * 64)[lane];
          }
          fs[f][jb] = frag_pieces<P>(rec, Rec::S, ft, jb, lane);
          fk[f][jb] = uni(ktf + (ft * 2 + jb) * 64)[lane];
        }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        f32x4 tk[PF], tq[PF];
#pragma unroll
        for (int f = 0; f < PF; ++f) tk[f] = tq[f] = zero4();
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) {
          __builtin_amdgcn_sched_barrier(0);  // at most six fragments of the token side at a time
          frag k0, k1, k2, k3, q0, q1;
          if constexpr (HASK) {
            k0 = bop[bop_dk(u, 0, jb) * 64 + lane]; k1 = bop[bop_dk(u, 1, jb) * 64 + lane];
            k2 = bop[bop_dk(u, 2, jb) * 64 + lane]; k3 = bop[bop_dk(u, 3, jb) * 64 + lane];
          }
          if constexpr (HASQ) { q0 = bop[bop_dq(u, 0, jb) * 64 + lane]; q1 = bop[bop_dq(u, 1, jb) * 64 + lane]; }
#pragma unroll
          for (int f = 0; f < PF; ++f) {
            if constexpr (HASK) tk[f] = P::mma(tk[f], fg[f][jb], k0);
            if constexpr (HASQ) tq[f] = P::mma(tq[f], fs[f][jb], q0);
            if constexpr (HASK) tk[f] = P::mma(tk[f], fs[f][jb], k1);
            if constexpr (HASQ) tq[f] = P::mma(tq[f], fk[f][jb], q1);
            if constexpr (HASK) tk[f] = P::mma(P::mma(tk[f], fq[f][jb], k2), fk[f][jb], k3);
          }
        }
#pragma unroll
        for (int f = 0; f < PF; ++f) {
          if constexpr (HASQ) acc[0][fs0 + f][u] = tq[f];
          if constexpr (HASK) acc[NWH - 1][fs0 + f][u] = tk[f];
        }
      }
    }
    // the lift backward of these 32 features, in place: acc <- dL/dtheta
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int f0 = fb + 32 * fp + 16 * f;
      const frag o0 = omega_frag<P>(omega, f0, 0, lane), o1 = omega_frag<P>(omega, f0, 32, lane);
      const f32x4 ph4 = *reinterpret_cast<const f32x4*>(phase + f0 + 4 * (lane >> 4));
      frag l0{}, l1{};
      if constexpr (LO) {
        l0 = omega_frag<P>(omega_lo, f0, 0, lane);
        l1 = omega_frag<P>(omega_lo, f0, 32, lane);
      }
#pragma unroll
      for (int wi = 0; wi < NWH; ++wi)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (u % 2 == 0) __builtin_amdgcn_sched_barrier(0);
          const frag x0 = sh.x[W0 + wi][u][0][lane], x1 = sh.x[W0 + wi][u][1][lane];
          const float inv_n = sh.inv[W0 + wi][16 * u + (lane & 15)], rd_n = sh.rdn[W0 + wi][16 * u + (lane & 15)];
          f32x4 sv = P::mma(P::mma(zero4(), o0, x0), o1, x1);
          if constexpr (LO) sv = P::mma(P::mma(sv, l0, x0), l1, x1);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float rv = (sv[i] * itau + ph4[i]) * 0.15915494309189535f;
            rv -= __builtin_rintf(rv);
            const float cs = amp * __builtin_amdgcn_cosf(rv), sn = amp * __builtin_amdgcn_sinf(rv);
            const float da = -sn * ((acc[wi][f][u][i] - cs * rd_n) * inv_n);
            acc[wi][f][u][i] = da;
            if constexpr (GEN) dit += da * sv[i];
          }
          if constexpr (GEN) asm volatile("" : "+v"(dit));  // summed here, not from held terms at the end
        }
    }
#pragma unroll
    for (int wi = 0; wi < NWH; ++wi)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        bs[wi][fp][u] = P::from_f32(pair_to8(acc[wi][0][u], acc[wi][1][u]));
        // in its packed form from here on: sunk to the use, the conversion would keep the fp32 values live
        asm volatile("" : "+v"(bs[wi][fp][u]));
      }
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (DxShared<P>::NBOP > 0) __syncthreads();  // the token-side operands' LDS takes the dx^ partials

  // dx^^T = Omega^T ds^T over this wave's features, then the waves' partials: two groups of four waves, each
  // into its own buffer, in turns (turn t: wave w takes input columns 16a .. 16a + 15, a = (w + t) & 3; the
  // first turn writes) so that the sums have a fixed order.
#pragma unroll
  for (int wi = 0; wi < NWH; ++wi) {
    f32x4 d[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int u = 0; u < 4; ++u) d[a][u] = zero4();
#pragma unroll
    for (int jj = 0; jj < NFT / 2; ++jj)
#pragma unroll
      for (int part = 0; part < (LO ? 2 : 1); ++part) {
        __builtin_amdgcn_sched_barrier(0);
        frag ob[4];
#pragma unroll
        for (int a = 0; a < 4; ++a) ob[a] = bf16_frag<P>(omt[part * OMT_ENTRIES + (a * 16 + fb / 32 + jj) * 64 + lane]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int a = 0; a < 4; ++a) d[a][u] = P::mma(d[a][u], ob[a], bs[wi][jj][u]);
      }
    const int le = fresh(lane);
    float* red = reinterpret_cast<float*>(sh.big) + ((w >> 2) * 2 + W0 + wi) * C * LD + (le & 15) * LD + 4 * (le >> 4);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int a = (w + t) & 3;
#pragma unroll
      for (int aa = 0; aa < 4; ++aa) {
        if (aa == a) {  // uniform over the wave
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            f32x4* px = reinterpret_cast<f32x4*>(red + 16 * u * LD + 16 * aa);
            *px = t == 0 ? d[aa][u] : *px + d[aa][u];
          }
        }
      }
      lds_barrier();
    }
  }
}

template <class P, typename InT, bool LO, bool GEN>
__global__ void __launch_bounds__(64 * DX_WAVES) bwd_dx_kernel(Params p) {
  using frag = typename P::frag;
  __shared__ DxShared<P> sh;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = (p.c0 + blockIdx.x) * C;
  const float* rec = record(p, b, h, blockIdx.x);
  // loaders: input `which` (0 q, 1 k), row r, features c0 .. c0 + 15
  const int which = w >> 2, r = (tid >> 2) & 63, c0 = (tid & 3) * 16;
  const bool rvalid = t0 + r < p.T;
  const InT* x = reinterpret_cast<const InT*>(which == 0 ? p.q : p.k);
  const int64_t xb = which == 0 ? b * p.qs0 + (t0 + r) * p.qs1 + h * p.qs2 + c0 : b * p.ks0 + (t0 + r) * p.ks1 + h * p.ks2 + c0;
  {
    const frag* bop = reinterpret_cast<const frag*>(rec + Rec::KXF);
    frag* s_bop = reinterpret_cast<frag*>(sh.big);
#pragma unroll
    for (int e = 0; e < DxShared<P>::NBOP / DX_WAVES; ++e) s_bop[e * 64 * DX_WAVES + tid] = bop[e * 64 * DX_WAVES + tid];
    if (tid < 2 * C) {
      const bool renorm = GEN ? !p.no_renorm : true;
      const float n = rec[Rec::V_NORM + tid];
      sh.inv[tid >> 6][tid & 63] = renorm ? 1.f / (n + 1e-8f) : 1.f;
      sh.rdn[tid >> 6][tid & 63] = renorm ? rec[Rec::V_RD + tid] / n : 0.f;
    }
    float part[16];
    load_x_part<InT>(x, xb, rvalid, p.normalize, part);
    round_like_input<InT>(p.normalize, part);
#pragma unroll
    for (int e8 = 0; e8 < 2; ++e8) {
      f32x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = part[8 * e8 + e];
      const int cc = c0 + 8 * e8;
      sh.x[which][r >> 4][cc >> 5][(r & 15) + 16 * ((cc & 31) >> 3)] = P::from_f32(v);
    }
  }
  __syncthreads();
  const float itau = GEN ? head_inv_tau(p, h) : p.inv_tau;
  float dit = 0.f;  // this lane's share of dL/d(1/tau)
  if constexpr (IsBf16Policy<P>::value) {
    dx_features<P, LO, GEN, 0, 2>(p, sh, rec, h, w, lane, itau, dit);
  } else {
    dx_features<P, LO, GEN, 1, 1>(p, sh, rec, h, w, lane, itau, dit);
    dx_features<P, LO, GEN, 0, 1>(p, sh, rec, h, w, fresh(lane), itau, dit);
  }
  {
    const int te = 64 * w + fresh(lane);  // the row and columns again
    const int re = (te >> 2) & 63, ce = (te & 3) * 16;
    const int64_t t = t0 + re;
    const bool valid = t < p.T;
    const float* d0 = reinterpret_cast<const float*>(sh.big) + which * C * LD;
    const float* d1 = d0 + 2 * C * LD;
    if (which == 0)
      write_dx<InT>(p, reinterpret_cast<const InT*>(p.q), b * p.qs0 + t * p.qs1 + h * p.qs2 + ce, p.dq,
                    b * p.dqs0 + t * p.dqs1 + h * p.dqs2 + ce, d0, d1, re, ce, valid, itau);
    else
      write_dx<InT>(p, reinterpret_cast<const InT*>(p.k), b * p.ks0 + t * p.ks1 + h * p.ks2 + ce, p.dk,
                    b * p.dks0 + t * p.dks1 + h * p.dks2 + ce, d0, d1, re, ce, valid, itau);
  }
  if (GEN && p.dit) {  // fixed order: lanes by a shuffle tree, then the waves in order
    dit += xor_shuffle<32>(dit);
    dit += xor_shuffle<16>(dit);
    dit += xor_shuffle<8>(dit);
    dit += xor_shuffle<4>(dit);
    dit += xor_shuffle<2>(dit);
    dit += xor_shuffle<1>(dit);
    if (lane == 0) sh.dit[w] = dit;
    __syncthreads();
    if (tid == 0) {
      float t = sh.dit[0];
#pragma unroll
      for (int v = 1; v < DX_WAVES; ++v) t += sh.dit[v];
      p.dit[(b * p.H + h) * p.nch + p.c0 + blockIdx.x] = t;
    }
  }
}

}  // namespace bwd

using namespace bwd;

static bool bwd_supported(const kdn_scan_args* f) {
  return f->d_k == DK && f->D == D && f->d_v == DV && (f->rule == 0 || f->rule == 1) && f->feature_mode == 0 &&
         f->omega_head_stride >= 0 && f->phase_head_stride >= 0 && !f->cu_seqlens && !f->state_slots;
}

static int bwd_check(const kdn_scan_bwd_args* a) {
  if (!a || !a->fwd) return KDN_ERR_INVALID_ARGUMENT;
  const kdn_scan_args* f = a->fwd;
  if (f->B <= 0 || f->T <= 0 || f->H <= 0 || !valid_dtype(f->in_dtype)) return KDN_ERR_INVALID_ARGUMENT;
  if (!bwd_supported(f)) return KDN_ERR_UNSUPPORTED;
  if (!f->q || !f->k || !f->v || !f->beta || !f->omega_bf16 || !f->phase) return KDN_ERR_INVALID_ARGUMENT;
  if (!a->dy || !a->dq || !a->dk || !a->dv || !a->dbeta) return KDN_ERR_INVALID_ARGUMENT;
  if (a->ddecay && !f->decay) return KDN_ERR_INVALID_ARGUMENT;
  for (int i = 0; i < 3; ++i)
    if (f->q_stride[i] < 0 || f->k_stride[i] < 0 || f->v_stride[i] < 0 || f->beta_stride[i] < 0 ||
        a->dy_stride[i] < 0)
      return KDN_ERR_INVALID_ARGUMENT;
  // the forward's pointer rules: 16-byte rows of q, k, v (element loads here, but the same buffers feed
  // the forward's vector loads), 16-byte phase (read four at a time) and Omega rows; fp32 gradients and
  // dL/dy at least 4-byte aligned
  const size_t isz = dtype_size(f->in_dtype);
  if (!aligned(f->q, 16) || !aligned(f->k, 16) || !aligned(f->v, 16)) return KDN_ERR_MISALIGNED;
  for (int i = 0; i < 3; ++i)
    if (((f->q_stride[i] * (int64_t)isz) % 16) != 0 || ((f->k_stride[i] * (int64_t)isz) % 16) != 0 ||
        ((f->v_stride[i] * (int64_t)isz) % 16) != 0)
      return KDN_ERR_MISALIGNED;
  if (!aligned(f->omega_bf16, 16) || !aligned(f->phase, 16)) return KDN_ERR_MISALIGNED;
  // per-head Omega rows and phases stay 16-byte aligned (Omega fragments and phases are vector loads)
  if ((f->omega_lo && !aligned(f->omega_lo, 16)) || (f->omega_head_stride * 2) % 16 != 0 ||
      (f->phase_head_stride * 4) % 16 != 0 || (a->dinv_tau && !aligned(a->dinv_tau, 4)))
    return KDN_ERR_MISALIGNED;
  if (!aligned(a->dy, 4) || !aligned(a->dq, 4) || !aligned(a->dk, 4) || !aligned(a->dv, 4) || !aligned(a->dbeta, 4))
    return KDN_ERR_MISALIGNED;
  return KDN_OK;
}

static int64_t bwd_chunks(const kdn_scan_args* f) { return (f->T + C - 1) / C; }

// The backward runs in segments of `seg` chunks (the last may be shorter), last segment first, so that
// its workspace grows with the segment, not with T:
//   nbuf record buffers (seg records per head each)   the per-chunk recompute and both carries of one
//                                                     segment, rotating so that up to three segments
//                                                     are in flight
//   nsegs - 1 states, fp32 [B][H][512][64] each       S^T at the start of segments 1 .. nsegs-1 (the
//                                                     checkpoint pass: the forward scan's prep and
//                                                     state kernels, kdn_scan.hip)
//   one such array                                    dL/dS^T carried from one segment to the previous
//   nfb buffers of the forward scan's records         for the checkpoint pass
//   the Omega^T fragment table
struct BwdLayout {
  int64_t seg, nsegs;
  int nbuf, nfb;
  size_t rec_buf, state_bytes, ckpt_off, carry_off, fwd_off, fwd_buf, omt_off, dit_off, total;
};

// Default segment: the largest power of two from 4 to 256 chunks whose records fit 4.5 GiB (256 chunks at
// B*H = 16: 4 segments, 15.52-15.55 ms per backward against 15.95 with 8 segments of 128, 16.43 with 16
// of 64, and 15.85-15.93 / 16.56-16.58 with 2 of 512 / 1 of 1024).
constexpr size_t BWD_SEGMENT_BUDGET = (size_t)4608 << 20;
constexpr int64_t BWD_SEGMENT_MAX = 256;

static BwdLayout bwd_layout(const kdn_scan_args* f, bool want_dit) {
  BwdLayout L;
  const int64_t nch = bwd_chunks(f), heads = f->B * f->H;
  const size_t per_chunk = (size_t)heads * Rec::floats * sizeof(float);
  int64_t seg = 4;
  if (f->segment_chunks > 0) {
    seg = f->segment_chunks;
  } else {
    const size_t fit = BWD_SEGMENT_BUDGET / per_chunk;
    while (seg < BWD_SEGMENT_MAX && (size_t)(2 * seg) <= fit) seg *= 2;
  }
  if (seg > nch) seg = nch;
  L.seg = seg;
  L.nsegs = (nch + seg - 1) / seg;
  L.nbuf = (int)(L.nsegs < 3 ? L.nsegs : 3);
  L.nfb = (int)(L.nsegs - 1 < 2 ? L.nsegs - 1 : 2);
  L.rec_buf = (size_t)seg * per_chunk;
  L.state_bytes = (size_t)heads * D * DV * sizeof(float);
  L.ckpt_off = (size_t)L.nbuf * L.rec_buf;
  L.carry_off = L.ckpt_off + (size_t)(L.nsegs - 1) * L.state_bytes;
  L.fwd_off = L.carry_off + (L.nsegs > 1 ? L.state_bytes : 0);
  L.fwd_buf = L.nfb > 0 ? (scan_checkpoint_buffer_bytes(f, seg) + 255) / 256 * 256 : 0;
  L.omt_off = L.fwd_off + (size_t)L.nfb * L.fwd_buf;
  // one Omega^T table, or one per head; twice with low parts
  const size_t tables = (f->omega_head_stride ? (size_t)f->H : 1) * (f->omega_lo ? 2 : 1);
  L.dit_off = L.omt_off + tables * OMT_BYTES;
  L.total = L.dit_off + (want_dit ? ((size_t)heads * nch * sizeof(float) + 255) / 256 * 256 : 0);
  return L;
}

namespace vsplit {
static bool applies(const kdn_scan_args* f);
static size_t workspace_bytes(const kdn_scan_bwd_args* a);
static int64_t segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks);
}  // namespace vsplit

namespace frep {
static size_t workspace_bytes(const kdn_scan_bwd_args* a);
static int64_t segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks);
}  // namespace frep

extern "C" size_t kdn_scan_bwd_workspace_bytes(const kdn_scan_bwd_args* a) {
  if (a && general_bwd_applies(a->fwd)) return general_bwd_workspace_bytes(a);
  if (a && a->fwd && frep_applies(a->fwd)) return frep::workspace_bytes(a);
  if (a && vsplit::applies(a->fwd)) return vsplit::workspace_bytes(a);
  if (bwd_check(a) != KDN_OK) return 0;
  return bwd_layout(a->fwd, a->dinv_tau != nullptr).total;
}

extern "C" int64_t kdn_scan_bwd_segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks) {
  if (a && general_bwd_applies(a->fwd)) return general_bwd_segments(a, segment_chunks);
  if (a && a->fwd && frep_applies(a->fwd)) return frep::segments(a, segment_chunks);
  if (a && vsplit::applies(a->fwd)) return vsplit::segments(a, segment_chunks);
  if (bwd_check(a) != KDN_OK) return 0;
  const BwdLayout L = bwd_layout(a->fwd, a->dinv_tau != nullptr);
  if (segment_chunks) *segment_chunks = L.seg;
  return L.nsegs;
}

// Omega^T as A fragments for the gradient kernel's dx^ = ds Omega: fragment (a, jb) lane l slot s holds
// Omega[32jb + kappa(l, s)][16a + (l & 15)] (a column gather done once per call instead of per chunk).
// grid (16, tables' heads, parts): part 0 from Omega (hi), part 1 from its low parts; head y's Omega at
// y * oms elements, its tables at y * parts * OMT_ENTRIES.
__global__ void __launch_bounds__(256) bwd_omega_t_kernel(const __bf16* omega, const __bf16* omega_lo, int64_t oms,
                                                          bf16x8* table) {
  const int idx = blockIdx.x * 256 + threadIdx.x;  // 16 blocks of 256 cover [a 4][jb 16][lane 64]
  const int lane = idx & 63, jb = (idx >> 6) & 15, a = idx >> 10;
  const int64_t hy = blockIdx.y;
  const int part = blockIdx.z;
  const __bf16* src = (part ? omega_lo : omega) + hy * oms;
  bf16x8 v;
#pragma unroll
  for (int s = 0; s < 8; ++s) v[s] = src[(size_t)(32 * jb + kappa(lane, s)) * DK + 16 * a + (lane & 15)];
  table[(hy * gridDim.z + part) * OMT_ENTRIES + idx] = v;
}

// The parameters of segment s: its chunks, its record buffer (rotating in processing order, last segment
// first), the state it starts from (initial_state or its checkpoint), the dL/dS^T it ends with
// (d_final_state or the carry) and where its reverse carry leaves dL/dS^T (the carry, or
// d_initial_state for segment 0).
static Params segment_params(const Params& base, const kdn_scan_bwd_args* a, const BwdLayout& L, int64_t s) {
  Params p = base;
  unsigned char* ws = static_cast<unsigned char*>(a->workspace);
  p.c0 = s * L.seg;
  p.nseg = (p.nch - p.c0 < L.seg) ? p.nch - p.c0 : L.seg;
  p.cap = L.seg;
  p.ws = reinterpret_cast<float*>(ws + (size_t)((L.nsegs - 1 - s) % L.nbuf) * L.rec_buf);
  const int64_t c0s = base.H * D * DV, c1s = D * DV, c2s = DV, c3s = 1;  // a contiguous [B][H][D][DV] state
  float* carry = reinterpret_cast<float*>(ws + L.carry_off);
  if (s > 0) {
    p.init = reinterpret_cast<const float*>(ws + L.ckpt_off + (size_t)(s - 1) * L.state_bytes);
    p.is0 = c0s; p.is1 = c1s; p.is2 = c2s; p.is3 = c3s;
    p.gout = carry;
    p.gos0 = c0s; p.gos1 = c1s; p.gos2 = c2s; p.gos3 = c3s;
  }
  if (s < L.nsegs - 1) {
    p.dfin = carry;
    p.fs0 = c0s; p.fs1 = c1s; p.fs2 = c2s; p.fs3 = c3s;
  }
  return p;
}

// One launch of segment p: 1 per-chunk recompute, 2 forward carry, 3 reverse carry, 4 gradients, or
// PH_CARRIES: both carries in one launch; PH_GRAD and PH_DX: the two launches of phase 4 (the gradient
// algebra, then dx) on their own.
// dL/d(1/tau) of head blockIdx.x: the per-(batch, chunk) partials summed in a fixed order (lane-strided
// sums, then a shuffle tree), so that the result does not depend on the schedule.
__global__ void __launch_bounds__(64) bwd_dit_reduce_kernel(const float* dit, int64_t B, int64_t H, int64_t nch,
                                                            float* out) {
  const int64_t h = blockIdx.x;
  const int lane = threadIdx.x;
  float t = 0.f;
  for (int64_t b = 0; b < B; ++b)
    for (int64_t c = lane; c < nch; c += 64) t += dit[(b * H + h) * nch + c];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o);
  if (lane == 0) out[h] = t;
}

constexpr int PH_CARRIES = 5, PH_GRAD = 6, PH_DX = 7;
template <class P, typename InT>
static int segment_phase(const Params& p, int phase, hipStream_t st) {
  const dim3 chunk_grid((unsigned)p.nseg, (unsigned)p.H, (unsigned)p.B);
  const unsigned chain_wgs = (unsigned)(((p.B * p.H + 7) / 8) * 8 * 4);
  if (phase == 1) {
    if (p.omega_lo) hipLaunchKernelGGL((bwd_prep_kernel<P, InT, true>), chunk_grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((bwd_prep_kernel<P, InT, false>), chunk_grid, dim3(256), 0, st, p);
  }
  if (phase == 2) hipLaunchKernelGGL((bwd_chain_kernel<P, false>), dim3(chain_wgs), dim3(64 * CHAIN_WAVES), 0, st, p);
  if (phase == 3) hipLaunchKernelGGL((bwd_chain_kernel<P, true>), dim3(chain_wgs), dim3(64 * CHAIN_WAVES), 0, st, p);
  if (phase == 4 || phase == PH_GRAD)
    hipLaunchKernelGGL((bwd_grad_kernel<P, InT>), chunk_grid, dim3(64 * GRAD_WAVES), 0, st, p);
  if (phase == 4 || phase == PH_DX) {
    const bool gen = p.omega_lo || p.oms || p.phs || p.inv_tau_head || p.no_renorm || p.dit;
    if (p.omega_lo) hipLaunchKernelGGL((bwd_dx_kernel<P, InT, true, true>), chunk_grid, dim3(64 * DX_WAVES), 0, st, p);
    else if (gen) hipLaunchKernelGGL((bwd_dx_kernel<P, InT, false, true>), chunk_grid, dim3(64 * DX_WAVES), 0, st, p);
    else hipLaunchKernelGGL((bwd_dx_kernel<P, InT, false, false>), chunk_grid, dim3(64 * DX_WAVES), 0, st, p);
    // segment 0 is the last one processed: every partial of dL/d(1/tau) is written
    if (p.dit && p.c0 == 0)
      hipLaunchKernelGGL(bwd_dit_reduce_kernel, dim3((unsigned)p.H), dim3(64), 0, st, p.dit, p.B, p.H, p.nch, p.dinv_tau);
  }
  if (phase == PH_CARRIES) hipLaunchKernelGGL((bwd_chains_kernel<P>), dim3(2 * chain_wgs), dim3(64 * CHAIN_WAVES), 0, st, p, chain_wgs);
  return launch_status();
}

// The start of a call: the Omega^T table, then the checkpoint pass (its prep kernels on aux if given).
static int bwd_start(const kdn_scan_bwd_args* a, const Params& base, const BwdLayout& L, hipStream_t st,
                     hipStream_t aux) {
  const unsigned heads = base.oms ? (unsigned)base.H : 1u, parts = base.omega_lo ? 2u : 1u;
  hipLaunchKernelGGL(bwd_omega_t_kernel, dim3(16, heads, parts), dim3(256), 0, st, base.omega, base.omega_lo, base.oms,
                     const_cast<bf16x8*>(base.omt));
  const int rc = launch_status();
  if (rc != KDN_OK) return rc;
  unsigned char* ws = static_cast<unsigned char*>(a->workspace);
  return scan_checkpoints(a->fwd, L.seg, L.nsegs - 1, reinterpret_cast<float*>(ws + L.ckpt_off), ws + L.fwd_off,
                          L.fwd_buf, L.nfb, st, aux);
}

// Serial: the start, then per segment (last first) recompute, both carries (one launch), gradients.
// With aux: the checkpoint pass's prep kernels run on aux beside its state kernels; then per segment
// (processing step i, segment s = nsegs - 1 - i, buffer i % nbuf)
//   aux: recompute(s) -> event R[i % nbuf]; dx(s + 1) after its gradient algebra (event G[(i - 1) % nbuf])
//   st:  both carries of s after R[i % nbuf] (the forward one after the checkpoint pass, which ends on
//        st), then the gradient algebra of s -> event G[i % nbuf]
// so that the carries, the sequential chain (two chain grids of B*H*4 workgroups), and the gradient
// algebra run back to back on st while aux recomputes and runs dx around them: per segment the two
// streams carry ~0.87 and ~0.75 ms of launches at config 3 (with the algebra on aux, 0.59 and 1.03).
// The recompute of step i reuses the buffer of step i - nbuf, whose dx precedes it on aux and waited for
// that step's algebra.  Every kernel reads and writes the same data in either schedule, so the results
// are identical bit for bit.
template <class P, typename InT>
static int bwd_schedule(const kdn_scan_bwd_args* a, const Params& base, const BwdLayout& L, hipStream_t st,
                        hipStream_t aux) {
#define KDN_TRY(x) do { if ((x) != hipSuccess) return KDN_ERR_DEVICE; } while (0)
#define KDN_TRYK(x) do { const int _rc = (x); if (_rc != KDN_OK) return _rc; } while (0)
  if (!aux || aux == st) {
    KDN_TRYK(bwd_start(a, base, L, st, nullptr));
    for (int64_t s = L.nsegs - 1; s >= 0; --s) {
      const Params p = segment_params(base, a, L, s);
      for (int ph : {1, PH_CARRIES, 4}) KDN_TRYK((segment_phase<P, InT>(p, ph, st)));
    }
    return KDN_OK;
  }
  EventSet evs;
  KDN_TRYK(evs.create(2 * L.nbuf + 2));
  hipEvent_t* evR = evs.ev;
  hipEvent_t* evG = evs.ev + L.nbuf;
  hipEvent_t evIn = evs.ev[2 * L.nbuf], evDone = evs.ev[2 * L.nbuf + 1];
  KDN_TRY(hipEventRecord(evIn, st));
  KDN_TRY(hipStreamWaitEvent(aux, evIn, 0));
  KDN_TRYK(bwd_start(a, base, L, st, aux));
  for (int64_t i = 0; i < L.nsegs; ++i) {
    const int64_t s = L.nsegs - 1 - i;
    const int bb = (int)(i % L.nbuf);
    const Params p = segment_params(base, a, L, s);
    KDN_TRYK((segment_phase<P, InT>(p, 1, aux)));
    KDN_TRY(hipEventRecord(evR[bb], aux));
    KDN_TRY(hipStreamWaitEvent(st, evR[bb], 0));
    KDN_TRYK((segment_phase<P, InT>(p, PH_CARRIES, st)));
    KDN_TRYK((segment_phase<P, InT>(p, PH_GRAD, st)));
    KDN_TRY(hipEventRecord(evG[bb], st));
    if (i > 0) {
      KDN_TRY(hipStreamWaitEvent(aux, evG[(i - 1) % L.nbuf], 0));
      KDN_TRYK((segment_phase<P, InT>(segment_params(base, a, L, s + 1), PH_DX, aux)));
    }
  }
  KDN_TRY(hipStreamWaitEvent(aux, evG[(L.nsegs - 1) % L.nbuf], 0));
  KDN_TRYK((segment_phase<P, InT>(segment_params(base, a, L, 0), PH_DX, aux)));
  KDN_TRY(hipEventRecord(evDone, aux));
  KDN_TRY(hipStreamWaitEvent(st, evDone, 0));
#undef KDN_TRY
#undef KDN_TRYK
  return KDN_OK;
}

// Checks the call and fills the parameters shared by every segment.
static int bwd_params(const kdn_scan_bwd_args* a, Params& p, BwdLayout& L) {
  const int rc = bwd_check(a);
  if (rc != KDN_OK) return rc;
  const kdn_scan_args* f = a->fwd;
  L = bwd_layout(f, a->dinv_tau != nullptr);
  if (!a->workspace || a->workspace_bytes < L.total) return KDN_ERR_WORKSPACE_TOO_SMALL;
  if (!aligned(a->workspace, 256)) return KDN_ERR_MISALIGNED;
  if (f->B > 65535 || f->H > 65535 || L.seg > 0x7fffffff) return KDN_ERR_UNSUPPORTED;
  p = Params{};
  p.B = f->B; p.T = f->T; p.H = f->H; p.nch = bwd_chunks(f);
  p.q = f->q; p.qs0 = f->q_stride[0]; p.qs1 = f->q_stride[1]; p.qs2 = f->q_stride[2];
  p.k = f->k; p.ks0 = f->k_stride[0]; p.ks1 = f->k_stride[1]; p.ks2 = f->k_stride[2];
  p.v = f->v; p.vs0 = f->v_stride[0]; p.vs1 = f->v_stride[1]; p.vs2 = f->v_stride[2];
  p.beta = f->beta; p.bs0 = f->beta_stride[0]; p.bs1 = f->beta_stride[1]; p.bs2 = f->beta_stride[2];
  p.decay = f->decay; p.ds0 = f->decay_stride[0]; p.ds1 = f->decay_stride[1]; p.ds2 = f->decay_stride[2];
  p.omega = reinterpret_cast<const __bf16*>(f->omega_bf16); p.phase = f->phase;
  p.inv_tau = f->inv_tau; p.normalize = f->normalize_input;
  p.init = f->initial_state;
  p.is0 = f->init_stride[0]; p.is1 = f->init_stride[1]; p.is2 = f->init_stride[2]; p.is3 = f->init_stride[3];
  p.dy = a->dy; p.ys0 = a->dy_stride[0]; p.ys1 = a->dy_stride[1]; p.ys2 = a->dy_stride[2];
  p.dfin = a->d_final_state;
  p.fs0 = a->dfinal_stride[0]; p.fs1 = a->dfinal_stride[1]; p.fs2 = a->dfinal_stride[2]; p.fs3 = a->dfinal_stride[3];
  p.dq = a->dq; p.dqs0 = a->dq_stride[0]; p.dqs1 = a->dq_stride[1]; p.dqs2 = a->dq_stride[2];
  p.dk = a->dk; p.dks0 = a->dk_stride[0]; p.dks1 = a->dk_stride[1]; p.dks2 = a->dk_stride[2];
  p.dv = a->dv; p.dvs0 = a->dv_stride[0]; p.dvs1 = a->dv_stride[1]; p.dvs2 = a->dv_stride[2];
  p.dbeta = a->dbeta; p.dbs0 = a->dbeta_stride[0]; p.dbs1 = a->dbeta_stride[1]; p.dbs2 = a->dbeta_stride[2];
  p.ddecay = a->ddecay; p.dds0 = a->ddecay_stride[0]; p.dds1 = a->ddecay_stride[1]; p.dds2 = a->ddecay_stride[2];
  p.gout = a->d_initial_state;
  p.gos0 = a->dinit_stride[0]; p.gos1 = a->dinit_stride[1]; p.gos2 = a->dinit_stride[2]; p.gos3 = a->dinit_stride[3];
  p.omt = reinterpret_cast<const bf16x8*>(static_cast<unsigned char*>(a->workspace) + L.omt_off);
  p.omega_lo = reinterpret_cast<const __bf16*>(f->omega_lo);
  p.oms = f->omega_head_stride; p.phs = f->phase_head_stride;
  p.inv_tau_head = f->inv_tau_head;
  p.no_renorm = f->no_renorm ? 1 : 0;
  p.linear = f->rule == 1 ? 1 : 0;
  p.omt_hs = f->omega_head_stride ? (f->omega_lo ? 2 : 1) * OMT_ENTRIES : 0;
  p.dinv_tau = a->dinv_tau;
  p.dit = a->dinv_tau ? reinterpret_cast<float*>(static_cast<unsigned char*>(a->workspace) + L.dit_off) : nullptr;
  return KDN_OK;
}

// bf16 inputs: the D = 512 contractions take bf16 operands with fp32 accumulation, the forward's policy
// for bf16 inputs; the lift and the 64 x 64 chunk algebra stay in fp32 MFMA.
static int bwd_run64(const kdn_scan_bwd_args* a, hipStream_t st, hipStream_t aux) {
  Params p;
  BwdLayout L;
  const int rc = bwd_params(a, p, L);
  if (rc != KDN_OK) return rc;
  if (a->fwd->in_dtype == KDN_DTYPE_BF16) return bwd_schedule<PrecBF16, __bf16>(a, p, L, st, aux);
  return bwd_schedule<PrecF32, float>(a, p, L, st, aux);
}

// ------------------------------------------------------------------------------------------------
// d_v = 16, 32 or 128 at D = 512: the kernels above are built for 64 value columns.  The value columns of
// the rule are independent given the keys, beta and lambda: row j of S evolves from column j of v alone
// (S_t[j] = lambda_t S_{t-1}[j] (I - beta_t k k^T) + beta_t v_t[j] k^T), and y[:, j] reads row j only.
// So the backward of d_v = 128 is the 64-wide backward of each column half, whose gradients of q, k,
// beta, lambda and 1/tau add up (the second half's go to workspace buffers, then are added in a fixed
// order); the backward of d_v = 16 or 32 is the 64-wide backward of v, dL/dy, the initial state and
// dL/dS_T padded with zero columns (zero columns of S and of dL/dS stay zero and add exact zeros to every
// shared gradient), with dv and dL/dS_0 cut back to d_v columns.
namespace vsplit {

static bool applies(const kdn_scan_args* f) {
  return f && f->D == D && f->feature_mode == 0 && (f->d_v == 16 || f->d_v == 32 || f->d_v == 128);
}

// The 64-wide request's arguments and the buffers after its workspace.
struct Plan {
  kdn_scan_args f64;
  size_t base, total;
  // d_v = 128: the second half's shared gradients (contiguous [B][T][H][64] / [B][T][H] / [H])
  size_t dq, dk, dbeta, ddecay, dit;
  // d_v < 64: padded copies (contiguous [B][T][H][64] rows, [B][H][512][64] states)
  size_t v, dy, s0, dfin, dv, gout;
};

static size_t up(size_t x) { return (x + 255) / 256 * 256; }

static Plan plan(const kdn_scan_bwd_args* a) {
  Plan P;
  P.f64 = *a->fwd;
  P.f64.d_v = DV;
  const kdn_scan_args* f = a->fwd;
  const size_t rows = (size_t)f->B * f->T * f->H, states = (size_t)f->B * f->H * D * DV;
  P.base = up(bwd_layout(&P.f64, a->dinv_tau != nullptr).total);
  size_t o = P.base;
  P.dq = P.dk = P.dbeta = P.ddecay = P.dit = P.v = P.dy = P.s0 = P.dfin = P.dv = P.gout = 0;
  if (f->d_v > DV) {
    P.dq = o; o += up(rows * DV * 4);
    P.dk = o; o += up(rows * DV * 4);
    P.dbeta = o; o += up(rows * 4);
    if (a->ddecay) { P.ddecay = o; o += up(rows * 4); }
    if (a->dinv_tau) { P.dit = o; o += up((size_t)f->H * 4); }
  } else {
    P.v = o; o += up(rows * DV * dtype_size(f->in_dtype));
    P.dy = o; o += up(rows * DV * 4);
    P.dv = o; o += up(rows * DV * 4);
    if (f->initial_state) { P.s0 = o; o += up(states * 4); }
    if (a->d_final_state) { P.dfin = o; o += up(states * 4); }
    if (a->d_initial_state) { P.gout = o; o += up(states * 4); }
  }
  P.total = o;
  return P;
}

// rows r = (b, t, h) of a (B, T, H, width) tensor given by three strides, and of a contiguous copy
struct Rows {
  int64_t T, H;
  __device__ __forceinline__ int64_t off(int64_t r, int64_t s0, int64_t s1, int64_t s2) const {
    const int64_t h = r % H, bt = r / H;
    return (bt / T) * s0 + (bt % T) * s1 + h * s2;
  }
};

// dst[r][c] = c < w ? src(r, c) : 0 for c < 64 (zero-padded contiguous copy)
template <typename T>
__global__ void __launch_bounds__(256) pad_rows(const T* src, int64_t s0, int64_t s1, int64_t s2, Rows R, int w,
                                                T* dst, int64_t n) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n * DV; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / DV;
    const int c = (int)(i % DV);
    dst[i] = c < w ? src[R.off(r, s0, s1, s2) + c] : (T)0.f;
  }
}

// dst(r, c) = src[r][c] for c < w
__global__ void __launch_bounds__(256) unpad_rows(const float* src, float* dst, int64_t s0, int64_t s1, int64_t s2,
                                                  Rows R, int w, int64_t n) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n * w; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / w;
    const int c = (int)(i % w);
    dst[R.off(r, s0, s1, s2) + c] = src[r * DV + c];
  }
}

// dst(r, c) += src[r][c] for c < w (src rows of w contiguous values)
__global__ void __launch_bounds__(256) add_rows(const float* src, float* dst, int64_t s0, int64_t s1, int64_t s2,
                                                Rows R, int w, int64_t n) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n * w; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / w;
    const int c = (int)(i % w);
    dst[R.off(r, s0, s1, s2) + c] += src[i];
  }
}

// states [b][h][d][c] (four strides) <-> contiguous [B][H][512][64], zero-padded / cut to w columns
__global__ void __launch_bounds__(256) pad_state(const float* src, int64_t s0, int64_t s1, int64_t s2, int64_t s3,
                                                 int64_t H, int w, float* dst, int64_t n) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int c = (int)(i % DV);
    const int64_t d = (i / DV) % D, bh = i / ((int64_t)DV * D);
    dst[i] = c < w ? src[(bh / H) * s0 + (bh % H) * s1 + d * s2 + c * s3] : 0.f;
  }
}
__global__ void __launch_bounds__(256) unpad_state(const float* src, float* dst, int64_t s0, int64_t s1, int64_t s2,
                                                   int64_t s3, int64_t H, int w, int64_t n) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int c = (int)(i % DV);
    if (c >= w) continue;
    const int64_t d = (i / DV) % D, bh = i / ((int64_t)DV * D);
    dst[(bh / H) * s0 + (bh % H) * s1 + d * s2 + c * s3] = src[i];
  }
}

static unsigned grid_for(int64_t n) {
  const int64_t g = (n + 255) / 256;
  return (unsigned)(g < 8192 ? (g > 0 ? g : 1) : 8192);
}

// the request's checks as the 64-wide one's (the pointers and strides of the d_v-wide tensors are what
// that one reads or writes, with the layouts above)
static int check(const kdn_scan_bwd_args* a, Plan& P) {
  if (!a || !a->fwd) return KDN_ERR_INVALID_ARGUMENT;
  P = plan(a);
  kdn_scan_bwd_args b = *a;
  b.fwd = &P.f64;
  return bwd_check(&b);
}

static size_t workspace_bytes(const kdn_scan_bwd_args* a) {
  Plan P;
  return check(a, P) == KDN_OK ? P.total : 0;
}

// the 64-wide backward's segments (each of its runs has the same ones)
static int64_t segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks) {
  Plan P;
  if (check(a, P) != KDN_OK) return 0;
  const BwdLayout L = bwd_layout(&P.f64, a->dinv_tau != nullptr);
  if (segment_chunks) *segment_chunks = L.seg;
  return L.nsegs;
}

static int run(const kdn_scan_bwd_args* a, hipStream_t st, hipStream_t aux) {
  const kdn_scan_args* f = a->fwd;
  Plan P;
  const int rc0 = check(a, P);
  if (rc0 != KDN_OK) return rc0;
  kdn_scan_bwd_args b = *a;
  b.fwd = &P.f64;
  if (!a->workspace || a->workspace_bytes < P.total) return KDN_ERR_WORKSPACE_TOO_SMALL;
  if (!aligned(a->workspace, 256)) return KDN_ERR_MISALIGNED;
  if (f->B > 65535 || f->H > 65535) return KDN_ERR_UNSUPPORTED;
  unsigned char* ws = static_cast<unsigned char*>(a->workspace);
  const Rows R = {f->T, f->H};
  const int64_t rows = f->B * f->T * f->H, states = f->B * f->H * (int64_t)D * DV;
  b.workspace_bytes = P.base;
  if (f->d_v > DV) {
    // first half: the caller's tensors as they are (64-column views)
    int rc = bwd_run64(&b, st, aux);
    if (rc != KDN_OK) return rc;
    // second half: columns 64 .. 127 of v, dL/dy, the states and dv; its shared gradients to the workspace
    kdn_scan_args g = P.f64;
    g.v = static_cast<const unsigned char*>(f->v) + DV * dtype_size(f->in_dtype);
    if (f->initial_state) g.initial_state = f->initial_state + DV * f->init_stride[3];
    kdn_scan_bwd_args c = *a;
    c.fwd = &g;
    c.workspace_bytes = P.base;
    c.dy = a->dy + DV;
    if (a->d_final_state) c.d_final_state = a->d_final_state + DV * a->dfinal_stride[3];
    c.dv = a->dv + DV;
    if (a->d_initial_state) c.d_initial_state = a->d_initial_state + DV * a->dinit_stride[3];
    const int64_t rs[3] = {f->T * f->H * DV, f->H * DV, DV}, ss[3] = {f->T * f->H, f->H, 1};
    c.dq = reinterpret_cast<float*>(ws + P.dq);
    c.dk = reinterpret_cast<float*>(ws + P.dk);
    c.dbeta = reinterpret_cast<float*>(ws + P.dbeta);
    c.ddecay = a->ddecay ? reinterpret_cast<float*>(ws + P.ddecay) : nullptr;
    c.dinv_tau = a->dinv_tau ? reinterpret_cast<float*>(ws + P.dit) : nullptr;
    for (int i = 0; i < 3; ++i) {
      c.dq_stride[i] = rs[i]; c.dk_stride[i] = rs[i];
      c.dbeta_stride[i] = ss[i]; c.ddecay_stride[i] = ss[i];
    }
    rc = bwd_run64(&c, st, aux);
    if (rc != KDN_OK) return rc;
    // first half + second half, element by element
    hipLaunchKernelGGL(add_rows, dim3(grid_for(rows * DV)), dim3(256), 0, st, c.dq, a->dq, a->dq_stride[0],
                       a->dq_stride[1], a->dq_stride[2], R, DV, rows);
    hipLaunchKernelGGL(add_rows, dim3(grid_for(rows * DV)), dim3(256), 0, st, c.dk, a->dk, a->dk_stride[0],
                       a->dk_stride[1], a->dk_stride[2], R, DV, rows);
    hipLaunchKernelGGL(add_rows, dim3(grid_for(rows)), dim3(256), 0, st, c.dbeta, a->dbeta, a->dbeta_stride[0],
                       a->dbeta_stride[1], a->dbeta_stride[2], R, 1, rows);
    if (a->ddecay)
      hipLaunchKernelGGL(add_rows, dim3(grid_for(rows)), dim3(256), 0, st, c.ddecay, a->ddecay, a->ddecay_stride[0],
                         a->ddecay_stride[1], a->ddecay_stride[2], R, 1, rows);
    if (a->dinv_tau) {
      const Rows Rh = {1, f->H};  // H rows of one value: offset h
      hipLaunchKernelGGL(add_rows, dim3(1), dim3(256), 0, st, c.dinv_tau, a->dinv_tau, (int64_t)0, (int64_t)0,
                         (int64_t)1, Rh, 1, f->H);
    }
    return launch_status();
  }
  // d_v < 64: zero-padded copies in, the 64-wide backward, d_v columns out
  kdn_scan_args g = P.f64;
  const int w = (int)f->d_v;
  const size_t isz = dtype_size(f->in_dtype);
  void* v64 = ws + P.v;
  if (isz == 2)
    hipLaunchKernelGGL(pad_rows<__bf16>, dim3(grid_for(rows * DV)), dim3(256), 0, st,
                       static_cast<const __bf16*>(f->v), f->v_stride[0], f->v_stride[1], f->v_stride[2], R, w,
                       static_cast<__bf16*>(v64), rows);
  else
    hipLaunchKernelGGL(pad_rows<float>, dim3(grid_for(rows * DV)), dim3(256), 0, st,
                       static_cast<const float*>(f->v), f->v_stride[0], f->v_stride[1], f->v_stride[2], R, w,
                       static_cast<float*>(v64), rows);
  g.v = v64;
  g.v_stride[0] = f->T * f->H * DV; g.v_stride[1] = f->H * DV; g.v_stride[2] = DV;
  if (f->initial_state) {
    float* s0 = reinterpret_cast<float*>(ws + P.s0);
    hipLaunchKernelGGL(pad_state, dim3(grid_for(states)), dim3(256), 0, st, f->initial_state, f->init_stride[0],
                       f->init_stride[1], f->init_stride[2], f->init_stride[3], f->H, w, s0, states);
    g.initial_state = s0;
    g.init_stride[0] = f->H * (int64_t)D * DV; g.init_stride[1] = (int64_t)D * DV; g.init_stride[2] = DV;
    g.init_stride[3] = 1;
  }
  kdn_scan_bwd_args c = *a;
  c.fwd = &g;
  c.workspace_bytes = P.base;
  float* dy64 = reinterpret_cast<float*>(ws + P.dy);
  hipLaunchKernelGGL(pad_rows<float>, dim3(grid_for(rows * DV)), dim3(256), 0, st, a->dy, a->dy_stride[0],
                     a->dy_stride[1], a->dy_stride[2], R, w, dy64, rows);
  c.dy = dy64;
  c.dy_stride[0] = f->T * f->H * DV; c.dy_stride[1] = f->H * DV; c.dy_stride[2] = DV;
  if (a->d_final_state) {
    float* df = reinterpret_cast<float*>(ws + P.dfin);
    hipLaunchKernelGGL(pad_state, dim3(grid_for(states)), dim3(256), 0, st, a->d_final_state, a->dfinal_stride[0],
                       a->dfinal_stride[1], a->dfinal_stride[2], a->dfinal_stride[3], f->H, w, df, states);
    c.d_final_state = df;
    c.dfinal_stride[0] = f->H * (int64_t)D * DV; c.dfinal_stride[1] = (int64_t)D * DV; c.dfinal_stride[2] = DV;
    c.dfinal_stride[3] = 1;
  }
  float* dv64 = reinterpret_cast<float*>(ws + P.dv);
  c.dv = dv64;
  c.dv_stride[0] = f->T * f->H * DV; c.dv_stride[1] = f->H * DV; c.dv_stride[2] = DV;
  float* go = a->d_initial_state ? reinterpret_cast<float*>(ws + P.gout) : nullptr;
  if (go) {
    c.d_initial_state = go;
    c.dinit_stride[0] = f->H * (int64_t)D * DV; c.dinit_stride[1] = (int64_t)D * DV; c.dinit_stride[2] = DV;
    c.dinit_stride[3] = 1;
  }
  int rc = launch_status();
  if (rc != KDN_OK) return rc;
  rc = bwd_run64(&c, st, aux);
  if (rc != KDN_OK) return rc;
  hipLaunchKernelGGL(unpad_rows, dim3(grid_for(rows * w)), dim3(256), 0, st, dv64, a->dv, a->dv_stride[0],
                     a->dv_stride[1], a->dv_stride[2], R, w, rows);
  if (go)
    hipLaunchKernelGGL(unpad_state, dim3(grid_for(states)), dim3(256), 0, st, go, a->d_initial_state,
                       a->dinit_stride[0], a->dinit_stride[1], a->dinit_stride[2], a->dinit_stride[3], f->H, w, states);
  return launch_status();
}

}  // namespace vsplit

static int bwd_run(const kdn_scan_bwd_args* a, void* stream, void* aux_stream);

// ------------------------------------------------------------------------------------------------
// D = 128 and 256 (feature replication, kdn_frep.hip): the 512-wide backward on replicated Omega and
// phases, from L(S_0) with dL/dS'_T = L(dL/dS_T); dL/dS_0 = P(dL/dS'_0).  Its workspace: the 512-wide
// request's, then the tables and three 512-wide states (S'_0, dL/dS'_T, dL/dS'_0).
namespace frep {

// The 512-wide request with the caller's pointers (for sizing and checks) and its workspace bytes.
static size_t base_bytes(const kdn_scan_bwd_args* a, kdn_scan_args* w) {
  *w = frep_wide(a->fwd, nullptr, nullptr);
  kdn_scan_bwd_args g = *a;
  g.fwd = w;
  return kdn_scan_bwd_workspace_bytes(&g);
}

static size_t workspace_bytes(const kdn_scan_bwd_args* a) {
  if (a->fwd->cu_seqlens || a->fwd->state_slots) return 0;
  kdn_scan_args w;
  const size_t base = base_bytes(a, &w);
  return base ? frep_layout(a->fwd, base, 3).total : 0;
}

static int64_t segments(const kdn_scan_bwd_args* a, int64_t* segment_chunks) {
  if (workspace_bytes(a) == 0) return 0;
  kdn_scan_args w = frep_wide(a->fwd, nullptr, nullptr);
  kdn_scan_bwd_args g = *a;
  g.fwd = &w;
  return kdn_scan_bwd_segments(&g, segment_chunks);
}

static int run(const kdn_scan_bwd_args* a, void* stream, void* aux) {
  const kdn_scan_args* f = a->fwd;
  const size_t need = workspace_bytes(a);
  if (!need) {  // the 512-wide request's own argument error (its checks at d_v = 64), else unsupported
    kdn_scan_args wc = frep_wide(f, nullptr, nullptr);
    wc.d_v = 64;
    kdn_scan_bwd_args gc = *a;
    gc.fwd = &wc;
    const int rc = bwd_check(&gc);
    return rc != KDN_OK ? rc : KDN_ERR_UNSUPPORTED;
  }
  if (!a->workspace || a->workspace_bytes < need) return KDN_ERR_WORKSPACE_TOO_SMALL;
  if (!aligned(a->workspace, 256)) return KDN_ERR_MISALIGNED;
  kdn_scan_args w0;
  const FrepLayout L = frep_layout(f, base_bytes(a, &w0), 3);
  kdn_scan_args w = frep_wide(f, &L, a->workspace);
  w.workspace = f->workspace;
  w.workspace_bytes = f->workspace_bytes;
  unsigned char* ws = static_cast<unsigned char*>(a->workspace);
  float* s0 = reinterpret_cast<float*>(ws + L.state[0]);
  float* dsT = reinterpret_cast<float*>(ws + L.state[1]);
  float* ds0 = reinterpret_cast<float*>(ws + L.state[2]);
  int64_t cs[4];
  frep_contiguous_strides(f, cs);
  kdn_scan_bwd_args g = *a;
  g.fwd = &w;
  g.workspace_bytes = L.base;
  if (f->initial_state) {
    w.initial_state = s0;
    for (int i = 0; i < 4; ++i) w.init_stride[i] = cs[i];
  }
  if (a->d_final_state) {
    g.d_final_state = dsT;
    for (int i = 0; i < 4; ++i) g.dfinal_stride[i] = cs[i];
  }
  if (a->d_initial_state) {
    g.d_initial_state = ds0;
    for (int i = 0; i < 4; ++i) g.dinit_stride[i] = cs[i];
  }
  const hipStream_t st = as_stream(stream);
  int rc = frep_tables(f, &L, a->workspace, st);
  if (rc == KDN_OK && f->initial_state) rc = frep_state_lift(f, f->initial_state, f->init_stride, s0, st);
  if (rc == KDN_OK && a->d_final_state) rc = frep_state_lift(f, a->d_final_state, a->dfinal_stride, dsT, st);
  if (rc != KDN_OK) return rc;
  rc = bwd_run(&g, stream, aux);
  if (rc != KDN_OK || !a->d_initial_state) return rc;
  return frep_state_fold(f, ds0, a->d_initial_state, a->dinit_stride, st);
}

}  // namespace frep

static int bwd_run(const kdn_scan_bwd_args* a, void* stream, void* aux_stream) {
  if (a && general_bwd_applies(a->fwd)) return general_bwd(a, stream);  // one stream
  if (a && a->fwd && frep_applies(a->fwd)) return frep::run(a, stream, aux_stream);
  const hipStream_t st = as_stream(stream), aux = aux_stream ? as_stream(aux_stream) : nullptr;
  if (a && vsplit::applies(a->fwd)) return vsplit::run(a, st, aux);
  return bwd_run64(a, st, aux);
}

extern "C" int kdn_delta_scan_bwd(const kdn_scan_bwd_args* a, void* stream) { return bwd_run(a, stream, nullptr); }

extern "C" int kdn_delta_scan_bwd_streams(const kdn_scan_bwd_args* a, void* stream, void* aux_stream) {
  return bwd_run(a, stream, aux_stream);
}

extern "C" int kdn_scan_bwd_phase(const kdn_scan_bwd_args* a, int phase, int64_t segment, void* stream) {
  if (phase < 0 || phase > 4) return KDN_ERR_INVALID_ARGUMENT;
  if (a && general_bwd_applies(a->fwd)) return KDN_ERR_UNSUPPORTED;  // no phase entry points at D = 1024
  if (a && vsplit::applies(a->fwd)) return KDN_ERR_UNSUPPORTED;        // nor for d_v other than 64
  if (a && a->fwd && frep_applies(a->fwd)) return KDN_ERR_UNSUPPORTED;  // nor for D = 128, 256
  Params p;
  BwdLayout L;
  const int rc = bwd_params(a, p, L);
  if (rc != KDN_OK) return rc;
  const hipStream_t st = as_stream(stream);
  if (phase == 0) return bwd_start(a, p, L, st, nullptr);
  if (segment < 0 || segment >= L.nsegs) return KDN_ERR_INVALID_ARGUMENT;
  const Params ps = segment_params(p, a, L, segment);
  if (a->fwd->in_dtype == KDN_DTYPE_BF16) return segment_phase<PrecBF16, __bf16>(ps, phase, st);
  return segment_phase<PrecF32, float>(ps, phase, st);
}

}  // namespace kdn
