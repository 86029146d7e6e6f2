// Learned per-cell preconditioner (no reference counterpart: the reference's psol is an
// identity, src/foeuler/foeuler.f90:434).  A 3x128 SiLU MLP with two rounds of one-hop message
// passing over face neighbours emits, per cell, a 5x5 block B^ = I + o[0:25] and 5 neighbour
// weights s = o[25:30] (the 4 face neighbours in neib slot order, then the cell itself):
//   t_c = B^_c (r_c / S),   z_c = S ((1 + s_4) t_c + sum_j s_j t_nb(j))
// (S = per-variable RMS of the state), a fixed linear operator for GMRES.  Trained with Adam on
// pairs (r, target) at the solver's states, loss |S^-1 (P r - target)|^2.
//
// Dense layers run on MFMA (v_mfma_f32_16x16x32_bf16): BF16 weights and activations, FP32 accumulation; the
// forward layers and the backward data products in persistent workgroups (mlp_layer_kernel), the weight
// gradients as reductions over cells (wgrad_kernel).  FP32 master weights and Adam moments.  Parameter packing (flat FP32): W0[20][128] b0 W1[256][128] b1 W2[256][128] b2
// W3[128][30] b3, the same as the oracle (oracle/learned.c).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <vector>

#include "context.h"
#include "learned_space.h"

namespace fos {

constexpr int NPAR = NI * NH + NH + 2 * NH * NH + NH + 2 * NH * NH + NH + NH * NO + NO;
constexpr int OFF_W0 = 0, OFF_B0 = OFF_W0 + NI * NH, OFF_W1 = OFF_B0 + NH, OFF_B1 = OFF_W1 + 2 * NH * NH;
constexpr int OFF_W2 = OFF_B1 + NH, OFF_B2 = OFF_W2 + 2 * NH * NH, OFF_W3 = OFF_B2 + NH, OFF_B3 = OFF_W3 + NH * NO;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __host__ inline uint16_t f2bf(float f) {  // round to nearest even
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(uint16_t, (__bf16)f);  // v_cvt_pk_bf16_f32 (round to nearest even)
#endif
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// sigmoid by the hardware reciprocal (1 ulp) instead of the IEEE division sequence
__device__ inline float sigm_f(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ inline float silu_f(float x) { return x * sigm_f(x); }
__device__ inline float dsilu_f(float x) {
  const float s = sigm_f(x);
  return s * (1.0f + x * (1.0f - s));
}

struct Learned : LearnedSpace<DBuf> {
  int nC = 0;
  bool ready = false, haveO = false;  // parameters set; network output O computed for the mesh
  long long step = 0;
  DBuf<float> par, m1, m2, grad, bias;  // bias: b0 b1 b2 b3(padded 32)
  // BF16 copies: forward operands (n-major, [out][in]) and backward-data operands ([in][out])
  DBuf<uint16_t> W0t, W1t, W2t, W3t, W1b, W2b, W3b;
  DBuf<int> nbr;          // [nC][4] cell neighbours (-1 none)
  DBuf<float> geo;        // [nC][13] log(v/vmean), area normals / v^(2/3) per neib slot
  DBuf<float> scale;      // [8]: S[5], then scratch
  double *pinned = nullptr, *dpinned = nullptr;  // the loss in host memory, and its device address
  ~Learned() {
    if (pinned) (void)hipHostFree(pinned);
  }
};

void destroy_learned(Learned *l) { delete l; }

namespace {

// ---------------------------------------------------------------- MFMA GEMMs

enum { EPI_SILU = 0, EPI_DSILU = 2, EPI_BF16 = 3 };

// One cell's 20 features, zero-padded to 32, as four octets (BF16): U/S, log(v/vmean), 4 area-normals /
// v^(2/3), gamma c / v^(1/3), |u|/c; from its state U and its 13 geometry features g.
struct FeatIn {
  double U[5];
  float g[13];
};
__device__ inline void feat_load(FeatIn &f, int c, int nC, const double *__restrict__ y, const float *__restrict__ geo) {
#pragma unroll
  for (int k = 0; k < 5; k++) f.U[k] = y[(size_t)k * nC + c];
#pragma unroll
  for (int k = 0; k < 13; k++) f.g[k] = geo[(size_t)13 * c + k];
}
__device__ inline void feat_row(const FeatIn &f, const float *__restrict__ S, float vm13, double gamma, double gm,
                                uint4 (&out)[NIP / 8]) {
  uint16_t x[NIP];
#pragma unroll
  for (int k = 0; k < NIP; k++) x[k] = 0;
#pragma unroll
  for (int k = 0; k < 5; k++) x[k] = f2bf((float)(f.U[k] / S[k]));
#pragma unroll
  for (int k = 0; k < 13; k++) x[5 + k] = f2bf(f.g[k]);
  const double ir = 1.0 / f.U[0];
  const double q2 = (f.U[1] * f.U[1] + f.U[2] * f.U[2] + f.U[3] * f.U[3]) * ir * ir;
  const double p = (gm - 1.0) * (f.U[4] - 0.5 * f.U[0] * q2);
  const double cs = sqrt(fmax(gm * p * ir, 1e-300));
  const double vol13 = exp(f.g[0] / 3.0) * (double)vm13;  // v^(1/3) = exp(log(v/vm)/3) vm^(1/3)
  x[18] = f2bf((float)(gamma * cs / vol13));
  x[19] = f2bf((float)(sqrt(q2) / cs));
#pragma unroll
  for (int q = 0; q < NIP / 8; q++)
    out[q] = make_uint4(x[8 * q] | (uint32_t)x[8 * q + 1] << 16, x[8 * q + 2] | (uint32_t)x[8 * q + 3] << 16,
                        x[8 * q + 4] | (uint32_t)x[8 * q + 5] << 16, x[8 * q + 6] | (uint32_t)x[8 * q + 7] << 16);
}
// features of the cells [c0, c0+R) alone (fos_learned_inputs)
__global__ void features_kernel(int R, int c0, int nC, const double *__restrict__ y, const float *__restrict__ geo,
                                const float *__restrict__ S, double gamma, double gm, uint16_t *__restrict__ X) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  FeatIn f;
  uint4 x[NIP / 8];
  feat_load(f, c0 + i, nC, y, geo);
  feat_row(f, S, geo[(size_t)13 * nC], gamma, gm, x);
#pragma unroll
  for (int q = 0; q < NIP / 8; q++) reinterpret_cast<uint4 *>(&X[(size_t)i * NIP])[q] = x[q];
}
// The output scale: O[c] *= k_c = min(1, x_c[18] (1 + x_c[19])) from the cell's (BF16) features,
// its CFL number gamma (c + |u|) / v^(1/3) capped at 1: the operator tends to the identity as the
// time step shrinks, where the Newton matrix I - gamma J differs from I by O(CFL).
__device__ inline float out_kappa(uint4 octet2) {
  return fminf(1.f, bf2f((uint16_t)octet2.y) * (1.f + bf2f((uint16_t)(octet2.y >> 16))));
}

// Layer out[r][c] = epi(sum_k A[r][k] Bn[c][k]) for all N columns -- EPI_SILU adds the bias (forward),
// EPI_DSILU multiplies by silu' of the forward pass's pre and EPI_BF16 rounds (the backward data
// products) -- on the gfx950 v_mfma_f32_16x16x32_bf16 (8 bf16 per lane and operand: lane l holds row l%16
// and the k-octet l/16 of each 32-wide k step; A and B use the same octets, so the product sums every k
// once).  Persistent workgroups keep the whole weight matrix in LDS and stream 16-row tiles per wave, so
// A is read from HBM once.
// The product is formed transposed (weights as the row operand), and the weight rows are dealt to the
// MFMAs' rows so that a lane ends up with 8 consecutive columns of one row in two accumulators: it stores
// them as one 16-byte vector, and they are the lane's own k-octet of the next layer.
// FEAT (layer 0): a wave takes 64 rows at a time; each lane forms one row's features from the state and
// leaves them in LDS for the four tiles.  kappa receives the rows' output scale and, when given, X the
// features (training).
// MEAN: the k >= 128 half of A is the mean of the row's neighbours' k < 128 half (message passing
// fused into the load, summed in slot order); meanOut, when given, receives it in the k >= 128 half of
// A's rows (training: the weight gradients read it).
// TAIL (layer 2): the output layer's 128 x 32 product and the output scale follow on the lane's own
// octets, so the last hidden layer is not stored (outb, when given, still receives it: training).
// At 1.5M cells, per layer: 0 with the features 48 + 184 -> 124 us, 1 399 -> 312 us, 2 with the output
// layer and its scale 399 + 110 + 102 -> 328 us (the whole set-up and apply 1,380 -> 831 us), all bitwise
// the same.  The mean layers are bound by the latency of the gathers and the arithmetic of the means and
// silu at two waves per SIMD (64 KB of weights per workgroup); 384 and 512 threads around the same weights
// were 14 % and 50 % slower (fewer registers per wave, spills).
struct LayerArgs {
  int R, lda, ldo;
  const uint16_t *A, *Bn;
  const int *nbr;
  const float *bias;
  float *pre;        // [R][N], null for inference
  uint16_t *outb, *meanOut;
  // FEAT
  const double *y;
  const float *geo, *S;
  double gamma, gm;
  int c0, nC;
  uint16_t *X;
  float *kappa;
  // TAIL
  const uint16_t *B3;
  const float *bias3;
  float *O;
};
// LDS octet slot of octet o in row n: the 16 rows that one operand read touches (8 apart in groups of
// four) land on distinct bank groups
template <int NOCT>
__device__ inline int oct_slot(int n, int o) {
  return n * NOCT + (o ^ (NOCT >= 16 ? (n & 3) | ((n >> 1) & 12) : (n >> 3) & 3));
}
// Memory is read and written with four consecutive lanes on 64 consecutive bytes of a row (lane l: row
// l / 4, 16-byte piece l % 4); the MFMAs want row l % 16, octet l / 16.  In that order no two neighbouring
// lanes share a row, every 16 bytes are an access of their own to the L1, and the L1 bounded the mean
// layers (1.5M cells: 181M accesses a layer, 0.79 per CU and cycle; now 38M, 0.22).  The neighbours are summed in memory order, and
// four lane permutations per octet change the order (to_mfma, from_mfma).
__device__ inline uint4 lane_perm(int from, uint4 v) {
  return make_uint4(__builtin_amdgcn_ds_bpermute(4 * from, v.x), __builtin_amdgcn_ds_bpermute(4 * from, v.y),
                    __builtin_amdgcn_ds_bpermute(4 * from, v.z), __builtin_amdgcn_ds_bpermute(4 * from, v.w));
}
constexpr int TPB = 256;
template <int K, int N, bool FEAT, bool MEAN, bool TAIL, int EPI>
__global__ __launch_bounds__(TPB) void mlp_layer_kernel(LayerArgs P) {
  static_assert(K % 32 == 0 && N % 32 == 0 && (!MEAN || K == 256) && (!FEAT || K == NIP) && (!TAIL || N == NH),
                "layer shape");
  constexpr int KS = K / 32, NT = N / 16, NOCT = K / 8;
  extern __shared__ uint4 lds_raw[];
  uint4 *sB = lds_raw, *s3 = lds_raw + N * NOCT;  // TAIL: the output layer's weights; FEAT: the waves' features
  for (int i = threadIdx.x; i < N * NOCT; i += TPB) {
    const int n = i / NOCT, o = i % NOCT;
    sB[oct_slot<NOCT>(n, o)] = *reinterpret_cast<const uint4 *>(&P.Bn[(size_t)n * K + 8 * o]);
  }
  if (TAIL)
    for (int i = threadIdx.x; i < NOP * NH / 8; i += TPB) {
      const int n = i / (NH / 8), o = i % (NH / 8);
      s3[oct_slot<NH / 8>(n, o)] = *reinterpret_cast<const uint4 *>(&P.B3[(size_t)n * NH + 8 * o]);
    }
  __shared__ float4 sBias[N / 4];
  if (EPI == EPI_SILU && threadIdx.x < N / 4) sBias[threadIdx.x] = reinterpret_cast<const float4 *>(P.bias)[threadIdx.x];
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, kq = lane >> 4, R = P.R;
  const int mr = lane >> 2, mp = lane & 3;  // row and piece in memory order
  auto to_mfma = [&](uint4 v) { return lane_perm(4 * lr + kq, v); };
  auto from_mfma = [&](uint4 v) { return lane_perm(mr + 16 * mp, v); };
  const int n0 = 8 * (lr >> 2) + (lr & 3);  // this lane's weight row within 32 columns, + 4 for the odd tile
  // XCD-aware tiling: workgroup b runs on XCD b % 8 (round-robin dispatch; the grid is a multiple of
  // 8), and each XCD walks its own contiguous eighth of the tiles, so the rows a tile's neighbours
  // read (nearby in the chunk numbering) sit in the same XCD's L2
  constexpr int ROWS = FEAT ? 64 : 16;  // rows a wave takes at a time
  const int nTiles = (R + ROWS - 1) / ROWS, wpb = TPB >> 6;
  const int xcd = blockIdx.x & 7, perX = (nTiles + 7) / 8;
  const int tBeg = min(nTiles, xcd * perX), tEnd = min(nTiles, tBeg + perX);
  const int stride = (gridDim.x >> 3) * wpb;
  constexpr int KA = MEAN ? KS / 2 : KS;  // k steps read directly from A
  auto load_a = [&](int tile, uint4 (&a)[KA]) {
    const int row = tile * 16 + mr;
    const bool in = tile < tEnd && row < R;
    const uint16_t *ar = P.A + (size_t)(in ? row : 0) * P.lda + 8 * mp;
#pragma unroll
    for (int st = 0; st < KA; st++) a[st] = in ? *reinterpret_cast<const uint4 *>(ar + 32 * st) : make_uint4(0u, 0u, 0u, 0u);
  };
  auto load_nb = [&](int tile) {
    const int row = tile * 16 + mr;
    return tile < tEnd && row < R ? *reinterpret_cast<const int4 *>(&P.nbr[(size_t)NBR * row]) : make_int4(-1, -1, -1, -1);
  };
  constexpr int GN = MEAN ? 4 : 1, GS = MEAN ? KS / 2 : 1;
  auto load_g = [&](int4 nb, uint4 (&g)[GN][GS]) {
    const int d[4] = {nb.x, nb.y, nb.z, nb.w};
#pragma unroll
    for (int j = 0; j < GN; j++)
#pragma unroll
      for (int st = 0; st < GS; st++)
        g[j][st] = d[j] >= 0 ? *reinterpret_cast<const uint4 *>(P.A + (size_t)d[j] * P.lda + 32 * st + 8 * mp)
                             : make_uint4(0u, 0u, 0u, 0u);
  };
  auto mma = [&](f32x4 (&acc)[NT], int st, uint4 av) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const uint4 bv = sB[oct_slot<NOCT>(32 * (t >> 1) + 4 * (t & 1) + n0, 4 * st + kq)];
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bv), __builtin_bit_cast(bf16x8, av),
                                                       acc[t], 0, 0, 0);
    }
  };
  auto finish = [&](int row0, const f32x4 (&acc)[NT]) {
    const int row = row0 + lr, mrow = row0 + mr;
    uint4 hid[N / 32];
#pragma unroll
    for (int u = 0; u < N / 32; u++) {
      const int col = 32 * u + 8 * kq;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] = acc[2 * u + e / 4][e % 4];
      if (EPI == EPI_SILU) {
        const float4 b0 = sBias[col / 4], b1 = sBias[col / 4 + 1];
        const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] += bb[e];
        if (P.pre && row < R) {
          float4 *p4 = reinterpret_cast<float4 *>(&P.pre[(size_t)row * N + col]);
          p4[0] = make_float4(v[0], v[1], v[2], v[3]);
          p4[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = silu_f(v[e]);
      } else if (EPI == EPI_DSILU && row < R) {
        const float4 *p4 = reinterpret_cast<const float4 *>(&P.pre[(size_t)row * N + col]);
        const float4 b0 = p4[0], b1 = p4[1];
        const float bb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] *= dsilu_f(bb[e]);
      }
      hid[u] = make_uint4(f2bf(v[0]) | (uint32_t)f2bf(v[1]) << 16, f2bf(v[2]) | (uint32_t)f2bf(v[3]) << 16,
                          f2bf(v[4]) | (uint32_t)f2bf(v[5]) << 16, f2bf(v[6]) | (uint32_t)f2bf(v[7]) << 16);
      if (!TAIL || P.outb) {
        const uint4 m = from_mfma(hid[u]);
        if (mrow < R) *reinterpret_cast<uint4 *>(&P.outb[(size_t)mrow * P.ldo + 32 * u + 8 * mp]) = m;
      }
    }
    if constexpr (TAIL) {
      f32x4 o3[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int st = 0; st < NH / 32; st++)
#pragma unroll
        for (int t = 0; t < 2; t++)
          o3[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, s3[oct_slot<NH / 8>(4 * t + n0, 4 * st + kq)]),
              __builtin_bit_cast(bf16x8, hid[st]), o3[t], 0, 0, 0);
      const float k = row < R ? P.kappa[row] : 0.f;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const float4 bb = *reinterpret_cast<const float4 *>(&P.bias3[8 * kq + 4 * t]);
        const float4 o = make_float4((o3[t][0] + bb.x) * k, (o3[t][1] + bb.y) * k, (o3[t][2] + bb.z) * k, (o3[t][3] + bb.w) * k);
        const uint4 m = from_mfma(__builtin_bit_cast(uint4, o));
        if (mrow < R) *reinterpret_cast<uint4 *>(&P.O[(size_t)mrow * NOP + 8 * mp + 4 * t]) = m;
      }
    }
  };
  int tile = tBeg + (blockIdx.x >> 3) * wpb + wave;
  if constexpr (FEAT) {
    uint4 *sX = s3 + wave * 64 * (NIP / 8);
    const float vm13 = P.geo[(size_t)13 * P.nC];
    FeatIn f;
    auto fetch = [&](int t) {
      if (t < tEnd && t * 64 + lane < R) feat_load(f, P.c0 + t * 64 + lane, P.nC, P.y, P.geo);
    };
    fetch(tile);
    for (; tile < tEnd; tile += stride) {
      const int mine = tile * 64 + lane;
      if (mine < R) {
        uint4 x[NIP / 8];
        feat_row(f, P.S, vm13, P.gamma, P.gm, x);
        P.kappa[mine] = out_kappa(x[2]);
#pragma unroll
        for (int q = 0; q < NIP / 8; q++) {
          sX[lane * (NIP / 8) + (q ^ ((lane >> 2) & 3))] = x[q];
          if (P.X) reinterpret_cast<uint4 *>(&P.X[(size_t)mine * NIP])[q] = x[q];
        }
      }
      fetch(tile + stride);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __asm__ volatile("" ::: "memory");
#pragma unroll
      for (int h = 0; h < 4; h++) {
        f32x4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int w = 16 * h + lr;
        mma(acc, 0, sX[w * (NIP / 8) + (kq ^ ((w >> 2) & 3))]);
        finish(tile * 64 + 16 * h, acc);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    return;
  }
  // Loads run ahead of their use in the registers that the current tile has done with: the next tile's own
  // rows once its own half is multiplied, its neighbours' rows once the means are formed (so that they are
  // in flight during the epilogue and the next own half), its neighbour list a tile earlier.
  uint4 a[KA], g[GN][GS];
  int4 nb = make_int4(-1, -1, -1, -1), nbn = nb;
  load_a(tile, a);
  if (MEAN) {
    nb = load_nb(tile);
    nbn = load_nb(tile + stride);
    load_g(nb, g);
  }
  for (; tile < tEnd; tile += stride) {
    // keep the weight fragments in LDS (read per tile) instead of letting them be hoisted into
    // registers, which would cost the occupancy that hides the A loads' latency
    __asm__ volatile("" ::: "memory");
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < KA; st++) mma(acc, st, to_mfma(a[st]));
    load_a(tile + stride, a);
    if (MEAN) {
      // mean over the present neighbours, summed in slot order
      const int d[4] = {nb.x, nb.y, nb.z, nb.w};
      const int cnt = (d[0] >= 0) + (d[1] >= 0) + (d[2] >= 0) + (d[3] >= 0);
      const float ic = cnt ? 1.0f / cnt : 0.f;
#pragma unroll
      for (int st = 0; st < GS; st++) {
        float sm[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < GN; j++) {
          if (d[j] < 0) continue;
          const uint16_t *h = reinterpret_cast<const uint16_t *>(&g[j][st]);
#pragma unroll
          for (int q = 0; q < 8; q++) sm[q] += bf2f(h[q]);
        }
        uint16_t o[8];
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = f2bf(sm[q] * ic);
        const uint4 m = *reinterpret_cast<const uint4 *>(o);
        mma(acc, GS + st, to_mfma(m));
        if (P.meanOut && tile * 16 + mr < R)
          *reinterpret_cast<uint4 *>(P.meanOut + (size_t)(tile * 16 + mr) * P.lda + K / 2 + 32 * st + 8 * mp) = m;
      }
      load_g(nbn, g);
      nb = nbn;
      nbn = load_nb(tile + 2 * stride);
    }
    finish(tile * 16, acc);
  }
}

// Weight gradient partials of one slice of rows: w[k][n] = sum_r A[r][k] D[r][n] for KB of A's columns and
// all N of D's, and from the first column block b[n] = sum_r D[r][n].  The row index is the MFMA
// reduction dimension, so both operands are needed by column: 32 rows of each are staged in LDS, an octet
// of each per thread, and read back by transposing LDS reads, four rows to a read.  Rows are padded by 32
// bytes: the eight rows that 32 lanes read then lie on different banks.  A slice is 16 stages of little
// work, so what bounded it was the latency of each: four stages are in flight, the LDS is double-buffered
// (one barrier per stage), and eight waves share a slice rather than two slices of four, whose partials
// would be twice the traffic.  Measured at 65,536 rows, wide layers / narrow ones: loaded from memory 2
// bytes at a time 64 us each, and the bias sums 86; staged in LDS and read 2 bytes at a time, the next
// stage in flight, 29 / 17 with the bias sums; transposing reads and eight waves 19 / 17; four stages in
// flight 15 / 13 (two or eight: the same within 1 %).  With the loads under conditions, which force a wait
// at each, four in flight took 32 / 28.
constexpr int WG_T = 512, WG_AHEAD = 4;  // threads (eight waves); stages of 32 rows in flight, an even number
template <int KB, int N>
__global__ __launch_bounds__(WG_T) void wgrad_kernel(int R, int rows, const uint16_t *__restrict__ A, int lda,
                                                     const uint16_t *__restrict__ D, float *__restrict__ w,
                                                     float *__restrict__ b) {
  constexpr int WK = KB == 32 ? 1 : N == 32 ? 8 : 2, WN = 8 / WK;   // waves along k and n
  constexpr int TK = KB / 16 / WK, TN = N / 16 / WN;                // 16 x 16 tiles per wave
  constexpr int SA = KB + 16, SD = N + 16, OA = KB / 8, OD = N / 8;  // LDS rows; octets per row
  constexpr int BUF = 32 * (SA + SD);
  static_assert(32 * OA <= WG_T && 32 * OD <= WG_T && WG_T % OD == 0, "an octet of each operand per thread");
  static_assert(2 * BUF * 2 >= WG_T * 8 * 4, "the bias sums fit the buffers");
  __shared__ alignas(16) uint16_t sm[2][BUF];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lk = (lane >> 4) * 4;
  const int kc = blockIdx.y * KB, kb = (wave % WK) * TK * 16, nb = (wave / WK) * TN * 16;
  const int rb = blockIdx.x * rows, re = min(R, rb + rows);
  const int ra = tid / OA, ca = 8 * (tid % OA), rd = tid / OD, cd = 8 * (tid % OD);  // this thread's octets
  uint4 a[WG_AHEAD], d[WG_AHEAD];
  // unconditional (rows past the slice repeat its last one and are zeroed on the way to LDS), so that no
  // wait is forced before the next stages' loads issue
  auto load = [&](int r0, uint4 &x, uint4 &y) {
    x = *reinterpret_cast<const uint4 *>(&A[(size_t)min(r0 + ra, re - 1) * lda + kc + ca]);
    y = *reinterpret_cast<const uint4 *>(&D[(size_t)min(r0 + rd, re - 1) * N + cd]);
  };
  // column lr of rows lk .. lk + 3 and 16 + lk .. 16 + lk + 3 of a 16-column tile: a transposing read gives
  // lane l of 16 column l of the four rows that the lanes hold, four lanes of 8 bytes to a row
  auto column = [&](const uint16_t *t, int stride) {
    const uint16_t *q = t + (lk + lr / 4) * stride + 4 * (lr % 4);
    typedef __attribute__((address_space(3))) bf16x4 *lp;
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(q));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(q + 16 * stride));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  f32x4 acc[TK][TN];
#pragma unroll
  for (int i = 0; i < TK; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float cs[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // column sums of this thread's octets of D (one column octet)
  auto stage = [&](uint16_t *sA, uint4 &x, uint4 &y, int r0) {
    uint16_t *sD = sA + 32 * SA;
    const unsigned mx = r0 + ra < re ? ~0u : 0u, my = r0 + rd < re ? ~0u : 0u;
    x = make_uint4(x.x & mx, x.y & mx, x.z & mx, x.w & mx);
    y = make_uint4(y.x & my, y.y & my, y.z & my, y.w & my);
    if (ra < 32) *reinterpret_cast<uint4 *>(&sA[ra * SA + ca]) = x;
    if (rd < 32) {
      *reinterpret_cast<uint4 *>(&sD[rd * SD + cd]) = y;
      const uint16_t *h = reinterpret_cast<const uint16_t *>(&y);
#pragma unroll
      for (int e = 0; e < 8; e++) cs[e] += bf2f(h[e]);
    }
    load(r0 + 32 * WG_AHEAD, x, y);
    __syncthreads();  // one per stage: the other buffer is written next, which every wave has read by then
    bf16x8 fa[TK], fd[TN];
#pragma unroll
    for (int i = 0; i < TK; i++) fa[i] = column(sA + kb + 16 * i, SA);
#pragma unroll
    for (int j = 0; j < TN; j++) fd[j] = column(sD + nb + 16 * j, SD);
#pragma unroll
    for (int i = 0; i < TK; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fd[j], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int q = 0; q < WG_AHEAD; q++) load(rb + 32 * q, a[q], d[q]);
  for (int r0 = rb; r0 < re; r0 += 32 * WG_AHEAD)
#pragma unroll
    for (int q = 0; q < WG_AHEAD; q++)
      stage(sm[q & 1], a[q], d[q], r0 + 32 * q);
  w += (size_t)blockIdx.x * NPART;
#pragma unroll
  for (int i = 0; i < TK; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) w[(size_t)(kc + kb + 16 * i + lk + e) * N + nb + 16 * j + lr] = acc[i][j][e];
  if (blockIdx.y) return;
  // thread tid summed column octet tid % OD
  float *sB = reinterpret_cast<float *>(sm[0]);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; e++) sB[tid * 8 + e] = cs[e];
  __syncthreads();
  if (tid < N) {
    float s = 0.f;
    for (int t = tid / 8; t < WG_T; t += OD) s += sB[t * 8 + tid % 8];
    b[(size_t)blockIdx.x * NPART + tid] = s;
  }
}

// The gradient in the flat parameter order, summed over the slices (64 parameters to a workgroup, its four
// waves a quarter of the slices each), and by a workgroup of its own the loss from its nl partials, straight
// into host memory: its copy in the middle of the pass held the host back until the forward pass was done,
// and the card then waited for the backward launches (65,536 cells: 334 -> 323 us a gradient)
__global__ __launch_bounds__(256) void wgrad_reduce(const float *__restrict__ part, int ns, float *__restrict__ g,
                                                    const double *__restrict__ lpart, int nl, double *loss) {
  __shared__ float sm[4][64];
  __shared__ double sl[4];
  if (blockIdx.x == gridDim.x - 1) {
    double s = 0.0;
    for (int k = threadIdx.x; k < nl; k += 256) s += lpart[k];
    for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
    if (threadIdx.x % 64 == 0) sl[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0) *loss = (sl[0] + sl[1]) + (sl[2] + sl[3]);
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (i < NPAR) {
    int at;
    if (i < OFF_B0) at = PW0 + i;  // the first NI of NIP rows
    else if (i < OFF_W1) at = PB0 + i - OFF_B0;
    else if (i < OFF_B1) at = PW1 + i - OFF_W1;
    else if (i < OFF_W2) at = PB1 + i - OFF_B1;
    else if (i < OFF_B2) at = PW2 + i - OFF_W2;
    else if (i < OFF_W3) at = PB2 + i - OFF_B2;
    else if (i < OFF_B3) at = PW3 + (i - OFF_W3) / NO * NOP + (i - OFF_W3) % NO;
    else at = PB3 + i - OFF_B3;
#pragma unroll 8
    for (int sl = wave; sl < ns; sl += 4) s += part[(size_t)sl * NPART + at];
  }
  sm[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && i < NPAR) g[i] = (sm[0][lane] + sm[1][lane]) + (sm[2][lane] + sm[3][lane]);
}

// ---------------------------------------------------------------- graph and elementwise kernels

// Backward of [h, mean_nb h] -> h, then silu': dP[c][k] = (dX[c][k] + sum_nb dX[nb][128+k]/cnt_nb) silu'(pre),
// 8 columns per thread (by single columns, each thread counting its neighbours' neighbours for itself:
// 62 us at 65,536 cells, 21 us now)
__global__ __launch_bounds__(256) void mp_backward_kernel(int R, const int *__restrict__ nbr,
                                                          const uint16_t *__restrict__ dX,
                                                          const float *__restrict__ pre, uint16_t *__restrict__ dP) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)R * (NH / 8)) return;
  const int c = (int)(t / (NH / 8)), k = (int)(t % (NH / 8)) * 8;
  const int4 *nb4 = reinterpret_cast<const int4 *>(nbr);
  const int4 nb = nb4[c];
  const int d[NBR] = {nb.x, nb.y, nb.z, nb.w};
  uint4 own = *reinterpret_cast<const uint4 *>(&dX[(size_t)c * 256 + k]), v[NBR];
  float cnt[NBR];
#pragma unroll
  for (int j = 0; j < NBR; j++) {
    if (d[j] < 0) continue;
    const int4 q = nb4[d[j]];
    cnt[j] = (float)((q.x >= 0) + (q.y >= 0) + (q.z >= 0) + (q.w >= 0));
    v[j] = *reinterpret_cast<const uint4 *>(&dX[(size_t)d[j] * 256 + 128 + k]);
  }
  const float4 p0 = *reinterpret_cast<const float4 *>(&pre[(size_t)c * NH + k]);
  const float4 p1 = *reinterpret_cast<const float4 *>(&pre[(size_t)c * NH + k + 4]);
  const float p[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
  uint16_t o[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    float s = bf2f(reinterpret_cast<const uint16_t *>(&own)[e]);
#pragma unroll
    for (int j = 0; j < NBR; j++)
      if (d[j] >= 0) s += bf2f(reinterpret_cast<const uint16_t *>(&v[j])[e]) / cnt[j];
    o[e] = f2bf(s * dsilu_f(p[e]));
  }
  *reinterpret_cast<uint4 *>(&dP[(size_t)c * NH + k]) = *reinterpret_cast<const uint4 *>(o);
}

// t[c][a] = rhat_a + sum_b O[c][5a+b] rhat_b, rhat = r / S (r: SoA with stride nC, cells [c0, c0+R));
// the 128-byte output row is read as 16-byte vectors, and its five weights go beside t, so that
// apply_z_kernel, which needs them and its neighbours' t, does not read the rows again (1.5M cells: 51 + 77 us
// -> 61 + 52 us for the two kernels)
__global__ void apply_t_kernel(int R, int c0, int nC, const float *__restrict__ O, const float *__restrict__ S,
                               const double *__restrict__ r, float *__restrict__ t, float *__restrict__ rh) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  float q[5];
  for (int b = 0; b < 5; b++) q[b] = (float)(r[(size_t)b * nC + c0 + i] / S[b]);
  const float4 *o4 = reinterpret_cast<const float4 *>(O + (size_t)NOP * i);
  float o[28];
#pragma unroll
  for (int k = 0; k < 7; k++) {
    const float4 v = o4[k];
    o[4 * k] = v.x;
    o[4 * k + 1] = v.y;
    o[4 * k + 2] = v.z;
    o[4 * k + 3] = v.w;
  }
  float ta[5];
#pragma unroll
  for (int a = 0; a < 5; a++) {
    float sa = q[a];
#pragma unroll
    for (int b = 0; b < 5; b++) sa += o[5 * a + b] * q[b];
    ta[a] = sa;
  }
  const float4 w = o4[7];  // o[28..29]
  float4 *t4 = reinterpret_cast<float4 *>(t + (size_t)NTR * i);
  t4[0] = make_float4(ta[0], ta[1], ta[2], ta[3]);
  t4[1] = make_float4(ta[4], o[25], o[26], o[27]);
  t4[2] = make_float4(w.x, w.y, 0.f, 0.f);
  if (rh)
    for (int a = 0; a < 5; a++) rh[(size_t)8 * i + a] = q[a];
}

// z_a[c] = S_a ((1 + s4[c]) t[c][a] + sum_j s_j[c] t[nb_j(c)][a]), s = O[c][25:30]: weights of the
// 4 face neighbours (neib slot order) and of the cell itself
__global__ void apply_z_kernel(int R, int nC, const int *__restrict__ nbr, const float *__restrict__ S, const float *__restrict__ t, double *__restrict__ z,
                               unsigned *__restrict__ nf) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= R) return;
  const float4 *t4 = reinterpret_cast<const float4 *>(t);
  constexpr int T4 = NTR / 4;
  const float4 tc0 = t4[T4 * (size_t)c], tc1 = t4[T4 * (size_t)c + 1], tc2 = t4[T4 * (size_t)c + 2];
  const float sw[5] = {tc1.y, tc1.z, tc1.w, tc2.x, tc2.y}, tc4 = tc1.x;
  const int4 nb = reinterpret_cast<const int4 *>(nbr)[c];
  const int d[4] = {nb.x, nb.y, nb.z, nb.w};
  float acc[5] = {(1.f + sw[4]) * tc0.x, (1.f + sw[4]) * tc0.y, (1.f + sw[4]) * tc0.z, (1.f + sw[4]) * tc0.w,
                  (1.f + sw[4]) * tc4};
#pragma unroll
  for (int j = 0; j < NBR; j++) {
    if (d[j] < 0) continue;
    const float4 a = t4[T4 * (size_t)d[j]];
    const float a4 = t4[T4 * (size_t)d[j] + 1].x;
    acc[0] += sw[j] * a.x;
    acc[1] += sw[j] * a.y;
    acc[2] += sw[j] * a.z;
    acc[3] += sw[j] * a.w;
    acc[4] += sw[j] * a4;
  }
  bool bad = false;
  for (int a = 0; a < 5; a++) {
    const double o = (double)S[a] * (double)acc[a];
    z[(size_t)a * nC + c] = o;
    bad |= !isfinite(o);
  }
  if (bad && nf) flag_nonfinite(nf);
}

// loss pieces: e = 2 (zhat - dhat) / R; ds[c][j] = e_c . t_nb(j) (j < 4), ds[c][4] = e_c . t_c (the
// weight gradients); part[block] = sum (zhat - dhat)^2
__global__ void loss_e_kernel(int R, int c0, int nC, const int *__restrict__ nbr, const float *__restrict__ O,
                              const float *__restrict__ S, const float *__restrict__ t, const double *__restrict__ delta,
                              float *__restrict__ e, float *__restrict__ ds, double *__restrict__ part) {
  __shared__ double sm[256];
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (c < R) {
    const float *o = O + (size_t)NOP * c;
    float zh[5];
    for (int a = 0; a < 5; a++) zh[a] = (1.f + o[29]) * t[(size_t)NTR * c + a];
    int nb[NBR];
    for (int j = 0; j < NBR; j++) {
      nb[j] = nbr[(size_t)NBR * c + j];
      if (nb[j] < 0) continue;
      for (int a = 0; a < 5; a++) zh[a] += o[25 + j] * t[(size_t)NTR * nb[j] + a];
    }
    float ea[5];
    for (int a = 0; a < 5; a++) {
      const float dd = zh[a] - (float)(delta[(size_t)a * nC + c0 + c] / S[a]);
      l += (double)dd * dd;
      ea[a] = 2.0f * dd / (float)R;
      e[(size_t)8 * c + a] = ea[a];
    }
    for (int j = 0; j < NBR; j++) {
      float g = 0.f;
      if (nb[j] >= 0)
        for (int a = 0; a < 5; a++) g += ea[a] * t[(size_t)NTR * nb[j] + a];
      ds[(size_t)8 * c + j] = g;
    }
    float g4 = 0.f;
    for (int a = 0; a < 5; a++) g4 += ea[a] * t[(size_t)NTR * c + a];
    ds[(size_t)8 * c + 4] = g4;
  }
  sm[threadIdx.x] = l;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) sm[threadIdx.x] += sm[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

// dt_c = (1 + s4_c) e_c + sum over neighbours d of c of s_j(d) e_d, j the slot of c in d's list;
// dO[5a+b] = dt_a rhat_b, dO[25+j] = ds[c][j], both times k_c (the output scale) for the last
// layer's gradient; bf16 dO [R][32]
__global__ void loss_dO_kernel(int R, const int *__restrict__ nbr, const float *__restrict__ O,
                               const float *__restrict__ e, const float *__restrict__ rh, const float *__restrict__ ds,
                               const float *__restrict__ kappa, uint16_t *__restrict__ dO) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= R) return;
  float dt[5];
  const float sc = 1.f + O[(size_t)NOP * c + 29];
  for (int a = 0; a < 5; a++) dt[a] = sc * e[(size_t)8 * c + a];
  for (int j = 0; j < NBR; j++) {
    const int d = nbr[(size_t)NBR * c + j];
    if (d < 0) continue;
    for (int q = 0; q < NBR; q++) {
      if (nbr[(size_t)NBR * d + q] != c) continue;
      const float w = O[(size_t)NOP * d + 25 + q];
      for (int a = 0; a < 5; a++) dt[a] += w * e[(size_t)8 * d + a];
    }
  }
  uint16_t *o = dO + (size_t)NOP * c;
  const float k = kappa[c];
  for (int a = 0; a < 5; a++)
    for (int b = 0; b < 5; b++) o[5 * a + b] = f2bf(k * dt[a] * rh[(size_t)8 * c + b]);
  for (int j = 0; j < 5; j++) o[25 + j] = f2bf(k * ds[(size_t)8 * c + j]);
  o[30] = o[31] = 0;
}

// batch-local neighbour table for cells [c0, c0+R)
__global__ void batch_nbr_kernel(int R, int c0, const int *__restrict__ nbr, int *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  for (int j = 0; j < NBR; j++) {
    const int d = nbr[(size_t)NBR * (c0 + i) + j];
    out[(size_t)NBR * i + j] = (d >= c0 && d < c0 + R) ? d - c0 : -1;
  }
}

__global__ void adam_kernel(int n, float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 operand copies from the FP32 master parameters
__global__ void pack_kernel(const float *__restrict__ p, uint16_t *W0t, uint16_t *W1t, uint16_t *W2t, uint16_t *W3t,
                            uint16_t *W1b, uint16_t *W2b, uint16_t *W3b, float *bias) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < NH * NIP) {  // W0t [128][32]
    const int n = i / NIP, k = i % NIP;
    W0t[i] = k < NI ? f2bf(p[OFF_W0 + k * NH + n]) : 0;
  }
  if (i < NH * 256) {  // W1t, W2t [128][256]; W1b, W2b [256][128]
    const int n = i / 256, k = i % 256;
    W1t[i] = f2bf(p[OFF_W1 + k * NH + n]);
    W2t[i] = f2bf(p[OFF_W2 + k * NH + n]);
    const int kk = i / NH, nn = i % NH;
    W1b[i] = f2bf(p[OFF_W1 + kk * NH + nn]);
    W2b[i] = f2bf(p[OFF_W2 + kk * NH + nn]);
  }
  if (i < NOP * NH) {  // W3t [32][128]; W3b [128][32]
    const int n = i / NH, k = i % NH;
    W3t[i] = n < NO ? f2bf(p[OFF_W3 + k * NO + n]) : 0;
    const int kk = i / NOP, nn = i % NOP;
    W3b[i] = nn < NO ? f2bf(p[OFF_W3 + kk * NO + nn]) : 0;
  }
  if (i < 3 * NH + NOP) {
    if (i < NH) bias[i] = p[OFF_B0 + i];
    else if (i < 2 * NH) bias[i] = p[OFF_B1 + i - NH];
    else if (i < 3 * NH) bias[i] = p[OFF_B2 + i - 2 * NH];
    else bias[i] = (i - 3 * NH) < NO ? p[OFF_B3 + i - 3 * NH] : 0.f;
  }
}

// per-variable state scale S = rms(rho), rms(|rhou|)/sqrt(3) (x3), rms(rhoE), floored at 1e-6 rms(rhoE)
// (1024 threads to a workgroup, since the last pass takes 256 partials: 1.5M cells 19.8 us with 256 threads, now 17.4)
constexpr int SC_T = 1024;
__global__ __launch_bounds__(SC_T) void scale_partial(int nC, const double *__restrict__ y, double *__restrict__ part) {
  __shared__ double sm[SC_T / 64][3];
  double a = 0, b = 0, c = 0;
#pragma unroll 4
  for (int i = blockIdx.x * SC_T + threadIdx.x; i < nC; i += gridDim.x * SC_T) {
    double v[5];
#pragma unroll
    for (int k = 0; k < 5; k++) v[k] = y[(size_t)k * nC + i];
    a += v[0] * v[0];
    b += v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    c += v[4] * v[4];
  }
  for (int m = 32; m > 0; m >>= 1) {
    a += __shfl_xor(a, m, 64);
    b += __shfl_xor(b, m, 64);
    c += __shfl_xor(c, m, 64);
  }
  if (threadIdx.x % 64 == 0) {
    sm[threadIdx.x / 64][0] = a;
    sm[threadIdx.x / 64][1] = b;
    sm[threadIdx.x / 64][2] = c;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double s = 0;
    for (int w = 0; w < SC_T / 64; w++) s += sm[w][threadIdx.x];
    part[blockIdx.x * 3 + threadIdx.x] = s;
  }
}

// one wave: lane l adds the partials l, l + 64, ...
__global__ __launch_bounds__(64) void scale_final(int nb, int nC, const double *__restrict__ part,
                                                  float *__restrict__ S) {
  double a = 0, b = 0, c = 0;
  for (int i = threadIdx.x; i < nb; i += 64) { a += part[3 * i]; b += part[3 * i + 1]; c += part[3 * i + 2]; }
  for (int m = 32; m > 0; m >>= 1) {
    a += __shfl_xor(a, m, 64);
    b += __shfl_xor(b, m, 64);
    c += __shfl_xor(c, m, 64);
  }
  if (threadIdx.x) return;
  const double ra = sqrt(a / nC), rb = sqrt(b / (3.0 * nC)), rc = sqrt(c / nC);
  const double fl = 1e-6 * rc + 1e-300;
  S[0] = (float)fmax(ra, fl);
  S[1] = S[2] = S[3] = (float)fmax(rb, fmax(1e-3 * ra, fl));
  S[4] = (float)fmax(rc, fl);
}

template <int K, int N, bool FEAT, bool MEAN, bool TAIL, int EPI>
void layer(hipStream_t s, const LayerArgs &P) {
  const size_t lds = sizeof(uint16_t) * ((size_t)N * K + (TAIL ? NOP * NH : FEAT ? TPB * NIP : 0));
  const int rows = FEAT ? 64 : 16, tiles = (P.R + rows - 1) / rows, wpb = TPB / 64;
  const int per = std::max(1, (int)(160 * 1024 / lds));  // workgroups per CU that the LDS allows
  const int grid = 8 * std::max(1, std::min((tiles + 8 * wpb - 1) / (8 * wpb), 32 * std::min(per, 1024 / TPB)));
  hipLaunchKernelGGL((mlp_layer_kernel<K, N, FEAT, MEAN, TAIL, EPI>), dim3(grid), dim3(TPB), lds, s, P);
}

int compute_scale(fos_euler *ctx, Learned *L, const double *y) {
  const int nb = std::max(1, std::min(256, (ctx->nC + SC_T - 1) / SC_T));
  hipLaunchKernelGGL(scale_partial, dim3(nb), dim3(SC_T), 0, ctx->stream, ctx->nC, y, L->red.p);
  hipLaunchKernelGGL(scale_final, dim3(1), dim3(64), 0, ctx->stream, nb, ctx->nC, L->red.p, L->scale.p);
  FOS_HIP_TRY(hipGetLastError());
  return 0;
}

// network forward on R cells starting at c0 (nbr: neighbour table with indices local to the range)
int forward(fos_euler *ctx, Learned *L, const double *y, int c0, int R, const int *nbr, double gamma, bool keepPre) {
  hipStream_t s = ctx->stream;
  const float *bias = L->bias.p;
  // training also stores the features, the means, the last hidden layer and the layers' inputs to silu
  // (the weight gradients read [h, mean h] as one row); inference keeps the hidden rows at 256 bytes
  const int ld = keepPre ? 256 : NH;
  uint16_t *h0 = keepPre ? L->HM0.p : L->H0.p, *h1 = keepPre ? L->HM1.p : L->H1.p;
  LayerArgs P{};
  P.R = R;
  P.lda = P.ldo = ld;
  P.nbr = nbr;
  P.kappa = L->kappa.p;
  P.y = y;
  P.geo = L->geo.p;
  P.S = L->scale.p;
  P.gamma = gamma;
  P.gm = ctx->gamm;
  P.c0 = c0;
  P.nC = ctx->nC;
  P.X = keepPre ? L->X.p : nullptr;
  P.Bn = L->W0t.p;
  P.bias = bias;
  P.pre = keepPre ? L->pre0.p : nullptr;
  P.outb = h0;
  layer<NIP, NH, true, false, false, EPI_SILU>(s, P);
  P.A = h0;
  P.Bn = L->W1t.p;
  P.bias = bias + NH;
  P.pre = keepPre ? L->pre1.p : nullptr;
  P.outb = h1;
  P.meanOut = keepPre ? h0 : nullptr;
  layer<256, NH, false, true, false, EPI_SILU>(s, P);
  P.A = h1;
  P.Bn = L->W2t.p;
  P.bias = bias + 2 * NH;
  P.pre = keepPre ? L->pre2.p : nullptr;
  P.outb = keepPre ? L->H2.p : nullptr;
  P.ldo = NH;
  P.meanOut = keepPre ? h1 : nullptr;
  P.B3 = L->W3t.p;
  P.bias3 = bias + 3 * NH;
  P.O = L->O.p;
  layer<256, NH, false, true, true, EPI_SILU>(s, P);
  FOS_HIP_TRY(hipGetLastError());
  return 0;
}

int repack(fos_euler *ctx, Learned *L) {
  hipLaunchKernelGGL(pack_kernel, dim3((NH * 256 + 255) / 256), dim3(256), 0, ctx->stream, L->par.p, L->W0t.p,
                     L->W1t.p, L->W2t.p, L->W3t.p, L->W1b.p, L->W2b.p, L->W3b.p, L->bias.p);
  FOS_HIP_TRY(hipGetLastError());
  return 0;
}

int create_learned(fos_euler *ctx) {
  if (ctx->learned) return 0;
  if (ctx->maxNF > NBR) {
    set_error("learned preconditioner: cells with %d faces (tetrahedra only)", ctx->maxNF);
    return -1;
  }
  Learned *L = new Learned();  // attached to the context only once complete
  const int nC = ctx->nC, mf = ctx->maxNF;
  L->nC = nC;
  std::vector<int> nbr((size_t)NBR * std::max(nC, 1), -1);
  for (int c = 0; c < nC; c++)
    for (int j = 0; j < mf; j++) {
      const int e = ctx->hNeib[(size_t)mf * c + j];
      nbr[(size_t)NBR * c + j] = (e >= 0 && e < nC) ? e : -1;
    }
  // static geometry features: log(v/vmean) and the 4 outward area vectors / v^(2/3) in neib order
  double vm = 0;
  for (int c = 0; c < nC; c++) vm += ctx->hV[c];
  vm /= std::max(nC, 1);
  std::vector<float> geo((size_t)13 * nC + 1, 0.f);
  for (int c = 0; c < nC; c++) geo[(size_t)13 * c] = (float)std::log(ctx->hV[c] / vm);
  for (int i = 0; i < ctx->nP; i++) {
    const int m = ctx->hIEP[2 * i], n = ctx->hIEP[2 * i + 1];
    const double a = ctx->hAP[i];
    for (int side = 0; side < 2; side++) {
      const int c = side ? n : m, o = side ? m : n;
      if (c >= nC) continue;
      for (int j = 0; j < mf; j++)
        if (ctx->hNeib[(size_t)mf * c + j] == o) {
          const double sc = (side ? -a : a) / std::pow(ctx->hV[c], 2.0 / 3.0);
          for (int d = 0; d < 3; d++) geo[(size_t)13 * c + 1 + 3 * j + d] = (float)(sc * ctx->hNormP[3 * (size_t)i + d]);
          break;
        }
    }
  }
  geo[(size_t)13 * nC] = (float)std::cbrt(vm);
  hipStream_t s = ctx->stream;
  if (L->nbr.upload(nbr.data(), nbr.size(), s) || L->geo.upload(geo.data(), geo.size(), s) || L->par.alloc(NPAR) ||
      L->m1.alloc(NPAR) || L->m2.alloc(NPAR) || L->grad.alloc(NPAR) || L->bias.alloc(3 * NH + NOP) ||
      L->W0t.alloc(NH * NIP) || L->W1t.alloc(NH * 256) || L->W2t.alloc(NH * 256) || L->W3t.alloc(NOP * NH) ||
      L->W1b.alloc(256 * NH) || L->W2b.alloc(256 * NH) || L->W3b.alloc(NH * NOP) || L->scale.alloc(8) ||
      hipHostMalloc((void **)&L->pinned, sizeof(double)) != hipSuccess ||
      hipHostGetDevicePointer((void **)&L->dpinned, L->pinned, 0) != hipSuccess) {
    if (!L->pinned) set_error("learned preconditioner: pinned host buffer allocation failed");
    delete L;
    return -1;
  }
  ctx->learned = L;
  return 0;
}

int set_params(fos_euler *ctx, const float *host) {
  Learned *L = ctx->learned;
  FOS_HIP_TRY(hipMemcpyAsync(L->par.p, host, sizeof(float) * NPAR, hipMemcpyHostToDevice, ctx->stream));
  FOS_HIP_TRY(hipMemsetAsync(L->m1.p, 0, sizeof(float) * NPAR, ctx->stream));
  FOS_HIP_TRY(hipMemsetAsync(L->m2.p, 0, sizeof(float) * NPAR, ctx->stream));
  L->step = 0;
  if (repack(ctx, L)) return -1;
  FOS_HIP_TRY(hipStreamSynchronize(ctx->stream));
  L->ready = true;
  return 0;
}

// forward + loss + backward for cells [c0, c0+R) of a snapshot; the gradient is left in L->grad
int loss_grad(fos_euler *ctx, const double *y, const double *r, const double *delta, double gamma, int c0, int R,
              double *loss) {
  Learned *L = ctx->learned;
  hipStream_t s = ctx->stream;
  L->haveO = false;
  if (L->train(R)) return -1;
  if (slice_count(R) * NPART > L->part.n) {  // slice_room's bound, checked before anything writes them
    set_error("learned: %zu slices of a %d-row batch exceed the workspace", slice_count(R), R);
    return -1;
  }
  if (compute_scale(ctx, L, y)) return -1;
  hipLaunchKernelGGL(batch_nbr_kernel, dim3((R + 255) / 256), dim3(256), 0, s, R, c0, L->nbr.p, L->bnbr.p);
  const int *nb = L->bnbr.p;
  if (forward(ctx, L, y, c0, R, nb, gamma, true)) return -1;
  const int gb = (R + 255) / 256;
  hipLaunchKernelGGL(apply_t_kernel, dim3(gb), dim3(256), 0, s, R, c0, ctx->nC, L->O.p, L->scale.p, r, L->t.p,
                     L->rh.p);
  hipLaunchKernelGGL(loss_e_kernel, dim3(gb), dim3(256), 0, s, R, c0, ctx->nC, nb, L->O.p, L->scale.p, L->t.p, delta,
                     L->e.p, L->ds.p, L->red.p);
  hipLaunchKernelGGL(loss_dO_kernel, dim3(gb), dim3(256), 0, s, R, nb, L->O.p, L->e.p, L->rh.p, L->ds.p, L->kappa.p,
                     L->dO16.p);
  const int rows = (int)slice_rows(R), ns = (int)slice_count(R);
  const dim3 gr((unsigned)(((size_t)R * (NH / 8) + 255) / 256)), blk(256);
  float *pt = L->part.p;
  // layer 3: dW3 = H2^T dO, db3 = sum dO; dP = (dO W3^T) silu'(pre2)
  hipLaunchKernelGGL((wgrad_kernel<NH, NOP>), dim3(ns, 1), dim3(WG_T), 0, s, R, rows, L->H2.p, NH, L->dO16.p, pt + PW3, pt + PB3);
  LayerArgs P{};
  P.R = R;
  P.A = L->dO16.p;
  P.lda = NOP;
  P.Bn = L->W3b.p;
  P.pre = L->pre2.p;
  P.outb = L->dP.p;
  P.ldo = NH;
  layer<NOP, NH, false, false, false, EPI_DSILU>(s, P);
  // layers 2 and 1: dW = [h, m]^T dP, db = sum dP; dX = dP W^T; dP <- mp-backward(dX) silu'(pre)
  const uint16_t *Hin[2] = {L->HM1.p, L->HM0.p};
  const uint16_t *Wb[2] = {L->W2b.p, L->W1b.p};
  float *preIn[2] = {L->pre1.p, L->pre0.p};
  const int offW[2] = {PW2, PW1}, offB[2] = {PB2, PB1};
  for (int l = 0; l < 2; l++) {
    hipLaunchKernelGGL((wgrad_kernel<NH, NH>), dim3(ns, 2), dim3(WG_T), 0, s, R, rows, Hin[l], 256, L->dP.p, pt + offW[l],
                       pt + offB[l]);
    P.A = L->dP.p;
    P.lda = NH;
    P.Bn = Wb[l];
    P.pre = nullptr;
    P.outb = L->dX.p;
    P.ldo = 256;
    layer<NH, 256, false, false, false, EPI_BF16>(s, P);
    hipLaunchKernelGGL(mp_backward_kernel, gr, blk, 0, s, R, nb, L->dX.p, preIn[l], L->dP.p);
  }
  // layer 0: dW0 = X^T dP, db0
  hipLaunchKernelGGL((wgrad_kernel<NIP, NH>), dim3(ns, 1), dim3(WG_T), 0, s, R, rows, L->X.p, NIP, L->dP.p, pt + PW0, pt + PB0);
  hipLaunchKernelGGL(wgrad_reduce, dim3((NPAR + 63) / 64 + 1), blk, 0, s, pt, ns, L->grad.p, L->red.p, gb, L->dpinned);
  FOS_HIP_TRY(hipGetLastError());
  FOS_HIP_TRY(hipStreamSynchronize(s));
  if (loss) *loss = *L->pinned / R;
  return 0;
}

}  // namespace

int learned_psetup(fos_euler *ctx, const double *y, double gamma) {
  Learned *L = ctx->learned;
  if (!L || !L->ready) {
    set_error("learned preconditioner: no parameters (fos_learned_init or fos_learned_set_params)");
    return -1;
  }
  L->haveO = false;  // training overwrites O with batch rows; the mesh output is recomputed here
  if (L->apply(ctx->nC) || compute_scale(ctx, L, y)) return -1;
  if (forward(ctx, L, y, 0, ctx->nC, L->nbr.p, gamma, false)) return -1;
  L->haveO = true;
  return 0;
}

int learned_psolve(fos_euler *ctx, const double *r, double *z) {
  Learned *L = ctx->learned;
  if (!L->haveO) {
    set_error("psolve_learned: called before psetup_learned");
    return -1;
  }
  const int nC = ctx->nC, gb = (nC + 255) / 256;
  hipLaunchKernelGGL(apply_t_kernel, dim3(gb), dim3(256), 0, ctx->stream, nC, 0, nC, L->O.p, L->scale.p, r, L->t.p,
                     nullptr);
  hipLaunchKernelGGL(apply_z_kernel, dim3(gb), dim3(256), 0, ctx->stream, nC, nC, L->nbr.p, L->scale.p, L->t.p,
                     z, ctx->dNonFinite + fos_euler::NF_SOLVE);
  FOS_HIP_TRY(hipGetLastError());
  return 0;
}

}  // namespace fos

using namespace fos;

extern "C" {

int fos_learned_nparams(void) { return NPAR; }

int fos_learned_init(fos_euler *ctx, uint64_t seed) {
  if (!ctx || create_learned(ctx)) return -1;
  // Glorot-uniform hidden layers, zero output layer: the untrained network is the identity
  std::mt19937_64 rng(seed);
  std::vector<float> p(NPAR, 0.f);
  auto fill = [&](int off, int fin, int fout) {
    const double a = std::sqrt(6.0 / (fin + fout));
    std::uniform_real_distribution<double> u(-a, a);
    for (int i = 0; i < fin * fout; i++) p[off + i] = (float)u(rng);
  };
  fill(OFF_W0, NI, NH);
  fill(OFF_W1, 2 * NH, NH);
  fill(OFF_W2, 2 * NH, NH);
  return set_params(ctx, p.data());
}

int fos_learned_set_params(fos_euler *ctx, const float *params) {
  if (!ctx || !params || create_learned(ctx)) return -1;
  return set_params(ctx, params);
}

int fos_learned_get_params(fos_euler *ctx, float *params) {
  if (!ctx || !params || !ctx->learned) return -1;
  FOS_HIP_TRY(hipMemcpyAsync(params, ctx->learned->par.p, sizeof(float) * NPAR, hipMemcpyDeviceToHost, ctx->stream));
  FOS_HIP_TRY(hipStreamSynchronize(ctx->stream));
  return 0;
}

int fos_learned_loss_grad(fos_euler *ctx, const double *y, const double *r, const double *delta, double gamma,
                          int batchStart, int batchSize, double *loss, float *grad) {
  if (!ctx || !ctx->learned || !ctx->learned->ready) { set_error("learned: not initialised"); return -1; }
  if (batchStart < 0 || batchSize <= 0 || batchStart + batchSize > ctx->nC) { set_error("learned: bad batch"); return -1; }
  if (loss_grad(ctx, y, r, delta, gamma, batchStart, batchSize, loss)) return -1;
  if (grad) {
    FOS_HIP_TRY(hipMemcpyAsync(grad, ctx->learned->grad.p, sizeof(float) * NPAR, hipMemcpyDeviceToHost, ctx->stream));
    FOS_HIP_TRY(hipStreamSynchronize(ctx->stream));
  }
  return 0;
}

int fos_learned_train_step(fos_euler *ctx, const double *y, const double *r, const double *delta, double gamma,
                           int batchStart, int batchSize, double lr, double *loss) {
  if (fos_learned_loss_grad(ctx, y, r, delta, gamma, batchStart, batchSize, loss, nullptr)) return -1;
  Learned *L = ctx->learned;
  L->step++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)L->step), c2 = 1.f - std::pow(b2, (float)L->step);
  hipLaunchKernelGGL(adam_kernel, dim3((NPAR + 255) / 256), dim3(256), 0, ctx->stream, NPAR, L->par.p, L->grad.p,
                     L->m1.p, L->m2.p, (float)lr, b1, b2, 1e-8f, c1, c2);
  return repack(ctx, L);
}

int fos_learned_inputs(fos_euler *ctx, const double *y, double gamma, float *X, float *S) {
  if (!ctx || create_learned(ctx)) return -1;
  Learned *L = ctx->learned;
  const int nC = ctx->nC;
  L->haveO = false;
  if (L->inputs(nC) || compute_scale(ctx, L, y)) return -1;
  hipLaunchKernelGGL(features_kernel, dim3((nC + 255) / 256), dim3(256), 0, ctx->stream, nC, 0, nC, y, L->geo.p,
                     L->scale.p, gamma, ctx->gamm, L->X.p);
  FOS_HIP_TRY(hipGetLastError());
  std::vector<uint16_t> xb((size_t)nC * NIP);
  float sc[8];
  FOS_HIP_TRY(hipMemcpyAsync(xb.data(), L->X.p, sizeof(uint16_t) * xb.size(), hipMemcpyDeviceToHost, ctx->stream));
  FOS_HIP_TRY(hipMemcpyAsync(sc, L->scale.p, sizeof(float) * 8, hipMemcpyDeviceToHost, ctx->stream));
  FOS_HIP_TRY(hipStreamSynchronize(ctx->stream));
  if (X)
    for (int c = 0; c < nC; c++)
      for (int k = 0; k < NI; k++) {
        uint32_t u = (uint32_t)xb[(size_t)c * NIP + k] << 16;
        std::memcpy(&X[(size_t)c * NI + k], &u, 4);
      }
  if (S)
    for (int k = 0; k < 5; k++) S[k] = sc[k];
  return 0;
}

int fos_euler_psetup_learned(double t, const double *y, const double *fy, int jok, int *jcur, double gamma,
                             void *user_data) {
  (void)t; (void)fy; (void)jok;
  fos_euler *ctx = static_cast<fos_euler *>(user_data);
  if (!ctx || !jcur) return -1;
  ctx->counters[2]++;
  *jcur = 1;
  return learned_psetup(ctx, y, gamma);
}

int fos_euler_psolve_learned(double t, const double *y, const double *fy, const double *r, double *z, double gamma,
                             double delta, int lr, void *user_data) {
  (void)t; (void)y; (void)fy; (void)gamma; (void)delta; (void)lr;
  fos_euler *ctx = static_cast<fos_euler *>(user_data);
  if (!ctx || !ctx->learned || !ctx->learned->ready) { set_error("psolve_learned: not set up"); return -1; }
  ctx->counters[3]++;
  if (learned_psolve(ctx, r, z)) return -1;
  return finish_call(ctx, "psolve_learned", fos_euler::NF_SOLVE);
}

}  // extern "C"
