// The learned warm start of the no-slip wall solve: a per-wall-node MLP
// (9 -> 64 -> 64 -> 64 -> 3, GELU) with BF16 weights and activations and FP32
// accumulation on the BF16 matrix cores, its training kernels (forward, backward,
// gradient reduction, Adam) and its inference kernel.
//
// Inputs per wall vertex: the cells' velocity there (3), the previous traction (3)
// and the vertex normal (3), standardised with a mean and 1/std per feature.  The
// network's output, scaled per component, is the traction increment over the
// previous traction; the predicted traction is f0 + scale * y.
//
// MFMA formulation.  A layer computes Z^T = W H^T + b with v_mfma_f32_16x16x16bf16_1k:
// A = W (rows: output features, k: input features), B = H^T (k: input features,
// columns: 16 nodes).  Lane l supplies A[l % 16][4 (l / 16) + j] and B[4 (l / 16) + j]
// [l % 16] and holds D[4 (l / 16) + i][l % 16]: for node l % 16 it holds the features
// 16 mt + 4 (l / 16) + i of output tile mt, which is exactly the B operand of K-step mt
// of the next layer, so activations never leave the registers.  The backward pass
// uses the same layout with W^T; the weight gradients dW = dZ^T H (k: nodes) take
// both operands through an LDS transpose and accumulate in registers; a workgroup's
// wavefronts and then the workgroups are summed in a fixed order.
#include <cmath>
#include <vector>

#include "internal.h"

typedef short mlp_s4 __attribute__((ext_vector_type(4)));
typedef float mlp_f4 __attribute__((ext_vector_type(4)));

#define MLP_NIN 9
#define MLP_H 64
#define MLP_NOUT 3
// FP32 parameter vector: W1[64][9] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[3][64] b4[3]
enum {
  MP_W1 = 0,
  MP_B1 = MP_W1 + MLP_H * MLP_NIN,
  MP_W2 = MP_B1 + MLP_H,
  MP_B2 = MP_W2 + MLP_H * MLP_H,
  MP_W3 = MP_B2 + MLP_H,
  MP_B3 = MP_W3 + MLP_H * MLP_H,
  MP_W4 = MP_B3 + MLP_H,
  MP_B4 = MP_W4 + MLP_NOUT * MLP_H,
  MP_N = MP_B4 + MLP_NOUT
};
// BF16 weights padded to MFMA tiles: W1p[64][16], W2[64][64], W3[64][64], W4p[16][64]
enum { WB_1 = 0, WB_2 = WB_1 + 64 * 16, WB_3 = WB_2 + 64 * 64, WB_4 = WB_3 + 64 * 64, WB_N = WB_4 + 16 * 64 };
// gradient accumulators in 16 x 16 tiles: layer 1 (4 x 1 tiles), 2 (4 x 4), 3 (4 x 4),
// 4 (1 x 4), then the biases b1 b2 b3 (64 each) and b4 (16, 3 used)
enum { GA_1 = 0, GA_2 = GA_1 + 4 * 256, GA_3 = GA_2 + 16 * 256, GA_4 = GA_3 + 16 * 256,
       GA_B = GA_4 + 4 * 256, GA_N = GA_B + 3 * 64 + 16 };
#define MLP_TS 72  // LDS row stride (bf16) of the transpose tiles and 64-wide weights: 64 + 8
#define MLP_TS1 24 // of the 16-wide ones: 16 + 8
// LDS copies of the weights with padded rows (16 rows of 128 bytes would share banks),
// and of W2^T, W3^T, W4^T for the backward pass
enum { SW_1 = 0, SW_2 = SW_1 + 64 * MLP_TS1, SW_3 = SW_2 + 64 * MLP_TS, SW_4 = SW_3 + 64 * MLP_TS,
       SW_N = SW_4 + 16 * MLP_TS,
       ST_2 = SW_N, ST_3 = ST_2 + 64 * MLP_TS, ST_4 = ST_3 + 64 * MLP_TS, ST_N = ST_4 + 64 * MLP_TS1 };
#define MLP_TW 4   // wavefronts per training workgroup
#define MLP_WG (64 * MLP_TW)  // threads of the forward's and the training's workgroups
// LDS copies of the biases b1 b2 b3 (64 each), b4 (3) and the norm
enum { SB_4 = 3 * 64, SB_NORM = SB_4 + 4, SB_N = SB_NORM + 2 * MLP_NIN + MLP_NOUT };

struct rbc3d_mlp {
  hipStream_t stream = nullptr;  // own stream, or `ext` once rbc3d_mlp_set_stream was
  hipStream_t ext = nullptr;     // called (which may name the null stream)
  bool use_ext = false;
  hipStream_t st() const { return use_ext ? ext : stream; }
  DBuf<float> p, m1, m2, grad, part, norm;
  DBuf<unsigned short> wb;
  DBuf<double> lpart;
  hipEvent_t ev = nullptr;  // marks the last work queued on st() (rbc_mlp_wait)
  int t = 0;
};

__device__ __forceinline__ unsigned short f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// GELU, tanh form (Hendrycks and Gimpel, 2016), and its derivative d.  With
// u = sqrt(2/pi) (x + 0.044715 x^3) and (1 + tanh u) / 2 = s = 1 / (1 + exp(-2u)):
// gelu = x s, d = s + x s (1 - s) 2 u'.  Seven instructions with the hardware's exponential
// and reciprocal (one unit in the last place each); through tanh with its division it was
// about thirty, which bound both kernels, and lost digits of 1 + tanh below zero.
#define GELU_2C 1.5957691216057308f  // 2 sqrt(2/pi)
#define GELU_A 0.044715f
#define GELU_LOG2E 1.4426950408889634f
__device__ __forceinline__ float gelu(float x, float &d) {
  const float x2 = x * x;
  const float e = x * fmaf(-GELU_2C * GELU_LOG2E * GELU_A, x2, -GELU_2C * GELU_LOG2E);
  const float s = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(e)), g = x * s;
  d = fmaf(g * (1.f - s), fmaf(3.f * GELU_2C * GELU_A, x2, GELU_2C), s);
  return g;
}

__device__ __forceinline__ mlp_f4 mfma(mlp_s4 a, mlp_s4 b, mlp_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// A operand from a row-major BF16 matrix W[rows][ld] (8-byte aligned rows): lane supplies
// W[r0 + l%16][k0 + 4q + j]
__device__ __forceinline__ mlp_s4 ldA(const unsigned short *W, int ld, int r0, int k0, int lane) {
  return *reinterpret_cast<const mlp_s4 *>(W + (r0 + (lane & 15)) * ld + k0 + 4 * (lane >> 4));
}
__device__ __forceinline__ mlp_s4 tobf(mlp_f4 v) {
  mlp_s4 r;
  r[0] = (short)f2bf(v[0]);
  r[1] = (short)f2bf(v[1]);
  r[2] = (short)f2bf(v[2]);
  r[3] = (short)f2bf(v[3]);
  return r;
}

// Forward pass of one tile of 16 nodes (node = node0 + lane % 16); keeps the
// activations' derivatives and the BF16 activations h (B-operand layout) for the backward.
struct MlpTile {
  mlp_s4 x;         // inputs (features 4q + j)
  mlp_f4 d[3][4];   // GELU' at the hidden layers' pre-activations, tile mt
  mlp_s4 h[3][4];   // BF16 activations of the hidden layers, K-step mt
  mlp_f4 y;         // outputs 4q + i (valid: q == 0, i < 3)
};

__device__ __forceinline__ void mlp_forward(const unsigned short *sW, const float *sb,
                                            const float *X, int n, int node0, int lane,
                                            MlpTile &T) {
  const float *norm = sb + SB_NORM;
  const int q = lane >> 4, node = node0 + (lane & 15);
  #pragma unroll
  for (int j = 0; j < 4; j++) {
    const int f = 4 * q + j;
    float v = 0.f;
    if (f < MLP_NIN && node < n) v = (X[(size_t)node * MLP_NIN + f] - norm[f]) * norm[MLP_NIN + f];
    T.x[j] = (short)f2bf(v);
  }
  // layer 1: W1p[64][16]
  #pragma unroll
  for (int mt = 0; mt < 4; mt++) {
    mlp_f4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = mfma(ldA(sW + SW_1, MLP_TS1, 16 * mt, 0, lane), T.x, acc);
    #pragma unroll
    for (int i = 0; i < 4; i++) acc[i] += sb[16 * mt + 4 * q + i];
    mlp_f4 g;
    #pragma unroll
    for (int i = 0; i < 4; i++) {
      float d;
      g[i] = gelu(acc[i], d);
      T.d[0][mt][i] = d;
    }
    T.h[0][mt] = tobf(g);
  }
  // layers 2 and 3: 64 x 64
  #pragma unroll
  for (int L = 1; L < 3; L++) {
    const unsigned short *W = sW + (L == 1 ? SW_2 : SW_3);
    const float *b = sb + 64 * L;
    #pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      mlp_f4 acc = {0.f, 0.f, 0.f, 0.f};
      #pragma unroll
      for (int kt = 0; kt < 4; kt++) acc = mfma(ldA(W, MLP_TS, 16 * mt, 16 * kt, lane), T.h[L - 1][kt], acc);
      #pragma unroll
      for (int i = 0; i < 4; i++) acc[i] += b[16 * mt + 4 * q + i];
      mlp_f4 g;
      #pragma unroll
      for (int i = 0; i < 4; i++) {
        float d;
        g[i] = gelu(acc[i], d);
        T.d[L][mt][i] = d;
      }
      T.h[L][mt] = tobf(g);
    }
  }
  // layer 4: W4p[16][64]
  mlp_f4 acc = {0.f, 0.f, 0.f, 0.f};
  #pragma unroll
  for (int kt = 0; kt < 4; kt++) acc = mfma(ldA(sW + SW_4, MLP_TS, 0, 16 * kt, lane), T.h[2][kt], acc);
  #pragma unroll
  for (int i = 0; i < 4; i++) acc[i] += (q == 0 && i < MLP_NOUT) ? sb[SB_4 + i] : 0.f;
  T.y = acc;
}

// the biases and the norm, which every tile reads, into LDS
__device__ __forceinline__ void load_biases(float *sb, const float *p, const float *norm) {
  for (int t = threadIdx.x; t < SB_N; t += blockDim.x)
    sb[t] = t < 64             ? p[MP_B1 + t]
            : t < 128          ? p[MP_B2 + t - 64]
            : t < SB_4         ? p[MP_B3 + t - 128]
            : t < SB_4 + 3     ? p[MP_B4 + t - SB_4]
            : t < SB_NORM      ? 0.f
                               : norm[t - SB_NORM];
}
// the BF16 weights into their padded LDS layout (tr: the transposes too)
__device__ __forceinline__ void load_weights(unsigned short *sW, const unsigned short *wb, bool tr) {
  static_assert(WB_N % 4 == 0, "four weights at a time");
  #pragma unroll 5
  for (int t4 = threadIdx.x; t4 < WB_N / 4; t4 += MLP_WG) {
    const mlp_s4 v = reinterpret_cast<const mlp_s4 *>(wb)[t4];
    const int t = 4 * t4;
    if (t < WB_2) {
      *reinterpret_cast<mlp_s4 *>(sW + SW_1 + (t >> 4) * MLP_TS1 + (t & 15)) = v;
    } else {
      const int o = t - WB_2, r = o >> 6, k = o & 63;  // rows of W2, W3, W4
      *reinterpret_cast<mlp_s4 *>(sW + SW_2 + r * MLP_TS + k) = v;
      if (tr)
        #pragma unroll
        for (int j = 0; j < 4; j++)
          sW[r < 128 ? ST_2 + ((r & 64) + k + j) * MLP_TS + (r & 63)
                     : ST_4 + (k + j) * MLP_TS1 + r - 128] = (unsigned short)v[j];
    }
  }
}

// inference: Y[node][c] = scale_c * y_c (the predicted traction increment)
__global__ void __launch_bounds__(MLP_WG) k_mlp_forward(int n, const float *__restrict__ X,
                                                     const unsigned short *__restrict__ wb,
                                                     const float *__restrict__ p,
                                                     const float *__restrict__ norm, float *Y) {
  __shared__ __align__(16) unsigned short sW[SW_N];
  __shared__ float sb[SB_N];
  load_biases(sb, p, norm);
  load_weights(sW, wb, false);
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ntile = (n + 15) / 16, nw = gridDim.x * (blockDim.x >> 6);
  for (int tile = blockIdx.x * (blockDim.x >> 6) + wv; tile < ntile; tile += nw) {
    MlpTile T;
    mlp_forward(sW, sb, X, n, 16 * tile, lane, T);
    const int node = 16 * tile + (lane & 15);
    if (lane < 16 && node < n)
      #pragma unroll
      for (int i = 0; i < MLP_NOUT; i++) Y[(size_t)node * MLP_NOUT + i] = T.y[i] * sb[SB_NORM + 2 * MLP_NIN + i];
  }
}

// transpose tile: S[node][feature] in LDS, row stride MLP_TS
__device__ __forceinline__ void st_tile(unsigned short *S, int f0, mlp_s4 v, int lane) {
  // lane holds node l%16, features f0 + 4q + j
  *reinterpret_cast<mlp_s4 *>(S + (lane & 15) * MLP_TS + f0 + 4 * (lane >> 4)) = v;
}
// operand from a transposed tile: lane supplies M[node 4q + j][c0 + l%16]
__device__ __forceinline__ mlp_s4 ld_tile(const unsigned short *S, int c0, int lane) {
  const unsigned short *r = S + 4 * (lane >> 4) * MLP_TS + c0 + (lane & 15);
  mlp_s4 v;
  #pragma unroll
  for (int j = 0; j < 4; j++) v[j] = (short)r[j * MLP_TS];
  return v;
}
// orders a wavefront's own LDS accesses
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// a wavefront's gradient sums: dW in MFMA output tiles, db per lane over its nodes
struct MlpAcc {
  mlp_f4 w1[4], w2[16], w3[16], w4[4], b[3][4], b4;
};
// dW tiles += dZ^T H over the 16 nodes of the tile held in the transpose tiles
template <int NM, int NN>
__device__ __forceinline__ void acc_dw(mlp_f4 *acc, const unsigned short *SZ,
                                       const unsigned short *SH, int lane) {
  mlp_s4 zf[NM], hf[NN];
  #pragma unroll
  for (int m = 0; m < NM; m++) zf[m] = ld_tile(SZ, 16 * m, lane);
  #pragma unroll
  for (int k = 0; k < NN; k++) hf[k] = ld_tile(SH, 16 * k, lane);
  #pragma unroll
  for (int m = 0; m < NM; m++)
    #pragma unroll
    for (int k = 0; k < NN; k++) acc[NN * m + k] = mfma(zf[m], hf[k], acc[NN * m + k]);
}
// the wavefront's sums added to (first: stored in) the workgroup's, in ga_slot's layout;
// all of a group's old sums are read before the first new one is stored, since one after
// the other every sum would wait for the LDS twice
template <int N>
__device__ __forceinline__ void put_tiles(float *red, const mlp_f4 *v, int lane, bool first) {
  float *t = red + 16 * (4 * (lane >> 4)) + (lane & 15);
  mlp_f4 o[N];
  #pragma unroll
  for (int m = 0; m < N; m++)
    #pragma unroll
    for (int i = 0; i < 4; i++) o[m][i] = first ? 0.f : t[256 * m + 16 * i];
  #pragma unroll
  for (int m = 0; m < N; m++)
    #pragma unroll
    for (int i = 0; i < 4; i++) t[256 * m + 16 * i] = o[m][i] + v[m][i];
}
__device__ __forceinline__ void put_bias(float *red, mlp_f4 v, int lane, bool first) {
  float *t = red + 4 * (lane >> 4);
  mlp_f4 o;
  #pragma unroll
  for (int i = 0; i < 4; i++) o[i] = first ? 0.f : t[i];
  #pragma unroll
  for (int i = 0; i < 4; i++)
    for (int k = 1; k < 16; k <<= 1) v[i] += __shfl_xor(v[i], k, 16);
  if ((lane & 15) == 0)
    #pragma unroll
    for (int i = 0; i < 4; i++) t[i] = o[i] + v[i];
}

// training: loss and gradient partial sums of one workgroup over the 16-node tiles its first
// nw <= MLP_TW wavefronts take in turn; targets are raw increments T[n][3].  A wavefront keeps
// all its sums in registers (160 of them matrix accumulators, one wavefront a SIMD): in
// LDS, where every tile's products were added before, a tile cost 640 more LDS accesses
// and 200 lane exchanges for the biases.  65,536 rows: 135 -> 58 us.
__global__ void __launch_bounds__(MLP_WG, 1) k_mlp_train(int n, int nw, const float *__restrict__ X,
                                                  const float *__restrict__ Tg,
                                                  const unsigned short *__restrict__ wb,
                                                  const float *__restrict__ p,
                                                  const float *__restrict__ norm, float *part,
                                                  double *lpart) {
  __shared__ __align__(16) unsigned short sW[ST_N];
  __shared__ __align__(16) unsigned short tz[MLP_TW][16 * MLP_TS], th[MLP_TW][16 * MLP_TS];
  __shared__ float red[GA_N];
  __shared__ double lred[MLP_TW];
  __shared__ float sb[SB_N];
  load_biases(sb, p, norm);
  load_weights(sW, wb, true);
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, q = lane >> 4;
  unsigned short *SZ = tz[wv], *SH = th[wv];
  const int ntile = (n + 15) / 16;
  const float gs = 2.f / (3.f * (float)n);
  double lsum = 0.;
  MlpAcc A;
  const mlp_f4 zero = {0.f, 0.f, 0.f, 0.f};
  #pragma unroll
  for (int t = 0; t < 16; t++) A.w2[t] = A.w3[t] = zero;
  #pragma unroll
  for (int t = 0; t < 4; t++) A.w1[t] = A.w4[t] = A.b[0][t] = A.b[1][t] = A.b[2][t] = zero;
  A.b4 = zero;
  for (int tile = wv < nw ? blockIdx.x * nw + wv : ntile; tile < ntile; tile += gridDim.x * nw) {
    MlpTile T;
    mlp_forward(sW, sb, X, n, 16 * tile, lane, T);
    const int node = 16 * tile + (lane & 15);
    // dL/dy of the normalised outputs
    mlp_f4 dy = zero;
    if (q == 0 && node < n)
      #pragma unroll
      for (int i = 0; i < MLP_NOUT; i++) {
        const float e = T.y[i] - Tg[(size_t)node * MLP_NOUT + i] / sb[SB_NORM + 2 * MLP_NIN + i];
        lsum += (double)e * e;
        dy[i] = gs * e;
      }
    const mlp_s4 dyb = tobf(dy);
    // layer 4: db4, dW4 = dY^T H3, dH3 = W4^T dY
    A.b4 += dy;
    wave_fence();
    st_tile(SZ, 0, dyb, lane);
    #pragma unroll
    for (int kt = 0; kt < 4; kt++) st_tile(SH, 16 * kt, T.h[2][kt], lane);
    wave_fence();
    acc_dw<1, 4>(A.w4, SZ, SH, lane);
    mlp_f4 dz[4];
    mlp_s4 dzb[4];
    #pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      mlp_f4 d = mfma(ldA(sW + ST_4, MLP_TS1, 16 * mt, 0, lane), dyb, zero);
      d *= T.d[2][mt];
      dz[mt] = d;
      dzb[mt] = tobf(d);
    }
    // layers 3 and 2: db, dW = dZ^T H_prev, dH_prev = W^T dZ
    #pragma unroll
    for (int L = 2; L >= 1; L--) {
      const unsigned short *WT = sW + (L == 2 ? ST_3 : ST_2);
      wave_fence();
      #pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        A.b[L][mt] += dz[mt];
        st_tile(SZ, 16 * mt, dzb[mt], lane);
        st_tile(SH, 16 * mt, T.h[L - 1][mt], lane);
      }
      wave_fence();
      acc_dw<4, 4>(L == 2 ? A.w3 : A.w2, SZ, SH, lane);
      mlp_s4 nzb[4];
      #pragma unroll
      for (int mt = 0; mt < 4; mt++) {
        mlp_f4 d = zero;
        #pragma unroll
        for (int kt = 0; kt < 4; kt++) d = mfma(ldA(WT, MLP_TS, 16 * mt, 16 * kt, lane), dzb[kt], d);
        d *= T.d[L - 1][mt];
        dz[mt] = d;
        nzb[mt] = tobf(d);
      }
      #pragma unroll
      for (int mt = 0; mt < 4; mt++) dzb[mt] = nzb[mt];
    }
    // layer 1: db1, dW1 = dZ1^T X
    wave_fence();
    #pragma unroll
    for (int mt = 0; mt < 4; mt++) {
      A.b[0][mt] += dz[mt];
      st_tile(SZ, 16 * mt, dzb[mt], lane);
    }
    st_tile(SH, 0, T.x, lane);
    wave_fence();
    acc_dw<4, 1>(A.w1, SZ, SH, lane);
  }
  for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
  if (lane == 0) lred[wv] = lsum;
  // the wavefronts that had a tile, one after the other
  const int nact = min(nw, ntile - nw * (int)blockIdx.x);
  for (int w = 0; w < nact; w++) {
    if (w == wv) {
      const bool first = w == 0;
      put_tiles<4>(red + GA_1, A.w1, lane, first);
      put_tiles<16>(red + GA_2, A.w2, lane, first);
      put_tiles<16>(red + GA_3, A.w3, lane, first);
      put_tiles<4>(red + GA_4, A.w4, lane, first);
      #pragma unroll
      for (int L = 0; L < 3; L++)
        #pragma unroll
        for (int t = 0; t < 4; t++) put_bias(red + GA_B + 64 * L + 16 * t, A.b[L][t], lane, first);
      put_bias(red + GA_B + 192, A.b4, lane, first);
    }
    __syncthreads();
  }
  for (int t = threadIdx.x; t < GA_N; t += MLP_WG) part[(size_t)blockIdx.x * GA_N + t] = red[t];
  if (threadIdx.x == 0) {
    double s = 0.;
    for (int w = 0; w < MLP_TW; w++) s += lred[w];
    lpart[blockIdx.x] = s;
  }
}

// accumulator slot of parameter p (the inverse of the tile layout above)
__device__ __forceinline__ int ga_slot(int p) {
  if (p < MP_B1) {
    const int o = p / MLP_NIN, i = p % MLP_NIN;
    return GA_1 + 256 * (o / 16) + 16 * (o % 16) + i;
  }
  if (p < MP_W2) return GA_B + (p - MP_B1);
  if (p < MP_B2 || (p >= MP_W3 && p < MP_B3)) {
    const int base = p < MP_B2 ? MP_W2 : MP_W3, g = p < MP_B2 ? GA_2 : GA_3;
    const int o = (p - base) / 64, i = (p - base) % 64;
    return g + 256 * (4 * (o / 16) + i / 16) + 16 * (o % 16) + i % 16;
  }
  if (p < MP_W3) return GA_B + 64 + (p - MP_B2);
  if (p < MP_W4) return GA_B + 128 + (p - MP_B3);
  if (p < MP_B4) {
    const int o = (p - MP_W4) / 64, i = (p - MP_W4) % 64;
    return GA_4 + 256 * (i / 16) + 16 * o + i % 16;
  }
  return GA_B + 192 + (p - MP_B4);
}

// grad[p] = sum over workgroups of the partials: a workgroup takes 64 parameters, each of
// its MLP_RW wavefronts the partials w, w + MLP_RW, ... in order, then the wavefronts in
// order.  (One thread a parameter walked all partials one after the other: 131 us at 512
// partials against 6 us at 256.)
#define MLP_RW 16
__global__ void __launch_bounds__(64 * MLP_RW) k_mlp_reduce(int nwg, const float *__restrict__ part,
                                                            float *grad) {
  __shared__ float red[MLP_RW][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, p = blockIdx.x * 64 + lane;
  const int s = p < MP_N ? ga_slot(p) : 0;
  float g = 0.f;
  #pragma unroll 4
  for (int w = wv; w < nwg; w += MLP_RW) g += part[(size_t)w * GA_N + s];
  red[wv][lane] = g;
  __syncthreads();
  if (wv == 0 && p < MP_N) {
    for (int w = 1; w < MLP_RW; w++) g += red[w][lane];
    grad[p] = g;
  }
}

// BF16 copy of the weights in the padded tile layout
__device__ __forceinline__ int wb_slot(int p) {
  if (p < MP_B1) return WB_1 + 16 * (p / MLP_NIN) + p % MLP_NIN;
  if (p >= MP_W2 && p < MP_B2) return WB_2 + (p - MP_W2);
  if (p >= MP_W3 && p < MP_B3) return WB_3 + (p - MP_W3);
  if (p >= MP_W4 && p < MP_B4) return WB_4 + (p - MP_W4);
  return -1;
}
__global__ void k_mlp_to_bf16(const float *__restrict__ p, unsigned short *wb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= MP_N) return;
  const int s = wb_slot(i);
  if (s >= 0) wb[s] = f2bf(p[i]);
}

// Adam (Kingma and Ba, 2015) on the FP32 master parameters, then their BF16 copy
__global__ void k_mlp_adam(float *p, float *m1, float *m2, const float *__restrict__ g, float lr,
                           float b1, float b2, float eps, float c1, float c2, unsigned short *wb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= MP_N) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi, b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float v = p[i] - lr * (a * c1) / (sqrtf(b * c2) + eps);
  p[i] = v;
  const int s = wb_slot(i);
  if (s >= 0) wb[s] = f2bf(v);
}

// ---------------------------------------------------------------------------
extern "C" int rbc3d_mlp_create(rbc3d_mlp **out) {
  if (!out) return RBC3D_EINVAL;
  rbc3d_mlp *m = new rbc3d_mlp();
  int r = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) == hipSuccess ? 0 : RBC3D_EHIP;
  if (!r) r = m->p.ensure(MP_N);
  if (!r) r = m->m1.ensure(MP_N);
  if (!r) r = m->m2.ensure(MP_N);
  if (!r) r = m->grad.ensure(MP_N);
  if (!r) r = m->norm.ensure(2 * MLP_NIN + MLP_NOUT);
  if (!r) r = m->wb.ensure(WB_N);
  if (!r && hipMemset(m->wb.p, 0, WB_N * 2) != hipSuccess) r = RBC3D_EHIP;
  if (!r && hipMemset(m->p.p, 0, MP_N * 4) != hipSuccess) r = RBC3D_EHIP;
  if (!r) {
    std::vector<float> nm(2 * MLP_NIN + MLP_NOUT, 1.f);
    #pragma unroll
    for (int i = 0; i < MLP_NIN; i++) nm[i] = 0.f;
    if (hipMemcpy(m->norm.p, nm.data(), nm.size() * 4, hipMemcpyHostToDevice) != hipSuccess) r = RBC3D_EHIP;
  }
  if (r) {
    rbc_set_error("rbc3d_mlp_create: device allocation");
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return r;
  }
  *out = m;
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_destroy(rbc3d_mlp *m) {
  if (!m) return RBC3D_OK;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  if (m->ev) (void)hipEventDestroy(m->ev);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_nparams(void) { return MP_N; }

extern "C" int rbc3d_mlp_set_stream(rbc3d_mlp *m, void *stream) {
  if (!m) return RBC3D_EINVAL;
  HIP_TRY(hipStreamSynchronize(m->st()));
  m->ext = (hipStream_t)stream;
  m->use_ext = true;
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_set_params(rbc3d_mlp *m, const float *params) {
  if (!m || !params) return RBC3D_EINVAL;
  for (int i = 0; i < MP_N; i++)
    if (!std::isfinite(params[i])) return RBC3D_ENONFINITE;
  HIP_TRY(hipStreamSynchronize(m->st()));
  HIP_TRY(hipMemcpy(m->p.p, params, MP_N * 4, hipMemcpyHostToDevice));
  HIP_TRY(hipMemset(m->m1.p, 0, MP_N * 4));
  HIP_TRY(hipMemset(m->m2.p, 0, MP_N * 4));
  m->t = 0;
  k_mlp_to_bf16<<<(MP_N + 255) / 256, 256, 0, m->stream>>>(m->p.p, m->wb.p);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(m->stream));
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_get_params(rbc3d_mlp *m, float *params) {
  if (!m || !params) return RBC3D_EINVAL;
  HIP_TRY(hipStreamSynchronize(m->st()));
  HIP_TRY(hipMemcpy(params, m->p.p, MP_N * 4, hipMemcpyDeviceToHost));
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_set_norm(rbc3d_mlp *m, const float *mean_in, const float *std_in,
                                  const float *scale_out) {
  if (!m || !mean_in || !std_in || !scale_out) return RBC3D_EINVAL;
  std::vector<float> nm(2 * MLP_NIN + MLP_NOUT);
  #pragma unroll
  for (int i = 0; i < MLP_NIN; i++) {
    if (!(std_in[i] > 0.f)) return RBC3D_EINVAL;
    nm[i] = mean_in[i];
    nm[MLP_NIN + i] = 1.f / std_in[i];
  }
  #pragma unroll
  for (int i = 0; i < MLP_NOUT; i++) {
    if (!(scale_out[i] > 0.f)) return RBC3D_EINVAL;
    nm[2 * MLP_NIN + i] = scale_out[i];
  }
  HIP_TRY(hipStreamSynchronize(m->st()));
  HIP_TRY(hipMemcpy(m->norm.p, nm.data(), nm.size() * 4, hipMemcpyHostToDevice));
  return RBC3D_OK;
}

int rbc_mlp_forward(rbc3d_mlp *m, int n, const float *d_x, float *d_y, hipStream_t st) {
  if (n <= 0) return RBC3D_OK;
  const int ntile = (n + 15) / 16;
  const unsigned nblk = (unsigned)std::min(1024, (ntile + 3) / 4);
  k_mlp_forward<<<nblk, MLP_WG, 0, st>>>(n, d_x, m->wb.p, m->p.p, m->norm.p, d_y);
  HIP_TRY(hipGetLastError());
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_forward_dev(rbc3d_mlp *m, int n, const float *d_x, float *d_y) {
  if (!m || n < 0 || (n > 0 && (!d_x || !d_y))) return RBC3D_EINVAL;
  RBC_TRY(rbc_mlp_forward(m, n, d_x, d_y, m->st()));
  HIP_TRY(hipStreamSynchronize(m->st()));
  return RBC3D_OK;
}

static int mlp_grad(rbc3d_mlp *m, int n, const float *d_x, const float *d_t, double *loss) {
  hipStream_t st = m->st();
  const int ntile = (n + 15) / 16;
  // A wavefront a workgroup up to 256 tiles, then more of them: the wavefronts add their sums
  // in turn, some 5 us each (gradient call of 100 rows 67.5 us with four, 53.5 with one;
  // 4,096 rows 70 and 62).
  const int nw = std::min(MLP_TW, (ntile + 255) / 256), nwg = std::min(256, (ntile + nw - 1) / nw);
  RBC_TRY(m->part.ensure((size_t)nwg * GA_N));
  RBC_TRY(m->lpart.ensure(nwg));
  k_mlp_train<<<nwg, MLP_WG, 0, m->st()>>>(n, nw, d_x, d_t, m->wb.p, m->p.p, m->norm.p,
                                                m->part.p, m->lpart.p);
  k_mlp_reduce<<<(MP_N + 63) / 64, 64 * MLP_RW, 0, m->st()>>>(nwg, m->part.p, m->grad.p);
  HIP_TRY(hipGetLastError());
  if (loss) {
    std::vector<double> lp(nwg);
    HIP_TRY(hipMemcpyAsync(lp.data(), m->lpart.p, nwg * 8, hipMemcpyDeviceToHost, m->st()));
    HIP_TRY(hipStreamSynchronize(m->st()));
    double s = 0;
    #pragma unroll
    for (int i = 0; i < nwg; i++) s += lp[i];
    *loss = s / (3.0 * n);
  }
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_grad_dev(rbc3d_mlp *m, int n, const float *d_x, const float *d_t,
                                  float *d_grad, double *loss) {
  if (!m || n <= 0 || !d_x || !d_t) return RBC3D_EINVAL;
  RBC_TRY(mlp_grad(m, n, d_x, d_t, loss));
  if (d_grad)
    HIP_TRY(hipMemcpyAsync(d_grad, m->grad.p, MP_N * 4, hipMemcpyDeviceToDevice, m->st()));
  HIP_TRY(hipStreamSynchronize(m->st()));
  return RBC3D_OK;
}

extern "C" int rbc3d_mlp_adam_step_dev(rbc3d_mlp *m, int n, const float *d_x, const float *d_t,
                                       float lr, double *loss) {
  if (!m || n <= 0 || !d_x || !d_t || !(lr > 0.f)) return RBC3D_EINVAL;
  RBC_TRY(mlp_grad(m, n, d_x, d_t, loss));
  m->t++;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = (float)(1.0 / (1.0 - std::pow((double)b1, m->t)));
  const float c2 = (float)(1.0 / (1.0 - std::pow((double)b2, m->t)));
  k_mlp_adam<<<(MP_N + 255) / 256, 256, 0, m->st()>>>(m->p.p, m->m1.p, m->m2.p, m->grad.p, lr, b1,
                                                        b2, 1e-8f, c1, c2, m->wb.p);
  HIP_TRY(hipGetLastError());
  // the update is complete when the call returns, so a caller may read or use the
  // parameters from any stream
  HIP_TRY(hipStreamSynchronize(m->st()));
  return RBC3D_OK;
}

// Make stream st wait for the work queued on the network's stream (an event, no host
// wait): a forward on another stream then reads the parameters after every update.
int rbc_mlp_wait(rbc3d_mlp *m, hipStream_t st) {
  if (m->st() == st) return RBC3D_OK;
  if (!m->ev) HIP_TRY(hipEventCreateWithFlags(&m->ev, hipEventDisableTiming));
  HIP_TRY(hipEventRecord(m->ev, m->st()));
  HIP_TRY(hipStreamWaitEvent(st, m->ev, 0));
  return RBC3D_OK;
}
