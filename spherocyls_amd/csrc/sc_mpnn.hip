// Message-passing network over the contact graph: warm starts for the
// minimiser (no reference counterpart).
//
// Network (hidden width 64, three message-passing layers, SiLU):
//   node input  x_i = (cos 2phi, sin 2phi, R, A)
//   edge input  e_ij = (1 - d/sigma, D_x/d, D_y/d, b_x, b_y) for every contact
//               (closest-point distance d < sigma), D the closest-approach
//               vector from j to i and b = r_j - r_i (sheared coordinates,
//               minimum image); both directions i<-j and j<-i are edges
//   h0_i   = silu(W_e [x_i, 1])
//   layer: z_ij = W_m [h_i, h_j, e_ij, 1];  M_i = sum_j silu(z_ij)
//          h_i <- h_i + silu(W_u [h_i, M_i, 1])
//   output y_i = W_o [h_i, 1]  (first three components), the displacement
//          (dx, dy, dphi) = scale * y_i in sheared coordinates.
// Every affine map carries its bias as the last weight row against a constant
// 1 column of its input, so the forward and backward passes are plain GEMMs:
//   forward    C[M x N] = A[M x K] . W[K x N]       (k_gemm_nt with Bt = W^T)
//   input grad dA       = dC . W^T                  (k_gemm_nt with Bt = W)
//   weight grad dW      = A^T . dC                   (k_gemm_tn, per-chunk
//                                                     partials summed in order)
// GEMM operands are BF16 and accumulate in FP32 on the MFMA units
// (v_mfma_f32_16x16x32_bf16 of gfx950 over 32-wide K steps, the
// 16x16x16 form for a remaining 16: a wavefront computes 16-row strips, one
// 16 x 16 tile per MFMA); the residual stream h, pre-activations, gradients,
// FP32 master weights and Adam moments stay FP32.  Edges are stored grouped by
// receiver (CSR), with the index of each edge's reverse, so every sum over
// edges runs in a fixed order: forward and backward are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/spherocyls.h"
#include "../../include/spherocyls_mpnn.h"
#include "sc_internal.h"
#include "sc_status.h"
#include "sc_physics.h"

namespace sc {
namespace mp {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

constexpr int kH = 64;        // hidden width
constexpr int kLayers = 3;
constexpr int kKx = 16;       // [x(4), 1, 0..]
constexpr int kKe = 144;      // [h_i, h_j, e(5), 1, 0..]
constexpr int kKu = 144;      // [h, M, 1, 0..]
constexpr int kKo = 80;       // [h, 1, 0..]
constexpr int kNo = 16;       // output width (3 used)
constexpr int kEdgeFeat = 5;
constexpr int kNodeFeat = 4;
// largest warm-start displacement per component (particle radii are ~0.5)
constexpr float kCapXY = 1.0f;
constexpr float kCapPhi = 0.5f;

// parameter blocks (FP32 master layout, each W row-major [K][N])
struct Layout {
  int we, wm[kLayers], wu[kLayers], wo, total;
  Layout() {
    int o = 0;
    we = o; o += kKx * kH;
    for (int l = 0; l < kLayers; ++l) { wm[l] = o; o += kKe * kH; wu[l] = o; o += kKu * kH; }
    wo = o; o += kKo * kNo;
    total = o;
  }
};

__device__ __forceinline__ bf16 to_bf16(float v) {
  // round to nearest even
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__device__ __forceinline__ float from_bf16(bf16 v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_grad(float z) {
  float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// ---------------------------------------------------------------------------
// GEMMs
// ---------------------------------------------------------------------------
enum Epi : int {
  kEpiStore = 0,     // C32 = acc
  kEpiSiluH = 1,     // C32 = acc (pre-activation); H32 = silu(acc)
  kEpiResid = 2,     // C32 = acc; H32 = Hin32 + silu(acc)
};

// One 16 x 16 x 32 MFMA step: lane group g = lane / 16 holds the eight K
// indices 8 g .. 8 g + 7 of its row of A and of its column of B.  The unit
// pairs A's and B's slots by lane group and position, so any assignment of K
// to slots that A and B share gives the same sum.
__device__ __forceinline__ f32x4 mfma32(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// C[M x NT*16] = A[M x K] . Bt^T, A row-major (lda), Bt row-major [N][ldb].
// One wavefront per 16-row strip, four per workgroup.  K % 16 == 0,
// lda % 8 == 0, ldb % 8 == 0 (16-byte operand loads in the 32-wide steps).
template <int NT, int EPI>
__global__ void __launch_bounds__(256) k_gemm_nt(const bf16* __restrict__ A, int lda,
                                                  const bf16* __restrict__ Bt, int ldb, int M, int K,
                                                  float* __restrict__ C, int ldc,
                                                  const float* __restrict__ Hin,
                                                  float* __restrict__ Hout, int ldh) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r0 = (blockIdx.x * 4 + wave) * 16;
  if (r0 >= M) return;
  const int ar = r0 + (lane & 15);
  const int kq = 4 * (lane >> 4);
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  int k0 = 0;
  const int k8 = 8 * (lane >> 4);
  for (; k0 + 32 <= K; k0 += 32) {
    s16x8 a = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (ar < M) a = *reinterpret_cast<const s16x8*>(A + (size_t)ar * lda + k0 + k8);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const s16x8 b =
          *reinterpret_cast<const s16x8*>(Bt + (size_t)(t * 16 + (lane & 15)) * ldb + k0 + k8);
      acc[t] = mfma32(a, b, acc[t]);
    }
  }
  for (; k0 < K; k0 += 16) {
    bf16x4 a = bf16x4{0, 0, 0, 0};
    if (ar < M) a = *reinterpret_cast<const bf16x4*>(A + (size_t)ar * lda + k0 + kq);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bf16x4 b =
          *reinterpret_cast<const bf16x4*>(Bt + (size_t)(t * 16 + (lane & 15)) * ldb + k0 + kq);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
    }
  }
  // acc[t][i] = C[r0 + 4 (lane / 16) + i][t * 16 + lane % 16]
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int col = t * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = r0 + kq + i;
      if (row >= M) continue;
      const float v = acc[t][i];
      C[(size_t)row * ldc + col] = v;
      if (EPI == kEpiSiluH) Hout[(size_t)row * ldh + col] = silu(v);
      if (EPI == kEpiResid)
        Hout[(size_t)row * ldh + col] = Hin[(size_t)row * ldh + col] + silu(v);
    }
  }
}

// Partial weight gradients: P[chunk][K][N] = A[rows of chunk]^T . D[rows of
// chunk], A row-major [M][lda] (K = KT*16 columns), D row-major [M][ldd] (N =
// NTN*16 columns).  One workgroup per chunk of `chunk` rows (a multiple of
// 32); its four wavefronts share the KT x NTN output tiles.
//
// The reduction runs down the rows, along which the operands are strided, so
// a lane that loaded its own operand would read 16 two-byte values per MFMA
// from 16 rows.  Instead a thread reads two neighbouring columns (4 bytes) of
// 8 rows, a wavefront 256 contiguous bytes of each row, and packs them into
// the two 16-byte operands those columns need; operands go through LDS
// ([8 rows][column], read back as one ds_read_b128 per operand) in two buffers,
// so a stage's loads are in flight while the previous stage multiplies.  What
// bounds it is reading A and D once (416 B a row for the 144 x 64 maps).
// 128000 edges, 144 x 64: 31 us (1.7 TB/s); 420 us with two-byte loads and 2048
// rows per chunk (63 workgroups).
template <int KT, int NTN>
__global__ void __launch_bounds__(256) k_gemm_tn(const bf16* __restrict__ A, int lda,
                                                  const bf16* __restrict__ D, int ldd, int M,
                                                  int chunk, float* __restrict__ P) {
  constexpr int kCols = (KT + NTN) * 16, kPairs = kCols / 2;
  constexpr int kTasks = kPairs * 4;                // column pairs x groups of 8 rows
  constexpr int kPer = (kTasks + 255) / 256;        // tasks per thread
  constexpr int kTiles = KT * NTN, kAcc = (kTiles + 3) / 4;
  __shared__ s16x8 s_op[2][4 * kCols];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m_begin = blockIdx.x * chunk, m_end = min(M, m_begin + chunk);
  uint32_t raw[kPer][8];
  auto load = [&](int m0) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int q = tid + 256 * k;
      const int col = 2 * (q % kPairs), mg = q / kPairs;
      const bool inA = col < KT * 16;
      const bf16* base = inA ? A + col : D + (col - KT * 16);
      const int ld = inA ? lda : ldd;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = m0 + 8 * mg + i;
        raw[k][i] = q < kTasks && m < m_end
                        ? *reinterpret_cast<const uint32_t*>(base + (size_t)m * ld)
                        : 0u;
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int q = tid + 256 * k;
      if (q >= kTasks) continue;
      const int col = 2 * (q % kPairs), mg = q / kPairs;
      s16x8 lo, hi;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        lo[i] = (short)(raw[k][i] & 0xffffu);
        hi[i] = (short)(raw[k][i] >> 16);
      }
      s_op[buf][mg * kCols + col] = lo;
      s_op[buf][mg * kCols + col + 1] = hi;
    }
  };
  f32x4 acc[kAcc];
#pragma unroll
  for (int t = 0; t < kAcc; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  load(m_begin);
  int buf = 0;
  for (int m0 = m_begin; m0 < m_end; m0 += 32, buf ^= 1) {
    // the other buffer is still being read by slower wavefronts; this one was
    // last read a stage earlier, before the previous barrier
    store(buf);
    __syncthreads();
    if (m0 + 32 < m_end) load(m0 + 32);
    const s16x8* op = s_op[buf] + (lane >> 4) * kCols + (lane & 15);
#pragma unroll
    for (int t = 0; t < kAcc; ++t) {
      const int tile = wave + 4 * t;
      if (tile < kTiles)
        acc[t] = mfma32(op[(tile / NTN) * 16], op[(KT + tile % NTN) * 16], acc[t]);
    }
  }
  float* Pc = P + (size_t)blockIdx.x * kTiles * 256;
  const int kq = 4 * (lane >> 4);
#pragma unroll
  for (int t = 0; t < kAcc; ++t) {
    const int tile = wave + 4 * t;
    if (tile >= kTiles) continue;
    const int kt = tile / NTN, nt = tile % NTN;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      Pc[(size_t)(kt * 16 + kq + i) * (NTN * 16) + nt * 16 + (lane & 15)] = acc[t][i];
  }
}

// Rows per partial of a weight gradient over M rows: 256, so that a few tens of
// thousands of rows already give every CU a workgroup, doubled while there
// would be more than 512 partials (each K x N floats, written and read back).
inline int chunk_rows(int M) {
  int c = 256;
  while ((M + c - 1) / c > 512) c *= 2;
  return c;
}
constexpr int kMaxChunks = 512;

// G[i] = sum over chunks of P[chunk][i].  A workgroup takes 32 elements; its 8
// groups of 32 threads each sum a contiguous eighth of the chunks in order,
// and the eight sums are added in order.  (One thread per element walks all
// chunks in one dependent chain: 17 us for 63 chunks of 9216 elements.)
__global__ void __launch_bounds__(256) k_sum_partials(const float* __restrict__ P, int nchunks,
                                                       int size, float* __restrict__ G) {
  __shared__ float s[256];
  const int t = threadIdx.x, part = t >> 5, i = blockIdx.x * 32 + (t & 31);
  const int per = (nchunks + 7) / 8, c0 = part * per, c1 = min(nchunks, c0 + per);
  float v = 0.0f;
  if (i < size)
#pragma unroll 8
    for (int c = c0; c < c1; ++c) v += P[(size_t)c * size + i];
  s[t] = v;
  __syncthreads();
  if (t < 32 && i < size) {
    float sum = s[t];
    for (int k = 1; k < 8; ++k) sum += s[t + 32 * k];
    G[i] = sum;
  }
}

// ---------------------------------------------------------------------------
// graph input builders (BF16 GEMM operands with the constant-1 column)
// ---------------------------------------------------------------------------
__global__ void k_build_x(const float* __restrict__ nf, int n, bf16* __restrict__ X) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bf16* r = X + (size_t)i * kKx;
  for (int c = 0; c < kKx; ++c) {
    float v = c < kNodeFeat ? nf[(size_t)i * kNodeFeat + c] : (c == kNodeFeat ? 1.0f : 0.0f);
    r[c] = to_bf16(v);
  }
}

// The input builders write 8 columns per thread: two 16-byte loads of FP32
// features, one 16-byte store of 8 BF16 values (each column is converted, and
// the node input summed over in-edges, in the same order as one thread per
// column would).
static_assert(kH % 8 == 0 && kKe % 8 == 0 && kKu % 8 == 0 && kKo % 8 == 0,
              "builder rows are whole 8-column chunks");
__device__ __forceinline__ void load8(const float* __restrict__ p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x;
  v[1] = a.y;
  v[2] = a.z;
  v[3] = a.w;
  v[4] = b.x;
  v[5] = b.y;
  v[6] = b.z;
  v[7] = b.w;
}

__device__ __forceinline__ void store8(bf16* __restrict__ p, const float (&v)[8]) {
  uint4 w;
  w.x = (unsigned)to_bf16(v[0]) | ((unsigned)to_bf16(v[1]) << 16);
  w.y = (unsigned)to_bf16(v[2]) | ((unsigned)to_bf16(v[3]) << 16);
  w.z = (unsigned)to_bf16(v[4]) | ((unsigned)to_bf16(v[5]) << 16);
  w.w = (unsigned)to_bf16(v[6]) | ((unsigned)to_bf16(v[7]) << 16);
  *reinterpret_cast<uint4*>(p) = w;
}

// Ein[e] = [h_dst, h_src, e_feat, 1, 0...]; one thread per (edge, 8 columns).
__global__ void k_build_edge_in(const float* __restrict__ H, const int* __restrict__ src,
                                const int* __restrict__ dst, const float* __restrict__ ef, int ne,
                                bf16* __restrict__ Ein) {
  constexpr int kCh = kKe / 8, kHc = kH / 8;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)ne * kCh) return;
  const int e = (int)(t / kCh), ch = (int)(t % kCh);
  float v[8];
  if (ch < kHc) {
    load8(H + (size_t)dst[e] * kH + 8 * ch, v);
  } else if (ch < 2 * kHc) {
    load8(H + (size_t)src[e] * kH + 8 * (ch - kHc), v);
  } else {
    for (int k = 0; k < 8; ++k) {
      const int c = 8 * ch + k;
      v[k] = c < 2 * kH + kEdgeFeat ? ef[(size_t)e * kEdgeFeat + (c - 2 * kH)]
                                    : (c == 2 * kH + kEdgeFeat ? 1.0f : 0.0f);
    }
  }
  store8(Ein + (size_t)e * kKe + 8 * ch, v);
}

// Uin[i] = [h_i, sum over in-edges of silu(z), 1, 0...]; one thread per (node, 8 columns).
__global__ void k_build_node_in(const float* __restrict__ H, const float* __restrict__ Z,
                                const int* __restrict__ off, int n, bf16* __restrict__ Uin) {
  constexpr int kCh = kKu / 8, kHc = kH / 8;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * kCh) return;
  const int i = (int)(t / kCh), ch = (int)(t % kCh);
  float v[8];
  if (ch < kHc) {
    load8(H + (size_t)i * kH + 8 * ch, v);
  } else if (ch < 2 * kHc) {
    for (int k = 0; k < 8; ++k) v[k] = 0.0f;
    for (int e = off[i]; e < off[i + 1]; ++e) {
      float z[8];
      load8(Z + (size_t)e * kH + 8 * (ch - kHc), z);
      for (int k = 0; k < 8; ++k) v[k] += silu(z[k]);
    }
  } else {
    for (int k = 0; k < 8; ++k) v[k] = 8 * ch + k == 2 * kH ? 1.0f : 0.0f;
  }
  store8(Uin + (size_t)i * kKu + 8 * ch, v);
}

// Hin[i] = [h_i, 1, 0...]; one thread per (node, 8 columns).
__global__ void k_build_out_in(const float* __restrict__ H, int n, bf16* __restrict__ Hin) {
  constexpr int kCh = kKo / 8, kHc = kH / 8;
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * kCh) return;
  const int i = (int)(t / kCh), ch = (int)(t % kCh);
  float v[8];
  if (ch < kHc) {
    load8(H + (size_t)i * kH + 8 * ch, v);
  } else {
    for (int k = 0; k < 8; ++k) v[k] = 8 * ch + k == kH ? 1.0f : 0.0f;
  }
  store8(Hin + (size_t)i * kKo + 8 * ch, v);
}

// ---------------------------------------------------------------------------
// backward helpers
// ---------------------------------------------------------------------------
// loss = mean over nodes and the 3 outputs of (y - t)^2; dY (BF16, 16 wide).
// Per-block partial losses, summed in order by k_sum_partials.
__global__ void k_loss(const float* __restrict__ Y, const float* __restrict__ T, int n,
                       bf16* __restrict__ dY, float* __restrict__ part) {
  __shared__ float sh[256];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.0f;
  if (i < n) {
    const float inv = 1.0f / (3.0f * (float)n);
    for (int c = 0; c < kNo; ++c) {
      float g = 0.0f;
      if (c < 3) {
        float d = Y[(size_t)i * kNo + c] - T[(size_t)i * 3 + c];
        l += d * d * inv;
        g = 2.0f * d * inv;
      }
      dY[(size_t)i * kNo + c] = to_bf16(g);
    }
  }
  sh[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// dPre = dH (given as columns [col0, col0+64) of dIn, row stride ldin) * silu'(Pre)
__global__ void k_act_grad(const float* __restrict__ dIn, int ldin, int col0,
                           const float* __restrict__ Pre, int rows, bf16* __restrict__ dPre) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)rows * kH) return;
  const int r = (int)(t / kH), c = (int)(t % kH);
  dPre[t] = to_bf16(dIn[(size_t)r * ldin + col0 + c] * silu_grad(Pre[t]));
}

// dH[i][c] = dIn[i][c], c < 64 (row stride ld)
__global__ void k_take_cols(const float* __restrict__ dIn, int ld, int n, float* __restrict__ dH) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * kH) return;
  dH[t] = dIn[(t / kH) * ld + t % kH];
}

// Edge pre-activation gradient: dZ[e] = dM[dst(e)] * silu'(Z[e]); dM is
// columns [64, 128) of dUin (row stride kKu).
__global__ void k_edge_grad(const float* __restrict__ dUin, const float* __restrict__ Z,
                            const int* __restrict__ dst, int ne, bf16* __restrict__ dZ) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)ne * kH) return;
  const int e = (int)(t / kH), c = (int)(t % kH);
  dZ[t] = to_bf16(dUin[(size_t)dst[e] * kKu + kH + c] * silu_grad(Z[t]));
}

// dH_prev[i] = dH[i] + dUin[i][0:64] + sum over in-edges e of dEin[e][0:64]
//             + sum over out-edges (= reverses of in-edges) of dEin[rev e][64:128]
__global__ void k_node_grad(const float* __restrict__ dH, const float* __restrict__ dUin,
                            const float* __restrict__ dEin, const int* __restrict__ off,
                            const int* __restrict__ rev, int n, float* __restrict__ dHprev) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)n * kH) return;
  const int i = (int)(t / kH), c = (int)(t % kH);
  float v = dH[t] + dUin[(size_t)i * kKu + c];
  for (int e = off[i]; e < off[i + 1]; ++e)
    v += dEin[(size_t)e * kKe + c] + dEin[(size_t)rev[e] * kKe + kH + c];
  dHprev[t] = v;
}

// ---------------------------------------------------------------------------
// parameters
// ---------------------------------------------------------------------------
// BF16 copies of every W: natural [K][N] (input gradients) and transposed
// [N][K] (forward).
__global__ void k_refresh(const float* __restrict__ W, int K, int N, bf16* __restrict__ Wn,
                          bf16* __restrict__ Wt) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= K * N) return;
  const int k = t / N, n = t % N;
  const bf16 v = to_bf16(W[t]);
  Wn[t] = v;
  Wt[(size_t)n * K + k] = v;
}

__global__ void k_adam(float* __restrict__ W, const float* __restrict__ G, float* __restrict__ m,
                       float* __restrict__ v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = G[i];
  const float mi = b1 * m[i] + (1.0f - b1) * g;
  const float vi = b2 * v[i] + (1.0f - b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  W[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// ---------------------------------------------------------------------------
// graph of a system's current state
// ---------------------------------------------------------------------------
// Closest-point contact of storage particles g and q evaluated with the lower
// caller id first (as the force kernels do), so both directions of a pair see
// the same contact; r.dx, r.dy are turned to point from q to g.
__device__ bool pair_canonical(const SystemView& v, int g, int q, double Lx, double Ly,
                               double gam, PairOut<double>& r) {
  const bool gFirst = v.b.id[g] < v.b.id[q];
  const int p = gFirst ? g : q, o = gFirst ? q : g;
  double dx = min_image(v.b.x[p] - v.b.x[o], Lx);
  double dy = min_image(v.b.y[p] - v.b.y[o], Ly);
  dx += gam * dy;
  if (!pair_contact_f64(dx, dy, v.b.nx[p], v.b.ny[p], v.b.nx[o], v.b.ny[o], v.b.A[p], v.b.A[o],
                        v.b.R[p] + v.b.R[o], r))
    return false;
  if (!gFirst) {
    r.dx = -r.dx;
    r.dy = -r.dy;
  }
  return true;
}

// Contacts of storage particle g (closest-point distance < sigma) over the 3 x 3
// cells around it, partner storage indices sorted by caller id; count only when
// out is null.
__device__ int contacts_of(const SystemView& v, int g, int* out, int cap) {
  const int pk = v.pack_of[g];
  const PackInfo P = v.packs[pk];
  const PackScal S = v.scal[pk];
  const double Lx = S.Lx, Ly = S.Ly, gam = S.gamma;
  double xw = v.b.x[g], yw = v.b.y[g];
  wrap_coord(xw, Lx);
  wrap_coord(yw, Ly);
  int col, row;
  cell_col_row(xw, yw, Lx, Ly, P, col, row);
  int rs[3], cs[3], nr = 0, nc = 0;
  for (int d = -1; d <= 1; ++d) {
    int r = (row + d + P.rows) % P.rows, c = (col + d + P.cols) % P.cols;
    bool dr = false, dc = false;
    for (int k = 0; k < nr; ++k) dr |= rs[k] == r;
    for (int k = 0; k < nc; ++k) dc |= cs[k] == c;
    if (!dr) rs[nr++] = r;
    if (!dc) cs[nc++] = c;
  }
  int n = 0;
  for (int i = 0; i < nr; ++i)
    for (int j = 0; j < nc; ++j) {
      const int cell = P.coff + rs[i] * P.cols + cs[j];
      const int m = min(v.cnt[cell], P.cap);
      for (int k = 0; k < m; ++k) {
        const int q = v.slot[(size_t)cell * P.cap + k];
        if (q == g) continue;
        PairOut<double> r;
        if (!pair_canonical(v, g, q, Lx, Ly, gam, r)) continue;
        if (out) {
          // insertion by caller id keeps every node's edge order fixed
          int pos = min(n, cap - 1);
          const int idq = v.b.id[q];
          while (pos > 0 && v.b.id[out[pos - 1]] > idq) {
            if (pos < cap) out[pos] = out[pos - 1];
            --pos;
          }
          if (n < cap) out[pos] = q;
        }
        ++n;
      }
    }
  return n;
}

// The graph kernels give a node 16 lanes, a cell around it to each of the first
// nine: a cell is a chain of dependent loads (count, slots, records), and with
// one lane a node walking nine of them one after the other, 68 thousand nodes
// were one wavefront a SIMD and took 57 us to count and 86 us to fill (now 40
// and 66).  A member beyond the bounding circles is no contact and is
// spared the pair math.
constexpr int kNodeLanes = 16, kNodeBlock = 256;
constexpr int kNodeList = 64;  // contacts a node's lanes order in LDS; more are left to one lane

// Calls hit(q) for the contacts of node g in this lane's cell.
template <class Hit>
__device__ __forceinline__ void contacts_in_cell(const SystemView& v, int g, int lane, Hit hit) {
  const int pk = v.pack_of[g];
  const PackInfo& P = v.packs[pk];
  const double Lx = v.scal[pk].Lx, Ly = v.scal[pk].Ly, gam = v.scal[pk].gamma;
  // each cell once: in grids of fewer than 3 rows (columns) the first nr (nc) of
  // row - 1, row, row + 1 differ
  const int nr = min(P.rows, 3), nc = min(P.cols, 3);
  if (lane >= nr * nc) return;
  const double2 xy = load2(v.b.x, g), ra = load2(v.b.R, g);
  double xw = xy.x, yw = xy.y;
  wrap_coord(xw, Lx);
  wrap_coord(yw, Ly);
  int col, row;
  cell_col_row(xw, yw, Lx, Ly, P, col, row);
  const int i = lane / nc, j = lane - i * nc;
  const int cell = P.coff + (row - 1 + i + P.rows) % P.rows * P.cols +
                   (col - 1 + j + P.cols) % P.cols;
  const int m = min(v.cnt[cell], P.cap);
  for (int k = 0; k < m; ++k) {
    const int q = v.slot[(size_t)cell * P.cap + k];
    const double2 xyq = load2(v.b.x, q), raq = load2(v.b.R, q);
    const double dy = min_image(xy.y - xyq.y, Ly);
    const double dx = min_image(xy.x - xyq.x, Lx) + gam * dy;
    const double reach = ra.x + ra.y + raq.x + raq.y;
    if (q == g || !(dx * dx + dy * dy < reach * reach * (1.0 + 1e-10))) continue;
    PairOut<double> r;
    if (pair_canonical(v, g, q, Lx, Ly, gam, r)) hit(q);
  }
}

__global__ void __launch_bounds__(kNodeBlock) k_graph_count(SystemView v, int* deg) {
  const size_t t = (size_t)blockIdx.x * kNodeBlock + threadIdx.x;
  const int g = (int)(t / kNodeLanes), lane = (int)(t % kNodeLanes);
  if (g >= v.ntot) return;
  int n = 0;
  contacts_in_cell(v, g, lane, [&](int) { ++n; });
  for (int off = kNodeLanes / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, kNodeLanes);
  if (lane == 0) deg[g] = n;
}

// Nodes in storage order; in-edges of node g (receiver g, senders = contacts)
// at off[g] .. off[g+1]-1, senders by caller id.  Writes node features, edge
// src / dst and features.
__global__ void __launch_bounds__(kNodeBlock)
    k_graph_fill(SystemView v, const int* __restrict__ off, int* __restrict__ src,
                 int* __restrict__ dst, float* __restrict__ nf, float* __restrict__ ef) {
  __shared__ int s_q[kNodeBlock / kNodeLanes][kNodeList], s_id[kNodeBlock / kNodeLanes][kNodeList];
  __shared__ int s_n[kNodeBlock / kNodeLanes];
  const size_t t = (size_t)blockIdx.x * kNodeBlock + threadIdx.x;
  const int g = (int)(t / kNodeLanes), lane = (int)(t % kNodeLanes);
  const int node = threadIdx.x / kNodeLanes;
  const bool live = g < v.ntot;
  const int o = live ? off[g] : 0, cap = live ? off[g + 1] - o : 0;
  if (lane == 0) s_n[node] = 0;
  __syncthreads();
  if (live && cap <= kNodeList) {
    contacts_in_cell(v, g, lane, [&](int q) {
      const int at = atomicAdd(&s_n[node], 1);
      if (at < kNodeList) {
        s_q[node][at] = q;
        s_id[node][at] = v.b.id[q];
      }
    });
  } else if (live && lane == 0) {
    contacts_of(v, g, src + o, cap);
  }
  __threadfence_block();  // (the one lane's list is read by the others)
  __syncthreads();
  if (!live) return;
  if (lane == 0) {
    const double phi = v.b.phi[g];
    nf[(size_t)g * kNodeFeat + 0] = (float)cos(2.0 * phi);
    nf[(size_t)g * kNodeFeat + 1] = (float)sin(2.0 * phi);
    nf[(size_t)g * kNodeFeat + 2] = (float)v.b.R[g];
    nf[(size_t)g * kNodeFeat + 3] = (float)v.b.A[g];
  }
  const PackScal& S = v.scal[v.pack_of[g]];
  for (int k = lane; k < cap; k += kNodeLanes) {
    int e = o + k, q;
    if (cap <= kNodeList) {  // its place among the senders
      q = s_q[node][k];
      const int id = s_id[node][k];
      e = o;
      for (int i = 0; i < cap; ++i) e += s_id[node][i] < id;
      src[e] = q;
    } else {
      q = src[e];
    }
    dst[e] = g;
    const double bx = min_image(v.b.x[q] - v.b.x[g], S.Lx);
    const double by = min_image(v.b.y[q] - v.b.y[g], S.Ly);
    PairOut<double> r;
    pair_canonical(v, g, q, S.Lx, S.Ly, S.gamma, r);
    const double sig = v.b.R[g] + v.b.R[q];
    float* f = ef + (size_t)e * kEdgeFeat;
    f[0] = (float)(1.0 - r.dist / sig);
    // crossed rods (d = 0) have no contact normal
    f[1] = r.dist > 0 ? (float)(r.dx / r.dist) : 0.0f;
    f[2] = r.dist > 0 ? (float)(r.dy / r.dist) : 0.0f;
    f[3] = (float)bx;
    f[4] = (float)by;
  }
}

// Exclusive prefix sums of the node degrees, off[g] = deg[0] + ... + deg[g-1]
// and off[n] = the number of edges, in three launches: the sum of each tile
// of kScanTile degrees, a one-workgroup scan of the tile sums, then each
// tile's offsets.  Integer sums: the offsets are exact.
constexpr int kScanTile = 1024;  // 256 threads x 4 degrees
__global__ void __launch_bounds__(256) k_scan_tiles(const int* __restrict__ deg, int n,
                                                    int* __restrict__ tsum) {
  __shared__ int s[256];
  const int t = threadIdx.x, base = blockIdx.x * kScanTile + 4 * t;
  int v = 0;
  for (int k = 0; k < 4; ++k)
    if (base + k < n) v += deg[base + k];
  s[t] = v;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) s[t] += s[t + h];
    __syncthreads();
  }
  if (t == 0) tsum[blockIdx.x] = s[0];
}

// One workgroup: exclusive scan of the nt tile sums in place, 1024 at a time.
__global__ void __launch_bounds__(1024) k_scan_tile_sums(int* tsum, int nt) {
  __shared__ int s[1024];
  __shared__ int carry;
  const int t = threadIdx.x;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < nt; base += 1024) {
    const int i = base + t;
    const int v = i < nt ? tsum[i] : 0;
    s[t] = v;
    __syncthreads();
    for (int h = 1; h < 1024; h <<= 1) {
      const int add = t >= h ? s[t - h] : 0;
      __syncthreads();
      s[t] += add;
      __syncthreads();
    }
    if (i < nt) tsum[i] = carry + s[t] - v;
    __syncthreads();  // every thread has read carry
    if (t == 1023) carry += s[1023];
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) k_scan_offsets(const int* __restrict__ deg, int n,
                                                      const int* __restrict__ tsum,
                                                      int* __restrict__ off) {
  __shared__ int s[256];
  const int t = threadIdx.x, base = blockIdx.x * kScanTile + 4 * t;
  int v[4], sum = 0;
  for (int k = 0; k < 4; ++k) {
    v[k] = base + k < n ? deg[base + k] : 0;
    sum += v[k];
  }
  s[t] = sum;
  __syncthreads();
  for (int h = 1; h < 256; h <<= 1) {
    const int add = t >= h ? s[t - h] : 0;
    __syncthreads();
    s[t] += add;
    __syncthreads();
  }
  int run = tsum[blockIdx.x] + s[t] - sum;
  for (int k = 0; k < 4; ++k) {
    if (base + k < n) off[base + k] = run;
    run += v[k];
  }
  // degrees past n count zero, so the last thread ends on the total
  if (blockIdx.x == gridDim.x - 1 && t == 255) off[n] = run;
}

// Reverse edge of each edge k (receiver dst[k], sender src[k]): the first edge
// of the sender's in-edges whose sender is that receiver.  A contact graph is
// symmetric; a missing reverse edge raises *bad.
__global__ void k_graph_rev(const int* __restrict__ off, const int* __restrict__ src,
                            const int* __restrict__ dst, int e, int* __restrict__ rev,
                            int* __restrict__ bad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= e) return;
  const int i = dst[k], j = src[k];
  int r = -1;
  for (int t = off[j]; t < off[j + 1]; ++t)
    if (src[t] == i) {
      r = t;
      break;
    }
  rev[k] = r;
  if (r < 0) atomicOr(bad, 1);
}

// x, y, phi of storage particle g += scale * y_g, each component clamped to
// +-cap (a proposal, not a step the minimiser must trust) and non-finite
// outputs dropped
__device__ __forceinline__ double proposal(float y, float scale, double cap) {
  double v = (double)(scale * y);
  if (!isfinite(v)) return 0.0;
  return fmin(fmax(v, -cap), cap);
}

// Checks of a graph handed over by the caller (offsets already checked), and
// the receivers and reverse edges that go with it.  Nodes: senders in range and
// increasing within a receiver's edges, finite node features.
enum GraphFault : int { kBadOrder = 1, kBadPair = 2, kBadNode = 4, kBadEdge = 8 };
__device__ __forceinline__ bool finite_bits(float v) {
  return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
}
__global__ void k_check_nodes(const int* __restrict__ off, const int* __restrict__ src,
                              const float* __restrict__ nf, int n, int* __restrict__ dst,
                              int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int fault = 0, last = 0;
  for (int k = off[i]; k < off[i + 1]; ++k) {
    const int j = src[k];
    dst[k] = i;
    if (k > off[i] && j <= last) fault |= kBadOrder;
    if (j < 0 || j >= n) fault |= kBadPair;
    last = j;
  }
  for (int c = 0; c < kNodeFeat; ++c)
    if (!finite_bits(nf[(size_t)i * kNodeFeat + c])) fault |= kBadNode;
  if (fault) atomicOr(bad, fault);
}

// Edges: the reverse of every edge by binary search in its sender's edges
// (where senders do not increase the search may miss, but stays inside), and
// finite edge features.
__global__ void k_check_edges(const int* __restrict__ off, const int* __restrict__ src,
                              const int* __restrict__ dst, const float* __restrict__ ef, int n,
                              int e, int* __restrict__ rev, int* __restrict__ bad) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= e) return;
  const int i = dst[k], j = src[k];
  int fault = 0;
  if (j >= 0 && j < n) {
    const int end = off[j + 1];
    int lo = off[j], hi = end;
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if (src[mid] < i) lo = mid + 1;
      else hi = mid;
    }
    if (lo >= end || src[lo] != i) fault |= kBadPair;
    rev[k] = lo;
  }
  for (int c = 0; c < kEdgeFeat; ++c)
    if (!finite_bits(ef[(size_t)k * kEdgeFeat + c])) fault |= kBadEdge;
  if (fault) atomicOr(bad, fault);
}

__global__ void k_apply(Bank b, const float* __restrict__ Y, float sx, float sy, float sp,
                        double cap_xy, double cap_phi, int n) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  b.x[g] += proposal(Y[(size_t)g * kNo + 0], sx, cap_xy);
  b.y[g] += proposal(Y[(size_t)g * kNo + 1], sy, cap_xy);
  b.phi[g] += proposal(Y[(size_t)g * kNo + 2], sp, cap_phi);
}

}  // namespace mp
}  // namespace sc

using namespace sc;
using namespace sc::mp;

struct sc_mpnn {
  int device = 0;
  // damped warm start: stashed positions and per-packing best energy / factor
  double *x0 = nullptr, *y0 = nullptr, *p0 = nullptr, *bestE = nullptr, *bestL = nullptr;
  int wcap = 0, wpack = 0;
  hipStream_t stream = nullptr;
  Layout lay;
  float scale[3] = {1.0f, 1.0f, 1.0f};
  std::string err;
  std::vector<void*> allocs;
  // parameters
  float *W = nullptr, *G = nullptr, *Am = nullptr, *Av = nullptr;
  bf16 *Wn = nullptr, *Wt = nullptr;  // same offsets as W
  // graph (capacity)
  int n = 0, e = 0, ncap = 0, ecap = 0;
  bool has_forward = false;
  int *off = nullptr, *src = nullptr, *dst = nullptr, *rev = nullptr;
  float *nf = nullptr, *ef = nullptr;
  // activations
  bf16* X = nullptr;
  float* Ze = nullptr;                 // encoder pre-activation [n][64]
  float* Hs[kLayers + 1] = {};         // residual stream per layer [n][64]
  bf16* Ein[kLayers] = {};             // [e][144]
  float* Z[kLayers] = {};              // [e][64]
  bf16* Uin[kLayers] = {};             // [n][144]
  float* U[kLayers] = {};              // [n][64]
  bf16* Hin = nullptr;                 // [n][80]
  float* Y = nullptr;                  // [n][16]
  float* T = nullptr;                  // [n][3] targets
  // backward scratch
  bf16 *dY = nullptr, *dPre = nullptr, *dZe = nullptr;
  float *dA = nullptr, *dH = nullptr, *dH2 = nullptr, *dEin = nullptr, *P = nullptr;
  float* part = nullptr;
  size_t pcap = 0;
  int* d_deg = nullptr;
  int* d_scan = nullptr;  // per-tile sums of the degree scan
  int* d_flag = nullptr;  // graph build: a contact without its reverse edge
  // a graph from the caller until it has passed its checks
  struct Incoming {
    int ncap = 0, ecap = 0;
    int *off = nullptr, *src = nullptr, *dst = nullptr, *rev = nullptr, *bad = nullptr;
    float *nf = nullptr, *ef = nullptr;
  } in;

  template <typename T>
  T* dalloc(size_t count) {
    void* p = nullptr;
    if (hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T)) != hipSuccess)
      throw std::string("hipMalloc failed");
    allocs.push_back(p);
    return static_cast<T*>(p);
  }
  void dfree(void*& p) {
    if (!p) return;
    auto it = std::find(allocs.begin(), allocs.end(), p);
    if (it != allocs.end()) allocs.erase(it);
    (void)hipFree(p);
    p = nullptr;
  }
};

namespace {

#define MPCK(expr)                                                      \
  do {                                                                  \
    hipError_t e_ = (expr);                                             \
    if (e_ != hipSuccess) throw std::string(#expr) + ": " + hipGetErrorString(e_); \
  } while (0)

int fail(sc_mpnn* m, int st, const std::string& msg) {
  if (m) m->err = msg;
  return st;
}

inline int blocks(size_t n, int b = 256) { return (int)((n + b - 1) / b); }

template <class T>
void realloc_dev(sc_mpnn* m, T*& p, size_t count) {
  void* q = p;
  p = nullptr;
  m->dfree(q);
  p = m->template dalloc<T>(count);
}

void ensure_capacity(sc_mpnn* m, int n, int e) {
  if (n <= m->ncap && e <= m->ecap) return;
  const int nc = std::max(n, m->ncap), ec = std::max(e, m->ecap);
  m->ncap = m->ecap = m->n = m->e = 0;  // until all of them are there
  realloc_dev(m, m->off, nc + 1);
  realloc_dev(m, m->src, ec);
  realloc_dev(m, m->dst, ec);
  realloc_dev(m, m->rev, ec);
  realloc_dev(m, m->nf, (size_t)nc * kNodeFeat);
  realloc_dev(m, m->ef, (size_t)ec * kEdgeFeat);
  realloc_dev(m, m->X, (size_t)nc * kKx);
  realloc_dev(m, m->Ze, (size_t)nc * kH);
  for (int l = 0; l <= kLayers; ++l) realloc_dev(m, m->Hs[l], (size_t)nc * kH);
  for (int l = 0; l < kLayers; ++l) {
    realloc_dev(m, m->Ein[l], (size_t)ec * kKe);
    realloc_dev(m, m->Z[l], (size_t)ec * kH);
    realloc_dev(m, m->Uin[l], (size_t)nc * kKu);
    realloc_dev(m, m->U[l], (size_t)nc * kH);
  }
  realloc_dev(m, m->Hin, (size_t)nc * kKo);
  realloc_dev(m, m->Y, (size_t)nc * kNo);
  realloc_dev(m, m->T, (size_t)nc * 3);
  realloc_dev(m, m->dY, (size_t)nc * kNo);
  realloc_dev(m, m->dPre, (size_t)std::max(nc, ec) * kH);
  realloc_dev(m, m->dZe, (size_t)nc * kH);
  realloc_dev(m, m->dA, (size_t)nc * kKu);
  realloc_dev(m, m->dH, (size_t)nc * kH);
  realloc_dev(m, m->dH2, (size_t)nc * kH);
  realloc_dev(m, m->dEin, (size_t)ec * kKe);
  realloc_dev(m, m->d_deg, nc + 1);
  realloc_dev(m, m->d_scan, (size_t)nc / 1024 + 2);
  if (!m->d_flag) m->d_flag = m->template dalloc<int>(1);
  m->pcap = (size_t)std::min(std::max(nc, ec) / 256 + 1, kMaxChunks) * kKe * kH;
  realloc_dev(m, m->P, m->pcap);
  realloc_dev(m, m->part, (size_t)blocks(nc) + 1);
  m->ncap = nc;
  m->ecap = ec;
}

void ensure_incoming(sc_mpnn* m, int n, int e) {
  sc_mpnn::Incoming& in = m->in;
  if (!in.bad) in.bad = m->dalloc<int>(1);
  if (n > in.ncap) {
    in.ncap = 0;
    realloc_dev(m, in.off, (size_t)n + 1);
    realloc_dev(m, in.nf, (size_t)n * kNodeFeat);
    in.ncap = n;
  }
  if (e > in.ecap) {
    in.ecap = 0;
    realloc_dev(m, in.src, e);
    realloc_dev(m, in.dst, e);
    realloc_dev(m, in.rev, e);
    realloc_dev(m, in.ef, (size_t)e * kEdgeFeat);
    in.ecap = e;
  }
}

// Nodes and edges of a graph that the host checks.
constexpr long kHostGraph = 12288;

// What k_check_nodes and k_check_edges do, on the host.
int check_graph(int n, const float* nf, int e, const int* off, const int* src, const float* ef,
                std::vector<int>& dst, std::vector<int>& rev) {
  dst.resize(e);
  rev.resize(e);
  int bad = 0;
  for (int i = 0; i < n; ++i)
    for (int k = off[i]; k < off[i + 1]; ++k) {
      dst[k] = i;
      if (k > off[i] && src[k] <= src[k - 1]) bad |= kBadOrder;
      if (src[k] < 0 || src[k] >= n) bad |= kBadPair;
    }
  if (bad) return bad;
  for (int k = 0; k < e; ++k) {
    const int i = dst[k], end = off[src[k] + 1];
    int lo = off[src[k]], hi = end;
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if (src[mid] < i) lo = mid + 1;
      else hi = mid;
    }
    if (lo >= end || src[lo] != i) return kBadPair;
    rev[k] = lo;
  }
  for (size_t i = 0; i < (size_t)n * kNodeFeat; ++i)
    if (!std::isfinite(nf[i])) return kBadNode;
  for (size_t i = 0; i < (size_t)e * kEdgeFeat; ++i)
    if (!std::isfinite(ef[i])) return kBadEdge;
  return 0;
}

void refresh_bf16(sc_mpnn* m) {
  const Layout& L = m->lay;
  auto one = [&](int o, int K, int N) {
    hipLaunchKernelGGL(k_refresh, dim3(blocks((size_t)K * N)), dim3(256), 0, m->stream, m->W + o,
                       K, N, m->Wn + o, m->Wt + o);
  };
  one(L.we, kKx, kH);
  for (int l = 0; l < kLayers; ++l) {
    one(L.wm[l], kKe, kH);
    one(L.wu[l], kKu, kH);
  }
  one(L.wo, kKo, kNo);
}

template <int NT, int EPI>
void gemm_nt(sc_mpnn* m, const bf16* A, int lda, const bf16* Bt, int ldb, int M, int K, float* C,
             int ldc, const float* Hin = nullptr, float* Hout = nullptr, int ldh = 0) {
  if (M <= 0) return;
  hipLaunchKernelGGL((k_gemm_nt<NT, EPI>), dim3(blocks((size_t)M, 64)), dim3(256), 0, m->stream,
                     A, lda, Bt, ldb, M, K, C, ldc, Hin, Hout, ldh);
}

template <int KT, int NTN>
void gemm_tn(sc_mpnn* m, const bf16* A, const bf16* D, int M, float* Gout) {
  const int size = KT * NTN * 256;
  if (M <= 0) return;
  const int chunk = chunk_rows(M), chunks = (M + chunk - 1) / chunk;
  hipLaunchKernelGGL((k_gemm_tn<KT, NTN>), dim3(chunks), dim3(256), 0, m->stream, A, KT * 16, D,
                     NTN * 16, M, chunk, m->P);
  hipLaunchKernelGGL(k_sum_partials, dim3(blocks((size_t)size, 32)), dim3(256), 0, m->stream, m->P,
                     chunks, size, Gout);
}

void forward(sc_mpnn* m) {
  const Layout& L = m->lay;
  const int n = m->n, e = m->e;
  hipStream_t st = m->stream;
  hipLaunchKernelGGL(k_build_x, dim3(blocks(n)), dim3(256), 0, st, m->nf, n, m->X);
  gemm_nt<4, kEpiSiluH>(m, m->X, kKx, m->Wt + L.we, kKx, n, kKx, m->Ze, kH, nullptr, m->Hs[0], kH);
  for (int l = 0; l < kLayers; ++l) {
    if (e > 0) {
      hipLaunchKernelGGL(k_build_edge_in, dim3(blocks((size_t)e * (kKe / 8))), dim3(256), 0, st,
                         m->Hs[l], m->src, m->dst, m->ef, e, m->Ein[l]);
      gemm_nt<4, kEpiStore>(m, m->Ein[l], kKe, m->Wt + L.wm[l], kKe, e, kKe, m->Z[l], kH);
    }
    hipLaunchKernelGGL(k_build_node_in, dim3(blocks((size_t)n * (kKu / 8))), dim3(256), 0, st,
                       m->Hs[l], m->Z[l], m->off, n, m->Uin[l]);
    gemm_nt<4, kEpiResid>(m, m->Uin[l], kKu, m->Wt + L.wu[l], kKu, n, kKu, m->U[l], kH, m->Hs[l],
                          m->Hs[l + 1], kH);
  }
  hipLaunchKernelGGL(k_build_out_in, dim3(blocks((size_t)n * (kKo / 8))), dim3(256), 0, st,
                     m->Hs[kLayers], n, m->Hin);
  gemm_nt<1, kEpiStore>(m, m->Hin, kKo, m->Wt + L.wo, kKo, n, kKo, m->Y, kNo);
  m->has_forward = true;
}

float backward(sc_mpnn* m) {
  const Layout& L = m->lay;
  const int n = m->n, e = m->e;
  hipStream_t st = m->stream;
  const int nb = blocks(n);
  hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, st, m->Y, m->T, n, m->dY, m->part);
  float* dloss = m->P;  // scratch for the reduced loss
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, st, m->part, nb, 1, dloss);
  float loss = 0.0f;
  MPCK(hipMemcpyAsync(&loss, dloss, sizeof(float), hipMemcpyDeviceToHost, st));
  MPCK(hipStreamSynchronize(st));
  // decoder
  gemm_tn<kKo / 16, kNo / 16>(m, m->Hin, m->dY, n, m->G + L.wo);
  gemm_nt<5, kEpiStore>(m, m->dY, kNo, m->Wn + L.wo, kNo, n, kNo, m->dA, kKo);
  // gradient of the last hidden state: the h columns of dHin
  hipLaunchKernelGGL(k_take_cols, dim3(blocks((size_t)n * kH)), dim3(256), 0, st, m->dA, kKo, n,
                     m->dH);
  float* dH = m->dH;
  float* dH2 = m->dH2;
  for (int l = kLayers - 1; l >= 0; --l) {
    // node update: U = Uin . Wu, h_{l+1} = h_l + silu(U)
    hipLaunchKernelGGL(k_act_grad, dim3(blocks((size_t)n * kH)), dim3(256), 0, st, dH, kH, 0,
                       m->U[l], n, m->dPre);
    gemm_tn<kKu / 16, kH / 16>(m, m->Uin[l], m->dPre, n, m->G + L.wu[l]);
    gemm_nt<9, kEpiStore>(m, m->dPre, kH, m->Wn + L.wu[l], kH, n, kH, m->dA, kKu);
    if (e > 0) {
      hipLaunchKernelGGL(k_edge_grad, dim3(blocks((size_t)e * kH)), dim3(256), 0, st, m->dA,
                         m->Z[l], m->dst, e, m->dPre);
      gemm_tn<kKe / 16, kH / 16>(m, m->Ein[l], m->dPre, e, m->G + L.wm[l]);
      gemm_nt<9, kEpiStore>(m, m->dPre, kH, m->Wn + L.wm[l], kH, e, kH, m->dEin, kKe);
    } else {
      MPCK(hipMemsetAsync(m->G + L.wm[l], 0, sizeof(float) * kKe * kH, st));
    }
    hipLaunchKernelGGL(k_node_grad, dim3(blocks((size_t)n * kH)), dim3(256), 0, st, dH, m->dA,
                       m->dEin, m->off, m->rev, n, dH2);
    std::swap(dH, dH2);
  }
  // encoder
  hipLaunchKernelGGL(k_act_grad, dim3(blocks((size_t)n * kH)), dim3(256), 0, st, dH, kH, 0, m->Ze,
                     n, m->dZe);
  gemm_tn<kKx / 16, kH / 16>(m, m->X, m->dZe, n, m->G + L.we);
  return loss;
}

void init_params(sc_mpnn* m, unsigned long long seed) {
  // SplitMix64 stream, uniform(-b, b) with b = sqrt(3 / fan_in) on real inputs;
  // bias rows and padding rows start at zero
  uint64_t z = seed;
  auto next = [&]() {
    z += 0x9e3779b97f4a7c15ull;
    uint64_t r = z;
    r = (r ^ (r >> 30)) * 0xbf58476d1ce4e5b9ull;
    r = (r ^ (r >> 27)) * 0x94d049bb133111ebull;
    return r ^ (r >> 31);
  };
  auto uni = [&]() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); };
  const Layout& L = m->lay;
  std::vector<float> h(L.total, 0.0f);
  auto fill = [&](int o, int K, int N, int fan_in, double gain) {
    double b = gain * std::sqrt(3.0 / fan_in);
    for (int k = 0; k < fan_in; ++k)
      for (int c = 0; c < N; ++c) h[o + k * N + c] = (float)((2.0 * uni() - 1.0) * b);
    (void)K;
  };
  fill(L.we, kKx, kH, kNodeFeat, 1.0);
  for (int l = 0; l < kLayers; ++l) {
    fill(L.wm[l], kKe, kH, 2 * kH + kEdgeFeat, 1.0);
    fill(L.wu[l], kKu, kH, 2 * kH, 0.5);
  }
  fill(L.wo, kKo, kNo, kH, 0.1);
  for (int k = 0; k < kKo; ++k)
    for (int c = 3; c < kNo; ++c) h[L.wo + k * kNo + c] = 0.0f;
  MPCK(hipMemcpy(m->W, h.data(), sizeof(float) * L.total, hipMemcpyHostToDevice));
  MPCK(hipMemset(m->G, 0, sizeof(float) * L.total));
  MPCK(hipMemset(m->Am, 0, sizeof(float) * L.total));
  MPCK(hipMemset(m->Av, 0, sizeof(float) * L.total));
  refresh_bf16(m);
  MPCK(hipStreamSynchronize(m->stream));
}

}  // namespace

#define MP_BEGIN                 \
  if (!m) return SC_ERR_ARG;     \
  try {                          \
    MPCK(hipSetDevice(m->device));
#define MP_END                                      \
  }                                                 \
  catch (const std::string& s) {                    \
    return fail(m, SC_ERR_HIP, s);                  \
  }                                                 \
  catch (...) {                                     \
    std::string m_;                                 \
    const int st_ = sc::current_exception_status(&m_); \
    return fail(m, st_, m_);                        \
  }

extern "C" {

int sc_mpnn_create(sc_mpnn** out, int device, unsigned long long seed) {
  if (!out) return SC_ERR_ARG;
  *out = nullptr;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return SC_ERR_NO_DEVICE;
  if (device < 0 || device >= count) return SC_ERR_ARG;
  sc_mpnn* m = new (std::nothrow) sc_mpnn();
  if (!m) return SC_ERR_HOST;
  m->device = device;
  try {
    MPCK(hipSetDevice(device));
    MPCK(hipStreamCreate(&m->stream));
    const int P = m->lay.total;
    m->W = m->dalloc<float>(P);
    m->G = m->dalloc<float>(P);
    m->Am = m->dalloc<float>(P);
    m->Av = m->dalloc<float>(P);
    m->Wn = m->dalloc<bf16>(P);
    m->Wt = m->dalloc<bf16>(P);
    init_params(m, seed);
  } catch (const std::string& s) {
    sc_mpnn_destroy(m);
    return SC_ERR_HIP;
  } catch (...) {
    const int st = sc::current_exception_status(nullptr);
    sc_mpnn_destroy(m);
    return st;
  }
  *out = m;
  return SC_OK;
}

int sc_mpnn_destroy(sc_mpnn* m) {
  if (!m) return SC_ERR_ARG;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  for (void* p : m->allocs) (void)hipFree(p);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return SC_OK;
}

const char* sc_mpnn_last_error(const sc_mpnn* m) { return m ? m->err.c_str() : ""; }

int sc_mpnn_num_params(const sc_mpnn* m, int* count) {
  if (!m || !count) return SC_ERR_ARG;
  *count = m->lay.total;
  return SC_OK;
}

int sc_mpnn_get_params(sc_mpnn* m, float* out) {
  if (!out) return SC_ERR_ARG;
  MP_BEGIN
  MPCK(hipStreamSynchronize(m->stream));
  MPCK(hipMemcpy(out, m->W, sizeof(float) * m->lay.total, hipMemcpyDeviceToHost));
  return SC_OK;
  MP_END
}

int sc_mpnn_set_params(sc_mpnn* m, const float* in) {
  if (!in) return SC_ERR_ARG;
  MP_BEGIN
  MPCK(hipStreamSynchronize(m->stream));
  MPCK(hipMemcpy(m->W, in, sizeof(float) * m->lay.total, hipMemcpyHostToDevice));
  refresh_bf16(m);
  MPCK(hipStreamSynchronize(m->stream));
  m->has_forward = false;
  return SC_OK;
  MP_END
}

int sc_mpnn_get_grads(sc_mpnn* m, float* out) {
  if (!out) return SC_ERR_ARG;
  MP_BEGIN
  MPCK(hipStreamSynchronize(m->stream));
  MPCK(hipMemcpy(out, m->G, sizeof(float) * m->lay.total, hipMemcpyDeviceToHost));
  return SC_OK;
  MP_END
}

int sc_mpnn_set_output_scale(sc_mpnn* m, const float* scale3) {
  if (!m || !scale3) return SC_ERR_ARG;
  for (int i = 0; i < 3; ++i) {
    if (!(scale3[i] > 0) || !std::isfinite(scale3[i])) return SC_ERR_ARG;
    m->scale[i] = scale3[i];
  }
  return SC_OK;
}

int sc_mpnn_get_output_scale(const sc_mpnn* m, float* scale3) {
  if (!m || !scale3) return SC_ERR_ARG;
  for (int i = 0; i < 3; ++i) scale3[i] = m->scale[i];
  return SC_OK;
}

int sc_mpnn_load_graph(sc_mpnn* m, int n, const float* node_feat, int e, const int* offsets,
                       const int* src, const float* edge_feat) {
  if (!m || n <= 0 || e < 0 || !node_feat || !offsets || (e > 0 && (!src || !edge_feat)))
    return SC_ERR_ARG;
  if (offsets[0] != 0 || offsets[n] != e) return fail(m, SC_ERR_ARG, "offsets must run from 0 to e");
  for (int i = 0; i < n; ++i) {  // (the senders of the nodes before are looked at first)
    if (offsets[i + 1] >= offsets[i]) continue;
    for (int j = 0; j < i; ++j)
      for (int k = offsets[j] + 1; k < std::min(offsets[j + 1], e); ++k)
        if (src[k] <= src[k - 1])
          return fail(m, SC_ERR_ARG, "senders must increase within a receiver's edges");
    return fail(m, SC_ERR_ARG, "offsets must not decrease");
  }
  MP_BEGIN
  // Receivers, reverse edges and the other checks: by the GPU, into buffers of
  // their own (until the graph has passed, the one loaded before stays), or, for
  // a small graph, by the host, whose arrays then go up once.  64 nodes and 256
  // edges 37 us by the host and 98 by the GPU, 512 and 2048 66 and 114, 3000 and
  // 12000 123 and 128, 16384 and 65536 357 and 189.
  hipStream_t st = m->stream;
  const bool small = (long)n + e <= kHostGraph;
  std::vector<int> dst, rev;
  int bad = 0;
  if (small) {
    bad = check_graph(n, node_feat, e, offsets, src, edge_feat, dst, rev);
  } else {
    ensure_incoming(m, n, e);
    const sc_mpnn::Incoming& in = m->in;
    MPCK(hipMemsetAsync(in.bad, 0, sizeof(int), st));
    MPCK(hipMemcpyAsync(in.off, offsets, sizeof(int) * (n + 1), hipMemcpyHostToDevice, st));
    MPCK(hipMemcpyAsync(in.nf, node_feat, sizeof(float) * n * kNodeFeat, hipMemcpyHostToDevice,
                        st));
    if (e > 0) {
      MPCK(hipMemcpyAsync(in.src, src, sizeof(int) * e, hipMemcpyHostToDevice, st));
      MPCK(hipMemcpyAsync(in.ef, edge_feat, sizeof(float) * e * kEdgeFeat, hipMemcpyHostToDevice,
                          st));
    }
    hipLaunchKernelGGL(k_check_nodes, dim3(blocks(n)), dim3(256), 0, st, in.off, in.src, in.nf, n,
                       in.dst, in.bad);
    if (e > 0)
      hipLaunchKernelGGL(k_check_edges, dim3(blocks(e)), dim3(256), 0, st, in.off, in.src, in.dst,
                         in.ef, n, e, in.rev, in.bad);
    MPCK(hipMemcpyAsync(&bad, in.bad, sizeof(int), hipMemcpyDeviceToHost, st));
    MPCK(hipStreamSynchronize(st));
  }
  if (bad)
    return fail(m, SC_ERR_ARG,
                bad & kBadOrder  ? "senders must increase within a receiver's edges"
                : bad & kBadPair ? "edges must be symmetric (every i<-j has j<-i)"
                : bad & kBadNode ? "non-finite node feature"
                                 : "non-finite edge feature");
  ensure_capacity(m, n, e);
  m->n = n;
  m->e = e;
  const sc_mpnn::Incoming& in = m->in;
  auto take = [&](void* to, const void* host, const void* checked, size_t bytes) {
    if (bytes)
      MPCK(hipMemcpyAsync(to, small ? host : checked, bytes,
                          small ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice, st));
  };
  take(m->off, offsets, in.off, sizeof(int) * (n + 1));
  take(m->nf, node_feat, in.nf, sizeof(float) * n * kNodeFeat);
  take(m->src, src, in.src, sizeof(int) * e);
  take(m->dst, dst.data(), in.dst, sizeof(int) * e);
  take(m->rev, rev.data(), in.rev, sizeof(int) * e);
  take(m->ef, edge_feat, in.ef, sizeof(float) * e * kEdgeFeat);
  if (small) MPCK(hipStreamSynchronize(st));  // the host arrays are the caller's
  m->has_forward = false;
  return SC_OK;
  MP_END
}

int sc_mpnn_forward(sc_mpnn* m, float* out) {
  MP_BEGIN
  if (m->n <= 0) return fail(m, SC_ERR_STATE, "no graph loaded");
  forward(m);
  if (out) {
    std::vector<float> y((size_t)m->n * kNo);
    MPCK(hipMemcpyAsync(y.data(), m->Y, sizeof(float) * y.size(), hipMemcpyDeviceToHost,
                        m->stream));
    MPCK(hipStreamSynchronize(m->stream));
    for (int i = 0; i < m->n; ++i)
      for (int c = 0; c < 3; ++c) out[(size_t)i * 3 + c] = y[(size_t)i * kNo + c];
  } else {
    MPCK(hipStreamSynchronize(m->stream));
  }
  return SC_OK;
  MP_END
}

int sc_mpnn_backward(sc_mpnn* m, const float* target, float* loss) {
  if (!target) return SC_ERR_ARG;
  MP_BEGIN
  if (!m->has_forward) return fail(m, SC_ERR_STATE, "backward needs a forward pass first");
  MPCK(hipMemcpyAsync(m->T, target, sizeof(float) * m->n * 3, hipMemcpyHostToDevice, m->stream));
  float l = backward(m);
  MPCK(hipStreamSynchronize(m->stream));
  if (loss) *loss = l;
  return SC_OK;
  MP_END
}

int sc_mpnn_adam(sc_mpnn* m, float lr, float beta1, float beta2, float eps, int step) {
  if (!m || !(lr > 0) || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1) || step < 1)
    return SC_ERR_ARG;
  MP_BEGIN
  const int P = m->lay.total;
  const float c1 = 1.0f - std::pow(beta1, (float)step), c2 = 1.0f - std::pow(beta2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(blocks(P)), dim3(256), 0, m->stream, m->W, m->G, m->Am, m->Av, P,
                     lr, beta1, beta2, eps, c1, c2);
  refresh_bf16(m);
  MPCK(hipStreamSynchronize(m->stream));
  m->has_forward = false;
  return SC_OK;
  MP_END
}

int sc_mpnn_graph_from_system(sc_mpnn* m, sc_system* s, int* n_out, int* e_out) {
  if (!s) return SC_ERR_ARG;
  MP_BEGIN
  SystemView v;
  if (system_view(s, &v) != SC_OK) return fail(m, SC_ERR_ARG, "no system");
  if (v.device != m->device) return fail(m, SC_ERR_ARG, "system and network on different devices");
  MPCK(hipStreamSynchronize(v.stream));
  const int n = v.ntot;
  const int nt = (n + kScanTile - 1) / kScanTile;
  // degrees, their prefix sums and the edge count, all on the device
  auto offsets = [&]() -> int {
    hipLaunchKernelGGL(k_graph_count, dim3(blocks((size_t)n * kNodeLanes)), dim3(kNodeBlock), 0,
                       m->stream, v, m->d_deg);
    hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(256), 0, m->stream, m->d_deg, n, m->d_scan);
    hipLaunchKernelGGL(k_scan_tile_sums, dim3(1), dim3(1024), 0, m->stream, m->d_scan, nt);
    hipLaunchKernelGGL(k_scan_offsets, dim3(nt), dim3(256), 0, m->stream, m->d_deg, n, m->d_scan,
                       m->off);
    int total = 0;
    MPCK(hipMemcpyAsync(&total, m->off + n, sizeof(int), hipMemcpyDeviceToHost, m->stream));
    MPCK(hipStreamSynchronize(m->stream));
    return total;
  };
  ensure_capacity(m, n, m->ecap);
  int e = offsets();
  if (e > m->ecap) {  // growing the edge arrays reallocates the offsets too: count again
    ensure_capacity(m, n, e);
    e = offsets();
  }
  hipLaunchKernelGGL(k_graph_fill, dim3(blocks((size_t)n * kNodeLanes)), dim3(kNodeBlock), 0,
                     m->stream, v, m->off, m->src, m->dst, m->nf, m->ef);
  MPCK(hipMemsetAsync(m->d_flag, 0, sizeof(int), m->stream));
  if (e > 0)
    hipLaunchKernelGGL(k_graph_rev, dim3(blocks(e)), dim3(256), 0, m->stream, m->off, m->src,
                       m->dst, e, m->rev, m->d_flag);
  int bad = 0;
  MPCK(hipMemcpyAsync(&bad, m->d_flag, sizeof(int), hipMemcpyDeviceToHost, m->stream));
  MPCK(hipStreamSynchronize(m->stream));
  if (bad) return fail(m, SC_ERR_STATE, "contact graph is not symmetric");
  m->n = n;
  m->e = e;
  m->has_forward = false;
  if (n_out) *n_out = n;
  if (e_out) *e_out = e;
  return SC_OK;
  MP_END
}

int sc_mpnn_export_graph(sc_mpnn* m, sc_system* s, float* node_feat, int* offsets, int* src,
                         float* edge_feat) {
  if (!s || !node_feat || !offsets) return SC_ERR_ARG;
  MP_BEGIN
  SystemView v;
  if (system_view(s, &v) != SC_OK || v.ntot != m->n)
    return fail(m, SC_ERR_STATE, "graph was not built from this system");
  const int n = m->n, e = m->e;
  std::vector<int> off(n + 1), sr(e), id(n), pack_of(n);
  std::vector<PackInfo> packs(v.npack);
  std::vector<float> nf((size_t)n * kNodeFeat), ef((size_t)e * kEdgeFeat);
  MPCK(hipMemcpy(off.data(), m->off, sizeof(int) * (n + 1), hipMemcpyDeviceToHost));
  MPCK(hipMemcpy(sr.data(), m->src, sizeof(int) * e, hipMemcpyDeviceToHost));
  MPCK(hipMemcpy(id.data(), v.b.id, sizeof(int) * n, hipMemcpyDeviceToHost));
  MPCK(hipMemcpy(pack_of.data(), v.pack_of, sizeof(int) * n, hipMemcpyDeviceToHost));
  MPCK(hipMemcpy(packs.data(), v.packs, sizeof(PackInfo) * v.npack, hipMemcpyDeviceToHost));
  // b.id is the index within the packing: caller index = packing offset + id
  for (int g = 0; g < n; ++g) id[g] += packs[pack_of[g]].poff;
  MPCK(hipMemcpy(nf.data(), m->nf, sizeof(float) * nf.size(), hipMemcpyDeviceToHost));
  MPCK(hipMemcpy(ef.data(), m->ef, sizeof(float) * ef.size(), hipMemcpyDeviceToHost));
  // caller order: node id[g] <- storage g; a receiver's edges keep their order
  // (senders ascending by caller index: a packing's particles are contiguous)
  std::vector<int> deg(n);
  for (int g = 0; g < n; ++g) deg[id[g]] = off[g + 1] - off[g];
  offsets[0] = 0;
  for (int i = 0; i < n; ++i) offsets[i + 1] = offsets[i] + deg[i];
  for (int g = 0; g < n; ++g) {
    const int i = id[g];
    for (int c = 0; c < kNodeFeat; ++c) node_feat[(size_t)i * kNodeFeat + c] = nf[(size_t)g * kNodeFeat + c];
    for (int k = 0; k < deg[i]; ++k) {
      const int eo = offsets[i] + k, es = off[g] + k;
      if (src) src[eo] = id[sr[es]];
      if (edge_feat)
        for (int c = 0; c < kEdgeFeat; ++c)
          edge_feat[(size_t)eo * kEdgeFeat + c] = ef[(size_t)es * kEdgeFeat + c];
    }
  }
  return SC_OK;
  MP_END
}

namespace {

__global__ void k_stash(Bank b, int n, double* x0, double* y0, double* p0) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  x0[g] = b.x[g];
  y0[g] = b.y[g];
  p0[g] = b.phi[g];
}

// x = x0 + lambda * proposal, lambda per packing (lam_pack) or one for all.
__global__ void k_apply_from(Bank b, const float* __restrict__ Y, float sx, float sy, float sp,
                             double cap_xy, double cap_phi, int n, const double* x0,
                             const double* y0, const double* p0, double lam,
                             const double* lam_pack, const int* pack_of) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  const double l = lam_pack ? lam_pack[pack_of[g]] : lam;
  b.x[g] = x0[g] + l * proposal(Y[(size_t)g * kNo + 0], sx, cap_xy);
  b.y[g] = y0[g] + l * proposal(Y[(size_t)g * kNo + 1], sy, cap_xy);
  b.phi[g] = p0[g] + l * proposal(Y[(size_t)g * kNo + 2], sp, cap_phi);
}

// Keep, per packing, the factor whose state has the lowest energy so far.
__global__ void k_take_best(const double* pack_sum, int npack, double lam, double* bestE,
                            double* bestL, int first) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npack) return;
  const double e = pack_sum[(size_t)k * kNSum + kSeE];
  if (first) {
    bestE[k] = e;
    bestL[k] = 0.0;
  } else if (e < bestE[k]) {
    bestE[k] = e;
    bestL[k] = lam;
  }
}

}  // namespace

int sc_mpnn_warm_start_damped(sc_mpnn* m, sc_system* s, int nlam, const double* lambdas,
                              double* e_before, double* e_after, double* lam_out) {
  if (!s || nlam < 0 || (nlam > 0 && !lambdas)) return SC_ERR_ARG;
  for (int i = 0; i < nlam; ++i)
    if (!std::isfinite(lambdas[i])) return SC_ERR_ARG;
  int st = sc_mpnn_graph_from_system(m, s, nullptr, nullptr);
  if (st != SC_OK) return st;
  MP_BEGIN
  forward(m);
  SystemView v;
  system_view(s, &v);
  if (v.ntot > m->wcap) {
    realloc_dev(m, m->x0, v.ntot);
    realloc_dev(m, m->y0, v.ntot);
    realloc_dev(m, m->p0, v.ntot);
    m->wcap = v.ntot;
  }
  if (v.npack > m->wpack) {
    realloc_dev(m, m->bestE, v.npack);
    realloc_dev(m, m->bestL, v.npack);
    m->wpack = v.npack;
  }
  // the system's kernels run on its own stream: order the two streams
  MPCK(hipStreamSynchronize(m->stream));
  hipLaunchKernelGGL(k_stash, dim3(blocks(v.ntot)), dim3(256), 0, v.stream, v.b, v.ntot, m->x0,
                     m->y0, m->p0);
  // the unmoved state, then each factor; the bank keeps its storage order
  // throughout (no re-sort until the end), so the stash stays aligned
  for (int i = -1; i < nlam; ++i) {
    if (i >= 0)
      hipLaunchKernelGGL(k_apply_from, dim3(blocks(v.ntot)), dim3(256), 0, v.stream, v.b, m->Y,
                         m->scale[0], m->scale[1], m->scale[2], (double)kCapXY, (double)kCapPhi,
                         v.ntot, m->x0, m->y0, m->p0, lambdas[i], nullptr, v.pack_of);
    st = system_energy_pass(s);
    if (st != SC_OK) return st;
    hipLaunchKernelGGL(k_take_best, dim3(blocks(v.npack)), dim3(256), 0, v.stream, v.pack_sum,
                       v.npack, i >= 0 ? lambdas[i] : 0.0, m->bestE, m->bestL, i < 0 ? 1 : 0);
    if (i < 0 && e_before) {
      std::vector<double> ps((size_t)v.npack * kNSum);
      MPCK(hipMemcpyAsync(ps.data(), v.pack_sum, sizeof(double) * ps.size(),
                          hipMemcpyDeviceToHost, v.stream));
      MPCK(hipStreamSynchronize(v.stream));
      for (int k = 0; k < v.npack; ++k) e_before[k] = ps[(size_t)k * kNSum + kSeE];
    }
  }
  hipLaunchKernelGGL(k_apply_from, dim3(blocks(v.ntot)), dim3(256), 0, v.stream, v.b, m->Y,
                     m->scale[0], m->scale[1], m->scale[2], (double)kCapXY, (double)kCapPhi,
                     v.ntot, m->x0, m->y0, m->p0, 0.0, m->bestL, v.pack_of);
  if (e_after)
    MPCK(hipMemcpyAsync(e_after, m->bestE, sizeof(double) * v.npack, hipMemcpyDeviceToHost,
                        v.stream));
  if (lam_out)
    MPCK(hipMemcpyAsync(lam_out, m->bestL, sizeof(double) * v.npack, hipMemcpyDeviceToHost,
                        v.stream));
  MPCK(hipStreamSynchronize(v.stream));
  return system_positions_changed(s);
  MP_END
}

int sc_mpnn_warm_start(sc_mpnn* m, sc_system* s) {
  if (!s) return SC_ERR_ARG;
  int st = sc_mpnn_graph_from_system(m, s, nullptr, nullptr);
  if (st != SC_OK) return st;
  MP_BEGIN
  forward(m);
  SystemView v;
  system_view(s, &v);
  hipLaunchKernelGGL(k_apply, dim3(blocks(v.ntot)), dim3(256), 0, m->stream, v.b, m->Y,
                     m->scale[0], m->scale[1], m->scale[2], (double)kCapXY, (double)kCapPhi,
                     v.ntot);
  MPCK(hipStreamSynchronize(m->stream));
  return system_positions_changed(s);
  MP_END
}

}  // extern "C"
