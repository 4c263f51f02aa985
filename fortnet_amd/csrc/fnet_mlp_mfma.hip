// FP32 element networks on the matrix cores of gfx950 (v_mfma_f32_16x16x4_f32).
//
// Same mathematics as the generic network kernel (fprop, network.F90:146-180 / iPredict :314-347;
// the input gradient of fdevi, network.F90:183-244, in reverse mode, one sweep per output), laid
// out for MFMA: each wave owns 16 atoms of one element and runs them through every layer as
//   Z^T [d_out x 16] = W^T [d_out x d_in] . X^T [d_in x 16]
// in 16 x 16 output blocks with K = 4 per instruction.  W^T fragments come from a copy of the
// FP32 weights packed at model upload so that each instruction's A operand is one coalesced
// 256-byte load (L1/L2-resident, shared by all waves); X^T fragments come from the wave's
// activation rows in LDS, 4 K-steps per ds_read_b128 (the K order inside a 16-wide chunk is
// permuted to k = 16 c + 4 g + s, identically in the packed weights, so lane group g reads four
// consecutive features).  The accumulator fragment (rows = outputs 4 g + r, column = atom) is
// activated in registers, f'(z) of every hidden layer is kept in LDS in fragment order, and the
// activations go back to LDS as the next layer's rows.  The reverse sweep runs the transposed
// products delta_l^T = W_l . delta_{l+1}^T on separately packed fragments.  Products and sums are
// FP32 (as the generic FP32 kernel); per-atom outputs and input gradients are written in FP64.
//
// BF16 modes: the products whose input and output are both hidden layers (the hidden-to-hidden
// weights, forward and reverse) run on v_mfma_f32_16x16x32_bf16 with FP32 accumulation, 32 K per
// instruction.  Each lane takes 8 consecutive features of its atom's row (k = 32 c + 8 g + e) and
// the weights are packed with the same k order, so the products pair up whatever order the
// instruction uses inside its K chunk.  Split mode (FNET_BF16) writes each operand as
// hi + lo, hi = bf16(x) and lo = bf16(x - hi), and accumulates hi.hi + hi.lo + lo.hi: about 16
// mantissa bits, enough for the 1e-5 eV/atom and 1e-4 eV/A gates; single mode (FNET_BF16_FAST)
// takes hi.hi only (8 bits; its errors are reported, not gated).  The input layer (z-scored
// features, which can be ill-conditioned) and the output layer stay FP32.
#include <algorithm>
#include <type_traits>

#include "../../include/fnet_hip.h"
#include "fnet_device.hpp"

namespace fnet {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// every layer width is padded to a multiple of 32: output blocks are computed in pairs
__host__ __device__ __forceinline__ int r32(int d) { return (d + 31) & ~31; }

__device__ __forceinline__ float actf(int id, float x) {
  switch (id) {
    case 7: return expf(-(x * x));                                // gaussian
    case 4: return logf(1.0f + expf(x));                          // softplus
    case 5: return (sqrtf(x * x + 1.0f) - 1.0f) / 2.0f + x;       // bent identity
    case 2: return x > 0.0f ? x : 0.0f;                           // relu
    case 3: return (0.01f * x > x) ? 0.01f * x : x;               // leaky relu
    case 1: return 1.0f / (1.0f + expf(-x));                      // sigmoid
    case 8: return x > 0.0f ? 1.0f : 0.0f;                        // heaviside
    case 6: return atanf(x);                                      // atan
    case 9: return x;                                             // linear
    default: return tanhf(x);                                     // tanh
  }
}

__device__ __forceinline__ float actd(int id, float x) {
  switch (id) {
    case 7: return -2.0f * x * expf(-(x * x));
    case 4: return 1.0f / (1.0f + expf(-x));
    case 5: return x / (2.0f * sqrtf(x * x + 1.0f)) + 1.0f;
    case 2: return x >= 0.0f ? 1.0f : 0.0f;
    case 3: return x >= 0.0f ? 1.0f : 0.01f;
    case 1: {
      const float s = 1.0f / (1.0f + expf(-x));
      return s * (1.0f - s);
    }
    case 8: return 0.0f;
    case 6: return 1.0f / (x * x + 1.0f);
    case 9: return 1.0f;
    default: {
      const float t = tanhf(x);
      return 1.0f - t * t;
    }
  }
}

// f(x) and f'(x) together: tanh and sigmoid share their transcendental (the same values as actf
// and actd, bit for bit), the others are evaluated one after the other.
__device__ __forceinline__ void actfd(int id, float x, float& f, float& d) {
  if (id == 0) {
    const float t = tanhf(x);
    f = t;
    d = 1.0f - t * t;
  } else if (id == 1) {
    const float s = 1.0f / (1.0f + expf(-x));
    f = s;
    d = s * (1.0f - s);
  } else {
    f = actf(id, x);
    d = actd(id, x);
  }
}

// f'(x) of tanh and sigmoid from y = f(x), as actd forms it
__device__ __forceinline__ float actd_post(int id, float y) {
  return id == 0 ? 1.0f - y * y : y * (1.0f - y);
}

struct MfmaArgs {
  NetShape sh;
  const float* wpack;
  long long pk_stride;
  long long fw[kMaxLayers], rw[kMaxLayers], pb[kMaxLayers];
  // BF16 fragments of the hidden-to-hidden layers (hi, then lo at + bsz): forward and reverse
  const bf8* bpack;
  long long bk_stride;  // per species, in bf8 units
  long long bfw[kMaxLayers], brw[kMaxLayers], bsz[kMaxLayers];
  int fpoff[kMaxLayers];  // offset (floats) of f'(z) of hidden activation layer m in the wave's store
  const float* params_f;  // [nspecies][nparams] FP32 (last-layer columns of the reverse sweep)
  const double* G;        // [N][nG]
  const double* ext;
  int next;
  const int* ext_in;
  int nG, nout;
  const double* zmean;
  const double* zinv;
  const int* perm;
  const int* tile_sp;
  const int* tile_start;
  const int* tile_cnt;
  int first_tile;
  int ldx;        // row stride (floats) of the wave's activation rows
  int wave_floats;
  double* Eatom;  // [N][nout]
  double* cG;     // [N][nout][nG]
  int nsub;       // 16-atom parts of a tile (blocks per tile when the waves share them)
  int ntiles;     // blocks beyond the tiles' search mirror entries
  MirrorArgs mr;
  unsigned long long* stamp;
};

// Row stride and per-wave LDS (floats) for a network shape: 16 activation rows of the widest
// layer (+4 floats so that rows start on different banks) and the fragment slots of every hidden
// layer, which hold z, then f'(z), then the reverse-sweep delta of that layer.
void wave_lds(const NetShape& sh, int& ldx, int& wave_floats, int* fpoff) {
  int dmax = 0;
  for (int l = 0; l < sh.nl; ++l) dmax = std::max(dmax, r32(sh.dims[l]));
  ldx = dmax + 4;
  int fp = 0;
  for (int m = 0; m < kMaxLayers; ++m) fpoff[m] = 0;
  for (int m = 1; m < sh.nl - 1; ++m) {
    fpoff[m] = fp;
    fp += r32(sh.dims[m]) * 16;
  }
  wave_floats = 16 * ldx + fp;
}

// Two 16 x 16 output blocks (ob0, ob0 + 1) of Z^T = A . X^T over Kc 16-wide K chunks: A fragments
// from the packed operand Af (block stride Kc * 256 floats), X^T fragments from the wave's rows.
__device__ __forceinline__ void gemm_pair(const float* __restrict__ Af, int ob0, int Kc,
                                          const float* X, int ldx, int lane, int j, int g,
                                          f4& c0, f4& c1) {
  const float* A0 = Af + (long long)ob0 * Kc * 256 + lane;
  const float* A1 = A0 + (long long)Kc * 256;
  float n0[4], n1[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    n0[s] = A0[s * 64];
    n1[s] = A1[s * 64];
  }
#pragma unroll 1
  for (int c = 0; c < Kc; ++c) {
    const f4 xb = *(const f4*)(X + j * ldx + 16 * c + 4 * g);
    float u0[4], u1[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u0[s] = n0[s];
      u1[s] = n1[s];
    }
    if (c + 1 < Kc) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        n0[s] = A0[((c + 1) * 4 + s) * 64];
        n1[s] = A1[((c + 1) * 4 + s) * 64];
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(u0[s], xb[s], c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(u1[s], xb[s], c1, 0, 0, 0);
    }
  }
}

// One output block of the same product (the same sums in the same order): the fragments of four
// chunks are fetched before the first is used, since a block that runs alone has nothing else to
// hide their latency behind.
__device__ __forceinline__ void gemm_one(const float* __restrict__ Af, int ob, int Kc,
                                         const float* X, int ldx, int lane, int j, int g, f4& c0) {
  const float* A0 = Af + (long long)ob * Kc * 256 + lane;
  for (int c = 0; c < Kc; c += 4) {
    float u[4][4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int s = 0; s < 4; ++s) u[d][s] = c + d < Kc ? A0[((c + d) * 4 + s) * 64] : 0.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      if (c + d < Kc) {
        const f4 xb = *(const f4*)(X + j * ldx + 16 * (c + d) + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s)
          c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(u[d][s], xb[s], c0, 0, 0, 0);
      }
  }
}

// hi and lo BF16 parts of 8 FP32 values
__device__ __forceinline__ void split8(const f4& x0, const f4& x1, bf8& h, bf8& l) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const __bf16 a = (__bf16)x0[e], b = (__bf16)x1[e];
    h[e] = a;
    h[e + 4] = b;
    l[e] = (__bf16)(x0[e] - (float)a);
    l[e + 4] = (__bf16)(x1[e] - (float)b);
  }
}

// gemm_pair on the BF16 matrix cores: Kc32 chunks of 32; A fragments Ah (hi) and Ah + bsz (lo),
// block stride Kc32 * 64 bf8; BF = 3 split products, 1 the hi products only.
template <int BF>
__device__ __forceinline__ void gemm_pair_bf(const bf8* __restrict__ Ah, long long bsz, int ob0,
                                             int Kc32, const float* X, int ldx, int lane, int j,
                                             int g, f4& c0, f4& c1) {
  const bf8* A0 = Ah + (long long)ob0 * Kc32 * 64 + lane;
  const bf8* A1 = A0 + (long long)Kc32 * 64;
  bf8 na0 = A0[0], na1 = A1[0], nl0, nl1;
  if (BF == 3) {
    nl0 = A0[bsz];
    nl1 = A1[bsz];
  }
#pragma unroll 1
  for (int c = 0; c < Kc32; ++c) {
    const float* xr = X + j * ldx + 32 * c + 8 * g;
    const f4 x0 = *(const f4*)xr, x1 = *(const f4*)(xr + 4);
    bf8 xh, xl;
    split8(x0, x1, xh, xl);
    const bf8 a0 = na0, a1 = na1;
    bf8 l0, l1;
    if (BF == 3) {
      l0 = nl0;
      l1 = nl1;
    }
    if (c + 1 < Kc32) {
      na0 = A0[(c + 1) * 64];
      na1 = A1[(c + 1) * 64];
      if (BF == 3) {
        nl0 = A0[bsz + (c + 1) * 64];
        nl1 = A1[bsz + (c + 1) * 64];
      }
    }
    c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, xh, c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, xh, c1, 0, 0, 0);
    if (BF == 3) {
      c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, xl, c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, xl, c1, 0, 0, 0);
      c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l0, xh, c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l1, xh, c1, 0, 0, 0);
    }
  }
}

// ... and one block of it
template <int BF>
__device__ __forceinline__ void gemm_one_bf(const bf8* __restrict__ Ah, long long bsz, int ob,
                                            int Kc32, const float* X, int ldx, int lane, int j,
                                            int g, f4& c0) {
  const bf8* A0 = Ah + (long long)ob * Kc32 * 64 + lane;
  for (int c = 0; c < Kc32; c += 2) {
    bf8 a[2], lo[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
      if (c + d < Kc32) {
        a[d] = A0[(c + d) * 64];
        if (BF == 3) lo[d] = A0[bsz + (c + d) * 64];
      }
#pragma unroll
    for (int d = 0; d < 2; ++d)
      if (c + d < Kc32) {
        const float* xr = X + j * ldx + 32 * (c + d) + 8 * g;
        bf8 xh, xl;
        split8(*(const f4*)xr, *(const f4*)(xr + 4), xh, xl);
        c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d], xh, c0, 0, 0, 0);
        if (BF == 3) {
          c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d], xl, c0, 0, 0, 0);
          c0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo[d], xh, c0, 0, 0, 0);
        }
      }
  }
}

// layer l (ww(d_l, d_{l+1})) maps a hidden layer to a hidden layer
__device__ __forceinline__ bool hidden_hidden(int l, int nl) { return l >= 1 && l + 1 <= nl - 2; }

// SPLIT: the four waves of a block share 16 atoms, each taking every fourth output block, instead
// of running 16 atoms each through all of them: a batch that leaves most of the chip idle waits
// for one wave's chain of loads, products and activations, which this cuts to about a third.  The
// sums are the same either way.  kOwn: output blocks of a hidden layer that one wave holds in
// registers, both of a layer up to 32 wide or every fourth of one up to 64, 128 or kMaxDim.
template <bool GRADIN, int BF, bool SPLIT, int kOwn>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(kOwn > 2 ? 4 : !SPLIT && BF == 3 ? 5 : 6)))
    k_mlp_mfma(MfmaArgs a) {
  extern __shared__ __align__(16) float smf[];
  const int lane = threadIdx.x & 63;
  // a scalar, and with it the tile and its addresses (500 boxes' weight gradients, whole iteration
  // 308 -> 295 us)
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  stamp(a.stamp);
  if ((int)blockIdx.x >= a.ntiles) {
    mirror_centre(a.mr, (long long)((int)blockIdx.x - a.ntiles) * (blockDim.x >> 6) + w, lane);
    return;
  }
  // waves a layer's blocks (and an activation's rows) are dealt to, and this one's number
  const int nw = SPLIT ? 4 : 1, me = SPLIT ? w : 0;
  const int tile = a.first_tile + (SPLIT ? (int)blockIdx.x / a.nsub : (int)blockIdx.x);
  const int a0 = 16 * (SPLIT ? (int)blockIdx.x % a.nsub : w);
  const int sp = a.tile_sp[tile], start = a.tile_start[tile], cnt = a.tile_cnt[tile];
  if (a0 >= cnt) return;  // whole wave (SPLIT: whole block)
  auto sync = [] {
    if constexpr (SPLIT) __syncthreads();
    else wave_sync();
  };
  const int nv = min(16, cnt - a0);
  const int nl = a.sh.nl;
  const int act = a.sh.act[sp];
  const int ldx = a.ldx;
  float* X = smf + (SPLIT ? 0 : (size_t)w * a.wave_floats);
  float* FP = X + 16 * ldx;
  const float* WP = a.wpack + (long long)sp * a.pk_stride;
  const bool valid = j < nv;
  const long long atom = valid ? (long long)a.perm[start + a0 + j] : 0;

  // input rows: standardised features (and external features), zero beyond d0 and nv; 32 lanes to
  // a row's chunk
  const int d0 = a.sh.dims[0], K0 = r32(d0);
  {
    const int t = SPLIT ? (int)threadIdx.x : lane, kl = t & 31;
    for (int r = t >> 5; r < 16; r += 2 * nw) {
      const long long at = r < nv ? a.perm[start + a0 + r] : 0;
      for (int k = kl; k < K0; k += 32) {
        float v = 0.0f;
        if (r < nv && k < d0)
          v = k < a.nG ? (float)((a.G[at * a.nG + k] - a.zmean[k]) * a.zinv[k])
                       : (float)a.ext[at * a.next + a.ext_in[k - a.nG]];
        X[r * ldx + k] = v;
      }
    }
  }
  sync();

  // this wave's output blocks of a hidden layer: q -> block (q < kOwn)
  auto own = [&](int q) { return SPLIT ? me + 4 * q : q; };
  float* row = X + j * ldx + 4 * g;  // a fragment's place in the rows: row + 16 * block
  // products of a hidden layer's own blocks, added to c
  auto product = [&](const float* Wf, const bf8* Bf, long long bsz, bool bf, int Kc, int Nb,
                     f4 (&c)[kOwn]) {
    if constexpr (SPLIT) {
#pragma unroll
      for (int q = 0; q < kOwn; ++q)
        if (own(q) < Nb) {
          if (bf) gemm_one_bf<BF ? BF : 1>(Bf, bsz, own(q), Kc >> 1, X, ldx, lane, j, g, c[q]);
          else gemm_one(Wf, own(q), Kc, X, ldx, lane, j, g, c[q]);
          __builtin_amdgcn_sched_barrier(0);
        }
    } else {
      if (bf) gemm_pair_bf<BF>(Bf, bsz, 0, Kc >> 1, X, ldx, lane, j, g, c[0], c[1]);
      else gemm_pair(Wf, 0, Kc, X, ldx, lane, j, g, c[0], c[1]);
    }
  };

  // hidden layers: the pre-activations stay in registers until every wave has read the layer's
  // rows, then the next rows y = f(z) and, in fragment order, f'(z), 16 bytes at a time (through
  // LDS value by value before: 8192 parts of 32-128-128-1 176 -> 147 us, whole step of 131 072 Si
  // atoms 2049 -> 2034)
  for (int l = 0; l < nl - 2; ++l) {
    const int Kc = r32(a.sh.dims[l]) >> 4, Nb = r32(a.sh.dims[l + 1]) >> 4;
    const float* Bp = WP + a.pb[l];
    f4 c[kOwn];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
      if (own(q) < Nb) c[q] = *(const f4*)(Bp + 16 * own(q) + 4 * g);
    product(WP + a.fw[l], a.bpack + (long long)sp * a.bk_stride + a.bfw[l], a.bsz[l],
            BF && hidden_hidden(l, nl), Kc, Nb, c);
    sync();
    float* ds = FP + a.fpoff[l + 1];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
      if (own(q) < Nb) {
        f4 f, d;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float fr, dr;
          actfd(act, c[q][r], fr, dr);
          f[r] = fr;
          d[r] = dr;
        }
        *(f4*)(row + 16 * own(q)) = f;
        if (GRADIN) *(f4*)(ds + (own(q) * 64 + lane) * 4) = d;
        __builtin_amdgcn_sched_barrier(0);  // (blocks interleaved take registers that cost waves)
      }
    sync();
  }
  // linear output layer (nout <= 16: one block): lane group g holds outputs 4 g + r of atom j
  if (!SPLIT || w == 0) {
    const int l = nl - 2;
    f4 c = *(const f4*)(WP + a.pb[l] + 4 * g);
    gemm_one(WP + a.fw[l], 0, r32(a.sh.dims[l]) >> 4, X, ldx, lane, j, g, c);
    if (valid)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * g + r < a.nout) a.Eatom[atom * a.nout + 4 * g + r] = (double)c[r];
  }
  if (!GRADIN) return;
  sync();

  // reverse sweep of the single output (input gradient = row of the Jacobian)
  double* out = a.cG + atom * a.nG;
  int m = nl - 2;
  {
    // delta of activation layer m from the one-hot output: column 0 of ww(m), times f'(z_m)
    const int dm = a.sh.dims[m], Nb = r32(dm) >> 4;
    const float* col = a.params_f + (long long)sp * a.sh.nparams + a.sh.woff[m];
    if (m >= 1) {
      const float* ds = FP + a.fpoff[m];
#pragma unroll
      for (int q = 0; q < kOwn; ++q)
        if (own(q) < Nb) {
          f4 d = *(const f4*)(ds + (own(q) * 64 + lane) * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int k = 16 * own(q) + 4 * g + r;
            d[r] = (k < dm ? col[k] : 0.0f) * d[r];
          }
          *(f4*)(row + 16 * own(q)) = d;
        }
      sync();
    } else if (valid) {
      for (int k = 4 * g + 16 * me; k < a.nG; k += 16 * nw)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k + r < a.nG) out[k + r] = (double)col[k + r] * a.zinv[k + r];
    }
  }
  // delta_{m-1}^T = W_{m-1} . delta_m^T (rows in X), times f'(z_{m-1})
  for (; m >= 2; --m) {
    const int Nb = r32(a.sh.dims[m - 1]) >> 4, Kc = r32(a.sh.dims[m]) >> 4;
    f4 c[kOwn];
#pragma unroll
    for (int q = 0; q < kOwn; ++q) c[q] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    product(WP + a.rw[m - 1], a.bpack + (long long)sp * a.bk_stride + a.brw[m - 1], a.bsz[m - 1],
            BF && hidden_hidden(m - 1, nl), Kc, Nb, c);
    sync();
    const float* ds = FP + a.fpoff[m - 1];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
      if (own(q) < Nb)
        *(f4*)(row + 16 * own(q)) = c[q] * *(const f4*)(ds + (own(q) * 64 + lane) * 4);
    sync();
  }
  // input layer: the ACSF part of d out / d x feeds the force adjoint (FP64, z-score factor)
  if (m == 1) {
    const int Mb = K0 >> 4, Kc = r32(a.sh.dims[1]) >> 4;
    const float* Rf = WP + a.rw[0];
    auto write_in = [&](const f4& c, int ib) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int f = 16 * ib + 4 * g + r;
        if (valid && f < a.nG) out[f] = (double)c[r] * a.zinv[f];
      }
    };
    if constexpr (SPLIT) {
      for (int ib = me; ib < Mb; ib += nw) {
        f4 c0 = {0.0f, 0.0f, 0.0f, 0.0f};
        gemm_one(Rf, ib, Kc, X, ldx, lane, j, g, c0);
        write_in(c0, ib);
      }
    } else {
      for (int ib0 = 0; ib0 < Mb; ib0 += 2) {
        f4 c0 = {0.0f, 0.0f, 0.0f, 0.0f}, c1 = {0.0f, 0.0f, 0.0f, 0.0f};
        gemm_pair(Rf, ib0, Kc, X, ldx, lane, j, g, c0, c1);
        write_in(c0, ib0);
        write_in(c1, ib0 + 1);
      }
    }
  }
}

// ---- weight gradient (bprop, network.F90:248-296, with sysTrain's scaling, bpnn.F90:692-702) ----
// One block = nw waves = 16 nw atoms of one element (a tile of the MFMA layout, or a fixed part of
// one).  Forward: every wave runs its 16 atoms through the hidden layers as above, keeping each
// layer's pre-activation rows z_l (tanh and sigmoid: f(z_l)) for all atoms of the block in LDS (R[l];
// R[0] holds the input rows) and, for other activations, its own current values in Xw.  Backward,
// top layer first, with delta_out = the loss gradient of each atom (nout = 1):
//  * the output layer (rank one) on the vector unit: dW[0][k] = sum_at delta_out a_l[at][k],
//    delta_l = W[0][k] delta_out f'(z_l);
//  * every other layer l: dW_l[o][k] = sum_at delta_{l+1}[at][o] a_l[at][k] on the matrix cores
//    with the block's atoms as the K dimension (A = delta rows, B = a_l = f(z_l) rows; a wave
//    takes a k-block with up to 8 o-blocks, so each element is activated once per 8 o-blocks), the bias
//    gradient as a column sum in atom order, then delta_l = (W_l^T delta_{l+1}) f'(z_l) with the
//    reverse fragments, written over z_l.
// Products and sums over the block's atoms are FP32 (column sums over the atoms in four fixed
// quarters, then the quarters in order); the block writes its FP32 partial vector
// (gpart + block * nparams), which k_grad_chunks / k_grad_reduce add in FP64 in a fixed order.
struct GradArgs {
  const double* lossgrad;  // [N][nout]
  float* gpart;            // [blocks][nparams]
  int nsub;                // blocks per tile
  int roff[kMaxLayers];    // LDS offsets (floats) of R[l], l = 0 .. nl - 2
  int ld[kMaxLayers];      // their row strides
  int doff;                // delta_out [16 nw]
  int woff;                // Xw of wave 0 (16 rows of stride ldw per wave); after the forward,
                           // scratch of the column sums (4 r32(widest layer) floats)
  int ldw;
};

// out[k] (k < n) = sum over the block's TA atoms of v(at, k) = wt[at] M[at][k] (ACT: f(M)), in
// four quarters of the atoms, each in order, then ((q0 + q1) + (q2 + q3)).  Ends synchronised.
template <bool WT, bool ACT>
__device__ __forceinline__ void col_sums(const float* M, int ld, int n, int TA, const float* wt,
                                         int act, float* red, float* out_f) {
  const int qa = TA >> 2;
  for (int idx = threadIdx.x; idx < 4 * n; idx += blockDim.x) {
    const int q = idx / n, k = idx - q * n;
    float s = 0.0f;
    for (int at = q * qa; at < (q + 1) * qa; ++at) {
      float v = M[at * ld + k];
      if (ACT) v = actf(act, v);
      s += WT ? wt[at] * v : v;
    }
    red[idx] = s;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < n; k += blockDim.x)
    out_f[k] = (red[k] + red[n + k]) + (red[2 * n + k] + red[3 * n + k]);
  __syncthreads();
}

template <int BF>
__global__ void __launch_bounds__(256) k_mlp_grad_mfma(MfmaArgs a, GradArgs ga) {
  extern __shared__ __align__(16) float smf[];
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int TA = 16 * nw;
  const int t = a.first_tile + (int)blockIdx.x / ga.nsub, sub = (int)blockIdx.x % ga.nsub;
  const int sp = a.tile_sp[t];
  const int start = a.tile_start[t] + sub * TA;
  const int cnt = min(TA, a.tile_cnt[t] - sub * TA);  // may be <= 0: the partial is then zero
  const int nl = a.sh.nl;
  const int act = a.sh.act[sp];
  const float* WP = a.wpack + (long long)sp * a.pk_stride;
  float* gp = ga.gpart + (long long)blockIdx.x * a.sh.nparams;
  float* dout = smf + ga.doff;
  float* Xw = smf + ga.woff + w * 16 * ga.ldw;
  float* red = smf + ga.woff;
  const int a0 = 16 * w;

  // entries without gradient: the dummy output weights and the input layer's biases
  for (int k = threadIdx.x; k < a.sh.dims[nl - 1]; k += blockDim.x) gp[a.sh.woff[nl - 1] + k] = 0.0f;
  for (int k = threadIdx.x; k < a.sh.dims[0]; k += blockDim.x) gp[a.sh.boff[0] + k] = 0.0f;

  // tanh and sigmoid: their derivative follows from their value, so the rows R[l] of hidden layers
  // hold f(z_l), which every later step needs, and no value is formed twice (four times before, which
  // bound the kernel: 96 000 atoms of 32-25-25-1 82 -> 58 us)
  const bool post = act == 0 || act == 1;

  // input rows (own atoms) and delta_out; 32 lanes to a row's chunk
  {
    float* X0 = smf + ga.roff[0] + a0 * ga.ld[0];
    const int d0 = a.sh.dims[0], K0 = r32(d0);
    for (int r = lane >> 5; r < 16; r += 2) {
      const bool in = a0 + r < cnt;
      const long long at = in ? a.perm[start + a0 + r] : 0;
      for (int k = lane & 31; k < K0; k += 32) {
        float v = 0.0f;
        if (in && k < d0)
          v = k < a.nG ? (float)((a.G[at * a.nG + k] - a.zmean[k]) * a.zinv[k])
                       : (float)a.ext[at * a.next + a.ext_in[k - a.nG]];
        X0[r * ga.ld[0] + k] = v;
      }
    }
    if (lane < 16)
      dout[a0 + lane] =
          a0 + lane < cnt ? (float)ga.lossgrad[(long long)a.perm[start + a0 + lane] * a.nout] : 0.0f;
  }
  wave_sync();

  // forward through the hidden layers: z_{l+1} rows into R[l+1], f(z_{l+1}) into Xw
  for (int l = 0; l + 2 < nl; ++l) {
    const int Kc = r32(a.sh.dims[l]) >> 4, Nb = r32(a.sh.dims[l + 1]) >> 4;
    const bool rows = l == 0 || post;
    const float* Xin = rows ? smf + ga.roff[l] + a0 * ga.ld[l] : Xw;
    const int ldin = rows ? ga.ld[l] : ga.ldw;
    const int ldz = ga.ld[l + 1];
    float* Z = smf + ga.roff[l + 1] + a0 * ldz;
    const float* Bp = WP + a.pb[l];
    const bool bf = BF && hidden_hidden(l, nl);
    for (int ob0 = 0; ob0 < Nb; ob0 += 2) {
      f4 c0 = *(const f4*)(Bp + 16 * ob0 + 4 * g);
      f4 c1 = *(const f4*)(Bp + 16 * ob0 + 16 + 4 * g);
      if (bf)
        gemm_pair_bf<BF>(a.bpack + (long long)sp * a.bk_stride + a.bfw[l], a.bsz[l], ob0, Kc >> 1,
                         Xin, ldin, lane, j, g, c0, c1);
      else
        gemm_pair(WP + a.fw[l], ob0, Kc, Xin, ldin, lane, j, g, c0, c1);
      if (post)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          c0[r] = actf(act, c0[r]);
          c1[r] = actf(act, c1[r]);
        }
      *(f4*)(Z + j * ldz + 16 * ob0 + 4 * g) = c0;
      *(f4*)(Z + j * ldz + 16 * ob0 + 16 + 4 * g) = c1;
    }
    wave_sync();
    if (post) continue;
    const int W = 16 * Nb;
    for (int idx = lane; idx < 16 * W; idx += 64) {
      const int r = idx / W, k = idx - r * W;
      Xw[r * ga.ldw + k] = actf(act, Z[r * ldz + k]);
    }
    wave_sync();
  }
  __syncthreads();  // the backward reads every wave's rows

  // output layer (one output): dW[0][k], the bias, and delta of the last hidden layer
  {
    const int l = nl - 2, dl = a.sh.dims[l], ldl = ga.ld[l];
    float* Z = smf + ga.roff[l];
    if (l == 0 || post) col_sums<true, false>(Z, ldl, dl, TA, dout, act, red, gp + a.sh.woff[l]);
    else col_sums<true, true>(Z, ldl, dl, TA, dout, act, red, gp + a.sh.woff[l]);
    col_sums<false, false>(dout, 1, 1, TA, nullptr, act, red, gp + a.sh.boff[nl - 1]);
    if (l >= 1) {
      const float* col = a.params_f + (long long)sp * a.sh.nparams + a.sh.woff[l];
      for (int idx = threadIdx.x; idx < TA * dl; idx += blockDim.x) {
        const int at = idx / dl, k = idx - at * dl;
        float* zp = Z + at * ldl + k;
        *zp = col[k] * dout[at] * (post ? actd_post(act, *zp) : actd(act, *zp));
      }
      __syncthreads();
    }
  }

  // the other layers, top down: R[l + 1] holds delta_{l+1}, R[l] holds z_l (x for l = 0)
  for (int l = nl - 3; l >= 0; --l) {
    const int dl = a.sh.dims[l], dn = a.sh.dims[l + 1];
    const int Kb = r32(dl) >> 4, Ob = r32(dn) >> 4;
    const int ldl = ga.ld[l], ldn = ga.ld[l + 1];
    float* Zl = smf + ga.roff[l];
    const float* Dn = smf + ga.roff[l + 1];
    // work items (k-block, group of up to 8 o-blocks); groups narrower than 8 when there are
    // fewer k-blocks than waves (the input layer), so that every wave has one
    const int gob = Kb >= nw ? 8 : max(1, min(8, (Ob * Kb) / nw));
    const int ngr = (Ob + gob - 1) / gob;
    for (int it = w; it < Kb * ngr; it += nw) {
      const int kb = it / ngr;
      {
        const int ob0 = (it - kb * ngr) * gob, ob1 = min(Ob, ob0 + gob);
        f4 c[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) c[q] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int s4 = 0; s4 < TA; s4 += 4) {
          const int at = s4 + g;
          const float z = Zl[at * ldl + 16 * kb + j];
          const float bv = l == 0 || post ? z : actf(act, z);
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (ob0 + q < ob1)
              c[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(Dn[at * ldn + 16 * (ob0 + q) + j], bv,
                                                          c[q], 0, 0, 0);
        }
        const int k = 16 * kb + j;
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (ob0 + q < ob1)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int o = 16 * (ob0 + q) + 4 * g + r;
              if (o < dn && k < dl) gp[a.sh.woff[l] + (long long)o * dl + k] = c[q][r];
            }
      }
    }
    col_sums<false, false>(Dn, ldn, dn, TA, nullptr, act, red, gp + a.sh.boff[l + 1]);
    if (l == 0) break;
    // delta_l = (W_l^T delta_{l+1}) f'(z_l), own atoms, over z_l
    const int Mb = Kb, Kc = Ob;
    const bool bf = BF && hidden_hidden(l, nl);
    float* zr = Zl + (a0 + j) * ldl;
    for (int ib0 = 0; ib0 < Mb; ib0 += 2) {
      f4 c0 = {0.0f, 0.0f, 0.0f, 0.0f}, c1 = {0.0f, 0.0f, 0.0f, 0.0f};
      if (bf)
        gemm_pair_bf<BF>(a.bpack + (long long)sp * a.bk_stride + a.brw[l], a.bsz[l], ib0, Kc >> 1,
                         Dn + a0 * ldn, ldn, lane, j, g, c0, c1);
      else
        gemm_pair(WP + a.rw[l], ib0, Kc, Dn + a0 * ldn, ldn, lane, j, g, c0, c1);
      f4* z0 = (f4*)(zr + 16 * ib0 + 4 * g);
      f4* z1 = (f4*)(zr + 16 * ib0 + 16 + 4 * g);
      f4 v0 = *z0, v1 = *z1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v0[r] = c0[r] * (post ? actd_post(act, v0[r]) : actd(act, v0[r]));
        v1[r] = c1[r] * (post ? actd_post(act, v1[r]) : actd(act, v1[r]));
      }
      *z0 = v0;
      *z1 = v1;
    }
    __syncthreads();
  }
}

}  // namespace

int mlp_mfma_waves(const NetShape& sh) {
  // single-output networks (the energy), layer widths up to kMaxDim
  if (sh.nl < 2 || sh.dims[sh.nl - 1] != 1) return 0;
  for (int l = 0; l < sh.nl; ++l)
    if (sh.dims[l] < 1 || sh.dims[l] > kMaxDim) return 0;
  int ldx, wf, fpoff[kMaxLayers];
  wave_lds(sh, ldx, wf, fpoff);
  int waves = 4;
  while (waves > 1 && (size_t)waves * wf * sizeof(float) > 64 * 1024) waves >>= 1;
  if ((size_t)waves * wf * sizeof(float) > 64 * 1024) return 0;
  return waves;
}

void mfma_layout(DevModel& m, size_t* floats, size_t* halves) {
  const NetShape& sh = m.shape;
  long long o = 0;
  for (int l = 0; l + 1 < sh.nl; ++l) {
    const long long sz = (long long)r32(sh.dims[l]) * r32(sh.dims[l + 1]);
    m.pk_fw[l] = o;
    o += sz;
    m.pk_rw[l] = o;
    o += sz;
    m.pk_b[l] = o;
    o += r32(sh.dims[l + 1]);
  }
  m.pk_stride = (o + 63) & ~63LL;
  *floats = (size_t)m.pk_stride * m.nspecies;
  // BF16 fragments of the hidden-to-hidden layers (none for networks with one hidden layer)
  long long h = 0;
  for (int l = 0; l < kMaxLayers; ++l) m.bk_fw[l] = m.bk_rw[l] = m.bk_sz[l] = 0;
  for (int l = 1; l + 2 < sh.nl; ++l) {
    const long long sz = (long long)r32(sh.dims[l]) * r32(sh.dims[l + 1]) / 8;
    m.bk_sz[l] = sz;
    m.bk_fw[l] = h;
    h += 2 * sz;
    m.bk_rw[l] = h;
    h += 2 * sz;
  }
  m.bk_stride = h;
  *halves = (size_t)(h * 8 * m.nspecies);
}

namespace {

// float -> bf16 bits, round to nearest even (finite values)
__device__ __forceinline__ uint16_t to_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

struct PackArgs {
  NetShape sh;
  int nspecies;
  const double* params;
  float* params_f;
  float* wpack;  // null: no matrix-core networks
  uint16_t* bpack;
  long long pk_stride, bk_stride;
  long long fw[kMaxLayers], rw[kMaxLayers], pb[kMaxLayers];
  long long bfw[kMaxLayers], brw[kMaxLayers], bsz[kMaxLayers];
};

// The FP32 copy of the parameters and the MFMA fragments of every species, one thread per value:
// after a parameter update nothing has to come to the host to be packed.
//
// A-operand fragments of FP32 layers, every width padded to a multiple of 32 with zeros.  Forward
// fragment of layer l: index ((ob * Kc + c) * 4 + s) * 64 + lane, lane = 16 g + i, holds
// ww_l(k = 16 c + 4 g + s, o = 16 ob + i); reverse fragment: ((ib * Oc + c) * 4 + s) * 64 + lane
// holds ww_l(k = 16 ib + i, o = 16 c + 4 g + s); then the layer's biases.
//
// BF16 fragments (hi, then lo = bf16(w - hi)) of the hidden-to-hidden layers for
// v_mfma_f32_16x16x32_bf16.  Forward: element ((ob * Kc32 + c) * 64 + lane) * 8 + e holds
// ww_l(k = 32 c + 8 g + e, o = 16 ob + i); reverse: ((ib * Oc32 + c) * 64 + lane) * 8 + e holds
// ww_l(k = 16 ib + i, o = 32 c + 8 g + e).  Offsets and sizes are in units of 8 values.
__global__ void __launch_bounds__(256) k_model_params(PackArgs a) {
  long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long np = a.sh.nparams * a.nspecies;
  if (q < np) {
    a.params_f[q] = (float)a.params[q];
    return;
  }
  q -= np;
  if (!a.wpack) return;
  const bool half = q >= a.pk_stride * a.nspecies;
  if (half) q -= a.pk_stride * a.nspecies;
  const long long stride = half ? 8 * a.bk_stride : a.pk_stride;
  if (stride == 0 || q >= stride * a.nspecies) return;
  const long long sp = q / stride, e = q - sp * stride;
  const double* P = a.params + sp * a.sh.nparams;
  float w = 0.0f;
  bool lo = false;
  for (int l = 0; l + 1 < a.sh.nl; ++l) {
    const int din = a.sh.dims[l], dout = a.sh.dims[l + 1];
    const long long sz = (long long)r32(din) * r32(dout);
    int k = -1, o = -1;
    if (half) {
      if (a.bsz[l] == 0) continue;
      const long long tf = e - 8 * a.bfw[l], tr = e - 8 * a.brw[l];
      const bool fwd = tf >= 0 && tf < 2 * sz, rev = tr >= 0 && tr < 2 * sz;
      if (!fwd && !rev) continue;
      long long t = fwd ? tf : tr;
      lo = t >= sz;
      if (lo) t -= sz;
      const int u = (int)(t & 7), lane = (int)(t >> 3) & 63, g = lane >> 4, i = lane & 15;
      const int nc = r32(fwd ? din : dout) >> 5, blk = (int)(t >> 9);
      const int ob = blk / nc, c = blk - ob * nc;
      k = fwd ? 32 * c + 8 * g + u : 16 * ob + i;
      o = fwd ? 16 * ob + i : 32 * c + 8 * g + u;
    } else {
      const long long tf = e - a.fw[l], tr = e - a.rw[l], tb = e - a.pb[l];
      if (tb >= 0 && tb < r32(dout)) {
        if (tb < dout) w = (float)P[a.sh.boff[l + 1] + tb];
        break;
      }
      const bool fwd = tf >= 0 && tf < sz, rev = tr >= 0 && tr < sz;
      if (!fwd && !rev) continue;
      const long long t = fwd ? tf : tr;
      const int lane = (int)t & 63, g = lane >> 4, i = lane & 15, s = (int)(t >> 6) & 3;
      const int nc = r32(fwd ? din : dout) >> 4, blk = (int)(t >> 8);
      const int ob = blk / nc, c = blk - ob * nc;
      k = fwd ? 16 * c + 4 * g + s : 16 * ob + i;
      o = fwd ? 16 * ob + i : 16 * c + 4 * g + s;
    }
    if (k < din && o < dout) w = (float)P[a.sh.woff[l] + (long long)o * din + k];
    break;
  }
  if (!half) {
    a.wpack[q] = w;
  } else {
    const uint16_t h = to_bf16(w);
    a.bpack[q] = lo ? to_bf16(w - __uint_as_float((uint32_t)h << 16)) : h;
  }
}

}  // namespace

hipError_t launch_model_params(const DevModel& m, hipStream_t s) {
  PackArgs a;
  a.sh = m.shape;
  a.nspecies = m.nspecies;
  a.params = m.params;
  a.params_f = m.params_f;
  a.wpack = m.wpack;
  a.bpack = m.bpack;
  a.pk_stride = m.pk_stride;
  a.bk_stride = m.bk_stride;
  for (int l = 0; l < kMaxLayers; ++l) {
    a.fw[l] = m.pk_fw[l];
    a.rw[l] = m.pk_rw[l];
    a.pb[l] = m.pk_b[l];
    a.bfw[l] = m.bk_fw[l];
    a.brw[l] = m.bk_rw[l];
    a.bsz[l] = m.bk_sz[l];
  }
  long long n = m.shape.nparams;
  if (m.wpack) n += m.pk_stride + 8 * m.bk_stride;
  n *= m.nspecies;
  if (n <= 0) return hipSuccess;
  k_model_params<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(a);
  return hipGetLastError();
}

namespace {
// Waves per weight-gradient block (the largest divisor of the tile's waves whose LDS fits 64 KiB),
// with the LDS layout of k_mlp_grad_mfma; 0 when the network has no MFMA tiles.
int mlp_grad_waves(const NetShape& sh, int tile_waves, GradArgs* ga, size_t* bytes) {
  if (tile_waves <= 0) return 0;
  for (int nw = tile_waves; nw >= 1; nw >>= 1) {
    if (tile_waves % nw) continue;
    const int TA = 16 * nw;
    GradArgs q{};
    int f = 0;
    for (int l = 0; l + 1 < sh.nl; ++l) {
      q.ld[l] = r32(sh.dims[l]) + 4;
      q.roff[l] = f;
      f += TA * q.ld[l];
    }
    q.doff = f;
    f += TA;
    q.ldw = 0;
    int wmax = 0;
    for (int l = 0; l < sh.nl; ++l) wmax = std::max(wmax, r32(sh.dims[l]));
    for (int l = 1; l + 1 < sh.nl; ++l) q.ldw = std::max(q.ldw, r32(sh.dims[l]) + 4);
    q.woff = f;
    f += std::max(nw * 16 * q.ldw, 4 * wmax);
    const size_t b = (size_t)f * sizeof(float);
    if (b <= 64 * 1024) {
      q.nsub = tile_waves / nw;
      if (ga) *ga = q;
      if (bytes) *bytes = b;
      return nw;
    }
  }
  return 0;
}
}  // namespace

// Weight-gradient blocks per MFMA tile (0: the network has no MFMA path)
int mlp_grad_subtiles(const NetShape& sh, int tile_waves) {
  GradArgs ga;
  return mlp_grad_waves(sh, tile_waves, &ga, nullptr) ? ga.nsub : 0;
}

hipError_t launch_mlp_grad_mfma(fnet_batch* b, const DevModel& m, hipStream_t s) {
  GradArgs ga;
  size_t lds = 0;
  const int nw = mlp_grad_waves(m.shape, b->mtile_waves, &ga, &lds);
  if (nw == 0) return hipErrorInvalidConfiguration;
  if (b->nmtiles <= 0) return hipSuccess;
  MfmaArgs a{};
  a.sh = m.shape;
  a.wpack = m.wpack;
  a.pk_stride = m.pk_stride;
  for (int l = 0; l < kMaxLayers; ++l) {
    a.fw[l] = m.pk_fw[l];
    a.rw[l] = m.pk_rw[l];
    a.pb[l] = m.pk_b[l];
    a.bfw[l] = m.bk_fw[l];
    a.brw[l] = m.bk_rw[l];
    a.bsz[l] = m.bk_sz[l];
  }
  a.params_f = m.params_f;
  a.G = (const double*)b->G;
  a.ext = b->ext;
  a.next = b->next;
  a.ext_in = m.ext_in;
  a.nG = m.nG;
  a.nout = m.nout;
  a.zmean = m.zmean;
  a.zinv = m.zinv;
  a.perm = b->perm;
  a.tile_sp = b->mtile_sp;
  a.tile_start = b->mtile_start;
  a.tile_cnt = b->mtile_cnt;
  a.first_tile = 0;
  a.bpack = (const bf8*)m.bpack;
  a.bk_stride = m.bk_stride;
  ga.lossgrad = b->lossgrad;
  ga.gpart = (float*)b->gpart;
  const int bf = (b->precision == FNET_BF16 && m.bpack) ? 3
               : (b->precision == FNET_BF16_FAST && m.bpack) ? 1 : 0;
  const dim3 grid((unsigned)((long long)b->nmtiles * ga.nsub)), block(64 * nw);
  if (bf == 3) k_mlp_grad_mfma<3><<<grid, block, lds, s>>>(a, ga);
  else if (bf == 1) k_mlp_grad_mfma<1><<<grid, block, lds, s>>>(a, ga);
  else k_mlp_grad_mfma<0><<<grid, block, lds, s>>>(a, ga);
  return hipGetLastError();
}

// 16-atom parts up to which the waves of a block share one (SPLIT): 1132 parts 26.2 -> 24.7 us,
// 2400 parts 27.1 -> 26.2 us; beyond that every CU has its fill of the other kind (6000 parts of
// 32-32-32: 26.7 -> 33 us).  Networks wider than 32, or whose rows and f'(z) let fewer than four waves
// of their own into 64 KB, share at every size: the other kind has few waves on a CU there (7700
// parts of 24-64-64-1: 123 -> 101 us; 8192 of 32-128-128-1 in split BF16: 294 -> 178 us).
constexpr long long kSplitTiles = 2560;

hipError_t launch_mlp_mfma(fnet_batch* b, const DevModel& m, int first_tile, int ntiles,
                           int want_grad_in, hipStream_t s, bool mirror,
                           unsigned long long* stamp) {
  if (ntiles <= 0) return hipSuccess;
  MfmaArgs a;
  a.sh = m.shape;
  a.wpack = m.wpack;
  a.pk_stride = m.pk_stride;
  for (int l = 0; l < kMaxLayers; ++l) {
    a.fw[l] = m.pk_fw[l];
    a.rw[l] = m.pk_rw[l];
    a.pb[l] = m.pk_b[l];
  }
  wave_lds(m.shape, a.ldx, a.wave_floats, a.fpoff);
  a.params_f = m.params_f;
  a.G = (const double*)b->G;
  a.ext = b->ext;
  a.next = b->next;
  a.ext_in = m.ext_in;
  a.nG = m.nG;
  a.nout = m.nout;
  a.zmean = m.zmean;
  a.zinv = m.zinv;
  a.perm = b->perm;
  a.tile_sp = b->mtile_sp;
  a.tile_start = b->mtile_start;
  a.tile_cnt = b->mtile_cnt;
  a.first_tile = first_tile;
  a.Eatom = b->Eatom;
  a.cG = (double*)b->cG;
  a.bpack = (const bf8*)m.bpack;
  a.bk_stride = m.bk_stride;
  for (int l = 0; l < kMaxLayers; ++l) {
    a.bfw[l] = m.bk_fw[l];
    a.brw[l] = m.bk_rw[l];
    a.bsz[l] = m.bk_sz[l];
  }
  const int bf = (b->precision == FNET_BF16 && m.bpack) ? 3
               : (b->precision == FNET_BF16_FAST && m.bpack) ? 1 : 0;
  const int waves = b->mtile_waves;
  a.nsub = waves;
  a.mr = mirror_args(b, 0, b->N);
  a.stamp = stamp;
  bool split = (long long)ntiles * waves <= kSplitTiles ||
               4 * a.wave_floats * sizeof(float) > 64 * 1024;
  int width = 0;  // of the widest hidden layer
  for (int l = 1; l + 1 < m.shape.nl; ++l) width = std::max(width, m.shape.dims[l]);
  split = split || width > 32;
  if (!want_grad_in) a.wave_floats = 16 * a.ldx;  // no f'(z) to keep
  const int bw = split ? 4 : waves;  // waves per block
  a.ntiles = split ? ntiles * waves : ntiles;
  const size_t lds = (size_t)(split ? 1 : waves) * a.wave_floats * sizeof(float);
  const dim3 grid((unsigned)(a.ntiles + (mirror ? (b->N + bw - 1) / bw : 0))), block(64 * bw);
  auto run = [&](void (*kern)(MfmaArgs)) { kern<<<grid, block, lds, s>>>(a); };
  auto go = [&](auto gradin, auto bfc) {
    constexpr bool G = decltype(gradin)::value;
    constexpr int B = decltype(bfc)::value;
    if (!split) run(k_mlp_mfma<G, B, false, 2>);
    else if (width <= 64) run(k_mlp_mfma<G, B, true, 1>);
    else if (width <= 128) run(k_mlp_mfma<G, B, true, 2>);
    else run(k_mlp_mfma<G, B, true, 4>);
  };
  auto mode = [&](auto gradin) {
    if (bf == 3) go(gradin, std::integral_constant<int, 3>());
    else if (bf == 1) go(gradin, std::integral_constant<int, 1>());
    else go(gradin, std::integral_constant<int, 0>());
  };
  if (want_grad_in) mode(std::true_type());
  else mode(std::false_type());
  return hipGetLastError();
}

}  // namespace fnet
