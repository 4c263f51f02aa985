// FP64 element networks on the matrix cores of gfx950 (v_mfma_f64_16x16x4_f64): forward, input
// gradient and weight gradient (the mathematics of fnet_mlp.hip, whose kernels keep the networks
// too wide for a block's LDS).
//
// A block of four waves takes 16 atoms of one element through the layers as
//   Z^T [d_out x 16] = W^T [d_out x d_in] . X^T [d_in x 16],
// each wave every fourth block of 16 outputs, the activation rows in LDS.  The scalar kernel gave
// one thread per (atom, output) a dot product of dependent loads from LDS and memory; on the few
// thousand atoms of an FP64 batch its 64-atom tiles also left most of the chip idle (16 water boxes:
// forward 41 -> 14 us, with input gradient 56 -> 22; 100 Si64 cells: weight gradient 38 -> 20 us).
// Operands:
// A lane 16 g + i = W(o = 16 ob + i, k = 4 s + g), read from the serialised parameters (a few KB,
// cached) four steps ahead, B lane 16 g + j = X[atom j][4 s + g]; register r of the result is
// output 16 ob + g + 4 r of atom j.  Rows are d + 2 doubles apart, which puts the 32 lanes of a read
// phase on different banks.
#include <algorithm>

#include "fnet_device.hpp"

namespace fnet {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ int r16(int d) { return (d + 15) & ~15; }

__device__ __forceinline__ double actf(int id, double x) {
  switch (id) {
    case 7: return exp(-(x * x));
    case 4: return log(1.0 + exp(x));
    case 5: return (sqrt(x * x + 1.0) - 1.0) / 2.0 + x;
    case 2: return x > 0.0 ? x : 0.0;
    case 3: return (0.01 * x > x) ? 0.01 * x : x;
    case 1: return 1.0 / (1.0 + exp(-x));
    case 8: return x > 0.0 ? 1.0 : 0.0;
    case 6: return atan(x);
    case 9: return x;
    default: return tanh(x);
  }
}

// f'(x) with y = f(x)
__device__ __forceinline__ double actd(int id, double x, double y) {
  switch (id) {
    case 7: return -2.0 * x * y;
    case 4: return 1.0 / (1.0 + exp(-x));
    case 5: return x / (2.0 * sqrt(x * x + 1.0)) + 1.0;
    case 2: return x >= 0.0 ? 1.0 : 0.0;
    case 3: return x >= 0.0 ? 1.0 : 0.01;
    case 1: return y * (1.0 - y);
    case 8: return 0.0;
    case 6: return 1.0 / (x * x + 1.0);
    case 9: return 1.0;
    default: return 1.0 - y * y;
  }
}

struct F64Args {
  NetShape sh;
  const double* params;
  const double* G;
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
  int nsub;    // 16-atom parts of a tile
  int aoff[kMaxLayers];  // LDS offsets (doubles): rows of layer l (weight gradient: all of them)
  int fpoff[kMaxLayers]; // f'(z) of hidden layer l, [r16(d_l)][16]
  int doff[2];           // two buffers of rows: activations / deltas in turn
  int ld;                // row stride of those (widest layer + 2)
  double* Eatom;
  double* cG;
  const double* lossgrad;
  double* gpart;         // [tiles][nparams]
  int nblocks;           // blocks beyond these search mirror entries
  MirrorArgs mr;
  unsigned long long* stamp;
};

// One block of 16 rows of M . X^T: M(i, k) = P[i * si + k * sk] for i < ni, k < nk (zero beyond), X
// rows of stride ld; four steps of K at a time, their M values fetched together.
__device__ __forceinline__ void gemm16(const double* __restrict__ P, long long si, long long sk,
                                       int ni, int nk, const double* X, int ld, int g, int j,
                                       d4& c) {
  const bool in = j < ni;
  for (int k0 = 0; k0 < nk; k0 += 16) {
    double m[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * s + g;
      m[s] = in && k < nk ? P[j * si + k * sk] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      c = __builtin_amdgcn_mfma_f64_16x16x4f64(m[s], X[j * ld + k0 + 4 * s + g], c, 0, 0, 0);
  }
}

// Input rows of 16 atoms (standardised features, external features; zero beyond d0 and nv).
__device__ __forceinline__ void input_rows(const F64Args& a, double* X, int ld, int start, int nv) {
  const int d0 = a.sh.dims[0], K0 = r16(d0);
  for (int idx = threadIdx.x; idx < 16 * K0; idx += 256) {
    const int r = idx / K0, k = idx - r * K0;
    double v = 0.0;
    if (r < nv && k < d0) {
      const long long at = a.perm[start + r];
      v = k < a.nG ? (a.G[at * a.nG + k] - a.zmean[k]) * a.zinv[k]
                   : a.ext[at * a.next + a.ext_in[k - a.nG]];
    }
    X[r * ld + k] = v;
  }
}

// Forward of 16 atoms; rows(l) gives layer l's row buffer and stride.  Hidden layers' f'(z) go to
// their slots when FP; the outputs are handed to out(o, atom j, value) by wave 0.
template <bool FP, typename Rows, typename Out>
__device__ __forceinline__ void forward16(const F64Args& a, const double* P, int act, double* sm,
                                          Rows rows, Out out) {
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nl = a.sh.nl;
  for (int l = 0; l < nl - 1; ++l) {
    const int din = a.sh.dims[l], dout = a.sh.dims[l + 1];
    const bool hidden = l < nl - 2;
    int ldi, ldo;
    const double* X = rows(l, ldi);
    double* Y = hidden ? rows(l + 1, ldo) : nullptr;
    const double* W = P + a.sh.woff[l];
    const double* b = P + a.sh.boff[l + 1];
    for (int ob = w; 16 * ob < dout; ob += 4) {
      d4 c = {0.0, 0.0, 0.0, 0.0};
      gemm16(W + 16LL * ob * din, din, 1, dout - 16 * ob, din, X, ldi, g, j, c);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = 16 * ob + g + 4 * r;
        const double z = c[r] + (o < dout ? b[o] : 0.0);
        if (!hidden) {
          if (o < dout) out(o, j, z);
        } else {
          const double y = o < dout ? actf(act, z) : 0.0;
          Y[j * ldo + o] = y;
          if (FP) sm[a.fpoff[l + 1] + 16 * o + j] = o < dout ? actd(act, z, y) : 0.0;
        }
      }
    }
    __syncthreads();
  }
}

// d[at][k] = (sum_o W(o, k) delta[at][o]) f'(z) for hidden layer l (rows D of stride a.ld into Y), or
// handed to in(k, atom j, value) for the input layer.
template <typename In>
__device__ __forceinline__ void reverse16(const F64Args& a, const double* P, int l, double* sm,
                                          const double* D, double* Y, int w, int g, int j, In in) {
  const int din = a.sh.dims[l], dout = a.sh.dims[l + 1];
  for (int ib = w; 16 * ib < din; ib += 4) {
    d4 c = {0.0, 0.0, 0.0, 0.0};
    gemm16(P + a.sh.woff[l] + 16 * ib, 1, din, din - 16 * ib, dout, D, a.ld, g, j, c);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = 16 * ib + g + 4 * r;
      if (l >= 1) Y[j * a.ld + k] = k < din ? c[r] * sm[a.fpoff[l] + 16 * k + j] : 0.0;
      else if (k < din) in(k, j, c[r]);
    }
  }
  __syncthreads();
}

template <bool GRADIN>
__global__ void __launch_bounds__(256) k_mlp_f64(F64Args a) {
  extern __shared__ __align__(16) double sm[];
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  stamp(a.stamp);
  if ((int)blockIdx.x >= a.nblocks) {
    mirror_centre(a.mr, (long long)((int)blockIdx.x - a.nblocks) * 4 + w, lane);
    return;
  }
  const int tile = a.first_tile + (int)blockIdx.x / a.nsub, a0 = 16 * ((int)blockIdx.x % a.nsub);
  const int sp = a.tile_sp[tile], start = a.tile_start[tile] + a0, nv = min(16, a.tile_cnt[tile] - a0);
  if (nv <= 0) return;
  const int nl = a.sh.nl, act = a.sh.act[sp];
  const double* P = a.params + (long long)sp * a.sh.nparams;
  const long long atom = j < nv ? (long long)a.perm[start + j] : -1;
  input_rows(a, sm + a.doff[0], a.ld, start, nv);
  __syncthreads();
  auto rows = [&](int l, int& ld) {
    ld = a.ld;
    return sm + a.doff[l & 1];
  };
  forward16<GRADIN>(a, P, act, sm, rows, [&](int o, int, double v) {
    if (atom >= 0) a.Eatom[atom * a.nout + o] = v;
  });
  if (!GRADIN) return;
  // reverse sweep of every output: the input gradient (row of the Jacobian)
  const int m = nl - 2;
  for (int t = 0; t < a.nout; ++t) {
    auto in = [&](int k, int, double v) {
      if (atom >= 0 && k < a.nG) a.cG[(atom * a.nout + t) * a.nG + k] = v * a.zinv[k];
    };
    const int dm = a.sh.dims[m];
    const double* row = P + a.sh.woff[m] + (long long)t * dm;
    if (m == 0) {
      for (int k = 4 * w + g; k < dm; k += 16) in(k, j, row[k]);
      continue;
    }
    double* D = sm + a.doff[m & 1];
    for (int k = 4 * w + g; k < r16(dm); k += 16)
      D[j * a.ld + k] = k < dm ? row[k] * sm[a.fpoff[m] + 16 * k + j] : 0.0;
    __syncthreads();
    for (int l = m - 1; l >= 0; --l)
      reverse16(a, P, l, sm, sm + a.doff[(l + 1) & 1], sm + a.doff[l & 1], w, g, j, in);
  }
}

// Weight gradient of one tile (bprop, network.F90:248-296, with sysTrain's scaling,
// bpnn.F90:692-702), 16 atoms at a time, into the tile's partial vector: dW(o, k) = sum over atoms
// of delta[o] a[k] with the atoms as the K dimension of the products.  The first 16 atoms write the
// partial, the others add to it, each value always by the same thread.
__global__ void __launch_bounds__(256) k_mlp_grad_f64(F64Args a) {
  extern __shared__ __align__(16) double sm[];
  const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = blockIdx.x;
  const int sp = a.tile_sp[tile], cnt = a.tile_cnt[tile];
  const int nl = a.sh.nl, act = a.sh.act[sp];
  const double* P = a.params + (long long)sp * a.sh.nparams;
  double* gp = a.gpart + (long long)tile * a.sh.nparams;
  // entries without gradient: the dummy output weights and the input layer's biases
  for (int k = threadIdx.x; k < a.sh.dims[nl - 1]; k += 256) gp[a.sh.woff[nl - 1] + k] = 0.0;
  for (int k = threadIdx.x; k < a.sh.dims[0]; k += 256) gp[a.sh.boff[0] + k] = 0.0;
  auto rows = [&](int l, int& ld) {
    ld = r16(a.sh.dims[l]) + 2;
    return sm + a.aoff[l];
  };
  for (int a0 = 0; a0 < cnt; a0 += 16) {
    const int start = a.tile_start[tile] + a0, nv = min(16, cnt - a0);
    const bool first = a0 == 0;
    int ld0;
    double* X0 = rows(0, ld0);
    input_rows(a, X0, ld0, start, nv);
    // delta of the (linear) output layer
    for (int q = threadIdx.x; q < 16 * 16; q += 256) {
      const int at = q >> 4, o = q & 15;
      sm[a.doff[(nl - 1) & 1] + at * a.ld + o] =
          at < nv && o < a.nout ? a.lossgrad[(long long)a.perm[start + at] * a.nout + o] : 0.0;
    }
    __syncthreads();
    // the outputs themselves are not needed: hidden layers only
    forward16<true>(a, P, act, sm, rows, [](int, int, double) {});
    for (int l = nl - 2; l >= 0; --l) {
      const int dl = a.sh.dims[l], dn = a.sh.dims[l + 1];
      const double* D = sm + a.doff[(l + 1) & 1];
      int ldl;
      const double* A = rows(l, ldl);
      const int Kb = (dl + 15) >> 4, Ob = (dn + 15) >> 4;
      for (int q = w; q < Kb * Ob; q += 4) {
        const int ob = q / Kb, kb = q - ob * Kb;
        d4 c = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s)
          c = __builtin_amdgcn_mfma_f64_16x16x4f64(D[(4 * s + g) * a.ld + 16 * ob + j],
                                                   A[(4 * s + g) * ldl + 16 * kb + j], c, 0, 0, 0);
        const int k = 16 * kb + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int o = 16 * ob + g + 4 * r;
          if (o < dn && k < dl) {
            double* p = gp + a.sh.woff[l] + (long long)o * dl + k;
            *p = first ? c[r] : *p + c[r];
          }
        }
      }
      for (int o = threadIdx.x; o < dn; o += 256) {
        double s = 0.0;
#pragma unroll
        for (int at = 0; at < 16; ++at) s += D[at * a.ld + o];
        double* p = gp + a.sh.boff[l + 1] + o;
        *p = first ? s : *p + s;
      }
      if (l >= 1)
        reverse16(a, P, l, sm, D, sm + a.doff[l & 1], w, g, j, [](int, int, double) {});
    }
    __syncthreads();
  }
}

// LDS layout: the two row buffers, f'(z) of the hidden layers, and (grad) the rows of every layer.
size_t layout(const NetShape& sh, bool grad, F64Args* out) {
  int wide = 16;
  for (int l = 0; l < sh.nl; ++l) wide = std::max(wide, r16(sh.dims[l]));
  F64Args a{};
  a.ld = wide + 2;
  int o = 0;
  for (int q = 0; q < 2; ++q) {
    a.doff[q] = o;
    o += 16 * a.ld;
  }
  for (int l = 1; l < sh.nl - 1; ++l) {
    a.fpoff[l] = o;
    o += 16 * r16(sh.dims[l]);
  }
  if (grad)
    for (int l = 0; l < sh.nl - 1; ++l) {
      a.aoff[l] = o;
      o += 16 * (r16(sh.dims[l]) + 2);
    }
  if (out)
    for (int l = 0; l < kMaxLayers; ++l) {
      out->aoff[l] = a.aoff[l];
      out->fpoff[l] = a.fpoff[l];
      out->doff[0] = a.doff[0];
      out->doff[1] = a.doff[1];
      out->ld = a.ld;
    }
  return sizeof(double) * (size_t)o;
}

F64Args make_args(const fnet_batch* b, const DevModel& m) {
  F64Args a{};
  a.sh = m.shape;
  a.params = m.params;
  a.G = (const double*)b->G;
  a.ext = b->ext;
  a.next = b->next;
  a.ext_in = m.ext_in;
  a.nG = m.nG;
  a.nout = m.nout;
  a.zmean = m.zmean;
  a.zinv = m.zinv;
  a.perm = b->perm;
  a.tile_sp = b->tile_sp;
  a.tile_start = b->tile_start;
  a.tile_cnt = b->tile_cnt;
  a.nsub = b->tile_atoms / 16;
  a.Eatom = b->Eatom;
  a.cG = (double*)b->cG;
  a.lossgrad = b->lossgrad;
  a.gpart = b->gpart;
  return a;
}

// One block's LDS (of the CU's 160 KB): hidden layers of 128 take 104 KB with the weight gradient.
constexpr size_t kF64Lds = 150 * 1024;
// Tiles (weight-gradient blocks) a batch is cut into: two for each CU.
constexpr long long kF64Tiles = 512;

}  // namespace

int mlp_f64_tile_atoms(const fnet_batch* b, const NetShape& sh) {
  if (layout(sh, true, nullptr) > std::min<size_t>(kF64Lds, b->ctx->lds_block)) return 0;
  const long long parts = (b->N + 15) / 16;
  return 16 * (int)std::max<long long>(1, std::min<long long>(64, (parts + kF64Tiles - 1) / kF64Tiles));
}

hipError_t launch_mlp_f64(fnet_batch* b, const DevModel& m, int first_tile, int ntiles,
                          int want_grad_in, hipStream_t s, bool mirror,
                          unsigned long long* stamp) {
  if (ntiles <= 0) return hipSuccess;
  F64Args a = make_args(b, m);
  const size_t lds = layout(m.shape, false, &a);
  a.first_tile = first_tile;
  a.nblocks = ntiles * a.nsub;
  a.mr = mirror_args(b, 0, b->N);
  a.stamp = stamp;
  const unsigned grid = a.nblocks + (mirror ? (unsigned)((b->N + 3) / 4) : 0u);
  if (want_grad_in) k_mlp_f64<true><<<grid, 256, lds, s>>>(a);
  else k_mlp_f64<false><<<grid, 256, lds, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_mlp_grad_f64(fnet_batch* b, const DevModel& m, hipStream_t s) {
  if (b->ntiles <= 0) return hipSuccess;
  F64Args a = make_args(b, m);
  const size_t lds = layout(m.shape, true, &a);
  k_mlp_grad_f64<<<b->ntiles, 256, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace fnet
