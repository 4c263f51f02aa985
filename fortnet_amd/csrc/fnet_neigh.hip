// Periodic neighbour lists for gfx950: one wavefront per centre atom, candidates tested 64 at a
// time in the reference's entry order and compacted with a ballot prefix count, so the CSR rows
// come out in exactly the order of dynneighlist.F90:233-320 without any sort.
//
// The distance test is the reference's FP64 arithmetic with FMA contraction disabled:
//   neighCoords = coords0(:,j) + latVecs . n          (dynneighlist.F90:291, latpointiter order)
//   dist2 = sum((coordsAtom1 - neighCoords)**2) <= cutoff**2   (dynneighlist.F90:292-294)
// so the set of (centre, neighbour, image) entries is bit-identical to the reference's.
//
// Whole lattice images are skipped when no atom of the structure can reach the centre from
// them: |row_a(inv L) . dr| <= rc |row_a(inv L)| bounds every fractional offset of a neighbour,
// so an image n with n_a outside [s_a(i) - smax_a - w_a, s_a(i) - smin_a + w_a] holds none; and
// an image whose translated Cartesian bounding box of the atoms lies farther than rc from the
// centre holds none either (on cubic cells this drops the corner images of the first test's
// box of images, ~10 % of the candidates on the Si cells).  The exact test still decides every
// candidate that is looked at.
#include <algorithm>

#include "fnet_device.hpp"

namespace fnet {
namespace {

// q / d for 0 <= q, d < 2^31 through the FP64 reciprocal rd = 1 / d: the estimate is within one of
// the quotient, and one correction step makes it exact (no integer division sequence)
__device__ __forceinline__ int udiv(int q, int d, double rd) {
  int a = (int)((double)q * rd);
  const long long r = (long long)q - (long long)a * d;
  a += r >= d ? 1 : (r < 0 ? -1 : 0);
  return a;
}

__device__ __forceinline__ unsigned long long lanemask_lt(int lane) {
  return (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
}

// Inverse lattice and image ranges, mirroring simplealgebra.F90:41-62,90-125 and
// latpointiter.F90:226-253 (extension 1, dynneighlist.F90:223-224).
__device__ void lattice_setup(const double* L, double rc, StructInfo& si) {
#pragma clang fp contract(off)
#define O(r, c) L[((c) - 1) * 3 + ((r) - 1)]
  double det = O(1, 1) * (O(2, 2) * O(3, 3) - O(3, 2) * O(2, 3));
  det = det - O(1, 2) * (O(2, 1) * O(3, 3) - O(3, 1) * O(2, 3));
  det = det + O(1, 3) * (O(2, 1) * O(3, 2) - O(3, 1) * O(2, 2));
  double* I = si.inv;
#define IV(r, c) I[((c) - 1) * 3 + ((r) - 1)]
  IV(1, 1) = -O(2, 3) * O(3, 2) + O(2, 2) * O(3, 3);
  IV(2, 1) = O(2, 3) * O(3, 1) - O(2, 1) * O(3, 3);
  IV(3, 1) = -O(2, 2) * O(3, 1) + O(2, 1) * O(3, 2);
  IV(1, 2) = O(1, 3) * O(3, 2) - O(1, 2) * O(3, 3);
  IV(2, 2) = -O(1, 3) * O(3, 1) + O(1, 1) * O(3, 3);
  IV(3, 2) = O(1, 2) * O(3, 1) - O(1, 1) * O(3, 2);
  IV(1, 3) = -O(1, 3) * O(2, 2) + O(1, 2) * O(2, 3);
  IV(2, 3) = O(1, 3) * O(2, 1) - O(1, 1) * O(2, 3);
  IV(3, 3) = -O(1, 2) * O(2, 1) + O(1, 1) * O(2, 2);
#undef IV
#undef O
  for (int q = 0; q < 9; ++q) I[q] = I[q] / det;
  for (int a = 0; a < 3; ++a) {
    double s = 0.0;
    for (int c = 0; c < 3; ++c) {
      double v = I[c * 3 + a];
      s = s + v * v;
    }
    double nrm = sqrt(s);
    int t = (int)floor(rc * nrm);
    si.lo[a] = -(t + 1);
    si.hi[a] = t + 1;
    si.w[a] = rc * nrm;
  }
}

// One block per structure: lattice set-up by thread 0, then the extent of the fractional
// coordinates (it only serves the image pruning of the direct search) or, for a structure with
// cell lists that fits one block (bin_lds), its bins: an LDS histogram, its prefix sums and the
// scatter, in place of seven launches over all atoms (24 ternary cells of 16 - 4096 atoms: eight
// launches and 99 us -> one of 13 us).  Block 0 clears the row maximum that the search raises.
struct PrepArgs {
  const double* xyz;
  const double* lat;
  const int* periodic;
  const long long* off;
  double rc;
  const int4* cellinfo;
  StructInfo* sinfo;
  const int* cell_off;
  int* cell_start;
  int* cell_atoms;
  int4* atom_m;
  int bin_lds;
  int* maxnb;
  unsigned long long* stamp;
};

__global__ void __launch_bounds__(1024) k_struct_prep(PrepArgs a) {
  extern __shared__ int hist[];  // [bin_lds]
  __shared__ StructInfo si;
  __shared__ double red[2][6][16];
  __shared__ int wsum[16];
  const int s = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  stamp(a.stamp);
  if (s == 0 && tid == 0) *a.maxnb = 0;
  if (tid == 0) {
    si.periodic = a.periodic[s];
    if (si.periodic) {
      lattice_setup(a.lat + 9 * s, a.rc, si);
    } else {
      for (int q = 0; q < 9; ++q) si.inv[q] = 0.0;
      for (int c = 0; c < 3; ++c) {
        si.lo[c] = 0;
        si.hi[c] = -1;
        si.w[c] = 0.0;
      }
    }
  }
  const long long a0 = a.off[s], a1 = a.off[s + 1];
  const int4 ci = a.cellinfo[s];
  const bool bin = ci.w && a.bin_lds > 0;
  const int nbins = bin ? ci.x * ci.y * ci.z : 0;
  for (int q = tid; q < nbins; q += blockDim.x) hist[q] = 0;
  __syncthreads();
  if (bin) {
    for (long long i = a0 + tid; i < a1; i += blockDim.x) {
      const int4 m = bin_of(si, a.xyz + 3 * i, ci);
      a.atom_m[i] = m;
      atomicAdd(&hist[m.w], 1);
    }
    __syncthreads();
    // exclusive prefix sums: each thread a run of bins, then the threads' totals
    const int per = (nbins + blockDim.x - 1) / blockDim.x;
    const int q0 = min(tid * per, nbins), q1 = min(q0 + per, nbins);
    int sum = 0;
    for (int q = q0; q < q1; ++q) sum += hist[q];
    int x = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int before = x - sum;
    for (int w = 0; w < wave; ++w) before += wsum[w];
    int* start = a.cell_start + a.cell_off[s];
    for (int q = q0; q < q1; ++q) {
      const int c = hist[q];
      start[q] = (int)a0 + before;
      hist[q] = before;
      before += c;
    }
    if (tid == 0) start[nbins] = (int)a1;
    __syncthreads();
    for (long long i = a0 + tid; i < a1; i += blockDim.x)
      a.cell_atoms[a0 + atomicAdd(&hist[a.atom_m[i].w], 1)] = (int)i;
  }
  // fractional extent (c = 0..2) and Cartesian bounding box (c = 3..5)
  double mn[6], mx[6];
  for (int c = 0; c < 6; ++c) {
    mn[c] = 1e300;
    mx[c] = -1e300;
  }
  const bool ext = si.periodic && !ci.w;
  if (ext) {
    for (long long i = a0 + tid; i < a1; i += blockDim.x) {
      const double x = a.xyz[3 * i], y = a.xyz[3 * i + 1], z = a.xyz[3 * i + 2];
      for (int c = 0; c < 3; ++c) {
        const double f = si.inv[0 * 3 + c] * x + si.inv[1 * 3 + c] * y + si.inv[2 * 3 + c] * z;
        mn[c] = fmin(mn[c], f);
        mx[c] = fmax(mx[c], f);
      }
      mn[3] = fmin(mn[3], x);
      mx[3] = fmax(mx[3], x);
      mn[4] = fmin(mn[4], y);
      mx[4] = fmax(mx[4], y);
      mn[5] = fmin(mn[5], z);
      mx[5] = fmax(mx[5], z);
    }
    for (int c = 0; c < 6; ++c) {
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) {
        mn[c] = fmin(mn[c], __shfl_xor(mn[c], o, 64));
        mx[c] = fmax(mx[c], __shfl_xor(mx[c], o, 64));
      }
      if (lane == 0) {
        red[0][c][wave] = mn[c];
        red[1][c][wave] = mx[c];
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    for (int c = 0; c < 6; ++c)
      for (int w = 0; ext && w < nw; ++w) {
        mn[c] = fmin(mn[c], red[0][c][w]);
        mx[c] = fmax(mx[c], red[1][c][w]);
      }
    for (int c = 0; c < 3; ++c) {
      si.smin[c] = mn[c];
      si.smax[c] = mx[c];
      si.bmin[c] = mn[c + 3];
      si.bmax[c] = mx[c + 3];
    }
    a.sinfo[s] = si;
  }
}

// Candidate test in the reference's arithmetic.  Returns the squared distance through d2.
__device__ __forceinline__ bool near_test(double ci0, double ci1, double ci2, const double* X,
                                          int j, double c0, double c1, double c2, double rc2,
                                          double& nd0, double& nd1, double& nd2, double& d2) {
#pragma clang fp contract(off)
  const double nc0 = X[3 * j] + c0, nc1 = X[3 * j + 1] + c1, nc2 = X[3 * j + 2] + c2;
  const double e0 = ci0 - nc0, e1 = ci1 - nc1, e2 = ci2 - nc2;
  double s = e0 * e0;
  s = s + e1 * e1;
  s = s + e2 * e2;
  nd0 = -e0;
  nd1 = -e1;
  nd2 = -e2;
  d2 = s;
  return s <= rc2;
}

// MODE: kCount writes the row lengths; kFill writes the rows at their CSR offsets; kPadded
// writes row i at i * cap (entries past cap dropped) and its full length, in one pass.
enum { kCount = 0, kFill = 1, kPadded = 2 };

// Bound by the tests of its candidates (FP64, a few dozen instructions for each 64 of them).  The
// wave's number is taken as a scalar, so that the atom, its structure and the image ranges are
// scalars too: 80 -> 46 registers, 8 waves to a SIMD instead of 6 (123 000 atoms of 8-512-atom Si
// cells 328 -> 259 us, 38 400 water atoms 125 -> 103 us).  Its vector units are busy
// all the time then; the strided loads of the coordinates do not bound it (a copy by component: no
// gain).
//
// SPLIT: the four waves of a block share one atom, each testing every fourth 64 of its candidates;
// a barrier per step exchanges their hit counts, so the row's order stays.  A small batch waits
// for one atom's serial walk over its candidates (192 water atoms 13.6 -> 9.2 us, 209 atoms of a
// request 13.6 -> 8.2 us).
template <int MODE, typename V, bool SPLIT = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6)))
    k_neigh(const double* __restrict__ xyz, const long long* __restrict__ off,
            const int* __restrict__ atom_struct, const StructInfo* __restrict__ sinfo,
            const double* __restrict__ lat, double rc, long long a0, long long a1,
            int* __restrict__ cnt, const int* __restrict__ rowptr,
            int* __restrict__ nj, int* __restrict__ nimg, V* __restrict__ nd,
            const int4* __restrict__ cellinfo, int cap, int* __restrict__ mir,
            int* __restrict__ maxnb, unsigned long long* __restrict__ t_end) {
  // nimg receives each entry's key (image + 1) n + (j - i) mod n; padded rows also set each
  // entry's mirror slot to -1 (no mirror) when mir is given, for the mirror search to fill in
#pragma clang fp contract(off)
  constexpr bool WRITE = MODE != kCount;
  const int lane = threadIdx.x & 63;
  // (the wave's number as a scalar: everything of the atom and its structure then is one too)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = SPLIT ? wave : 0;  // this wave's turn in a step of 64 kW candidates
  constexpr int kW = SPLIT ? 4 : 1;
  const long long i = a0 + (SPLIT ? (long long)blockIdx.x : (long long)blockIdx.x * 4 + wave);
  if (i >= a1) return;
  const int s = atom_struct[i];
  if (cellinfo[s].w) return;  // structure handled by the cell-list kernels
  const long long o = off[s];
  const int n = (int)(off[s + 1] - o);
  const int li = (int)(i - o);
  const double* X = xyz + 3 * o;
  const double ci0 = X[3 * li], ci1 = X[3 * li + 1], ci2 = X[3 * li + 2];
  const double rc2 = rc * rc;
  const long long base = MODE == kFill ? rowptr[i] : (MODE == kPadded ? i * cap : 0);
  int count = 0;

  __shared__ double4 tab[4][64];  // per wave: translation L . n (x, y, z), image index (w)
  double4* tw = tab[wave];
  auto order = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // key of an entry: (image + 1) n + (j - i) mod n, which increases along the row (the image
  // index is key / n - 1); the force gather's mirror search reads it
  auto put = [&](int q, int j, int key, double nd0, double nd1, double nd2, double d2) {
    if (MODE == kPadded && q >= cap) return;
    const long long pos = base + q;
    nj[pos] = (int)(o + j);
    nimg[pos] = key;
    V v;
    v.x = nd0;
    v.y = nd1;
    v.z = nd2;
    entry_d2(v, d2);
    nd[pos] = v;
    if (MODE == kPadded && mir) mir[pos] = -1;
  };
  // QUEUE: the hits wait in a ring of (t, slot of tab or -1: central cell) until 64 of them, or a
  // table of images, are complete; they are then tested once more for their vectors and written
  // one to a lane.  A step of 64 candidates has a few hits, whose write would cost all lanes half
  // as much as the test (123 000 atoms of 8-512-atom Si cells 259 -> 235 us, 38 400 water atoms
  // 103 -> 91 us).
  constexpr bool QUEUE = WRITE && !SPLIT;
  __shared__ int2 ring[QUEUE ? 4 : 1][QUEUE ? 128 : 1];
  int2* rw = ring[QUEUE ? wave : 0];
  int head = 0;  // hits so far; count of them are written
  auto flush = [&](int nf) {
    order();
    if (lane < nf) {
      const int2 h = rw[(count + lane) & 127];
      double4 c = make_double4(0.0, 0.0, 0.0, -1.0);
      if (h.y >= 0) c = tw[h.y];
      int j = li + h.x;
      if (j >= n) j -= n;
      double nd0, nd1, nd2, d2;
      near_test(ci0, ci1, ci2, X, j, c.x, c.y, c.z, rc2, nd0, nd1, nd2, d2);
      put(count + lane, j, ((int)c.w + 1) * n + h.x, nd0, nd1, nd2, d2);
    }
    count += nf;
    order();
  };
  __shared__ int hits[2][4];  // SPLIT: the waves' hits of this step and the one before
  int par = 0;
  auto emit = [&](bool hit, int j, int t, int slot, int img, double nd0, double nd1, double nd2,
                  double d2) {
    const unsigned long long mask = __ballot(hit);
    int before = 0, all = __popcll(mask);
    if constexpr (QUEUE) {
      if (hit) rw[(head + __popcll(mask & lanemask_lt(lane))) & 127] = make_int2(t, slot);
      head += all;
      if (head - count >= 64) flush(64);
      return;
    }
    if constexpr (SPLIT) {
      if (lane == 0) hits[par][w] = all;
      __syncthreads();
      all = 0;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int h = hits[par][v];
        before += v < w ? h : 0;
        all += h;
      }
      par ^= 1;
    }
    if (WRITE && hit)
      put(count + before + __popcll(mask & lanemask_lt(lane)), j, (img + 1) * n + t, nd0, nd1, nd2,
          d2);
    count += all;
  };

  // central cell: j = i+1 .. n-1, 0 .. i-1
  for (int t0 = 1; t0 < n; t0 += 64 * kW) {
    const int t = t0 + 64 * w + lane;
    int j = li + t;
    if (j >= n) j -= n;
    double nd0 = 0, nd1 = 0, nd2 = 0, d2 = 0;
    bool hit = false;
    if (t < n) hit = near_test(ci0, ci1, ci2, X, j, 0.0, 0.0, 0.0, rc2, nd0, nd1, nd2, d2);
    emit(hit, j, t, -1, -1, nd0, nd1, nd2, d2);
  }
  const StructInfo& si = sinfo[s];
  if (si.periodic) {
    // Lattice images in the reference's lexicographic order (third index fastest, origin
    // skipped), 64 at a time: the ones that can hold a neighbour are compacted in order into an
    // LDS table with their translation, then the (image, atom) pairs of the table are tested as
    // one list, 64 per step, so small cells (n << 64) still fill the wave.
    const double* L = lat + 9 * s;
    double sf[3];
    for (int a = 0; a < 3; ++a)
      sf[a] = si.inv[0 * 3 + a] * ci0 + si.inv[1 * 3 + a] * ci1 + si.inv[2 * 3 + a] * ci2;
    double wlo[3], whi[3];
    for (int a = 0; a < 3; ++a) {
      const double m = 1e-8 * (1.0 + fabs(sf[a]) + fabs(si.smin[a]) + fabs(si.smax[a]) + si.w[a]);
      wlo[a] = sf[a] - si.smax[a] - si.w[a] - m;
      whi[a] = sf[a] - si.smin[a] + si.w[a] + m;
    }
    const int m1 = si.hi[0] - si.lo[0] + 1, m2 = si.hi[1] - si.lo[1] + 1,
              m3 = si.hi[2] - si.lo[2] + 1;
    const int nq = m1 * m2 * m3;
    const int m23 = m2 * m3;
    const double rm23 = 1.0 / (double)m23, rm3 = 1.0 / (double)m3;
    const int qorig = ((0 - si.lo[0]) * m2 + (0 - si.lo[1])) * m3 + (0 - si.lo[2]);
    const int qs = 64 * kW / n, rs = 64 * kW % n;
    for (int q0 = 0; q0 < nq; q0 += 64) {
      const int q = q0 + lane;
      bool keep = false;
      double4 tv = make_double4(0.0, 0.0, 0.0, 0.0);
      if (q < nq && q != qorig) {
        // q = ((p1 - lo0) m2 + (p2 - lo1)) m3 + (p3 - lo2)
        const int a1 = udiv(q, m23, rm23), rem = q - a1 * m23, a2 = udiv(rem, m3, rm3);
        const int p1 = si.lo[0] + a1, p2 = si.lo[1] + a2, p3 = si.lo[2] + (rem - a2 * m3);
        keep = !(p1 < wlo[0] || p1 > whi[0] || p2 < wlo[1] || p2 > whi[1] || p3 < wlo[2] ||
                 p3 > whi[2]);
        const double pv0 = (double)p1, pv1 = (double)p2, pv2 = (double)p3;
        double cv[3];
        for (int r = 0; r < 3; ++r) {
          double acc = 0.0;
          acc = acc + L[0 * 3 + r] * pv0;
          acc = acc + L[1 * 3 + r] * pv1;
          acc = acc + L[2 * 3 + r] * pv2;
          cv[r] = acc;
        }
        // distance from the centre to the image's box of atoms; the margin covers the
        // rounding of this estimate against the exact test's
        const double ci[3] = {ci0, ci1, ci2};
        double q2 = 0.0;
        for (int r = 0; r < 3; ++r) {
          const double g = fmax(0.0, fmax(si.bmin[r] + cv[r] - ci[r], ci[r] - si.bmax[r] - cv[r]));
          q2 += g * g;
        }
        keep = keep && q2 <= rc2 * (1.0 + 1e-9) + 1e-12;
        tv = make_double4(cv[0], cv[1], cv[2], (double)(q > qorig ? q - 1 : q));
      }
      const unsigned long long km = __ballot(keep);
      if (QUEUE && head != count) flush(head - count);  // (their images are still in the table)
      if (keep) tw[__popcll(km & lanemask_lt(lane))] = tv;
      order();
      // flat index u = slot n + t over the kept images, t = 0 .. n - 1 from the centre on
      const int tot = __popcll(km) * n;
      int slot = (64 * w + lane) / n, t = (64 * w + lane) % n;
      for (int u0 = 64 * w; u0 - 64 * w < tot; u0 += 64 * kW) {
        double nd0 = 0, nd1 = 0, nd2 = 0, d2 = 0;
        bool hit = false;
        int j = 0, img = 0;
        if (u0 + lane < tot) {
          const double4 c = tw[slot];
          j = li + t;
          if (j >= n) j -= n;
          img = (int)c.w;
          hit = near_test(ci0, ci1, ci2, X, j, c.x, c.y, c.z, rc2, nd0, nd1, nd2, d2);
        }
        emit(hit, j, t, slot, img, nd0, nd1, nd2, d2);
        slot += qs;
        t += rs;
        if (t >= n) {
          t -= n;
          slot += 1;
        }
      }
      order();
    }
  }
  if (QUEUE && head != count) flush(head - count);
  if (MODE != kFill && lane == 0 && w == 0) cnt[i] = count;
  if (MODE == kPadded && lane == 0 && w == 0) {
    raise_max(maxnb, count);
    if (blockIdx.x == gridDim.x - 1) stamp_now(t_end);
  }
}

// Copies the padded rows (cap entries per atom) to their CSR offsets.
template <typename V>
__global__ void __launch_bounds__(256)
    k_compact_rows(long long n, int cap, const int* __restrict__ cnt,
                   const int* __restrict__ rowptr, const int* __restrict__ pnj,
                   const int* __restrict__ pnimg, const V* __restrict__ pnd,
                   int* __restrict__ nj, int* __restrict__ nimg, V* __restrict__ nd) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long i = t / cap;
  const int e = (int)(t - i * cap);
  if (i >= n || e >= cnt[i]) return;
  const long long src = t, dst = (long long)rowptr[i] + e;
  nj[dst] = pnj[src];
  nimg[dst] = pnimg[src];
  nd[dst] = pnd[src];
}

// ---- exclusive scan of the per-atom counts -------------------------------------------------
constexpr int kScanBlock = 1024;

__global__ void __launch_bounds__(kScanBlock) k_scan_block(const int* __restrict__ in,
                                                          int* __restrict__ out, long long n,
                                                          int* __restrict__ totals,
                                                          int* __restrict__ bmax) {
  __shared__ int buf[kScanBlock];
  __shared__ int wmax[kScanBlock / 64];
  const long long g = (long long)blockIdx.x * kScanBlock + threadIdx.x;
  const int v = (g < n) ? in[g] : 0;
  if (bmax) {
    int m = v;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  }
  buf[threadIdx.x] = v;
  __syncthreads();
  if (bmax && threadIdx.x == 0) {
    int m = wmax[0];
    for (int w = 1; w < kScanBlock / 64; ++w) m = max(m, wmax[w]);
    bmax[blockIdx.x] = m;
  }
  for (int st = 1; st < kScanBlock; st <<= 1) {
    int add = (threadIdx.x >= st) ? buf[threadIdx.x - st] : 0;
    __syncthreads();
    buf[threadIdx.x] += add;
    __syncthreads();
  }
  if (g < n) out[g] = buf[threadIdx.x] - v;
  if (threadIdx.x == kScanBlock - 1) totals[blockIdx.x] = buf[threadIdx.x];
}

__global__ void __launch_bounds__(kScanBlock) k_scan_totals(int* __restrict__ totals,
                                                           long long nb, int* __restrict__ last,
                                                           const int* __restrict__ bmax,
                                                           int* __restrict__ maxout) {
  __shared__ int buf[kScanBlock];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  if (maxout && threadIdx.x == 0) {
    int m = 0;
    for (long long b = 0; b < nb; ++b) m = max(m, bmax[b]);
    *maxout = m;
  }
  __syncthreads();
  for (long long b0 = 0; b0 < nb; b0 += kScanBlock) {
    const long long g = b0 + threadIdx.x;
    const int v = (g < nb) ? totals[g] : 0;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int st = 1; st < kScanBlock; st <<= 1) {
      int add = (threadIdx.x >= st) ? buf[threadIdx.x - st] : 0;
      __syncthreads();
      buf[threadIdx.x] += add;
      __syncthreads();
    }
    if (g < nb) totals[g] = carry + buf[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 0) carry += buf[kScanBlock - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) *last = carry;
}

__global__ void k_scan_add(int* __restrict__ out, long long n, const int* __restrict__ totals) {
  const long long g = (long long)blockIdx.x * kScanBlock + threadIdx.x;
  if (g < n) out[g] += totals[blockIdx.x];
}

}  // namespace

// scratch of launch_scan: block totals (nb + 1) and block maxima (nb)
long long scan_tmp_size(long long n) { return 2 * ((n + kScanBlock - 1) / kScanBlock) + 1; }

// Exclusive scan of cnt[0..n) into rowptr[0..n] (rowptr[n] = total); with maxout, also the
// largest count (the reduction rides on the scan's own pass over the counts).
hipError_t launch_scan(int* cnt, int* rowptr, long long n, int* tmp, hipStream_t s,
                       int* maxout) {
  const long long nb = (n + kScanBlock - 1) / kScanBlock;
  if (nb == 0) {
    FNET_HIP_TRY(hipMemsetAsync(rowptr, 0, sizeof(int), s));
    if (maxout) FNET_HIP_TRY(hipMemsetAsync(maxout, 0, sizeof(int), s));
    return hipSuccess;
  }
  int* bmax = maxout ? tmp + nb + 1 : nullptr;
  k_scan_block<<<(unsigned)nb, kScanBlock, 0, s>>>(cnt, rowptr, n, tmp, bmax);
  k_scan_totals<<<1, kScanBlock, 0, s>>>(tmp, nb, rowptr + n, bmax, maxout);
  k_scan_add<<<(unsigned)nb, kScanBlock, 0, s>>>(rowptr, n, tmp);
  return hipGetLastError();
}

hipError_t launch_struct_prep(fnet_batch* b, double rc, hipStream_t s, unsigned long long* stamp) {
  if (b->S == 0) return hipSuccess;
  PrepArgs a;
  a.xyz = b->xyz;
  a.lat = b->lat;
  a.periodic = b->periodic;
  a.off = b->off;
  a.rc = rc;
  a.cellinfo = b->cellinfo;
  a.sinfo = b->sinfo;
  a.cell_off = b->cell_off;
  a.cell_start = b->cell_start;
  a.cell_atoms = b->cell_atoms;
  a.atom_m = b->atom_m;
  a.bin_lds = b->bin_lds;
  a.maxnb = b->d_maxnb;
  a.stamp = stamp;
  // wide blocks only where they bin a structure
  k_struct_prep<<<b->S, b->bin_lds ? 1024 : 256, sizeof(int) * b->bin_lds, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_neigh_count(fnet_batch* b, double rc, long long a0, long long a1,
                              hipStream_t s) {
  const long long n = a1 - a0;
  if (n <= 0 || b->n_cell_struct == b->S) return hipSuccess;
  const unsigned grid = (unsigned)((n + 3) / 4);
  k_neigh<kCount, double4><<<grid, 256, 0, s>>>(b->xyz, b->off, b->atom_struct, b->sinfo,
                                                 b->lat, rc, a0, a1, b->cnt, nullptr, nullptr,
                                                 nullptr, nullptr, b->cellinfo, 0, nullptr,
                                                 nullptr, nullptr);
  return hipGetLastError();
}

hipError_t launch_neigh_fill(fnet_batch* b, double rc, long long a0, long long a1, int fp64,
                             hipStream_t s) {
  const long long n = a1 - a0;
  if (n <= 0 || b->n_cell_struct == b->S) return hipSuccess;
  const unsigned grid = (unsigned)((n + 3) / 4);
  if (fp64) {
    k_neigh<kFill, double4><<<grid, 256, 0, s>>>(b->xyz, b->off, b->atom_struct, b->sinfo,
                                                 b->lat, rc, a0, a1, nullptr, b->rowptr, b->nj,
                                                 b->nimg, (double4*)b->nd, b->cellinfo, 0,
                                                 nullptr, nullptr, nullptr);
  } else {
    k_neigh<kFill, float4><<<grid, 256, 0, s>>>(b->xyz, b->off, b->atom_struct, b->sinfo,
                                                b->lat, rc, a0, a1, nullptr, b->rowptr, b->nj,
                                                b->nimg, (float4*)b->nd, b->cellinfo, 0,
                                                nullptr, nullptr, nullptr);
  }
  return hipGetLastError();
}

// Atoms up to which the direct search gives each four waves: beyond about a wave to every SIMD the
// barriers cost more than the shorter walk gains (3072 water atoms 21.5 us with one, 23.6 with four).
constexpr long long kNeighSplit = 1024;

hipError_t launch_neigh_pad(fnet_batch* b, double rc, int fp64, hipStream_t s, int* mir,
                            unsigned long long* stamp) {
  const long long n = b->N;
  if (n <= 0 || b->n_cell_struct == b->S) return hipSuccess;
  const bool split = n <= kNeighSplit;
  const unsigned grid = (unsigned)(split ? n : (n + 3) / 4);
  auto go = [&](auto* kern, auto* nd) {
    kern<<<grid, 256, 0, s>>>(b->xyz, b->off, b->atom_struct, b->sinfo, b->lat, rc, 0, n, b->cnt,
                              nullptr, b->pnj, b->pnimg, nd, b->cellinfo, b->nb_cap, mir,
                              b->d_maxnb, stamp);
  };
  if (fp64)
    go(split ? k_neigh<kPadded, double4, true> : k_neigh<kPadded, double4>, (double4*)b->pnd);
  else
    go(split ? k_neigh<kPadded, float4, true> : k_neigh<kPadded, float4>, (float4*)b->pnd);
  return hipGetLastError();
}

hipError_t launch_compact_rows(fnet_batch* b, int fp64, hipStream_t s) {
  const long long tot = (long long)b->N * b->nb_cap;
  if (tot <= 0) return hipSuccess;
  const unsigned grid = (unsigned)((tot + 255) / 256);
  if (fp64) {
    k_compact_rows<double4><<<grid, 256, 0, s>>>(b->N, b->nb_cap, b->cnt, b->rowptr, b->pnj,
                                                 b->pnimg, (const double4*)b->pnd, b->nj,
                                                 b->nimg, (double4*)b->nd);
  } else {
    k_compact_rows<float4><<<grid, 256, 0, s>>>(b->N, b->nb_cap, b->cnt, b->rowptr, b->pnj,
                                                b->pnimg, (const float4*)b->pnd, b->nj, b->nimg,
                                                (float4*)b->nd);
  }
  return hipGetLastError();
}

}  // namespace fnet
