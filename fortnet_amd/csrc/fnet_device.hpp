// Device functions that kernels of several translation units share: the mirror search of one
// centre and the energy sum of one chunk, each run by blocks of their own or by extra blocks of
// another stage's launch.
#pragma once

#include "fnet_internal.hpp"

namespace fnet {

// Raises *p to v.  A row's count rarely passes the largest so far, so the plain read (a stale
// value only costs an atomic) keeps the rows of a large batch from queueing on one address.
__device__ __forceinline__ void raise_max(int* p, int v) {
  if (v > __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(p, v);
}

// Integer part of an atom's fractional coordinates and its bin among the ci.x ci.y ci.z bins of
// its cell.
__device__ __forceinline__ int4 bin_of(const StructInfo& si, const double* x, const int4& ci) {
  const int nb[3] = {ci.x, ci.y, ci.z};
  int m[3], bn[3];
  for (int a = 0; a < 3; ++a) {
    const double f = si.inv[0 * 3 + a] * x[0] + si.inv[1 * 3 + a] * x[1] + si.inv[2 * 3 + a] * x[2];
    const double fl = floor(f);
    m[a] = (int)fl;
    const int b = (int)((f - fl) * nb[a]);
    bn[a] = b < 0 ? 0 : (b >= nb[a] ? nb[a] - 1 : b);
  }
  return make_int4(m[0], m[1], m[2], (bn[0] * nb[1] + bn[1]) * nb[2] + bn[2]);
}

struct RowLayout {
  const int* rowptr;  // CSR rows (cap == 0)
  const int* cnt;     // padded rows: row i at i * cap with cnt[i] entries
  int cap;
  __device__ __forceinline__ long long base(long long i) const {
    return cap ? i * (long long)cap : (long long)rowptr[i];
  }
  __device__ __forceinline__ int len(long long i) const {
    return cap ? min(cnt[i], cap) : rowptr[i + 1] - rowptr[i];
  }
};

struct MirrorArgs {
  RowLayout rl;
  const int* nj;
  const int* key;
  const long long* off;
  const int* atom_struct;
  const StructInfo* sinfo;
  long long a0, a1;
  int* mir;
};

// The mirror entries of centre i, by one wave; lanes over the centre's entries.  The entries store
// their keys (image + 1) n + (j - i) mod n.  Each mirror pair is searched once, from the entry with
// i < j (or, for the centre's own images, from the one with the lower image index), which writes
// both directions; entries left at -1 (filled before) have no mirror.
__device__ __forceinline__ void mirror_centre(const MirrorArgs& a, long long i, int lane) {
  if (i >= a.a1) return;
  const int s = a.atom_struct[i];
  const long long o = a.off[s];
  const int n = (int)(a.off[s + 1] - o);
  const StructInfo& si = a.sinfo[s];
  const int nimages =
      si.periodic ? (si.hi[0] - si.lo[0] + 1) * (si.hi[1] - si.lo[1] + 1) *
                            (si.hi[2] - si.lo[2] + 1) - 1
                  : 0;
  const int li = (int)(i - o);
  const long long bi = a.rl.base(i);
  const int len = a.rl.len(i);
  for (int e = lane; e < len; e += 64) {
    const int k = a.key[bi + e];
    const int j = a.nj[bi + e];
    const int lj = j - (int)o;
    const int img = k / n - 1;
    const int t = k - (img + 1) * n;  // (j - i) mod n
    const int mimg = img < 0 ? -1 : nimages - 1 - img;
    if (!(li < lj || (li == lj && img < mimg))) continue;
    const int target = (mimg + 1) * n + (t == 0 ? 0 : n - t);
    const long long bj = a.rl.base(j);
    const int lenj = a.rl.len(j);
    int lo = 0, hi = lenj;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (a.key[bj + mid] < target) lo = mid + 1;
      else hi = mid;
    }
    if (lo < lenj && a.key[bj + lo] == target) {
      a.mir[bi + e] = (int)(bj + lo);
      a.mir[bj + lo] = (int)(bi + e);
    }
  }
}

inline MirrorArgs mirror_args(const fnet_batch* b, long long a0, long long a1) {
  MirrorArgs m;
  m.rl.rowptr = b->rowptr;
  m.rl.cnt = b->cnt;
  m.rl.cap = b->nl_padded ? b->nb_cap : 0;
  m.nj = b->nl_padded ? b->pnj : b->nj;
  m.key = b->nl_padded ? b->pnimg : b->nimg;
  m.off = b->off;
  m.atom_struct = b->atom_struct;
  m.sinfo = b->sinfo;
  m.a0 = a0;
  m.a1 = a1;
  m.mir = b->mir;
  return m;
}

// Per-structure sums of the atomic outputs (predictBatch sums, bpnn.F90:1040-1047;
// forces.F90:381-385) in FP64 with a fixed order: each block sums one chunk of kEnergyChunk atoms
// of one structure (thread t takes atoms t, t + 256, ... in order; the four wave sums combine in a
// fixed order), then a structure's chunks are added in order.  The result does not depend on
// scheduling, and a large cell is spread over many blocks instead of one.  `single`: every
// structure is one chunk, whose sum is the structure's.
struct EnergyArgs {
  const double* Eatom;
  const long long* off;
  const int* chunk_struct;
  const int* chunk_first;
  int nout, single;
  double* Epart;
  double* Estruct;
  const int* maxnb;  // longest row of the list, handed to the host with the energies
  int* h_maxnb;      // pinned host memory, or null
  double* h_Eatom;   // pinned copies of the energies, or null
  double* h_Estruct;
};

// chunk c by a block of 256 threads
__device__ __forceinline__ void energy_chunk(const EnergyArgs& a, int c, double* ws) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = a.chunk_struct[c];
  const long long a0 = a.off[s] + (long long)(c - a.chunk_first[s]) * kEnergyChunk;
  const long long a1 = min(a0 + (long long)kEnergyChunk, a.off[s + 1]);
  for (int t = 0; t < a.nout; ++t) {
    double v = 0.0;
    for (long long i = a0 + threadIdx.x; i < a1; i += 256) {
      const double e = a.Eatom[i * a.nout + t];
      if (a.h_Eatom) a.h_Eatom[i * a.nout + t] = e;
      v += e;
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    if (lane == 0) ws[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      const double e = (ws[0] + ws[1]) + (ws[2] + ws[3]);
      if (a.single) {
        a.Estruct[(long long)s * a.nout + t] = e;
        if (a.h_Estruct) a.h_Estruct[(long long)s * a.nout + t] = e;
      } else {
        a.Epart[(long long)c * a.nout + t] = e;
      }
    }
    __syncthreads();
  }
}

// (structure, output) pair q of the structures s0 .. s1 - 1: its chunks in order
__device__ __forceinline__ void energy_total(const EnergyArgs& a, long long q, int s0, int s1) {
  const long long s = s0 + q / a.nout;
  const int t = (int)(q % a.nout);
  if (s >= s1) return;
  double v = 0.0;
  for (int c = a.chunk_first[s]; c < a.chunk_first[s + 1]; ++c)
    v += a.Epart[(long long)c * a.nout + t];
  a.Estruct[s * a.nout + t] = v;
  if (a.h_Estruct) a.h_Estruct[s * a.nout + t] = v;
}

// host: with the pinned copies
inline EnergyArgs energy_args(const fnet_batch* b, const DevModel& m, bool host) {
  EnergyArgs e;
  e.Eatom = b->Eatom;
  e.off = b->off;
  e.chunk_struct = b->chunk_struct;
  e.chunk_first = b->chunk_first;
  e.nout = m.nout;
  e.single = b->single_chunks;
  e.Epart = b->Epart;
  e.Estruct = b->Estruct;
  e.maxnb = b->d_maxnb;
  e.h_maxnb = host ? b->h_maxnb : nullptr;
  e.h_Eatom = host && b->h_res ? host_Eatom(b) : nullptr;
  e.h_Estruct = host && b->h_res ? host_Estruct(b) : nullptr;
  return e;
}

// Time stamp of a stage boundary (the device's constant-rate counter): the start of a launch, by its
// first thread.
__device__ __forceinline__ void stamp(unsigned long long* p) {
  if (p && blockIdx.x == 0 && threadIdx.x == 0) *p = wall_clock64();
}

// Stamps near the end of a launch are taken in its last block: blocks dispatched before it may still
// run, and stores be on their way, a few microseconds longer.  (A maximum over the last 512 blocks,
// each after its stores, cost a 64-atom step 4 us and a request of 209 atoms 14 us.)
__device__ __forceinline__ void stamp_now(unsigned long long* p) {
  if (p) *p = wall_clock64();
}
__device__ __forceinline__ void stamp_last(unsigned long long* p) {
  if (p && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *p = wall_clock64();
}

}  // namespace fnet
