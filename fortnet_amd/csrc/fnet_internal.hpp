// Internal declarations shared by the HIP translation units of libfnet_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <string>
#include <map>
#include <vector>

namespace fnet {

constexpr int kMaxLayers = 8;   // input + hidden + output layers of one element network
constexpr int kMaxDim = 256;    // widest layer of the generic network kernels
constexpr int kMaxMembers = 16; // functions sharing one angular neighbour-pair loop
constexpr int kMaxZ = 16;       // distinct atomic numbers referenced by one model
constexpr int kLadSlots = 10;   // (lambda, 2^m) slots of an exponent-ladder group: 2 x 5
constexpr int kProgLen = 8;     // exponents per lambda of a progression group
constexpr int kMaxOut = 8;      // network outputs (targets)
constexpr double kPi = 3.14159265358979323846; // lib_dftbp/constants.F90:15

// One radial function (G1/G2/G3), acsf.F90:1287-1373.
// A model whose z-score divides some radial feature by a sigma below |mean| / kRadial64Kappa has
// its radial functions summed in FP64 in the FP32 modes too.  Summed in FP32 over a few dozen
// neighbours they carry a relative error of up to ~4e-7, which the z-score turns into ~1e-5 of a
// network input at this ratio; on a perturbed diamond lattice (|mean| / sigma up to 124) that
// error alone moved the forces by 1.6e-4 eV/A RMS.
constexpr double kRadial64Kappa = 25.0;

struct RadialFn {
  int col;     // output column in G
  int type;    // 1, 2, 3
  int zc;      // element code of neighbour species, -1 = any
  int atomid;  // 0 = none, else 1-based ext column
  double rc, eta, rs, kappa;
};

// Angular functions (G4/G5, acsf.F90:1377-1492) that share type, cutoff, eta, species pair and
// atom-id column: they are evaluated in one pass over the neighbour pairs.
struct AngGroup {
  int type;   // 4 or 5
  int zc1, zc2;
  int same;   // both neighbour lists identical (unresolved or Z1 == Z2): ordered pairs + diagonal
  int atomid;
  int nmem;
  double rc, eta;
  int col[kMaxMembers];
  int xint[kMaxMembers]; // xi as an integer power, or -1 for a general real power
  double xi[kMaxMembers];
  double lam[kMaxMembers];
  double scale[kMaxMembers]; // 2^(1 - xi)
  double pdiag[kMaxMembers]; // (1 + lam)^xi: the j == k terms, where cos(theta) = 1
  // Exponent-ladder form (lad > 0): every member has xi = 2^m with m <= lad <= 4 and one of at
  // most two lambda values; slot 5 i + m stands for (lamv[i], 2^m) and names its member (or -1).
  int lad;
  int lmask;  // bit m set when some member has xi = 2^m
  double lamv[2];
  int smem[kLadSlots];
  double lpdiag[kLadSlots]; // (1 + lamv[i])^(2^m)
  // Progression form (np > 0, groups without the ladder form): the exponents are x0 + k s, k < np
  // <= kProgLen, x0 >= 1, with the lambdas in lamv (the reference's automatic scheme); slot
  // kProgLen i + k stands for (lamv[i], x0 + k s).  The powers of 1 + lambda cos(theta) then are
  // P^(x0 - 1) and P R^k with R = P^s, both exponents split into integer and fraction.
  int np;
  int sint, bint;       // integer parts of s and x0 - 1
  double sfrac, bfrac;  // their fractions
  double pdelta[kProgLen];  // xi_k - (x0 + k s), a few ulp of xi_k at most
  int pexact;               // some exponent is no integer
  int pmem[2 * kProgLen];
  // Adjoint pass: a G5 ladder group and another one over the same lists with the same ladder
  // and lambdas but another eta are evaluated together (partner >= 0 on the first one,
  // follower = 1 on the second).
  int partner;
  int follower;
};

// Network shape of every element network.
struct NetShape {
  int nl;                  // number of layers
  int dims[kMaxLayers];
  long long woff[kMaxLayers]; // offset of ww(l) (d_l x d_{l+1}) in the serialised vector
  long long boff[kMaxLayers]; // offset of bb(l)
  long long nparams;
  int act[64];             // hidden activation per species (<= 64 species)
};

// Per-structure neighbour-search data, computed on the device each step.
struct StructInfo {
  double inv[9];    // inverse lattice, inv[c*3+r] = inv(r,c)
  double smin[3], smax[3]; // extent of fractional coordinates
  double bmin[3], bmax[3]; // Cartesian bounding box of the atoms
  double w[3];      // rc * |row_a(inv L)|: largest fractional offset of a neighbour
  int lo[3], hi[3]; // reference image ranges (latpointiter.F90:226-253)
  int periodic;
  int pad;
};

// Scalar state of one element network's optimizer (fnet_optim.hip); the vectors live in
// fnet_ctx::opt_vecs.
struct OptState {
  int kind, converged, mem, line_search;
  double tol, max_disp, lr;
  // line minimiser (linemin.F90)
  int lm_state, lm_it, lm_conv, lm_maxiter;
  double lm_tol, lm_xx[2], lm_dx[2], lm_xcur, lm_first, lm_maxx;
  int cg_state;        // conjugate gradients: 1 before the first direction
  int lb_it;           // L-BFGS: directions computed so far
  int f_it, f_reset;   // FIRE
  double f_a, f_dt;
};

// Device copy of the model.
struct DevModel {
  int nG = 0, nR = 0, nAG = 0, nZ = 0;
  int maxmem = 1;               // largest angular group
  int form = 0;                 // angular groups: 1 all exponent ladders, 2 ladders and
                                // progressions, 0 some group has neither
  int maxprog = 0;              // longest progression
  int has_pairs = 0;            // some angular groups are evaluated in pairs by the adjoint
  int n_followers = 0;          // ... second groups of them
  int radial_resolved = 0;      // some radial function is restricted to one neighbour element
  int radial64 = 0;             // FP32 modes sum the radial functions in FP64 (kRadial64Kappa)
  int need_ext = 0;             // external feature columns the model reads
  int zlist[kMaxZ];
  int nspecies = 0, nout = 0, nin = 0, next_in = 0;
  double rcmax = 0.0;
  NetShape shape{};
  RadialFn* radial = nullptr;   // [nR]
  AngGroup* groups = nullptr;   // [nAG]
  double* zmean = nullptr;      // [nG] (0 where no standardisation)
  double* zinv = nullptr;       // [nG] (1 where no standardisation)
  int* ext_in = nullptr;        // [next_in] 0-based ext columns
  double* params = nullptr;     // [nspecies][nparams]
  float* params_f = nullptr;    // FP32 copy
  // FP32 weights packed as MFMA operand fragments (per species, stride pk_stride floats):
  // forward fragments of every layer at pk_fw[l], reverse (transposed) fragments at pk_rw[l],
  // biases zero-padded to a multiple of 16 at pk_b[l]
  float* wpack = nullptr;
  long long pk_stride = 0;
  long long pk_fw[kMaxLayers] = {}, pk_rw[kMaxLayers] = {}, pk_b[kMaxLayers] = {};
  // BF16 hi / lo fragments of the hidden-to-hidden layers (BF16 modes), in units of 8 values
  uint16_t* bpack = nullptr;
  long long bk_stride = 0;
  long long bk_fw[kMaxLayers] = {}, bk_rw[kMaxLayers] = {}, bk_sz[kMaxLayers] = {};
  bool valid = false;
};

// Launch parameters of the batched kernels chosen by the autotuner (fnet_autotune) for a model,
// precision and batch size; 0 / -1 leave the built-in choice.
struct Tune {
  int fwd_wpb = 0;    // waves per block of the forward ACSF kernel (1, 2, 4)
  int adj_wpb = 0;    // waves per block of the adjoint ACSF kernel (1, 2)
  int mlp_waves = 0;  // waves of 16 atoms per block of the MFMA network kernels (1, 2, 4)
  int rbal = -1;      // forward radial lanes in proportion to the element ranges (0, 1)
  int persist = 0;    // ACSF kernels on a persistent grid (1)
  bool operator==(const Tune& o) const {
    return fwd_wpb == o.fwd_wpb && adj_wpb == o.adj_wpb && mlp_waves == o.mlp_waves &&
           rbal == o.rbal && persist == o.persist;
  }
};

// Host I/O through pinned memory (fnet_stage.hip): segments that one kernel copies.  The largest array
// and the ring bound the pinned memory of a context.  At the line (21 760 atoms, 522 KB of coordinates)
// an upload alone takes 26 us by command and 29 through the ring, a whole MD call 310 and 292, since
// results of up to half of it come back without a copy command; the latter goes on beyond (43 520
// atoms 500 and 477).
constexpr int kStageSegs = 24;
constexpr size_t kStageRing = 2u << 20;  // pinned bytes of one context
constexpr size_t kStageMax = 512u << 10; // larger arrays keep their own copy command
struct StageSegs {
  int n = 0;
  unsigned first[kStageSegs];
  const void* src[kStageSegs];
  void* dst[kStageSegs];
  size_t bytes[kStageSegs];
};
struct StageOut {
  void* host;
  const void* dev;
  size_t bytes;
};

}  // namespace fnet

struct fnet_batch;

struct fnet_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // side stream of the steady-state step (the mirror entries run beside the ACSF forward and
  // the networks) and the events that fork it from and join it to the main stream
  hipStream_t side = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  std::string err;
  char* ring = nullptr;      // pinned ring of the staged copies
  size_t ring_at = 0;
  fnet::StageSegs segs;      // copies in that have not been launched yet
  bool stage_direct = false; // ... and a copy command was enqueued beside them
  fnet::DevModel model;
  hipEvent_t ev[8] = {};
  int n_ev = 0;
  // stage boundaries of the last steady-state step, written by its kernels (an event between two
  // kernels costs a barrier packet each); stamped: the last step's times are these
  unsigned long long* stamps = nullptr;
  double stamp_khz = 0.0;
  bool stamped = false;
  double* d_grad = nullptr; // [nspecies][nparams] FP64 gradient of the last train call
  long long grad_cap = 0;
  bool have_grad = false;
  int loss = 0;               // fnet_loss of the training gradient and loss value
  int use_graph = 0;          // fnet_run replays a captured HIP graph of its steady-state step
  double last_loss = 0.0;     // loss of the last training-gradient call
  // device optimizers (fnet_optimizer_init / _step)
  int opt_kind = -1;
  fnet::OptState* opt_states = nullptr;  // [nspecies]
  double* opt_vecs = nullptr;            // [nspecies][opt_vstride]
  int* opt_conv = nullptr;               // [nspecies]
  long long opt_vstride = 0, opt_cap = 0;
  long long model_gen = 0;    // bumped by every model upload (new device tables)
  long long params_gen = 0;   // bumped by every change of the parameters (uploads, optimizer steps)
  double reg_strength = 0.0;  // elastic-net regularisation of the weight gradients
  double reg_alpha = 0.0;
  int n_cu = 0;               // compute units of the device (persistent grids)
  int lds_block = 64 * 1024;  // LDS bytes one block may allocate (the device's limit)
  // autotuned launch parameters per (model generation, precision, log2 of the atom count)
  std::map<std::vector<long long>, fnet::Tune> tunes;
};

struct fnet_batch {
  fnet_ctx* ctx = nullptr;
  int S = 0;
  long long N = 0;
  int next = 0;
  int precision = 1;
  int launch = 0;
  long long capN = 0, capS = 0, capExt = 0;     // allocated capacities (reused by reload)
  long long res_N = 0, res_S = 0;               // capacity of the result buffers
  int res_nG = -1, res_nout = -1;
  std::vector<long long> h_off;
  std::vector<int> h_species;
  int max_species = -1;        // largest of them
  // inputs
  double* xyz = nullptr;       // [N][3]
  double* lat = nullptr;       // [S][9]
  int* periodic = nullptr;     // [S]
  long long* off = nullptr;    // [S+1]
  int* atom_struct = nullptr;  // [N]
  int* species = nullptr;      // [N]
  int* zcode = nullptr;        // [N] element slot of each atom under the current model
  std::vector<int> h_atnum;    // atomic numbers (host): element slots follow model uploads
  int zone = 0;                // one element slot, taken by every atom (staging skips the sort)
  unsigned long long zcode_gen = 0;  // model generation zcode was derived with
  double* ext = nullptr;       // [N][next]
  fnet::StructInfo* sinfo = nullptr; // [S]
  // per-species tiles of the network kernels; the tables share one allocation (tab)
  int* tab = nullptr;
  size_t tab_cap = 0;
  std::vector<int> h_tab;
  int* perm = nullptr;         // [N] atoms grouped by species
  int* tile_sp = nullptr;      // [ntiles]
  int* tile_start = nullptr;   // [ntiles] into perm
  int* tile_cnt = nullptr;     // [ntiles]
  int ntiles = 0;
  int tile_atoms = 0;
  int tile_launch = -1;          // launch mode the tiles were built for
  std::vector<int> h_tile_first; // [S+1] tiles of each structure (per-structure launches)
  // block tiles of the MFMA network kernel (16 atoms per wave, mtile_waves waves per block)
  int* mtile_sp = nullptr;
  int* mtile_start = nullptr;
  int* mtile_cnt = nullptr;
  int nmtiles = 0;
  int mtile_waves = 0;
  std::vector<int> h_mtile_first; // [S+1]
  // neighbour list (CSR)
  int* cnt = nullptr;          // [N]
  int* rowptr = nullptr;       // [N+1]
  int* scan_tmp = nullptr;
  long long scan_tmp_cap = 0;
  int* nj = nullptr;           // [P]
  int* nimg = nullptr;         // [P]
  void* nd = nullptr;          // [P] double4 or float4: image position - centre, and r^2
  long long pcap = 0;
  long long npairs = 0;
  int max_nb = 0;
  int* d_maxnb = nullptr;
  // one-pass search (batched launches): row i at i * nb_cap, then compacted into the CSR list;
  // nb_cap comes from the previous list (0: count pass + fill pass)
  int nb_cap = 0;
  bool nl_padded = false;      // the current list is the padded rows (compacted on download)
  long long pad_len = 0;       // allocated padded entries
  int* pnj = nullptr;
  int* pnimg = nullptr;
  void* pnd = nullptr;         // double4 (room for either precision)
  // cell lists of large periodic structures
  int4* cellinfo = nullptr;    // [S] bins per axis (x, y, z) and use flag (w)
  int* cell_off = nullptr;     // [S+1] first global cell of each structure
  int* cell_count = nullptr;   // [ncells] (reused as the scatter cursor)
  int* cell_start = nullptr;   // [ncells+1]
  int* cell_atoms = nullptr;   // [N]
  int* atom_cell = nullptr;    // [N]
  int4* atom_m = nullptr;      // [N] integer part of the fractional coordinates, local bin
  int* cell_scan_tmp = nullptr;
  long long ncells = 0;        // cells of the structures with cell lists, one more per structure
  long long cell_cap = 0;      // allocated cells
  int n_cell_struct = 0;       // structures with cell lists
  int bin_lds = 0;             // > 0: every such structure is binned by its struct-prep block, with
                               // this many LDS bins; 0: binning kernels over all atoms
  std::vector<int> h_cellinfo; // [4*S]
  std::vector<double> h_lat;   // [S][9]
  std::vector<int> h_periodic; // [S]
  // results
  void* G = nullptr;           // [N][nG] FP64 (accumulated in FP64 in both precisions)
  void* cG = nullptr;          // [N][nout][nG] T
  double* Eatom = nullptr;     // [N][nout]
  double* Estruct = nullptr;   // [S][nout]
  void* F = nullptr;           // [N][nout][3] FP64
  double* lossgrad = nullptr;  // [N][nout]
  // force assembly (fnet_gather.hip): per-entry adjoint gradients and mirror entries, sized for
  // the list layout (padded rows or CSR)
  double* gvec = nullptr;      // [entries][nout][3], FP64 values (FP64 mode) or FP32 values
  int* mir = nullptr;          // [entries] mirror entry (j, i, -n) of each entry, -1 if none
  int* orph = nullptr;         // [entries] entries without a mirror
  int* d_norph = nullptr;      // number of them
  long long gv_entries = 0;    // allocated entries of mir / orph
  long long gv_len = 0;        // allocated doubles of gvec
  bool have_mirror = false;
  bool mir_clear = false;      // every entry of the current padded list has its mirror slot at -1
  // energy reduction in fixed-size chunks of atoms (two passes, fixed order)
  int* chunk_tab = nullptr;    // allocation of the two tables
  size_t chunk_cap = 0;
  int* chunk_struct = nullptr; // [nchunks]
  int* chunk_first = nullptr;  // [S+1]
  double* Epart = nullptr;     // [nchunks][nout]
  std::vector<int> h_chunk_first;
  int nchunks = 0;
  int single_chunks = 0;       // every structure has exactly one chunk
  long long epart_len = 0;
  // weight gradient: one FP64 partial vector per network tile, reduced in tile order
  double* gpart = nullptr;
  long long gpart_len = 0;
  // steady-state step of fnet_run (no host read-back): the longest row of the list it built is
  // copied to pinned host memory with the step and checked when results are next read
  int* h_maxnb = nullptr;
  // small batches: pinned copies of the results, written by the kernels that produce them
  // (kHostAtoms), and which of them hold the current results
  double* h_res = nullptr;
  size_t h_res_cap = 0;
  bool host_E = false, host_F = false;
  bool loaded = false;          // the last load or update got through
  bool pending = false;
  int pending_level = 0;        // what was computed on that list: 1 features, 2 energies, 3 forces
  long long gen = 0;            // bumped whenever a buffer the step uses is reallocated
  // HIP graph of the steady-state step and the launch parameters it was captured with
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::vector<long long> gkey;
  int graph_failed = 0;         // capture or instantiation failed once: run the step eagerly
  int last_graph = 0;           // the last fnet_run replayed the graph
  double* d_targets = nullptr; // staging of training inputs
  long long targets_cap = 0;
  bool have_nl = false, have_G = false, have_E = false, have_F = false;
  // model and parameter generations the batch's results were computed with
  long long seen_model_gen = -1, seen_params_gen = -1;
  int result_precision = -1;
};

namespace fnet {

// The launch parameters for a batch: the tuned entry of its model, precision and size, else
// the defaults.
const Tune& tune_of(const fnet_batch* b);
std::vector<long long> tune_key(const fnet_batch* b);

// Distance of a neighbour entry.  The neighbour kernels store the squared distance of the FP64
// membership test in V.w, in the list's precision (FP32 rows: rounded to FP32); the ACSF kernels
// take the square root when they stage the entry (entry_r): FP64 rows the FP64 root, FP32 rows
// (the FP32 path, held to its accuracy gates) the FP32 root of the rounded value.  Taking it
// there costs one root per entry instead of one per tested candidate (the compiler evaluates
// the root before the store's branch; ~27 candidates per entry on the Si cells).
__device__ __forceinline__ void entry_d2(double4& v, double d2) { v.w = d2; }
__device__ __forceinline__ void entry_d2(float4& v, double d2) { v.w = (float)d2; }
__device__ __forceinline__ double entry_r(double w) { return sqrt(w); }
__device__ __forceinline__ float entry_r(float w) { return sqrtf(w); }

// staged host I/O (fnet_stage.hip), on the context's stream: stage_in copies `src` now and to the
// device with the next stage_flush; stage_out brings n results to the host and waits for them
hipError_t stage_in(fnet_ctx* ctx, void* dst, const void* src, size_t bytes);
hipError_t stage_flush(fnet_ctx* ctx);
hipError_t stage_out(fnet_ctx* ctx, const StageOut* out, int n);

// Batches of up to this many outputs have their energies and forces written to pinned host memory
// as they are formed: an MD call of 1 024 atoms 100 -> 78 us, of 8 192 167 -> 146.  The line bounds the
// pinned memory that a batch holds (256 KB); the gain goes on beyond it (32 768 atoms 405 -> 367).
constexpr long long kHostAtoms = 8192;
inline double* host_Estruct(const fnet_batch* b);
inline double* host_Eatom(const fnet_batch* b);
inline double* host_F(const fnet_batch* b);

// launchers (fnet_neigh.hip)
// lattices, extents and (bin_lds > 0) cell bins; clears the batch's row maximum
hipError_t launch_struct_prep(fnet_batch* b, double rc, hipStream_t s,
                              unsigned long long* stamp = nullptr);
// Largest structure, and most bins, that a struct-prep block bins: one block's walk over the atoms
// against four launches over all of them.  An MD call of one structure of 1 000 Si atoms 96 -> 84 us,
// 4 096 133 -> 115, 8 000 169 -> 154, 21 952 335 either way, four of those 1 020 -> 1 037.
constexpr int kPrepBins = 4096;
constexpr int kPrepBinAtoms = 8192;
hipError_t launch_neigh_count(fnet_batch* b, double rc, long long a0, long long a1, hipStream_t s);
hipError_t launch_neigh_fill(fnet_batch* b, double rc, long long a0, long long a1, int fp64,
                             hipStream_t s);
// padded rows; a non-null mir (sized for the padded layout) gets -1 at every entry written
// (stamp: end of the launch, near enough: stamp_now)
hipError_t launch_neigh_pad(fnet_batch* b, double rc, int fp64, hipStream_t s,
                            int* mir = nullptr, unsigned long long* stamp = nullptr);
hipError_t launch_cells_pad(fnet_batch* b, double rc, int fp64, hipStream_t s,
                            int* mir = nullptr, unsigned long long* stamp = nullptr);
hipError_t launch_compact_rows(fnet_batch* b, int fp64, hipStream_t s);
hipError_t launch_scan(int* cnt, int* rowptr, long long n, int* tmp, hipStream_t s,
                       int* maxout);
long long scan_tmp_size(long long n);

// launchers (fnet_cells.hip)
constexpr int kCellMinAtoms = 64; // structures at least this large may use cell lists
// Cost of one cell-list candidate (bin walk, LDS sort into the reference's order) in units of
// one direct-scan candidate: 8192 Si cells of 290-512 atoms (3 bins of width rc per axis, the
// 27 stencil bins covering the whole cell, ~4 images per atom in the direct scan) took 1.83 ms
// with cell lists and 1.69 ms with the direct scan.
constexpr double kCellCandidateCost = 5.0;
hipError_t launch_cell_bin(fnet_batch* b, hipStream_t s);
// sort capacity of one wave of the cell-list search (power of two >= need, at least 64) and its
// LDS bytes in the writing passes
int cells_sort_capacity(int need);
size_t cells_lds_bytes(int need, int fp64);
hipError_t launch_cells_count(fnet_batch* b, double rc, long long a0, long long a1, hipStream_t s);
hipError_t launch_cells_fill(fnet_batch* b, double rc, long long a0, long long a1, int fp64,
                             hipStream_t s);

// launchers (fnet_optim.hip)
long long opt_vec_doubles(long long n, int mem);
hipError_t launch_opt_init(const double* params, double* vecs, long long n, long long vstride,
                           int mem, int nspecies, hipStream_t s);
hipError_t launch_opt_step(OptState* states, double* params, const double* grad, double* vecs,
                           long long n, long long vstride, double fx, int* conv, int nspecies,
                           hipStream_t s);

// entries of a batch's current neighbour-list layout: padded rows or CSR
inline long long layout_entries(const fnet_batch* b);

// no-allocation force assembly (fnet_gather.hip): static device scratch of kNoallocScratchBytes
// per GPU, its address resolved per device by scratch_init (called by fnet_ctx_create)
constexpr long long kNoallocScratchBytes = 32LL << 20;
hipError_t scratch_init(int device);
void* scratch_ptr(int device);

// launchers (fnet_gather.hip)
hipError_t launch_zero_int(int* p, int n, hipStream_t s);
hipError_t launch_mirror(fnet_batch* b, long long a0, long long a1, long long fill_entries,
                         hipStream_t s);
// energies: also the energy chunks of the whole batch, in blocks of their own
hipError_t launch_force_gather(fnet_batch* b, const DevModel& m, long long a0, long long a1,
                               bool energies, hipStream_t s);
// the orphans' part of the forces; energies: also the sums over the chunks; host: also the pinned
// copy of the forces; stamps: {start, end} of the launch (stamp_last)
hipError_t launch_force_finish(fnet_batch* b, const DevModel& m, bool energies, hipStream_t s,
                               bool host, unsigned long long* stamps = nullptr);

// launchers (fnet_acsf.hip)
hipError_t launch_acsf_fwd(fnet_batch* b, const DevModel& m, long long a0, long long a1, int fp64,
                           hipStream_t s);
// norph: orphan counter that the launch clears, or null
hipError_t launch_acsf_adj(fnet_batch* b, const DevModel& m, long long a0, long long a1, int fp64,
                           hipStream_t s, int* norph, unsigned long long* stamp = nullptr);

// launchers (fnet_mlp.hip)
// mirror: extra blocks of the launch search the mirror entries of the whole batch
hipError_t launch_mlp_fwd(fnet_batch* b, const DevModel& m, int first_tile, int ntiles, int fp64,
                          int want_grad_in, hipStream_t s, bool mirror = false,
                          unsigned long long* stamp = nullptr);
constexpr int kEnergyChunk = 2048;  // atoms per block of the energy reduction
// host: also the pinned copies (longest row, energies of small batches)
hipError_t launch_energy_reduce(fnet_batch* b, const DevModel& m, int s0, int s1, hipStream_t s,
                                bool host = false);
// Training targets and weights on the device, and where the loss goes: part [3 nchunks] (per energy
// chunk), out [1]
struct LossInput {
  int n_global, loss;
  const double* gt;
  const double* at;
  const double* aw;   // null: 1
  const double* dpw;  // null: 1
  double inv_wsum;
  double* part;
  double* out;
};
// loss gradient of every atomic output and the loss of every chunk
hipError_t launch_lossgrad(fnet_batch* b, const DevModel& m, const LossInput& in, hipStream_t s);
// weight gradient: per-tile partials into b->gpart, then their sum in a fixed order into grad; with
// it the loss, from the chunks of launch_lossgrad
hipError_t launch_mlp_grad(fnet_batch* b, const DevModel& m, int fp64, double* grad,
                           const LossInput& in, hipStream_t s);
// number of weight-gradient partial vectors launch_mlp_grad writes into b->gpart
int grad_parts(const fnet_batch* b, const DevModel& m, int fp64);
// MFMA weight gradient (FP32 / BF16 modes): blocks per MFMA tile, 0 without an MFMA path
int mlp_grad_subtiles(const NetShape& sh, int tile_waves);
hipError_t launch_mlp_grad_mfma(fnet_batch* b, const DevModel& m, hipStream_t s);
// elastic-net term (scale = strength / sum of datapoint weights) added to the device gradient
hipError_t launch_regularize(const DevModel& m, double* grad, double scale, double alpha,
                             hipStream_t s);
hipError_t launch_sd_step(double* params, const double* grad, long long n, double lr,
                          double max_disp, double tol, double* scratch, int nspecies,
                          hipStream_t s);
// atoms per generic tile of the batch
int mlp_tile_atoms(const fnet_batch* b, const NetShape& sh, int fp64);
int grad_chunks(int ntiles);  // chunks of the weight-gradient reduction

// launchers (fnet_mlp_f64.hip): FP64 element networks on MFMA 16x16x4 f64.  Atoms per tile of the
// batch (a multiple of 16), 0 if the network is too wide for a block's LDS
int mlp_f64_tile_atoms(const fnet_batch* b, const NetShape& sh);
hipError_t launch_mlp_f64(fnet_batch* b, const DevModel& m, int first_tile, int ntiles,
                          int want_grad_in, hipStream_t s, bool mirror, unsigned long long* stamp);
hipError_t launch_mlp_grad_f64(fnet_batch* b, const DevModel& m, hipStream_t s);

// launchers (fnet_mlp_mfma.hip): FP32 element networks on MFMA 16x16x4 f32
int mlp_mfma_waves(const NetShape& sh);  // waves per block, 0 if the shape is not supported
// sizes of the packed fragments (floats, bf16 values) and where each layer's lie
void mfma_layout(DevModel& m, size_t* floats, size_t* halves);
hipError_t launch_mlp_mfma(fnet_batch* b, const DevModel& m, int first_tile, int ntiles,
                           int want_grad_in, hipStream_t s, bool mirror = false,
                           unsigned long long* stamp = nullptr);
// FP32 copy of the resident parameters and, for networks on the matrix cores, their fragments
hipError_t launch_model_params(const DevModel& m, hipStream_t s);

size_t lds_bytes_acsf(int max_nb, int nZ, int fp64, int adj);
int acsf_slice_entries(int max_nb);  // entries of one wave's LDS slice for rows up to max_nb

}  // namespace fnet

#define FNET_HIP_TRY(expr)                                   \
  do {                                                       \
    hipError_t _e = (expr);                                  \
    if (_e != hipSuccess) return _e;                         \
  } while (0)

namespace fnet {
inline double* host_Estruct(const fnet_batch* b) { return b->h_res; }
inline double* host_Eatom(const fnet_batch* b) { return b->h_res + b->S * b->ctx->model.nout; }
inline double* host_F(const fnet_batch* b) { return host_Eatom(b) + b->N * b->ctx->model.nout; }
inline long long layout_entries(const fnet_batch* b) {
  return b->nl_padded ? (long long)b->N * b->nb_cap : b->npairs;
}
}  // namespace fnet
