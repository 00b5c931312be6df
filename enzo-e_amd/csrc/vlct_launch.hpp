// vlct_launch.hpp -- host-side launch sequence of the VL+CT step, shared by
// the FP64 translation unit (vlct_capi.hip, built without FMA contraction
// for bitwise reference parity), the mixed-precision one (vlct_mixed.hip, FP32
// reconstruction and Riemann fluxes) and the contracted FP64 one
// (vlct_fp64c.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>
#include <map>
#include <string>
#include <cmath>
#include <type_traits>
#include <vector>

#include "../../include/enzoe_vlct.h"
#include "vlct_kernels.hpp"
#include "vlct_march.hpp"

namespace enzoe {

// ----------------------------------------------------------- profiling
// Launches are bracketed by HIP events on their stream while profiling is
// on; the events are resolved only when a report is asked for.
struct ProfEntry {
  double total_ms = 0;
  long count = 0;
};
struct PendingTiming {
  const char *name;
  hipEvent_t a, b;
};
extern bool g_profiling;
extern std::map<std::string, ProfEntry> g_prof;
extern std::vector<PendingTiming> g_pending;
extern std::vector<hipEvent_t> g_event_pool;

hipEvent_t pool_event();
void resolve_pending();

struct KernelTimer {
  hipStream_t s;
  const char *name;
  hipEvent_t a = nullptr, b = nullptr;
  bool on;
  KernelTimer(hipStream_t s_, const char *n, bool allowed = true)
      : s(s_), name(n), on(allowed && g_profiling) {
    if (on) {
      a = pool_event();
      b = pool_event();
      (void)hipEventRecord(a, s);
    }
  }
  ~KernelTimer() {
    if (on) {
      (void)hipEventRecord(b, s);
      g_pending.push_back({name, a, b});
      if (g_pending.size() > 4096) resolve_pending();
    }
  }
};

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }
// workgroup count padded to a multiple of the 8 XCDs (see wg_coords)
inline unsigned nblk8(long n, int bs) { return (nblk(n, bs) + 7u) & ~7u; }

}  // namespace enzoe

// --------------------------------------------------------------- method

struct enzoe_vlct_method {
  int mhd = 1;
  int riemann = ENZOE_KNS::RS_HLLD;
  int recon[2] = {ENZOE_KNS::RC_NN, ENZOE_KNS::RC_PLM};
  int nstages = 2;
  int precision = ENZOE_PREC_DOUBLE;
  // kernels launched in XCD-contiguous workgroup order (StageParams mask);
  // measured on the 256^3 Orszag-Tang block it pays for k_edge only
  int xcd_remap = 2;
  double theta = 1.5, courant = 0.3, gamma = 5.0 / 3.0;
  double dfloor = 1e-200, pfloor = 1e-200;
  // launch structure of the stages: for MHD constrained transport and the
  // cell update as three launches (0: k_edge, k_faces, k_cells) or fused
  // launches over tiles (1..4, ctu_variant); 5: each stage as one
  // persistent launch (k_stage, MHD or hydro); same bits every way; -1
  // (the default): the autotuner's choice per block shape, three launches
  // until it has run
  int ctu = -1;
  int force_ctu = -1;                    // set while the autotuner times one
  std::map<long long, int> tuned_ctu;    // the autotuner's choice per shape
  // the autotuner's choice between those separate launches (0) and a whole
  // stage as one launch (MARCH_STRUCTURE, TILE_STRUCTURE), per shape, ghost
  // depth and size of the launch (whole_key): which of them wins goes with
  // the number of blocks
  std::map<std::pair<long long, int>, int> tuned_whole;
  // rows of the tiled cell order per block shape (the autotuner's choice;
  // tile_rows_for otherwise) and the value forced while it times one
  std::map<long long, int> tuned_rows;
  int force_rows = -1;
  // the shape of the flux launch for blocks of this shape (flux_shape_of:
  // 0 three faces per thread, 1 one face per thread, 2 z pencils for the
  // nearest-neighbour stage): the autotuner's choice, the value forced
  // while it times one, and the method's setting (-1: the autotuner's)
  std::map<long long, int> tuned_shape;
  int force_shape = -1;
  int flux_shape = -1;
  // the persistent stage kernel's grid barrier (a GridBarrier in device
  // memory, zeroed once), or null until first needed
  void *d_bar = nullptr;
  // dual-energy formalism ("modern" formulation) and its eta
  int dual = 0;
  double eta = 0.001;

  // scratch pool (grown on demand)
  void *scratch = nullptr;
  size_t scratch_bytes = 0;
  // descriptor table
  void *d_desc = nullptr;
  size_t desc_bytes = 0;
  std::vector<char> last_desc;
  // the CFL minimum of a pass of its own and of device-driven cycles, whose
  // launches a caller's graph may hold and replay at any time
  unsigned long long *d_dt = nullptr;
  // the CFL minimum that a host-driven step takes, a word that no captured
  // work touches, and whether k_dt_out has left it ready for the next one
  unsigned long long *d_step_dt = nullptr;
  bool step_dt_ready = false;
  // a CFL minimum on its way to the host: a pinned word that k_dt_out writes
  // (null: not allocated)
  unsigned long long *h_dt = nullptr;
  void *d_ptrtab = nullptr;
  size_t ptrtab_bytes = 0;
  std::vector<char> last_dt_desc;  // host copy of the dt descriptor table
  void *d_rtab = nullptr;          // refresh pointer table
  size_t rtab_bytes = 0;
  std::vector<double *> last_rtab;
  size_t scratch_budget = 0;       // bytes of the chunk scratch pool
  bool dry = false;                // prepare buffers and tables, launch nothing
  // fixed workspace of the allocation-free entry point while it runs (the
  // descriptor table, then the stage scratch), or null
  char *arena = nullptr;
  size_t arena_bytes = 0;
  // launch-order mask chosen by enzoe_vlct_autotune per block shape, and a
  // mask forced while the autotuner times a candidate (-1: none)
  std::map<long long, int> tuned_mask;
  int force_mask = -1;
  void *d_dts = nullptr;  // per-block dt uploaded by enzoe_vlct_compute_dt
  size_t dts_bytes = 0;
  // device tables of the flux-correction calls (FluxData pointers of
  // enzoe_vlct_compute_store_fluxes, links of the batched send, blocks of
  // the batched correction), re-uploaded only when they change
  void *d_fdtab = nullptr, *d_fltab = nullptr, *d_fbtab = nullptr;
  size_t fdtab_bytes = 0, fltab_bytes = 0, fbtab_bytes = 0;
  std::vector<char> last_fdtab, last_fltab, last_fbtab;
  // debug counters (DBG_* in vlct_kernels.hpp): device memory while the
  // checks are on (enzoe_vlct_set_debug_checks), null otherwise
  unsigned long long *d_dbg = nullptr;
  // transfer tables of enzoe_vlct_transfer_batch: two, so that the
  // restriction and prolongation batches of a cycle both stay cached
  void *d_trtab[2] = {nullptr, nullptr};
  size_t trtab_bytes[2] = {0, 0};
  std::vector<char> last_trtab[2];
};

namespace ENZOE_KNS {
// the profiling helpers above stay in `enzoe` (one set for the library)
using namespace ::enzoe;


inline long long shape_key(int mx, int my, int mz) {
  return ((long long)mx << 40) | ((long long)my << 20) | (long long)mz;
}

// The launch structure of the stages for blocks of this shape where they do
// not run marched (march_ok): 0 = k_flux, then k_edge + k_faces + k_cells; for MHD 1..3 = k_ctu with tile
// CtuTile1..3, 4 = k_edge + k_ctu without its edge phase (faces and cells
// fused); 5 = the persistent k_stage (persistent_ok); the method's
// setting, or the autotuner's choice for the shape when the setting is
// "auto" (-1).  Until it has run, tile 32 x 4 x 2 for MHD below 2^19 cells,
// ghost zones included: those calls are bound by latency, and k_ctu is two
// launches fewer a stage (cycle of one FP64 block of 16^3: 93 against 77 us,
// of 32^3 100, 91, of 56^3 152, 143; 32 of 16^3 187, 177; 4 of 32^3 151, 153).
inline int ctu_variant(const enzoe_vlct_method *m, int mx, int my, int mz, int nb) {
  if (m->force_ctu >= 0) return m->force_ctu;
  if (m->ctu >= 0) return m->ctu;
  auto it = m->tuned_ctu.find(shape_key(mx, my, mz));
  if (it != m->tuned_ctu.end()) return it->second;
  return (m->mhd && m->nstages == 2 && (long)mx * my * mz * nb < (1L << 19)) ? 2 : 0;
}

// ... and, chosen by march_ok and tile_ok and not by enzoe_vlct_set_fused_ct,
// the marched stages and the tiled ones
constexpr int MARCH_STRUCTURE = 6, TILE_STRUCTURE = 7;

inline long active_cells(int mx, int my, int mz, int ghost) {
  return (long)(mx - 2 * ghost) * (my - 2 * ghost) * (mz - 2 * ghost);
}
// Key of tuned_whole: launches of one shape and ghost depth whose active
// cells lie in the same octave tune together; from 2^20 on (four waves a SIMD
// at a cell a thread) the device is full and they are all alike.
inline std::pair<long long, int> whole_key(int mx, int my, int mz, int ghost, int nb) {
  const unsigned long cells = (unsigned long)active_cells(mx, my, mz, ghost) * nb;
  int octave = 0;
  while (octave < 20 && (cells >> (octave + 1)) != 0) octave++;
  return {shape_key(mx, my, mz), ghost * 32 + octave};
}

// The fused CT update needs the two stages of the VL scheme (its final
// stage reads the first stage's copy of the start-of-step faces); the
// scratch holds that copy whenever the fused launch may be chosen.
inline bool ctu_possible(const enzoe_vlct_method *m) {
  return m->mhd && m->nstages == 2 && (m->ctu != 0 || m->force_ctu > 0);
}

// The persistent stage launch (structure 5) exists for HLLD MHD and for
// hydro without the dual-energy formalism, and not on the allocation-free
// path (its barrier is a buffer of the method).
inline bool persistent_ok(const enzoe_vlct_method *m) {
  return !m->dual && (!m->mhd || m->riemann == RS_HLLD) && m->arena == nullptr;
}

// The method's grid barrier, allocated and zeroed on first use (not while
// a graph is being captured: compute_group takes it before any launch,
// also in the dry run that precedes a capture).
inline int ensure_barrier(enzoe_vlct_method *m) {
  if (m->d_bar) return 0;
  void *p = nullptr;
  if (hipMalloc(&p, sizeof(GridBarrier)) != hipSuccess) return ENZOE_ERR_ALLOC;
  if (hipMemset(p, 0, sizeof(GridBarrier)) != hipSuccess) {
    (void)hipFree(p);
    return ENZOE_ERR_HIP;
  }
  m->d_bar = p;
  return 0;
}

// Workgroups of a persistent stage kernel the current device holds at once
// (occupancy x CUs), cached per device; 0 on failure.
template <typename FluxT, int RECON, int RIEMANN, bool MHD, bool PRIMF>
int stage_capacity() {
  static std::atomic<int> cap[16];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 0;
  int c = cap[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    int per = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, k_stage<FluxT, FluxT, RECON, RIEMANN, MHD, PRIMF>, 256, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    c = per * cus;
    cap[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

// One stage as one persistent launch: as many workgroups as the largest
// phase needs, at most what the device holds at once (a multiple of 8).
template <typename FluxT, int RECON, int RIEMANN, bool MHD, bool PRIMF>
int launch_stage(const enzoe_vlct_method *m, const BlockDesc<FluxT> *d, int nb,
                 const int nwg[4], StageParams sp, hipStream_t s) {
  const int cap = stage_capacity<FluxT, RECON, RIEMANN, MHD, PRIMF>() & ~7;
  if (cap < 8 || !m->d_bar) return ENZOE_ERR_HIP;
  long need = 0;
  for (int q = 0; q < 4; q++) need = std::max(need, (long)nwg[q] * nb);
  const int G = (int)std::min<long>(cap, std::max<long>(8, (need + 7) & ~7L));
  PersistParams pp;
  pp.nb = nb;
  for (int q = 0; q < 4; q++) pp.nwg[q] = nwg[q];
  pp.bar = (GridBarrier *)m->d_bar;
  pp.limit = 1u << 22;
  sp.xcd_remap = 0;  // the phases walk their boxes in the plain order
  hipLaunchKernelGGL((k_stage<FluxT, FluxT, RECON, RIEMANN, MHD, PRIMF>), dim3(G), dim3(256),
                     0, s, d, sp, pp);
  return 0;
}

template <typename FluxT, bool MHD>
int dispatch_stage(const enzoe_vlct_method *m, int recon, bool primf,
                   const BlockDesc<FluxT> *d, int nb, const int nwg[4],
                   const StageParams &sp, hipStream_t s) {
  constexpr int RS = MHD ? RS_HLLD : RS_HLLC;
  if constexpr (std::is_same<FluxT, float>::value) {
    if (primf) {
      if (recon == RC_NN) return launch_stage<FluxT, RC_NN, RS, MHD, true>(m, d, nb, nwg, sp, s);
      if (recon == RC_PLM)
        return launch_stage<FluxT, RC_PLM, RS, MHD, true>(m, d, nb, nwg, sp, s);
      return launch_stage<FluxT, RC_PLM_ATHENA, RS, MHD, true>(m, d, nb, nwg, sp, s);
    }
  }
  if (recon == RC_NN) return launch_stage<FluxT, RC_NN, RS, MHD, false>(m, d, nb, nwg, sp, s);
  if (recon == RC_PLM) return launch_stage<FluxT, RC_PLM, RS, MHD, false>(m, d, nb, nwg, sp, s);
  return launch_stage<FluxT, RC_PLM_ATHENA, RS, MHD, false>(m, d, nb, nwg, sp, s);
}
template <typename FluxT, bool DE, class Tile, bool EDGES_LDS = true>
void launch_ctu(const BlockDesc<FluxT> *d, int nb, int mx, int my, int mz, int lo,
                StageParams sp, hipStream_t s) {
  int nt[3];
  ctu_tiles<Tile>(mx, my, mz, lo, nt);
  const long tiles = (long)nt[0] * nt[1] * nt[2];
  hipLaunchKernelGGL((k_ctu<FluxT, DE, Tile, EDGES_LDS>),
                     dim3(nblk8(tiles * Tile::NT, Tile::NT), nb), dim3(Tile::NT), 0, s, d, sp);
}

inline int total_staling(int r) { return r == RC_NN ? 1 : 2; }
inline int immediate_staling(int r) { return r == RC_NN ? 0 : 1; }

inline int parse_recon(const std::string &n, int *out) {
  if (n == "nn") { *out = RC_NN; return 0; }
  if (n == "plm" || n == "plm_enzo") { *out = RC_PLM; return 0; }
  if (n == "plm_athena") { *out = RC_PLM_ATHENA; return 0; }
  return ENZOE_ERR_CONFIG;
}

// The mixed path (FP32 fluxes, no dual energy) keeps its half-step state as
// FP32 primitives.
template <typename FluxT>
inline constexpr bool half_f32(int dual) {
  return std::is_same<FluxT, float>::value && !dual;
}

// bytes of scratch per block
template <typename FluxT>
inline size_t scratch_per_block(int mx, int my, int mz, int mhd, int dual = 0, int ctu = 0) {
  size_t ncc = (size_t)mx * my * mz;
  size_t nq = mhd ? 8 : 5;
  size_t bytes = 0;
  // half-step state: FP64 integration quantities (Ut), or in the mixed path
  // FP32 primitives (Up)
  bytes += nq * ncc * (half_f32<FluxT>(dual) ? sizeof(float) : sizeof(double));
  if (mhd) {
    const size_t faces = ((size_t)mz * my * (mx + 1) + (size_t)mz * (my + 1) * mx +
                          (size_t)(mz + 1) * my * mx) * sizeof(double);
    bytes += faces;                                    // bft
    if (ctu) bytes += faces;                           // bf0
    bytes += 6 * ncc * sizeof(double);                 // E, Ec
    if (half_f32<FluxT>(dual)) bytes += 3 * ncc * sizeof(double);  // Ech
  }
  bytes += 3 * (mhd ? 7 : 5) * ncc * sizeof(FluxT);    // F
  if (dual) bytes += 7 * ncc * sizeof(double);         // eit, Fe, Vb
  return bytes;
}

inline int ensure_bytes(void **ptr, size_t *have, size_t need) {
  if (*have >= need) return 0;
  // work queued earlier may still read the old buffer
  if (*ptr) {
    (void)hipDeviceSynchronize();
    (void)hipFree(*ptr);
  }
  *ptr = nullptr;
  *have = 0;
  if (hipMalloc(ptr, need) != hipSuccess) return ENZOE_ERR_ALLOC;
  *have = need;
  return 0;
}

// Copies a host table to a device buffer unless the buffer already holds
// exactly these bytes; the stream is synchronised after a copy, so the
// host table may change as soon as the call returns.
inline int upload_table(void **dptr, size_t *have, std::vector<char> *last,
                        const void *host, size_t bytes, hipStream_t s) {
  const char *raw = (const char *)host;
  if (*dptr && last->size() == bytes && std::memcmp(last->data(), raw, bytes) == 0)
    return 0;
  if (int rc = ensure_bytes(dptr, have, bytes)) return rc;
  if (hipMemcpyAsync(*dptr, raw, bytes, hipMemcpyHostToDevice, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return ENZOE_ERR_HIP;
  last->assign(raw, raw + bytes);
  return 0;
}

inline int check_block(const enzoe_vlct_method *m, const enzoe_block &b) {
  if (b.mx < 7 || b.my < 7 || b.mz < 7) return ENZOE_ERR_ARG;
  // cell indices of the tiled order are 32-bit
  if ((long long)(b.mx + 1) * (b.my + 1) * (b.mz + 1) >= (1LL << 31)) return ENZOE_ERR_ARG;
  // EnzoMethodMHDVlct.cpp:124-133: ghost depth >= sum of staling rates
  int req = 0;
  for (int s = 0; s < m->nstages; s++) req += total_staling(m->recon[s]);
  if (b.ghost < req) return ENZOE_ERR_ARG;
  if (!b.density || !b.velocity[0] || !b.velocity[1] || !b.velocity[2] ||
      !b.total_energy)
    return ENZOE_ERR_ARG;
  if (m->mhd) {
    for (int d = 0; d < 3; d++)
      if (!b.bfield[d] || !b.bfieldi[d]) return ENZOE_ERR_ARG;
  }
  // the dual-energy formalism integrates the internal_energy field
  if (m->dual && !b.internal_energy) return ENZOE_ERR_ARG;
  return 0;
}

// Rows of the tiled cell order for a block with planes of mx x my cells:
// the largest of 64, 32, 16, 8 rows whose slab planes hold the flux
// kernel's z stencil (about 5 planes of 11 words per cell) in 2 MB, half an
// XCD's L2; 0 (plain order) when a whole plane of that already fits in 4 MB.
inline int tile_rows_for(int mx, int my) {
  const double row = (double)mx * 11 * 8 * 5;
  if (row * my <= double(4 << 20)) return 0;
  int rows = 64;
  while (rows > 8 && row * rows > double(2 << 20)) rows /= 2;
  return rows;
}


// The flux launch for blocks of this shape: 0, three faces per thread
// (k_flux); 1, one face per thread (k_flux over three z slices, for blocks
// too small to fill the device); 2, the nearest-neighbour stage as z
// pencils with LDS-staged planes (k_flux_zp; the other stages as 0).  The
// setting, else the autotuner's choice, else 1 for launches of fewer than
// 2^18 cells, ghost zones included (under 4 waves a SIMD with one cell a
// thread; cycle in us with 0 and 1: 16^3 MHD 77, 67, hydro 53, 48; 4 blocks of
// 32^3 153, 149 and 86, 83; equal at 56^3).
inline int flux_shape_of(const enzoe_vlct_method *m, int mx, int my, int mz, int nb) {
  if (m->force_shape >= 0) return m->force_shape;
  if (m->flux_shape >= 0) return m->flux_shape;
  auto it = m->tuned_shape.find(shape_key(mx, my, mz));
  if (it != m->tuned_shape.end()) return it->second;
  return (long)mx * my * mz * nb < (1L << 18) ? 1 : 0;
}

// Rows of the tiled cell order for blocks of this shape.
inline int tile_rows_of(const enzoe_vlct_method *m, int mx, int my, int mz) {
  if (m->force_rows >= 0) return m->force_rows;
  auto it = m->tuned_rows.find(shape_key(mx, my, mz));
  return it != m->tuned_rows.end() ? it->second : tile_rows_for(mx, my);
}

// Fills descriptors for blocks [b0, b1) into out[0 .. b1-b0), their scratch
// laid out from `base`.
// accel: 3 acceleration pointers per block of the call (x, y, z), or null
template <typename FluxT>
void fill_desc_at(const enzoe_vlct_method *m, char *base, const enzoe_block *blocks,
                  int b0, int b1, BlockDesc<FluxT> *out,
                  const double *const *accel = nullptr) {
  for (int bi = b0; bi < b1; bi++) {
    const enzoe_block &b = blocks[bi];
    BlockDesc<FluxT> d;
    std::memset(&d, 0, sizeof(d));
    d.U[S_RHO] = b.density;
    for (int a = 0; a < 3; a++) d.U[S_VX + a] = b.velocity[a];
    d.U[S_E] = b.total_energy;
    if (m->mhd)
      for (int a = 0; a < 3; a++) {
        d.U[S_BX + a] = b.bfield[a];
        d.bfi[a] = b.bfieldi[a];
      }
    d.pressure = b.pressure;
    d.mx = b.mx; d.my = b.my; d.mz = b.mz;
    d.g = b.ghost;
    d.tile_rows = tile_rows_of(m, b.mx, b.my, b.mz);
    if (accel)
      for (int a = 0; a < 3; a++) d.acc[a] = accel[3 * bi + a];
    for (int a = 0; a < 3; a++) d.cw[a] = b.cell_width[a];
    const size_t ncc = (size_t)b.mx * b.my * b.mz;
    const int nq = m->mhd ? 8 : 5;
    for (int q = 0; q < S_N; q++) {
      if (!m->mhd && q >= S_BX) continue;
      if (half_f32<FluxT>(m->dual)) {
        d.Up[q] = (float *)base;
        base += ncc * sizeof(float);
      } else {
        d.Ut[q] = (double *)base;
        base += ncc * sizeof(double);
      }
    }
    (void)nq;
    if (m->mhd) {
      d.bft[0] = (double *)base; base += (size_t)b.mz * b.my * (b.mx + 1) * sizeof(double);
      d.bft[1] = (double *)base; base += (size_t)b.mz * (b.my + 1) * b.mx * sizeof(double);
      d.bft[2] = (double *)base; base += (size_t)(b.mz + 1) * b.my * b.mx * sizeof(double);
      if (ctu_possible(m)) {
        d.bf0[0] = (double *)base; base += (size_t)b.mz * b.my * (b.mx + 1) * sizeof(double);
        d.bf0[1] = (double *)base; base += (size_t)b.mz * (b.my + 1) * b.mx * sizeof(double);
        d.bf0[2] = (double *)base; base += (size_t)(b.mz + 1) * b.my * b.mx * sizeof(double);
      }
      for (int a = 0; a < 3; a++) {
        d.E[a] = (double *)base;
        base += ncc * sizeof(double);
      }
      for (int a = 0; a < 3; a++) {
        d.Ec[a] = (double *)base;
        base += ncc * sizeof(double);
      }
      if (half_f32<FluxT>(m->dual))
        for (int a = 0; a < 3; a++) {
          d.Ech[a] = (double *)base;
          base += ncc * sizeof(double);
        }
    }
    for (int dd = 0; dd < 3; dd++) {
      for (int q = 0; q < S_N; q++) {
        if (!m->mhd && q >= S_BX) continue;
        if (m->mhd && q == S_BX + dd) continue;  // normal-B flux is 0
        d.F[dd][q] = (FluxT *)base;
        base += ncc * sizeof(FluxT);
      }
    }
    if (m->dual) {
      d.ei = b.internal_energy;
      d.eit = (double *)base;
      base += ncc * sizeof(double);
      for (int a = 0; a < 3; a++) {
        d.Fe[a] = (double *)base;
        base += ncc * sizeof(double);
        d.Vb[a] = (double *)base;
        base += ncc * sizeof(double);
      }
    }
    out[bi - b0] = d;
  }
}

// fill_desc_at over the method's scratch pool, into a vector
template <typename FluxT>
void fill_desc(const enzoe_vlct_method *m, const enzoe_block *blocks, int b0,
               int b1, std::vector<BlockDesc<FluxT>> &out,
               const double *const *accel = nullptr) {
  out.resize(b1 - b0);
  fill_desc_at<FluxT>(m, (char *)m->scratch, blocks, b0, b1, out.data(), accel);
}

// cells of the box [lo, m - hi_trim) of a block
inline long cube(int mx, int my, int mz, int lo, int hi_trim) {
  long a = mx - lo - hi_trim, b = my - lo - hi_trim, c = mz - lo - hi_trim;
  if (a <= 0 || b <= 0 || c <= 0) return 0;
  return a * b * c;
}

// flux launch of one stage; shape as flux_shape_of (2 applies to the
// nearest-neighbour reconstruction only)
template <typename FluxT, int RECON, int RIEMANN, bool MHD, bool DE, bool PRIMF>
void launch_flux(const BlockDesc<FluxT> *d, int nb, int mx, int my, int mz,
                 StageParams sp, hipStream_t s, int shape) {
  const int cs = sp.cur_stale;
  if (RECON == RC_NN && shape == 2) {
    // z pencils: ZP_TX x ZP_TY tiles, each marching through a segment of
    // planes; about 2048 workgroups per block
    const int nx = mx - 2 * cs, ny = my - 2 * cs, nz = mz - 2 * cs;
    const int tiles = ((nx + ZP_TX - 1) / ZP_TX) * ((ny + ZP_TY - 1) / ZP_TY);
    const int want = std::max(1, std::min(nz, (2048 + tiles - 1) / tiles));
    const int zplanes = (nz + want - 1) / want;
    const int nseg = (nz + zplanes - 1) / zplanes;
    hipLaunchKernelGGL((k_flux_zp<FluxT, FluxT, RIEMANN, MHD, DE, PRIMF>),
                       dim3(tiles * nseg, nb), dim3(256), 0, s, d, sp, zplanes);
    return;
  }
  const long nthreads = cube(mx, my, mz, cs, cs);
  dim3 grid(nblk8(nthreads, 256), nb, shape == 1 ? 3 : 1);
  hipLaunchKernelGGL((k_flux<FluxT, FluxT, RECON, RIEMANN, MHD, DE, PRIMF>), grid,
                     dim3(256), 0, s, d, sp);
}

template <typename FluxT, bool MHD, bool DE, bool PRIMF>
void dispatch_flux_p(const enzoe_vlct_method *m, int recon,
                     const BlockDesc<FluxT> *d, int nb, int mx, int my, int mz,
                     StageParams sp, hipStream_t s, int shape) {
  constexpr int RS = MHD ? RS_HLLD : RS_HLLC;
  if (MHD && m->riemann != RS_HLLD) {
    if (recon == RC_NN)
      launch_flux<FluxT, RC_NN, RS_HLLE, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
    else if (recon == RC_PLM)
      launch_flux<FluxT, RC_PLM, RS_HLLE, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
    else
      launch_flux<FluxT, RC_PLM_ATHENA, RS_HLLE, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
    return;
  }
  if (recon == RC_NN)
    launch_flux<FluxT, RC_NN, RS, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
  else if (recon == RC_PLM)
    launch_flux<FluxT, RC_PLM, RS, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
  else
    launch_flux<FluxT, RC_PLM_ATHENA, RS, MHD, DE, PRIMF>(d, nb, mx, my, mz, sp, s, shape);
}

// primf: the stage reads the mixed path's FP32 primitive half-step state;
// shape: flux_shape_of
template <typename FluxT, bool MHD, bool DE>
void dispatch_flux(const enzoe_vlct_method *m, int recon, bool primf,
                   const BlockDesc<FluxT> *d, int nb, int mx, int my, int mz,
                   StageParams sp, hipStream_t s, int shape) {
  if constexpr (half_f32<FluxT>(DE ? 1 : 0)) {
    if (primf) {
      dispatch_flux_p<FluxT, MHD, DE, true>(m, recon, d, nb, mx, my, mz, sp, s, shape);
      return;
    }
  }
  dispatch_flux_p<FluxT, MHD, DE, false>(m, recon, d, nb, mx, my, mz, sp, s, shape);
}

// gamma (gamma - 1) as the reference's synchronisation holds it: a float
// (EnzoPhysicsFluidProps.cpp:236)
inline double sync_ggm1(double gamma) {
  return (double)(float)(gamma * (gamma - 1.));
}


// XCD-order mask of the stage kernels for blocks of this shape
inline int launch_mask(const enzoe_vlct_method *m, int mx, int my, int mz) {
  if (m->force_mask >= 0) return m->force_mask;
  auto it = m->tuned_mask.find(shape_key(mx, my, mz));
  return it != m->tuned_mask.end() ? it->second : m->xcd_remap;
}

// Saving the final stage's face fluxes for flux corrections: the fields and
// the device table of one FluxData pointer per block of the call.
struct StoreArgs {
  StoreSlots sl;
  double *const *d_fdtab;
};

// ------------------------------------------------------- marched stages

// Whether the two stages of nb blocks of this shape run marched (k_march,
// k_march_hd): the VL scheme, fields whose byte offsets fit 32 bits, no debug
// counts (the marched tiles solve the faces of their rings more than once),
// and no structure or flux-launch shape asked for; then the autotuner's
// choice for launches like this one, or else from 2^18 active cells on (FP64
// hydro: 3 2^17).  Below that the launches are bound by latency, a plane after
// the other costs more than it saves, and the separate launches win.  Cycle
// in us, separate and marched -- MHD: 4 blocks of 32^3 158, 177; one of 48^3
// 137, 144; 8 of 32^3 229, 230; one of 64^3 202, 202; 4 of 48^3 293, 268; 16
// of 64^3 2180, 1545.  FP64 hydro: 8 of 32^3 123, 140; one of 64^3 106, 114;
// 16 of 32^3 201, 163.  Mixed hydro: 4 of 32^3 70, 75; one of 64^3 77, 76;
// 64 of 16^3 125, 107.
inline bool march_possible(const enzoe_vlct_method *m, int mx, int my, int mz) {
  return (!m->mhd || ctu_possible(m)) && m->nstages == 2 && !m->d_dbg &&
         8ull * (mx + 1) * (my + 1) * (mz + 1) < (1ull << 32);
}
inline bool march_ok(const enzoe_vlct_method *m, int mx, int my, int mz, int ghost, int nb) {
  if (!march_possible(m, mx, my, mz)) return false;
  if (m->force_ctu >= 0) return m->force_ctu == MARCH_STRUCTURE;
  if (m->ctu >= 0 || m->flux_shape >= 0) return false;
  auto it = m->tuned_whole.find(whole_key(mx, my, mz, ghost, nb));
  if (it != m->tuned_whole.end()) return it->second == MARCH_STRUCTURE;
  const bool light = m->mhd || m->precision == ENZOE_PREC_MIXED;
  return active_cells(mx, my, mz, ghost) * nb >= (light ? 1L << 18 : 3L << 17);
}

// Compute units of the current device, cached per device; 256 if unknown.
inline int device_cus() {
  static std::atomic<int> cus[16];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
  int c = cus[dev].load(std::memory_order_relaxed);
  if (c == 0) {
    if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        c <= 0)
      c = 256;
    cus[dev].store(c, std::memory_order_relaxed);
  }
  return c;
}

// The tiling of one marched stage over nb blocks with NT-thread workgroups,
// PER of them on a CU: the tile that covers the update box of a plane with
// the fewest workgroups (ties: the longer rows), and the workgroups' shares
// of the planes.  cost: the launch's time in units of one plane of 512
// threads a CU with the device full; a piece of work costs 3 planes more
// than it updates (the flux work of the planes around it, and its start).
template <int NT, int PER, bool MHD>
MarchParams march_tiling(int mx, int my, int mz, int cs, int nb, int cus, double &cost) {
  constexpr double UNIT = NT * PER / 512.0;
  const int nx = mx - 2 * (cs + 1), ny = my - 2 * (cs + 1), nz = mz - 2 * (cs + 1);
  MarchParams p{};
  long tiles = -1;
  for (int w2 = 10; w2 <= NT / 9; w2++) {
    if (w2 > nx + 2 && tiles >= 0) break;
    int h2 = std::min(NT / w2, ny + 2);
    while ((w2 + 2) * (h2 + 2) > march_plane_cells<MHD>(NT)) h2--;
    const int ntx = (nx + w2 - 3) / (w2 - 2), nty = (ny + h2 - 3) / (h2 - 2);
    if (tiles < 0 || (long)ntx * nty <= tiles) {
      tiles = (long)ntx * nty;
      p.w2 = w2;
      p.h2 = h2;
      p.ntx = ntx;
      p.nty = nty;
    }
  }
  p.nz = nz;
  const long slots = (long)cus * PER;
  // even shares over the whole launch (the rings then come from memory
  // instead of the L2: about an eighth more time a plane)
  p.zseg = nz;
  p.nseg = 1;
  p.total = tiles * nz * nb;
  p.share = (int)std::min<long>(std::max<long>((p.total + slots - 1) / slots, 4), INT_MAX);
  cost = 1.12 * UNIT * (p.share + 3.0 * (1.0 + (double)p.share / nz));
  // or a segment of a tile to a workgroup, in rounds over the device
  for (int seg = 1; seg <= std::max(1, nz / 4); seg++) {
    const int zseg = (nz + seg - 1) / seg;
    const long wgs = tiles * seg * nb;
    const double c = UNIT * (double)((wgs + slots - 1) / slots) * (zseg + 3);
    if (c < cost) {
      cost = c;
      p.zseg = p.share = zseg;
      p.nseg = (nz + zseg - 1) / zseg;
      p.total = tiles * p.nseg * nb * (long)zseg;
    }
  }
  return p;
}

template <typename T, int RECON, int RIEMANN, bool DE, bool HALF, int NT, int WAVES>
void launch_march_nt(const BlockDesc<T> *d, const MarchParams &mp, const StageParams &sp,
                     hipStream_t s) {
  const unsigned wgs = (unsigned)((mp.total + mp.share - 1) / mp.share);
  hipLaunchKernelGGL((k_march<T, RECON, RIEMANN, DE, HALF, NT, WAVES>), dim3((wgs + 7u) & ~7u),
                     dim3(NT), 0, s, d, sp, mp);
}
// One marched stage: 512-thread tiles, one a CU, or 256-thread ones, two a
// CU, whichever covers the blocks' planes in less time (the smaller tile
// repeats more of its ring but fits small blocks better).  The mixed
// nearest-neighbour march fits three waves a SIMD (168 registers, 120 KB of
// LDS): 768-thread tiles or three of 256.  Its Orszag-Tang 256^3 stage took
// 1.20 ms with two waves, 1.09 with three; the reconstructing one would spill
// 36 registers.
template <typename T, int RECON, int RIEMANN, bool DE, bool HALF>
void launch_march(const BlockDesc<T> *d, int nb, int mx, int my, int mz, const StageParams &sp,
                  hipStream_t s) {
  const int cus = device_cus();
  double big, small;
  constexpr int W = std::is_same<T, float>::value && RECON == RC_NN && !DE ? 3 : 2;
  constexpr int NT = 256 * W;
  const MarchParams p5 = march_tiling<NT, 1, true>(mx, my, mz, sp.cur_stale, nb, cus, big);
  const MarchParams p2 = march_tiling<256, W, true>(mx, my, mz, sp.cur_stale, nb, cus, small);
  if (big <= small)
    launch_march_nt<T, RECON, RIEMANN, DE, HALF, NT, W>(d, p5, sp, s);
  else
    launch_march_nt<T, RECON, RIEMANN, DE, HALF, 256, W>(d, p2, sp, s);
}
template <typename T, int RIEMANN, bool DE>
void dispatch_march(int recon, const BlockDesc<T> *d, int nb, int mx, int my, int mz,
                    const StageParams &sp, hipStream_t s) {
  if (sp.stage == 0)
    launch_march<T, RC_NN, RIEMANN, DE, false>(d, nb, mx, my, mz, sp, s);
  else if (recon == RC_NN)
    launch_march<T, RC_NN, RIEMANN, DE, true>(d, nb, mx, my, mz, sp, s);
  else if (recon == RC_PLM)
    launch_march<T, RC_PLM, RIEMANN, DE, true>(d, nb, mx, my, mz, sp, s);
  else
    launch_march<T, RC_PLM_ATHENA, RIEMANN, DE, true>(d, nb, mx, my, mz, sp, s);
}

template <typename T, int RECON, bool DE, bool HALF, int NT, int PER>
void launch_march_hd_nt(const BlockDesc<T> *d, const MarchParams &mp, const StageParams &sp,
                        hipStream_t s) {
  const unsigned wgs = (unsigned)((mp.total + mp.share - 1) / mp.share);
  hipLaunchKernelGGL((k_march_hd<T, RECON, DE, HALF, NT, NT * PER / 256>),
                     dim3((wgs + 7u) & ~7u), dim3(NT), 0, s, d, sp, mp);
}
// The tiles of the hydrodynamic march by what its registers allow: 167 in the
// FP64 reconstructing stage (three waves a SIMD: one workgroup of 768 on a
// CU), 124 in FP64 nearest neighbour and the mixed reconstructing one (four:
// two of 512), 81 in mixed nearest neighbour (six: three of 512); with
// dual energy the reconstructing stage takes 192 (two: one of 512).  Beside
// them 256-thread tiles, as many on a CU.  8 blocks of 128^3, FP64, PLM
// stage: 1.17 ms with 768, 1.21 with 512, 1.31 with 256, 1.69 with two of
// 384 (whose registers spill).
template <typename T, int RECON, bool DE, bool HALF, int NT, int PER, int NT2, int PER2>
void launch_march_hd_of(const BlockDesc<T> *d, int nb, int mx, int my, int mz,
                        const StageParams &sp, hipStream_t s) {
  const int cus = device_cus();
  double big, small;
  const MarchParams p = march_tiling<NT, PER, false>(mx, my, mz, sp.cur_stale, nb, cus, big);
  const MarchParams q = march_tiling<NT2, PER2, false>(mx, my, mz, sp.cur_stale, nb, cus, small);
  if (big <= small)
    launch_march_hd_nt<T, RECON, DE, HALF, NT, PER>(d, p, sp, s);
  else
    launch_march_hd_nt<T, RECON, DE, HALF, NT2, PER2>(d, q, sp, s);
}
template <typename T, int RECON, bool DE, bool HALF>
void launch_march_hd(const BlockDesc<T> *d, int nb, int mx, int my, int mz,
                     const StageParams &sp, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    if constexpr (RECON == RC_NN)
      launch_march_hd_of<T, RECON, DE, HALF, 512, 3, 256, 6>(d, nb, mx, my, mz, sp, s);
    else
      launch_march_hd_of<T, RECON, DE, HALF, 512, 2, 256, 4>(d, nb, mx, my, mz, sp, s);
  } else {
    if constexpr (RECON == RC_NN)
      launch_march_hd_of<T, RECON, DE, HALF, 512, 2, 256, 4>(d, nb, mx, my, mz, sp, s);
    else if constexpr (DE)
      launch_march_hd_of<T, RECON, DE, HALF, 512, 1, 256, 2>(d, nb, mx, my, mz, sp, s);
    else
      launch_march_hd_of<T, RECON, DE, HALF, 768, 1, 256, 3>(d, nb, mx, my, mz, sp, s);
  }
}
template <typename T, bool DE>
void dispatch_march_hd(int recon, const BlockDesc<T> *d, int nb, int mx, int my, int mz,
                       const StageParams &sp, hipStream_t s) {
  if (sp.stage == 0)
    launch_march_hd<T, RC_NN, DE, false>(d, nb, mx, my, mz, sp, s);
  else if (recon == RC_NN)
    launch_march_hd<T, RC_NN, DE, true>(d, nb, mx, my, mz, sp, s);
  else if (recon == RC_PLM)
    launch_march_hd<T, RC_PLM, DE, true>(d, nb, mx, my, mz, sp, s);
  else
    launch_march_hd<T, RC_PLM_ATHENA, DE, true>(d, nb, mx, my, mz, sp, s);
}

// Whether a hydrodynamic stage of small blocks is one launch of k_tile: a
// scheme of two stages (the one stage of the other updates the state in
// place, which tiles beside it still read), no debug counts (the faces between
// tiles are solved twice), and no structure or flux-launch shape asked for;
// then the autotuner's choice for launches like this one, or else fewer than
// 2^16 cells with ghosts (dual energy: 2^15), where a launch costs more than
// the repeated faces.  Cycle in
// us, separate and tiled -- FP64: one block of 12^3 38.4, 36.0; 16^3 39.1,
// 36.1; 24^3 41.7, 37.0; 32^3 (54872 cells) 48.4, 45.7; 8 of 16^3 (85184)
// 54.8, 57.5; 48^3 65.9, 70.8.  Dual energy: 24^3 44.2, 38.6; 32^3 51.9, 52.3.
// Mixed: 16^3 35.8, 30.8; 32^3 40.2, 36.7; 8 of 16^3 46.5, 46.0.
inline bool tile_possible(const enzoe_vlct_method *m, int mx, int my, int mz) {
  return !m->mhd && m->nstages == 2 && !m->d_dbg && std::min(mx, std::min(my, mz)) >= 7;
}
inline bool tile_ok(const enzoe_vlct_method *m, int mx, int my, int mz, int ghost, int nb) {
  if (!tile_possible(m, mx, my, mz)) return false;
  if (m->force_ctu >= 0) return m->force_ctu == TILE_STRUCTURE;
  if (m->force_shape >= 0 || m->ctu >= 0 || m->flux_shape >= 0) return false;
  auto it = m->tuned_whole.find(whole_key(mx, my, mz, ghost, nb));
  if (it != m->tuned_whole.end()) return it->second == TILE_STRUCTURE;
  return (long)mx * my * mz * nb < (m->dual ? 1L << 15 : 1L << 16);
}
template <typename FluxT, bool DE>
void dispatch_tile(int recon, bool primf, const BlockDesc<FluxT> *d, int nb, int mx, int my,
                   int mz, int lo, const StageParams &sp, hipStream_t s) {
  using Tile = FluxTile<FluxT>;
  const dim3 grid(((mx - 2 * lo + Tile::TX - 1) / Tile::TX) *
                      ((my - 2 * lo + Tile::TY - 1) / Tile::TY) *
                      ((mz - 2 * lo + Tile::TZ - 1) / Tile::TZ),
                  nb);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(576), 0, s, d, sp);
  };
  constexpr bool F32 = half_f32<FluxT>(DE ? 1 : 0);
  if (F32 && primf) {
    if (recon == RC_NN) launch(k_tile<FluxT, FluxT, RC_NN, DE, F32>);
    else if (recon == RC_PLM) launch(k_tile<FluxT, FluxT, RC_PLM, DE, F32>);
    else launch(k_tile<FluxT, FluxT, RC_PLM_ATHENA, DE, F32>);
  } else {
    if (recon == RC_NN) launch(k_tile<FluxT, FluxT, RC_NN, DE, false>);
    else if (recon == RC_PLM) launch(k_tile<FluxT, FluxT, RC_PLM, DE, false>);
    else launch(k_tile<FluxT, FluxT, RC_PLM_ATHENA, DE, false>);
  }
}

// Bytes of the chunk scratch pool: the larger of 4 GiB and a third of the
// free device memory, at most 16 GiB (taken once per method).
inline size_t scratch_budget(enzoe_vlct_method *m) {
  if (m->scratch_budget == 0) {
    size_t budget = (size_t)4 << 30;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess)
      budget = std::max(budget, std::min((size_t)16 << 30, free_b / 3));
    m->scratch_budget = budget;
  }
  return m->scratch_budget;
}

// The launch sequence of compute_group over chunks of `chunk` blocks whose
// descriptors are table[0 .. n) in device memory.  timers: bracket the
// kernels with profiling events (when profiling is on).
template <typename FluxT, bool MHD, bool DE>
int launch_chunks(enzoe_vlct_method *m, const enzoe_block *blocks, int n, int chunk,
                  const BlockDesc<FluxT> *table, double dt, const double *dts,
                  hipStream_t s, const StoreArgs *st, unsigned long long *cfl,
                  bool timers) {
  const int mx = blocks[0].mx, my = blocks[0].my, mz = blocks[0].mz;
  // (stored fluxes come from the separate launches' flux arrays)
  const bool march =
      !st && march_ok(m, mx, my, mz, blocks[0].ghost, std::min(n, chunk));
  const bool tile =
      !MHD && !st && !march && tile_ok(m, mx, my, mz, blocks[0].ghost, std::min(n, chunk));
  for (int c0 = 0; c0 < n; c0 += chunk) {
    const int c1 = std::min(n, c0 + chunk);
    const int nb = c1 - c0;
    const BlockDesc<FluxT> *d = table + c0;

    int stale = 0;
    for (int stage = 0; stage < m->nstages; stage++) {
      const bool is_final = (stage + 1) == m->nstages;
      const int recon = m->recon[stage];
      StageParams sp;
      sp.stage = stage;
      sp.is_final = is_final ? 1 : 0;
      sp.stale = stale;
      sp.cur_stale = stale + immediate_staling(recon);
      // EnzoMethodMHDVlct.cpp:462: dt/2 for the partial step
      sp.dt = (!is_final) ? dt / 2. : dt;
      sp.dts = dts ? dts + c0 : nullptr;
      sp.dt_factor = (!is_final) ? 0.5 : 1.0;
      sp.gamma = m->gamma;
      sp.igm1 = 1. / (m->gamma - 1.);
      sp.density_floor = m->dfloor;
      sp.pressure_floor = m->pfloor;
      sp.theta = m->theta;
      sp.xcd_remap = launch_mask(m, mx, my, mz);
      sp.eta = m->eta;
      sp.ggm1 = sync_ggm1(m->gamma);
      sp.cfl = is_final ? cfl : nullptr;
      sp.dbg = m->d_dbg;
      const int cs = sp.cur_stale;
      const bool primf = stage > 0 && half_f32<FluxT>(DE ? 1 : 0);
      // with the fused CFL the final update's launch covers the block
      const int lo = sp.cfl ? 0 : (is_final ? cs : cs + 1);
      const int structure = ctu_variant(m, mx, my, mz, nb);
      if (march) {
        {
          KernelTimer kt(s, recon == RC_NN ? "k_march_nn" : "k_march_plm", timers);
          if constexpr (!MHD)
            dispatch_march_hd<FluxT, DE>(recon, d, nb, mx, my, mz, sp, s);
          else if (m->riemann == RS_HLLD)
            dispatch_march<FluxT, RS_HLLD, DE>(recon, d, nb, mx, my, mz, sp, s);
          else
            dispatch_march<FluxT, RS_HLLE, DE>(recon, d, nb, mx, my, mz, sp, s);
        }
        if (is_final && (MHD || sp.cfl)) {
          // the cells around the update: ring centre B, CFL, pressure
          const int blo = sp.cfl ? 0 : cs;
          const long shell = cube(mx, my, mz, blo, blo) - cube(mx, my, mz, cs + 1, cs + 1);
          KernelTimer kt(s, "k_shell", timers);
          hipLaunchKernelGGL((k_shell<FluxT, MHD, DE>), dim3(nblk(shell, 256), nb), dim3(256), 0,
                             s, d, sp);
        }
        stale += total_staling(recon);
        continue;
      }
      if constexpr (!MHD) {
        if (tile) {
          KernelTimer kt(s, recon == RC_NN ? "k_tile_nn" : "k_tile_plm", timers);
          dispatch_tile<FluxT, DE>(recon, primf, d, nb, mx, my, mz, lo, sp, s);
          stale += total_staling(recon);
          continue;
        }
      }
      if constexpr (!DE) {
        if (structure == 5 && persistent_ok(m) && m->d_bar) {
          // the stage's four kernels as one persistent launch
          const int nwg[4] = {(int)nblk(cube(mx, my, mz, cs, cs), 256),
                              (int)nblk(cube(mx, my, mz, cs, cs), 256),
                              (int)nblk(cube(mx, my, mz, cs + 1, cs), 256),
                              (int)nblk(cube(mx, my, mz, lo, lo), 256)};
          KernelTimer kt(s, recon == RC_NN ? "k_stage_nn" : "k_stage_plm", timers);
          if (int rc = dispatch_stage<FluxT, MHD>(m, recon, primf, d, nb, nwg, sp, s)) return rc;
          stale += total_staling(recon);
          continue;
        }
      }
      {
        KernelTimer kt(s, recon == RC_NN ? "k_flux_nn" : "k_flux_plm", timers);
        dispatch_flux<FluxT, MHD, DE>(m, recon, primf, d, nb, mx, my, mz, sp, s,
                                      flux_shape_of(m, mx, my, mz, nb));
      }
      const int variant =
          (MHD && ctu_possible(m) && structure >= 1 && structure <= 4) ? structure : 0;
      if (variant == 4) {
        {
          KernelTimer kt(s, "k_edge", timers);
          hipLaunchKernelGGL((k_edge<FluxT>), dim3(nblk8(cube(mx, my, mz, cs, cs), 256), nb),
                             dim3(256), 0, s, d, sp);
        }
        KernelTimer kt(s, "k_fc", timers);
        launch_ctu<FluxT, DE, CtuTile1, false>(d, nb, mx, my, mz, lo, sp, s);
      } else if (variant > 0) {
        KernelTimer kt(s, "k_ctu", timers);
        if (variant == 2)
          launch_ctu<FluxT, DE, CtuTile2>(d, nb, mx, my, mz, lo, sp, s);
        else if (variant == 3)
          launch_ctu<FluxT, DE, CtuTile3>(d, nb, mx, my, mz, lo, sp, s);
        else
          launch_ctu<FluxT, DE, CtuTile1>(d, nb, mx, my, mz, lo, sp, s);
      } else {
        if (MHD) {
          {
            KernelTimer kt(s, "k_edge", timers);
            hipLaunchKernelGGL((k_edge<FluxT>), dim3(nblk8(cube(mx, my, mz, cs, cs), 256), nb),
                               dim3(256), 0, s, d, sp);
          }
          {
            KernelTimer kt(s, "k_faces", timers);
            hipLaunchKernelGGL((k_faces<FluxT>),
                               dim3(nblk8(cube(mx, my, mz, cs + 1, cs), 256), nb), dim3(256),
                               0, s, d, sp);
          }
        }
        KernelTimer kt(s, "k_cells", timers);
        hipLaunchKernelGGL((k_cells<FluxT, MHD, DE>),
                           dim3(nblk8(cube(mx, my, mz, lo, lo), 256), nb), dim3(256), 0,
                           s, d, sp);
      }
      stale += total_staling(recon);
    }
    if (st) {
      // the chunk's flux scratch still holds the final stage's fluxes
      long work = 0;
      for (int bi = c0; bi < c1; bi++) {
        const int g = blocks[bi].ghost;
        FluxLayout L;
        L.init(mx - 2 * g, my - 2 * g, mz - 2 * g);
        work = std::max(work, L.per_field * st->sl.nf);
      }
      KernelTimer kt(s, "k_store_fluxes", timers);
      hipLaunchKernelGGL((k_store_fluxes<FluxT>), dim3(nblk8(work, 256), nb),
                         dim3(256), 0, s, d, st->d_fdtab + c0, st->sl, dt,
                         dts ? dts + c0 : nullptr);
    }
  }
  if (hipGetLastError() != hipSuccess) return ENZOE_ERR_HIP;
  return 0;
}

// One VL+CT step (EnzoMethodMHDVlct::compute) on blocks of equal shape.
// dts: per-block dt in device memory (n values) or null (all blocks use dt).
// st: store the final stage's face fluxes (hydro only) or null.
// DE: the dual-energy formalism (FP64 path only).
// cfl (non-null): the final stage's k_cells also takes the CFL minimum of
// its cells and writes their pressure.
template <typename FluxT, bool MHD, bool DE = false>
int compute_group(enzoe_vlct_method *m, const enzoe_block *blocks, int n,
                  double dt, const double *dts, hipStream_t s,
                  const StoreArgs *st = nullptr,
                  const double *const *accel = nullptr,
                  unsigned long long *cfl = nullptr) {
  const int mx = blocks[0].mx, my = blocks[0].my, mz = blocks[0].mz;
  if (DE != (m->dual != 0)) return ENZOE_ERR_CONFIG;
  const size_t per = scratch_per_block<FluxT>(mx, my, mz, m->mhd, m->dual, ctu_possible(m));
  if (m->arena) {
    // the allocation-free path: descriptor table and scratch in the fixed
    // workspace; nothing is allocated, nothing cached across calls
    const size_t dbytes = ((size_t)n * sizeof(BlockDesc<FluxT>) + 255) & ~(size_t)255;
    if (dbytes >= m->arena_bytes || m->arena_bytes - dbytes < per) return ENZOE_ERR_SIZE;
    const int chunk =
        (int)std::max<size_t>(1, std::min<size_t>(n, (m->arena_bytes - dbytes) / per));
    std::vector<BlockDesc<FluxT>> desc(n);
    for (int c0 = 0; c0 < n; c0 += chunk)
      fill_desc_at<FluxT>(m, m->arena + dbytes, blocks, c0, std::min(n, c0 + chunk),
                          desc.data() + c0, accel);
    if (hipMemcpyAsync(m->arena, desc.data(), n * sizeof(BlockDesc<FluxT>),
                       hipMemcpyHostToDevice, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return ENZOE_ERR_HIP;
    return launch_chunks<FluxT, MHD, DE>(m, blocks, n, chunk, (const BlockDesc<FluxT> *)m->arena,
                                         dt, dts, s, st, cfl, false);
  }
  // chunk size: as many blocks as fit the scratch budget (at least 1); the
  // chunks run one after the other on the stream and share the pool
  const size_t budget = scratch_budget(m);
  int chunk = (int)std::max<size_t>(1, std::min<size_t>(n, budget / per));
  if (int rc = ensure_bytes(&m->scratch, &m->scratch_bytes, per * chunk)) return rc;

  // descriptor table of every chunk, uploaded once (and only when changed)
  std::vector<BlockDesc<FluxT>> desc, part;
  for (int c0 = 0; c0 < n; c0 += chunk) {
    fill_desc<FluxT>(m, blocks, c0, std::min(n, c0 + chunk), part, accel);
    desc.insert(desc.end(), part.begin(), part.end());
  }
  {
    const size_t dbytes = desc.size() * sizeof(BlockDesc<FluxT>);
    const char *raw = (const char *)desc.data();
    bool same = (m->last_desc.size() == dbytes) &&
                std::memcmp(m->last_desc.data(), raw, dbytes) == 0;
    if (!same) {
      if (int rc = ensure_bytes(&m->d_desc, &m->desc_bytes, dbytes)) return rc;
      if (hipMemcpyAsync(m->d_desc, raw, dbytes, hipMemcpyHostToDevice, s) !=
          hipSuccess)
        return ENZOE_ERR_HIP;
      // the host copy must stay valid until the copy has been consumed
      if (hipStreamSynchronize(s) != hipSuccess) return ENZOE_ERR_HIP;
      m->last_desc.assign(raw, raw + dbytes);
    }
  }
  if (!DE && persistent_ok(m) && (m->ctu == -1 || m->ctu == 5 || m->force_ctu == 5))
    if (int rc = ensure_barrier(m)) return rc;
  if (m->dry) return 0;
  return launch_chunks<FluxT, MHD, DE>(m, blocks, n, chunk,
                                       (const BlockDesc<FluxT> *)m->d_desc, dt, dts, s, st,
                                       cfl, true);
}

// The launch sequence of n blocks (chunks of `chunk`) of the FP32 flux path
// over a descriptor table prepared in device memory, per-block dt in dts
// (device); compiled in vlct_mixed.hip.
int launch_prepared_mixed(enzoe_vlct_method *m, const enzoe_block *blocks, int n, int chunk,
                          const void *table, const double *dts, hipStream_t s);

// FP32 flux path, compiled in vlct_mixed.hip
int compute_mixed(enzoe_vlct_method *m, const enzoe_block *blocks, int n,
                  double dt, const double *dts, hipStream_t s,
                  const StoreArgs *st = nullptr,
                  const double *const *accel = nullptr,
                  unsigned long long *cfl = nullptr);

}  // namespace ENZOE_KNS

namespace enzoe {

// FP64 step with multiply-adds contracted into FMAs, compiled in
// vlct_fp64c.hip: compute_runs' and the prepared launch sequence's
// counterparts (st: the StoreArgs of the flux store, or null)
int compute_contracted(enzoe_vlct_method *m, const enzoe_block *blocks, int n, double dt,
                       const double *dts, hipStream_t s, const void *st,
                       const double *const *accel, unsigned long long *cfl);
int launch_prepared_contracted(enzoe_vlct_method *m, const enzoe_block *blocks, int n,
                               int chunk, const void *table, const double *dts,
                               hipStream_t s);

}  // namespace enzoe
