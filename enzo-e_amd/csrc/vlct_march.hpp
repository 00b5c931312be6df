// vlct_march.hpp -- one stage of the VL+CT step as one launch whose
// workgroups march tiles of columns up through the planes of a block.
//
// The separate launches (k_flux, k_edge, k_faces, k_cells) write 24 words per
// cell and stage (fluxes, centre E, edge EMFs) to memory and read about 46
// back, and every cell's state is loaded and converted to primitives four
// to ten times and every slope limited twice.  k_march keeps all of that on
// the chip: a thread owns one column, a workgroup a tile of columns with one
// ring of columns around it (constrained transport needs the fluxes of the
// ring), and the planes go by one after the other.  A step of the march, at
// plane k:
//   z   the face below plane k, from the column's own left state (kept from
//       the last step) and the slope of this plane's cell;
//   x,y the faces towards i + 1 and j + 1, the neighbour's right state
//       through LDS;
//   E   the edge EMFs of plane k (E_z) and of the level below it (E_x, E_y);
//   B   the faces of plane k - 1 and the level between, from those EMFs;
//   U   the cell of plane k - 1.
// The expressions are the ones of the separate kernels (solve_face,
// edge_value, face_b_update, cell_finish), so the results are the same bits,
// FP64 and mixed (in the contracted build the compiler fuses them as it finds
// them in each kernel).
//
// What bounds it: FP64 instruction issue.  A 256^3 block's stages execute
// 2020 (nearest neighbour) and 2400 (PLM) VALU instructions a column and
// plane, a quarter of them for the rings (512 threads of 34 x 15 columns
// cover 32 x 13 cells), at about two thirds of the issue rate; the rest is
// waiting at the 4 (NN) or 6 (PLM) barriers of a plane and on dependent
// operations with two waves a SIMD, all that 256 registers and 119 or 147 KB
// of LDS allow.  The mixed path has registers over, and waits for memory and
// on dependent operations too: three waves a SIMD in its first stage, one
// barrier and a load of the column's cell less (LATE, CARRY below).
// Orszag-Tang 256^3, FP64: 1.88 + 2.60 ms for the two stages against 3.19 +
// 3.82 of the separate launches; mixed 1.09 + 1.64 against 2.35 + 2.23; 64
// turbulence blocks of 64^3: 2.28 + 2.72 against 3.87 + 4.19 (FP64), 1.43 +
// 1.79 (mixed).
#pragma once

#include "vlct_kernels.hpp"

namespace ENZOE_KNS {

// The work of a launch is the planes of every tile of every block in one
// row, ordered by block, segment of planes, tile and plane; workgroup g takes
// the `share` planes from g * share, in one piece for each (segment, tile)
// they touch.  share = zseg: a workgroup does one segment of one tile, and
// neighbouring tiles run beside each other, which share their rings in the
// L2.  One segment and another share: every workgroup has the same number of
// planes however the tiles come out.
struct MarchParams {
  int w2, h2;      // threads of a tile along x and y (its columns + the ring)
  int ntx, nty;    // tiles along x and y
  int nz;          // updated planes of a block
  int zseg, nseg;  // planes of a segment, segments
  int share;       // planes of a workgroup
  long total;      // planes of the launch (segments counted whole)
};

// Cells of the LDS plane of a reconstructing march (the tile, its ring and
// one more cell around; MHD: one less, with dual energy the FP64 march fills
// the 160 KB).
template <bool MHD>
constexpr int march_plane_cells(int nt) {
  return nt + nt / 4 - (MHD ? 1 : 0);
}

// dU - dtdx (F_hi - F_lo), never contracted (cell_stage's divergence).
__device__ __forceinline__ double flux_difference(double dU, double dtdx, double hi, double lo) {
#pragma clang fp contract(off)
  return dU - dtdx * (hi - lo);
}
__device__ __forceinline__ double source_difference(double dU, double dtdx, double p, double hi,
                                                    double lo) {
#pragma clang fp contract(off)
  return dU - dtdx * p * (hi - lo);
}
__device__ __forceinline__ double half_sum(double a, double b) {
#pragma clang fp contract(off)
  return 0.5 * (a + b);
}

// A value that every lane holds, in scalar registers.
__device__ __forceinline__ double uniform(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Waits for the workgroup's LDS accesses only: global loads issued ahead
// stay in flight (a workgroup's threads exchange nothing through memory).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// PLM states of a cell's two faces along one axis from its neighbours am,
// ap: lo = a - s/2 (its low face), hi = a + s/2, floored for a density
// or pressure.  EXACT = false (FP64, the Enzo limiter): for values whose
// magnitudes are below MARCH_TAME, so that no difference overflows or is NaN:
// the limiter's sign factor from the sign bits and the floors by the
// hardware maximum, 11 instructions instead of 22 a slope.  The values are
// those of the general form but for the sign of a zero.
constexpr double MARCH_TAME = 0x1p996;
template <int RECON, bool EXACT, typename T>
__device__ __forceinline__ void march_states(int q, T am, T a, T ap, T theta,
                                             const FluxConsts &fc, T &lo, T &hi) {
  T s;
  if constexpr (RECON == RC_PLM_ATHENA) {
    s = limiter_athena(am, a, ap);
  } else if constexpr (EXACT || std::is_same<T, float>::value) {
    s = limiter_enzo(am, a, ap, theta);
  } else {
    const double c = 0.5 * (ap - am), l = (a - am) * theta, r = (ap - a) * theta;
    const double m = __builtin_fmin(__builtin_fmin(fabs(l), fabs(r)), fabs(c));
    const bool same = (__double2hiint(l) ^ __double2hiint(r)) >= 0;
    s = same ? copysign(m, l) : 0.0;
  }
  lo = a - s * T(0.5);
  hi = a + s * T(0.5);
  if (q == S_RHO || q == S_E) {
    const T f = (T)(q == S_RHO ? fc.dfloor : fc.pfloor);
    if constexpr (EXACT) {
      lo = dmax(lo, f);
      hi = dmax(hi, f);
    } else {
      lo = fmax(lo, f);
      hi = fmax(hi, f);
    }
  }
}
// Whether a cell's state is outside the range of EXACT = false.
template <bool MHD, typename T>
__device__ __forceinline__ bool march_wild(const T w[S_N]) {
  T s = fabs(w[0]);
#pragma unroll
  for (int q = 1; q < (MHD ? S_N : S_BX); q++) s += fabs(w[q]);
  return !(s < (T)MARCH_TAME);
}

// Minimum of `local` over a workgroup of any whole number of waves into
// *result (block_min_to's encoding).
template <int NT>
__device__ __forceinline__ void march_min_to(unsigned long long *result, double local,
                                             unsigned long long *wmin) {
  unsigned long long bits = __double_as_longlong(local);
  if (!(local >= 0.0)) bits = 0x7FF8000000000000ull;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    unsigned long long o = __shfl_xor(bits, off, 64);
    bits = (o < bits) ? o : bits;
  }
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = bits;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long m = wmin[0];
    for (int w = 1; w < NT / 64; w++) m = (wmin[w] < m) ? wmin[w] : m;
    if (m < __hip_atomic_load(result, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin(result, m);
  }
}

// A cell's state as it comes from memory, ahead of its use: HALF, the
// primitives the first stage stored; else the integration quantities.
template <typename T, bool DE, bool HALF>
struct RawCell {
  typename std::conditional<HALF, T, double>::type d[S_N];
  double ei;
};
// off: the cell's byte offset in an FP64 field
template <bool MHD, typename T, bool DE, bool HALF>
__device__ __forceinline__ void march_load(const BlockDesc<T> &b, unsigned off,
                                           RawCell<T, DE, HALF> &r) {
#pragma unroll
  for (int q = 0; q < (MHD ? S_N : S_BX); q++) {
    if constexpr (HALF) {
      if constexpr (std::is_same<T, float>::value)
        r.d[q] = ldo(b.Up[q], off >> 1);
      else
        r.d[q] = ldo(b.Ut[q], off);
    } else {
      if (!(DE && q == S_E)) r.d[q] = ldo(b.U[q], off);
    }
  }
  if (DE && !HALF) r.ei = ldo(b.ei, off);
}
// The centre E of a cell from its velocity and B.
template <typename P>
__device__ __forceinline__ void march_center_e(const P w[S_N], double ec[3]) {
  ec[0] = center_efield((double)w[S_VY], (double)w[S_VZ], (double)w[S_BY], (double)w[S_BZ]);
  ec[1] = center_efield((double)w[S_VZ], (double)w[S_VX], (double)w[S_BZ], (double)w[S_BX]);
  ec[2] = center_efield((double)w[S_VX], (double)w[S_VY], (double)w[S_BX], (double)w[S_BY]);
}
// ... as primitives (load_prim's expressions)
template <bool MHD, typename T, bool DE, bool HALF>
__device__ __forceinline__ void march_prim(const RawCell<T, DE, HALF> &r, double gm1, T w[S_N]) {
#pragma unroll
  for (int q = 0; q < (MHD ? S_N : S_BX); q++)
    if (HALF || q != S_E) w[q] = (T)r.d[q];
  if constexpr (!HALF) {
    if (DE)
      w[S_E] = (T)(gm1 * r.d[S_RHO] * r.ei);
    else
      w[S_E] = (T)prim_pressure<MHD>(r.d[S_RHO], r.d[S_VX], r.d[S_VY], r.d[S_VZ], r.d[S_E],
                                     MHD ? r.d[S_BX] : 0., MHD ? r.d[S_BY] : 0.,
                                     MHD ? r.d[S_BZ] : 0., gm1);
  }
}

// One piece of a workgroup's planes: the column of this thread and the
// offsets the marches use.  False when the piece holds no plane to update.
struct MarchPiece {
  int by, tix, tiy, z0;  // block, tile, first updated plane of the piece
  int ks, ke;            // updated planes [ks, ke)
};
__device__ __forceinline__ bool march_piece(const MarchParams &mp, int cs, long &pos, long last,
                                            MarchPiece &p) {
  const unsigned column = (unsigned)((unsigned long)pos / (unsigned)mp.zseg);
  const int zin = (int)(pos - (long)column * mp.zseg);
  int zn = (last - pos < mp.zseg - zin) ? (int)(last - pos) : mp.zseg - zin;
  pos += zn;
  const int ntile = mp.ntx * mp.nty;
  const unsigned part = column / (unsigned)ntile;
  const int tile = (int)(column - part * (unsigned)ntile);
  p.by = (int)(part / (unsigned)mp.nseg);
  p.z0 = (int)(part - (unsigned)p.by * (unsigned)mp.nseg) * mp.zseg + zin;
  if (zn > mp.nz - p.z0) zn = mp.nz - p.z0;  // the last segment may be shorter
  if (zn <= 0) return false;
  p.tiy = tile / mp.ntx;
  p.tix = tile - p.tiy * mp.ntx;
  p.ks = cs + 1 + p.z0;
  p.ke = p.ks + zn;
  return true;
}
// The cell of the outer ring that thread r of a reconstructing march brings
// in: tile coordinates (rx, ry); false for the threads past the ring.
__device__ __forceinline__ bool march_ring(int r, int w2, int h2, int &rx, int &ry) {
  const bool ring = r < 2 * (w2 + h2);
  if (r < 2 * h2) {
    rx = (r & 1) ? w2 : -1;
    ry = r >> 1;
  } else {
    r -= 2 * h2;
    rx = r >> 1;
    ry = (r & 1) ? h2 : -1;
  }
  if (!ring) rx = ry = 0;
  return ring;
}

// Launch: total / share workgroups (rounded up to a multiple of 8) of NT
// threads, WAVES waves to a SIMD; the XCD-contiguous order of wg_coords.  T
// is the arithmetic and flux type (float: the mixed path).  HALF: the stage reads the half-step state, which the first stage
// stored as primitives (mixed path: FP32 and the FP64 centre E beside
// them; FP64: with the pressure in the place of the total energy); the
// first stage of the VL scheme is the nearest-neighbour one and reads the
// start-of-step state.
template <typename T, int RECON, int RIEMANN, bool DE, bool HALF, int NT, int WAVES>
__global__ void __launch_bounds__(NT, WAVES)
k_march(const BlockDesc<T> *__restrict__ blocks, StageParams sp, MarchParams mp) {
  constexpr bool PLM = RECON != RC_NN;
  constexpr bool F32 = std::is_same<T, float>::value;
  // the limiter's fast form needs its operands' range checked
  constexpr bool CHECK = RECON == RC_PLM && !F32;
  static_assert(HALF || !PLM, "the first stage is the nearest-neighbour one");
  // the stage that reads the half-step state is the final one; the debug
  // counts take the separate launches
  constexpr bool FINAL = HALF;
  // Mixed path, whose FP32 solves leave registers over: the cell k + 1 stays
  // in registers until it is the plane's (CARRY; FP64 would spill, and loads
  // it twice, a plane apart), and the cell update comes after the barrier
  // that ends the plane instead of a barrier of its own (LATE; in FP64 the
  // same time with and without spills).  Orszag-Tang 256^3, second stage: 1.77
  // ms with neither, 1.73 LATE, 1.64 both; first stage 1.30, 1.20 LATE, 1.085
  // with three waves a SIMD as well.
  constexpr bool LATE = F32, CARRY = PLM && F32;
  sp.stage = sp.is_final = FINAL ? 1 : 0;
  sp.dbg = nullptr;
  if (!FINAL) sp.cfl = nullptr;
  const unsigned g = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const long last = ((long)g + 1) * mp.share < mp.total ? ((long)g + 1) * mp.share : mp.total;

  const FluxConsts fc = flux_consts<T>(sp, nullptr);
  const T theta = (T)sp.theta;
  // LDS.  sW: the plane's primitives; sEc: the centre E of plane k; sF: the z
  // and x face quantities by slot; sX: the x right states on their way to the
  // neighbour, then the y fluxes; sP: the y right states, then the edge EMFs
  // (sE).  sB, the face B of plane k - 1: with LATE behind sE, else in the
  // first rows of sF, whose values (FZ*, FXB) are spent by then.  What takes
  // an area's place is written at least one barrier after its last read.
  constexpr int WN = PLM ? march_plane_cells<true>(NT) : NT;
  enum { FZD, FZBX, FZBY, FXB, FX0, FN = FX0 + 5 };
  enum { FY0, FYB = FY0 + 5, FYN };
  constexpr int EB = LATE ? 40 : 24, PB = PLM && 7 * sizeof(T) > EB ? 7 * sizeof(T) : EB;
  __shared__ T sW[S_N][WN];
  __shared__ __align__(16) T sF[PLM ? FN : FN + FYN][NT];
  __shared__ double sEc[3][NT];
  __shared__ T sXs[PLM ? S_N - 1 : 1][PLM ? NT : 1];
  __shared__ __align__(16) char sP[PB * NT];
  __shared__ double sD[DE ? 4 : 1][DE ? NT : 1];
  __shared__ int sWild;
  T(*sY)[NT] = reinterpret_cast<T(*)[NT]>(sP);
  double(*sE)[NT] = reinterpret_cast<double(*)[NT]>(sP);
  double(*sB)[NT] = LATE ? sE + 3 : reinterpret_cast<double(*)[NT]>(&sF[0][0]);
  T(*sX)[NT] = PLM ? reinterpret_cast<T(*)[NT]>(&sXs[0][0]) : &sF[FN];

  const int tid = (int)threadIdx.x;
  const int w2 = mp.w2, h2 = mp.h2;
  const int cs = sp.cur_stale;
  double local = 1.7976931348623157e308;

  for (long pos = (long)g * mp.share; pos < last;) {
    MarchPiece piece;
    if (!march_piece(mp, cs, pos, last, piece)) continue;
    const int by = piece.by, tix = piece.tix, tiy = piece.tiy, z0 = piece.z0;
    const int ks = piece.ks, ke = piece.ke;
    if (zero_step(sp, by)) continue;
    const BlockDesc<T> &b = blocks[by];
    const int mx = b.mx, my = b.my, mz = b.mz;

    const bool lane = tid < w2 * h2;
    const int ty = lane ? tid / w2 : 0, tx = lane ? tid - ty * w2 : 0;
    const int i = cs + tix * (w2 - 2) + tx, j = cs + tiy * (h2 - 2) + ty;
    // columns past the block (in the last tiles) read its last one and write
    // nothing
    const int ic = i < mx ? i : mx - 1, jc = j < my ? j : my - 1;
    const bool in_x = tx >= 1 && tx < w2 - 1 && i < mx - cs - 1;
    const bool in_y = ty >= 1 && ty < h2 - 1 && j < my - cs - 1;
    const bool upd = lane && in_x && in_y;
    // faces this tile writes: the high faces of its cells and, in the first
    // tile along an axis, the low face of its first cell
    const bool own_x = lane && in_y && (in_x || (tx == 0 && tix == 0));
    const bool own_y = lane && in_x && (in_y || (ty == 0 && tiy == 0));
    const double dt = sp.dts ? sp.dts[by] * sp.dt_factor : sp.dt;
    const double dtdx = uniform(dt / b.cw[0]), dtdy = uniform(dt / b.cw[1]),
                 dtdz = uniform(dt / b.cw[2]);

    // LDS neighbours of this column (clamped: the outermost columns' results
    // are not used where a neighbour is missing)
    const int xp = tid + 1 < NT ? tid + 1 : NT - 1, xm = tid > 0 ? tid - 1 : 0;
    const int yp = tid + w2 < NT ? tid + w2 : NT - 1, ym = tid >= w2 ? tid - w2 : 0;
    const int xyp = tid + w2 + 1 < NT ? tid + w2 + 1 : NT - 1;
    const int ws = PLM ? w2 + 2 : w2;  // row of sW
    const int wi = PLM ? (ty + 1) * ws + tx + 1 : tid;
    // in the nearest-neighbour march sW is indexed by column (wi = tid)
    const int wxp = PLM ? wi + 1 : xp, wyp = PLM ? wi + ws : yp;
    // byte offsets in an FP64 field's plane: this column's cell, its faces
    // towards i + 1 and j + 1
    const unsigned plane = 8u * (unsigned)(mx * my);
    const unsigned planex = 8u * (unsigned)((mx + 1) * my);
    const unsigned planey = 8u * (unsigned)(mx * (my + 1));
    const unsigned col = 8u * (unsigned)(jc * mx + ic);
    const unsigned colx = 8u * (unsigned)(jc * (mx + 1) + ic + 1);
    const unsigned coly = 8u * (unsigned)((jc + 1) * mx + ic);
    // the cell of the outer ring this thread brings in (reconstruction only)
    bool ring = false;
    unsigned rcol = 0;
    int rw = 0;
    if constexpr (PLM) {
      int rx, ry;
      ring = march_ring(tid, w2, h2, rx, ry);
      int ri = cs + tix * (w2 - 2) + rx, rj = cs + tiy * (h2 - 2) + ry;
      ri = ri < mx ? ri : mx - 1;
      rj = rj < my ? rj : my - 1;
      rcol = 8u * (unsigned)(rj * mx + ri);
      rw = (ry + 1) * ws + rx + 1;
    }
    const double *const *bfr = HALF ? b.bft : b.bfi;
    const double *const *bf0 = FINAL ? b.bf0 : b.bfi;
    double *const *bout = FINAL ? b.bfi : b.bft;

    // state carried from plane to plane
    T Lz[S_N], wm[S_N], wp[S_N];
    T Fz[5];
    T FxBz = T(0), FyBz = T(0), FxD = T(0), FyD = T(0);
    double dU[5], dUe = 0., pc = 0.;  // of the cell of plane k - 1
    T FzE = T(0), FzV = T(0);
    double ecx0 = 0., ecx1 = 0., ecy0 = 0., ecy1 = 0.;
    double Ex = 0., Ey = 0., Ez = 0., Bz = 0.;
#pragma unroll
    for (int q = 0; q < 5; q++) {
      Fz[q] = T(0);
      dU[q] = 0.;
    }
#pragma unroll
    for (int q = 0; q < S_N; q++) Lz[q] = wm[q] = wp[q] = T(0);

    const int k0 = ks - 1;
    double fbx, fby, fbz;
    if (CHECK && tid == 0) sWild = 0;
    if (CHECK) lds_barrier();
    {
      RawCell<T, DE, HALF> raw;
      double ec[3];
      T w[S_N];
      const unsigned c0 = (unsigned)k0 * plane + col;
      bool wild = false;
      march_load<true>(b, c0, raw);
      march_prim<true>(raw, fc.gm1, w);
      if constexpr (F32 && HALF) {
#pragma unroll
        for (int a = 0; a < 3; a++) ec[a] = ldo(b.Ech[a], c0);
      } else {
        march_center_e(raw.d, ec);
      }
      if (CHECK) wild = march_wild<true>(w);
      if (lane) {
#pragma unroll
        for (int q = 0; q < S_N; q++) sW[q][wi] = w[q];
      }
#pragma unroll
      for (int a = 0; a < 3; a++) sEc[a][tid] = ec[a];
      if constexpr (PLM) {
        march_load<true>(b, c0 - plane, raw);
        march_prim<true>(raw, fc.gm1, wm);
        march_load<true>(b, c0 + plane, raw);
        march_prim<true>(raw, fc.gm1, wp);
        march_load<true>(b, (unsigned)k0 * plane + rcol, raw);
        march_prim<true>(raw, fc.gm1, w);
        if (CHECK) wild = wild || march_wild<true>(wm) || march_wild<true>(wp) || march_wild<true>(w);
        if (ring) {
#pragma unroll
          for (int q = 0; q < S_N; q++) sW[q][rw] = w[q];
        }
      }
      if (CHECK && wild) sWild = 1;
      fbx = ldo(bfr[0], (unsigned)k0 * planex + colx);
      fby = ldo(bfr[1], (unsigned)k0 * planey + coly);
      fbz = ldo(bfr[2], c0);
    }
    lds_barrier();

    for (int k = k0; k <= ke; k++) {
      // a state out of the fast limiter's range was seen in this tile
      const bool exact = CHECK && __builtin_amdgcn_readfirstlane(sWild) != 0;
      // ---- z: the face between planes k - 1 and k
      {
        T a[S_N], R[S_N], Ln[S_N];
#pragma unroll
        for (int q = 0; q < S_N; q++) a[q] = sW[q][wi];
        if constexpr (PLM) {
          auto states = [&](auto ex) {
#pragma unroll
            for (int q = 0; q < S_N; q++)
              if (q != S_BZ)
                march_states<RECON, decltype(ex)::value>(q, wm[q], a[q], wp[q], theta, fc, R[q],
                                                         Ln[q]);
          };
          if (!CHECK || exact)
            states(std::true_type());
          else
            states(std::false_type());
        } else {
#pragma unroll
          for (int q = 0; q < S_N; q++) R[q] = Ln[q] = a[q];
        }
        if (k > k0) {
          FaceFlux<T> f;
          solve_face<T, RIEMANN, true, 2, DE, PLM, HALF>(Lz, R, (T)fbz, fc, f);
          if (k > ks) {
            // the divergence of cell k - 1 (its x and y parts are in dU)
#pragma unroll
            for (int q = 0; q < 5; q++)
              dU[q] = flux_difference(dU[q], dtdz, (double)f.u[q], (double)Fz[q]);
            if (DE) {
              dUe = flux_difference(dUe, dtdz, (double)f.e, (double)FzE);
              dUe = source_difference(dUe, dtdz, pc, (double)f.vb, (double)FzV);
            }
          }
#pragma unroll
          for (int q = 0; q < 5; q++) Fz[q] = f.u[q];
          if (DE) {
            FzE = f.e;
            FzV = f.vb;
          }
          sF[FZD][tid] = f.u[S_RHO];
          sF[FZBX][tid] = f.bj;
          sF[FZBY][tid] = f.bk;
        }
#pragma unroll
        for (int q = 0; q < S_N; q++)
          if (!(PLM && q == S_BZ)) Lz[q] = Ln[q];
      }
      // the right states along an axis through LDS: this column's own left
      // state in L, the neighbour's right state in R (lo / hi: sW of the
      // cells before and after, nb: the neighbour column, SKIP: the slot of
      // the normal B)
      auto exchange = [&](auto skip_slot, T(*sR)[NT], int lo, int hi, int nb, T L[S_N],
                          T R[S_N]) {
        constexpr int SKIP = decltype(skip_slot)::value;
        if constexpr (PLM) {
          auto states = [&](auto ex) {
#pragma unroll
            for (int q = 0; q < S_N; q++) {
              if (q == SKIP) continue;
              T right;
              march_states<RECON, decltype(ex)::value>(q, sW[q][lo], sW[q][wi], sW[q][hi], theta,
                                                       fc, right, L[q]);
              sR[q > SKIP ? q - 1 : q][tid] = right;
            }
          };
          if (!CHECK || exact)
            states(std::true_type());
          else
            states(std::false_type());
          lds_barrier();
#pragma unroll
          for (int q = 0; q < S_N; q++)
            if (q != SKIP) R[q] = sR[q > SKIP ? q - 1 : q][nb];
        } else {
#pragma unroll
          for (int q = 0; q < S_N; q++) {
            L[q] = sW[q][wi];
            R[q] = sW[q][hi];
          }
        }
      };
      // ---- x: the face towards i + 1
      T FxBz_k, FyBz_k;
      {
        T L[S_N], R[S_N];
        exchange(std::integral_constant<int, S_BX>(), sX, wi - 1, wxp, xp, L, R);
        FaceFlux<T> f;
        solve_face<T, RIEMANN, true, 0, DE, PLM, HALF>(L, R, (T)fbx, fc, f);
#pragma unroll
        for (int q = 0; q < 5; q++) sF[FX0 + q][tid] = f.u[q];
        sF[FXB][tid] = f.bj;
        FxBz_k = f.bk;
        if (DE) {
          sD[0][tid] = (double)f.e;
          sD[1][tid] = (double)f.vb;
        }
      }
      // ---- y: the face towards j + 1
      {
        T L[S_N], R[S_N];
        exchange(std::integral_constant<int, S_BY>(), sY, wi - ws, wyp, yp, L, R);
        FaceFlux<T> f;
        solve_face<T, RIEMANN, true, 1, DE, PLM, HALF>(L, R, (T)fby, fc, f);
#pragma unroll
        for (int q = 0; q < 5; q++) sX[FY0 + q][tid] = f.u[q];
        FyBz_k = f.bj;
        sX[FYB][tid] = f.bk;
        if (DE) {
          sD[2][tid] = (double)f.e;
          sD[3][tid] = (double)f.vb;
        }
      }
      // loads for the rest of this step and for the next plane go out now (the
      // FP64 reconstruction loads the column's cell twice, a plane apart,
      // instead of keeping it through the solves: 16 registers)
      const unsigned kn = (unsigned)((k + 1 < mz) ? k + 1 : mz - 1);
      const unsigned ku = (unsigned)(k > 0 ? k - 1 : 0);  // the plane to update
      const unsigned cn = kn * plane + col;
      const unsigned cu = ku * plane + col;
      const unsigned fxu = ku * planex + colx;
      const unsigned fyu = ku * planey + coly;
      const unsigned fzk = (unsigned)k * plane + col;
      const bool face_step = k >= ks;  // the level below plane k
      const bool cell_step = k > ks;   // plane k - 1
      const double b0z = ldo(bf0[2], fzk), b0x = ldo(bf0[0], fxu), b0y = ldo(bf0[1], fyu);
      CellBase u0;
      auto load_base = [&]() {
        u0.rho = ldo(b.U[S_RHO], cu);
        u0.v[0] = ldo(b.U[S_VX], cu);
        u0.v[1] = ldo(b.U[S_VY], cu);
        u0.v[2] = ldo(b.U[S_VZ], cu);
        u0.e = ldo(b.U[S_E], cu);
        if (DE) u0.ei = ldo(b.ei, cu);
      };
      if constexpr (!LATE) load_base();
      RawCell<T, DE, HALF> nxt, nx2, halo;
      if constexpr (!CARRY) march_load<true>(b, cn, nxt);
      fbx = ldo(bfr[0], kn * planex + colx);
      fby = ldo(bfr[1], kn * planey + coly);
      fbz = ldo(bfr[2], cn);
      double echn[3];
      if constexpr (F32 && HALF) {
#pragma unroll
        for (int a = 0; a < 3; a++) echn[a] = ldo(b.Ech[a], cn);
      }
      if constexpr (PLM) {
        march_load<true>(b, kn * plane + rcol, halo);
        const unsigned kn2 = (unsigned)((k + 2 < mz) ? k + 2 : mz - 1);
        march_load<true>(b, kn2 * plane + col, nx2);
      }
      lds_barrier();  // the plane's fluxes are in LDS
      // ---- E: edge EMFs
      const double Ex_b = Ex, Ey_b = Ey, Ez_b = Ez;  // levels k - 3/2, plane k - 1
      {
        const double dxm = (double)sF[FX0][tid], dym = (double)sX[FY0][tid];
        Ez = edge_value(sEc[2][tid], sEc[2][xp], sEc[2][yp], sEc[2][xyp], (double)sF[FXB][tid],
                        (double)sF[FXB][yp], (double)sX[FYB][tid], (double)sX[FYB][xp], dxm,
                        (double)sF[FX0][yp], dym, (double)sX[FY0][xp]);
        const double cx0 = sEc[0][tid], cx1 = sEc[0][yp], cy0 = sEc[1][tid], cy1 = sEc[1][xp];
        if (face_step) {
          const double dz = (double)sF[FZD][tid];
          Ex = edge_value(ecx0, ecx1, cx0, cx1, (double)FyBz, (double)FyBz_k,
                          (double)sF[FZBY][tid], (double)sF[FZBY][yp], (double)FyD, dym, dz,
                          (double)sF[FZD][yp]);
          Ey = edge_value(ecy0, cy0, ecy1, cy1, (double)sF[FZBX][tid], (double)sF[FZBX][xp],
                          (double)FxBz, (double)FxBz_k, dz, (double)sF[FZD][xp], (double)FxD, dxm);
        }
        ecx0 = cx0; ecx1 = cx1; ecy0 = cy0; ecy1 = cy1;
        FxBz = FxBz_k;
        FyBz = FyBz_k;
        FxD = (T)dxm;
        FyD = (T)dym;
      }
      sE[0][tid] = Ex;
      sE[1][tid] = Ey;
      sE[2][tid] = Ez_b;
      lds_barrier();
      // ---- B: the level below plane k, and the faces of plane k - 1
      const double Bz_b = Bz;
      double Bx = 0., By = 0.;
      if (face_step) {
        Bz = face_b_update(b0z, dtdx, dtdy, Ey, sE[1][xm], Ex, sE[0][ym]);
        if (upd && (k > ks || z0 == 0)) {
          sto(bout[2], fzk, Bz);
          if (!FINAL) sto(b.bf0[2], fzk, b0z);
        }
      }
      if (cell_step) {
        Bx = face_b_update(b0x, dtdy, dtdz, Ez_b, sE[2][ym], Ey, Ey_b);
        By = face_b_update(b0y, dtdz, dtdx, Ex, Ex_b, Ez_b, sE[2][xm]);
        sB[0][tid] = Bx;
        sB[1][tid] = By;
        if (own_x) {
          sto(bout[0], fxu, Bx);
          if (!FINAL) sto(b.bf0[0], fxu, b0x);
        }
        if (own_y) {
          sto(bout[1], fyu, By);
          if (!FINAL) sto(b.bf0[1], fyu, b0y);
        }
      }
      // ---- U: the cell of plane k - 1
      auto update = [&]() {
        if (!cell_step || !upd) return;
        const double bc[3] = {half_sum(sB[0][xm], Bx), half_sum(sB[1][ym], By),
                              half_sum(Bz_b, Bz)};
        if (!F32 || FINAL) {
          double *const *Uo = FINAL ? b.U : b.Ut;
          sto(Uo[S_BX], cu, bc[0]);
          sto(Uo[S_BY], cu, bc[1]);
          sto(Uo[S_BZ], cu, bc[2]);
        }
        const double t = cell_finish<T, true, DE, true>(b, sp, dt, CellOffset{cu}, u0, dU, dUe, bc);
        local = t < local ? t : local;
      };
      if constexpr (!LATE) {
        lds_barrier();
        update();
      }
      // ---- the x and y parts of plane k's divergence
      double dUn[5], dUen = 0., pcn = 0.;
#pragma unroll
      for (int q = 0; q < 5; q++) {
        dUn[q] = flux_difference(0., dtdx, (double)sF[FX0 + q][tid], (double)sF[FX0 + q][xm]);
        dUn[q] = flux_difference(dUn[q], dtdy, (double)sX[FY0 + q][tid], (double)sX[FY0 + q][ym]);
      }
      if (DE) {
        pcn = dmax((double)sW[S_E][wi], sp.pressure_floor);
        dUen = flux_difference(0., dtdx, sD[0][tid], sD[0][xm]);
        dUen = source_difference(dUen, dtdx, pcn, sD[1][tid], sD[1][xm]);
        dUen = flux_difference(dUen, dtdy, sD[2][tid], sD[2][ym]);
        dUen = source_difference(dUen, dtdy, pcn, sD[3][tid], sD[3][ym]);
      }
      // ---- the next plane into LDS
      {
        T w[S_N];
        double ec[3];
        if constexpr (CARRY) {
#pragma unroll
          for (int q = 0; q < S_N; q++) w[q] = wp[q];
        } else {
          march_prim<true>(nxt, fc.gm1, w);
        }
        if constexpr (F32 && HALF) {
#pragma unroll
          for (int a = 0; a < 3; a++) ec[a] = echn[a];
        } else {
          march_center_e(nxt.d, ec);
        }
        if constexpr (PLM) {
#pragma unroll
          for (int q = 0; q < S_N; q++) wm[q] = sW[q][wi];
          T h[S_N];
          march_prim<true>(halo, fc.gm1, h);
          if (ring) {
#pragma unroll
            for (int q = 0; q < S_N; q++) sW[q][rw] = h[q];
          }
          march_prim<true>(nx2, fc.gm1, wp);
          if (CHECK && (march_wild<true>(h) || march_wild<true>(wp))) sWild = 1;
        }
        if (lane) {
#pragma unroll
          for (int q = 0; q < S_N; q++) sW[q][wi] = w[q];
        }
#pragma unroll
        for (int a = 0; a < 3; a++) sEc[a][tid] = ec[a];
      }
      if constexpr (LATE) load_base();
      lds_barrier();
      if constexpr (LATE) update();  // (the next solves cover its stores)
#pragma unroll
      for (int q = 0; q < 5; q++) dU[q] = dUn[q];
      dUe = dUen;
      pc = pcn;
    }
  }
  // (sF: last read before the barrier that ended the last plane)
  if (sp.cfl != nullptr)
    march_min_to<NT>(sp.cfl, local, reinterpret_cast<unsigned long long *>(&sF[0][0]));
}

// The hydrodynamic march: as k_march, with the HLLC solve and without
// constrained transport.  A step at plane k: the z face below it, which
// completes the divergence and the update of the cell of plane k - 1; then
// the x and y faces of plane k.  The right states travel through the rows of
// LDS that take the fluxes afterwards.  Bound as k_march; 8 blocks of 128^3,
// FP64: 0.89 + 1.25 ms for the two stages against 1.66 + 1.94 of the separate
// launches (a third of which wrote the 15 fluxes of a cell and read them
// back); mixed 0.46 + 0.61 against 1.12 + 1.11.  WAVES: a SIMD's waves that its
// registers are held to.
template <typename T, int RECON, bool DE, bool HALF, int NT, int WAVES>
__global__ void __launch_bounds__(NT, WAVES)
k_march_hd(const BlockDesc<T> *__restrict__ blocks, StageParams sp, MarchParams mp) {
  constexpr bool PLM = RECON != RC_NN;
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr bool CHECK = RECON == RC_PLM && !F32;
  constexpr bool FINAL = HALF;
  constexpr int NQ = 5;  // density, velocity, pressure
  static_assert(HALF || !PLM, "the first stage is the nearest-neighbour one");
  sp.stage = sp.is_final = FINAL ? 1 : 0;
  sp.dbg = nullptr;
  if (!FINAL) sp.cfl = nullptr;
  const unsigned g = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const long last = ((long)g + 1) * mp.share < mp.total ? ((long)g + 1) * mp.share : mp.total;

  const FluxConsts fc = flux_consts<T>(sp, nullptr);
  const T theta = (T)sp.theta;

  constexpr int WN = PLM ? march_plane_cells<false>(NT) : NT;
  __shared__ T sW[NQ][WN];
  __shared__ T sF[2 * NQ][NT];  // right states, then fluxes: x rows, y rows
  __shared__ double sD[DE ? 4 : 1][DE ? NT : 1];
  __shared__ unsigned long long wmin[NT / 64];
  __shared__ int sWild;

  const int tid = (int)threadIdx.x;
  const int w2 = mp.w2, h2 = mp.h2;
  const int cs = sp.cur_stale;
  double local = 1.7976931348623157e308;

  for (long pos = (long)g * mp.share; pos < last;) {
    MarchPiece piece;
    if (!march_piece(mp, cs, pos, last, piece)) continue;
    const int by = piece.by, tix = piece.tix, tiy = piece.tiy;
    const int ks = piece.ks, ke = piece.ke;
    if (zero_step(sp, by)) continue;
    const BlockDesc<T> &b = blocks[by];
    const int mx = b.mx, my = b.my, mz = b.mz;

    const bool lane = tid < w2 * h2;
    const int ty = lane ? tid / w2 : 0, tx = lane ? tid - ty * w2 : 0;
    const int i = cs + tix * (w2 - 2) + tx, j = cs + tiy * (h2 - 2) + ty;
    const int ic = i < mx ? i : mx - 1, jc = j < my ? j : my - 1;
    const bool upd = lane && tx >= 1 && tx < w2 - 1 && i < mx - cs - 1 && ty >= 1 &&
                     ty < h2 - 1 && j < my - cs - 1;
    const double dt = sp.dts ? sp.dts[by] * sp.dt_factor : sp.dt;
    const double dtdx = uniform(dt / b.cw[0]), dtdy = uniform(dt / b.cw[1]),
                 dtdz = uniform(dt / b.cw[2]);
    const int xp = tid + 1 < NT ? tid + 1 : NT - 1, xm = tid > 0 ? tid - 1 : 0;
    const int yp = tid + w2 < NT ? tid + w2 : NT - 1, ym = tid >= w2 ? tid - w2 : 0;
    const int ws = PLM ? w2 + 2 : w2;
    const int wi = PLM ? (ty + 1) * ws + tx + 1 : tid;
    const unsigned plane = 8u * (unsigned)(mx * my);
    const unsigned col = 8u * (unsigned)(jc * mx + ic);
    bool ring = false;
    unsigned rcol = 0;
    int rw = 0;
    if constexpr (PLM) {
      int rx, ry;
      ring = march_ring(tid, w2, h2, rx, ry);
      int ri = cs + tix * (w2 - 2) + rx, rj = cs + tiy * (h2 - 2) + ry;
      ri = ri < mx ? ri : mx - 1;
      rj = rj < my ? rj : my - 1;
      rcol = 8u * (unsigned)(rj * mx + ri);
      rw = (ry + 1) * ws + rx + 1;
    }

    // carried from plane to plane
    T Lz[S_N], wm[S_N], wp[S_N], Fz[NQ];
    double dU[NQ], dUe = 0., pc = 0.;
    T FzE = T(0), FzV = T(0);
    CellBase u0{};
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      Fz[q] = T(0);
      dU[q] = 0.;
    }
#pragma unroll
    for (int q = 0; q < S_N; q++) Lz[q] = wm[q] = wp[q] = T(0);

    // the left state of the first z face, the planes around the first one
    if (CHECK && tid == 0) sWild = 0;
    if (CHECK) lds_barrier();
    {
      RawCell<T, DE, HALF> raw;
      T w[S_N], h[S_N];
      const unsigned c0 = (unsigned)ks * plane + col;
      march_load<false>(b, c0 - plane, raw);
      march_prim<false>(raw, fc.gm1, wm);
      march_load<false>(b, c0, raw);
      march_prim<false>(raw, fc.gm1, w);
      if constexpr (PLM) {
        march_load<false>(b, c0 - 2u * plane, raw);
        march_prim<false>(raw, fc.gm1, wp);
        bool wild = CHECK && (march_wild<false>(wm) || march_wild<false>(w) ||
                              march_wild<false>(wp));
        // (the general form of the limiter: one state a piece)
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          T low;
          march_states<RECON, true>(q, wp[q], wm[q], w[q], theta, fc, low, Lz[q]);
        }
        march_load<false>(b, (unsigned)(ks + 1 < mz ? ks + 1 : mz - 1) * plane + col, raw);
        march_prim<false>(raw, fc.gm1, wp);
        march_load<false>(b, (unsigned)ks * plane + rcol, raw);
        march_prim<false>(raw, fc.gm1, h);
        if (CHECK) wild = wild || march_wild<false>(wp) || march_wild<false>(h);
        if (CHECK && wild) sWild = 1;
        if (ring) {
#pragma unroll
          for (int q = 0; q < NQ; q++) sW[q][rw] = h[q];
        }
      } else {
#pragma unroll
        for (int q = 0; q < NQ; q++) Lz[q] = wm[q];
      }
      if (lane) {
#pragma unroll
        for (int q = 0; q < NQ; q++) sW[q][wi] = w[q];
      }
    }
    lds_barrier();

    for (int k = ks; k <= ke; k++) {
      const bool exact = CHECK && __builtin_amdgcn_readfirstlane(sWild) != 0;
      // ---- z: the face between planes k - 1 and k
      {
        T a[S_N], R[S_N], Ln[S_N];
#pragma unroll
        for (int q = 0; q < NQ; q++) a[q] = sW[q][wi];
        if constexpr (PLM) {
          auto states = [&](auto ex) {
#pragma unroll
            for (int q = 0; q < NQ; q++)
              march_states<RECON, decltype(ex)::value>(q, wm[q], a[q], wp[q], theta, fc, R[q],
                                                       Ln[q]);
          };
          if (!CHECK || exact)
            states(std::true_type());
          else
            states(std::false_type());
        } else {
#pragma unroll
          for (int q = 0; q < NQ; q++) R[q] = Ln[q] = a[q];
        }
        FaceFlux<T> f;
        solve_face<T, RS_HLLC, false, 2, DE, PLM, HALF>(Lz, R, T(0), fc, f);
        if (k > ks) {
#pragma unroll
          for (int q = 0; q < NQ; q++)
            dU[q] = flux_difference(dU[q], dtdz, (double)f.u[q], (double)Fz[q]);
          if (DE) {
            dUe = flux_difference(dUe, dtdz, (double)f.e, (double)FzE);
            dUe = source_difference(dUe, dtdz, pc, (double)f.vb, (double)FzV);
          }
          if (upd) {
            const double bc[3] = {0., 0., 0.};
            const double t = cell_finish<T, false, DE, true>(
                b, sp, dt, CellOffset{(unsigned)(k - 1) * plane + col}, u0, dU, dUe, bc);
            local = t < local ? t : local;
          }
        }
        if (k == ke) break;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          Fz[q] = f.u[q];
          Lz[q] = Ln[q];
        }
        if (DE) {
          FzE = f.e;
          FzV = f.vb;
        }
      }
      // ---- x, y: the faces towards i + 1 and j + 1
      FaceFlux<T> fx, fy;
      {
        T Lx[S_N], Ly[S_N], Rx[S_N], Ry[S_N];
        if constexpr (PLM) {
          auto states = [&](auto ex) {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
              constexpr bool EX = decltype(ex)::value;
              const T a = sW[q][wi];
              T rx, ry;
              march_states<RECON, EX>(q, sW[q][wi - 1], a, sW[q][wi + 1], theta, fc, rx, Lx[q]);
              march_states<RECON, EX>(q, sW[q][wi - ws], a, sW[q][wi + ws], theta, fc, ry,
                                      Ly[q]);
              sF[q][tid] = rx;
              sF[NQ + q][tid] = ry;
            }
          };
          if (!CHECK || exact)
            states(std::true_type());
          else
            states(std::false_type());
          lds_barrier();
#pragma unroll
          for (int q = 0; q < NQ; q++) {
            Rx[q] = sF[q][xp];
            Ry[q] = sF[NQ + q][yp];
          }
          lds_barrier();
        } else {
#pragma unroll
          for (int q = 0; q < NQ; q++) {
            Lx[q] = Ly[q] = sW[q][wi];
            Rx[q] = sW[q][xp];
            Ry[q] = sW[q][yp];
          }
        }
        solve_face<T, RS_HLLC, false, 0, DE, PLM, HALF>(Lx, Rx, T(0), fc, fx);
        solve_face<T, RS_HLLC, false, 1, DE, PLM, HALF>(Ly, Ry, T(0), fc, fy);
      }
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        sF[q][tid] = fx.u[q];
        sF[NQ + q][tid] = fy.u[q];
      }
      if (DE) {
        sD[0][tid] = (double)fx.e;
        sD[1][tid] = (double)fx.vb;
        sD[2][tid] = (double)fy.e;
        sD[3][tid] = (double)fy.vb;
      }
      // loads for the next step: the base of this plane's update, the next
      // planes
      const unsigned kn = (unsigned)((k + 1 < mz) ? k + 1 : mz - 1);
      const unsigned cu = (unsigned)k * plane + col;
      RawCell<T, DE, HALF> nxt, nx2, halo;
      march_load<false>(b, kn * plane + col, nxt);
      if constexpr (PLM) {
        march_load<false>(b, kn * plane + rcol, halo);
        const unsigned kn2 = (unsigned)((k + 2 < mz) ? k + 2 : mz - 1);
        march_load<false>(b, kn2 * plane + col, nx2);
      }
      u0.rho = ldo(b.U[S_RHO], cu);
      u0.v[0] = ldo(b.U[S_VX], cu);
      u0.v[1] = ldo(b.U[S_VY], cu);
      u0.v[2] = ldo(b.U[S_VZ], cu);
      u0.e = ldo(b.U[S_E], cu);
      if (DE) u0.ei = ldo(b.ei, cu);
      lds_barrier();  // the plane's fluxes are in LDS
      // ---- the x and y parts of plane k's divergence
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        dU[q] = flux_difference(0., dtdx, (double)fx.u[q], (double)sF[q][xm]);
        dU[q] = flux_difference(dU[q], dtdy, (double)fy.u[q], (double)sF[NQ + q][ym]);
      }
      if (DE) {
        pc = dmax((double)sW[S_E][wi], sp.pressure_floor);
        dUe = flux_difference(0., dtdx, sD[0][tid], sD[0][xm]);
        dUe = source_difference(dUe, dtdx, pc, sD[1][tid], sD[1][xm]);
        dUe = flux_difference(dUe, dtdy, sD[2][tid], sD[2][ym]);
        dUe = source_difference(dUe, dtdy, pc, sD[3][tid], sD[3][ym]);
      }
      // ---- the next plane into LDS
      {
        T w[S_N];
        march_prim<false>(nxt, fc.gm1, w);
        if constexpr (PLM) {
#pragma unroll
          for (int q = 0; q < NQ; q++) wm[q] = sW[q][wi];
          T h[S_N];
          march_prim<false>(halo, fc.gm1, h);
          if (ring) {
#pragma unroll
            for (int q = 0; q < NQ; q++) sW[q][rw] = h[q];
          }
          march_prim<false>(nx2, fc.gm1, wp);
          if (CHECK && (march_wild<false>(h) || march_wild<false>(wp))) sWild = 1;
        }
        if (lane) {
#pragma unroll
          for (int q = 0; q < NQ; q++) sW[q][wi] = w[q];
        }
      }
      lds_barrier();
    }
    lds_barrier();  // the piece's last reads of LDS
  }
  if (sp.cfl != nullptr) march_min_to<NT>(sp.cfl, local, wmin);
}

// The cells around a marched final stage's update: the cell-centred B of the
// layer at the edge of the flux region (its faces have been updated), and
// with the CFL minimum the term and pressure of every cell outside the
// update.  One thread per cell of the shell, enumerated as the ghost shell.
template <typename FluxT, bool MHD, bool DE>
__global__ void __launch_bounds__(256)
k_shell(const BlockDesc<FluxT> *__restrict__ blocks, StageParams sp) {
  const int by = (int)blockIdx.y;
  if (zero_step(sp, by)) return;
  const BlockDesc<FluxT> &b = blocks[by];
  const int m[3] = {b.mx, b.my, b.mz};
  const int lo = sp.cur_stale;
  const bool cfl = sp.cfl != nullptr;
  const int blo = cfl ? 0 : lo;
  int ext[3], l[3], h[3];
  for (int a = 0; a < 3; a++) {
    ext[a] = m[a] - 2 * blo;
    l[a] = lo + 1 - blo;
    h[a] = m[a] - lo - 1 - blo;
  }
  int k, j, i;
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  double local = 1.7976931348623157e308;
  if (ghost_coords<unsigned>(t, ext, l, h, k, j, i)) {
    k += blo;
    j += blo;
    i += blo;
    const bool in_box = k >= lo && j >= lo && i >= lo && k < m[2] - lo && j < m[1] - lo &&
                        i < m[0] - lo;
    const FaceBGlobal<FluxT> fb{b, b.bfi};
    local = cell_stage<FluxT, MHD, DE>(b, sp, by, k, j, i, true, in_box, fb,
                                       FluxGlobal<FluxT>{b});
  }
  if (cfl) block_min_to(sp.cfl, local);
}

// --------------------------------------------------- small hydro blocks

// One hydrodynamic stage of small blocks as one launch: a workgroup has a
// tile of 8 x 4 x 4 cells, solves the faces around them, one to a thread
// (144, 160 and 160 along x, y and z, each axis in three waves of its own),
// leaves the fluxes in LDS and updates the cells.  Bound by latency: the
// kernel takes about as long as the two it replaces (one 16^3 block, FP64:
// 9.2 us against 6.4 + 4.0, second stage 12.6 against 8.3 + 4.0), and the gap
// between them goes.  The faces between tiles are solved twice (464 for 384
// owned ones).
template <typename FluxT>
struct FluxTile {
  static constexpr int TX = 8, TY = 4, TZ = 4, PER = 192, NF = 160;
  const FluxT (*f)[5][NF];
  const double (*e)[2][NF];
  int x, y, z;  // the cell in the tile
  __device__ __forceinline__ int face(int d, int side) const {
    return d == 0 ? (z * TY + y) * (TX + 1) + x + side
                  : (d == 1 ? (z * (TY + 1) + y + side) * TX + x : ((z + side) * TY + y) * TX + x);
  }
  __device__ __forceinline__ void operator()(int d, int q, long, long, double &lo,
                                             double &hi) const {
    lo = (double)f[d][q][face(d, 0)];
    hi = (double)f[d][q][face(d, 1)];
  }
  __device__ __forceinline__ void energy(int d, long, long, double &elo, double &ehi,
                                         double &vlo, double &vhi) const {
    elo = e[d][0][face(d, 0)];
    ehi = e[d][0][face(d, 1)];
    vlo = e[d][1][face(d, 0)];
    vhi = e[d][1][face(d, 1)];
  }
};
// Launch: grid (tiles of [lo, m - lo), blocks), lo as update_cells takes it;
// 576 threads.
template <typename T, typename FluxT, int RECON, bool DE, bool PRIMF>
__global__ void __launch_bounds__(576)
k_tile(const BlockDesc<FluxT> *__restrict__ blocks, StageParams sp) {
  using Tile = FluxTile<FluxT>;
  constexpr int TX = Tile::TX, TY = Tile::TY, TZ = Tile::TZ;
  __shared__ FluxT sF[3][5][Tile::NF];
  __shared__ double sD[DE ? 3 : 1][2][DE ? Tile::NF : 1];
  __shared__ unsigned long long wmin[9];
  const int by = blockIdx.y;
  if (zero_step(sp, by)) return;
  const BlockDesc<FluxT> &b = blocks[by];
  const int mx = b.mx, my = b.my, mz = b.mz;
  const int ul = sp.cur_stale + 1, lo = sp.is_final ? ul - 1 : ul;
  const bool cfl = sp.cfl != nullptr;
  const int blo = cfl ? 0 : lo;
  const int ntx = (mx - 2 * blo + TX - 1) / TX, nty = (my - 2 * blo + TY - 1) / TY;
  const int t = (int)blockIdx.x, tz = t / (ntx * nty), ty = (t - tz * ntx * nty) / ntx;
  const int i0 = blo + (t - (tz * nty + ty) * ntx) * TX, j0 = blo + ty * TY, k0 = blo + tz * TZ;
  const int tid = (int)threadIdx.x;

  {
    double *const *U = (sp.stage == 0) ? b.U : b.Ut;
    const FluxConsts fc = flux_consts<T>(sp, nullptr);
    const double *ei = DE ? ((sp.stage == 0) ? b.ei : b.eit) : nullptr;
    const PrimSource<T, false, DE, PRIMF> src{U, ei, b.Up, fc.gm1};
    // thread r of axis D: the low face of the cell (i, j, k); solved where
    // a cell beside it is updated
    auto solve = [&](auto axis) {
      constexpr int D = decltype(axis)::value;
      constexpr int NX = TX + (D == 0), NY = TY + (D == 1), NZ = TZ + (D == 2);
      const int r = tid - D * Tile::PER;
      const int z = r / (NX * NY), y = (r - z * (NX * NY)) / NX, x = r - (z * NY + y) * NX;
      const int i = i0 + x, j = j0 + y, k = k0 + z;
      if (r >= NX * NY * NZ || i < ul || j < ul || k < ul || i >= mx - ul + (D == 0) ||
          j >= my - ul + (D == 1) || k >= mz - ul + (D == 2))
        return;
      const int c = (k * my + j) * mx + i - (D == 0 ? 1 : D == 1 ? mx : mx * my);
      T wc[S_N];
      src(c, wc);
      FaceFlux<T> f;
      face_flux<T, FluxT, RECON, RS_HLLC, false, D, DE, PRIMF>(b, src, nullptr, k, j, i, c, wc,
                                                              fc, f);
#pragma unroll
      for (int q = 0; q < 5; q++) sF[D][q][r] = (FluxT)f.u[q];
      if (DE) {
        sD[DE ? D : 0][0][DE ? r : 0] = (double)f.e;
        sD[DE ? D : 0][1][DE ? r : 0] = (double)f.vb;
      }
    };
    if (tid < Tile::PER)
      solve(std::integral_constant<int, 0>());
    else if (tid < 2 * Tile::PER)
      solve(std::integral_constant<int, 1>());
    else
      solve(std::integral_constant<int, 2>());
  }
  __syncthreads();
  double local = 1.7976931348623157e308;
  if (tid < TX * TY * TZ) {
    const int z = tid / (TX * TY), y = (tid - z * (TX * TY)) / TX, x = tid % TX;
    const int i = i0 + x, j = j0 + y, k = k0 + z;
    const bool in_launch = i < mx - blo && j < my - blo && k < mz - blo;
    const bool in_box = in_launch && k >= lo && j >= lo && i >= lo && k < mz - lo &&
                        j < my - lo && i < mx - lo;
    const FaceBGlobal<FluxT> fb{b, nullptr};
    const Tile flux{sF, reinterpret_cast<const double(*)[2][Tile::NF]>(&sD[0][0][0]), x, y, z};
    local = cell_stage<FluxT, false, DE>(b, sp, by, k, j, i, in_launch, in_box, fb, flux);
  }
  if (cfl) march_min_to<576>(sp.cfl, local, wmin);
}

}  // namespace ENZOE_KNS
