// amcafe_device.hip -- HIP kernels of the CAFE time step for CDNA4 (gfx950) and
// the internal launcher API declared in amcafe_dev.h.
//
// One step of one or many independent domains ("instances") runs as:
//   k_step_in          the step's records from the pinned staging area
//   k_temperature      TempField::AnalyticTempCurr (S/TempField.C:139-217), optionally
//                      fused with SetLiquid3 (S/VoxelsCA.C:1098-1116).  (k_easm: the
//                      EASM temperature, S/TempField.C:79-137, when asked for;
//                      k_temp_commit after a temperature on its own.)
//   k_setliquid        SetLiquid3 alone, when the temperature was a separate call
//   k_solid_to_mushy   ConvertSolid1(1) (S/VoxelsCA.C:780-797)
//   k_active_flags     active-set membership (S/VoxelsCA.C:262-273) + per-block counts
//   k_scan             two-level exclusive scan of the block counts, the step's loop state
//   k_compact          ordered active list, voxel->active map, gathers, ruq draws
//                      (S/VoxelsCA.C:274-303, 336-380)
//   k_active_setup     active-neighbour table (S/VoxelsCA.C:304-335) and growing list;
//   k_grow_lists       the growing cells' sorted candidate lists (the per-pair part of
//                      S/VoxelsCA.C:386-445) with each entry's capture re-centring
//   k_event_loop       the serial capture/nucleation loop (S/VoxelsCA.C:381-610), one
//                      workgroup per instance, FP64 throughout
//   k_finish           active arrays back to the grid (S/VoxelsCA.C:633-643) and
//                      ConvertSolid1(0) over the active cells (S/VoxelsCA.C:739-758)
//   k_step_out         the output records to the pinned staging area
// Per-voxel passes take runs of 16 voxels per thread (one 16-byte state load; the temperature
// four).  Layer kernels: k_voronoi, k_site_rank, k_write_layer (base plate and powder layers,
// S/BasePlate.C, S/VoxelsCA.C AddLayer1/CleanLayer); k_grain_presence, k_remap (grain
// renumbering).
// Grid-wide kernels take a flattened block list over all instances, so a batch of
// domains of different sizes is one launch per stage.
//
// Must be compiled with -ffp-contract=off: every floating-point expression that
// restates the reference is evaluated with its own rounding, in its own order.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <string>
#include <vector>

#include <atomic>

#include "amcafe_dev.h"
#include "ddmath.h"
#include "gl25.h"

// A pointer known to address global memory.  The capture loop reads its array pointers
// from a descriptor copied to LDS, so the compiler cannot tell their address space and
// would emit flat accesses, which also count against the LDS wait counter: every LDS
// wait would then wait for the outstanding memory loads, and for the stores to be
// acknowledged, as well.  A flat store may also alias the descriptor in LDS, so each one
// makes the compiler read the next array pointer from LDS again.
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gmem(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}
// 8-byte vector records (int2, float2) read and written through a global pointer as one
// 64-bit access (HIP's vector types have no assignment in that address space)
template <class V>
__device__ __forceinline__ V gload8(const V* p) {
  static_assert(sizeof(V) == 8, "8-byte records only");
  return __builtin_bit_cast(V, *gmem((const unsigned long long*)p));
}
template <class V>
__device__ __forceinline__ void gstore8(V* p, V v) {
  static_assert(sizeof(V) == 8, "8-byte records only");
  *gmem((unsigned long long*)p) = __builtin_bit_cast(unsigned long long, v);
}

// LDS words that the waves of a workgroup exchange while they run, each one access in program order (a
// wave's LDS operations are performed in order: what was stored before a word is there when the word
// is seen).  As accesses through a generic pointer to volatile they were flat and system-wide, each
// with a wait for its acknowledgement.
template <class T>
__device__ __forceinline__ void lds_put(T* p, T v) {
  typedef __attribute__((address_space(3))) unsigned u32;
  typedef __attribute__((address_space(3))) unsigned long long u64;
  asm volatile("" ::: "memory");
  if constexpr (sizeof(T) == 8)
    __hip_atomic_store((u64*)p, __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else
    __hip_atomic_store((u32*)p, __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class T>
__device__ __forceinline__ T lds_get(T* p) {
  typedef __attribute__((address_space(3))) unsigned u32;
  typedef __attribute__((address_space(3))) unsigned long long u64;
  T v;
  if constexpr (sizeof(T) == 8)
    v = __builtin_bit_cast(T, __hip_atomic_load((u64*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  else
    v = __builtin_bit_cast(T, __hip_atomic_load((u32*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  asm volatile("" ::: "memory");
  return v;
}

// lane l's value of v (l must be the same in every lane)
__device__ static inline double lane_f64(double v, int l) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// another lane's value by a DPP row operation
template <int CTRL, int ROWS = 0xf>
__device__ static inline int dpp(int v) {
  if constexpr (ROWS == 0xf && (CTRL < 0x100 || CTRL == 0x140 || CTRL == 0x141))  // every lane reads an active one
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, false);
  else
    return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS = 0xf>
__device__ static inline float dpp(float v) {
  return __int_as_float(dpp<CTRL, ROWS>(__float_as_int(v)));
}
template <int CTRL, int ROWS = 0xf>
__device__ static inline double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)dpp<CTRL, ROWS>((int)b), hi = (unsigned)dpp<CTRL, ROWS>((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

#define ZB 1024     // voxels per compaction block (one wave, 16 per thread)
#define GB 256      // threads per grid-wide block
#define SB 4096     // voxels per solid->mushy block (GB threads, 16 voxels each)
// Workgroups of a pass over the active cells, per instance; they go round when there are more cells.  A
// grid for the whole capacity of a 512x512x128 domain, 16 thousand workgroups for 20 thousand cells,
// took 20.7 us in k_active_setup, this one 11.3.
constexpr int kActiveBlocks = 1024;

// -------------------------------------------------------------------------------------
// device structures
struct LoopState {
  int nslots;        // growing-list length
  int vSind2;        // next scan position (S/VoxelsCA.C:346-353, 487-488, 520-521)
  int nGrain;
  int pool_used;
  unsigned int rng;  // minstd_rand0 state
  int nslots_pre;    // slots whose entries have a CapRec (-1 before the loop runs)
  long long draws;
  double tinc;
  int events, captures, nucs, done;
  int pending;       // 1: a nucleation was decided but the pool was empty
  int pend_tgt;      // active index of the voxel to nucleate
  int Na, nmushy0;
  int npre;          // entries of the lists built ahead
  int zhot0, zhot1;  // z planes the last temperature evaluation could have melted
  int zold0, zold1;  // the same of the evaluation that tvalid speaks of
  // T holds the analytic field of a laser plane at lz_prev (tvalid = 1): every voxel is xi
  // where its hot flag (vs bit 7) is set, else T0 above lz_prev and tS below it
  int tvalid;
  int fin;      // the step's loop has finished: its results may go to the grid
  double lz_prev;
  int zpar;     // which half of zliq the last active-set pass wrote
  int chunks;   // chunks of the active-set scan that are done
};

// One entry of a growing cell's candidate list: everything the capture loop reads of it in one
// 32-byte record (four to a cache line; as an array per field, an entry cost five lines).
struct alignas(16) CandRec {
  double D, r;  // capture distance, ruqs
  int tgt;      // target (active index)
  float tn;     // lower bound on the time from a capture through this entry to the first capture
                // by the cell it creates (-inf: unknown)
  float back;   // lower bound on how far the clock may step back after it before that cell's
                // half-diagonal is zero (-inf: unknown)
  short nb;     // neighbour rank
  short n;      // entries from this one to the list's end
};
// What the capture loop reads of an active cell whose voxel is captured, in one cache line.
struct alignas(128) CellRow {
  int nbr[AMCD_NB];  // active indices of the Moore neighbours (-1: outside or not active)
  int vox, cold;     // voxel; all active neighbours below tL (S/VoxelsCA.C:396-397)
  double T;
  int pad[2];
};
// What a capture through an entry of a list the set-up built does: the re-centred octahedron, the
// grain, the new cell's velocity and its list built ahead (-1: none).
struct alignas(16) CapRec {
  double x, y, z, E;
  int pre, G;
  double V;
};
// A growing cell's constants; n: entries of its list (-1: the cell carries no valid grain).
struct alignas(16) SlotRec {
  double c[3];
  int vox, G, act, scan, base, n;
};
// A performed event, for the active arrays at the loop's end.
struct alignas(16) EventRec {
  int i1, G;
  double E, x, y, z, pad;
};
struct Inst {
  amcd_params p;
  int N, nxy, nblkZ, nblkG, nblkS, nblkT;
  // grid fields
  uint8_t* vs;
  int* gid;
  double* ext;
  double *cx, *cy, *cz;
  double* T;
  uint8_t* bj;
  uint8_t* build;  // VoxelsCA::Build (changes only where the driver calls SetBuild)
  int* amap;
  // per z plane: bit 0 = had liquid at the last active-set pass (or unknown); two halves of nz planes,
  // the pass writes the one that ls->zpar does not name, which is clear
  unsigned* zliq;
  int *bcA, *bcM;  // per-ZB-block counts -> exclusive offsets within chunks of 1024 blocks
  int *chA, *chM;  // per chunk: totals -> exclusive offsets
  // active list
  int acap;
  int* aVox;
  uint8_t* aVS;
  int* aG;
  double *aT, *aExt, *aCx, *aCy, *aCz, *ruq;
  CellRow* aRow;
  EventRec* events;
  int* aScan;
  // growing list + candidates (26 slots per growing cell)
  SlotRec* slots;
  double *gExt, *gVhat;
  float2* gLH;      // per slot: capture-clock bounds (lo, hi) of the memory-resident tier
  int2* gHd;        // per slot: list head (entry, target) of the memory-resident tier
  // Lists: first those that the set-up built ahead for the cells that captures would create (`precap`
  // entries at most), then slot s's at precap + 26 s, when the set-up or the loop built it.
  // The entries ahead and those of the set-up's first `capslots` lists have a CapRec, the others their
  // shape factor (at the entry's place less precap), from which a capture is re-centred when it
  // happens: far fewer cells grow than are active, and a CapRec for every active cell took 1.25 of 3.3 KB.
  CandRec* cand;
  CapRec* cap;
  double* cF;
  int precap, capslots;
  // grains
  int gcap;
  double* rot;
  int poolcap;
  double* pool;
  LoopState* ls;
};

// -------------------------------------------------------------------------------------
// minstd_rand0 (x <- 16807 x mod 2^31-1) and libstdc++'s generate_canonical<double,53>
// (/usr/include/c++/11/bits/random.tcc:3345-3381): two engine outputs per double,
//   sum = (x1-1) + (x2-1)*R,  R = 2^31-2,  result = sum / RN(R*R),  clamp below 1.
#define MINSTD_M 2147483647u
__host__ __device__ static inline unsigned int mod_m(unsigned long long x) {
  unsigned long long r = (x & MINSTD_M) + (x >> 31);
  r = (r & MINSTD_M) + (r >> 31);
  return (unsigned int)(r >= MINSTD_M ? r - MINSTD_M : r);
}
__host__ __device__ static inline unsigned int lcg_next(unsigned int x) { return mod_m((unsigned long long)x * 16807u); }
__host__ __device__ static inline unsigned int lcg_pow(unsigned long long e) {  // 16807^e mod m
  unsigned long long b = 16807u, r = 1;
  while (e) {
    if (e & 1) r = mod_m(r * b);
    b = mod_m(b * b);
    e >>= 1;
  }
  return (unsigned int)r;
}
// 16807^(2 d 256^q) mod m: digit q (base 256) of a cell's index, so that the engine is at a cell's two
// outputs after four products (by squaring, as many dependent pairs as its index has bits)
struct LcgTable {
  unsigned p[4][256];
};
constexpr LcgTable lcg_table() {
  LcgTable t = {};
  unsigned long long base = 16807ull * 16807ull % MINSTD_M;
  for (int q = 0; q < 4; ++q) {
    unsigned long long x = 1;
    for (int d = 0; d < 256; ++d) {
      t.p[q][d] = (unsigned)x;
      x = x * base % MINSTD_M;
    }
    base = x;
  }
  return t;
}
__constant__ LcgTable kLcg = lcg_table();
__device__ static inline unsigned lcg_skip_cells(unsigned x, unsigned a) {  // x 16807^(2a)
  for (int q = 0; q < 4 && (a >> (8 * q)) != 0; ++q) x = mod_m((unsigned long long)x * kLcg.p[q][(a >> (8 * q)) & 255u]);
  return x;
}
__host__ __device__ static inline unsigned int lcg_seed(unsigned long long s) {
  unsigned int x = (unsigned int)(s % MINSTD_M);
  return x == 0 ? 1u : x;
}
__host__ __device__ static inline double canonical(unsigned int x1, unsigned int x2) {
  double sum = (double)(x1 - 1u);
  sum = sum + (double)(x2 - 1u) * 2147483646.0;
  double ret = sum / 4611686009837453312.0;  // RN((2^31-2)^2)
  if (ret >= 1.0) ret = 0x1.fffffffffffffp-1;
  return ret;
}

// -------------------------------------------------------------------------------------
__device__ static inline int find_inst(const int* start, int n, int b) {
  int lo = 0, hi = n;  // start[lo] <= b < start[hi]
  while (hi - lo > 1) {
    int mid = (lo + hi) >> 1;
    if (start[mid] <= b) lo = mid; else hi = mid;
  }
  return lo;
}
template <class DI>
__device__ static inline void decode(DI& d, int v, int& i, int& j, int& k) {
  k = v / d.nxy;
  int r = v - k * d.nxy;
  j = r / d.p.nx;
  i = r - j * d.p.nx;
}

// -------------------------------------------------------------------------------------
// TempField::AnalyticTempCurr, S/TempField.C:155-197, with the optional SetLiquid3.
// T takes one of three values, T0 (above the laser plane), xi = tL(1+eps) (inside the melt
// pool) or tS.  Two shortcuts keep the result bit-identical while touching little memory:
//  * a voxel whose |offset| along some semi-axis exceeds that semi-axis by a relative 2^-40
//    is outside the ellipsoid without the divisions (RN is monotone, so the rounded
//    quotient is >= 1 and so is the rounded sum of squares);
//  * while tvalid holds, the previous T of a voxel is known from its hot flag and the
//    previous laser plane, so T, the flag byte and BuildjID are stored only where they change;
//  * a run of voxels whose row segments lie farther from the laser than the melt pool's
//    extent plus two voxels (in the unrotated frame: the rotation about the plate centre
//    preserves distances up to rounding far below that margin) cannot reach tL, so in the
//    planes the pool can reach it changes nothing unless one of its voxels was hot.
//  * planes that neither this evaluation nor the last could melt keep everything while the laser
//    stays in its plane: the workgroups go over the others only.
// A thread takes four voxels (one state word): what bounds it is the chain of a thread whose voxels
// are near the laser, some FP64 instructions and two or three divisions one after another for
// each, and the stores.  20 us for 512x512x128, 8.8 for 256x192x64, 7.2 for 40x24x20; with sixteen voxels a
// thread, a workgroup to every block of the domain and the melt flag of the step set by an atomic
// per wave 32, 20 and 14.
#define TV 4  // voxels per thread
__global__ __launch_bounds__(GB) void k_temperature(Inst* I, const int* bstart, int ninst, const amcd_step* S,
                                                    amcd_out* O, int setliquid) {
  int ii = find_inst(bstart, ninst, blockIdx.x);
  // The descriptor and the step record are copied: read through references, every field would
  // be read again from memory after each store of the voxel loop (a store could alias them).
  const Inst d = I[ii];
  const amcd_step st = S[ii];
  if (st.skip) return;
  const amcd_params& p = d.p;
  // planes with (k+.5)dz in (lz - max depth, lz] are the only ones T can reach tL in (with a plane of
  // margin; the ellipsoid tests need |zp - lz| < depth): elsewhere T is T0 or tS without geometry
  const double depth = fmax(p.a1[2], p.a1[5]);
  const int kh0 = (int)floor((st.lz - depth) / p.dz - 0.5) - 1, kh1 = (int)floor(st.lz / p.dz - 0.5) + 1;
  if (blockIdx.x == bstart[ii] && threadIdx.x == 0) {
    d.ls->zhot0 = max(0, kh0);
    d.ls->zhot1 = min(p.nz - 1, kh1);
  }
  bool anyhot = false;
  // the three temperatures as values (selected through their struct fields, the compiler
  // would keep the struct in scratch memory and load through the selected address)
  const double T0 = p.T0, tS = p.tS, tL = p.tL, xi = p.xi;
  const bool valid = d.ls->tvalid != 0 && tS < tL && T0 < tL;
  const double lzp = d.ls->lz_prev;
  const int zold0 = d.ls->zold0, zold1 = d.ls->zold1;
  const double e1 = 1 + 0x1p-40;
  const double lim1 = p.a1[1] * e1, lim2 = p.a1[2] * e1, lim3 = p.a1[3] * e1, lim4 = p.a1[4] * e1,
               lim5 = p.a1[5] * e1;
  int first = 0, last = d.nblkT - 1;
  if (valid && st.lz == lzp && !(tS < T0)) {  // (tS < T0: the melt flags of planes below the laser's are cleared)
    first = max(0, min(p.nz - 1, min(kh0, zold0))) * d.nxy / (GB * TV);
    last = min(last, ((max(0, min(p.nz - 1, max(kh1, zold1))) + 1) * d.nxy - 1) / (GB * TV));
  }
  const int nb = bstart[ii + 1] - bstart[ii];
  for (int blk = first + (int)blockIdx.x - bstart[ii]; blk <= last; blk += nb) {
    const int v0 = (blk * GB + (int)threadIdx.x) * TV;
    if (v0 >= d.N) continue;
    uint8_t sv[TV];
    if (v0 + TV <= d.N) {
      const unsigned w = *reinterpret_cast<const unsigned*>(d.vs + v0);
#pragma unroll
      for (int q = 0; q < TV; ++q) sv[q] = (uint8_t)(w >> (8 * q));
    } else {
#pragma unroll
      for (int q = 0; q < TV; ++q) sv[q] = v0 + q < d.N ? d.vs[v0 + q] : 0;
    }
    int i, j, k;
    decode(d, v0, i, j, k);
    // Nothing changes for a run of voxels in one plane outside [kh0, kh1] when none of them
    // is hot (and no state byte carries bits the pass clears) and the plane lies on the
    // same side of the previous and the current laser plane: T stays T0 or tS as before,
    // and no state, grain or melt flag is written (below the laser plane the flag is
    // cleared when T < T0, so tS < T0 rules the shortcut out there).
    bool quiet = false;
    if (valid && v0 + TV <= d.N && (v0 + TV - 1) / d.nxy == k) {
      unsigned busy = 0;
#pragma unroll
      for (int q = 0; q < TV; ++q) busy |= sv[q] & 0xbc;
      const double zp = ((double)k + .5) * p.dz;
      bool cold = k < kh0 || k > kh1 || zp > st.lz;  // no geometry reaches these voxels
      if (!cold) {  // the run's distance to the laser (of its rows' when it spans several)
        const double Lx = p.hx + st.cg * (st.lx - p.hx) - st.sg * (st.ly - p.hy);
        const double Ly = p.hy + st.sg * (st.lx - p.hx) + st.cg * (st.ly - p.hy);
        const bool one = i + TV <= p.nx;
        const int ia = one ? i : 0, ib = one ? i + TV - 1 : p.nx - 1, jb = one ? j : j + (i + TV - 1) / p.nx;
        const double xa = ((double)ia + .5) * p.dx, xb = ((double)ib + .5) * p.dx;
        const double ya = ((double)j + .5) * p.dy, yb = ((double)jb + .5) * p.dy;
        const double ex = fmax(0.0, fmax(xa - Lx, Lx - xb)), ey = fmax(0.0, fmax(ya - Ly, Ly - yb));
        const double A = fmax(p.bmDX0, p.a1[3]), B = fmax(p.a1[1], p.a1[4]);
        const double R = sqrt(A * A + B * B) + 2.0 * fmax(p.dx, p.dy);
        cold = ex * ex + ey * ey > R * R;
      }
      quiet = busy == 0 && cold && (zp > st.lz) == (zp > lzp) && ((zp > st.lz) || !(tS < T0));
    }
    if (!quiet)
#pragma unroll
    for (int q = 0; q < TV; ++q) {
      const int v = v0 + q;
      if (v >= d.N) break;
      const double x0 = ((double)i + .5) * p.dx;
      const double y0 = ((double)j + .5) * p.dy;
      const double zp = ((double)k + .5) * p.dz;
      double T = T0;
      if (k < kh0 || k > kh1) {
        if (!(zp > st.lz)) T = tS;
      } else if (!(zp > st.lz)) {
        const double xp = st.cg * (x0 - p.hx) + st.sg * (y0 - p.hy) + p.hx;
        const double yp = (-st.sg) * (x0 - p.hx) + st.cg * (y0 - p.hy) + p.hy;
        const double r0 = xp - st.lx, r1 = yp - st.ly, r2 = zp - st.lz;
        T = tS;
        if (st.dirp * r0 > 0) {
          if (fabs(r0) < p.bmDX0 && !(fabs(r1) > lim1) && !(fabs(r2) > lim2)) {
            const double q1 = r1 / p.a1[1], q2 = r2 / p.a1[2];
            const double dsq = q1 * q1 + q2 * q2;
            if (dsq < 1.0) T = xi;
          }
        } else if (!(fabs(r0) > lim3) && !(fabs(r1) > lim4) && !(fabs(r2) > lim5)) {
          const double q0 = r0 / p.a1[3], q1 = r1 / p.a1[4], q2 = r2 / p.a1[5];
          const double dsq = q0 * q0 + q1 * q1 + q2 * q2;
          if (dsq < 1.0) T = xi;
        }
      }
      const uint8_t s0 = sv[q];
      const bool hot = T >= tL;
      const double Told = (s0 & 0x80) ? xi : (zp > lzp ? T0 : tS);
      if (!valid || T != Told) d.T[v] = T;
      if (!(zp > st.lz)) {
        if (T > tL) {
          if (d.bj[v] != 1) d.bj[v] = 1;
        } else if (T < T0) {
          d.bj[v] = 0;
        }
      }
      uint8_t s = s0 & 3;
      if (setliquid && hot) {
        if (v < d.nxy) {
          s = 2;
        } else if (v < st.ilaserLoc * d.nxy) {
          s = 1;
          d.gid[v] = 0;
        }
        d.ext[v] = 0.0;
      }
      const uint8_t s1 = s | (s0 & 0x40) | (hot ? 0x80 : 0);
      if (s1 != s0) d.vs[v] = s1;
      anyhot = anyhot || hot;
      if (++i == p.nx) {
        i = 0;
        if (++j == p.ny) {
          j = 0;
          ++k;
        }
      }
    }
  }
  if (__any(anyhot) && (threadIdx.x & 63) == 0) O[ii].any_melt = 1;  // (every writer stores 1)
}
// After a temperature pass: the field now matches this step's laser plane.
__global__ void k_temp_commit(Inst* I, const amcd_step* S, int valid) {
  const Inst& d = I[blockIdx.x];
  if (threadIdx.x != 0 || S[blockIdx.x].skip) return;
  d.ls->tvalid = valid;
  d.ls->lz_prev = S[blockIdx.x].lz;
  d.ls->zold0 = d.ls->zhot0;
  d.ls->zold1 = d.ls->zhot1;
}

// -------------------------------------------------------------------------------------
// TempField::EASM (S/TempField.C:79-137): the temperature of a Gaussian moving source with
// 316L properties, Utilities::EASM_Temp_LG (S/Utilities.C:128-140).  Every voxel is an
// independent FP64 fixed-point problem: T -> (T + F(T))/2 with F the source integral, until a step is
// at most 10 K, or 100 times.  The properties jump at 1660 K, so where F crosses that temperature
// the iteration goes round for all 100 steps: 2.5% of the voxels of a 128x64x32 domain, the others
// take 1 to 11.  With a thread to a voxel the launch lasted for those: 101 integrals of 25
// nodes one after the other, 4250 us.  Now a thread takes its voxel through EASM_FIRST integrals, and
// what is left of a block's voxels goes to groups of 16 lanes, one or two nodes a lane, until the
// iteration repeats itself: the map has no other state than T, so a value that came back to the
// bit gives every later one.  Per node one reciprocal and one exponential (a power, three divisions
// and an exponential before).  A whole call now takes 220 us; bound by FP64 issue and the chain of
// the last voxels.
__constant__ double kGLx[AMC_GL25_N] = AMC_GL25_X;
__constant__ double kGLw[AMC_GL25_N] = AMC_GL25_W;

// Utilities::Materials_316L (S/Utilities.C:60-96): cP, k, rho at temperature T (alpha = k/(rho cP))
// (pow(10, -n) written as the literal it folds to)
__device__ static inline void mat316(double T, double& cP, double& k, double& rho) {
  if (T < 1660)
    rho = 8084.2 - 0.42086 * T - 3.8942 * 1e-5 * T * T;
  else if (T >= 1660 && T < 3090)
    rho = 7432.7 + 3.9338 * 1e-2 * T - 1.8007 * 1e-4 * T * T;
  else
    rho = 6124.72;
  cP = T < 1660 ? 458.984 + 0.1328 * T : 769.855;
  if (T < 1660)
    k = 9.248 + 1.571 * 1e-2 * T;
  else if (T >= 1660 && T < 3090)
    k = 12.41 + 3.279 * 1e-3 * T;
  else
    k = 21.6465;
}

// 1/x and 1/sqrt(x) for normal x by Newton's iteration on the hardware's estimates (within 1 ulp).
__device__ static inline double rcp_f64(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}
__device__ static inline double rsqrt_f64(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
  return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}
// exp(x) for x <= 0: 2^n times the Taylor sum of the rest, |r| <= ln(2)/2, to r^13/13! (the next term
// is 4e-18); ln(2) in two parts, the first short enough for exact products with n.
__device__ static inline double exp_neg_f64(double x) {
  x = fmax(x, -800.0);
  const double n = rint(x * 0x1.71547652b82fep+0);
  const double r = fma(-n, 0x1.ef35793c76730p-45, fma(-n, 0x1.62e42fefa3800p-1, x));
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return __builtin_amdgcn_ldexp(p, (int)n);
}

// Utilities::Integral (S/Utilities.C:105-124): 300 + the 25-point Gauss-Legendre sum over
// s in [0, t] of Temp_Fun_G (S/Utilities.C:228-249), t = 8e-4 s, sigma 50 um, eta 0.56,
// properties at the iterate T.  Nodes x = t/2 + (t/2) xi, weights (t/2) w.
constexpr double kEasmT = 80.0e-5, kEasmSigma = 50.0e-6, kEasmEta = 0.56;
struct EasmNodes {
  double x[AMC_GL25_N];   // the source's position along the track
  double ts[AMC_GL25_N];  // its age
  double w[AMC_GL25_N];   // weight / sqrt(age)
};
struct EasmProps {
  double a4;  // 4 alpha
  double C2;  // twice eta Q / (pi rho cP sqrt(4 pi alpha))
};
__device__ static inline EasmProps easm_props(double T, double Q) {
  double cP, k, rho;
  mat316(T, cP, k, rho);
  const double q = rho * cP;  // 2 / (pi rho cP sqrt(4 pi alpha)) = pi^(-3/2) / sqrt(k rho cP)
  return {4 * k * rcp_f64(q), kEasmEta * Q * 0x1.6fcb5f827b97fp-3 * rsqrt_f64(k * q)};
}
// one node's share of the sum; r2, z2: squared distances across and along z
__device__ static inline double easm_node(const EasmProps& m, double ts, double w, double r2, double z2) {
  const double a = m.a4 * ts, D = fma(m.a4, ts, 2 * (kEasmSigma * kEasmSigma));
  const double inv = rcp_f64(a * D);
  return w * exp_neg_f64(-(r2 * a + z2 * D) * inv) * (a * inv);
}

// TempField::EASM's voxel loop (S/TempField.C:90-115): 0 K above the laser plane, 0.99 T0
// ahead of the laser in the top layer, EASM_Temp_LG from 0 K elsewhere; BuildjID as the
// analytic model sets it; the "T >= tL" flag for SetLiquid3; O.any_melt collects whether
// some voxel stayed below tL (the all_of test of S/TempField.C:121-124 is its negation).
constexpr int EASM_LIM = 100, EASM_FIRST = 12;
constexpr double EASM_TOL = 10;
__global__ __launch_bounds__(GB) void k_easm(Inst* I, const int* bstart, int ninst, const amcd_step* S, amcd_out* O,
                                             double Q, double layerT, unsigned long long* n_evals) {
  __shared__ EasmNodes nd;
  __shared__ double lx[GB], ly[GB], lz[GB], lT[GB];  // voxels left after the first integrals
  __shared__ int lown[GB], nleft;
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  const amcd_step st = S[ii];
  if (st.skip) return;
  const int tid = threadIdx.x, v = (blockIdx.x - bstart[ii]) * GB + tid;
  const amcd_params& p = d.p;
  if (v == 0) {  // planes that can melt: up to the laser's (with a plane of margin)
    d.ls->zhot0 = 0;
    d.ls->zhot1 = min(p.nz - 1, (int)floor(st.lz / p.dz - 0.5) + 1);
  }
  if (tid < AMC_GL25_N) {
    const double slp = kEasmT / 2.0, x = slp + slp * kGLx[tid];
    nd.x[tid] = (st.lx - p.bmV * kEasmT) + p.bmV * x;
    nd.ts[tid] = kEasmT - x;
    nd.w[tid] = kGLw[tid] * slp / sqrt(kEasmT - x);
  }
  if (tid == 0) nleft = 0;
  __syncthreads();
  int evals = 0;
  double T = 0.0, zp = 0.0, xp = 0.0, y2 = 0.0, z2 = 0.0;
  bool solve = false;
  if (v < d.N) {
    int i, j, k;
    decode(d, v, i, j, k);
    const double x0 = ((double)i + .5) * p.dx, y0 = ((double)j + .5) * p.dy;
    zp = ((double)k + .5) * p.dz;
    if (!(zp > st.lz)) {
      xp = st.cg * (x0 - p.hx) + st.sg * (y0 - p.hy) + p.hx;
      const double yp = (-st.sg) * (x0 - p.hx) + st.cg * (y0 - p.hy) + p.hy;
      const double dy = yp - st.ly, dz = zp - st.lz;
      y2 = dy * dy;
      z2 = dz * dz;
      solve = !((x0 > st.lx) && (zp > (st.lz - layerT)));
      if (!solve) T = .99 * p.T0;
    }
  }
  bool go = solve;
  for (int n = 0; n < EASM_FIRST && __any(go); ++n) {
    const EasmProps m = easm_props(T, Q);
    double sum = 0.0;
#pragma unroll 5
    for (int q = 0; q < AMC_GL25_N; ++q) {
      const double dx = xp - nd.x[q];
      sum += easm_node(m, nd.ts[q], nd.w[q], fma(dx, dx, y2), z2);
    }
    const double F = 300 + m.C2 * sum, Tn = n == 0 ? F : 0.5 * (T + F);
    if (go) {
      ++evals;
      go = fabs(T - Tn) > EASM_TOL;
      T = Tn;
    }
  }
  // the voxels that go on, to groups of 16 lanes
  if (go) {
    const int at = atomicAdd(&nleft, 1);
    lx[at] = xp;
    ly[at] = y2;
    lz[at] = z2;
    lT[at] = T;
    lown[at] = tid;
  }
  __syncthreads();
  const int left = nleft, sub = tid & 15;
  for (int at = tid >> 4; at < left; at += GB / 16) {  // (whole groups: a voxel's lanes stay together)
    const double y2g = ly[at], z2g = lz[at], dxa = lx[at] - nd.x[sub];
    const bool two = sub + 16 < AMC_GL25_N;
    const int q2 = two ? sub + 16 : sub;
    const double dxb = lx[at] - nd.x[q2], ra = fma(dxa, dxa, y2g), rb = fma(dxb, dxb, y2g);
    const double tsa = nd.ts[sub], tsb = nd.ts[q2], wa = nd.w[sub], wb = two ? nd.w[q2] : 0.0;
    double Tg = lT[at], anchor = Tg;
    int n = EASM_FIRST - 1, lim = EASM_LIM, seen = n, next = 2 * n;
    while (n < lim) {
      const EasmProps m = easm_props(Tg, Q);
      double s = easm_node(m, tsa, wa, ra, z2g) + easm_node(m, tsb, wb, rb, z2g);
      s += dpp<0xb1>(s);   // quad_perm [1, 0, 3, 2]
      s += dpp<0x4e>(s);   // quad_perm [2, 3, 0, 1]
      s += dpp<0x141>(s);  // row_half_mirror
      s += dpp<0x140>(s);  // row_mirror
      const double Tn = 0.5 * (Tg + (300 + m.C2 * s));
      ++n;
      const bool stop = !(fabs(Tg - Tn) > EASM_TOL);
      Tg = Tn;
      if (stop) break;
      if (lim == EASM_LIM && Tg == anchor) {
        // period n - seen: the values go round until the limit, and only the rest of the last round is
        // evaluated (all of them count)
        lim = n + (EASM_LIM - n) % (n - seen);
      } else if (lim == EASM_LIM && n == next) {
        anchor = Tg;
        seen = n;
        next = 2 * n;
      }
    }
    if (sub == 0) {
      lT[at] = Tg;
      lx[at] = (double)(n == lim ? EASM_LIM + 1 : n + 1);  // integrals of this voxel
    }
  }
  __syncthreads();
  if (tid < left) {  // results back to the voxels' threads
    ly[lown[tid]] = lT[tid];
    lz[lown[tid]] = lx[tid];
  }
  __syncthreads();
  if (go) {
    T = ly[tid];
    evals = (int)lz[tid];
  }
  bool cold = false;
  if (v < d.N) {
    if (!(zp > st.lz)) {
      if (T > p.tL) d.bj[v] = 1;
      else if (T < p.T0) d.bj[v] = 0;
    }
    d.T[v] = T;
    const bool hot = T >= p.tL;
    cold = !hot;
    d.vs[v] = (d.vs[v] & 3) | (hot ? 0x80 : 0);
  }
  if (__any(cold) && (tid & 63) == 0) O[ii].any_melt = 1;
  for (int m = 32; m >= 1; m >>= 1) evals += __shfl_xor(evals, m);
  if ((tid & 63) == 0 && evals) atomicAdd(n_evals, (unsigned long long)evals);
}

// SetLiquid3 (S/VoxelsCA.C:1098-1116) when the temperature kernel ran without it.
__global__ __launch_bounds__(GB) void k_setliquid(Inst* I, const int* bstart, int ninst, const amcd_step* S) {
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  if (S[ii].skip) return;
  int v = (blockIdx.x - bstart[ii]) * GB + threadIdx.x;
  if (v >= d.N) return;
  uint8_t s = d.vs[v];
  if (!(s & 0x80)) return;
  uint8_t st = s & 3;
  if (v < d.nxy) {
    st = 2;
  } else if (v < S[ii].ilaserLoc * d.nxy) {
    st = 1;
    d.gid[v] = 0;
  }
  d.ext[v] = 0.0;
  d.vs[v] = st | 0x80;
}

// A run of up to 16 consecutive voxels from v0 on, whatever rows it lies in: bit q of xlo, xhi, ylo,
// yhi, zlo, zhi says that voxel v0 + q is on that side of the domain.
struct RunEdges {
  unsigned xlo, xhi, ylo, yhi, zlo, zhi;
};
__device__ static inline RunEdges run_edges(const Inst& d, int v0) {
  const int nx = d.p.nx, ny = d.p.ny, nz = d.p.nz;
  int i, j, k;
  decode(d, v0, i, j, k);
  RunEdges e = {0, 0, 0, 0, 0, 0};
  if (i + 16 <= nx) {  // within a row
    e.xlo = i == 0 ? 1u : 0u;
    e.xhi = i + 16 == nx ? 1u << 15 : 0u;
    e.ylo = j == 0 ? ~0u : 0u;
    e.yhi = j == ny - 1 ? ~0u : 0u;
    e.zlo = k == 0 ? ~0u : 0u;
    e.zhi = k == nz - 1 ? ~0u : 0u;
    return e;
  }
  for (int q = 0; q < 16;) {  // row by row
    const int len = min(16 - q, nx - i);
    const unsigned m = ((1u << len) - 1) << q;
    e.xlo |= i == 0 ? 1u << q : 0u;
    e.xhi |= i + len == nx ? 1u << (q + len - 1) : 0u;
    e.ylo |= j == 0 ? m : 0u;
    e.yhi |= j == ny - 1 ? m : 0u;
    e.zlo |= k == 0 ? m : 0u;
    e.zhi |= k >= nz - 1 ? m : 0u;
    q += len;
    i = 0;
    if (++j == ny) {
      j = 0;
      ++k;
    }
  }
  return e;
}
// Four state bytes at a time: bit 0 of each byte of the result is set for ...
__device__ static inline unsigned bytes_liquid(unsigned x) { return x & ~(x >> 1) & 0x01010101u; }
__device__ static inline unsigned bytes_solid(unsigned x) { return x & (x >> 1) & 0x01010101u; }
__device__ static inline unsigned bytes_cool(unsigned x) {  // mushy, or liquid below tL
  return ((x >> 1) & ~x & 0x01010101u) | (x & ~(x >> 1) & ~(x >> 7) & 0x01010101u);
}
// bit 0 of the four bytes to four adjacent bits
__device__ static inline unsigned pack_bytes(unsigned b) { return (b * 0x10204080u) >> 28; }
// Bit q: a Moore neighbour of voxel v0 + q has a state byte that `pred` marks.  Each of the nine rows
// around the run is a run of 18 bytes itself (the run moved by the row's offset, and one byte to
// either side), read with one 16-byte and one 4-byte load at whatever alignment it has; neighbours
// across the domain's sides are masked out.  (Reads reach up to 20 bytes beyond the array, inside
// the 256 that every device array is allocated beyond its length.)  Runs that span rows had gone
// voxel by voxel, byte by byte: on 40x24x20 voxels k_solid_to_mushy 58 -> 4.8 us and k_active_flags
// 62 -> 5.1 us; rows of a multiple of 16 (512x512x128, aligned loads before) 14.9 -> 15.3 and 20.3 ->
// 16.8 us, so this is the only form.
template <class Pred>
__device__ static inline unsigned moore_marks(const Inst& d, int v0, const RunEdges& e, Pred pred) {
  // (all nine rows' loads before the first use: one round of latency; a row outside the domain reads
  // its nearest bytes and is masked)
  uint4 w[9];
  unsigned w4[9];
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int at = min(max(v0 + (r / 3 - 1) * d.nxy + (r % 3 - 1) * d.p.nx - 1, 0), d.N);
    __builtin_memcpy(&w[r], d.vs + at, 16);
    __builtin_memcpy(&w4[r], d.vs + at + 16, 4);
  }
  unsigned near = 0;
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int dz = r / 3 - 1, dy = r % 3 - 1, first = v0 + dz * d.nxy + dy * d.p.nx - 1;
    const unsigned out = (dz < 0 ? e.zlo : dz > 0 ? e.zhi : 0u) | (dy < 0 ? e.ylo : dy > 0 ? e.yhi : 0u);
    unsigned m = pack_bytes(pred(w[r].x)) | pack_bytes(pred(w[r].y)) << 4 | pack_bytes(pred(w[r].z)) << 8 |
                 pack_bytes(pred(w[r].w)) << 12 | (pack_bytes(pred(w4[r])) & 3u) << 16;
    m <<= min(max(-first, 0), 18);  // bit q: voxel v0 + q - 1 of the row
    near |= ((m & ~e.xlo) | (m >> 1) | ((m >> 2) & ~e.xhi)) & ~out;
  }
  return near;
}

// ConvertSolid1(1): solid -> mushy when any Moore neighbour is liquid.  Updating in
// place is equivalent to the reference's collect-then-apply, because the update
// (3 -> 2) never changes the predicate (some neighbour == 1) of any other voxel.
__global__ __launch_bounds__(GB) void k_solid_to_mushy(Inst* I, const int* bstart, int ninst, const amcd_step* S) {
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  if (S[ii].skip) return;
  const int nz = d.p.nz;
  const int b0 = (blockIdx.x - bstart[ii]) * SB;
  const int bend = min(d.N, b0 + SB);
  // liquid exists only in planes that held it at the last active-set pass or that the
  // last temperature evaluation could melt: a block with no such plane within one plane
  // of its own leaves at once
  const int h0 = d.ls->zhot0, h1 = d.ls->zhot1;
  const int zb0 = b0 / d.nxy, zb1 = (bend - 1) / d.nxy;
  bool any = false;
  const unsigned* zliq = d.zliq + (size_t)d.ls->zpar * nz;
  for (int z = max(0, zb0 - 1); z <= min(nz - 1, zb1 + 1); ++z) any = any || (zliq[z] & 1u) || (z >= h0 && z <= h1);
  if (!any) return;
  // A solid voxel with a liquid Moore neighbour turns mushy.  Each thread takes 16 consecutive
  // voxels and reads the nine rows around them (moore_marks).  Liquid voxels are not changed by
  // the pass, so every test reads settled states, and each thread writes its own voxels only.
  // Bound by latency: 15 us for 512x512x128 (mostly blocks that leave at once), 4.8 us for 40x24x20.
  constexpr int PT = SB / GB;
  const int v0 = b0 + (int)threadIdx.x * PT;
  if (v0 >= bend) return;
  const uint4 c = *reinterpret_cast<const uint4*>(d.vs + v0);  // (beyond the domain's end: not solid)
  const unsigned cw[4] = {c.x, c.y, c.z, c.w};
  unsigned sol = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) sol |= pack_bytes(bytes_solid(cw[r])) << (4 * r);
  if (v0 + PT > d.N) sol &= (1u << (d.N - v0)) - 1;
  if (!sol) return;
  const unsigned m = sol & moore_marks(d, v0, run_edges(d, v0), bytes_liquid);
  if (!m) return;
  unsigned nw[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) nw[r] = cw[r] & ~(((m >> (4 * r)) & 15u) * 0x204081u & 0x01010101u);  // 3 -> 2
  if (v0 + PT <= d.N) {
    *reinterpret_cast<uint4*>(d.vs + v0) = make_uint4(nw[0], nw[1], nw[2], nw[3]);
  } else {
    for (int q = 0; q < d.N - v0; ++q) d.vs[v0 + q] = (uint8_t)(nw[q >> 2] >> (8 * (q & 3)));
  }
}

// Active set: {mushy} U {liquid below tL} U {neighbours at or above tL of those}.
// Writes bit 6 of vs and the per-block (ZB voxels) counts of active and mushy cells.
// One wave per block of ZB voxels (four per workgroup), 16 consecutive voxels per thread,
// four state bytes at a time: per byte, bit 0 of lo/hi/hb is state bit 0, state bit 1
// and the hot flag.
__global__ __launch_bounds__(256) void k_active_flags(Inst* I, const int* bstart, int ninst, const amcd_step* S) {
  constexpr int PT = ZB / 64;
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  if (S[ii].skip) return;
  const int blk = (blockIdx.x - bstart[ii]) * 4 + (int)(threadIdx.x >> 6);
  if (blk >= d.nblkZ) return;  // whole waves leave: nothing below synchronises the block
  const int lane = threadIdx.x & 63;
  const int v0 = blk * ZB + lane * PT;
  int na = 0, nm = 0;
  unsigned liq = 0;  // bit q: voxel v0 + q is liquid
  if (v0 < d.N) {
    const int nq = min(PT, d.N - v0);
    unsigned w[4] = {0, 0, 0, 0};
    if (nq == PT) {
      const uint4 x = *reinterpret_cast<const uint4*>(d.vs + v0);
      w[0] = x.x;
      w[1] = x.y;
      w[2] = x.z;
      w[3] = x.w;
    } else {
      for (int q = 0; q < nq; ++q) w[q >> 2] |= (unsigned)d.vs[v0 + q] << (8 * (q & 3));
    }
    const unsigned valid = nq == PT ? 0xffffu : (1u << nq) - 1;
    // hot voxels that are neither mushy nor cool liquid ask their Moore neighbours
    unsigned hotpend = 0;  // bit q: voxel v0 + q is hot and not active by itself
#pragma unroll
    for (int r = 0; r < 4; ++r) hotpend |= pack_bytes((w[r] >> 7) & 0x01010101u & ~bytes_cool(w[r])) << (4 * r);
    hotpend &= valid;
    unsigned nearA = 0;  // bit q: a Moore neighbour of voxel v0 + q is mushy or cool liquid
    if (hotpend) nearA = moore_marks(d, v0, run_edges(d, v0), bytes_cool);
    unsigned nw[4];
    bool changed = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned x = w[r];
      const unsigned lo = x & 0x01010101u, hi = (x >> 1) & 0x01010101u, hb = (x >> 7) & 0x01010101u;
      // bytes of this word inside the domain; hot bytes with an active neighbour
      const unsigned vb = ((valid >> (4 * r)) & 15u) * 0x204081u & 0x01010101u;
      const unsigned nb = (((hotpend & nearA) >> (4 * r)) & 15u) * 0x204081u & 0x01010101u;
      const unsigned mu = hi & ~lo & vb, lq = lo & ~hi & vb;
      const unsigned ac = mu | (lq & ~hb) | nb;
      nw[r] = (x & ~0x40404040u) | (ac << 6);
      changed = changed || nw[r] != x;
      na += __popc(ac);
      nm += __popc(mu);
      liq |= pack_bytes(lq) << (4 * r);
    }
    if (changed) {
      if (nq == PT) {
        *reinterpret_cast<uint4*>(d.vs + v0) = make_uint4(nw[0], nw[1], nw[2], nw[3]);
      } else {
        for (int q = 0; q < nq; ++q) d.vs[v0 + q] = (uint8_t)(nw[q >> 2] >> (8 * (q & 3)));
      }
    }
  }
  // planes holding liquid now (for the next step's solid->mushy pass): one atomic per
  // wave and plane, and none once the flag is seen set.  A run of 16 spans at most two
  // planes unless a plane holds fewer than 16 voxels.
  unsigned* zliq = d.zliq + (size_t)(1 - d.ls->zpar) * d.p.nz;
  int lp0 = -1, lp1 = -1;
  if (liq) {
    lp0 = (v0 + __builtin_ctz(liq)) / d.nxy;
    lp1 = (v0 + 31 - __builtin_clz(liq)) / d.nxy;
    if (d.nxy < PT)
      for (unsigned m = liq; m; m &= m - 1) {
        const int kz = (v0 + __builtin_ctz(m)) / d.nxy;
        if (!(zliq[kz] & 1u)) atomicOr(&zliq[kz], 1u);
      }
  }
  for (int pass = 0; pass < 2; ++pass) {
    const int pz = pass ? lp1 : lp0;
    unsigned long long pend = __ballot(pz >= 0);
    while (pend) {
      const int leader = __builtin_ctzll(pend);
      const int zl = __builtin_amdgcn_readlane(pz, leader);
      pend &= ~__ballot(pz == zl);
      if (lane == leader && !(zliq[zl] & 1u)) atomicOr(&zliq[zl], 1u);
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    na += __shfl_xor(na, o);
    nm += __shfl_xor(nm, o);
  }
  if (lane == 0) {
    d.bcA[blk] = na;
    d.bcM[blk] = nm;
  }
}

// Exclusive scan of the per-block counts in two levels, and the step's loop state: chunks of 1024
// blocks scanned by one workgroup each (offsets within the chunk, chunk totals); the instance's last
// chunk to be done scans the totals.  It also seeds the loop's engine (after the Na cells' two
// draws each, S/VoxelsCA.C:380), takes over the laser plane of the temperature (`commit`) and swaps
// the liquid-plane marks.  A pass of a few microseconds that is launch latency, so everything
// that is one workgroup's work between the flags and the compaction is in it: as five launches
// (chunks, totals, engine, laser plane, marks) it took 23 us of a step.
__global__ __launch_bounds__(1024) void k_scan(Inst* I, const int* cstart, int ninst, const amcd_step* S, amcd_out* O,
                                               int commit) {
  __shared__ int wa[16], wm[16], last;
  const int ii = find_inst(cstart, ninst, blockIdx.x);
  const Inst& d = I[ii];
  const int c = blockIdx.x - cstart[ii], nc = cstart[ii + 1] - cstart[ii];
  const int b = c * 1024 + (int)threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  LoopState* ls = d.ls;
  int a = 0, m = 0;
  if (b < d.nblkZ) {
    a = d.bcA[b];
    m = d.bcM[b];
  }
  int ia = a, im = m;
  for (int o = 1; o < 64; o <<= 1) {
    const int ta = __shfl_up(ia, o), tm = __shfl_up(im, o);
    if (lane >= o) {
      ia += ta;
      im += tm;
    }
  }
  if (lane == 63) {
    wa[w] = ia;
    wm[w] = im;
  }
  __syncthreads();
  int pa = 0, pm = 0;
  for (int q = 0; q < w; ++q) {
    pa += wa[q];
    pm += wm[q];
  }
  if (b < d.nblkZ) {
    d.bcA[b] = pa + ia - a;
    d.bcM[b] = pm + im - m;
  }
  if (threadIdx.x == 1023) {
    __hip_atomic_store(&d.chA[c], pa + ia, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&d.chM[c], pm + im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // every chunk's totals are there when the count is complete
    last = nc == 1 || __hip_atomic_fetch_add(&ls->chunks, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == nc - 1;
  }
  __syncthreads();
  if (!last) return;
  const amcd_step st = S[ii];
  if (!st.skip) {
    const int zp = ls->zpar;
    for (int z = threadIdx.x; z < d.p.nz; z += 1024) d.zliq[(size_t)zp * d.p.nz + z] = 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
      ls->zpar = 1 - zp;
      if (commit) {
        ls->tvalid = 1;
        ls->lz_prev = st.lz;
        ls->zold0 = ls->zhot0;
        ls->zold1 = ls->zhot1;
      }
    }
  }
  if (w != 0) return;
  // the chunk totals, 64 at a time
  int Na = 0, Nm = 0;
  for (int c0 = 0; c0 < nc; c0 += 64) {
    const bool in = c0 + lane < nc;
    const int va = in ? __hip_atomic_load(&d.chA[c0 + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    const int vm = in ? __hip_atomic_load(&d.chM[c0 + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    int xa = va, xm = vm;
    for (int o = 1; o < 64; o <<= 1) {
      const int ta = __shfl_up(xa, o), tm = __shfl_up(xm, o);
      if (lane >= o) {
        xa += ta;
        xm += tm;
      }
    }
    if (in) {
      d.chA[c0 + lane] = Na + xa - va;
      d.chM[c0 + lane] = Nm + xm - vm;
    }
    Na += __shfl(xa, 63);
    Nm += __shfl(xm, 63);
  }
  if (lane == 0) {
    if (st.skip) Na = Nm = 0;
    ls->chunks = 0;
    ls->Na = Na;
    ls->nmushy0 = Nm;
    ls->nslots = 0;
    ls->nslots_pre = -1;
    ls->npre = 0;
    ls->vSind2 = Nm;
    ls->tinc = 0.0;
    ls->events = ls->captures = ls->nucs = 0;
    ls->pool_used = 0;
    ls->pending = 0;
    ls->fin = 0;
    ls->done = st.skip || Na > d.acap;
    ls->nGrain = st.nGrain;
    if (!ls->done) {
      ls->rng = lcg_skip_cells(lcg_seed(30ull * (unsigned long long)st.tInd + d.p.seed1), (unsigned)Na);
      ls->draws = 2ll * Na;
    }
    amcd_out& o = O[ii];
    o.n_active = Na;
    o.n_mushy0 = Nm;
    if (Na > d.acap) {
      o.overflow = 1;
      o.status = -2;
    }
  }
}

// Ordered compaction: the active list in ascending voxel id, the voxel -> active map,
// gathers of the per-cell state, the scan position of mushy cells and the uniform
// draws ruq (S/VoxelsCA.C:380): the engine is seeded with 30*tInd+seed1 and active
// cell a takes engine outputs 2a+1 and 2a+2 (jump-ahead 16807^(2a)).
__global__ __launch_bounds__(256) void k_compact(Inst* I, const int* bstart, int ninst, const amcd_step* S) {
  // one wave per block of ZB voxels (four per workgroup), 16 consecutive voxels per thread
  constexpr int PT = ZB / 64;
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  if (d.ls->done) return;
  const int blk = (blockIdx.x - bstart[ii]) * 4 + (int)(threadIdx.x >> 6);
  if (blk >= d.nblkZ) return;
  // a block without active cells (its global offset equals the next block's) has nothing
  // to write; most of the domain is such blocks
  const int o0 = d.bcA[blk] + d.chA[blk >> 10];
  const int o1 = blk + 1 < d.nblkZ ? d.bcA[blk + 1] + d.chA[(blk + 1) >> 10] : d.ls->Na;
  if (o1 == o0) return;
  const int lane = threadIdx.x & 63;
  const int v0 = blk * ZB + lane * PT;
  unsigned am = 0, mm = 0;  // bit q: voxel v0 + q is active / mushy
  if (v0 < d.N) {
    const int nq = min(PT, d.N - v0);
    if (nq == PT) {
      const uint4 x = *reinterpret_cast<const uint4*>(d.vs + v0);
      const unsigned w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int q = 0; q < PT; ++q) {
        const unsigned b = (w[q >> 2] >> (8 * (q & 3))) & 0xffu;
        am |= ((b >> 6) & 1u) << q;
        mm |= ((b & 3u) == 2u ? 1u : 0u) << q;
      }
    } else {
      for (int q = 0; q < nq; ++q) {
        const unsigned b = d.vs[v0 + q];
        am |= ((b >> 6) & 1u) << q;
        mm |= ((b & 3u) == 2u ? 1u : 0u) << q;
      }
    }
  }
  // exclusive prefix over the wave's lanes of the active and mushy counts (voxel order)
  const int ca = __popc(am), cm = __popc(mm);  // (mushy voxels are active)
  int ia = ca, im = cm;
  for (int o = 1; o < 64; o <<= 1) {
    const int ta = __shfl_up(ia, o), tm = __shfl_up(im, o);
    if (lane >= o) {
      ia += ta;
      im += tm;
    }
  }
  const int ea = ia - ca, em = im - cm;  // this lane's exclusive prefixes
  const int total = __shfl(ia, 63);
  const int m0 = d.bcM[blk] + d.chM[blk >> 10];
  const unsigned int x0 = lcg_seed(30ull * (unsigned long long)S[ii].tInd + d.p.seed1);
  // the block's active voxels, 64 at a time: lane L takes the (base + L)-th of them, found
  // by a binary search over the lanes' prefixes and a walk over that lane's mask
  for (int base = 0; base < total; base += 64) {
    const int idx = base + lane;
    int t = 0;  // the lane holding voxel idx: the last lane whose prefix is <= idx
    for (int step = 32; step >= 1; step >>= 1) {
      const int c = t + step;
      const int ec = __shfl(ea, c < 64 ? c : 63);
      if (c < 64 && ec <= idx) t = c;
    }
    const unsigned mt = (unsigned)__shfl((int)am, t), mmt = (unsigned)__shfl((int)mm, t);
    const int et = __shfl(ea, t), emt = __shfl(em, t);
    if (idx >= total) continue;
    unsigned m = mt;
    for (int r = idx - et; r > 0; --r) m &= m - 1;
    const int q = __builtin_ctz(m);
    const int v = blk * ZB + t * PT + q;
    const int a = o0 + idx;
    const bool mushy = (mmt >> q) & 1u;
    d.aVox[a] = v;
    d.amap[v] = a;
    d.aVS[a] = d.vs[v] & 3;
    d.aT[a] = d.T[v];
    if (mushy) {  // (a liquid cell's are written when it is captured)
      d.aG[a] = d.gid[v];
      d.aExt[a] = d.ext[v];
      d.aCx[a] = d.cx[v];
      d.aCy[a] = d.cy[v];
      d.aCz[a] = d.cz[v];
    }
    d.aScan[a] = mushy ? m0 + emt + __popc(mmt & ((1u << q) - 1)) : -1;
    const unsigned int x1 = lcg_next(lcg_skip_cells(x0, (unsigned)a));
    const unsigned int x2 = lcg_next(x1);
    d.ruq[a] = (canonical(x1, x2) - .5) * d.p.dx / 100.;
  }
}

// Voxel centre, S/VoxelsCA.C:409-414.
template <class DI>
__device__ static inline void centre(DI& d, int v, double* c) {
  int i, j, k;
  decode(d, v, i, j, k);
  c[0] = ((double)i + .5) * d.p.dx;
  c[1] = ((double)j + .5) * d.p.dy;
  c[2] = ((double)k + .5) * d.p.dz;
}

// Capture candidate of growing cell a (centroid c, rotation R) towards liquid voxel
// vt: D = pow(cos th sin ph,.5) * |R^T dnx|_1 and the factor f (S/VoxelsCA.C:409-424).
__device__ static inline void candidate_at(const double* ct, const double* c, const double* R, double* D, double* f) {
  double dnx0 = ct[0] - c[0], dnx1 = ct[1] - c[1], dnx2 = ct[2] - c[2];
  double ff = amc_shape_factor(dnx0, dnx1, dnx2);
  double d0 = fabs(R[0] * dnx0 + R[3] * dnx1 + R[6] * dnx2);
  double d1 = fabs(R[1] * dnx0 + R[4] * dnx1 + R[7] * dnx2);
  double d2 = fabs(R[2] * dnx0 + R[5] * dnx1 + R[8] * dnx2);
  *D = ff * (d0 + d1 + d2);
  *f = ff;
}
__device__ static inline void candidate(const Inst& d, const double* c, const double* R, int vt, double* D,
                                        double* f) {
  double ct[3];
  centre(d, vt, ct);
  double dnx0 = ct[0] - c[0], dnx1 = ct[1] - c[1], dnx2 = ct[2] - c[2];
  double ff = amc_shape_factor(dnx0, dnx1, dnx2);
  double d0 = fabs(R[0] * dnx0 + R[3] * dnx1 + R[6] * dnx2);
  double d1 = fabs(R[1] * dnx0 + R[4] * dnx1 + R[7] * dnx2);
  double d2 = fabs(R[2] * dnx0 + R[5] * dnx1 + R[8] * dnx2);
  *D = ff * (d0 + d1 + d2);
  *f = ff;
}

// vhat = Avel * pow(tL - T, nvel) (S/VoxelsCA.C:405), pow rounded to nearest; the two
// temperatures of the analytic model are precomputed, any other (EASM) is evaluated here.
template <class P>
__device__ static inline double growth_velocity(P& p, double T) {
  if (T >= p.tL) return 0.0;
  if (T == p.tS) return p.vhat_tS;
  if (T == p.T0) return p.vhat_T0;
  return p.Avel * amc_pow_cr(p.tL - T, p.nvel);
}

// Active-neighbour table and, for every growing cell (mushy, some liquid active
// neighbour, all active neighbours below tL; S/VoxelsCA.C:396-397), its slot in the
// growing list and its capture candidates.  Slot order is irrelevant: the event loop
// compares candidates by (time, ruqs, scan position, neighbour rank).  Bound by the latency of its
// loads: as 26 indices with a temperature and a state behind each, 11.8 us for 40x24x20 voxels and 15.4
// for 256x192x64; as nine rows of three indices and four state bytes, side by side, 6.5 and 9.8.
__device__ static inline bool cand_less(double Da, double Ra, int ka, double Db, double Rb, int kb);

__global__ __launch_bounds__(GB) void k_active_setup(Inst* I, const int* bstart, int ninst, amcd_out* O) {
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const int Na = I[ii].ls->Na, nb = bstart[ii + 1] - bstart[ii], b0 = blockIdx.x - bstart[ii];
  if (I[ii].ls->done || b0 * GB >= Na) return;  // (before the descriptor is read)
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  for (int a = b0 * GB + (int)threadIdx.x; __any(a < Na); a += nb * GB) {
    bool grow = false;
    if (a < Na) {
      int v = d.aVox[a];
      int i, j, k;
      decode(d, v, i, j, k);
      CellRow row;
      // A row of three neighbours at a time: their active indices and state bytes (active: bit 6, at or
      // above tL: bit 7), all rows' loads before the first use; a row outside the domain reads the
      // voxel's own and is masked.
      struct Three {
        int n[3];
      };
      Three tn[9];
      unsigned ts[9];
#pragma unroll
      for (int r = 0; r < 9; ++r) {
        const int y = j + r % 3 - 1, z = k + r / 3 - 1;
        const bool in = y >= 0 && y < d.p.ny && z >= 0 && z < d.p.nz;
        const int at = max(in ? v + (r / 3 - 1) * d.nxy + (r % 3 - 1) * d.p.nx - 1 : v - 1, 0);
        __builtin_memcpy(&tn[r], d.amap + at, 12);
        __builtin_memcpy(&ts[r], d.vs + at, 4);
      }
      bool cold = true, liq = false;
#pragma unroll
      for (int r = 0; r < 9; ++r) {
        const int y = j + r % 3 - 1, z = k + r / 3 - 1;
        const bool in = y >= 0 && y < d.p.ny && z >= 0 && z < d.p.nz;
        const bool first = v + (r / 3 - 1) * d.nxy + (r % 3 - 1) * d.p.nx == 0;  // (its left neighbour is before the array)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          if (r == 4 && c == 1) continue;
          const int x = i + c - 1, q = 3 * r + c - (3 * r + c > 13 ? 1 : 0);
          const int n3 = first ? tn[r].n[c > 0 ? c - 1 : 0] : tn[r].n[c];
          const unsigned b = (first ? ts[r] << 8 : ts[r]) >> (8 * c);
          const int n = in && x >= 0 && x < d.p.nx ? n3 : -1;
          row.nbr[q] = n;
          cold = cold && !(n >= 0 && (b & 0x80u));
          liq = liq || (n >= 0 && (b & 3u) == 1u);
        }
      }
      row.vox = v;
      row.cold = cold;
      row.T = d.aT[a];
      row.pad[0] = row.pad[1] = 0;
      d.aRow[a] = row;
      grow = cold && liq && d.aVS[a] == 2;
    }
    unsigned long long bal = __ballot(grow);
    if (!bal) continue;
    int lane = threadIdx.x & 63;
    int leader = __ffsll((long long)bal) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&d.ls->nslots, __popcll(bal));
    base = __shfl(base, leader);
    if (!grow) continue;
    unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int slot = base + __popcll(bal & lt);
    d.gExt[slot] = d.aExt[a];
    d.gVhat[slot] = growth_velocity(d.p, d.aT[a]);
    const int G = d.aG[a];
    const bool bad = G < 1 || G > d.gcap;  // a growing cell must carry a valid grain
    if (bad) atomicOr(&O[ii].err_state, 1);
    d.slots[slot] = {{d.aCx[a], d.aCy[a], d.aCz[a]}, d.aVox[a], G, a, d.aScan[a], d.precap + slot * AMCD_NB, bad ? -1 : 0};
  }
}

// Re-centring of the decentred octahedron after a capture, S/VoxelsCA.C:528-605 and
// the helpers S/VoxelsCA.h:56-93.  R is row-major (local -> global), f is the
// capturing candidate's shape factor.  Outputs the new centroid and half-diagonal.
__device__ static inline void project_point_line(const double* A, const double* x0, const double* x1, double* xp) {
  double n[3], snorm, dd, t;
  snorm = sqrt((x1[0] - x0[0]) * (x1[0] - x0[0]) + (x1[1] - x0[1]) * (x1[1] - x0[1]) +
               (x1[2] - x0[2]) * (x1[2] - x0[2]));
  n[0] = (x1[0] - x0[0]) / snorm;
  n[1] = (x1[1] - x0[1]) / snorm;
  n[2] = (x1[2] - x0[2]) / snorm;
  dd = -(n[0] * A[0] + n[1] * A[1] + n[2] * A[2]);
  t = (-dd - n[0] * x0[0] - n[1] * x0[1] - n[2] * x0[2]) /
      (n[0] * (x1[0] - x0[0]) + n[1] * (x1[1] - x0[1]) + n[2] * (x1[2] - x0[2]));
  xp[0] = x0[0] + (x1[0] - x0[0]) * t;
  xp[1] = x0[1] + (x1[1] - x0[1]) * t;
  xp[2] = x0[2] + (x1[2] - x0[2]) * t;
}
__device__ static inline double dist3(const double* p, const double* q) {
  return sqrt((p[0] - q[0]) * (p[0] - q[0]) + (p[1] - q[1]) * (p[1] - q[1]) + (p[2] - q[2]) * (p[2] - q[2]));
}
template <class DI>
__device__ static inline void recentre(DI& d, int vcap, int vnew, const double* cen, const double* R, double f,
                                double* ncen, double* next) {
  auto& p = d.p;
  int jx0, jx1, jx2, jy0, jy1, jy2;
  decode(d, vnew, jx0, jx1, jx2);
  decode(d, vcap, jy0, jy1, jy2);
  double l0 = (jx0 - jy0) * p.dx, l1 = (jx1 - jy1) * p.dy, l2 = (jx2 - jy2) * p.dz;
  double l = sqrt(l0 * l0 + l1 * l1 + l2 * l2);
  double dnx[3], locX[3];
  dnx[0] = ((double)jx0 + .5) * p.dx - cen[0];
  dnx[1] = ((double)jx1 + .5) * p.dy - cen[1];
  dnx[2] = ((double)jx2 + .5) * p.dz - cen[2];
  locX[0] = R[0] * dnx[0] + R[3] * dnx[1] + R[6] * dnx[2];
  locX[1] = R[1] * dnx[0] + R[4] * dnx[1] + R[7] * dnx[2];
  locX[2] = R[2] * dnx[0] + R[5] * dnx[1] + R[8] * dnx[2];
  double dr = fabs(locX[0]) + fabs(locX[1]) + fabs(locX[2]);
  // octahedron vertices +-dr e_i (vertex c is +dr e_c, vertex c+3 is -dr e_c); the octant's
  // three vertices in ascending vertex order, the reference's table of S/VoxelsCA.h:61-76
  // ({0,1,2},{1,2,3},{0,2,4},{2,3,4},{0,1,5},{1,3,5},{0,4,5},{3,4,5} by octant), computed
  // instead of looked up so that no memory access sits in the chain
  const int a0 = signbit(locX[0]) ? 3 : 0, a1 = signbit(locX[1]) ? 4 : 1, a2 = signbit(locX[2]) ? 5 : 2;
  const int vlo = min(min(a0, a1), a2), vhi = max(max(a0, a1), a2);
  const int vsel[3] = {vlo, a0 + a1 + a2 - vlo - vhi, vhi};
  double V[3][3], S0[3][3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    int vi = vsel[q];
    for (int c = 0; c < 3; ++c) {
      double sgn = (vi % 3 == c) ? (vi < 3 ? 1.0 : -1.0) : 0.0;
      S0[q][c] = sgn;
      V[q][c] = sgn * dr;
    }
  }
  double dn[3];
  for (int q = 0; q < 3; ++q)
    dn[q] = (locX[0] - V[q][0]) * (locX[0] - V[q][0]) + (locX[1] - V[q][1]) * (locX[1] - V[q][1]) +
            (locX[2] - V[q][2]) * (locX[2] - V[q][2]);
  int k0 = 0, k2 = 0;
  for (int q = 1; q < 3; ++q) {
    if (dn[q] < dn[k0]) k0 = q;   // std::min_element: first minimum
    if (dn[k2] < dn[q]) k2 = q;   // std::max_element: first maximum
  }
  int k1;
  if (k0 == k2) {
    k0 = 0; k1 = 1; k2 = 2;
  } else {
    k1 = 3 - k0 - k2;
  }
  double xI[3], xJ[3];
  project_point_line(locX, V[k0], V[k1], xI);
  project_point_line(locX, V[k0], V[k2], xJ);
  double d1I = dist3(V[k0], xI), dI2 = dist3(V[k1], xI), d1J = dist3(V[k0], xJ), dJ3 = dist3(V[k2], xJ);
  const double sq3 = 0x1.bb67ae8584caap+0;   // pow(3.0,.5), folded by the reference's compiler
  const double s23 = 0x1.a20bd700c2c3ep-1;   // pow(2.0/3.0,.5)
  double m = sq3 * l;
  double L12 = .5 * ((m < d1I ? m : d1I) + (m < dI2 ? m : dI2));
  double L13 = .5 * ((m < d1J ? m : d1J) + (m < dJ3 ? m : dJ3));
  double Lmud = sq3 * (s23 * (L12 < L13 ? L13 : L12));
  *next = f * Lmud * 1.0;
  dnx[0] = V[k0][0] - Lmud * S0[k0][0];
  dnx[1] = V[k0][1] - Lmud * S0[k0][1];
  dnx[2] = V[k0][2] - Lmud * S0[k0][2];
  locX[0] = R[0] * dnx[0] + R[1] * dnx[1] + R[2] * dnx[2];
  locX[1] = R[3] * dnx[0] + R[4] * dnx[1] + R[5] * dnx[2];
  locX[2] = R[6] * dnx[0] + R[7] * dnx[1] + R[8] * dnx[2];
  ncen[0] = cen[0] + locX[0];
  ncen[1] = cen[1] + locX[1];
  ncen[2] = cen[2] + locX[2];
}

// Candidate lists of the growing cells (S/VoxelsCA.C:396-440): one wave per slot, lane q
// evaluates neighbour q when it is liquid, and the entries are placed by rank in (D, ruqs,
// neighbour) order -- the order the capture loop reads the list in.
//
// What a capture through an entry does depends, but for the voxels captured before it, on the
// entry alone: the re-centred octahedron, the new cell's velocity and its candidates.  They are
// evaluated here for every entry, over the whole chip, instead of on the capture loop's one compute
// unit: the re-centring by the entry's lane, the new cell's sorted list two entries at a time (a
// half wave each), with the re-centring of its own entries and a single-precision bound on the time
// to the captures after them.  Only for the captures that the step has time for: a cell grows half a
// voxel a step, which leaves about a third of the entries.  Bound by the latency of a wave's own
// chain, not by the chip (a few thousand waves): averaged over a run's steps 36 us for the 512x512x128
// raster (49 us at its 3.2 thousand growing cells), 38 us for 256x192x64 (106 us at 6 thousand) and 21 us
// for 40x24x20 (33 us at 200).  With lists ahead for every entry the runs' averages were 64, 109 and
// 38 us, in the first and last without any 18 and 15 us; with the lists ahead the loop's windows end
// later: 3291 -> 2863 cycles per event in the first deck.
__device__ static inline int list_rank(double D, double r, bool on, int half) {
  // position in (D, ruqs, neighbour) order among the entries of this lane's half wave (all of it
  // for half < 0), NaN distances last
  const int lane = threadIdx.x & 63, q = half < 0 ? lane : lane & 31;
  const unsigned long long bal = __ballot(on);
  const unsigned mine = half < 0 ? (unsigned)bal : (half ? (unsigned)(bal >> 32) : (unsigned)bal);
  const unsigned any = half < 0 ? (unsigned)bal : (unsigned)bal | (unsigned)(bal >> 32);
  int rank = 0;
  for (unsigned b = any; b != 0; b &= b - 1) {
    const int j = __builtin_ctz(b);
    double Dj = lane_f64(D, j), rj = lane_f64(r, j);
    if (half >= 0) {
      const double Dh = lane_f64(D, j + 32), rh = lane_f64(r, j + 32);
      Dj = half ? Dh : Dj;
      rj = half ? rh : rj;
    }
    rank += ((mine >> j) & 1u) != 0 && j != q && cand_less(Dj, rj, j, D, r, q) ? 1 : 0;
  }
  return rank;
}
// Capture distance D for an offset (x, y, z), in single precision: the shape factor's cosine and
// sine are ratios of the offsets; within 1e-5 of the exact one.
__device__ static inline float distance_f32(float x, float y, float z, const float* R) {
  const float rho = sqrtf(x * x + y * y), rr = sqrtf(rho * rho + z * z);
  const float cs = rho > 0.0f ? fmaxf(fabsf(x), fabsf(y)) / rho : 1.0f;
  const float sn = rr > 0.0f ? fmaxf(rho, fabsf(z)) / rr : 1.0f;
  return sqrtf(cs * sn) * (fabsf(R[0] * x + R[3] * y + R[6] * z) + fabsf(R[1] * x + R[4] * y + R[7] * z) +
                           fabsf(R[2] * x + R[5] * y + R[8] * z));
}
// Lower bound, in single precision, on the time to grow by `lead` at velocity V (-inf: none).
__device__ static inline float time_bound(double lead, double V) {
  if (!(lead > 0.0) || !(V >= 0.0)) return -__builtin_inff();
  const double x = lead / V * (1.0 - 1e-6);  // (+inf for V = 0: it never captures)
  const float f = (float)x;
  return (double)f > x ? nextafterf(f, 0.0f) : f;
}
// Lower bound on the time that takes a half-diagonal E back to zero at velocity V (-inf: none).
__device__ static inline float back_bound(double E, double V) {
  if (!(E >= 0.0) || !(V >= 0.0)) return -__builtin_inff();
  return V > 0.0 ? (float)(E / V * (1.0 - 1e-6)) : __builtin_inff();
}
// Lower bound on the time from the capture of active cell t (voxel v; new centroid c, rotation R,
// half-diagonal E0) to the first capture by the cell it becomes, over the neighbours that are
// liquid before the loop, and (*back) on the step back that takes E0 to zero.  -inf: no useful
// bound; +inf: the cell does not grow.
__device__ static inline float first_capture_after(const Inst& d, int t, int v, const double* c, double E0,
                                                   const float* Rf, float* back) {
  *back = __builtin_inff();
  if (!d.aRow[t].cold) return __builtin_inff();
  const amcd_params& p = d.p;
  const double T = d.aRow[t].T;
  const double V = T == p.tS ? p.vhat_tS : (T == p.T0 ? p.vhat_T0 : p.Avel * pow(p.tL - T, p.nvel) * (1 + 1e-9));
  *back = back_bound(E0, V);
  if (!(V > 0.0) || !(E0 == E0)) return -__builtin_inff();
  int i, j, k;
  decode(d, v, i, j, k);
  float Dm = __builtin_inff();
  bool bad = false;
  for (int dz = -1; dz <= 1; ++dz) {
    const int z = k + dz;
    if (z < 0 || z >= p.nz) continue;
    for (int dy = -1; dy <= 1; ++dy) {
      const int y = j + dy;
      if (y < 0 || y >= p.ny) continue;
      const uint8_t* row = d.vs + (size_t)z * d.nxy + (size_t)y * p.nx;
      const float fy = (float)(((double)y + .5) * p.dy - c[1]), fz = (float)(((double)z + .5) * p.dz - c[2]);
#pragma unroll
      for (int dx = -1; dx <= 1; ++dx) {
        const int x = i + dx;
        if (x < 0 || x >= p.nx || (dx == 0 && dy == 0 && dz == 0)) continue;
        if ((row[x] & 3) != 1) continue;
        const float D = distance_f32((float)(((double)x + .5) * p.dx - c[0]), fy, fz, Rf);
        bad |= !(D == D);
        Dm = fminf(Dm, D);
      }
    }
  }
  return bad ? -__builtin_inff() : time_bound((double)Dm * (1.0 - 1e-5) - E0, V);
}

__device__ static inline void grow_list(const Inst& d, int slot, int lane) {
  const amcd_params& p = d.p;
  const SlotRec sr = d.slots[slot];
  if (sr.n < 0) return;
  const int a = sr.act;
  const int t = lane < AMCD_NB ? d.aRow[a].nbr[lane] : -1;
  const bool liq = t >= 0 && d.aVS[t] == 1;
  double D = __builtin_inf(), f = 0.0, r = __builtin_inf();
  int tv = -1, cold = 0;
  float tnew = __builtin_inff();
  double4 rc = make_double4(0.0, 0.0, 0.0, 0.0);
  double V = 0.0, R[9];
  float Rf[9];
  for (int q = 0; q < 9; ++q) {
    R[q] = d.rot[9 * (size_t)(sr.G - 1) + q];
    Rf[q] = (float)R[q];
  }
  if (liq) {
    const double c[3] = {sr.c[0], sr.c[1], sr.c[2]};
    tv = d.aRow[t].vox;
    cold = d.aRow[t].cold;
    const double T = d.aRow[t].T;
    V = !(T < p.tL) ? 0.0 : T == p.tS ? p.vhat_tS : T == p.T0 ? p.vhat_T0 : growth_velocity(p, T);
    candidate(d, c, R, tv, &D, &f);
    r = .5 * (d.ruq[a] + d.ruq[t]);
    double nc[3], ne;
    recentre(d, sr.vox, tv, c, R, f, nc, &ne);
    rc = make_double4(nc[0], nc[1], nc[2], ne);
  }
  const unsigned long long bal = __ballot(liq);
  const int n = (int)__popcll(bal);
  const size_t cb = d.precap + (size_t)slot * AMCD_NB;
  const int rank = list_rank(D, r, liq, -1);
  int pre = -1;
  // the lists ahead, for the entries whose target would grow
  const int half = lane >> 5, q = lane & 31;
  const int qq = q < 13 ? q : q + 1, ddx = qq % 3 - 1, ddy = (qq / 3) % 3 - 1, ddz = qq / 9 - 1;
  // and whose capture the step has time for (a step's last event may come later: its list is made then)
  const bool recs = slot < d.capslots;  // the entries have a CapRec
  const bool soon = recs && !(D > d.gExt[slot] + d.gVhat[slot] * p.DelT * (1 + 1e-6));
  for (unsigned todo = (unsigned)__ballot(liq && cold && soon); todo != 0;) {
    const int j0 = __builtin_ctz(todo);
    todo &= todo - 1;
    const bool two = todo != 0;
    const int j1 = two ? __builtin_ctz(todo) : j0;
    todo &= todo - 1;
    const int tj = half ? __builtin_amdgcn_readlane(t, j1) : __builtin_amdgcn_readlane(t, j0);
    const int vj = half ? __builtin_amdgcn_readlane(tv, j1) : __builtin_amdgcn_readlane(tv, j0);
    double c[3], E0;
    c[0] = half ? lane_f64(rc.x, j1) : lane_f64(rc.x, j0);
    c[1] = half ? lane_f64(rc.y, j1) : lane_f64(rc.y, j0);
    c[2] = half ? lane_f64(rc.z, j1) : lane_f64(rc.z, j0);
    E0 = half ? lane_f64(rc.w, j1) : lane_f64(rc.w, j0);
    const double Vj = half ? lane_f64(V, j1) : lane_f64(V, j0);
    const int t2 = q < AMCD_NB && (two || !half) ? d.aRow[tj].nbr[q] : -1;
    const bool on = t2 >= 0 && d.aVS[t2] == 1;
    double D2 = __builtin_inf(), f2 = 0.0, r2 = __builtin_inf();
    float tn2 = -__builtin_inff(), back2 = -__builtin_inff();
    CapRec cr = {0.0, 0.0, 0.0, 0.0, -1, sr.G, 0.0};
    if (on) {
      r2 = .5 * (d.ruq[tj] + d.ruq[t2]);
      int vi, vy, vk;
      decode(d, vj, vi, vy, vk);
      const double ct[3] = {((double)(vi + ddx) + .5) * p.dx, ((double)(vy + ddy) + .5) * p.dy,
                            ((double)(vk + ddz) + .5) * p.dz};
      candidate_at(ct, c, R, &D2, &f2);
      // and the bound for the cell that a capture through this entry would create
      const int v2 = vj + ddz * d.nxy + ddy * p.nx + ddx;
      double nc[3], ne;
      recentre(d, vj, v2, c, R, f2, nc, &ne);
      tn2 = first_capture_after(d, t2, v2, nc, ne, Rf, &back2);
      cr.x = nc[0];
      cr.y = nc[1];
      cr.z = nc[2];
      cr.E = ne;
    }
    const unsigned long long b2 = __ballot(on);
    const int na = __popc((unsigned)b2), nb = __popc((unsigned)(b2 >> 32));
    const int rank2 = list_rank(D2, r2, on, half);
    int base = 0;
    if (lane == 0) base = atomicAdd(&d.ls->npre, na + nb);
    base = __builtin_amdgcn_readfirstlane(base);
    const bool fits = base >= 0 && base <= d.precap - na - nb;
    const int at = half ? base + na : base;
    if (on && fits) {
      d.cand[at + rank2] = {D2, r2, t2, tn2, back2, (short)q, (short)((half ? nb : na) - rank2)};
      d.cap[at + rank2] = cr;
    }
    // the time to the new cell's first capture
    const float tn = time_bound(D2 - E0, Vj);
    const unsigned long long first = __ballot(on && rank2 == 0);
    const unsigned fa = (unsigned)first, fb = (unsigned)(first >> 32);
    if (fa != 0) {
      const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tn), __builtin_ctz(fa)));
      tnew = lane == j0 ? x : tnew;
      pre = lane == j0 && fits ? base : pre;
    }
    if (fb != 0) {
      const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tn), 32 + __builtin_ctz(fb)));
      tnew = lane == j1 ? x : tnew;
      pre = lane == j1 && fits ? base + na : pre;
    }
  }
  if (liq) {
    if (cold && !soon) tnew = -__builtin_inff();
    d.cand[cb + rank] = {D, r, t, tnew, cold ? back_bound(rc.w, V) : __builtin_inff(), (short)lane, (short)(n - rank)};
    if (!recs) d.cF[(size_t)slot * AMCD_NB + rank] = f;
    else d.cap[cb + rank] = {rc.x, rc.y, rc.z, rc.w, pre, sr.G, V};
  }
  if (lane == 0) d.slots[slot].n = n;
}
// every wave of an instance's blocks takes slots wave, wave + (its waves), ...
__global__ __launch_bounds__(GB) void k_grow_lists(Inst* I, const int* bstart, int ninst) {
  int ii = find_inst(bstart, ninst, blockIdx.x);
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  if (d.ls->done) return;
  const int lane = threadIdx.x & 63;
  const int nw = (bstart[ii + 1] - bstart[ii]) * (GB / 64);
  const int ns = d.ls->nslots;
  for (int slot = ((blockIdx.x - bstart[ii]) * GB + (int)threadIdx.x) >> 6; slot < ns; slot += nw)
    grow_list(d, slot, lane);
}

// (before the pass is run again in one step: the lists built ahead are allocated anew)
__global__ void k_clear_npre(Inst* I) {
  if (threadIdx.x == 0) I[blockIdx.x].ls->npre = 0;
}

// The capture / nucleation loop of one instance (S/VoxelsCA.C:381-610): one workgroup of NT
// threads per instance.  The reference looks at every growing cell for every event; here an
// event's only serial work is one wave's, and everything else happens once per window of
// events.
//
// A candidate is a pair (growing cell, liquid neighbour) with the capture time
// t = (D - E)/V of the cell's present half-diagonal E.  Between events E grows by V*Dt as the
// clock T grows by Dt, so tau = T + t stays fixed up to rounding: float bounds [lo, hi] are kept
// on the tau of each cell's first live candidate, and a thread holds E and V of its cells, j,
// j + NT, ... in registers.  A window is a clock value W and every candidate with lo <= W (its
// entries, at most 64):
//   SELECT   a histogram of the lower bounds gives the W that takes about `want` heads (at least
//            the smallest upper bound); the threads write the entries of their cells to LDS, and,
//            where a cell that a capture creates may itself capture before W, the entries of the
//            list built ahead for it, relative to the capture's own bounds;
//   ENGINE   wave 0, one entry per lane, performs events while the smallest upper bound of its
//            live entries stays below W: exact times (S/VoxelsCA.C:420-440), the first by (t, ruqs,
//            scan order), the event's uniform draw, T += Dt, E += V*Dt of its lanes, and the
//            captured voxel's entries drop out.  No candidate outside the window can come first:
//            their lower bounds exceed W, and the earliest capture by a cell that an event creates
//            is bounded from below by the set-up (CandRec::tn) or, for a list made in the loop, by
//            BUILD, which the engine waits for then; the window ends where the bound falls below W
//            and the cell's candidates are not entries themselves.  A step back of the clock goes
//            on like any other unless it could take some half-diagonal below zero (CandRec::back);
//   BUILD    meanwhile the other waves create the cells of the events as they are published:
//            grain, centre, half-diagonal, list (S/VoxelsCA.C:396-440, 486-506, 528-605);
//   APPLY    heads that died move to the next live candidate (the cells are listed in LDS first, so
//            that their list reads run side by side), new cells are taken over, and the window's
//            growth E += V*Dt is replayed event by event, in the reference's order of additions,
//            so every half-diagonal has the reference's bits.
// A window that does not fit takes less of the clock; one too full even at W = the smallest upper
// bound (many candidates within rounding of each other) takes the exact best of every wave as its
// entries and performs one event.
//
// What bounds it: a chain of dependent instructions.  An event is about 100 instructions of one
// wave (11 to 13 cycles each), and every window pays five barriers and two rounds of list reads;
// hence as many events per window as its 64 entries give (31 where the interface is wide, 18 in the
// memory tier, 8 where there are few cells), records that are one cache line, and lists and capture constants made by the
// set-up's parallel pass.  One decision per barrier with the lists built around each event took
// 6.9K cycles an event in these decks and 13.7K with the state in memory; now (cycles per event, 2.4
// GHz): 5.3K with few growing cells (at most 300), 2.7K with 3 thousand of a single track or of a
// raster over a wide plate, 6.0K with 15 thousand (state in memory; 10.1K while a cell without a
// bound from the set-up, or any step back, ended the window, 6.5K while ties shrank the span).
typedef const __attribute__((address_space(4))) Inst CInst;
struct Best {
  double t, r;
  int key;   // scan position * 32 + neighbour rank: the reference's scan order
  int cand;  // candidate entry, or the lane that holds it
  int tgt;   // active index of the captured voxel
};
__device__ static inline Best best_none() {
  Best b;
  b.t = __builtin_inf();
  b.r = __builtin_inf();
  b.key = 0x7fffffff;
  b.cand = -1;
  b.tgt = -1;
  return b;
}
// a strictly before b in (t, ruqs, scan order).  The ordering predicates are written
// without short-circuit branches, and a winner is taken field by field with selects on one
// predicate value, so that every field of the result comes from the same operand whatever
// the compiler does with the comparison chain.
__device__ static inline bool better(const Best& a, const Best& b) {
  const bool tl = a.t < b.t, tg = a.t > b.t, rl = a.r < b.r, rg = a.r > b.r;
  return tl | (!tg & (rl | (!rg & (a.key < b.key))));
}
// Wave-wide reductions by DPP row operations: two quad permutes, the half-row and row
// mirrors leave a row's result in all 16 of its lanes, row_bcast:15 and row_bcast:31
// carry rows 0 and 2 into rows 1 and 3 and then row 1 into rows 2 and 3, so that lane
// 63 ends with the result for the whole wave.  Every lane must be active.
constexpr int kQuadX1 = 0xb1, kQuadX2 = 0x4e, kHalfMirror = 0x141, kMirror = 0x140, kBcast15 = 0x142,
              kBcast31 = 0x143;
__device__ static inline float wave_min(float v) {
  v = fminf(v, dpp<kQuadX1>(v));
  v = fminf(v, dpp<kQuadX2>(v));
  v = fminf(v, dpp<kHalfMirror>(v));
  v = fminf(v, dpp<kMirror>(v));
  v = fminf(v, dpp<kBcast15, 0xa>(v));
  v = fminf(v, dpp<kBcast31, 0xc>(v));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ static inline double wave_min_f64(double v) {
  v = fmin(v, dpp<kQuadX1>(v));
  v = fmin(v, dpp<kQuadX2>(v));
  v = fmin(v, dpp<kHalfMirror>(v));
  v = fmin(v, dpp<kMirror>(v));
  v = fmin(v, dpp<kBcast15, 0xa>(v));
  v = fmin(v, dpp<kBcast31, 0xc>(v));
  return lane_f64(v, 63);
}
template <int CTRL, int ROWS = 0xf>
__device__ static inline void best_step(Best& b) {
  Best o;
  o.t = dpp<CTRL, ROWS>(b.t);
  o.r = dpp<CTRL, ROWS>(b.r);
  o.key = dpp<CTRL, ROWS>(b.key);
  o.cand = dpp<CTRL, ROWS>(b.cand);
  o.tgt = dpp<CTRL, ROWS>(b.tgt);
  const bool bt = better(o, b);
  b.t = bt ? o.t : b.t;
  b.r = bt ? o.r : b.r;
  b.key = bt ? o.key : b.key;
  b.cand = bt ? o.cand : b.cand;
  b.tgt = bt ? o.tgt : b.tgt;
}
__device__ static inline Best lane_best(const Best& b, int l) {
  Best o;
  o.t = lane_f64(b.t, l);
  o.r = lane_f64(b.r, l);
  o.key = __builtin_amdgcn_readlane(b.key, l);
  o.cand = __builtin_amdgcn_readlane(b.cand, l);
  o.tgt = __builtin_amdgcn_readlane(b.tgt, l);
  return o;
}
// best over a wave.  (t, ruqs, key) is a strict total order on candidates -- keys are
// unique -- so the order in which lanes are combined does not change the result.  A
// single candidate, or a single one at the smallest time, is the best without the full
// comparison.
__device__ static inline Best wave_best(Best b) {
  const unsigned long long m = __ballot(b.cand >= 0);
  if (m == 0) return best_none();
  if (__popcll(m) == 1) return lane_best(b, __builtin_ctzll(m));
  const double tmin = wave_min_f64(b.cand >= 0 ? b.t : __builtin_inf());
  const unsigned long long at = __ballot((b.cand >= 0) & (b.t == tmin));
  if (__popcll(at) == 1) return lane_best(b, __builtin_ctzll(at));
  best_step<kQuadX1>(b);
  best_step<kQuadX2>(b);
  best_step<kHalfMirror>(b);
  best_step<kMirror>(b);
  best_step<kBcast15, 0xa>(b);
  best_step<kBcast31, 0xc>(b);
  return lane_best(b, 63);
}
// candidate order inside a growing cell's list: (D, ruqs, key), NaN distances last
// (branch-free for the reason given at better())
__device__ static inline bool cand_less(double Da, double Ra, int ka, double Db, double Rb, int kb) {
  const bool na = Da != Da, nb = Db != Db;
  const bool c1 = na != nb;             // exactly one NaN: the other one is first
  const bool c2 = !na & !nb & (Da != Db);  // both numbers, different
  const bool rne = Ra != Rb;
  const bool tail = (rne & (Ra < Rb)) | (!rne & (ka < kb));
  return (c1 & nb) | (!c1 & c2 & (Da < Db)) | (!c1 & !c2 & tail);
}

// Liveness of candidate targets: an LDS bitmap over the active cells, bit set = "not liquid"
// (filled from the states at launch, set for every voxel captured or nucleated), or, for
// interfaces of more than AMCD_DEAD_BITS cells, the state bytes themselves.  Every list entry was
// liquid when its list was built, so "not dead" means live, and a dead entry stays dead.
#define AMCD_DEAD_BITS (1 << 19)
template <bool GD>
struct Liveness {
  unsigned* bits;
  uint8_t* vs;
  __device__ __forceinline__ bool dead(int t) const {
    if constexpr (GD)
      return gmem(vs)[t] != 1;
    else
      return (bits[t >> 5] >> (t & 31)) & 1u;
  }
  __device__ __forceinline__ void kill(int t) const {  // (lanes of one wave, each its own voxel)
    if constexpr (!GD) atomicOr(&bits[t >> 5], 1u << (t & 31));
  }
};

// A list record as two 16-byte loads.
__device__ static inline CandRec load_rec(const CandRec* p) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  const auto q = gmem((const v2d*)p);
  const v2d x = q[0], y = q[1];
  const unsigned long long a = (unsigned long long)__double_as_longlong(y.x);
  const unsigned long long b = (unsigned long long)__double_as_longlong(y.y);
  return {x.x, x.y, (int)a, __int_as_float((int)(a >> 32)), __int_as_float((int)b), (short)(b >> 32), (short)(b >> 48)};
}
// First live entry of a sorted list from entry `from` on, four records at a time with no branches
// between the loads.  Positions past the list's end read what follows it, at the array's end the
// 256 bytes every device array is allocated beyond its length; they are never used.
struct SlotHead {
  double D1;
  int c1, tgt1;  // head entry and its target (-1: no live entry)
};
template <bool GD>
__device__ static inline SlotHead slot_head(CInst& d, const Liveness<GD>& live, int from) {
  SlotHead h;
  h.tgt1 = -1;
  h.D1 = __builtin_inf();
  h.c1 = from;
  for (int p = from;; p += 4) {
    CandRec e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) e[q] = load_rec(d.cand + p + q);
    const int n = e[0].n;  // entries from position p on
    bool dd[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // (an entry past the list end asks about cell 0)
      const int t = q < n ? e[q].tgt : 0;
      dd[q] = live.dead(t) | (q >= n);
    }
    int hit = -1;
#pragma unroll
    for (int q = 3; q >= 0; --q) hit = dd[q] ? hit : q;
    if (hit < 0) {
      if (n <= 4) break;
      continue;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q == hit) {
        h.c1 = p + q;
        h.tgt1 = e[q].tgt;
        h.D1 = e[q].D;
      }
    break;
  }
  return h;
}

// Float bounds [lo, hi] on tau = T + t, the event clock at which the cell's head would
// be captured, t = (D1 - E)/V.  While the head does not change, every event adds Dt to
// T and V*Dt to E, so tau stays fixed up to rounding; the margin, 2^-26 of the
// magnitudes involved, exceeds that drift for more than 2^20 events (the loop
// re-evaluates every cell before that).  lo = hi = +inf: never a candidate (t NaN or
// +inf); lo = -inf, hi = +inf: evaluated at every event (V <= 0 or t = -inf).
__device__ static inline float f_down(double x) {
  float f = (float)x;
  return ((double)f > x) ? nextafterf(f, -__builtin_inff()) : f;
}
__device__ static inline float f_up(double x) {
  float f = (float)x;
  return ((double)f < x) ? nextafterf(f, __builtin_inff()) : f;
}
__device__ static inline void tau_bounds(double D1, double e, double v, double T, float& lo, float& hi) {
  const double t = (D1 - e) / v;
  if (t != t || t == __builtin_inf()) {
    lo = hi = __builtin_inff();
  } else if (!(v > 0.0) || t == -__builtin_inf()) {
    lo = -__builtin_inff();
    hi = __builtin_inff();
  } else {
    const double m = 0x1p-26 * (fabs(t) + fabs(T) + (fabs(D1) + fabs(e)) / v);
    const double tau = T + t;
    lo = f_down(tau - m);
    hi = f_up(tau + m);
  }
}

// Phase timers of the loop (shader-clock cycles of wave 0), compiled in only with
// -DAMCD_PHASE_PROFILE; read with amcd_phase_profile().
#ifdef AMCD_PHASE_PROFILE
__device__ unsigned long long g_phase[32];
#define PHASE_INIT(v) unsigned long long v = clock64()
#define PHASE(v, slot)                                        \
  do {                                                        \
    const unsigned long long t_ = clock64();                  \
    if (threadIdx.x == 0) atomicAdd(&g_phase[slot], t_ - v);  \
    v = t_;                                                   \
  } while (0)
#else
#define PHASE_INIT(v)
#define PHASE(v, slot)
#endif

// ---- windows
// Clock span of a window (the histogram's scale), adapted to the heads it gets: about half of the growing
// cells have a candidate within a step.  A window that had to fall back to its smallest clock value (mode
// 2 or more: a flat front's ties) says nothing of the span.  Bounded on both sides: hundreds of
// windows in a row that take a few heads, or too many, would bring it to infinity or zero, and every
// later window to one event.
__host__ __device__ static inline double first_span(double DelT, int cells) {
  return DelT * fmin(1.0, 80.0 / (double)(cells > 1 ? cells : 1));
}
__host__ __device__ static inline double next_span(double span, int bins, int mode, double DelT, int cells) {
  if (mode < 2) span *= bins >= 32 ? 1.6 : fmax(0.4, (bins + 8) / 26.0);
  return fmin(fmax(span, 0x1p-10 * first_span(DelT, cells)), 64 * DelT);
}
// How far the clock may step back before a half-diagonal e of velocity v is zero, in single precision (the
// loop takes 2^-16 off for the rounding): e/v; nothing for a velocity whose reciprocal would leave that
// range (0 times infinity, not a number, would be dropped from the minimum over the cells).
__host__ __device__ static inline float step_back(double e, double v) {
  const float f = (float)v;
#ifdef __HIP_DEVICE_COMPILE__
  const float y = __builtin_amdgcn_rcpf(f);
#else
  const float y = 1.0f / f;
#endif
  return f > 1e-30f ? fmaxf((float)e * y, 0.0f) : v > 0.0 ? 0.0f : __builtin_inff();
}
constexpr int WCAP = 64;   // entries of a window: one per lane of the engine wave
constexpr int TCAP = 256;  // touched cells (heads that died) listed per window
struct Window {
  // entries
  double D[WCAP], E[WCAP], V[WCAP], r[WCAP];
  int tgt[WCAP], key[WCAP], cand[WCAP], own[WCAP];  // own: the entry's cell (slot)
  int lo[WCAP], hi[WCAP];  // bounds, as order keys
  int lim[WCAP];  // after a capture through the entry: the largest bound that the new cell cannot precede
  double y[WCAP];   // reciprocal of V
  int parent[WCAP]; // the entry whose capture creates this one's cell (-1: the cell is there)
  int rank[WCAP];   // position by hi
  float back[WCAP]; // CandRec::back
  // events, in order: entry (-1: nucleation, -2: not performed yet) and voxel, published one by
  // one; growth time; the slot of the cell it created (-1: none)
  int2 ev[WCAP];
  double dt[WCAP];
  int slot[WCAP], base[WCAP];  // (base: its list's first entry)
  double E0[WCAP], V0[WCAP];
  int first[WCAP];  // after an event: CandRec::tn of the cell as BUILD has made it, as bits (kPending: not yet)
  int n;        // entries asked for (more than WCAP: the window is too full)
  int m;        // events
  int decided;  // events decided in this window (one more than m when the last waits for the pool)
  int scan0;    // scan position of the first event's voxel
  int G, pool;  // the nucleation's grain and pool entry (a window has at most one, its last event)
  int done;     // the engine has published its last event
  unsigned x2[WCAP];         // random engine states after the window's draws
  unsigned long long draws;  // bit m: event m nucleates
};
struct LoopShared {
  Window win;
  // cells whose head died in the window, with their half-diagonal before it (for a cell that ran
  // out of candidates: after it)
  double tE[TCAP], tV[TCAP];
  int tS[TCAP], tn;
  float red[16];
  int back;      // CandRec::back's minimum over the cells, as float bits (they order like the values)
  int hist[32];  // heads by lower bound, in thirty-seconds of twice the window's span
  int nslots;
  int fin;  // 1: goes on, 0: finished, -1: pool refill, -2: larger tier, -4: no progress
  double T;
  int go, r_i1, all, neg, nexec;
  int tied;  // cells whose head can be the first, where a window takes the exact best of every wave
  unsigned cur;  // random engine state
  unsigned long long units;
  unsigned seen[8], exact[8];  // per wave: cells that the windows looked at, and exact times of theirs
};

// The workgroup's exchange: the window, the liveness bitmap and, for the register tiers, every
// cell's bounds and list head (one workgroup runs on a CU at a time).  File scope, for the routine
// that is kept out of line.
constexpr int LDS_CELLS = 4096;
__shared__ LoopShared s_loop;
__shared__ unsigned s_dead_bits[AMCD_DEAD_BITS / 32];
__shared__ float2 s_lh[LDS_CELLS];
__shared__ int2 s_hd[LDS_CELLS];

// A cell's bounds and head: in LDS for the register tiers, else in memory.
template <bool MEM>
__device__ static inline float2 get_lh(CInst& d, int s) {
  if constexpr (MEM) return gload8(d.gLH + s);
  else return s_lh[s];
}
template <bool MEM>
__device__ static inline void set_lh(CInst& d, int s, float lo, float hi) {
  if constexpr (MEM) gstore8(d.gLH + s, make_float2(lo, hi));
  else s_lh[s] = make_float2(lo, hi);
}
template <bool MEM>
__device__ static inline int2 get_hd(CInst& d, int s) {
  if constexpr (MEM) return gload8(d.gHd + s);
  else return s_hd[s];
}
template <bool MEM>
__device__ static inline void set_hd(CInst& d, int s, int c1, int tgt) {
  if constexpr (MEM) gstore8(d.gHd + s, make_int2(c1, tgt));
  else s_hd[s] = make_int2(c1, tgt);
}

// A thread's half-diagonals and velocities: K cells in registers (or a batch of K streamed from
// memory).  A cell without candidates has velocity 0.
template <int K>
struct Cells {
  double E[K], V[K];
};

__device__ static inline double pack2(int lo, int hi) {
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
// Float bounds as integers in the same order (no NaN among them): minima and comparisons are
// then one instruction each, with the lane permutation as an operand modifier.
__device__ static inline int order_key(float f) {
  const int i = __float_as_int(f);
  return i ^ ((i >> 31) & 0x7fffffff);
}
// +inf; after every bound; as an entry's limit: BUILD is asked when it is captured
constexpr int kKeyInf = 0x7f800000, kKeyNone = 0x7fffffff, kKeyAsk = 0x7ffffffe;
__device__ static inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ static inline double uni(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)uni((int)b), hi = (unsigned)uni((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <int CTRL, int ROWS = 0xf>
__device__ static inline int dpp_min_shift(int v) {  // with the lane's lower neighbour by the row shift
  return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, ROWS, 0xf, false));
}

// An event for BUILD to start on: one 8-byte store (a wave's LDS stores are performed in order, so
// what was stored before it is there when it is seen).
__device__ static inline void publish(Window& win, int m, int ent, int i1) {
  lds_put(&win.ev[m], make_int2(ent, i1));
}

// ENGINE: the events of window `win`, by one wave.  The entries are sorted by their upper
// bounds once per window (the first to come in the highest lane), so an event takes the first
// live lane without a search; only where a later entry's lower bound reaches it (they are equal
// up to rounding) are the exact times compared.  Every value that steers the loop is made uniform
// on entry (scalar branches, no loads).  The time is the quotient (D - E)/V rounded to nearest,
// from V's reciprocal rounded to nearest and two residual corrections (Markstein's theorem: the
// first makes the quotient faithful, the second correctly rounded); where a residual could leave
// the normal range, by a division.
struct EngineState {
  double T;
  int vSind2, nGrain, pool_used, events, captures, nucs;
  int nd;  // draws consumed
  long long visits;  // candidates bounded as entries, and times compared
};
constexpr int kPending = 0x7fc00bad;  // (no float result has these bits)
struct EngineRun {
  double T, rdt;
  int m, used, visits, fin, ri1, rent;
  bool nuc;
};
// The body is straight: one branch leaves the loop, whatever the reason, and only near-ties, asking
// BUILD and steps back branch inside (a taken branch costs as much as three instructions).
template <bool PLAIN>
__device__ static inline void engine_run(EngineRun& o, Window& win, double D, double E, double V, double y, double r,
                                         int tgt, int key, int src, int parent, int lo, int hi, int lim_,
                                         unsigned long long live, unsigned long long close, unsigned long long draws, int W,
                                         double DelT, int scan0, float back) {
  const int lane = threadIdx.x & 63;
  double T = o.T, rdt = 0.0;
  const double T0 = T;
  int m = 0, ri1 = -1, rent = -2, visits = 0, lim = W, fin = 1, used = 0;
  bool nuc = false;
  bool ask = false;  // the last event's cell has no bound yet
  unsigned long long killed = 0;
  double Vg = parent < 0 ? V : 0.0;  // a cell grows from the event that creates it on
  while (live != 0) {
    int wl = 63 - __builtin_clzll(live);
    const int u = __builtin_amdgcn_readlane(hi, wl);
    if (__builtin_expect(ask, 0)) {  // BUILD's (it is at work on the event, whatever this wave does)
      int b;
      while ((b = uni(lds_get(&win.first[m - 1]))) == kPending) __builtin_amdgcn_s_sleep(1);
      const float f = __int_as_float(b), Tf = (float)T;
      const float x = Tf + f - 0x1p-20f * (fabsf(Tf) + fabsf(f));
      lim = min(lim, f == -__builtin_inff() ? (int)0x80000000 : f == __builtin_inff() ? kKeyNone : uni(order_key(x)) - 2);
      ask = false;
    }
    const bool late = u > lim;
    const double a = D - E;
    double t;
    if constexpr (PLAIN) {
      double q = a * y;
      q = fma(fma(-V, q, a), y, q);
      t = fma(fma(-V, q, a), y, q);
    } else {
      t = a / V;
    }
    int seen = 1;
    bool none = false;
    if ((close >> wl) & 1ull) {
      // several within rounding: the smallest time, then (ruqs, key) among the equal ones
      const unsigned long long c = __ballot(lo <= u) & live;
      seen = __popcll(c);
      const bool ok = ((c >> lane) & 1ull) && t <= 1e6;
      const double tmin = wave_min_f64(ok ? t : __builtin_inf());
      unsigned long long at = __ballot(ok && t == tmin);
      none = at == 0;
      if (!none) {
        wl = __builtin_ctzll(at);
        at &= at - 1;
        if (at != 0) {
          double rb = lane_f64(r, wl);
          int kb = __builtin_amdgcn_readlane(key, wl);
          for (; at != 0; at &= at - 1) {
            const int l = __builtin_ctzll(at);
            const double rl = lane_f64(r, l);
            const int kl = __builtin_amdgcn_readlane(key, l);
            const bool first = rl < rb || (!(rl > rb) && kl < kb);
            wl = first ? l : wl;
            rb = first ? rl : rb;
            kb = first ? kl : kb;
          }
        }
      }
    }
    const double tw = lane_f64(t, wl);
    const int th = (int)(__double_as_longlong(tw) >> 32);
    const int i1 = __builtin_amdgcn_readlane(tgt, wl), ent = __builtin_amdgcn_readlane(src, wl);
    const bool me = lane == m;
    const int over = __ballot(T < DelT) == 0;         // loop condition (S/VoxelsCA.C:381)
    const int far = th >= 0x412e8480;                 // 1e6 or more, or not a number (S/VoxelsCA.C:480)
    const int draw = (int)((draws >> m) & 1ull);      // nucleation (S/VoxelsCA.C:483)
    if ((int)late | over | (int)none | far | draw) {
      if (!late) {
        fin = over ? 0 : none ? (m == 0 ? 0 : 1) : far ? 0 : 1;
        visits += over ? 0 : seen;
        nuc = !over && !none && !far;
        if (nuc) {
          ri1 = me ? i1 : ri1;
          used = m + 1;
        }
      }
      break;
    }
    visits += seen;
    // capture: growth of every cell (S/VoxelsCA.C:511-516); the lanes' cells all have a live
    // candidate.  A step back in time (negative Dt) ends the window if it may clamp a
    // half-diagonal at zero and so move a capture time.
    bool clamp = false;
    if (__builtin_expect(th < 0, 0)) {
      double Tk = rdt;  // the clock after each event so far (to rounding, which `back` has room for)
      for (int s = 1; s < 64; s <<= 1) {
        const double p = __shfl_up(Tk, s);
        Tk += lane >= s ? p : 0.0;
      }
      Tk += T0 + 0x1p-40 * (fabs(T0) + fabs(Tk));
      const double f = lane < m ? Tk - (double)win.back[rent < 0 ? 0 : rent] : -__builtin_inf();
      clamp = !(T + tw > fmax(-wave_min_f64(-f), T0 + 0x1p-40 * fabs(T0) - (double)back));
    }
    ri1 = me ? i1 : ri1;
    rent = me ? ent : rent;
    lds_put(&win.ev[lane], make_int2(rent, ri1));
    T = T + tw;
    E = E + Vg * tw;
    rdt = me ? tw : rdt;
    killed |= __ballot(tgt == i1);
    const unsigned long long kids = __ballot(parent == ent);
    if (kids != 0) {  // candidates of the cell that this event creates
      live |= kids;
      const bool mine = parent == ent;
      Vg = mine ? V : Vg;
      key = mine ? (scan0 + m) * 32 + key : key;
    }
    live &= ~killed;
    const int bound = __builtin_amdgcn_readlane(lim_, wl);
    ask = bound == kKeyAsk;
    lim = min(lim, bound);
    lim = clamp ? (int)0x80000000 : lim;
    ++m;
  }
  o.T = T;
  o.rdt = rdt;
  o.m = m;
  o.used = nuc ? used : m;
  o.visits = visits;
  o.fin = fin;
  o.ri1 = ri1;
  o.rent = rent;
  o.nuc = nuc;
}
__device__ static inline void engine_window(CInst& d, LoopShared& sh, Window& win, EngineState& es, float W,
                                            double DelT_, int n_pool, LoopState* ls) {
  const int lane = threadIdx.x & 63;
  const int n = uni(win.n);
  // sorted by the upper bounds, the first to come in the highest lane
  const int src = __builtin_amdgcn_ds_permute((63 - (lane < n ? win.rank[lane] : lane)) << 2, lane);
  const bool in = lane >= 64 - n;
  const double D = in ? win.D[src] : 0.0, V = in ? win.V[src] : 1.0, r = in ? win.r[src] : 0.0;
  const double E = in ? win.E[src] : 0.0, y = in ? win.y[src] : 1.0;
  const int tgt = in ? win.tgt[src] : -1, key = in ? win.key[src] : 0;
  const int lo = in ? win.lo[src] : kKeyNone, hi = in ? win.hi[src] : kKeyNone, lim = in ? win.lim[src] : kKeyNone;
  const int parent = in ? win.parent[src] : -1;
  const bool plain = __all(!in || (V > 0x1p-300 && V < 0x1p300 && D > 0x1p-300 && D < 0x1p300 && fabs(E) < 0x1p300));
  // entries that a later one's lower bound reaches: the smallest lower bound over the lower lanes
  int sm = dpp_min_shift<0x111>(lo);  // row_shr:1, :2, :4, :8, then the rows below
  sm = dpp_min_shift<0x112>(sm);
  sm = dpp_min_shift<0x114>(sm);
  sm = dpp_min_shift<0x118>(sm);
  sm = dpp_min_shift<kBcast15, 0xa>(sm);
  sm = dpp_min_shift<kBcast31, 0xc>(sm);
  sm = __builtin_amdgcn_update_dpp(0x7fffffff, sm, 0x138, 0xf, 0xf, false);  // wave_shr:1
  const unsigned long long close = __ballot(sm <= hi), live = __ballot(in && parent < 0);
  const unsigned dlo = uni((int)win.draws), dhi = uni((int)(win.draws >> 32));
  const unsigned long long draws = ((unsigned long long)dhi << 32) | dlo;
  const double DelT = uni(DelT_);
  EngineRun o;
  o.T = uni(es.T);
  const int Wk = uni(order_key(W));
  const float back = __int_as_float(uni(sh.back));
  if (plain)
    engine_run<true>(o, win, D, E, V, y, r, tgt, key, src, parent, lo, hi, lim, live, close, draws, Wk, DelT,
                      uni(es.vSind2), back);
  else
    engine_run<false>(o, win, D, E, V, y, r, tgt, key, src, parent, lo, hi, lim, live, close, draws, Wk, DelT,
                      uni(es.vSind2), back);
  int fin = n == 0 ? 0 : o.fin, m = o.m;  // n == 0: no candidate left
  es.captures += m;
  if (fin == 1 && o.nuc) {  // S/VoxelsCA.C:483-506
    const int i1 = __builtin_amdgcn_readlane(o.ri1, m);
    if (es.pool_used >= n_pool || es.pool_used >= d.poolcap || es.nGrain >= d.gcap) {
      if (lane == 0) {
        *gmem(&ls->pending) = 1;  // the host refills the pool and resumes
        *gmem(&ls->pend_tgt) = i1;
      }
      fin = -1;
    } else {
      // (the nucleus's first capture is not bounded: the window ends)
      es.nGrain++;
      if (lane == 0) {
        win.G = es.nGrain;
        win.pool = es.pool_used;
        publish(win, m, -1, i1);
      }
      es.pool_used++;
      es.nucs++;
      ++m;
    }
  }
  if (lane == 0) lds_put(&win.done, 1);
  if (lane < m) {
    win.dt[lane] = o.rdt;
    gmem(d.aScan)[o.ri1] = es.vSind2 + lane;
  }
  es.events += o.used;
  es.nd += o.used;
  es.visits += o.visits;
  es.T = o.T;
  if (lane == 0) {
    if (o.used > 0) sh.cur = win.x2[o.used - 1];
    win.m = m;
    win.decided = o.used;
    sh.T = o.T;
    sh.fin = fin;
  }
  es.vSind2 += m;
}

// The rare parts of BUILD out of line, so that their registers do not add to the cells' own: the
// re-centring of a capture by a cell made in this launch, a velocity that is not tabulated (EASM
// temperatures).
struct Octahedron {
  double x, y, z, E;
};
__device__ __attribute__((noinline)) static Octahedron recentre_out(const Inst* I, int sw, int cand, int v1) {
  CInst& d = *(CInst*)I;
  const auto q = gmem(d.slots) + sw;
  const double c[3] = {q->c[0], q->c[1], q->c[2]};
  const int G = q->G;
  double R[9], o[3], e;
#pragma unroll
  for (int q = 0; q < 9; ++q) R[q] = gmem(d.rot)[9 * (size_t)(G - 1) + q];
  recentre(d, q->vox, v1, c, R, gmem(d.cF)[cand - d.precap], o, &e);
  return {o[0], o[1], o[2], e};
}
__device__ __attribute__((noinline)) static double velocity_out(const Inst* I, double T) {
  CInst& d = *(CInst*)I;
  return growth_velocity(d.p, T);
}

// The sorted list of a cell that no set-up list was built ahead for (a nucleus, or a capture by a
// cell of this launch), out of line as the other rare parts.
__device__ __attribute__((noinline)) static void list_out(const Inst* I, int cb, int i1, int G, int v1, int tn, int liq,
                                                          double c0, double c1, double c2, double E0, double V0, int k) {
  CInst& d = *(CInst*)I;
  auto& p = d.p;
  const int lane = threadIdx.x & 63;
  double R[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) R[q] = gmem(d.rot)[9 * (size_t)(G - 1) + q];
  double D = __builtin_inf(), f = 0, r = __builtin_inf();
  // neighbour `lane` of v1, in the order of the active-neighbour table
  int vi, vj, vk;
  decode(d, v1, vi, vj, vk);
  const int qq = lane < 13 ? lane : lane + 1;
  const int ddx = qq % 3 - 1, ddy = (qq / 3) % 3 - 1, ddz = qq / 9 - 1;
  if (liq) {
    const double cen[3] = {c0, c1, c2};
    const double ct[3] = {((double)(vi + ddx) + .5) * p.dx, ((double)(vj + ddy) + .5) * p.dy,
                          ((double)(vk + ddz) + .5) * p.dz};
    candidate_at(ct, cen, R, &D, &f);
    r = .5 * (gmem(d.ruq)[i1] + gmem(d.ruq)[tn]);
  }
  const bool bad = __any(liq && !(D == D));
  const double Dm = wave_min_f64(liq ? D : __builtin_inf());
  // (first of all: the engine may wait for it)
  if (lane == 0) lds_put(&s_loop.win.first[k], __float_as_int(bad ? -__builtin_inff() : time_bound(Dm - E0, V0)));
  const int rank = list_rank(D, r, liq != 0, -1), n = (int)__popcll(__ballot(liq != 0));
  if (liq) {
    typedef double v2d __attribute__((ext_vector_type(2)));
    const auto q = gmem((v2d*)(d.cand + cb + rank));
    q[0] = v2d{D, r};
    const int none = __float_as_int(-__builtin_inff());
    q[1] = v2d{pack2(tn, none), pack2(none, lane | (n - rank) << 16)};
    gmem(d.cF)[cb - d.precap + rank] = f;
  }
}

// BUILD: the cell that event k of the window creates (one wave, while the engine goes on).  The
// liveness is that of the window's start; the voxels of the events up to k are known.  One round
// of loads: the captured cell's row by lanes 0..31, the entry's capture by lanes 32..43.
template <bool GD>
__device__ static inline void build_cell(CInst& d, const Inst* I, LoopShared& sh, Window& win, const Liveness<GD>& live,
                                         int ent, int k, int nrec, int nm0) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  const int lane = threadIdx.x & 63;
  auto& p = d.p;
  const int evi = lane <= k ? lds_get(&win.ev[lane]).y : -1;  // lane j: voxel of event j
  const int i1 = __builtin_amdgcn_readlane(evi, k), scan = uni(win.scan0) + k;
  const int cand = ent >= 0 ? uni(win.cand[ent]) : -1, sw = ent >= 0 ? uni(win.own[ent]) : -1;
  const bool first = cand >= 0 && cand < nrec;  // it has a CapRec
  const int* at = (const int*)(d.aRow + i1) + (lane & 31);
  if (lane >= 32) at = first ? (const int*)(d.cap + cand) + min(lane - 32, 11) : at;
  const int x = gmem(at)[0];
  const int tn = lane < AMCD_NB ? x : -1;
  bool liq = tn >= 0 && !live.dead(tn >= 0 ? tn : 0);
  for (int j = 0; j < k; ++j) liq &= tn != __builtin_amdgcn_readlane(evi, j);
  const unsigned long long bal = __ballot(liq);  // liquid just after the event
  const int v1 = __builtin_amdgcn_readlane(x, 26), cold = __builtin_amdgcn_readlane(x, 27);
  auto word2 = [&](int l) {
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane(x, l + 1) << 32) |
                                            (unsigned)__builtin_amdgcn_readlane(x, l)));
  };
  const double T1 = word2(28);
  double cen[3], E0;
  int G, pre = -1;
  if (first) {            // capture (S/VoxelsCA.C:507-605)
    cen[0] = word2(32);
    cen[1] = word2(34);
    cen[2] = word2(36);
    E0 = word2(38);
    pre = __builtin_amdgcn_readlane(x, 40);
    G = __builtin_amdgcn_readlane(x, 41);
  } else if (ent >= 0) {  // by a cell made in this launch, or beyond the slots with a CapRec
    G = uni(gmem(d.slots)[sw].G);
    const Octahedron o = recentre_out(I, sw, cand, v1);
    cen[0] = uni(o.x);
    cen[1] = uni(o.y);
    cen[2] = uni(o.z);
    E0 = uni(o.E);
  } else {                // nucleation (S/VoxelsCA.C:486-506)
    G = uni(win.G);
    centre(d, v1, cen);
    E0 = 0.0;
    if (lane < 9) gmem(d.rot)[9 * (size_t)(G - 1) + lane] = gmem(d.pool)[9 * (size_t)uni(win.pool) + lane];
  }
  int slot = -1, cb = 0;
  const bool grows = cold && bal;
  if (grows) {
    if (lane == 0) slot = atomicAdd(&sh.nslots, 1);
    slot = uni(slot);
    cb = pre >= 0 ? pre : d.precap + slot * AMCD_NB;
    const double V0 = (T1 == p.tS) & (T1 < p.tL) ? p.vhat_tS : velocity_out(I, T1);
    if (lane == 0 && ent >= 0 && win.lim[ent] == kKeyAsk) win.back[ent] = back_bound(E0, V0);
    if (pre < 0) {
      if (ent < 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the nucleus's rotation, read back
      list_out(I, cb, i1, G, v1, tn, liq, cen[0], cen[1], cen[2], E0, V0, k);
    }
    if (lane == 0) {
      win.base[k] = cb;
      win.E0[k] = E0;
      win.V0[k] = V0;
    }
  }
  if (lane == 0) {
    win.slot[k] = slot;
    if (!grows && ent >= 0 && win.lim[ent] == kKeyAsk) win.back[ent] = __builtin_inff();
    // (the set-up's list for the cell gave the engine no bound)
    if (!grows || pre >= 0) lds_put(&win.first[k], __float_as_int(grows ? -__builtin_inff() : __builtin_inff()));
  }
  // the slot's record by lanes 0..2 and the event's by lanes 3..5, 16 bytes each
  const int q = lane < 3 ? lane : lane - 3;
  const double c02 = q == 0 ? cen[0] : cen[2];
  const double a = lane < 3 ? (q == 2 ? pack2(i1, scan) : c02) : (q == 0 ? pack2(i1, G) : q == 1 ? cen[0] : cen[2]);
  const double b = lane < 3 ? (q == 0 ? cen[1] : q == 1 ? pack2(v1, G) : pack2(cb, 1))
                            : (q == 0 ? E0 : q == 1 ? cen[1] : 0.0);
  if (lane < 6 && (lane >= 3 || grows)) {
    v2d* to = lane < 3 ? (v2d*)(d.slots + slot) + q : (v2d*)(d.events + (scan - nm0)) + q;
    gmem(to)[0] = v2d{a, b};
  }
}
// BUILD for a wave's share of a window's events, as the engine publishes them (or all of them,
// when it is done); out of line: its registers do not add to those that hold the cells.  The
// engine ends after at most WCAP events whatever these waves do, so the wait ends.
template <bool GD>
__device__ __attribute__((noinline)) static void build_cells(const Inst* I, int first, int step, int nrec, int nm0) {
  CInst& d = *(CInst*)I;
  Window& win = s_loop.win;
  const Liveness<GD> live = {s_dead_bits, d.aVS};
  for (int k = first; k < WCAP; k += step) {
    int ent;
    for (;;) {
      const int done = uni(lds_get(&win.done));
      ent = uni(lds_get(&win.ev[k]).x);  // (read after `done`: a set flag means all is published)
      if (ent != -2 || done) break;
      __builtin_amdgcn_s_sleep(1);
    }
    if (ent == -2) break;
    build_cell<GD>(d, I, s_loop, win, live, ent, k, nrec, nm0);
  }
}

// A cell whose last candidate died in this window grows through the event that took it: the
// largest event of its targets from the former head on (those before it died in earlier windows).
__device__ static inline int last_event(CInst& d, int from, int scan0) {
  int mx = -1;
  for (int p = from;; p += 4) {
    CandRec e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) e[q] = load_rec(d.cand + p + q);
    const int n = e[0].n;
    int sc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sc[q] = gmem(d.aScan)[q < n ? e[q].tgt : e[0].tgt] - scan0;
#pragma unroll
    for (int q = 0; q < 4; ++q) mx = max(mx, sc[q]);
    if (n <= 4) break;
  }
  return mx;
}

// One cell after a window: its head moves from entry c0 to the next live candidate; bounds for it.  e is the
// half-diagonal before the window's growth (of a cell that event k0 created: after that event);
// `grown` returns it with the window's growth, through the event that took the last candidate
// when there is none left.  dtl: lane j holds the growth time of event j (whole waves call this).
struct Refreshed {
  double grown;
  float lo, hi;
  int c1, tgt;
};
template <bool GD>
__device__ static inline Refreshed refresh_cell(CInst& d, const Liveness<GD>& live, bool on, int c0, double e, double v,
                                                int k0, int m, int scan0, double dtl, double T0, double T) {
  Refreshed o;
  o.lo = o.hi = __builtin_inff();
  o.c1 = 0;
  o.tgt = -1;
  o.grown = e;
  double D1 = 0.0;
  int last = -1;
  if (on) {
    const SlotHead h = slot_head<GD>(d, live, c0);
    o.c1 = h.c1;
    o.tgt = h.tgt1;
    D1 = h.D1;
    last = h.tgt1 >= 0 ? m - 1 : last_event(d, c0, scan0);
  }
  if (__any(on && (k0 >= 0 || o.tgt < 0))) {
    for (int j = 0; j < m; ++j) {
      const double g = o.grown + v * lane_f64(dtl, j);
      o.grown = (j > k0) & (j <= last) ? g : o.grown;
    }
    if (o.grown < 0.0) o.grown = 0.0;  // (only a window's last event can take it below zero)
  }
  // tau is the same before and after the growth; a new cell's is taken after it
  if (o.tgt >= 0) tau_bounds(D1, k0 >= 0 ? o.grown : e, v, k0 >= 0 ? T : T0, o.lo, o.hi);
  return o;
}

// A cell's entries up to clock W into the window: its head, and the live candidates after it
// while their bounds reach W (two list positions per round of loads; the one past the list's end
// is masked).
__device__ static inline int put_entry(Window& win, const CandRec& e, double E, double V, int key, int cand, int own,
                                       int parent, int lo, int hi) {
  const int i = atomicAdd(&win.n, 1);
  if (i >= WCAP) return -1;
  win.D[i] = e.D;
  win.E[i] = E;
  win.V[i] = V;
  win.r[i] = e.r;
  win.tgt[i] = e.tgt;
  win.key[i] = key;
  win.cand[i] = cand;
  win.own[i] = own;
  win.parent[i] = parent;
  win.lo[i] = lo;
  win.hi[i] = hi;
  win.back[i] = e.back;
  return i;
}
template <bool GD>
__device__ static inline void push_cell(CInst& d, const Liveness<GD>& live, Window& win, int s, double E, double V,
                                        int c1, float lo, float hi, double T, float W, int nrec) {
  const int scan = gmem(d.slots)[s].scan;
  bool first = true;
  for (int p = c1;; p += 2) {
    CandRec e[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) e[q] = load_rec(d.cand + p + q);
    const int n = e[0].n;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (q >= n) return;
      if (!first) {
        tau_bounds(e[q].D, E, V, T, lo, hi);
        if (!(lo <= W) || lo == __builtin_inff()) return;  // and so are all later ones
        if (live.dead(e[q].tgt)) continue;
      }
      first = false;
      const int i = put_entry(win, e[q], E, V, scan * 32 + e[q].nb, p + q, s, -1, order_key(lo), order_key(hi));
      if (i < 0) return;
      // the clock after the capture is at least lo: when the new cell may capture within the
      // window, its candidates join it
      const float tn = e[q].tn;
      const float x = lo + tn - 0x1p-20f * (fabsf(lo) + fabsf(tn));
      int lim = tn == -__builtin_inff() ? kKeyAsk : tn == __builtin_inff() ? kKeyNone : order_key(x) - 2;
      if ((lim < order_key(W) || lim == kKeyAsk) && p + q >= d.precap && p + q < nrec) {
        const CapRec cr = d.cap[p + q];
        if (cr.pre >= 0) {
          lim = kKeyNone;
          for (int pc = cr.pre;; ++pc) {
            const CandRec ec = load_rec(d.cand + pc);
            float l, h;
            tau_bounds(ec.D, cr.E, cr.V, 0.0, l, h);
                const int lk = order_key(lo + l) - 1, hk = order_key(hi + h) + 1;
            if (l == __builtin_inff() || lk > order_key(W)) break;
            if (l == -__builtin_inff()) {  // (no bound)
              lim = kKeyAsk;
              break;
            }
            if (!live.dead(ec.tgt)) {
              const int ic = put_entry(win, ec, cr.E, cr.V, ec.nb, pc, -1, i, lk, hk);
              if (ic < 0) return;
              const float xc = lo + l + ec.tn - 0x1p-20f * (fabsf(lo) + fabsf(l) + fabsf(ec.tn));
              win.lim[ic] = ec.tn == -__builtin_inff() ? kKeyAsk : ec.tn == __builtin_inff() ? kKeyNone : order_key(xc) - 2;
            }
            if (ec.n <= 1) break;
          }
        }
      }
      win.lim[i] = lim;
    }
    if (n <= 2) return;
  }
}

// The exact best candidate of one cell (its head and the entries tied with it in time) against
// b (S/VoxelsCA.C:420-440).  Returns the times evaluated.
template <bool GD>
__device__ static inline int exact_cell(CInst& d, const Liveness<GD>& live, int s, double E, double V, int c1, Best& b,
                                         int& bs, double& be, double& bv) {
  const int scan = gmem(d.slots)[s].scan;
  double t1 = 0.0;
  int evals = 0;
  for (int p = c1;; ++p) {
    const CandRec e = load_rec(d.cand + p);
    const double t = (e.D - E) / V;
    ++evals;
    if (p == c1) {
      t1 = t;
      if (!(t1 <= 1e6)) break;
    }
    if (!(t == t1)) break;
    Best z;
    z.t = t;
    z.r = e.r;
    z.key = scan * 32 + e.nb;
    z.cand = p;
    z.tgt = e.tgt;
    if (!live.dead(e.tgt) && better(z, b)) {
      b = z;
      bs = s;
      be = E;
      bv = V;
    }
    if (e.n <= 1) break;
  }
  return evals;
}

// GD: an interface of more than AMCD_DEAD_BITS cells, whose liveness is read from the states
// (instantiated with the memory-resident tier only).  K = 0: every cell's state in memory
// (gExt, gVhat, gHd, gLH), streamed MB cells per thread at a time, for growing lists larger
// than the register tiers hold.
template <int NT, int K, bool GD = false>
__global__ __launch_bounds__(NT) void k_event_loop(Inst* I, const amcd_step* S, amcd_out* O) {
  constexpr int NW = NT / 64;
  constexpr bool MEM = K == 0;                  // half-diagonals and velocities in memory
  constexpr bool HM = MEM || NT * K > LDS_CELLS;  // bounds and heads in memory
  constexpr int KR = MEM ? 4 : K;  // cells a thread holds in registers at a time
  // slots this tier holds: K per thread in registers, or every slot of the domain's arrays
  const int CAP = MEM ? I[blockIdx.x].acap : NT * K;
  LoopShared& sh = s_loop;
  if (I[blockIdx.x].ls->done) return;
  // The descriptor through the constant address space (no launch writes it while it is read): its
  // fields are scalar loads that no store can alias, so the compiler keeps or repeats them as its
  // registers allow; as a copy they spilled 420 scalar registers.
  CInst& d = *(CInst*)(I + blockIdx.x);
  LoopState* ls = d.ls;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const float fInf = __builtin_inff();
  const double DelT = d.p.DelT, rX = d.p.rX;
  const int n_pool = S[blockIdx.x].n_pool;
  const int Na = ls->Na;
  const int ns_first = ls->nslots;
  const int ns_pre = min(ls->nslots_pre < 0 ? ns_first : ls->nslots_pre, d.capslots);  // slots whose entries have a CapRec
  const int nrec = uni(d.precap + ns_pre * AMCD_NB);  // entries that have one
  const Liveness<GD> live = {s_dead_bits, d.aVS};
  if (!GD && Na <= AMCD_DEAD_BITS) {  // liveness bitmap from the current states
    for (int wd = tid; wd < (Na + 31) / 32; wd += NT) {
      typedef unsigned v4u __attribute__((ext_vector_type(4)));
      const auto q = gmem((const v4u*)(d.aVS + 32 * (size_t)wd));  // (256 bytes are allocated beyond the end)
      const v4u x = q[0], y = q[1];
      unsigned b = 0;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        const unsigned v = j < 16 ? x[j / 4] : y[(j - 16) / 4];
        b |= (((v >> (8 * (j & 3))) & 0xffu) != 1u ? 1u : 0u) << j;
      }
      const int left = Na - 32 * wd;
      s_dead_bits[wd] = left < 32 ? b | ~0u << left : b;
    }
  }
  const unsigned long long c_start = clock64();  // the loop's own duration (stats)
  if (tid == 0) {
    int go = 1;
    if (!GD && Na > AMCD_DEAD_BITS)
      go = -3;  // more interface cells than the LDS bitmap holds: the host relaunches with GD
    else if (ns_first > CAP)
      go = -2;  // more growing cells than this tier holds
    else if (ls->pending)
      // resume with the pending nucleation, or ask again: another instance's larger tier relaunches the
      // loop for all of them, before the host has refilled this one's pool
      go = ls->pool_used >= n_pool || ls->pool_used >= d.poolcap || ls->nGrain >= d.gcap ? -1 : 2;
    else if (ls->events == 0 && Na == ls->nmushy0)
      go = 0;   // loop condition vSind2 != countS fails at once (S/VoxelsCA.C:381)
    sh.go = go;
    sh.r_i1 = ls->pend_tgt;
    sh.nslots = ns_first;
    sh.T = ls->tinc;
    sh.fin = go > 0 ? 1 : go == -3 ? -2 : go;  // (-1: pool refill, -2: larger tier)
    sh.units = 0;
    sh.back = 0;
    sh.cur = ls->rng;
  }
  if (tid < 32) sh.hist[tid] = 0;
  __syncthreads();
  const int go = sh.go;
  const int nm0 = ls->nmushy0;
  // engine state (meaningful in wave 0 only)
  EngineState es;
  es.T = sh.T;
  es.vSind2 = ls->vSind2;
  es.nGrain = ls->nGrain;
  es.pool_used = ls->pool_used;
  es.events = ls->events;
  es.captures = ls->captures;
  es.nucs = ls->nucs;
  es.nd = 0;
  es.visits = 0;
  unsigned long long units = 0;
  unsigned seen = 0, exact = 0;  // cells whose candidates this thread has looked at, and exact times of theirs
  Cells<KR> c;
  if (go > 0) {
    const unsigned int aj = lcg_pow(2ull * lane + 1);
    Window& win = sh.win;
    double T = sh.T;
#pragma unroll
    for (int k = 0; k < KR; ++k) c.E[k] = c.V[k] = 0.0;
    int ns = ns_first;  // slots the threads have taken over
    // Refresh of every cell whose head died (or of all) by its own thread.
    auto refresh_own = [&](bool all, int m, int scan0, double dtl, double T0) {
      for (int it = 0, s0 = w * 64; s0 < ns; ++it, s0 += NT) {
        const int s = s0 + lane;
        const int2 h = s < ns ? get_hd<HM>(d, s) : make_int2(0, -1);
        const bool on = h.y >= 0 && (all || live.dead(h.y));
        if (!__any(on)) continue;
        double e = 0.0, v = 0.0;
        if constexpr (MEM) {
          e = on ? gmem(d.gExt)[s] : 0.0;
          v = on ? gmem(d.gVhat)[s] : 0.0;
        } else {
#pragma unroll
          for (int k = 0; k < KR; ++k) {
            e = k == it ? c.E[k] : e;
            v = k == it ? c.V[k] : v;
          }
        }
        const Refreshed o = refresh_cell<GD>(d, live, on, h.x, e, v, -1, m, scan0, dtl, T0, T);
        if (on) {
          set_hd<HM>(d, s, o.c1, o.tgt);
          set_lh<HM>(d, s, o.lo, o.hi);
          if (o.tgt < 0) {
            if constexpr (MEM) {
              gmem(d.gExt)[s] = o.grown;
              gmem(d.gVhat)[s] = 0.0;
            } else {
#pragma unroll
              for (int k = 0; k < KR; ++k) {
                c.E[k] = k == it ? o.grown : c.E[k];
                c.V[k] = k == it ? 0.0 : c.V[k];
              }
            }
          }
        }
      }
    };
    // every cell starts at its list's first entry
    for (int s = tid; s < ns; s += NT) {
      const bool any = gmem(d.slots)[s].n > 0;
      set_hd<HM>(d, s, any ? gmem(d.slots)[s].base : 0, any ? 0 : -1);
      set_lh<HM>(d, s, fInf, fInf);
      if (MEM && !any) gmem(d.gVhat)[s] = 0.0;
    }
    if constexpr (!MEM) {
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int s = tid + k * NT;
        if (s < ns) {
          c.E[k] = gmem(d.gExt)[s];
          c.V[k] = get_hd<HM>(d, s).y >= 0 ? gmem(d.gVhat)[s] : 0.0;
        }
      }
    }
    refresh_own(true, 0, 0, 0.0, T);
    double step = first_span(DelT, ns_first);  // clock span of a window
    int nev = 0;  // events since the bounds were last recomputed
    int want = 44;  // heads asked for
    int start = 0;  // the first way of filling that the next window tries
    bool resume = go == 2;
    PHASE_INIT(pt);
    for (;;) {
      const double T0 = T;
      // ---- SELECT
      float u = fInf;
      const float Tf = (float)T, ibin = (float)(16.0 / step), top = Tf + 2.0f * (float)step;
      for (int s0 = w * 64; s0 < ns; s0 += 4 * NT) {
        float2 b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int s = s0 + lane + q * NT;
          b[q] = s < ns ? get_lh<HM>(d, s) : make_float2(fInf, fInf);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          u = fminf(u, b[q].y);
          if (b[q].x <= top) atomicAdd(&sh.hist[max(0, min(31, (int)((b[q].x - Tf) * ibin)))], 1);
        }
      }
      u = wave_min(u);
      if (lane == 0) sh.red[w] = u;
      if (tid < WCAP) {
        win.ev[tid] = make_int2(-2, -1);
        win.first[tid] = kPending;
        win.rank[tid] = 0;
      }
      if (w == 1) {  // the window's uniforms, one per lane (S/VoxelsCA.C:483)
        const unsigned int x1 = mod_m((unsigned long long)sh.cur * aj), x2 = lcg_next(x1);
        const unsigned long long nuc = __ballot(canonical(x1, x2) < rX);
        win.x2[lane] = x2;
        if (lane == 0) win.draws = nuc;
      }
      if (tid == 0) {
        win.n = 0;
        win.done = 0;
        win.scan0 = es.vSind2;
        sh.tn = 0;
        if constexpr (MEM) sh.tied = 0;
      }
      __syncthreads();
      PHASE(pt, 0);
      if (!resume) {
        u = wave_min(lane < NW ? sh.red[lane] : fInf);
        // the span that takes `want` heads (later entries of their cells and new cells' come on
        // top); the spans of the next windows follow it
        int cum = lane < 32 ? sh.hist[lane] : 0;
        cum += __builtin_amdgcn_update_dpp(0, cum, 0x111, 0xf, 0xf, false);
        cum += __builtin_amdgcn_update_dpp(0, cum, 0x112, 0xf, 0xf, false);
        cum += __builtin_amdgcn_update_dpp(0, cum, 0x114, 0xf, 0xf, false);
        cum += __builtin_amdgcn_update_dpp(0, cum, 0x118, 0xf, 0xf, false);
        cum += __builtin_amdgcn_update_dpp(0, cum, kBcast15, 0xa, 0xf, false);
        const int bins = __popcll(__ballot(lane < 32 && cum <= want));
        float W = fmaxf(Tf + (float)bins / ibin, u);
        // ---- the window's entries
        // 0: clock span, 1: less of it, 2: up to u, 3: exact best of every wave, one event.  Where one
        // window needed that, the next ones hold the same ties (a flat front's cells reach their
        // neighbours at one time), so in the memory tier, where each way costs a pass over every cell's
        // state, they begin there while more than a window's are left (118x93x74, 12 thousand growing
        // cells: 10.9K -> 10.3K cycles per event, 9.1K since ties leave the span alone; in the register
        // tiers the first ways cost little).
        int mode = start;
        for (;; ++mode) {
          if (mode > 0) W = mode == 1 ? fmaxf(Tf + 0.4f * (W - Tf), u) : u;
          if (mode < 3) {
            for (int s0 = tid; s0 < ns; s0 += KR * NT) {
              unsigned todo = 0;
#pragma unroll
              for (int k = 0; k < KR; ++k) {
                const int s = s0 + k * NT;
                const float lo = s < ns ? get_lh<HM>(d, s).x : fInf;
                todo |= (unsigned)(lo != fInf && lo <= W) << k;
              }
              while (todo != 0) {
                const int k1 = __builtin_ctz(todo);
                todo &= todo - 1;
                const int s = s0 + k1 * NT;
                double E = 0, V = 0;
                if constexpr (MEM) {
                  E = gmem(d.gExt)[s];
                  V = gmem(d.gVhat)[s];
                } else {
#pragma unroll
                  for (int k = 0; k < KR; ++k) {
                    E = k == k1 ? c.E[k] : E;
                    V = k == k1 ? c.V[k] : V;
                  }
                }
                const float2 b = get_lh<HM>(d, s);
                ++seen;
                push_cell<GD>(d, live, win, s, E, V, get_hd<HM>(d, s).x, b.x, b.y, T, W, nrec);
              }
              if (!MEM) break;
            }
          } else {  // exact best of every wave
            Best b = best_none();
            int bs = 0, near = 0;
            double be = 0, bv = 0;
            for (int s0 = tid; s0 < ns; s0 += KR * NT) {
#pragma unroll
              for (int k = 0; k < KR; ++k) {
                const int s = s0 + k * NT;
                const float lo = s < ns ? get_lh<HM>(d, s).x : fInf;
                if constexpr (MEM) near += lo != fInf && lo <= u;
                if (lo != fInf && lo <= u) {
                  ++seen;
                  exact += exact_cell<GD>(d, live, s, MEM ? gmem(d.gExt)[s] : c.E[k], MEM ? gmem(d.gVhat)[s] : c.V[k],
                                          get_hd<HM>(d, s).x, b, bs, be, bv);
                }
              }
              if (!MEM) break;
            }
            if (MEM && near != 0) atomicAdd(&sh.tied, near);
            const Best wb = wave_best(b);
            if (wb.cand >= 0 && wb.cand == b.cand) {
              const int i = put_entry(win, load_rec(d.cand + b.cand), be, bv, b.key, b.cand, bs, -1, order_key(-fInf),
                                      order_key(u));
              win.lim[i] = (int)0x80000000;
            }
          }
          __syncthreads();
          if (win.n <= WCAP) break;
          es.visits += win.n;
          __syncthreads();
          if (tid == 0) win.n = 0;
          __syncthreads();
        }
        step = next_span(step, bins, mode, DelT, ns_first);
        // (as many heads as leave room for what comes on top of them)
        if (start == 0) want = mode > 0 ? max(8, want * 5 / 8) : win.n < 44 ? min(56, want + 2) : win.n > 56 ? want - 1 : want;
        if constexpr (MEM) start = mode < 3 ? 0 : sh.tied > WCAP ? 3 : 2;
        {
          // every entry's position by its upper bound: each wave counts a share of the others
          const int n = win.n, j0 = w * (WCAP / NW);
          es.visits += mode < 3 ? n : 0;
          if (lane < n && j0 < n) {
            const int h = win.hi[lane];
            int before = 0;
#pragma unroll
            for (int j = 0; j < WCAP / NW; ++j) {
              const int hj = win.hi[j0 + j];
              before += (j0 + j < n) & ((hj < h) | ((hj == h) & (j0 + j < lane))) ? 1 : 0;
            }
            if (before) atomicAdd(&win.rank[lane], before);
          }
          if (w == NW - 1 && lane < n) win.y[lane] = 1.0 / win.V[lane];
        }
        __syncthreads();
        PHASE(pt, 1);
        // ---- ENGINE
        if (w == 0) {
          __builtin_amdgcn_s_setprio(3);
          engine_window(d, sh, win, es, W, DelT, n_pool, ls);
          __builtin_amdgcn_s_setprio(0);
        }
      } else if (w == 0) {
        // a resumed nucleation: the window's one event, decided before the suspension
        es.nGrain++;
        if (lane == 0) {
          const int i1 = sh.r_i1;
          win.dt[0] = 0.0;
          win.G = es.nGrain;
          win.pool = es.pool_used;
          win.m = 1;
          win.decided = 0;
          gmem(d.aScan)[i1] = es.vSind2;
          *gmem(&ls->pending) = 0;
          publish(win, 0, -1, i1);
          lds_put(&win.done, 1);
        }
        es.vSind2++;
        es.pool_used++;
        es.nucs++;
      }
      resume = false;
      PHASE(pt, 2);
      // ---- BUILD, while the engine goes on
      if (w > 0) build_cells<GD>(I + blockIdx.x, w - 1, NW - 1, nrec, nm0);
      __syncthreads();
      PHASE(pt, 3);
      T = sh.T;
      int fin = sh.fin;
      const int m = uni(win.m), scan0 = uni(win.scan0), ns1 = sh.nslots;
      if (w == 0) {
        units += (unsigned long long)win.decided * (unsigned)ns;
        if (lane < m) {
          const int i1 = win.ev[lane].y;
          live.kill(i1);
          gmem(d.aVS)[i1] = 2;
          const int later = win.decided - 1 - lane;  // events that the reference scans its cell for
          if (win.slot[lane] >= 0 && later > 0) atomicAdd(&sh.units, (unsigned long long)later);
        }
        nev += m;
        if (lane == 0) {
          sh.all = nev >= (1 << 20);
          sh.neg = 0;
          sh.back = kKeyInf;
        }
        nev = nev >= (1 << 20) ? 0 : nev;
      }
      if (m == 0 && fin == 1) fin = -4;  // a window always performs an event or ends the loop
      __syncthreads();
      // ---- APPLY: the cells whose head died (or, now and then, all), listed so that their list
      // reads run side by side over the workgroup
      const bool all = sh.all;
      if (tid < 32) sh.hist[tid] = 0;  // (read before ENGINE, filled again after APPLY)
      unsigned touched = 0;  // the thread's listed cells (register tiers)
      for (int s0 = w * 64; s0 < ns; s0 += KR * NT) {
        unsigned bits = 0;
        int total = 0;
#pragma unroll
        for (int k = 0; k < KR; ++k) {
          const int s = s0 + lane + k * NT;
          const int tg = s < ns ? get_hd<HM>(d, s).y : -1;
          const bool dd = live.dead(tg >= 0 ? tg : 0);
          const bool on = tg >= 0 && (dd || all);
          bits |= (unsigned)on << k;
          total += __popcll(__ballot(on));
        }
        if (total != 0) {
          int base = 0;
          if (lane == 0) base = atomicAdd(&sh.tn, total);
          base = uni(base);
#pragma unroll
          for (int k = 0; k < KR; ++k) {
            const bool on = (bits >> k) & 1u;
            const unsigned long long bal = __ballot(on);
            if (bal == 0) continue;
            const int i = base + __popcll(bal & ((1ull << lane) - 1));
            base += __popcll(bal);
            if (on && i < TCAP) {
              const int s = s0 + lane + k * NT;
              sh.tS[i] = s;
              sh.tE[i] = MEM ? gmem(d.gExt)[s] : c.E[k];
              sh.tV[i] = MEM ? gmem(d.gVhat)[s] : c.V[k];
            }
          }
        }
        touched = bits;
        if (!MEM) break;
      }
      __syncthreads();
      PHASE(pt, 4);
      const double dtl = lane < m ? win.dt[lane] : 0.0;  // lane j: growth time of event j
      int nt = sh.tn;
      if (nt > TCAP || all) {  // more than the list holds
        refresh_own(all, m, scan0, dtl, T0);
        nt = 0;
        touched = 0;
      }
      // growth, event by event in the reference's order (S/VoxelsCA.C:511-516), of the cells of
      // before the window; a nucleation's time is 0: E + V*0 = E
      bool neg = false;
      float back = fInf;  // CandRec::back over the cells, after the window
      for (int s0 = w * 64; s0 < ns; s0 += KR * NT) {
        if constexpr (MEM) {
#pragma unroll
          for (int k = 0; k < KR; ++k) {
            const int s = s0 + lane + k * NT;
            c.E[k] = s < ns ? gmem(d.gExt)[s] : 0.0;
            c.V[k] = s < ns ? gmem(d.gVhat)[s] : 0.0;
          }
        }
        for (int j = 0; j < m; ++j) {
          const double dt = lane_f64(dtl, j);
#pragma unroll
          for (int k = 0; k < KR; ++k) c.E[k] = c.E[k] + c.V[k] * dt;
        }
#pragma unroll
        for (int k = 0; k < KR; ++k) {
          neg |= c.E[k] < 0.0;
          if (s0 + lane + k * NT < ns) back = fminf(back, step_back(c.E[k], c.V[k]));
          if constexpr (MEM) {
            const int s = s0 + lane + k * NT;
            if (s < ns) gmem(d.gExt)[s] = c.E[k];
          }
        }
        if (!MEM) break;
      }
      int fixs = -1;  // a cell out of candidates, and its final half-diagonal (memory tier)
      double fixe = 0.0;
      static_assert(!MEM || TCAP + WCAP <= NT, "one round over the list");
      for (int i0 = 0; i0 < nt + m; i0 += NT) {
        const int i = i0 + lane * NW + w;  // spread over the waves
        int s = -1, k0 = -1, c0 = 0;
        double e = 0.0, v = 0.0;
        if (i < nt) {
          s = sh.tS[i];
          e = sh.tE[i];
          v = sh.tV[i];
          c0 = get_hd<HM>(d, s).x;
        } else if (i < nt + m) {
          k0 = i - nt;
          s = win.slot[k0];
          if (s >= 0) {
            c0 = win.base[k0];
            e = win.E0[k0];
            v = win.V0[k0];
          }
        }
        const Refreshed o = refresh_cell<GD>(d, live, s >= 0, c0, e, v, k0, m, scan0, dtl, T0, T);
        if (s >= 0) {
          if (i < nt) {
            sh.tE[i] = o.grown;
          } else {
            gmem(d.gExt)[s] = o.grown;
            gmem(d.gVhat)[s] = v;
            back = fminf(back, step_back(o.grown, v));
          }
          if (HM || s < CAP) {
            set_hd<HM>(d, s, o.tgt >= 0 ? o.c1 : i, o.tgt);
            set_lh<HM>(d, s, o.lo, o.hi);
          }
          if (MEM && o.tgt < 0) {
            fixs = s;
            fixe = o.grown;
          }
        }
      }
      if (neg) sh.neg = 1;
      back = wave_min(back);
      if (lane == 0) atomicMin(&sh.back, __float_as_int(back * (1.0f - 0x1p-16f)));
      __syncthreads();
      PHASE(pt, 5);
      // what the list's threads found: cells out of candidates, and the new cells
      if constexpr (MEM) {
        if (fixs >= 0) {
          gmem(d.gExt)[fixs] = fixe;
          gmem(d.gVhat)[fixs] = 0.0;
        }
      } else {
#pragma unroll
        for (int k = 0; k < KR; ++k) {
          const int s = tid + k * NT;
          if ((touched >> k) & 1u) {
            const int2 h = get_hd<HM>(d, s);
            if (h.y < 0) {
              c.E[k] = sh.tE[h.x];
              c.V[k] = 0.0;
            }
          }
          if (s >= ns && s < ns1) {
            c.E[k] = gmem(d.gExt)[s];
            c.V[k] = get_hd<HM>(d, s).y >= 0 ? gmem(d.gVhat)[s] : 0.0;
          }
        }
      }
      if (sh.neg) {
        // the reference's clamp at zero, which moves the cell's capture times: only a window's
        // last event can take a half-diagonal there and so need it
        if constexpr (MEM) __syncthreads();
        for (int s0 = tid; s0 < ns; s0 += KR * NT) {
#pragma unroll
          for (int k = 0; k < KR; ++k) {
            const int s = s0 + k * NT;
            if (s >= ns) continue;
            if ((MEM ? gmem(d.gExt)[s] : c.E[k]) < 0.0) {
              if constexpr (MEM) gmem(d.gExt)[s] = 0.0;
              else c.E[k] = 0.0;
              const int2 h = get_hd<HM>(d, s);
              if (h.y >= 0) {
                float lo, hi;
                tau_bounds(load_rec(d.cand + h.x).D, 0.0, MEM ? gmem(d.gVhat)[s] : c.V[k], T, lo, hi);
                set_lh<HM>(d, s, lo, hi);
              }
            }
          }
          if (!MEM) break;
        }
      }
      if (MEM) __syncthreads();  // (another thread's stores of a cell's state)
      ns = min(ns1, CAP);
      PHASE(pt, 6);
      if (ns1 > CAP && fin == 1) fin = T < DelT ? -2 : 0;  // cells beyond this tier: the host resumes
      if (fin != 1) {
        if (tid == 0) sh.fin = fin;
        break;
      }
    }
    // half-diagonals back to the growing list (the cells not taken over are current there)
    if constexpr (!MEM) {
#pragma unroll
      for (int k = 0; k < KR; ++k) {
        const int s = tid + k * NT;
        if (s < ns) gmem(d.gExt)[s] = c.E[k];
      }
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    seen += __shfl_xor(seen, o);
    exact += __shfl_xor(exact, o);
  }
  if (lane == 0) {
    sh.seen[w] = seen;
    sh.exact[w] = exact;
  }
  if (tid == 0) sh.nexec = es.vSind2 - nm0;
  __syncthreads();
  // ---- loop state and counters
  const int ns = sh.nslots;
  const int fin = sh.fin;
  if (fin == 0) {
    // the step's events, and the half-diagonals of every growing cell, to the active arrays
    for (int q = tid; q < sh.nexec; q += NT) {
      const EventRec e = d.events[q];
      gmem(d.aG)[e.i1] = e.G;
      gmem(d.aCx)[e.i1] = e.x;
      gmem(d.aCy)[e.i1] = e.y;
      gmem(d.aCz)[e.i1] = e.z;
      gmem(d.aExt)[e.i1] = e.E;
    }
    __syncthreads();
    for (int s = tid; s < ns; s += NT) gmem(d.aExt)[gmem(d.slots)[s].act] = gmem(d.gExt)[s];
  }
  if (tid == 0) {
    const int status = go == -3 ? -3 : fin == -1 ? 1 : fin == -2 ? 2 : fin == 0 ? 0 : -4;
    ls->nslots_pre = ns_pre;
    ls->tinc = es.T;
    ls->vSind2 = es.vSind2;
    ls->nGrain = es.nGrain;
    ls->pool_used = es.pool_used;
    ls->events = es.events;
    ls->captures = es.captures;
    ls->nucs = es.nucs;
    ls->rng = sh.cur;
    ls->draws += 2ll * es.nd;
    ls->nslots = ns;
    ls->done = ls->fin = status == 0 ? 1 : 0;
    amcd_out& o = O[blockIdx.x];
    o.status = status;
    o.n_events = es.events;
    o.n_captures = es.captures;
    o.n_nucleations = es.nucs;
    o.n_slots = ns;
    o.nGrain = es.nGrain;
    o.pool_used = es.pool_used;
    o.tinc = es.T;
    o.draws = ls->draws;
    o.interface_events += (long long)(units + sh.units);
    o.cand_evals += es.visits;
    for (int q = 0; q < NW; ++q) {
      o.slot_visits += sh.seen[q];
      o.cand_evals += sh.exact[q];
    }
    o.loop_cycles += (long long)(clock64() - c_start);
  }
}

// The step's results back to the grid (S/VoxelsCA.C:633-643) and ConvertSolid1(0)
// (S/VoxelsCA.C:739-758): mushy -> solid when every Moore neighbour is mushy or solid.  Every mushy
// voxel is in the active list, so only those are visited, and so is every liquid neighbour of one: a
// neighbour whose state in the grid is liquid has been captured when its active state is mushy,
// whether its own thread has written the grid yet or not, and a state that has been written (2, or
// 3 from 2) counts the same.  One pass instead of two: only what a step changes is written (the
// octahedra of captured voxels, half-diagonals of mushy ones), 6.9 + 9.1 -> 12.8 us for the 512x512x128
// raster.  Also clears the voxel -> active map for the next step.  The pass leaves the grid as it is
// while the step will be run again (an overflow in any instance) or the loop be resumed; run a second
// time it writes the same values.
__global__ __launch_bounds__(GB) void k_finish(Inst* I, const int* astart, int ninst, const amcd_out* O) {
  int ii = find_inst(astart, ninst, blockIdx.x);
  const int Na = I[ii].ls->Na, nb = astart[ii + 1] - astart[ii], b0 = blockIdx.x - astart[ii];
  if (!I[ii].ls->fin || b0 * GB >= Na) return;  // (before the descriptor is read)
  int again = 0;
  for (int q = threadIdx.x; q < ninst; q += GB) again |= O[q].overflow;
  if (__syncthreads_or(again)) return;
  const Inst d = I[ii];  // a copy: stores in the loops cannot alias it
  const int end = min(Na, d.acap);
  for (int a = b0 * GB + (int)threadIdx.x; a < end; a += nb * GB) {
    const int v = d.aVox[a];
    d.amap[v] = -1;
    if (d.aVS[a] != 2) continue;
    const uint8_t s0 = d.vs[v];
    int i, j, k;
    decode(d, v, i, j, k);
    const int* nbr = d.aRow[a].nbr;
    uint8_t sn[AMCD_NB];
#pragma unroll
    for (int q = 0; q < AMCD_NB; ++q) {  // (the nine rows' bytes side by side; outside the domain: solid)
      const int qq = q < 13 ? q : q + 1, x = i + qq % 3 - 1, y = j + (qq / 3) % 3 - 1, z = k + qq / 9 - 1;
      const bool in = x >= 0 && x < d.p.nx && y >= 0 && y < d.p.ny && z >= 0 && z < d.p.nz;
      sn[q] = in ? d.vs[v + (qq / 9 - 1) * d.nxy + ((qq / 3) % 3 - 1) * d.p.nx + qq % 3 - 1] : 3;
    }
    unsigned liq = 0, none = 0;
#pragma unroll
    for (int q = 0; q < AMCD_NB; ++q) {
      liq |= ((sn[q] & 3) == 1 ? 1u : 0u) << q;
      none |= (sn[q] & 3) == 0 ? 1u : 0u;
    }
    bool solid = none == 0;
    for (; solid && liq != 0; liq &= liq - 1) {
      const int n = nbr[__builtin_ctz(liq)];
      solid = n >= 0 && d.aVS[n] == 2;
    }
    const uint8_t s1 = (s0 & 0xC0) | (solid ? 3 : 2);
    if (s1 != s0) d.vs[v] = s1;
    d.ext[v] = solid ? 0.0 : d.aExt[a];
    if ((s0 & 3) == 1) {  // captured in this step
      d.gid[v] = d.aG[a];
      d.cx[v] = d.aCx[a];
      d.cy[v] = d.aCy[a];
      d.cz[v] = d.aCz[a];
    }
  }
}

// ---- per-layer helpers ---------------------------------------------------------------
// A step's records: in from the pinned staging area with fresh output records (`clear` words) and the
// instances' nucleation pools (a workgroup each, after the first `nrec`), and the outputs back.  As
// kernels in the step's graph they cost 3.5 us each; as stream copies beside it, 10.
__global__ void k_step_in(unsigned* steps, const unsigned* staged, int nwords, unsigned* outs, int clear, const Inst* I,
                          int nrec, const double* dpool, const double* hpool) {
  if ((int)blockIdx.x < nrec) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < nwords) steps[q] = staged[q];
    if (q < clear) outs[q] = 0u;
    return;
  }
  const int i = blockIdx.x - nrec;
  const int n = 9 * min(((const amcd_step*)staged)[i].n_pool, I[i].poolcap);
  double* to = I[i].pool;
  const double* from = hpool + (to - dpool);
  for (int q = threadIdx.x; q < n; q += blockDim.x) to[q] = from[q];
}
__global__ void k_step_out(unsigned* staged, const unsigned* outs, int nwords) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nwords) staged[q] = outs[q];
}
// After a host upload of vState: the "T >= tL" flag (bit 7) follows the device's current
// temperature field, so SetLiquid3 still sees the caller's melt pool.
__global__ void k_rehot(uint8_t* vs, const double* T, int N, double tL) {
  size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= (size_t)N) return;
  vs[v] = (uint8_t)((vs[v] & 0x7f) | (T[v] >= tL ? 0x80 : 0));
}
__global__ void k_grain_presence(const int* gid, int N, int* present, int ngrain) {
  size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= (size_t)N) return;
  int g = gid[v];
  if (g > 0 && g <= ngrain && present[g - 1] == 0) present[g - 1] = 1;
}
__global__ void k_remap(int* gid, int N, const int* remap, int ngrain) {
  size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= (size_t)N) return;
  int g = gid[v];
  if (g > 0 && g <= ngrain) gid[v] = remap[g - 1];
}
// Voronoi labelling of a z-slab: each voxel takes the first site (in draw
// order) at the smallest FP64 squared distance, ((ax*ax + ay*ay) + az*az) with no
// contraction, the order the reference evaluates it in.
//   plate (S/BasePlate.C:74-78, 104-117): voxel centres ((i + .5) dx, ...), planes
//     0..nz-1; the first site is taken unconditionally (start at +inf, strict <).
//   powder layer (S/VoxelsCA.C:920-933): voxel corners (i dx, j dy, (z0 + k) dz), planes
//     z0..z0+nz-1 (planes above the domain included, as the reference labels them);
//     best distance starts at 1e6, strict <.
// A block takes a brick of 8x8x4 voxels at a time.  No site whose distance from the brick's box exceeds the
// least of the sites' largest distances to it can be a voxel's nearest (with a margin far
// above rounding), so the block first finds that least distance, one site a thread, and then every voxel
// looks at the remaining sites, in draw order, from LDS: some tens of them instead of all.  Plate mode
// writes the base-plate fields of S/VoxelsCA.C:125-161 directly; layer mode writes the label and marks
// the site used.  512x512x80 voxels, 2000 sites: 16.0 -> 0.47 ms (FP64 bound then, site reads from the L2
// now).
#define VOR_B 256  // threads, voxels of a brick, sites looked at together
template <bool LAYER>
__global__ __launch_bounds__(VOR_B) void k_voronoi(Inst* I, int ii, int z0, int nz, const double* __restrict__ xs,
                                                   int ng, int* __restrict__ label, int* __restrict__ used) {
  __shared__ double sx[VOR_B], sy[VOR_B], sz[VOR_B], su[VOR_B / 64];
  __shared__ int si[VOR_B], sn[VOR_B / 64];
  const Inst& d = I[ii];
  const int nx = d.p.nx, ny = d.p.ny, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int bx = (nx + 7) / 8, by = (ny + 7) / 8, nb = bx * by * ((nz + 3) / 4);
  const double dx = d.p.dx, dy = d.p.dy, dz = d.p.dz;
  auto at = [&](int i, int j, int k, double& x, double& y, double& z) {
    if (LAYER) {
      x = i * dx;
      y = j * dy;
      z = (z0 + k) * dz;
    } else {
      x = ((double)i + .5) * dx;
      y = ((double)j + .5) * dy;
      z = ((double)(z0 + k) + .5) * dz;
    }
  };
  for (int b = blockIdx.x; b < nb; b += gridDim.x) {
    const int kb = b / (bx * by), jb = (b - kb * bx * by) / bx, ib = b - (kb * by + jb) * bx;
    const int i = 8 * ib + (tid & 7), j = 8 * jb + ((tid >> 3) & 7), k = 4 * kb + (tid >> 6);
    const bool in = i < nx && j < ny && k < nz;
    double x, y, z, lo[3], hi[3];
    at(i, j, k, x, y, z);
    at(8 * ib, 8 * jb, 4 * kb, lo[0], lo[1], lo[2]);
    at(min(nx, 8 * ib + 8) - 1, min(ny, 8 * jb + 8) - 1, min(nz, 4 * kb + 4) - 1, hi[0], hi[1], hi[2]);
    double far = __builtin_huge_val();
    for (int q = tid; q < ng; q += VOR_B) {
      double s2 = 0.0;
      for (int c = 0; c < 3; ++c) {
        const double s = xs[3 * q + c], m = fmax(fabs(s - lo[c]), fabs(s - hi[c]));
        s2 += m * m;
      }
      far = fmin(far, s2);
    }
    for (int o = 32; o >= 1; o >>= 1) far = fmin(far, __shfl_xor(far, o));
    if (lane == 0) su[w] = far;
    __syncthreads();
    for (int q = 0; q < VOR_B / 64; ++q) far = fmin(far, su[q]);
    far *= 1 + 1e-9;
    double bd = LAYER ? 1e6 : __builtin_huge_val();
    int best = 0;
    for (int c0 = 0; c0 < ng; c0 += VOR_B) {
      double s[3] = {0.0, 0.0, 0.0}, near = 0.0;
      bool keep = false;
      if (c0 + tid < ng) {
        for (int c = 0; c < 3; ++c) {
          s[c] = xs[3 * (c0 + tid) + c];
          const double m = fmax(0.0, fmax(lo[c] - s[c], s[c] - hi[c]));
          near += m * m;
        }
        keep = !(near > far);
      }
      const unsigned long long bal = __ballot(keep);
      if (lane == 0) sn[w] = __popcll(bal);
      __syncthreads();  // (the last sites have been looked at)
      int base = 0, m = 0;
      for (int q = 0; q < VOR_B / 64; ++q) {
        base += q < w ? sn[q] : 0;
        m += sn[q];
      }
      if (keep) {
        const int p = base + __popcll(bal & ((1ull << lane) - 1));
        sx[p] = s[0];
        sy[p] = s[1];
        sz[p] = s[2];
        si[p] = c0 + tid;
      }
      __syncthreads();
      for (int q = 0; q < m; ++q) {
        const double ax = x - sx[q], ay = y - sy[q], az = z - sz[q];
        const double dd = ax * ax + ay * ay + az * az;
        const bool lt = dd < bd;
        bd = lt ? dd : bd;
        best = lt ? si[q] : best;
      }
      __syncthreads();
    }
    const long long v = (long long)d.nxy * k + (long long)nx * j + i;
    if (in && LAYER) {
      label[v] = best;
      used[best] = 1;
    } else if (in) {
      d.gid[v] = best + 1;
      d.vs[v] = (v < (long long)d.nxy * (nz - 1)) ? 3 : 2;
      d.cx[v] = x;
      d.cy[v] = y;
      d.cz[v] = z;
    }
  }
}

// AddLayer1's continuous renumbering (S/VoxelsCA.C:935-947): rank[s] = number of used
// sites before s; the total goes to *n_used.  One workgroup.
__global__ __launch_bounds__(1024) void k_site_rank(const int* __restrict__ used, int ng, int* __restrict__ rank,
                                                    int* __restrict__ n_used) {
  __shared__ int wsum[16];
  __shared__ int carry;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int c0 = 0; c0 < ng; c0 += 1024) {
    const int s = c0 + threadIdx.x;
    const int u = (s < ng && used[s]) ? 1 : 0;
    int inc = u;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(inc, o);
      inc += lane >= o ? t : 0;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int before = carry;
    for (int q = 0; q < w; ++q) before += wsum[q];
    if (s < ng) rank[s] = before + inc - u;
    __syncthreads();
    if (threadIdx.x == 1023) carry = before + inc;
    __syncthreads();
  }
  if (threadIdx.x == 0) *n_used = carry;
}

// AddLayer1's voxel writes (S/VoxelsCA.C:952-981): the new layer takes the renumbered
// Voronoi labels as solid grains gbase + 1.., everything at or above the laser plane is
// emptied.
__global__ void k_write_layer(Inst* I, int ii, int iz1, int ilaserLoc, int gbase, const int* __restrict__ label,
                              const int* __restrict__ rank) {
  const Inst& d = I[ii];
  size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= (size_t)d.N) return;
  int i, j, k;
  decode(d, (int)v, i, j, k);
  if (k >= iz1 && k < ilaserLoc) {
    int jind = d.nxy * (k - iz1) + d.p.nx * j + i;
    d.gid[v] = gbase + rank[label[jind]] + 1;
    d.vs[v] = 3;
    d.cx[v] = ((double)i + .5) * d.p.dx;
    d.cy[v] = ((double)j + .5) * d.p.dy;
    d.cz[v] = ((double)k + .5) * d.p.dz;
  }
  if ((long long)v >= (long long)d.nxy * ilaserLoc) {
    d.vs[v] = 0;
    d.gid[v] = 0;
  }
}

// -------------------------------------------------------------------------------------
// host side of the device library
struct amcd_batch {
  int n = 0;
  int dev = 0;
  hipStream_t stream = nullptr;
  std::vector<Inst> h;      // host mirror of the descriptors
  Inst* d_inst = nullptr;
  int *d_bstartG = nullptr, *d_bstartZ = nullptr, *d_astart = nullptr, *d_bstartS = nullptr, *d_bstartT = nullptr,
      *d_lstart = nullptr, *d_cstart = nullptr, *d_bstartF = nullptr;
  std::vector<int> bstartG, bstartZ, astart, bstartS, bstartT, lstart, cstart, bstartF;
  amcd_step* d_steps = nullptr;
  amcd_out* d_outs = nullptr;
  amcd_step* h_steps = nullptr;  // pinned
  amcd_out* h_outs = nullptr;    // pinned
  bool staged = false;  // launched work may still have to read h_steps
  std::vector<void*> allocs;
  hipEvent_t ev[16];
  double last_ms[16] = {0};
  bool timing = false;
  int tier = 1;  // capture-loop capacity tier (see launch_event_loop)
  int min_tier = 0;  // lowest tier a step starts in (AMCAFE_CAPTURE_TIER_MIN; tests use it to
                     // run small decks in the larger tiers; 5 = memory tier, bitmap in memory)
  // nucleation pools of every instance in one device region (instance i's at pool_off[i]
  // entries of 9 doubles), staged in pinned memory, from which the step takes them
  double* d_pool = nullptr;
  double* h_pool = nullptr;  // pinned
  uint8_t* d_mark = nullptr;  // SetBuild's grain marks (mark_cap bytes)
  size_t mark_cap = 0;
  std::vector<size_t> pool_off;
  std::vector<std::pair<void**, size_t>> wanted;  // device arrays of the next allocation
  unsigned long long* d_evals = nullptr;  // source integrals of an EASM evaluation
  // The driver's step as HIP graphs (AMCAFE_GRAPH=0 launches the stages one by one): the stages up
  // to the capture loop, per capture tier, and the finishing pass; each is captured again when the
  // block counts it was captured with change (capacity growth)
  bool graphs = true;
  hipGraphExec_t gstep[6] = {};
  long long gstep_key[6] = {};
  hipGraphExec_t gfin = nullptr;
  long long gfin_key = -1;
  std::vector<int> astart_up, lstart_up;  // the block lists the device holds
  // Active-list chunking: blocks per instance of the candidate-list pass, picked by timing
  // the pass (which only rebuilds lists from their inputs) at each candidate, again each time
  // the largest growing list has doubled (AMCAFE_AUTOTUNE=0 keeps the default)
  int list_cap = 2048;
  bool autotune = true, tuned = false;
  bool tune_pending = false;  // the next step tunes (between its list pass and its capture loop)
  int tuned_at = 0;  // largest growing list at the last tuning
  int n_tunings = 0;
  float tune_ms[8] = {0};
};

static thread_local std::string g_dev_err;
#define HIPT(x)                                                                        \
  do {                                                                                 \
    hipError_t e_ = (x);                                                               \
    if (e_ != hipSuccess) {                                                            \
      g_dev_err = std::string(#x) + ": " + hipGetErrorString(e_);                      \
      return -1;                                                                       \
    }                                                                                  \
  } while (0)

// Device arrays are asked for one by one and come out of one allocation: freeing an allocation
// waits for the device, 95 us each; twelve domains' 505 took 48 ms to close, as one 2 ms.
// Every array has 256 bytes beyond its length: the list-block reads of the
// capture loop run up to four entries past the last slot's list.
template <class T>
static void want(amcd_batch* b, T** p, size_t n) {
  b->wanted.emplace_back((void**)p, (n * sizeof(T) + 256 + 255) & ~(size_t)255);
}
static int alloc_wanted(amcd_batch* b) {
  std::vector<std::pair<void**, size_t>> wanted;
  wanted.swap(b->wanted);
  size_t total = 0;
  for (const auto& w : wanted) total += w.second;
  char* q = nullptr;
  HIPT(hipMalloc((void**)&q, total));
  b->allocs.push_back(q);
  for (const auto& w : wanted) {
    *w.first = q;
    q += w.second;
  }
  return 0;
}

static void want_active(amcd_batch* b, Inst& d, int acap) {
  d.acap = acap;
  size_t c = (size_t)acap;
  // Growing cells are a tenth of the active ones in a raster, and what they need beyond a list of their
  // own is sized for a quarter: records of captures, and about 27 entries of lists ahead each.  2.15 KB per
  // active cell in all; cells beyond that go without (see Inst::cand).
  d.capslots = (int)(c / 4);
  d.precap = (int)std::min<size_t>(6 * c, (size_t)1 << 26);
  if (c * AMCD_NB + (size_t)d.precap > 0x7fffff00ull) d.precap = 0;  // entries are counted in 32 bits
  want(b, &d.aVox, c);
  want(b, &d.aVS, c);
  want(b, &d.aG, c);
  want(b, &d.aT, c);
  want(b, &d.aExt, c);
  want(b, &d.aCx, c);
  want(b, &d.aCy, c);
  want(b, &d.aCz, c);
  want(b, &d.ruq, c);
  want(b, &d.aRow, c);
  want(b, &d.events, c);
  want(b, &d.aScan, c);
  want(b, &d.slots, c);
  want(b, &d.gExt, c);
  want(b, &d.gVhat, c);
  want(b, &d.gLH, c);
  want(b, &d.gHd, c);
  want(b, &d.cand, c * AMCD_NB + d.precap);
  want(b, &d.cap, (size_t)d.capslots * AMCD_NB + d.precap);
  want(b, &d.cF, c * AMCD_NB);
}

static int push_inst(amcd_batch* b) {
  HIPT(hipMemcpyAsync(b->d_inst, b->h.data(), sizeof(Inst) * b->n, hipMemcpyHostToDevice, b->stream));
  return 0;
}

extern "C" {

const char* amcd_last_error() { return g_dev_err.c_str(); }

int amcd_device_name(char* buf, int len) {
  hipDeviceProp_t pr;
  int dev = 0;
  HIPT(hipGetDevice(&dev));
  HIPT(hipGetDeviceProperties(&pr, dev));
  snprintf(buf, len, "%s (%s, %d CUs)", pr.name, pr.gcnArchName, pr.multiProcessorCount);
  return 0;
}

int amcd_create(const amcd_params* p, int n, amcd_batch** out, char* err, int errlen) {
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
    snprintf(err, errlen, "no HIP device");
    return -1;
  }
  amcd_batch* b = new amcd_batch();
  b->n = n;
  b->h.resize(n);
  if (const char* g = getenv("AMCAFE_GRAPH")) b->graphs = atoi(g) != 0;
  if (const char* t = getenv("AMCAFE_AUTOTUNE")) b->autotune = atoi(t) != 0;
  if (const char* mt = getenv("AMCAFE_CAPTURE_TIER_MIN")) {
    b->min_tier = std::max(0, std::min(5, atoi(mt)));  // 5: the memory tier with the bitmap in memory
    b->tier = std::max(b->tier, b->min_tier);
  }
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    snprintf(err, errlen, "hipStreamCreate failed");
    delete b;
    return -1;
  }
  for (int q = 0; q < 16; ++q)
    if (hipEventCreate(&b->ev[q]) != hipSuccess) {
      snprintf(err, errlen, "hipEventCreate failed");
      amcd_destroy(b);
      return -1;
    }
  b->bstartG.assign(n + 1, 0);
  b->bstartS.assign(n + 1, 0);
  b->bstartT.assign(n + 1, 0);
  b->lstart.assign(n + 1, 0);
  b->cstart.assign(n + 1, 0);
  b->bstartZ.assign(n + 1, 0);
  b->bstartF.assign(n + 1, 0);
  b->astart.assign(n + 1, 0);
  for (int i = 0; i < n; ++i) {
    Inst& d = b->h[i];
    memset(&d, 0, sizeof(Inst));
    d.p = p[i];
    long long N = (long long)p[i].nx * p[i].ny * p[i].nz;
    if (N <= 0 || N > 0x7fffffffLL - 4096) {
      snprintf(err, errlen, "domain %d: voxel count %lld out of range", i, N);
      amcd_destroy(b);
      return -1;
    }
    d.N = (int)N;
    d.nxy = p[i].nx * p[i].ny;
    d.nblkZ = (d.N + ZB - 1) / ZB;
    d.nblkG = (d.N + GB - 1) / GB;
    d.nblkS = (d.N + SB - 1) / SB;
    d.nblkT = (d.N + GB * TV - 1) / (GB * TV);
    size_t Nn = (size_t)d.N;
    want(b, &d.vs, Nn);
    want(b, &d.gid, Nn);
    want(b, &d.ext, Nn);
    want(b, &d.cx, Nn);
    want(b, &d.cy, Nn);
    want(b, &d.cz, Nn);
    want(b, &d.T, Nn);
    want(b, &d.bj, Nn);
    want(b, &d.build, Nn);
    want(b, &d.amap, Nn);
    want(b, &d.bcA, (size_t)d.nblkZ);
    want(b, &d.bcM, (size_t)d.nblkZ);
    want(b, &d.chA, (size_t)d.nblkZ / 1024 + 1);
    want(b, &d.chM, (size_t)d.nblkZ / 1024 + 1);
    want(b, &d.zliq, 2 * (size_t)p[i].nz);
    want(b, &d.ls, 1);
    // (it grows on overflow; 2^23 interface cells are far more than a domain this size needs)
    int acap = (int)std::min<long long>(N, std::max<long long>(1 << 16, std::min<long long>(N / 8, 1 << 23)));
    if (const char* ac = getenv("AMCAFE_ACTIVE_CAP_INIT"))  // tests: start small to exercise the growth path
      acap = (int)std::min<long long>(N, std::max(64, atoi(ac)));
    want_active(b, d, acap);
    d.gcap = 0;
    d.rot = nullptr;
    d.poolcap = 0;
    d.pool = nullptr;
    b->bstartG[i + 1] = b->bstartG[i] + d.nblkG;
    b->bstartS[i + 1] = b->bstartS[i] + d.nblkS;
    b->bstartT[i + 1] = b->bstartT[i] + std::min(d.nblkT, std::max(64, 2048 / n));  // (what the chip holds at a time)
    b->cstart[i + 1] = b->cstart[i] + (d.nblkZ + 1023) / 1024;
    b->bstartZ[i + 1] = b->bstartZ[i] + d.nblkZ;
    b->bstartF[i + 1] = b->bstartF[i] + (d.nblkZ + 3) / 4;
  }
  want(b, &b->d_inst, (size_t)n);
  for (int** starts : {&b->d_bstartG, &b->d_bstartS, &b->d_bstartT, &b->d_lstart, &b->d_cstart, &b->d_bstartZ, &b->d_astart,
                       &b->d_bstartF})
    want(b, starts, (size_t)n + 1);
  want(b, &b->d_steps, (size_t)n);
  want(b, &b->d_outs, (size_t)n);
  want(b, &b->d_evals, 1);
  if (alloc_wanted(b)) {
    snprintf(err, errlen, "%s", g_dev_err.c_str());
    amcd_destroy(b);
    return -1;
  }
  for (Inst& d : b->h) {
    size_t Nn = (size_t)d.N;
    hipError_t me = hipSuccess;
    auto zero = [&](void* q, int val, size_t bytes) {
      const hipError_t e = hipMemsetAsync(q, val, bytes, b->stream);
      if (me == hipSuccess) me = e;
    };
    zero(d.vs, 0, Nn);
    zero(d.gid, 0, Nn * 4);
    zero(d.ext, 0, Nn * 8);
    zero(d.cx, 0, Nn * 8);
    zero(d.cy, 0, Nn * 8);
    zero(d.cz, 0, Nn * 8);
    zero(d.T, 0, Nn * 8);
    zero(d.bj, 0, Nn);
    zero(d.build, 0, Nn);
    zero(d.zliq, 0xff, (size_t)d.p.nz * 8);  // unknown: every plane may hold liquid
    zero(d.amap, 0xff, Nn * 4);
    zero(d.ls, 0, sizeof(LoopState));
    if (me != hipSuccess) {
      snprintf(err, errlen, "hipMemsetAsync: %s", hipGetErrorString(me));
      amcd_destroy(b);
      return -1;
    }
  }
  if (hipHostMalloc((void**)&b->h_steps, sizeof(amcd_step) * n, 0) != hipSuccess ||
      hipHostMalloc((void**)&b->h_outs, sizeof(amcd_out) * n, 0) != hipSuccess) {
    snprintf(err, errlen, "hipHostMalloc failed");
    amcd_destroy(b);
    return -1;
  }
  const std::pair<int*, const std::vector<int>*> starts[] = {{b->d_bstartG, &b->bstartG}, {b->d_bstartS, &b->bstartS},
                                                             {b->d_bstartT, &b->bstartT}, {b->d_cstart, &b->cstart},
                                                             {b->d_bstartZ, &b->bstartZ}, {b->d_bstartF, &b->bstartF}};
  for (const auto& st : starts)
    if (hipMemcpyAsync(st.first, st.second->data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, b->stream) !=
        hipSuccess) {
      snprintf(err, errlen, "hipMemcpyAsync of block starts failed");
      amcd_destroy(b);
      return -1;
    }
  if (push_inst(b) || hipStreamSynchronize(b->stream) != hipSuccess) {
    snprintf(err, errlen, "%s", g_dev_err.c_str());
    amcd_destroy(b);
    return -1;
  }
  *out = b;
  return 0;
}

void amcd_destroy(amcd_batch* b) {  // best effort: errors while tearing down are not reported
  if (!b) return;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  for (void* q : b->allocs) (void)hipFree(q);
  for (int q = 0; q < 16; ++q)
    if (b->ev[q]) (void)hipEventDestroy(b->ev[q]);
  if (b->h_steps) (void)hipHostFree(b->h_steps);
  if (b->h_outs) (void)hipHostFree(b->h_outs);
  for (auto& g : b->gstep)
    if (g) (void)hipGraphExecDestroy(g);
  if (b->gfin) (void)hipGraphExecDestroy(b->gfin);
  if (b->h_pool) (void)hipHostFree(b->h_pool);
  if (b->d_pool) (void)hipFree(b->d_pool);
  if (b->d_mark) (void)hipFree(b->d_mark);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

void amcd_set_timing(amcd_batch* b, int on) { b->timing = on != 0; }

int amcd_upload(amcd_batch* b, int i, const int* gid, const int* vstate, const double* ext, const double* cen,
                const int* bj) {
  if (i < 0 || i >= b->n) return -1;
  Inst& d = b->h[i];
  HIPT(hipStreamSynchronize(b->stream));
  size_t N = d.N;
  std::vector<uint8_t> tmp(N);
  if (vstate) {
    for (size_t v = 0; v < N; ++v) tmp[v] = (uint8_t)(vstate[v] & 3);
    HIPT(hipMemcpy(d.vs, tmp.data(), N, hipMemcpyHostToDevice));
    // (on the batch's stream: a fill on the null stream need not be done when it returns, and the batch's
    // stream does not wait for it)
    HIPT(hipMemsetAsync(d.zliq, 0xff, (size_t)d.p.nz * 8, b->stream));
    HIPT(hipMemsetAsync(&d.ls->tvalid, 0, sizeof(int), b->stream));
    hipLaunchKernelGGL(k_rehot, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, b->stream, d.vs, d.T, d.N, d.p.tL);
    HIPT(hipGetLastError());
    HIPT(hipStreamSynchronize(b->stream));
  }
  if (bj) {
    for (size_t v = 0; v < N; ++v) tmp[v] = (uint8_t)(bj[v] ? 1 : 0);
    HIPT(hipMemcpy(d.bj, tmp.data(), N, hipMemcpyHostToDevice));
  }
  if (gid) HIPT(hipMemcpy(d.gid, gid, N * 4, hipMemcpyHostToDevice));
  if (ext) HIPT(hipMemcpy(d.ext, ext, N * 8, hipMemcpyHostToDevice));
  if (cen) {
    std::vector<double> c(N);
    double* dst[3] = {d.cx, d.cy, d.cz};
    for (int q = 0; q < 3; ++q) {
      for (size_t v = 0; v < N; ++v) c[v] = cen[3 * v + q];
      HIPT(hipMemcpy(dst[q], c.data(), N * 8, hipMemcpyHostToDevice));
    }
  }
  return 0;
}

int amcd_download(amcd_batch* b, int i, int* gid, int* vstate, double* ext, double* cen, int* bj, double* T) {
  if (i < 0 || i >= b->n) return -1;
  Inst& d = b->h[i];
  HIPT(hipStreamSynchronize(b->stream));
  size_t N = d.N;
  std::vector<uint8_t> tmp(N);
  if (vstate) {
    HIPT(hipMemcpy(tmp.data(), d.vs, N, hipMemcpyDeviceToHost));
    for (size_t v = 0; v < N; ++v) vstate[v] = tmp[v] & 3;
  }
  if (bj) {
    HIPT(hipMemcpy(tmp.data(), d.bj, N, hipMemcpyDeviceToHost));
    for (size_t v = 0; v < N; ++v) bj[v] = tmp[v];
  }
  if (gid) HIPT(hipMemcpy(gid, d.gid, N * 4, hipMemcpyDeviceToHost));
  if (ext) HIPT(hipMemcpy(ext, d.ext, N * 8, hipMemcpyDeviceToHost));
  if (T) HIPT(hipMemcpy(T, d.T, N * 8, hipMemcpyDeviceToHost));
  if (cen) {
    std::vector<double> c(N);
    double* src[3] = {d.cx, d.cy, d.cz};
    for (int q = 0; q < 3; ++q) {
      HIPT(hipMemcpy(c.data(), src[q], N * 8, hipMemcpyDeviceToHost));
      for (size_t v = 0; v < N; ++v) cen[3 * v + q] = c[v];
    }
  }
  return 0;
}

static int ensure_grains(amcd_batch* b, Inst& d, int need) {
  if (need <= d.gcap) return 0;
  int ncap = std::max(need, std::max(1024, d.gcap * 2));
  double* nr = nullptr;
  HIPT(hipMalloc(&nr, sizeof(double) * 9 * (size_t)ncap));
  if (d.rot) {
    HIPT(hipMemcpyAsync(nr, d.rot, sizeof(double) * 9 * (size_t)d.gcap, hipMemcpyDeviceToDevice, b->stream));
    HIPT(hipStreamSynchronize(b->stream));
    for (auto& q : b->allocs)
      if (q == d.rot) q = nr;
    HIPT(hipFree(d.rot));
  } else {
    b->allocs.push_back(nr);
  }
  d.rot = nr;
  d.gcap = ncap;
  return push_inst(b);
}

int amcd_set_rot(amcd_batch* b, int i, const double* rot9, int ngrain) {
  Inst& d = b->h[i];
  if (ensure_grains(b, d, ngrain + 256)) return -1;
  if (ngrain > 0)
    HIPT(hipMemcpyAsync(d.rot, rot9, sizeof(double) * 9 * (size_t)ngrain, hipMemcpyHostToDevice, b->stream));
  HIPT(hipStreamSynchronize(b->stream));
  return 0;
}

int amcd_get_rot(amcd_batch* b, int i, double* rot9, int ngrain) {
  Inst& d = b->h[i];
  if (ngrain > d.gcap) return -1;
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipMemcpy(rot9, d.rot, sizeof(double) * 9 * (size_t)ngrain, hipMemcpyDeviceToHost));
  return 0;
}

// Every instance's pool lives in one device region behind one pinned staging area, from which the
// step's first kernel takes it.  A pool larger than its instance's capacity
// re-lays the region out for every instance (capacities at least double).
int amcd_set_pools(amcd_batch* b, const double* const* rot9, const int* n) {
  bool grow = b->d_pool == nullptr;
  for (int i = 0; i < b->n; ++i) grow = grow || n[i] > b->h[i].poolcap;
  HIPT(hipStreamSynchronize(b->stream));  // no launch reads the staging area or the old pools any more
  b->staged = false;
  if (grow) {
    for (auto& g : b->gstep) {  // (captured with the old region)
      if (g) (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
    std::vector<size_t> off(b->n + 1, 0);
    for (int i = 0; i < b->n; ++i) {
      Inst& d = b->h[i];
      int cap = std::max(64, d.poolcap);
      while (cap < n[i]) cap *= 2;
      d.poolcap = cap;
      off[i + 1] = off[i] + (size_t)cap;
    }
    double *dp = nullptr, *hp = nullptr;
    HIPT(hipMalloc(&dp, sizeof(double) * 9 * off[b->n]));
    if (hipHostMalloc((void**)&hp, sizeof(double) * 9 * off[b->n], 0) != hipSuccess) {
      (void)hipFree(dp);
      g_dev_err = "hipHostMalloc of the pool staging area failed";
      return -1;
    }
    if (b->d_pool) HIPT(hipFree(b->d_pool));
    if (b->h_pool) HIPT(hipHostFree(b->h_pool));
    b->d_pool = dp;
    b->h_pool = hp;
    b->pool_off = off;
    for (int i = 0; i < b->n; ++i) b->h[i].pool = dp + 9 * off[i];
    if (push_inst(b)) return -1;
  }
  for (int i = 0; i < b->n; ++i)
    if (n[i] > 0 && rot9[i]) memcpy(b->h_pool + 9 * b->pool_off[i], rot9[i], sizeof(double) * 9 * (size_t)n[i]);
  return 0;
}

int amcd_set_pool(amcd_batch* b, int i, const double* rot9, int n) {
  if (i < 0 || i >= b->n) return -1;
  std::vector<const double*> r(b->n, nullptr);
  std::vector<int> c(b->n, 0);
  r[i] = rot9;
  c[i] = n;
  return amcd_set_pools(b, r.data(), c.data());
}

// grain-table capacity for the coming step: current grains + pool size
int amcd_reserve_grains(amcd_batch* b, int i, int need) { return ensure_grains(b, b->h[i], need); }

static int put_steps(amcd_batch* b, const amcd_step* steps) {
  if (b->staged) {  // (a temperature whose output records nobody has read)
    HIPT(hipStreamSynchronize(b->stream));
    b->staged = false;
  }
  memcpy(b->h_steps, steps, sizeof(amcd_step) * b->n);
  return 0;
}
// the staged step records and pools to the device, with fresh output records when `clear`
static int launch_step_in(amcd_batch* b, bool clear) {
  static_assert(sizeof(amcd_step) % 4 == 0 && sizeof(amcd_out) % 4 == 0, "records copied as words");
  const int ns = (int)(sizeof(amcd_step) / 4) * b->n, no = clear ? (int)(sizeof(amcd_out) / 4) * b->n : 0;
  const int nrec = (std::max(ns, no) + 255) / 256;
  b->staged = true;
  hipLaunchKernelGGL(k_step_in, dim3(nrec + (b->d_pool ? b->n : 0)), dim3(256), 0, b->stream, (unsigned*)b->d_steps,
                     (const unsigned*)b->h_steps, ns, (unsigned*)b->d_outs, no, b->d_inst, nrec, b->d_pool, b->h_pool);
  HIPT(hipGetLastError());
  return 0;
}
static int launch_step_out(amcd_batch* b) {
  const int no = (int)(sizeof(amcd_out) / 4) * b->n;
  hipLaunchKernelGGL(k_step_out, dim3((no + 255) / 256), dim3(256), 0, b->stream, (unsigned*)b->h_outs,
                     (const unsigned*)b->d_outs, no);
  HIPT(hipGetLastError());
  return 0;
}

static void tmark(amcd_batch* b, int q) {
  if (b->timing) (void)hipEventRecord(b->ev[q], b->stream);  // timing only
}

static int run_temperature(amcd_batch* b, int setliquid) {
  int nb = b->bstartT[b->n];
  hipLaunchKernelGGL(k_temperature, dim3(nb), dim3(GB), 0, b->stream, b->d_inst, b->d_bstartT, b->n, b->d_steps,
                     b->d_outs, setliquid);
  HIPT(hipGetLastError());
  return 0;
}
static int commit_temperature(amcd_batch* b, int valid) {  // (in the fused step the scan does it)
  hipLaunchKernelGGL(k_temp_commit, dim3(b->n), dim3(64), 0, b->stream, b->d_inst, b->d_steps, valid);
  HIPT(hipGetLastError());
  return 0;
}
// the device T no longer follows the analytic layout (upload, new layer, EASM)
static int invalidate_T(amcd_batch* b, int i) {
  HIPT(hipMemsetAsync(&b->h[i].ls->tvalid, 0, sizeof(int), b->stream));
  return 0;
}

int amcd_temperature(amcd_batch* b, const amcd_step* steps) {
  if (put_steps(b, steps) || launch_step_in(b, true) || run_temperature(b, 0)) return -1;
  return commit_temperature(b, 1);
}

static int read_outs(amcd_batch* b, amcd_out* outs);
int amcd_easm(amcd_batch* b, const amcd_step* steps, double Q, double layerT, amcd_out* outs,
              unsigned long long* n_evals) {
  if (put_steps(b, steps) || launch_step_in(b, true)) return -1;
  unsigned long long* dn = b->d_evals;
  HIPT(hipMemsetAsync(dn, 0, sizeof(unsigned long long), b->stream));
  tmark(b, 0);
  hipLaunchKernelGGL(k_easm, dim3(b->bstartG[b->n]), dim3(GB), 0, b->stream, b->d_inst, b->d_bstartG, b->n,
                     b->d_steps, b->d_outs, Q, layerT, dn);
  if (commit_temperature(b, 0)) return -1;
  tmark(b, 1);
  unsigned long long hn = 0;
  HIPT(hipMemcpyAsync(&hn, dn, sizeof(hn), hipMemcpyDeviceToHost, b->stream));
  if (read_outs(b, outs)) return -1;
  if (b->timing) {
    float ms = 0;
    (void)hipEventElapsedTime(&ms, b->ev[0], b->ev[1]);
    b->last_ms[0] = ms;
  }
  if (n_evals) *n_evals = hn;
  return 0;
}

static int launch_update(amcd_batch* b, bool fused_temperature) {
  const int n = b->n;
  tmark(b, 0);
  if (fused_temperature) {
    if (run_temperature(b, 1)) return -1;
  } else {
    hipLaunchKernelGGL(k_setliquid, dim3(b->bstartG[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_bstartG, n,
                       b->d_steps);
  }
  tmark(b, 1);
  hipLaunchKernelGGL(k_solid_to_mushy, dim3(b->bstartS[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_bstartS, n,
                     b->d_steps);
  tmark(b, 2);
  hipLaunchKernelGGL(k_active_flags, dim3(b->bstartF[n]), dim3(256), 0, b->stream, b->d_inst, b->d_bstartF, n,
                     b->d_steps);
  hipLaunchKernelGGL(k_scan, dim3(b->cstart[n]), dim3(1024), 0, b->stream, b->d_inst, b->d_cstart, n, b->d_steps,
                     b->d_outs, fused_temperature ? 1 : 0);
  hipLaunchKernelGGL(k_compact, dim3(b->bstartF[n]), dim3(256), 0, b->stream, b->d_inst, b->d_bstartF, n,
                     b->d_steps);
  tmark(b, 3);
  HIPT(hipGetLastError());
  return 0;
}

// Capacity tiers of the capture loop: threads per workgroup x growing cells per thread.  The
// last but one keeps the cells in memory (no limit below the active capacity); the last one is
// that with the liveness read from the states (interfaces beyond AMCD_DEAD_BITS).
static const int kNTiers = 5;
static const int kTierCap[kNTiers] = {256 * 4, 512 * 4, 512 * 8, 512 * 16, 0x7fffffff};
extern "C++" template <int NT, int K, bool GD = false>
static int launch_loop(amcd_batch* b) {
  hipLaunchKernelGGL((k_event_loop<NT, K, GD>), dim3(b->n), dim3(NT), 0, b->stream, b->d_inst, b->d_steps, b->d_outs);
  HIPT(hipGetLastError());
  return 0;
}
static int launch_event_loop_wide(amcd_batch* b) { return launch_loop<512, 0, true>(b); }
static int launch_event_loop(amcd_batch* b) {
  switch (b->tier) {
    case 0: return launch_loop<256, 4>(b);
    case 1: return launch_loop<512, 4>(b);
    case 2: return launch_loop<512, 8>(b);
    case 3: return launch_loop<512, 16>(b);
    case 4: return launch_loop<512, 0>(b);
    default: return launch_event_loop_wide(b);
  }
}

static int wait_outs(amcd_batch* b, amcd_out* outs) {
  HIPT(hipStreamSynchronize(b->stream));
  b->staged = false;
  memcpy(outs, b->h_outs, sizeof(amcd_out) * b->n);
  return 0;
}
static int read_outs(amcd_batch* b, amcd_out* outs) { return launch_step_out(b) || wait_outs(b, outs); }

// The active-cell block lists, sized by the capacities up to kActiveBlocks (idle workgroups exit, so no
// host round trip is needed mid-step), uploaded when a capacity has changed.
static int prep_active(amcd_batch* b) {
  const int n = b->n;
  b->astart[0] = 0;
  for (int i = 0; i < n; ++i) b->astart[i + 1] = b->astart[i] + std::min((b->h[i].acap + GB - 1) / GB, kActiveBlocks);
  b->lstart[0] = 0;
  for (int i = 0; i < n; ++i) b->lstart[i + 1] = b->lstart[i] + std::min(b->list_cap, (b->h[i].acap + 3) / 4);
  if (b->astart != b->astart_up) {
    HIPT(hipMemcpyAsync(b->d_astart, b->astart.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, b->stream));
    b->astart_up = b->astart;
  }
  if (b->lstart != b->lstart_up) {
    HIPT(hipMemcpyAsync(b->d_lstart, b->lstart.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, b->stream));
    b->lstart_up = b->lstart;
  }
  // the vectors stay unchanged until the next capacity change, so the copies may read them late
  return 0;
}
static int autotune_lists(amcd_batch* b);
static int launch_active_kernels(amcd_batch* b) {
  const int n = b->n;
  hipLaunchKernelGGL(k_active_setup, dim3(b->astart[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_astart, n,
                     b->d_outs);
  hipLaunchKernelGGL(k_grow_lists, dim3(b->lstart[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_lstart, n);
  if (b->tune_pending && !b->timing) {  // stage by stage only: the graphs never tune
    b->tune_pending = false;
    if (autotune_lists(b)) return -1;
  }
  tmark(b, 4);
  if (launch_event_loop(b)) return -1;
  tmark(b, 5);
  HIPT(hipGetLastError());
  return 0;
}
static int launch_active(amcd_batch* b) { return prep_active(b) || launch_active_kernels(b); }

static int launch_finish(amcd_batch* b) {
  const int n = b->n;
  hipLaunchKernelGGL(k_finish, dim3(b->astart[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_astart, n, b->d_outs);
  tmark(b, 6);
  HIPT(hipGetLastError());
  return 0;
}

static void collect_timing(amcd_batch* b) {
  if (!b->timing) return;
  (void)hipEventSynchronize(b->ev[6]);
  for (int q = 0; q < 6; ++q) {
    float ms = 0;
    (void)hipEventElapsedTime(&ms, b->ev[q], b->ev[q + 1]);
    b->last_ms[q] = ms;
  }
}

int amcd_read_outs(amcd_batch* b, amcd_out* outs) { return read_outs(b, outs); }

// capture-loop phase timers (zeros unless built with -DAMCD_PHASE_PROFILE); reading resets them
int amcd_phase_profile(unsigned long long* out32) {
#ifdef AMCD_PHASE_PROFILE
  HIPT(hipDeviceSynchronize());
  HIPT(hipMemcpyFromSymbol(out32, HIP_SYMBOL(g_phase), sizeof(unsigned long long) * 32));
  unsigned long long z[32] = {0};
  HIPT(hipMemcpyToSymbol(HIP_SYMBOL(g_phase), z, sizeof(z)));
#else
  for (int q = 0; q < 32; ++q) out32[q] = 0;
#endif
  return 0;
}

int amcd_last_timings(amcd_batch* b, double* ms, int n) {
  for (int q = 0; q < n && q < 6; ++q) ms[q] = b->last_ms[q];
  return 0;
}

// growth of the active capacity after an overflow; the step is then repeated (the
// stages before the compaction are idempotent for the same temperature field)
static int grow_active(amcd_batch* b, const amcd_out* outs) {
  bool any = false;
  for (int i = 0; i < b->n; ++i) {
    if (!outs[i].overflow) continue;
    Inst& d = b->h[i];
    int need = outs[i].n_active;
    int ncap = (int)std::min<long long>(d.N, std::max<long long>((long long)need * 3 / 2, (long long)d.acap * 2));
    // old arrays stay allocated until destroy; they are simply no longer referenced
    want_active(b, d, ncap);
    any = true;
  }
  if (any && (alloc_wanted(b) || push_inst(b))) return -1;
  return 0;
}

// An instance whose interface is larger than the LDS liveness bitmap returns from the
// launch before its loop starts (status -3); the loop then runs for it in the memory-
// resident tier with the bitmap in memory (instances already done return at once).
static int widen(amcd_batch* b, amcd_out* outs) {
  bool need = false;
  for (int i = 0; i < b->n; ++i) need = need || outs[i].status == -3;
  if (!need) return 0;
  if (launch_event_loop_wide(b) || read_outs(b, outs)) return -1;
  return 0;
}

// Relaunch (resume) the capture loop with a larger tier while some instance has more
// growing cells than the current tier holds.
static int regrow_tier(amcd_batch* b, amcd_out* outs) {
  for (;;) {
    bool need = false;
    for (int i = 0; i < b->n; ++i) need = need || outs[i].status == 2;
    if (!need) return 0;
    if (b->tier >= kNTiers - 1) {
      int worst = 0;
      for (int i = 0; i < b->n; ++i)
        if (outs[i].status == 2 && outs[i].n_slots >= outs[worst].n_slots) worst = i;
      g_dev_err = "instance " + std::to_string(worst) + ": " + std::to_string(outs[worst].n_slots) +
                  " growing cells and the memory-resident capture tier still asks for more";
      return -1;
    }
    b->tier++;
    if (launch_event_loop(b) || read_outs(b, outs)) return -1;
  }
}
// smallest tier holding 1/32 more than the largest growing list of the step just done (a
// step that outgrows it resumes in the next tier)
static void pick_tier(amcd_batch* b, const amcd_out* outs) {
  int mx = 0;
  for (int i = 0; i < b->n; ++i) mx = std::max(mx, outs[i].n_slots);
  int t = 0;
  while (t < kNTiers - 1 && kTierCap[t] < mx + mx / 32) ++t;
  b->tier = std::max(t, b->min_tier);
}

// Capture of the step's stages into an executable graph: with `step` the step records in, the
// temperature and state passes, the active-list and candidate-list passes and the capture loop of the
// current tier; otherwise the results to the grid (of the instances whose loop has finished) and the
// output records out.
static int capture_graph(amcd_batch* b, bool step, hipGraphExec_t* out) {
  hipGraph_t g = nullptr;
  HIPT(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  const int rc = step ? launch_step_in(b, true) || launch_update(b, true) || launch_active_kernels(b)
                      : launch_finish(b) || launch_step_out(b);
  const hipError_t e = hipStreamEndCapture(b->stream, &g);
  if (rc || e != hipSuccess) {
    if (g) (void)hipGraphDestroy(g);
    if (g_dev_err.empty() || e != hipSuccess) g_dev_err = std::string("step graph capture: ") + hipGetErrorString(e);
    return -1;
  }
  const hipError_t ei = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (ei != hipSuccess) {
    g_dev_err = std::string("hipGraphInstantiate: ") + hipGetErrorString(ei);
    return -1;
  }
  return 0;
}
static std::atomic<long long> g_graph_launches{0};
long long amcd_graph_launches(void) { return g_graph_launches.load(); }
// graph of the step's stages for the current tier, captured again when the block counts change
static int launch_step_graph(amcd_batch* b) {
  const int n = b->n, t = std::min(b->tier, 5);
  const long long key = ((long long)b->astart[n] << 32) | (unsigned)b->lstart[n];
  hipGraphExec_t& g = b->gstep[t];
  if (g && b->gstep_key[t] != key) {
    HIPT(hipGraphExecDestroy(g));
    g = nullptr;
  }
  if (!g) {
    if (capture_graph(b, true, &g)) return -1;
    b->gstep_key[t] = key;
  }
  b->staged = true;
  HIPT(hipGraphLaunch(g, b->stream));
  g_graph_launches++;
  return 0;
}
static int launch_finish_graph(amcd_batch* b) {
  const long long key = b->astart[b->n];
  if (b->gfin && b->gfin_key != key) {
    HIPT(hipGraphExecDestroy(b->gfin));
    b->gfin = nullptr;
  }
  if (!b->gfin) {
    if (capture_graph(b, false, &b->gfin)) return -1;
    b->gfin_key = key;
  }
  HIPT(hipGraphLaunch(b->gfin, b->stream));
  g_graph_launches++;
  return 0;
}

// Candidate chunkings of the candidate-list pass (blocks per instance).  The pass rebuilds every
// live slot's list from inputs it does not write, so running it again right after itself, before
// the capture loop, changes nothing; each candidate is timed three times after a warm-up on the
// step's interface.  The device's block list is left with the last candidate's and uploaded
// again for the chosen one at the next step.
static const int kListCaps[5] = {256, 512, 1024, 2048, 4096};
static int autotune_lists(amcd_batch* b) {
  const int n = b->n;
  std::vector<int> ls(n + 1);
  float best = 1e30f;
  int pick = b->list_cap;
  for (int c = 0; c < 5; ++c) {
    ls[0] = 0;
    for (int i = 0; i < n; ++i) ls[i + 1] = ls[i] + std::min(kListCaps[c], (b->h[i].acap + 3) / 4);
    HIPT(hipMemcpyAsync(b->d_lstart, ls.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, b->stream));
    for (int r = 0; r < 4; ++r) {
      if (r == 1) HIPT(hipEventRecord(b->ev[14], b->stream));
      hipLaunchKernelGGL(k_clear_npre, dim3(n), dim3(64), 0, b->stream, b->d_inst);
      hipLaunchKernelGGL(k_grow_lists, dim3(ls[n]), dim3(GB), 0, b->stream, b->d_inst, b->d_lstart, n);
    }
    HIPT(hipEventRecord(b->ev[15], b->stream));
    HIPT(hipGetLastError());
    HIPT(hipEventSynchronize(b->ev[15]));
    float ms = 0;
    HIPT(hipEventElapsedTime(&ms, b->ev[14], b->ev[15]));
    b->tune_ms[c] = ms / 3;
    if (ms < best) {
      best = ms;
      pick = kListCaps[c];
    }
  }
  b->list_cap = pick;
  b->tuned = true;
  b->lstart_up.clear();  // the device's list now holds the last candidate's: upload at the next step
  return 0;
}
// after a finished step: the next step tunes once the largest growing list has reached 256
// cells, and again each time it has doubled since
static int maybe_autotune(amcd_batch* b, const amcd_out* outs) {
  if (!b->autotune) return 0;
  int mx = 0;
  for (int i = 0; i < b->n; ++i) mx = std::max(mx, outs[i].n_slots);
  if (mx < 256 || mx < 2 * b->tuned_at) return 0;
  b->tuned_at = mx;
  b->n_tunings++;
  b->tune_pending = true;
  return 0;
}
int amcd_tuning(amcd_batch* b, int* list_cap, int* n_tunings, int* cells, float* ms, int nms) {
  if (list_cap) *list_cap = b->tuned ? b->list_cap : 0;
  if (n_tunings) *n_tunings = b->n_tunings;
  if (cells) *cells = b->tuned_at;
  for (int c = 0; c < nms && c < 5; ++c) ms[c] = b->tune_ms[c];
  return b->tuned ? 1 : 0;
}

static bool all_finished(const amcd_batch* b, const amcd_out* outs) {
  for (int i = 0; i < b->n; ++i)
    if (outs[i].status != 0) return false;
  return true;
}
// The step, as graphs (the driver's fused form) or stage by stage: per-stage timing needs events
// between the stages, a tuning step runs the list pass several times, and the seam form keeps the
// output records its temperature call wrote.  One synchronisation: the results of instances whose
// loop has finished are in the grid when the output records are read.  Suspensions (pool refill,
// larger tier, wide bitmap) take further launches, and the finishing pass then runs again (the same
// values, for the instances that had finished).
static int update_common(amcd_batch* b, const amcd_step* steps, amcd_out* outs, bool fused) {
  const bool graph = b->graphs && !b->timing && fused && !b->tune_pending;
  if (put_steps(b, steps)) return -1;
  for (int attempt = 0; attempt < 8; ++attempt) {
    if (graph) {
      if (prep_active(b) || launch_step_graph(b) || launch_finish_graph(b) || wait_outs(b, outs)) return -1;
    } else {
      // A retry repeats the step's stages with the same temperature source: the fused form
      // re-evaluates the same laser (idempotent), the seam form keeps the caller's field and
      // re-applies SetLiquid3 to it (idempotent for the same T).
      if (launch_step_in(b, fused || attempt > 0) || launch_update(b, fused) || launch_active(b) || launch_finish(b) ||
          read_outs(b, outs))
        return -1;
    }
    bool ovf = false;
    for (int i = 0; i < b->n; ++i) ovf = ovf || outs[i].overflow;
    if (!ovf) break;
    if (grow_active(b, outs)) return -1;
  }
  const bool finished = all_finished(b, outs);
  if (!finished) {
    if (widen(b, outs) || regrow_tier(b, outs)) return -1;
    for (int i = 0; i < b->n; ++i)
      if (outs[i].status == 1) return 0;  // (the caller refills the pool and resumes)
    if (launch_finish(b)) return -1;
    HIPT(hipStreamSynchronize(b->stream));
  }
  collect_timing(b);
  pick_tier(b, outs);
  return maybe_autotune(b, outs);
}

int amcd_update_voxels(amcd_batch* b, const amcd_step* steps, amcd_out* outs) {
  return update_common(b, steps, outs, false);
}

int amcd_step_fused(amcd_batch* b, const amcd_step* steps, amcd_out* outs) {
  return update_common(b, steps, outs, true);
}

int amcd_resume(amcd_batch* b, const amcd_step* steps, amcd_out* outs) {
  if (put_steps(b, steps) || launch_step_in(b, false)) return -1;
  if (launch_event_loop(b)) return -1;
  if (read_outs(b, outs)) return -1;
  if (widen(b, outs) || regrow_tier(b, outs)) return -1;
  bool pend = false;
  for (int i = 0; i < b->n; ++i) pend = pend || outs[i].status == 1;
  if (!pend) {
    if (launch_finish(b)) return -1;
    HIPT(hipStreamSynchronize(b->stream));
  }
  return 0;
}

// VoxelsCA::SetBuild (S/VoxelsCA.C:76-115) as two rounds of grain-set membership: mark the
// grains of the flagged voxels (BuildjID == 1, then Build == 1), then flag every voxel of a
// marked grain as built.  Grain ids lie in 1..ngrain.
__global__ void k_build_mark(const int* __restrict__ gid, const uint8_t* __restrict__ flag, int N, int ngrain,
                             uint8_t* __restrict__ mark) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= N || flag[v] != 1) return;
  const int g = gid[v];
  if (g > 0 && g <= ngrain) mark[g] = 1;
}
__global__ void k_build_apply(const int* __restrict__ gid, int N, int ngrain, const uint8_t* __restrict__ mark,
                              uint8_t* __restrict__ build) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= N) return;
  const int g = gid[v];
  if (g > 0 && g <= ngrain && mark[g]) build[v] = 1;
}
int amcd_set_build(amcd_batch* b, int i, int ngrain) {
  const Inst& d = b->h[i];
  if (b->mark_cap < (size_t)ngrain + 1) {
    HIPT(hipStreamSynchronize(b->stream));
    if (b->d_mark) HIPT(hipFree(b->d_mark));
    b->d_mark = nullptr;
    b->mark_cap = 0;
    const size_t cap = std::max<size_t>(4096, 2 * ((size_t)ngrain + 1));
    HIPT(hipMalloc(&b->d_mark, cap));
    b->mark_cap = cap;
  }
  uint8_t* mk = b->d_mark;
  const dim3 grid((d.N + 255) / 256);
  for (int round = 0; round < 2; ++round) {
    HIPT(hipMemsetAsync(mk, 0, (size_t)ngrain + 1, b->stream));
    hipLaunchKernelGGL(k_build_mark, grid, dim3(256), 0, b->stream, d.gid, round == 0 ? d.bj : d.build, d.N,
                       ngrain, mk);
    hipLaunchKernelGGL(k_build_apply, grid, dim3(256), 0, b->stream, d.gid, d.N, ngrain, mk, d.build);
  }
  HIPT(hipGetLastError());
  return 0;
}
// Build = 1 on the first n_built voxels (the base plate, S/VoxelsCA.C:157-160), 0 elsewhere
int amcd_build_init(amcd_batch* b, int i, long long n_built) {
  const Inst& d = b->h[i];
  HIPT(hipMemsetAsync(d.build, 0, (size_t)d.N, b->stream));
  if (n_built > 0) HIPT(hipMemsetAsync(d.build, 1, (size_t)std::min<long long>(n_built, d.N), b->stream));
  HIPT(hipStreamSynchronize(b->stream));
  return 0;
}
int amcd_get_build(amcd_batch* b, int i, int* out) {
  const Inst& d = b->h[i];
  std::vector<uint8_t> tmp((size_t)d.N);
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipMemcpy(tmp.data(), d.build, (size_t)d.N, hipMemcpyDeviceToHost));
  for (size_t v = 0; v < tmp.size(); ++v) out[v] = tmp[v];
  return 0;
}

int amcd_grain_presence(amcd_batch* b, int i, int ngrain, int* present) {
  Inst& d = b->h[i];
  int* dp = nullptr;
  HIPT(hipMalloc(&dp, sizeof(int) * (size_t)(ngrain + 1)));
  HIPT(hipMemsetAsync(dp, 0, sizeof(int) * (size_t)(ngrain + 1), b->stream));
  hipLaunchKernelGGL(k_grain_presence, dim3((d.N + 255) / 256), dim3(256), 0, b->stream, d.gid, d.N, dp, ngrain);
  HIPT(hipMemcpyAsync(present, dp, sizeof(int) * (size_t)ngrain, hipMemcpyDeviceToHost, b->stream));
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipFree(dp));
  return 0;
}

int amcd_remap_grains(amcd_batch* b, int i, const int* remap, int ngrain) {
  Inst& d = b->h[i];
  int* dr = nullptr;
  HIPT(hipMalloc(&dr, sizeof(int) * (size_t)(ngrain + 1)));
  HIPT(hipMemcpyAsync(dr, remap, sizeof(int) * (size_t)ngrain, hipMemcpyHostToDevice, b->stream));
  hipLaunchKernelGGL(k_remap, dim3((d.N + 255) / 256), dim3(256), 0, b->stream, d.gid, d.N, dr, ngrain);
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipFree(dr));
  return 0;
}

// workgroups of k_voronoi: one to a brick, up to a number whose threads a launch can count (a domain one voxel
// wide has as many bricks as an eighth or a quarter of its voxels)
static unsigned voronoi_blocks(int nx, int ny, int nz) {
  const long long bricks = (long long)((nx + 7) / 8) * ((ny + 7) / 8) * ((nz + 3) / 4);
  return (unsigned)std::min<long long>(bricks, 1 << 20);
}
int amcd_init_plate(amcd_batch* b, int i, int nzh, const double* xs, int ng) {
  if (i < 0 || i >= b->n || ng <= 0 || nzh <= 0) return -1;
  Inst& d = b->h[i];
  if (nzh > d.p.nz) nzh = d.p.nz;
  double* dx = nullptr;
  HIPT(hipMalloc(&dx, sizeof(double) * 3 * (size_t)ng));
  HIPT(hipMemcpyAsync(dx, xs, sizeof(double) * 3 * (size_t)ng, hipMemcpyHostToDevice, b->stream));
  hipLaunchKernelGGL(k_voronoi<false>, dim3(voronoi_blocks(d.p.nx, d.p.ny, nzh)), dim3(VOR_B), 0, b->stream, b->d_inst, i, 0, nzh, dx,
                     ng, nullptr, nullptr);
  HIPT(hipGetLastError());
  HIPT(hipMemsetAsync(d.zliq, 0xff, (size_t)d.p.nz * 8, b->stream));
  if (invalidate_T(b, i)) return -1;
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipFree(dx));
  return 0;
}

int amcd_add_layer(amcd_batch* b, int i, int iz1, int ilaserLoc, int gbase, const double* xs, int ng, int* n_used) {
  if (i < 0 || i >= b->n || ng <= 0) return -1;
  Inst& d = b->h[i];
  const int nl = ilaserLoc - iz1;
  const size_t cnt = (size_t)d.nxy * (size_t)(nl > 0 ? nl : 0);
  double* dx = nullptr;
  int *lab = nullptr, *used = nullptr;
  HIPT(hipMalloc(&dx, sizeof(double) * 3 * (size_t)ng));
  HIPT(hipMalloc(&lab, sizeof(int) * (cnt + 1)));
  HIPT(hipMalloc(&used, sizeof(int) * (2 * (size_t)ng + 1)));  // used[ng], rank[ng], total
  int* rank = used + ng;
  int* tot = used + 2 * ng;
  HIPT(hipMemcpyAsync(dx, xs, sizeof(double) * 3 * (size_t)ng, hipMemcpyHostToDevice, b->stream));
  HIPT(hipMemsetAsync(used, 0, sizeof(int) * (2 * (size_t)ng + 1), b->stream));
  if (cnt)
    hipLaunchKernelGGL(k_voronoi<true>, dim3(voronoi_blocks(d.p.nx, d.p.ny, nl)), dim3(VOR_B), 0, b->stream, b->d_inst, i, iz1, nl, dx,
                       ng, lab, used);
  hipLaunchKernelGGL(k_site_rank, dim3(1), dim3(1024), 0, b->stream, used, ng, rank, tot);
  hipLaunchKernelGGL(k_write_layer, dim3((d.N + 255) / 256), dim3(256), 0, b->stream, b->d_inst, i, iz1, ilaserLoc,
                     gbase, lab, rank);
  HIPT(hipGetLastError());
  HIPT(hipMemsetAsync(d.zliq, 0xff, (size_t)d.p.nz * 8, b->stream));
  if (invalidate_T(b, i)) return -1;
  HIPT(hipMemcpyAsync(n_used, tot, sizeof(int), hipMemcpyDeviceToHost, b->stream));
  HIPT(hipStreamSynchronize(b->stream));
  HIPT(hipFree(dx));
  HIPT(hipFree(lab));
  HIPT(hipFree(used));
  return 0;
}

// pow(x, y) rounded to nearest, the host build of the device routine (velocity table)
double amcd_host_pow(double x, double y) { return amc_pow_cr(x, y); }
int amcd_host_pow_n(const double* x, const double* y, int n, double* out) {
  for (int i = 0; i < n; ++i) out[i] = amc_pow_cr(x[i], y[i]);
  return 0;
}

// the clock span of the window after one that took `bins` of the histogram in `mode` (for tests)
double amcd_window_span(double span, int bins, int mode, double DelT, int cells) {
  return span < 0.0 ? first_span(DelT, cells) : next_span(span, bins, mode, DelT, cells);
}
// the step back that a cell allows (for tests)
float amcd_step_back(double e, double v) { return step_back(e, v); }
// device memory that an active-list capacity takes (for tests)
size_t amcd_active_bytes(int acap) {
  amcd_batch b;
  Inst d = {};
  want_active(&b, d, acap);
  size_t total = 0;
  for (const auto& w : b.wanted) total += w.second;
  return total;
}

// the capture shape factor evaluated by the host build of the device math
int amcd_host_shape_factor(const double* dnx, int n, double* out) {
  for (int i = 0; i < n; ++i) out[i] = amc_shape_factor(dnx[3 * i], dnx[3 * i + 1], dnx[3 * i + 2]);
  return 0;
}

// engine stream of libstdc++'s uniform_real_distribution<double>(0,1) over
// minstd_rand0(seed), as the device computes it (for known-answer tests)
int amcd_uniform_stream(unsigned long long seed, int n, double* out) {
  unsigned int x = lcg_seed(seed);
  for (int q = 0; q < n; ++q) {
    unsigned int x1 = lcg_next(x), x2 = lcg_next(x1);
    x = x2;
    out[q] = canonical(x1, x2);
  }
  return 0;
}
// the same stream from jump-ahead positions (the ruq path of k_compact)
int amcd_uniform_jump(unsigned long long seed, int n, double* out) {
  unsigned int x0 = lcg_seed(seed);
  for (int a = 0; a < n; ++a) {
    unsigned int x1 = mod_m((unsigned long long)x0 * lcg_pow(2ull * a + 1));
    out[a] = canonical(x1, lcg_next(x1));
  }
  return 0;
}

}  // extern "C"
