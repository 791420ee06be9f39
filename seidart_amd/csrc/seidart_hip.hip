// seidart_hip.hip -- MI355X (gfx950) FDTD time-stepping core of SeidarT.
//
// Hand-written HIP kernels for the four reference schemes plus the C ABI
// declared in include/seidart_hip.h.  One source, templated on the
// arithmetic type T (double or float).  The scheme of every kernel is the
// legacy Fortran loop it cites; the numerical conventions (which psi array
// decays with which profile, which coefficient average feeds which stress)
// are kept exactly, including the legacy's shared psi arrays.
//
// Data layout in HBM (all x fastest, padded grid, one plane per shot):
//   fields        nx*nz (2-D) or nx*ny*nz (2.5-D), precision T
//   coefficients  nx*nz per model, shared by every shot on that model
//   psi           slab storage: x-axis memory variables only on the
//                 i < lx / i >= nx-lx columns, z-axis ones only on the
//                 j < lz / j >= nz-lz rows (likewise y in 2.5-D), so the
//                 interior carries no C-PML state at all.
//   traces        [it][comp][rec] per shot
//
// Execution: the 2-D kinds take several time steps per launch on regions
// (k_el2_multi, k_em2_multi), or one or two with the walking kernels (short
// runs, and launch shapes that a caller sets), and write their receiver
// samples themselves.  A 2.5-D step is two launches (stress then velocity, or
// H then E) and a receiver gather.  Every launch goes over one work list that
// covers the shots of every model.  The walking kernels' items are ordered so
// that all shots of one tile land on the same XCD (blocks are dealt to the 8
// XCDs round-robin), which serves the model's coefficients from its L2; the
// other lists give each XCD a contiguous run of neighbouring items.  The
// adjoint kernels (2-D elastic and EM) sit after the forward kernels of their
// scheme.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/seidart_hip.h"

#ifndef SDT_NT_STORE
#define SDT_NT_STORE 0
#endif
#ifndef SDT_NT_LOAD
#define SDT_NT_LOAD 0
#endif

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                          \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess)                                                      \
      return fail(SDT_EDEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int TX = 64;  // tile width in x (one wavefront row)
constexpr int TZ = 4;   // tile height in z
constexpr int NT = TX * TZ;

// Device copies of the descriptors.
struct DModel {
  int nx, ny, nz, lx, ly, lz;
  double dx, dy, dz, dt;
  double scal[4];
  const void* coef[40];
  const void* prof[3][6];
  const void* aux;
};

struct DShot {
  int model, isrc, jsrc, ksrc;
  void* f[9];
  void* psi;
  void* g[9];     // second state buffer (ping-pong kinds)
  void* psi2;
  const void* src[3];
  int nrec;
  const int* rec;
  void* trace;
  int* blowup;
  const void* msrc[6];  // stress increments xx yy zz xy xz yz (elastic)
  // receivers by row (ELASTIC2, EM2): those on row k are rxid[rrow[k] .. rrow[k+1]),
  // each a pair (column, receiver index), columns ascending
  const int* rrow;
  const int* rxid;
};

// Adjoint-side buffers of one shot (elastic 2-D), see sdt_adj_shot.
struct DAdj {
  void* trail[2];   // forward states, slot k at trail + k * slot (two buffers)
  long slot;        // elements of one state: fields then psi
  int trail_len;    // slots available
  void* lam[2];     // adjoint state ping-pong: lambda_t in lam[t & 1]
  void* work;       // 12 scratch planes nx*nz
  const void* resid;
  double* grad;     // [12][nz][nx]
  double* gsrc;     // [nt][3]
  float* g32;       // FP32 plans: per-call staging of grad (same layout)
};

// FP32 gradient staging of one distinct grad array, flushed into it.
struct DFlush {
  double* grad;
  float* g32;
  long n;           // cells of the model
};

enum { PK = 0, PA, PB, PKH, PAH, PBH };

// Array pointers live in descriptors in device memory, so the compiler would
// treat them as generic (flat) addresses; flat loads also count against the
// LDS/scalar wait counter, which serialises every shuffle and scalar load
// with all outstanding memory traffic.  Every array access therefore goes
// through explicitly global (address space 1) pointers.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
using gcptr = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gcptr<T> cp(const void* p) {
  return (gcptr<T>)p;
}
template <typename T>
__device__ __forceinline__ gptr<T> mp(void* p) {
  return (gptr<T>)p;
}

// Read-only array through the constant address space: a wave-uniform index
// becomes a scalar load into SGPRs (only for data no kernel of the launch
// writes).
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* kp(const void* p) {
  return (const __attribute__((address_space(4))) T*)p;
}

// C-PML profile table of a model: P[axis * 6 + q] (q as in PK..PBH).
template <typename T>
struct Prof {
  const void* const* p;
  __device__ explicit Prof(const void* const* q) : p(q) {}
  __device__ gcptr<T> operator[](int q) const { return cp<T>(p[q]); }
};

// Receiver samples of step itn at row b of one shot (2-D kinds), called by
// every lane of a wavefront that owns lanes lo..hi of row b (lane l holds
// column col0 + l; a, c: the two components on each lane).  The receivers
// of the row (DShot::rrow / rxid) are taken 64 at a time, one per lane,
// which fetches its value from the lane that holds its column and writes it
// if this wavefront owns that column; trace layout [it][comp][rec].
template <typename T>
__device__ __forceinline__ void gather_row(const DShot& S, int b, int itn, int lane, int col0, int lo,
                                           int hi, T a, T c) {
  const int q0 = S.rrow[b], q1 = S.rrow[b + 1];
  const int nrec = S.nrec;
  auto tr = mp<T>(S.trace) + (long)itn * 2 * nrec;
  for (int e0 = q0; e0 < q1; e0 += 64) {
    const int e = e0 + lane;
    const bool has = e < q1;
    const int rx = has ? S.rxid[2 * e] : col0 - 1, id = has ? S.rxid[2 * e + 1] : 0;
    const int src = rx - col0;  // lane holding column rx
    const bool mine = has && src >= lo && src <= hi;
    const T va = __shfl(a, src & 63, 64), vc = __shfl(c, src & 63, 64);
    if (mine) {
      tr[id] = va;
      tr[nrec + id] = vc;
    }
  }
}

// Flag instability: |v|^2 > 1e50 or non-finite (seismicfdtd.f95:378-379).
__device__ __forceinline__ void check_blowup(double v2, int* flag, int it) {
  if (!(v2 <= 1.0e50)) atomicMin(flag, it);
}

// The work item of this block in a launch over n consecutive items, -1 for
// none (the grid is n rounded up to a multiple of 8): each XCD (blockIdx % 8)
// takes a contiguous run of them.
__device__ __forceinline__ int item8(int n) {
  const int run = (int)(gridDim.x >> 3), q = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  return q < n ? q : -1;
}

// slab offset helpers: position of column i inside the two x slabs
__device__ __forceinline__ int slab_pos(int i, int n, int l) { return i < l ? i : i - n + 2 * l; }
__device__ __forceinline__ bool in_slab(int i, int n, int l) { return i < l || i >= n - l; }

// ===========================================================================
// ELASTIC2: seismic2, legacy/fortran/seismicfdtd.f95:12-385
//
// One fused kernel per time step.  A wavefront owns a tile of EW columns x
// eh rows of one shot and walks it top to bottom.  Lane l holds column
// xo - 1 + l; lanes 1..EW own their column, lane 0 and lanes EW+1, EW+2 are
// halo.  At row r the wave updates the stresses of row r (both legacy stress
// loops, sharing the velocity-derivative psi as the legacy does) and then
// the velocities of row r-1, which need the new stresses of rows r-2..r.
// The previous and next velocity rows live in registers; x neighbours come
// from the neighbouring lanes (wave shuffles).  Stresses of the halo row
// above and below the tile and of the halo lanes are recomputed, so every
// tile is independent; the state therefore ping-pongs between two buffers
// (step `it` reads buffer it&1 and writes the other), which keeps halo reads
// of neighbouring tiles on old values.  Each cell's fields, psi and
// coefficients cross HBM once per step.
//
// psi slabs: x [nz][2lx]: dvx_dx dvz_dx dsxx_dx dsxz_dx (+ dvx_dx dvz_dx of
//                          the shear loop in the split variant)
//            z [2lz][nx]: dvz_dz dvx_dz dszz_dz dsxz_dz (+ dvz_dz dvx_dz)
// ===========================================================================
#ifndef SDT_EL2_ROWS
#define SDT_EL2_ROWS 32
#endif
#ifndef SDT_EL2_GRID
#define SDT_EL2_GRID 1000000
#endif
#ifndef SDT_EL2_WAVES_PER_SIMD
#define SDT_EL2_WAVES_PER_SIMD 4
#endif
#ifndef SDT_EL2_PREFETCH
#define SDT_EL2_PREFETCH 0
#endif
#ifndef SDT_EL2_WAVES_PER_BLOCK
#define SDT_EL2_WAVES_PER_BLOCK 4
#endif
constexpr int EW = 61;            // owned columns per wavefront
// Tile shape: wavefronts per block (side by side in x; a template
// parameter, 1, 2 or 4) and rows per tile (run time); sdt_plan_set_tiles
// changes both, and the autotuner picks them per plan.

// Array addressed by 32-bit element offsets: the scalar base plus a 32-bit
// vector byte offset maps onto the global load/store form with an SGPR base
// and a VGPR offset, so no per-access 64-bit address arithmetic.  Every
// array it indexes is smaller than 4 GiB (checked at plan creation).
template <typename T>
struct A32 {
  using PT = __attribute__((address_space(1))) T*;
  PT p;
  __device__ explicit A32(const void* q) : p((PT)q) {}
  __device__ __forceinline__ __attribute__((address_space(1))) T& operator[](uint32_t e) const {
    return *(PT)((__attribute__((address_space(1))) char*)p + e * (uint32_t)sizeof(T));
  }
};

template <typename T>
__device__ __forceinline__ T lane_next(T v) {  // value of lane l+1
  return __shfl_down(v, 1, 64);
}
template <typename T>
__device__ __forceinline__ T lane_prev(T v) {  // value of lane l-1
  return __shfl_up(v, 1, 64);
}

// The same by DPP wavefront shifts (a VALU move the compiler folds into the
// instruction that uses it, no LDS round trip): dpp_next gives lane l the
// value of lane l+1, dpp_prev that of lane l-1; the lane with no neighbour
// (63, resp. 0) gets 0.  Faster in the two-step kernel; in the one-step
// kernels the LDS form measured faster (they are latency-bound at lower
// occupancy, and a VALU result feeding a DPP read needs wait states).
__device__ __forceinline__ int dpp_next_i(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ int dpp_prev_i(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false); }
template <typename T>
__device__ __forceinline__ T dpp_next(T v) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, dpp_next_i(__builtin_bit_cast(int, v)));
  } else {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)dpp_next_i((int)(unsigned)b), hi = (unsigned)dpp_next_i((int)(unsigned)(b >> 32));
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  }
}
template <typename T>
__device__ __forceinline__ T dpp_prev(T v) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, dpp_prev_i(__builtin_bit_cast(int, v)));
  } else {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)dpp_prev_i((int)(unsigned)b), hi = (unsigned)dpp_prev_i((int)(unsigned)(b >> 32));
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  }
}

template <typename T, bool SPLIT, bool PML, bool R1>
__device__ __forceinline__ void el2_tile(const DModel* __restrict__ models,
                                         const DShot* __restrict__ shots, const int4 wi, const int it,
                                         const int lane, const int eh, const int par);

// Work: a block of WB wavefronts takes one item (shot, xo, zo): wave w owns
// columns xo + w*EW .. +EW-1 of rows zo .. zo+eh-1, so the block's row
// accesses are WB*EW contiguous cells of each array.  The grid is
// persistent: block b takes items b, b + gridDim.x, ...; gridDim.x is a
// multiple of 8, so item w always runs on XCD w % 8.
// SPLIT: the split C-PML variant (see SDT_SPLIT_CPML).
// R1: tiles of one row (eh == 1), whose three row steps take their loads
// all at once (a latency-bound shape: register budget of one wavefront per
// SIMD).
// The state of step it is read from buffer it & 1 (A = field/psi, B =
// field_b/psi_b) and written to the other; with prun (the first step of a
// run of two-step launches, k_el2_step2) it is read from buffer
// ((it - *prun) / 2) & 1 instead, the buffer those launches leave it in.
template <typename T, bool SPLIT, int WB, bool R1 = false>
__global__ void __launch_bounds__(64 * WB, R1 ? 1 : (sizeof(T) == 4 ? SDT_EL2_WAVES_PER_SIMD : 3))
k_el2_step(const DModel* __restrict__ models, const DShot* __restrict__ shots,
           const int4* __restrict__ work, int nitems, const int* __restrict__ base, int rel,
           int eh, const int* __restrict__ prun) {
  // wave-uniform values kept in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = __builtin_amdgcn_readfirstlane(*base + rel);
  const int par = prun ? __builtin_amdgcn_readfirstlane(((it - *prun) >> 1) & 1) : (it & 1);
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const int4 wv = work[w];
    // .w: the shot's model, so its record loads beside the shot's
    const int4 wi = make_int4(__builtin_amdgcn_readfirstlane(wv.x),
                              __builtin_amdgcn_readfirstlane(wv.y) + wave * EW,
                              __builtin_amdgcn_readfirstlane(wv.z), __builtin_amdgcn_readfirstlane(wv.w));
    if (wi.x < 0) continue;
    const DModel& M = models[wi.w];
    if (wi.y >= M.nx) continue;
    // a wave whose columns and rows (halo included) avoid every C-PML slab
    // runs the body without memory variables
    const bool interior = wi.y - 1 >= M.lx && wi.y + 62 < M.nx - M.lx && wi.z - 2 >= M.lz &&
                          wi.z + eh + 1 < M.nz - M.lz;
    if (interior)
      el2_tile<T, SPLIT, false, R1>(models, shots, wi, it, threadIdx.x & 63, eh, par);
    else
      el2_tile<T, SPLIT, true, R1>(models, shots, wi, it, threadIdx.x & 63, eh, par);
  }
}

template <typename T, bool SPLIT, bool PML, bool R1>
__device__ __forceinline__ void el2_tile(const DModel* __restrict__ models,
                                         const DShot* __restrict__ shots, const int4 wi, const int it,
                                         const int lane, const int eh, const int par) {
  // Every fused multiply-add is written out; nothing else is contracted, so
  // the interior and C-PML bodies (and every tile shape) round identically.
#pragma clang fp contract(off)
  const DShot& S = shots[wi.x];
  const DModel& M = models[wi.w];  // the shot's model (carried by the work item)
  const int nx = M.nx, nz = M.nz;
  const int xo = wi.y, zo = wi.z;
  const int i = xo - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);  // clamped column: every load stays in bounds
  const bool own = incol && lane >= 1 && lane <= EW;
  const int zend = min(zo + eh, nz);
  const bool has_rec = S.nrec > 0 && S.rrow[zend] > S.rrow[zo];  // receivers on own rows
  const long nn = (long)nx * nz;
  const A32<const T> vxi(par ? S.g[0] : S.f[0]);
  const A32<const T> vzi(par ? S.g[1] : S.f[1]);
  const A32<const T> sxxi(par ? S.g[2] : S.f[2]);
  const A32<const T> szzi(par ? S.g[3] : S.f[3]);
  const A32<const T> sxzi(par ? S.g[4] : S.f[4]);
  const A32<T> vxo(par ? S.f[0] : S.g[0]);
  const A32<T> vzo(par ? S.f[1] : S.g[1]);
  const A32<T> sxxo(par ? S.f[2] : S.g[2]);
  const A32<T> szzo(par ? S.f[3] : S.g[3]);
  const A32<T> sxzo(par ? S.f[4] : S.g[4]);
  const A32<const T> pin(par ? S.psi2 : S.psi);
  const A32<T> pout(par ? S.psi : S.psi2);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dt = T(M.dt);
  const int lx = M.lx, lz = M.lz;
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const uint32_t ZB = (SPLIT ? 6 : 4) * SX;  // first z-slab array
  const bool inx = PML && incol && in_slab(i, nx, lx);
  const int xs = inx ? slab_pos(i, nx, lx) : 0;
  const Prof<T> P(&M.prof[0][0]);
  const T ikx = P[PK][ic], ax = P[PA][ic], bx = P[PB][ic];
  const T ikxh = P[PKH][ic], axh = P[PAH][ic], bxh = P[PBH][ic];
  const auto ikz = P[12 + PK], az = P[12 + PA], bz = P[12 + PB];
  const auto ikzh = P[12 + PKH], azh = P[12 + PAH], bzh = P[12 + PBH];
  const auto brow = cp<T>(M.aux);
  const A32<const T> N11(M.coef[0]), N13(M.coef[1]), N15(M.coef[2]);
  const A32<const T> N33(M.coef[3]), N35(M.coef[4]);
  const A32<const T> S15(M.coef[5]), S35(M.coef[6]), S55(M.coef[7]);
  const A32<const T> DTX(M.coef[8]), DTZ(M.coef[9]);
  const A32<const T> OMX(M.coef[10]), OMZ(M.coef[11]);
  const bool mono = M.coef[2] != nullptr;   // c15 / c35 terms present
  const bool atten = M.coef[10] != nullptr; // gamma present
  const bool can_n = incol && lane <= EW + 1 && i <= nx - 2;          // normal stress (needs i+1)
  const bool can_s = incol && lane >= 1 && lane <= EW + 1 && i >= 1;  // shear (needs i-1)
  const bool ux = own && i >= 1, uz = own && i <= nx - 2;              // vx / vz columns
  const bool is_src_col = (i == S.isrc);
  const int ksrc = S.ksrc;
  const auto srcx = cp<T>(S.src[0]), srcz = cp<T>(S.src[2]);
  const T incx = (srcx != nullptr) ? srcx[it] : T(0);
  const T incz = (srcz != nullptr) ? srcz[it] : T(0);
  // stress-rate (moment-tensor) source: xx, zz, xz increments of this step
  const bool msrc = S.msrc[0] || S.msrc[2] || S.msrc[4];
  const T incsxx = S.msrc[0] ? cp<T>(S.msrc[0])[it] : T(0);
  const T incszz = S.msrc[2] ? cp<T>(S.msrc[2])[it] : T(0);
  const T incsxz = S.msrc[4] ? cp<T>(S.msrc[4])[it] : T(0);

  auto row = [&](int r) { return (uint32_t)(r < 0 ? 0 : (r >= nz ? nz - 1 : r)) * nx + ic; };
  auto valid = [&](int r) { return incol && r >= 0 && r < nz; };
  T vx_m = valid(zo - 2) ? vxi[row(zo - 2)] : T(0);  // velocity row r-1
  T vz_m = valid(zo - 2) ? vzi[row(zo - 2)] : T(0);
  T vx_c = valid(zo - 1) ? vxi[row(zo - 1)] : T(0);  // velocity row r
  T vz_c = valid(zo - 1) ? vzi[row(zo - 1)] : T(0);
  T sxx_p = 0, szz_p = 0, sxz_p = 0, sxz_pp = 0;      // new stresses of rows r-1, r-2

  // Every load a row needs (addresses clamped in bounds).  With
  // SDT_EL2_PREFETCH the loads of row r+1 are issued before row r is
  // computed, so each wave keeps two rows of loads in flight.
  struct Row {
    T vxn, vzn, sxx, szz, sxz, n11, n13, n33, s55, n15, n35, s15, s35, dtx, dtz, omx, omz;
    T m_vxx, m_vzx, m_vzz, m_vxz, s_vxx, s_vzx, s_vzz, s_vxz, m_sxx, m_sxzx, m_szz, m_sxzz;
  };
  auto load_row = [&](int r) {
    Row L;
    const int rr = r - 1;
    const uint32_t c = row(r), cv = row(rr), cn = row(r + 1);
    L.vxn = vxi[cn];
    L.vzn = vzi[cn];
    L.sxx = sxxi[c];
    L.szz = szzi[c];
    L.sxz = sxzi[c];
    L.n11 = N11[c];
    L.n13 = N13[c];
    L.n33 = N33[c];
    L.s55 = S55[c];
    // monoclinic couplings and attenuation are optional (null = 0 and 1)
    L.n15 = mono ? N15[c] : T(0);
    L.n35 = mono ? N35[c] : T(0);
    L.s15 = mono ? S15[c] : T(0);
    L.s35 = mono ? S35[c] : T(0);
    L.dtx = DTX[cv];
    L.dtz = DTZ[cv];
    L.omx = atten ? OMX[cv] : T(1);
    L.omz = atten ? OMZ[cv] : T(1);
    const int rs = r < 0 ? 0 : (r >= nz ? nz - 1 : r);
    const int rvs = rr < 0 ? 0 : (rr >= nz ? nz - 1 : rr);
    const bool inz = PML && in_slab(rs, nz, lz), inzv = PML && in_slab(rvs, nz, lz);
    const uint32_t oxs = inx ? (uint32_t)rs * 2 * lx + xs : 0, oxvs = inx ? (uint32_t)rvs * 2 * lx + xs : 0;
    const uint32_t oz = ZB + (inz ? (uint32_t)slab_pos(rs, nz, lz) * nx + ic : 0);
    const uint32_t ozv = ZB + (inzv ? (uint32_t)slab_pos(rvs, nz, lz) * nx + ic : 0);
    // psi loads only where the cell has that memory (a zero-width slab has no storage)
    const bool inzc = incol && inz, inzvc = incol && inzv;
    L.m_vxx = inx ? pin[oxs] : T(0);  // x-slab, stress row
    L.m_vzx = inx ? pin[SX + oxs] : T(0);
    L.m_vzz = inzc ? pin[oz] : T(0);  // z-slab, stress row
    L.m_vxz = inzc ? pin[SZ + oz] : T(0);
    // split C-PML: the shear loop's own memory (x slab arrays 4, 5; z 4, 5)
    L.s_vxx = (SPLIT && inx) ? pin[4 * SX + oxs] : T(0);
    L.s_vzx = (SPLIT && inx) ? pin[5 * SX + oxs] : T(0);
    L.s_vzz = (SPLIT && inzc) ? pin[4 * SZ + oz] : T(0);
    L.s_vxz = (SPLIT && inzc) ? pin[5 * SZ + oz] : T(0);
    L.m_sxx = inx ? pin[2 * SX + oxvs] : T(0);  // velocity row
    L.m_sxzx = inx ? pin[3 * SX + oxvs] : T(0);
    L.m_szz = inzvc ? pin[2 * SZ + ozv] : T(0);
    L.m_sxzz = inzvc ? pin[3 * SZ + ozv] : T(0);
    return L;
  };
  // (FP64 keeps one row in flight: two would spill at its register budget)
  constexpr bool PF = SDT_EL2_PREFETCH && sizeof(T) == 4;
  Row ahead{};
  if constexpr (PF) ahead = load_row(zo - 1);

  // row step r: the stresses of row r, then the velocities of row r - 1
  auto step_row = [&](const int r, const Row& L) {
    const int rr = r - 1;                             // velocity row
    const uint32_t c = row(r), cv = row(rr);
    const bool rv = valid(r);
    const T ld_vxn = L.vxn, ld_vzn = L.vzn, ld_sxx = L.sxx, ld_szz = L.szz, ld_sxz = L.sxz;
    const T n11 = L.n11, n13 = L.n13, n33 = L.n33, s55 = L.s55;
    const T n15 = L.n15, n35 = L.n35, s15 = L.s15, s35 = L.s35;
    const T dtx = L.dtx, dtz = L.dtz, omx = L.omx, omz = L.omz;
    const int rs = r < 0 ? 0 : (r >= nz ? nz - 1 : r);
    const int rvs = rr < 0 ? 0 : (rr >= nz ? nz - 1 : rr);
    const bool inz = PML && in_slab(rs, nz, lz), inzv = PML && in_slab(rvs, nz, lz);
    const uint32_t ox = (uint32_t)rs * 2 * lx + xs, oxv = (uint32_t)rvs * 2 * lx + xs;
    const uint32_t oz = ZB + (inz ? (uint32_t)slab_pos(rs, nz, lz) * nx + ic : 0);
    const uint32_t ozv = ZB + (inzv ? (uint32_t)slab_pos(rvs, nz, lz) * nx + ic : 0);
    T m_vxx = L.m_vxx, m_vzx = L.m_vzx, m_vzz = L.m_vzz, m_vxz = L.m_vxz;
    T s_vxx = L.s_vxx, s_vzx = L.s_vzx, s_vzz = L.s_vzz, s_vxz = L.s_vxz;
    T m_sxx = L.m_sxx, m_sxzx = L.m_sxzx, m_szz = L.m_szz, m_sxzz = L.m_sxzz;
    const T bzr = bz[rs], azr = az[rs], ikzr = ikz[rs], bzhr = bzh[rs], azhr = azh[rs], ikzhr = ikzh[rs];
    const T browr = SPLIT ? bxh : brow[rs];  // b_x_half(j) (A2), or b_x_half(i)
    const T bzv = bz[rvs], azv = az[rvs], ikzv = ikz[rvs], bzhv = bzh[rvs], azhv = azh[rvs], ikzhv = ikzh[rvs];
    const bool nxt = (r + 1 <= zend) && valid(r + 1);
    const T vx_n = nxt ? ld_vxn : T(0), vz_n = nxt ? ld_vzn : T(0);  // velocity row r+1

    // ---- stresses of row r (seismicfdtd.f95:247-312) ----
    const T vx_e = lane_next(vx_c), vz_e = lane_next(vz_c);
    const T vx_w = lane_prev(vx_c), vz_w = lane_prev(vz_c);
    T sxx_c = rv ? ld_sxx : T(0), szz_c = rv ? ld_szz : T(0), sxz_c = rv ? ld_sxz : T(0);
    const bool inx_r = inx && rv, inz_r = incol && rv && inz;
    if (rv && can_n && r >= 1) {
      T dvx_dx = (vx_e - vx_c) * idx;
      T dvz_dz = (vz_c - vz_m) * idz;
      T dvz_dx = (vz_e - vz_c) * idx;
      T dvx_dz = (vx_c - vx_m) * idz;
      if (inx_r) {
        m_vxx = fma(browr, m_vxx, axh * dvx_dx);  // :255
        m_vzx = fma(bx, m_vzx, ax * dvz_dx);
        dvx_dx = fma(dvx_dx, ikxh, m_vxx);
        dvz_dx = fma(dvz_dx, ikx, m_vzx);
      }
      if (inz_r) {
        m_vzz = fma(bzr, m_vzz, azr * dvz_dz);
        m_vxz = fma(bzhr, m_vxz, azhr * dvx_dz);
        dvz_dz = fma(dvz_dz, ikzr, m_vzz);
        dvx_dz = fma(dvx_dz, ikzhr, m_vxz);
      }
      const T sh = dvz_dx + dvx_dz;
      sxx_c = fma(fma(n15, sh, fma(n13, dvz_dz, n11 * dvx_dx)), dt, sxx_c);
      szz_c = fma(fma(n35, sh, fma(n33, dvz_dz, n13 * dvx_dx)), dt, szz_c);
    }
    if (rv && can_s && r <= nz - 2 && r < zend) {  // same psi arrays (A1) unless split
      T& q_vxx = SPLIT ? s_vxx : m_vxx;
      T& q_vzx = SPLIT ? s_vzx : m_vzx;
      T& q_vzz = SPLIT ? s_vzz : m_vzz;
      T& q_vxz = SPLIT ? s_vxz : m_vxz;
      T dvx_dx = (vx_c - vx_w) * idx;
      T dvz_dz = (vz_n - vz_c) * idz;
      T dvz_dx = (vz_c - vz_w) * idx;
      T dvx_dz = (vx_n - vx_c) * idz;
      if (inx_r) {
        q_vxx = fma(bxh, q_vxx, axh * dvx_dx);
        q_vzx = fma(bx, q_vzx, ax * dvz_dx);
        dvx_dx = fma(dvx_dx, ikxh, q_vxx);
        dvz_dx = fma(dvz_dx, ikx, q_vzx);
      }
      if (inz_r) {
        q_vzz = fma(bzr, q_vzz, azr * dvz_dz);
        q_vxz = fma(bzhr, q_vxz, azhr * dvx_dz);
        dvz_dz = fma(dvz_dz, ikzr, q_vzz);
        dvx_dz = fma(dvx_dz, ikzhr, q_vxz);
      }
      sxz_c = fma(fma(s55, dvz_dx + dvx_dz, fma(s35, dvz_dz, s15 * dvx_dx)), dt, sxz_c);
    }
    if (msrc && rv && is_src_col && r == ksrc) {  // every lane that computes the cell adds it
      sxx_c += incsxx;
      szz_c += incszz;
      sxz_c += incsxz;
    }
    if (own && rv && r >= zo && r < zend) {
      sxxo[c] = sxx_c;
      szzo[c] = szz_c;
      sxzo[c] = sxz_c;
      if (inx) {
        pout[ox] = m_vxx;
        pout[SX + ox] = m_vzx;
        if (SPLIT) {
          pout[4 * SX + ox] = s_vxx;
          pout[5 * SX + ox] = s_vzx;
        }
      }
      if (inz) {
        pout[oz] = m_vzz;
        pout[SZ + oz] = m_vxz;
        if (SPLIT) {
          pout[4 * SZ + oz] = s_vzz;
          pout[5 * SZ + oz] = s_vxz;
        }
      }
    }

    // ---- velocities of row rr = r - 1 (seismicfdtd.f95:317-375) ----
    const T sxx_w = lane_prev(sxx_p);  // sigma_xx(i-1, rr)
    const T sxz_e = lane_next(sxz_p);  // sigma_xz(i+1, rr)
    T gvx = 0, gvz = 0;  // new velocities of the owned cells (receiver samples)
    if (own && rr >= zo && rr < zend) {
      T vxn = vx_m, vzn = vz_m;
      if (ux && rr >= 1) {
        T a = (sxx_p - sxx_w) * idx;
        T b = (sxz_p - sxz_pp) * idz;
        if (inx) {
          m_sxx = fma(bx, m_sxx, ax * a);
          a = fma(a, ikx, m_sxx);
        }
        if (inzv) {
          m_sxzz = fma(bzv, m_sxzz, azv * b);
          b = fma(b, ikzv, m_sxzz);
        }
        vxn = fma(vxn, omx, (a + b) * dtx);
      }
      if (uz && rr <= nz - 2) {
        T a = (sxz_e - sxz_p) * idx;
        T b = (szz_c - szz_p) * idz;
        if (inx) {
          m_sxzx = fma(bxh, m_sxzx, axh * a);
          a = fma(a, ikxh, m_sxzx);
        }
        if (inzv) {
          m_szz = fma(bzhv, m_szz, azhv * b);
          b = fma(b, ikzhv, m_szz);
        }
        vzn = fma(vzn, omz, (a + b) * dtz);
      }
      if (inx) { pout[2 * SX + oxv] = m_sxx; pout[3 * SX + oxv] = m_sxzx; }
      if (inzv) { pout[2 * SZ + ozv] = m_szz; pout[3 * SZ + ozv] = m_sxzz; }
      if (is_src_col && rr == ksrc) { vxn += incx; vzn += incz; }   // source, :359-361
      if (i == 0 || i == nx - 1 || rr == 0 || rr == nz - 1) { vxn = 0; vzn = 0; }  // :365-375
      check_blowup((double)vxn * vxn + (double)vzn * vzn, S.blowup, it);
      vxo[cv] = vxn;
      vzo[cv] = vzn;
      gvx = vxn;
      gvz = vzn;
    }
    if (has_rec && rr >= zo && rr < zend) gather_row<T>(S, rr, it, lane, xo - 1, 1, EW, gvx, gvz);
    sxz_pp = sxz_p;
    sxx_p = sxx_c;
    szz_p = szz_c;
    sxz_p = sxz_c;
    vx_m = vx_c;
    vz_m = vz_c;
    vx_c = vx_n;
    vz_c = vz_n;
  };
  if constexpr (R1) {
    // one row (zend == zo + 1): the loads of rows zo-1, zo, zo+1 read only
    // the previous state, so all three are in flight before the first step
    const Row L0 = load_row(zo - 1), L1 = load_row(zo), L2 = load_row(zo + 1);
    step_row(zo - 1, L0);
    step_row(zo, L1);
    step_row(zo + 1, L2);
  } else {
    for (int r = zo - 1; r <= zend; ++r) {
      Row L;
      if constexpr (PF) {
        L = ahead;
        ahead = load_row(r + 1);
      } else {
        L = load_row(r);
      }
      step_row(r, L);
    }
  }
}

// ===========================================================================
// ELASTIC2, two time steps per launch.
//
// The walk of k_el2_step with the second step pipelined behind the first.
// At row r a wavefront computes
//   A  the stresses of step it at row r      (velocities of it-1, rows r-1..r+1)
//   B  the velocities of step it at row r-1  (stresses from A, rows r-2..r)
//   C  the stresses of step it+1 at row r-2  (velocities from B, rows r-3..r-1)
//   D  the velocities of step it+1 at row r-3 (stresses from C, rows r-4..r-2)
// so the state of step it lives only in registers and each field, memory
// variable and coefficient crosses HBM once per two steps.
// One step makes a cell depend on columns i-1 .. i+2 and rows k-2 .. k+1 of
// the previous state (the shear stress updates the C-PML memory the normal
// stresses just updated, quirk A1, so it sees the normal loop's neighbours);
// two steps on columns i-2 .. i+4 and rows k-4 .. k+2.  Lane l therefore
// holds column xo - 2 + l and lanes 2 .. 2+EW2-1 are exact after two steps;
// rows zo-4 .. zo+eh+1 are read to produce rows zo .. zo+eh-1.  Every stage
// evaluates the expressions of k_el2_step in the same order, so both kernels
// give identical bits.  The state of step it is never stored, so this kernel
// also writes the receiver samples of both steps.
// The state of step it is read from buffer ((it - *it0) / 2) & 1 and the
// state of it+2 written to the other (it0: first step of the run).
// ===========================================================================
// Owned columns per wavefront (at most 58: two halo lanes on the left, four
// on the right).  56 makes every wavefront's row of stores start and end on
// a 32-byte boundary (56 floats = 224 bytes, tiles at multiples of 56), so
// no HBM sector is written in pieces by two wavefronts: 134.3 against 131.4
// Gcell-updates/s with 58 on the 96-shot layered workload, same bits.
#ifndef SDT_EL2X2_EW
#define SDT_EL2X2_EW 56
#endif
constexpr int EW2 = SDT_EL2X2_EW;
static_assert(EW2 >= 1 && EW2 <= 58, "two-step wavefront: 2 halo lanes left, 4 right");
#ifndef SDT_EL2X2_WAVES
#define SDT_EL2X2_WAVES 4   // FP32 wavefronts per SIMD the register budget allows
#endif
#ifndef SDT_EL2X2_PREFETCH
#define SDT_EL2X2_PREFETCH 0
#endif
#ifndef SDT_EL2X2_WAVES_SPLIT
// the same for the split C-PML variant's edge kernel: at 4 wavefronts it
// spills a few registers and is still faster than at 3 (1.178 against
// 1.228 ms per two-step launch pair of the 96-shot layered workload)
#define SDT_EL2X2_WAVES_SPLIT 4
#endif
#ifndef SDT_EL2X2_WAVES_INT
#define SDT_EL2X2_WAVES_INT 5  // the same for the interior-only kernel
#endif

template <typename T, bool SPLIT, int BODY>
__device__ __forceinline__ void el2x2_tile(const DModel* __restrict__ models,
                                           const DShot* __restrict__ shots, const int4 wi, const int it,
                                           const int q, const int lane, const int eh) {
#pragma clang fp contract(off)
  // BODY 0: an interior wave (no C-PML) reads only columns 1..nx-2 and rows
  // 1..nz-2, so every edge condition of the scheme holds on every lane;
  // BODY 1: its columns are interior (every condition on the column holds,
  // no x slab) but its rows may reach a z slab or the outer rows;
  // BODY 2: anything else; BODY 3 (below): x-slab columns of a tile whose
  // rows are all off the z slabs and the outer rows.
  // BODY 3: as 2, but every row the wave reads is off the z slabs and the
  // outer rows (x-slab columns of a z-interior tile).
  constexpr bool INT = BODY == 0, XI = BODY < 2, PML = BODY > 0, ZI = BODY == 3;
  const DShot& S = shots[wi.x];
  const DModel& M = models[S.model];
  const int nx = M.nx, nz = M.nz;
  const int xo = wi.y, zo = wi.z;
  const int i = xo - 2 + lane;
  const bool incol = XI || (i >= 0 && i < nx);
  const int ic = XI ? i : (incol ? i : (i < 0 ? 0 : nx - 1));  // clamped column: every load stays in bounds
  const bool own = incol && lane >= 2 && lane < 2 + EW2;
  const int ze = min(zo + eh, nz);
  const A32<const T> vxi(q ? S.g[0] : S.f[0]);
  const A32<const T> vzi(q ? S.g[1] : S.f[1]);
  const A32<const T> sxxi(q ? S.g[2] : S.f[2]);
  const A32<const T> szzi(q ? S.g[3] : S.f[3]);
  const A32<const T> sxzi(q ? S.g[4] : S.f[4]);
  const A32<T> vxo(q ? S.f[0] : S.g[0]);
  const A32<T> vzo(q ? S.f[1] : S.g[1]);
  const A32<T> sxxo(q ? S.f[2] : S.g[2]);
  const A32<T> szzo(q ? S.f[3] : S.g[3]);
  const A32<T> sxzo(q ? S.f[4] : S.g[4]);
  const A32<const T> pin(q ? S.psi2 : S.psi);
  const A32<T> pout(q ? S.psi : S.psi2);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dt = T(M.dt);
  const int lx = M.lx, lz = M.lz;
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const uint32_t ZB = (SPLIT ? 6 : 4) * SX;  // first z-slab array
  const bool inx = !XI && incol && in_slab(i, nx, lx);
  const int xs = inx ? slab_pos(i, nx, lx) : 0;
  const Prof<T> P(&M.prof[0][0]);
  const T ikx = P[PK][ic], ax = P[PA][ic], bx = P[PB][ic];
  const T ikxh = P[PKH][ic], axh = P[PAH][ic], bxh = P[PBH][ic];
  // z profiles and b_x_half by row: one value per row, read through the
  // scalar (constant) path into SGPRs; nothing writes them during a launch
  const auto ikz = kp<T>(M.prof[2][PK]), az = kp<T>(M.prof[2][PA]), bz = kp<T>(M.prof[2][PB]);
  const auto ikzh = kp<T>(M.prof[2][PKH]), azh = kp<T>(M.prof[2][PAH]), bzh = kp<T>(M.prof[2][PBH]);
  const auto brow = kp<T>(M.aux);
  const A32<const T> N11(M.coef[0]), N13(M.coef[1]), N15(M.coef[2]);
  const A32<const T> N33(M.coef[3]), N35(M.coef[4]);
  const A32<const T> S15(M.coef[5]), S35(M.coef[6]), S55(M.coef[7]);
  const A32<const T> DTX(M.coef[8]), DTZ(M.coef[9]);
  const A32<const T> OMX(M.coef[10]), OMZ(M.coef[11]);
  const bool mono = M.coef[2] != nullptr;   // c15 / c35 terms present
  const bool atten = M.coef[10] != nullptr; // gamma present
  const bool is_src_col = (i == S.isrc);
  const int ksrc = S.ksrc;
  const auto srcx = cp<T>(S.src[0]), srcz = cp<T>(S.src[2]);
  const T incx0 = srcx ? srcx[it] : T(0), incx1 = srcx ? srcx[it + 1] : T(0);
  const T incz0 = srcz ? srcz[it] : T(0), incz1 = srcz ? srcz[it + 1] : T(0);
  const bool msrc = S.msrc[0] || S.msrc[2] || S.msrc[4];
  const T ms0xx = S.msrc[0] ? cp<T>(S.msrc[0])[it] : T(0), ms1xx = S.msrc[0] ? cp<T>(S.msrc[0])[it + 1] : T(0);
  const T ms0zz = S.msrc[2] ? cp<T>(S.msrc[2])[it] : T(0), ms1zz = S.msrc[2] ? cp<T>(S.msrc[2])[it + 1] : T(0);
  const T ms0xz = S.msrc[4] ? cp<T>(S.msrc[4])[it] : T(0), ms1xz = S.msrc[4] ? cp<T>(S.msrc[4])[it + 1] : T(0);

  auto crow = [&](int r) { return r < 0 ? 0 : (r >= nz ? nz - 1 : r); };
  auto cell = [&](int r) { return (uint32_t)crow(r) * nx + ic; };
  auto valid = [&](int r) { return INT || (incol && r >= 0 && r < nz); };

  struct CN { T n11, n13, n33, s55, n15, n35, s15, s35; };  // stress coefficients of a row
  struct CV { T dtx, dtz, omx, omz; };                      // velocity coefficients of a row
  struct MV { T vxx, vzx, vzz, vxz, svxx, svzx, svzz, svxz; };  // memory of velocity derivatives
  struct MS { T sxx, sxzx, szz, sxzz; };                    // memory of stress derivatives

  auto load_cn = [&](int r) {
    CN k;
    const uint32_t c = cell(r);
    k.n11 = N11[c];
    k.n13 = N13[c];
    k.n33 = N33[c];
    k.s55 = S55[c];
    k.n15 = mono ? N15[c] : T(0);
    k.n35 = mono ? N35[c] : T(0);
    k.s15 = mono ? S15[c] : T(0);
    k.s35 = mono ? S35[c] : T(0);
    return k;
  };
  auto load_cv = [&](int r) {
    CV k;
    const uint32_t c = cell(r);
    k.dtx = DTX[c];
    k.dtz = DTZ[c];
    k.omx = atten ? OMX[c] : T(1);
    k.omz = atten ? OMZ[c] : T(1);
    return k;
  };
  // slab offsets of row r: x slab (valid where inx), z slab (ZB-based)
  auto offx = [&](int r) { return inx ? (uint32_t)crow(r) * 2 * lx + xs : 0u; };
  auto inzs = [&](int r) { return PML && !ZI && in_slab(crow(r), nz, lz); };
  auto offz = [&](int r) { return ZB + (inzs(r) ? (uint32_t)slab_pos(crow(r), nz, lz) * nx + ic : 0u); };
  auto load_mv = [&](int r) {
    MV m{};
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      const bool inzc = incol && inzs(r);
      m.vxx = inx ? pin[ox] : T(0);
      m.vzx = inx ? pin[SX + ox] : T(0);
      m.vzz = inzc ? pin[oz] : T(0);
      m.vxz = inzc ? pin[SZ + oz] : T(0);
      if (SPLIT) {
        m.svxx = inx ? pin[4 * SX + ox] : T(0);
        m.svzx = inx ? pin[5 * SX + ox] : T(0);
        m.svzz = inzc ? pin[4 * SZ + oz] : T(0);
        m.svxz = inzc ? pin[5 * SZ + oz] : T(0);
      }
    }
    return m;
  };
  auto load_ms = [&](int r) {
    MS m{};
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      const bool inzc = incol && inzs(r);
      m.sxx = inx ? pin[2 * SX + ox] : T(0);
      m.sxzx = inx ? pin[3 * SX + ox] : T(0);
      m.szz = inzc ? pin[2 * SZ + oz] : T(0);
      m.sxzz = inzc ? pin[3 * SZ + oz] : T(0);
    }
    return m;
  };
  auto store_mv = [&](int r, const MV& m) {  // own cells only
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      if (inx) {
        pout[ox] = m.vxx;
        pout[SX + ox] = m.vzx;
        if (SPLIT) {
          pout[4 * SX + ox] = m.svxx;
          pout[5 * SX + ox] = m.svzx;
        }
      }
      if (inzs(r)) {
        pout[oz] = m.vzz;
        pout[SZ + oz] = m.vxz;
        if (SPLIT) {
          pout[4 * SZ + oz] = m.svzz;
          pout[5 * SZ + oz] = m.svxz;
        }
      }
    }
  };
  auto store_ms = [&](int r, const MS& m) {  // own cells only
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      if (inx) { pout[2 * SX + ox] = m.sxx; pout[3 * SX + ox] = m.sxzx; }
      if (inzs(r)) { pout[2 * SZ + oz] = m.szz; pout[3 * SZ + oz] = m.sxzz; }
    }
  };

  // Stresses of one step at row a (seismicfdtd.f95:247-312): velocities of
  // rows a-1, a, a+1 in, the row's stresses and memory updated in place.
  auto stress = [&](int a, T vxm, T vzm, T vxc, T vzc, T vxn, T vzn, T& sxx, T& szz, T& sxz,
                    const CN& k, MV& m, T isxx, T iszz, T isxz) {
    const T vx_e = dpp_next(vxc), vz_e = dpp_next(vzc);
    const T vx_w = dpp_prev(vxc), vz_w = dpp_prev(vzc);
    const bool rv = valid(a);
    const int rs = crow(a);
    const bool inx_r = inx && rv, inz_r = incol && rv && inzs(a);
    T bzr = 0, azr = 0, ikzr = 0, bzhr = 0, azhr = 0, ikzhr = 0, browr = 0;
    if constexpr (PML) {
      bzr = bz[rs]; azr = az[rs]; ikzr = ikz[rs];
      bzhr = bzh[rs]; azhr = azh[rs]; ikzhr = ikzh[rs];
      browr = SPLIT ? bxh : brow[rs];  // b_x_half(j) (A2), or b_x_half(i)
    }
    if (INT || (rv && (XI || i <= nx - 2) && a >= 1)) {
      T dvx_dx = (vx_e - vxc) * idx;
      T dvz_dz = (vzc - vzm) * idz;
      T dvz_dx = (vz_e - vzc) * idx;
      T dvx_dz = (vxc - vxm) * idz;
      if (PML && inx_r) {
        m.vxx = fma(browr, m.vxx, axh * dvx_dx);
        m.vzx = fma(bx, m.vzx, ax * dvz_dx);
        dvx_dx = fma(dvx_dx, ikxh, m.vxx);
        dvz_dx = fma(dvz_dx, ikx, m.vzx);
      }
      if (PML && inz_r) {
        m.vzz = fma(bzr, m.vzz, azr * dvz_dz);
        m.vxz = fma(bzhr, m.vxz, azhr * dvx_dz);
        dvz_dz = fma(dvz_dz, ikzr, m.vzz);
        dvx_dz = fma(dvx_dz, ikzhr, m.vxz);
      }
      const T sh = dvz_dx + dvx_dz;
      sxx = fma(fma(k.n15, sh, fma(k.n13, dvz_dz, k.n11 * dvx_dx)), dt, sxx);
      szz = fma(fma(k.n35, sh, fma(k.n33, dvz_dz, k.n13 * dvx_dx)), dt, szz);
    }
    if (INT || (rv && (XI || i >= 1) && a <= nz - 2)) {  // same memory arrays (A1) unless split
      T& q_vxx = SPLIT ? m.svxx : m.vxx;
      T& q_vzx = SPLIT ? m.svzx : m.vzx;
      T& q_vzz = SPLIT ? m.svzz : m.vzz;
      T& q_vxz = SPLIT ? m.svxz : m.vxz;
      T dvx_dx = (vxc - vx_w) * idx;
      T dvz_dz = (vzn - vzc) * idz;
      T dvz_dx = (vzc - vz_w) * idx;
      T dvx_dz = (vxn - vxc) * idz;
      if (PML && inx_r) {
        q_vxx = fma(bxh, q_vxx, axh * dvx_dx);
        q_vzx = fma(bx, q_vzx, ax * dvz_dx);
        dvx_dx = fma(dvx_dx, ikxh, q_vxx);
        dvz_dx = fma(dvz_dx, ikx, q_vzx);
      }
      if (PML && inz_r) {
        q_vzz = fma(bzr, q_vzz, azr * dvz_dz);
        q_vxz = fma(bzhr, q_vxz, azhr * dvx_dz);
        dvz_dz = fma(dvz_dz, ikzr, q_vzz);
        dvx_dz = fma(dvx_dz, ikzhr, q_vxz);
      }
      sxz = fma(fma(k.s55, dvz_dx + dvx_dz, fma(k.s35, dvz_dz, k.s15 * dvx_dx)), dt, sxz);
    }
    if (msrc && a == ksrc && rv && is_src_col) {
      sxx += isxx;
      szz += iszz;
      sxz += isxz;
    }
  };
  // Velocities of one step at row b (seismicfdtd.f95:317-375): the new
  // stresses of rows b-1 (sxz), b, b+1 (szz) in.
  auto vel = [&](int b, T sxx_b, T szz_b, T sxz_b, T sxz_bm, T szz_bn, T vx_old, T vz_old,
                 const CV& k, MS& m, T ix, T iz, T& vxn, T& vzn) {
    const T sxx_w = dpp_prev(sxx_b);  // sigma_xx(i-1, b)
    const T sxz_e = dpp_next(sxz_b);  // sigma_xz(i+1, b)
    const bool rv = valid(b);
    const int rs = crow(b);
    const bool inzv = PML && inzs(b);
    T bzv = 0, azv = 0, ikzv = 0, bzhv = 0, azhv = 0, ikzhv = 0;
    if constexpr (PML) {
      bzv = bz[rs]; azv = az[rs]; ikzv = ikz[rs];
      bzhv = bzh[rs]; azhv = azh[rs]; ikzhv = ikzh[rs];
    }
    vxn = vx_old;
    vzn = vz_old;
    if (INT || (rv && (XI || i >= 1) && b >= 1)) {
      T a = (sxx_b - sxx_w) * idx;
      T c = (sxz_b - sxz_bm) * idz;
      if (PML && inx) {
        m.sxx = fma(bx, m.sxx, ax * a);
        a = fma(a, ikx, m.sxx);
      }
      if (PML && inzv) {
        m.sxzz = fma(bzv, m.sxzz, azv * c);
        c = fma(c, ikzv, m.sxzz);
      }
      vxn = fma(vxn, k.omx, (a + c) * k.dtx);
    }
    if (INT || (rv && (XI || i <= nx - 2) && b <= nz - 2)) {
      T a = (sxz_e - sxz_b) * idx;
      T c = (szz_bn - szz_b) * idz;
      if (PML && inx) {
        m.sxzx = fma(bxh, m.sxzx, axh * a);
        a = fma(a, ikxh, m.sxzx);
      }
      if (PML && inzv) {
        m.szz = fma(bzhv, m.szz, azhv * c);
        c = fma(c, ikzhv, m.szz);
      }
      vzn = fma(vzn, k.omz, (a + c) * k.dtz);
    }
    if (b == ksrc && is_src_col) { vxn += ix; vzn += iz; }   // source, :359-361
    if (!INT && (!rv || (!XI && (i == 0 || i == nx - 1)) || b == 0 || b == nz - 1)) {  // :365-375
      vxn = 0;
      vzn = 0;
    }
  };
  // receiver samples of step itn at row b (an own row; every lane calls)
  const int nrec = S.nrec;
  auto gather = [&](int b, int itn, T vx, T vz) { gather_row<T>(S, b, itn, lane, xo - 2, 2, 1 + EW2, vx, vz); };

  T vx0_m = valid(zo - 4) ? vxi[cell(zo - 4)] : T(0);  // velocities of step it-1, row r-1
  T vz0_m = valid(zo - 4) ? vzi[cell(zo - 4)] : T(0);
  T vx0_c = valid(zo - 3) ? vxi[cell(zo - 3)] : T(0);  // row r
  T vz0_c = valid(zo - 3) ? vzi[cell(zo - 3)] : T(0);
  T s1xx_p = 0, s1zz_p = 0, s1xz_p = 0, s1xx_pp = 0, s1zz_pp = 0, s1xz_pp = 0;  // step it, rows r-1, r-2
  T v1x_m = 0, v1z_m = 0, v1x_c = 0, v1z_c = 0;  // step it, rows r-3, r-2
  T s2xx_p = 0, s2zz_p = 0, s2xz_p = 0, s2xz_pp = 0;  // step it+1, rows r-3 (and r-4)
  CN kn_p{}, kn_pp{};  // stress coefficients of rows r-1, r-2
  CV kv_p{}, kv_pp{};  // velocity coefficients of rows r-2, r-3
  MV mv_p{}, mv_pp{};  // memory after step it, rows r-1, r-2
  MS ms_p{}, ms_pp{};  // memory after step it, rows r-2, r-3
  // receivers on the tile's own rows at all (one test per tile, not per row)
  const bool has_rec = nrec > 0 && S.rrow[ze] > S.rrow[zo];
  bool bad0 = false, bad1 = false;  // own cell above the blow-up bound at step it / it+1

  // Every load of iteration r (addresses clamped in bounds).  With
  // SDT_EL2X2_PREFETCH the loads of iteration r+1 are issued before
  // iteration r computes, so each wavefront keeps two rows in flight.
  struct Ld {
    T vx, vz, sxx, szz, sxz;
    CN kn;
    MV mv;
    CV kv;
    MS ms;
  };
  auto load_it = [&](int r) {
    Ld L;
    L.vx = vxi[cell(r + 1)];
    L.vz = vzi[cell(r + 1)];
    const uint32_t cA = cell(r);
    L.sxx = sxxi[cA];
    L.szz = szzi[cA];
    L.sxz = sxzi[cA];
    L.kn = load_cn(r);
    L.mv = load_mv(r);
    L.kv = load_cv(r - 1);
    L.ms = load_ms(r - 1);
    return L;
  };
  constexpr bool PF = SDT_EL2X2_PREFETCH && INT;
  Ld ahead{};
  if constexpr (PF) ahead = load_it(zo - 3);

  for (int r = zo - 3; r <= ze + 2; ++r) {
    const bool actA = r <= ze + 1, actB = r >= zo - 1 && r <= ze + 1;
    const bool actC = r >= zo + 1, actD = r >= zo + 3;
    Ld L;
    if constexpr (PF) {
      L = ahead;
      ahead = load_it(r + 1);
    } else {
      L = load_it(r);
    }
    const T ld_vx = L.vx, ld_vz = L.vz, ld_sxx = L.sxx, ld_szz = L.szz, ld_sxz = L.sxz;
    const CN kn = L.kn;
    MV mv = L.mv;
    const CV kv = L.kv;
    MS ms = L.ms;
    const bool nxt = r + 1 <= ze + 1 && valid(r + 1);
    const T vx0_n = nxt ? ld_vx : T(0), vz0_n = nxt ? ld_vz : T(0);

    // A: stresses of step it, row r
    const bool rvA = valid(r);
    T s1xx_c = rvA ? ld_sxx : T(0), s1zz_c = rvA ? ld_szz : T(0), s1xz_c = rvA ? ld_sxz : T(0);
    if (actA)
      stress(r, vx0_m, vz0_m, vx0_c, vz0_c, vx0_n, vz0_n, s1xx_c, s1zz_c, s1xz_c, kn, mv, ms0xx, ms0zz,
             ms0xz);
    // B: velocities of step it, row r-1
    T v1x_n = 0, v1z_n = 0;
    if (actB) {
      vel(r - 1, s1xx_p, s1zz_p, s1xz_p, s1xz_pp, s1zz_c, vx0_m, vz0_m, kv, ms, incx0, incz0, v1x_n, v1z_n);
      if (r - 1 >= zo && r - 1 < ze) {
        bad0 |= own && !((double)v1x_n * v1x_n + (double)v1z_n * v1z_n <= 1.0e50);
        if (has_rec) gather(r - 1, it, v1x_n, v1z_n);
      }
    }
    // C: stresses of step it+1, row r-2
    T s2xx_c = s1xx_pp, s2zz_c = s1zz_pp, s2xz_c = s1xz_pp;
    if (actC) {
      MV mc = mv_pp;
      stress(r - 2, v1x_m, v1z_m, v1x_c, v1z_c, v1x_n, v1z_n, s2xx_c, s2zz_c, s2xz_c, kn_pp, mc, ms1xx,
             ms1zz, ms1xz);
      if (own && r - 2 >= zo && r - 2 < ze) {
        const uint32_t c = cell(r - 2);
        sxxo[c] = s2xx_c;
        szzo[c] = s2zz_c;
        sxzo[c] = s2xz_c;
        store_mv(r - 2, mc);
      }
    }
    // D: velocities of step it+1, row r-3
    if (actD) {
      MS md = ms_pp;
      T v2x, v2z;
      vel(r - 3, s2xx_p, s2zz_p, s2xz_p, s2xz_pp, s2zz_c, v1x_m, v1z_m, kv_pp, md, incx1, incz1, v2x, v2z);
      if (r - 3 < ze) {
        bad1 |= own && !((double)v2x * v2x + (double)v2z * v2z <= 1.0e50);
        if (own) {
          const uint32_t c = cell(r - 3);
          vxo[c] = v2x;
          vzo[c] = v2z;
          store_ms(r - 3, md);
        }
        if (has_rec) gather(r - 3, it + 1, v2x, v2z);
      }
    }
    vx0_m = vx0_c; vz0_m = vz0_c; vx0_c = vx0_n; vz0_c = vz0_n;
    s1xx_pp = s1xx_p; s1zz_pp = s1zz_p; s1xz_pp = s1xz_p;
    s1xx_p = s1xx_c; s1zz_p = s1zz_c; s1xz_p = s1xz_c;
    v1x_m = v1x_c; v1z_m = v1z_c; v1x_c = v1x_n; v1z_c = v1z_n;
    s2xz_pp = s2xz_p; s2xx_p = s2xx_c; s2zz_p = s2zz_c; s2xz_p = s2xz_c;
    kn_pp = kn_p; kn_p = kn; kv_pp = kv_p; kv_p = kv;
    mv_pp = mv_p; mv_p = mv; ms_pp = ms_p; ms_p = ms;
  }
  if (bad0)
    check_blowup(HUGE_VAL, S.blowup, it);
  else if (bad1)
    check_blowup(HUGE_VAL, S.blowup, it + 1);
}

// Work: as k_el2_step, with EW2 owned columns per wavefront.  INT: every
// item of the work list is an interior block (el2x2_interior), so the kernel
// holds only the interior body and its smaller register budget allows more
// wavefronts per SIMD; otherwise each wavefront picks its body.
template <typename T, bool SPLIT, int WB, bool INT>
// (the split variant's C-PML body needs a larger budget: fewer wavefronts)
__global__ void __launch_bounds__(64 * WB, sizeof(T) == 4 ? (INT ? SDT_EL2X2_WAVES_INT : SPLIT ? SDT_EL2X2_WAVES_SPLIT : SDT_EL2X2_WAVES)
                                                          : (INT ? 3 : SPLIT ? 1 : 2))
k_el2_step2(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const int4* __restrict__ work, int nitems, const int* __restrict__ base, int rel,
            const int* __restrict__ it0, int eh0) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = __builtin_amdgcn_readfirstlane(*base + rel);
  const int q = __builtin_amdgcn_readfirstlane(((it - *it0) >> 1) & 1);
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const int4 wv = work[w];
    const int4 wi = make_int4(__builtin_amdgcn_readfirstlane(wv.x),
                              __builtin_amdgcn_readfirstlane(wv.y) + wave * EW2,
                              __builtin_amdgcn_readfirstlane(wv.z), 0);
    if (wi.x < 0) continue;
    const DModel& M = models[shots[wi.x].model];
    if (wi.y >= M.nx) continue;
    const int eh = wv.w > 0 ? __builtin_amdgcn_readfirstlane(wv.w) : eh0;  // rows of this tile
    // the columns (lanes), resp. rows (zo-4 .. ze+1), the wave reads outside
    // the C-PML slabs and off the outer ring (columns 0, nx-1 and rows 0,
    // nz-1 and their neighbours)
    const int ze = min(wi.z + eh, M.nz);
    const bool xint = wi.y - 2 >= M.lx + 1 && wi.y + 61 <= M.nx - M.lx - 2;
    const bool zint = wi.z - 4 >= M.lz + 1 && ze + 1 <= M.nz - M.lz - 2;
    if (INT || (xint && zint))
      el2x2_tile<T, SPLIT, 0>(models, shots, wi, it, q, threadIdx.x & 63, eh);
    else if (xint)
      el2x2_tile<T, SPLIT, 1>(models, shots, wi, it, q, threadIdx.x & 63, eh);
    else if (zint)
      el2x2_tile<T, SPLIT, 3>(models, shots, wi, it, q, threadIdx.x & 63, eh);
    else
      el2x2_tile<T, SPLIT, 2>(models, shots, wi, it, q, threadIdx.x & 63, eh);
  }
}

// After a run whose last step wrote buffer B, copy B's fields and psi into A
// so the caller always finds the state in field[] / psi (A); B keeps an
// identical copy, which the next (odd) step reads.  With to_b the copy runs
// the other way (a run of two-step launches that ends in A before an odd
// step).  blockIdx.z: the field, or psi after the last.  Every short run with an
// odd number of launches waits for it: 16 bytes per lane where the two arrays
// are aligned alike (us, element by element with a division per element, then
// so: 36 shots of 1064x808 elastic FP32 475, 259, FP64 541, 496, where it reaches
// 5 TB/s; 32 shots EM FP32 257, 139; 6 shots 33, 19).
template <typename T>
__global__ void __launch_bounds__(256)
k_copy_back(const DShot* __restrict__ shots, int nfield, const long* __restrict__ nel,
            const long* __restrict__ npsi, int to_b) {
  using V = __attribute__((ext_vector_type(4))) uint32_t;
  constexpr int E = 16 / sizeof(T);
  const int s = blockIdx.y, f = blockIdx.z;
  const DShot& S = shots[s];
  const long n = f < nfield ? nel[s] : npsi[s];
  void* const a = f < nfield ? S.f[f] : S.psi;
  void* const b = f < nfield ? S.g[f] : S.psi2;
  void* const src = to_b ? a : b;
  void* const dst = to_b ? b : a;
  // elements before the first 16-byte boundary, then whole vectors
  long head = n, nv = 0;
  if ((((uintptr_t)src ^ (uintptr_t)dst) & 15) == 0) {
    head = min(n, (long)((16 - ((uintptr_t)src & 15)) & 15) / (long)sizeof(T));
    nv = (n - head) / E;
  }
  const long t0 = (long)blockIdx.x * blockDim.x + threadIdx.x, step = (long)gridDim.x * blockDim.x;
  const auto sv = (gcptr<V>)((const T*)src + head);
  const auto dv = (gptr<V>)((T*)dst + head);
  for (long q = t0; q < nv; q += step) dv[q] = sv[q];
  for (long q = t0; q < n - nv * E; q += step) {
    const long e = q < head ? q : q + nv * E;
    mp<T>(dst)[e] = cp<T>(src)[e];
  }
}

// ===========================================================================
// ELASTIC2 adjoint: the transpose of one k_el2_step, for gradients of a
// trace misfit.  No counterpart in the reference (it has no adjoint).
//
// A step maps u_t = (v, sigma, psi) to u_{t+1} through the legacy sub-loops
// N (normal stresses), S (shear stress), V (velocities), source and
// Dirichlet edges, each linear in the state.  Its transpose runs them in
// reverse: with lambda_{t+1} = dJ/du_{t+1} (residual already injected at
// the receivers), adjoint step t produces lambda_t and adds
//   dJ/dcoef += lambda' * (d new state / d coef)
// where the partial products are recomputed from u_t and u_{t+1}, both
// read from the trail of recomputed forward states.  Three launches:
//   k_el2_adj_v  V^T : lambda of the new velocities -> partial lambda_v,
//                psi_s adjoint, and per-cell stress-derivative adjoints
//                (scratch planes 0..3);
//   k_el2_adj_s  gathers those into lambda_sigma, then S^T and N^T with
//                the shared velocity-derivative psi, writing per-cell
//                velocity-derivative adjoints (planes 4..11);
//   k_el2_adj_g  gathers those into lambda_v.
// Gradient slots are the kernel coefficient slots of the model
// (n11 n13 n15 n33 n35 s15 s35 s55 dt/rho_x dt/rho_z 1-gx 1-gz), FP64,
// accumulated atomically so shots of one model may share one array.
// ===========================================================================
__device__ __forceinline__ void gadd(double* g, double v) {
  if (v != 0.0) unsafeAtomicAdd(g, v);
}
// FP32 plans stage the gradient in FP32 within one sdt_adjoint_run call (at
// most a segment of steps) and flush it into the FP64 array at the end:
// half the atomic bytes, so a model's staging stays in L2.
__device__ __forceinline__ void gadd(float* g, double v) {
  const float f = (float)v;
  if (f != 0.0f) unsafeAtomicAdd(g, f);
}
__device__ __forceinline__ void gadd(__attribute__((address_space(1))) double* g, double v) {
  gadd((double*)g, v);
}
__device__ __forceinline__ void gadd(__attribute__((address_space(1))) float* g, double v) {
  gadd((float*)g, v);
}
template <typename T>
struct GAcc;
template <>
struct GAcc<double> {
  static __device__ __forceinline__ double* of(const DAdj& a) { return a.grad; }
};
template <>
struct GAcc<float> {
  static __device__ __forceinline__ float* of(const DAdj& a) { return a.g32; }
};

// grad += staging; staging = 0 (slots of the mask only)
__global__ void k_grad_flush(const DFlush* __restrict__ fl, unsigned gmask) {
  const DFlush& F = fl[blockIdx.y];
  for (int q = 0; q < 12; ++q) {
    if (!(gmask & (1u << q))) continue;
    double* g = F.grad + (long)q * F.n;
    float* h = F.g32 + (long)q * F.n;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < F.n; e += (long)gridDim.x * blockDim.x) {
      g[e] += (double)h[e];
      h[e] = 0.0f;
    }
  }
}

// lambda_{t+1}(v) += dJ/dtrace(t) at the receivers (the trace of step t is
// read from u_{t+1}).
template <typename T>
__global__ void k_el2_adj_inject(const DModel* __restrict__ models, const DShot* __restrict__ shots,
                                 const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase,
                                 int k) {
  const int t = *tbase + k;
  const int s = blockIdx.y;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DAdj& A = adj[s];
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= S.nrec || A.resid == nullptr) return;
  const DModel& M = models[S.model];
  const long n = (long)M.nx * M.nz;
  const auto q = cp<int>(S.rec) + 3 * r;
  const long c = (long)q[2] * M.nx + q[0];
  const auto res = cp<T>(A.resid) + (long)t * 2 * S.nrec + r;
  T* L = static_cast<T*>(A.lam[(t + 1) & 1]);
  atomicAdd(L + c, res[0]);
  atomicAdd(L + n + c, res[S.nrec]);
}

template <typename T, bool SPLIT>
__global__ void __launch_bounds__(NT)
k_el2_adj_v(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k,
            const int* __restrict__ tsel) {
  const int t = *tbase + k, t0 = *tbase;
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  const int lx = M.lx, lz = M.lz;
  const long SX = (long)nz * 2 * lx, SZ = (long)2 * lz * nx;
  const auto Lin = cp<T>(A.lam[(t + 1) & 1]);
  auto Lout = mp<T>(A.lam[t & 1]);
  const auto u1 = cp<T>(A.trail[*tsel]) + (long)(t + 1 - t0) * A.slot;
  const auto u0 = cp<T>(A.trail[*tsel]) + (long)(t - t0) * A.slot;
  auto W = mp<T>(A.work);
  double* G = A.grad;
  const Prof<T> P(&M.prof[0][0]);
  const bool inx = in_slab(i, nx, lx), inz = in_slab(j, nz, lz);
  const long ox = 5 * n + (inx ? (long)j * 2 * lx + slab_pos(i, nx, lx) : 0);
  const long oz = 5 * n + (SPLIT ? 6 : 4) * SX + (inz ? (long)slab_pos(j, nz, lz) * nx + i : 0);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz);
  // Dirichlet edges come last in the step: nothing flows back through them
  const bool edge = (i == 0 || i == nx - 1 || j == 0 || j == nz - 1);
  const T lvx = edge ? T(0) : Lin[c], lvz = edge ? T(0) : Lin[n + c];
  if (A.gsrc && i == S.isrc && j == S.ksrc) {  // d J / d source increment of step t
    A.gsrc[3 * (long)t + 0] = (double)lvx;
    A.gsrc[3 * (long)t + 2] = (double)lvz;
  }
  // vx(i,j) = vx * (1 - gx) + (dsxx_dx + dsxz_dz) * dt / rho, seismicfdtd.f95:317-337
  T ax1 = 0, ax2 = 0;
  if (i >= 1 && j >= 1) {
    const T w = cp<T>(M.coef[8])[c] * lvx;
    const T h1 = (u1[2 * n + c] - u1[2 * n + c - 1]) * idx;
    const T h2 = (u1[4 * n + c] - u1[4 * n + c - nx]) * idz;
    T b1 = h1, b2 = h2;
    ax1 = w;
    ax2 = w;
    if (inx) {
      const T lr = Lin[ox + 2 * SX] + w;
      ax1 = P[PK][i] * w + P[PA][i] * lr;
      Lout[ox + 2 * SX] = P[PB][i] * lr;
      b1 = P[PK][i] * h1 + u1[ox + 2 * SX];
    }
    if (inz) {
      const T lr = Lin[oz + 3 * SZ] + w;
      ax2 = P[12 + PK][j] * w + P[12 + PA][j] * lr;
      Lout[oz + 3 * SZ] = P[12 + PB][j] * lr;
      b2 = P[12 + PK][j] * h2 + u1[oz + 3 * SZ];
    }
    gadd(G + 8 * n + c, (double)lvx * (double)(b1 + b2));
    gadd(G + 10 * n + c, (double)lvx * (double)u0[c]);
    Lout[c] = (M.coef[10] ? cp<T>(M.coef[10])[c] : T(1)) * lvx;
  } else {
    if (inx) Lout[ox + 2 * SX] = Lin[ox + 2 * SX];
    if (inz) Lout[oz + 3 * SZ] = Lin[oz + 3 * SZ];
    Lout[c] = lvx;
  }
  // vz(i,j), seismicfdtd.f95:339-357
  T az1 = 0, az2 = 0;
  if (i <= nx - 2 && j <= nz - 2) {
    const T w = cp<T>(M.coef[9])[c] * lvz;
    const T k1 = (u1[4 * n + c + 1] - u1[4 * n + c]) * idx;
    const T k2 = (u1[3 * n + c + nx] - u1[3 * n + c]) * idz;
    T b1 = k1, b2 = k2;
    az1 = w;
    az2 = w;
    if (inx) {
      const T lr = Lin[ox + 3 * SX] + w;
      az1 = P[PKH][i] * w + P[PAH][i] * lr;
      Lout[ox + 3 * SX] = P[PBH][i] * lr;
      b1 = P[PKH][i] * k1 + u1[ox + 3 * SX];
    }
    if (inz) {
      const T lr = Lin[oz + 2 * SZ] + w;
      az2 = P[12 + PKH][j] * w + P[12 + PAH][j] * lr;
      Lout[oz + 2 * SZ] = P[12 + PBH][j] * lr;
      b2 = P[12 + PKH][j] * k2 + u1[oz + 2 * SZ];
    }
    gadd(G + 9 * n + c, (double)lvz * (double)(b1 + b2));
    gadd(G + 11 * n + c, (double)lvz * (double)u0[n + c]);
    Lout[n + c] = (M.coef[11] ? cp<T>(M.coef[11])[c] : T(1)) * lvz;
  } else {
    if (inx) Lout[ox + 3 * SX] = Lin[ox + 3 * SX];
    if (inz) Lout[oz + 2 * SZ] = Lin[oz + 2 * SZ];
    Lout[n + c] = lvz;
  }
  W[c] = ax1;          // adjoint of dsxx_dx at the vx node
  W[n + c] = ax2;      // adjoint of dsxz_dz at the vx node
  W[2 * n + c] = az1;  // adjoint of dsxz_dx at the vz node
  W[3 * n + c] = az2;  // adjoint of dszz_dz at the vz node
}

template <typename T, bool SPLIT>
__global__ void __launch_bounds__(NT)
k_el2_adj_s(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k,
            const int* __restrict__ tsel) {
  const int t = *tbase + k, t0 = *tbase;
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  const int lx = M.lx, lz = M.lz;
  const long SX = (long)nz * 2 * lx, SZ = (long)2 * lz * nx;
  const auto Lin = cp<T>(A.lam[(t + 1) & 1]);
  auto Lout = mp<T>(A.lam[t & 1]);
  const auto u1 = cp<T>(A.trail[*tsel]) + (long)(t + 1 - t0) * A.slot;
  const auto u0 = cp<T>(A.trail[*tsel]) + (long)(t - t0) * A.slot;
  auto W = mp<T>(A.work);
  double* G = A.grad;
  const Prof<T> P(&M.prof[0][0]);
  const bool inx = in_slab(i, nx, lx), inz = in_slab(j, nz, lz);
  const long ox = 5 * n + (inx ? (long)j * 2 * lx + slab_pos(i, nx, lx) : 0);
  const long oz = 5 * n + (SPLIT ? 6 : 4) * SX + (inz ? (long)slab_pos(j, nz, lz) * nx + i : 0);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dt = T(M.dt);
  // stresses feed the velocity update through their differences
  const T lsxx = Lin[2 * n + c] + idx * (W[c] - (i + 1 < nx ? W[c + 1] : T(0)));
  const T lszz = Lin[3 * n + c] + idz * ((j >= 1 ? W[3 * n + c - nx] : T(0)) - W[3 * n + c]);
  const T lsxz = Lin[4 * n + c] + idz * (W[n + c] - (j + 1 < nz ? W[n + c + nx] : T(0))) +
                 idx * ((i >= 1 ? W[2 * n + c - 1] : T(0)) - W[2 * n + c]);
  Lout[2 * n + c] = lsxx;
  Lout[3 * n + c] = lszz;
  Lout[4 * n + c] = lsxz;
  // adjoints of the velocity-derivative psi: shared by both stress loops
  // (A1), or the shear loop's own ones ls* in the split variant
  T lm1 = inx ? Lin[ox] : T(0), lm3 = inx ? Lin[ox + SX] : T(0);
  T lm2 = inz ? Lin[oz] : T(0), lm4 = inz ? Lin[oz + SZ] : T(0);
  T ls1 = 0, ls3 = 0, ls2 = 0, ls4 = 0;
  if (SPLIT) {
    ls1 = inx ? Lin[ox + 4 * SX] : T(0);
    ls3 = inx ? Lin[ox + 5 * SX] : T(0);
    ls2 = inz ? Lin[oz + 4 * SZ] : T(0);
    ls4 = inz ? Lin[oz + 5 * SZ] : T(0);
  }
  T& q1 = SPLIT ? ls1 : lm1;
  T& q2 = SPLIT ? ls2 : lm2;
  T& q3 = SPLIT ? ls3 : lm3;
  T& q4 = SPLIT ? ls4 : lm4;
  const long xq = SPLIT ? 4 * SX : 0, zq = SPLIT ? 4 * SZ : 0;  // shear-loop psi
  const T ikx = P[PK][i], ax = P[PA][i], bx = P[PB][i];
  const T ikxh = P[PKH][i], axh = P[PAH][i], bxh = P[PBH][i];
  const T ikz = P[12 + PK][j], az = P[12 + PA][j], bz = P[12 + PB][j];
  const T ikzh = P[12 + PKH][j], azh = P[12 + PAH][j], bzh = P[12 + PBH][j];
  // S^T: sigma_xz, seismicfdtd.f95:283-312 (psi after it is u_{t+1}'s)
  T lf1 = 0, lf2 = 0, lf3 = 0, lf4 = 0;
  if (j <= nz - 2 && i >= 1) {
    const T mu = dt * lsxz;
    const T f1 = (u0[c] - u0[c - 1]) * idx, f2 = (u0[n + c + nx] - u0[n + c]) * idz;
    const T f3 = (u0[n + c] - u0[n + c - 1]) * idx, f4 = (u0[c + nx] - u0[c]) * idz;
    const bool mono = M.coef[5] != nullptr;
    const T s15 = mono ? cp<T>(M.coef[5])[c] : T(0), s35 = mono ? cp<T>(M.coef[6])[c] : T(0);
    const T s55 = cp<T>(M.coef[7])[c];
    const T lg1 = s15 * mu, lg2 = s35 * mu, lg3 = s55 * mu;
    T g1 = f1, g2 = f2, g3 = f3, g4 = f4;
    lf1 = lg1; lf2 = lg2; lf3 = lg3; lf4 = lg3;
    if (inx) {
      g1 = ikxh * f1 + u1[ox + xq];
      T l = q1 + lg1;
      lf1 = ikxh * lg1 + axh * l;
      q1 = bxh * l;
      g3 = ikx * f3 + u1[ox + xq + SX];
      l = q3 + lg3;
      lf3 = ikx * lg3 + ax * l;
      q3 = bx * l;
    }
    if (inz) {
      g2 = ikz * f2 + u1[oz + zq];
      T l = q2 + lg2;
      lf2 = ikz * lg2 + az * l;
      q2 = bz * l;
      g4 = ikzh * f4 + u1[oz + zq + SZ];
      l = q4 + lg3;
      lf4 = ikzh * lg3 + azh * l;
      q4 = bzh * l;
    }
    const double m = (double)mu;
    gadd(G + 5 * n + c, m * (double)g1);
    gadd(G + 6 * n + c, m * (double)g2);
    gadd(G + 7 * n + c, m * ((double)g3 + (double)g4));
  }
  // N^T: sigma_xx, sigma_zz, seismicfdtd.f95:247-281 (psi before it is u_t's)
  T le1 = 0, le2 = 0, le3 = 0, le4 = 0;
  if (j >= 1 && i <= nx - 2) {
    const T mux = dt * lsxx, muz = dt * lszz;
    const T e1 = (u0[c + 1] - u0[c]) * idx, e2 = (u0[n + c] - u0[n + c - nx]) * idz;
    const T e3 = (u0[n + c + 1] - u0[n + c]) * idx, e4 = (u0[c] - u0[c - nx]) * idz;
    const bool mono = M.coef[2] != nullptr;
    const T n11 = cp<T>(M.coef[0])[c], n13 = cp<T>(M.coef[1])[c], n33 = cp<T>(M.coef[3])[c];
    const T n15 = mono ? cp<T>(M.coef[2])[c] : T(0), n35 = mono ? cp<T>(M.coef[4])[c] : T(0);
    const T ld1 = n11 * mux + n13 * muz, ld2 = n13 * mux + n33 * muz, lsh = n15 * mux + n35 * muz;
    T d1 = e1, d2 = e2, d3 = e3, d4 = e4;
    le1 = ld1; le2 = ld2; le3 = lsh; le4 = lsh;
    if (inx) {
      const T brow = SPLIT ? bxh : cp<T>(M.aux)[j];  // b_x_half(j), :255 (A2)
      d1 = ikxh * e1 + (brow * u0[ox] + axh * e1);
      T l = lm1 + ld1;
      le1 = ikxh * ld1 + axh * l;
      lm1 = brow * l;
      d3 = ikx * e3 + (bx * u0[ox + SX] + ax * e3);
      l = lm3 + lsh;
      le3 = ikx * lsh + ax * l;
      lm3 = bx * l;
    }
    if (inz) {
      d2 = ikz * e2 + (bz * u0[oz] + az * e2);
      T l = lm2 + ld2;
      le2 = ikz * ld2 + az * l;
      lm2 = bz * l;
      d4 = ikzh * e4 + (bzh * u0[oz + SZ] + azh * e4);
      l = lm4 + lsh;
      le4 = ikzh * lsh + azh * l;
      lm4 = bzh * l;
    }
    const double mx = (double)mux, mz = (double)muz, sh = (double)d3 + (double)d4;
    gadd(G + c, mx * (double)d1);
    gadd(G + n + c, mx * (double)d2 + mz * (double)d1);
    gadd(G + 2 * n + c, mx * sh);
    gadd(G + 3 * n + c, mz * (double)d2);
    gadd(G + 4 * n + c, mz * sh);
  }
  if (inx) {
    Lout[ox] = lm1;
    Lout[ox + SX] = lm3;
    if (SPLIT) {
      Lout[ox + 4 * SX] = ls1;
      Lout[ox + 5 * SX] = ls3;
    }
  }
  if (inz) {
    Lout[oz] = lm2;
    Lout[oz + SZ] = lm4;
    if (SPLIT) {
      Lout[oz + 4 * SZ] = ls2;
      Lout[oz + 5 * SZ] = ls4;
    }
  }
  W[4 * n + c] = le1;   // dvx_dx at the normal-stress node
  W[5 * n + c] = le2;   // dvz_dz
  W[6 * n + c] = le3;   // dvz_dx
  W[7 * n + c] = le4;   // dvx_dz
  W[8 * n + c] = lf1;   // dvx_dx at the shear node
  W[9 * n + c] = lf2;   // dvz_dz
  W[10 * n + c] = lf3;  // dvz_dx
  W[11 * n + c] = lf4;  // dvx_dz
}

template <typename T>
__global__ void __launch_bounds__(NT)
k_el2_adj_g(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k) {
  const int t = *tbase + k;
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  auto Lout = mp<T>(A.lam[t & 1]);
  const auto W = cp<T>(A.work);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz);
  const bool w_ = i >= 1, e_ = i + 1 < nx, n_ = j >= 1, s_ = j + 1 < nz;
  auto at = [&](int q, long o, bool ok) { return ok ? W[q * n + c + o] : T(0); };
  const T gx = idx * (at(4, -1, w_) - W[4 * n + c]) + idz * (W[7 * n + c] - at(7, nx, s_)) +
               idx * (W[8 * n + c] - at(8, 1, e_)) + idz * (at(11, -nx, n_) - W[11 * n + c]);
  const T gz = idz * (W[5 * n + c] - at(5, nx, s_)) + idx * (at(6, -1, w_) - W[6 * n + c]) +
               idz * (at(9, -nx, n_) - W[9 * n + c]) + idx * (W[10 * n + c] - at(10, 1, e_));
  Lout[c] = Lout[c] + gx;
  Lout[n + c] = Lout[n + c] + gz;
}

// ---------------------------------------------------------------------------
// Fused adjoint step: the same transpose as the three kernels above, in one
// launch.  A block holds 64 columns x AR rows of one shot, one cell per thread
// and one row per wavefront, and owns all but a ring of them (AdjOwn): V^T of
// every cell, then the stress gathers with S^T and N^T, then the velocity
// gather.  x neighbours come from the neighbouring lanes, z neighbours through
// LDS.  Blocks recompute the ring, so they are independent (lambda
// ping-pongs); only owned cells write lambda_t and add to the gradient.  The
// residual of the step is added to lambda_{t+1} as it is read.
// The interior body (and the whole EM kernel) issues all loads of a cell before
// the first use, and no load follows a store (loads and stores complete in
// order, so that a walk down the rows waits for the gradient's atomics with
// every row).  The elastic slab body still loads memory variables and their
// adjoints between its phases, after stores.  Against wavefronts
// walking tiles of 1 to 64 rows (us per step, elastic FP32 with six gradient
// slots then EM FP64 with four): 120x90 14.7 -> 10.0 and 15.8 -> 5.1, 740x440
// x 6 shots 73 -> 51 and 90 -> 53, 1064x552 x 16 shots 260 -> 209 and 322 -> 221;
// elastic FP64 16.3 -> 10.5, 133 -> 107, 423 -> 422.  Bound at the largest: 0.53
// GB of state (106 us at 5 TB/s, 186 without the gradient) and the atomics (22
// us for six slots); at the smallest three dependent scalar loads, one round
// of loads and two barriers.
// ---------------------------------------------------------------------------
// Rows of a block: 16 where two such blocks fit on a CU (elastic FP32, 64
// registers), else 8, of which two to four fit.  Measured (us per step, blocks
// of 8 / 12 / 16 rows): elastic FP32 120x90 8.4 / 9.6 / 9.9, 1064x552 x 16 shots 227
// / 231 / 203 (legacy C-PML); FP64 740x440 x 6 shots 105 / 115 / 104, 120x90 10.0 /
// 12.2 / 12.9; EM FP32 x 6 shots 29 / 31 / 29, FP64 54 / 53 / 59, 120x90 5.2 / 6.2 / 7.0.
template <typename T, bool EM>
constexpr int AR = !EM && sizeof(T) == 4 ? 16 : 8;

// Owned cells of a block: columns x0 .. x0 + w - 1, rows 1 .. h of its 64 x AR.
// The stress adjoints of a row and column need V^T one cell away, the
// velocities those of their neighbours: a ring of one cell.  The legacy C-PML
// passes the shear loop's memory adjoints on to the normal loop's, which
// reaches one cell further to the west and to the south.
template <int ROWS, bool LEGACY>
struct AdjOwn {
  static constexpr int x0 = LEGACY ? 2 : 1, w = 63 - x0, h = LEGACY ? ROWS - 3 : ROWS - 2;
};
template <typename T, bool SPLIT>
using ElAdjOwn = AdjOwn<AR<T, false>, !SPLIT>;
template <typename T>
using EmAdjOwn = AdjOwn<AR<T, true>, false>;

// Orders a wavefront's LDS accesses before and after it, lanes among each other
// (the hardware takes them in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The residuals of step t of the receivers on this wavefront's row r of the
// grid, summed per column: lane l's column is xl + l.  buf: 2 x 64 of the
// wavefront's own.
template <typename T>
__device__ __forceinline__ void adj_residual(const DShot& S, const DAdj& A, int t, int r, int xl, int lane,
                                             T* b0, T* b1, T& a0, T& a1) {
  const int q0 = S.rrow[r], q1 = S.rrow[r + 1];
  if (q1 <= q0) return;
  const auto res = cp<T>(A.resid) + (long)t * 2 * S.nrec;
  b0[lane] = 0;
  b1[lane] = 0;
  wave_lds_fence();
  for (int e = q0 + lane; e < q1; e += 64) {
    const int l = S.rxid[2 * e] - xl, id = S.rxid[2 * e + 1];
    if (l >= 0 && l < 64) {
      atomicAdd(&b0[l], res[id]);
      atomicAdd(&b1[l], res[S.nrec + id]);
    }
  }
  wave_lds_fence();
  a0 += b0[lane];
  a1 += b1[lane];
}

template <typename T>
struct ElAdjLds {
  static constexpr int R = AR<T, false>;
  T u[4][R][64];   // u_t's vx, vz; u_{t+1}'s sxz, szz
  T bd[2][R][64];  // V^T: adjoints of dsxz_dz (at vx), dszz_dz (at vz)
  T ef[4][R][64];  // stress phase: adjoints of dvz_dz, dvx_dz (normal), dvz_dz, dvx_dz (shear)
};

// PML false: no cell of the block lies in a slab or outside the grid's inner cells.
template <typename T, bool SPLIT, bool PML>
__device__ __forceinline__ void el2_adj_block(const DModel& M, const DShot& S, const DAdj& A, const int x0,
                                              const int z0, const int t, const int t0, const int tb,
                                              const unsigned gmask, ElAdjLds<T>& L) {
  using Own = ElAdjOwn<T, SPLIT>;
  constexpr int R = AR<T, false>;
  const int nx = M.nx, nz = M.nz, lx = M.lx, lz = M.lz;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = x0 + lane, r = z0 + w;
  const bool in = !PML || (i >= 0 && i < nx && r >= 0 && r < nz);
  const int ic = PML ? min(max(i, 0), nx - 1) : i, rc = PML ? min(max(r, 0), nz - 1) : r;
  const bool own = in && lane >= Own::x0 && lane < Own::x0 + Own::w && w >= 1 && w <= Own::h;
  // 32-bit element offsets within one state / gradient array (checked at setup)
  const uint32_t n = (uint32_t)nx * nz, c = (uint32_t)rc * nx + ic;
  const A32<const T> Li(A.lam[(t + 1) & 1]);
  const A32<T> Lo(A.lam[t & 1]);
  const T* trail = static_cast<const T*>(A.trail[tb]);
  const A32<const T> u1(trail + (long)(t + 1 - t0) * A.slot), u0(trail + (long)(t - t0) * A.slot);
  T lvx = Li[c], lvz = Li[n + c];
  T lsxx = Li[2 * n + c], lszz = Li[3 * n + c], lsxz = Li[4 * n + c];
  const T sxx1 = u1[2 * n + c], szz1 = u1[3 * n + c], sxz1 = u1[4 * n + c];
  const T vx = u0[c], vz = u0[n + c];
  const bool mono = M.coef[2] != nullptr, atten = M.coef[10] != nullptr;
  const T dtx = A32<const T>(M.coef[8])[c], dtz = A32<const T>(M.coef[9])[c];
  const T omx = atten ? A32<const T>(M.coef[10])[c] : T(1), omz = atten ? A32<const T>(M.coef[11])[c] : T(1);
  const T n11 = A32<const T>(M.coef[0])[c], n13 = A32<const T>(M.coef[1])[c], n33 = A32<const T>(M.coef[3])[c];
  const T s55 = A32<const T>(M.coef[7])[c];
  const T n15 = mono ? A32<const T>(M.coef[2])[c] : T(0), n35 = mono ? A32<const T>(M.coef[4])[c] : T(0);
  const T s15 = mono ? A32<const T>(M.coef[5])[c] : T(0), s35 = mono ? A32<const T>(M.coef[6])[c] : T(0);
  // memory variables: offsets, and profiles of the column and of the row
  const bool inx = PML && in && in_slab(i, nx, lx), inz = PML && in && in_slab(r, nz, lz);
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const uint32_t ox = 5 * n + (inx ? (uint32_t)r * 2 * lx + slab_pos(i, nx, lx) : 0);
  const uint32_t oz = 5 * n + (SPLIT ? 6 : 4) * SX + (inz ? (uint32_t)slab_pos(r, nz, lz) * nx + i : 0);
  const Prof<T> P(&M.prof[0][0]);
  T ikx = 0, ax = 0, bx = 0, ikxh = 0, axh = 0, bxh = 0, ikz = 0, az = 0, bz = 0, ikzh = 0, azh = 0, bzh = 0;
  if (inx) {
    ikx = P[PK][ic]; ax = P[PA][ic]; bx = P[PB][ic];
    ikxh = P[PKH][ic]; axh = P[PAH][ic]; bxh = P[PBH][ic];
  }
  if (inz) {
    ikz = P[12 + PK][rc]; az = P[12 + PA][rc]; bz = P[12 + PB][rc];
    ikzh = P[12 + PKH][rc]; azh = P[12 + PAH][rc]; bzh = P[12 + PBH][rc];
  }
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dt = T(M.dt);
  const A32<typename std::remove_pointer<decltype(GAcc<T>::of(A))>::type> G(GAcc<T>::of(A));
  if (S.nrec > 0 && A.resid && r >= 0 && r < nz)
    adj_residual<T>(S, A, t, r, x0, lane, L.ef[0][w], L.ef[1][w], lvx, lvz);

  // ---- V^T: velocity updates, seismicfdtd.f95:317-375 ----
  const bool edge = PML && (i <= 0 || i >= nx - 1 || r <= 0 || r >= nz - 1);
  if (edge) lvx = lvz = 0;
  if (own && i == S.isrc && r == S.ksrc && A.gsrc) {
    A.gsrc[3 * (long)t + 0] = (double)lvx;
    A.gsrc[3 * (long)t + 2] = (double)lvz;
  }
  const bool dox = !PML || (in && i >= 1 && r >= 1), doz = !PML || (in && i <= nx - 2 && r <= nz - 2);
  T An = 0, Bn = 0, Cn = 0, Dn = 0, pvx = lvx, pvz = lvz;
  if (dox) {
    const T q = dtx * lvx;
    An = q;
    Bn = q;
    pvx = omx * lvx;
    if (inx) {
      const T lr = Li[ox + 2 * SX] + q;
      An = ikx * q + ax * lr;
      if (own) Lo[ox + 2 * SX] = bx * lr;
    }
    if (inz) {
      const T lr = Li[oz + 3 * SZ] + q;
      Bn = ikz * q + az * lr;
      if (own) Lo[oz + 3 * SZ] = bz * lr;
    }
  } else if (own) {
    if (inx) Lo[ox + 2 * SX] = Li[ox + 2 * SX];
    if (inz) Lo[oz + 3 * SZ] = Li[oz + 3 * SZ];
  }
  if (doz) {
    const T q = dtz * lvz;
    Cn = q;
    Dn = q;
    pvz = omz * lvz;
    if (inx) {
      const T lr = Li[ox + 3 * SX] + q;
      Cn = ikxh * q + axh * lr;
      if (own) Lo[ox + 3 * SX] = bxh * lr;
    }
    if (inz) {
      const T lr = Li[oz + 2 * SZ] + q;
      Dn = ikzh * q + azh * lr;
      if (own) Lo[oz + 2 * SZ] = bzh * lr;
    }
  } else if (own) {
    if (inx) Lo[ox + 3 * SX] = Li[ox + 3 * SX];
    if (inz) Lo[oz + 2 * SZ] = Li[oz + 2 * SZ];
  }
  L.u[0][w][lane] = vx;
  L.u[1][w][lane] = vz;
  L.u[2][w][lane] = sxz1;
  L.u[3][w][lane] = szz1;
  L.bd[0][w][lane] = Bn;
  L.bd[1][w][lane] = Dn;
  __syncthreads();

  // ---- stresses: gathers, then S^T and N^T, :247-312 ----
  const int wu = w > 0 ? w - 1 : 0, wd = w < R - 1 ? w + 1 : R - 1;
  const T A_e = dpp_next(An), C_w = dpp_prev(Cn);
  const T vx_w = dpp_prev(vx), vz_w = dpp_prev(vz), vx_e = dpp_next(vx), vz_e = dpp_next(vz);
  const T sxx_w = dpp_prev(sxx1), sxz_e = dpp_next(sxz1);
  lsxx += idx * (An - A_e);
  lszz += idz * (L.bd[1][wu][lane] - Dn);
  lsxz += idz * (Bn - L.bd[0][wd][lane]) + idx * (C_w - Cn);
  if (own) {
    if (dox) {
      T b1 = (sxx1 - sxx_w) * idx, b2 = (sxz1 - L.u[2][wu][lane]) * idz;
      if (inx) b1 = ikx * b1 + u1[ox + 2 * SX];
      if (inz) b2 = ikz * b2 + u1[oz + 3 * SZ];
      if (gmask & (1u << 8)) gadd(&G[8 * n + c], (double)lvx * (double)(b1 + b2));
      if (gmask & (1u << 10)) gadd(&G[10 * n + c], (double)lvx * (double)vx);
    }
    if (doz) {
      T b1 = (sxz_e - sxz1) * idx, b2 = (L.u[3][wd][lane] - szz1) * idz;
      if (inx) b1 = ikxh * b1 + u1[ox + 3 * SX];
      if (inz) b2 = ikzh * b2 + u1[oz + 2 * SZ];
      if (gmask & (1u << 9)) gadd(&G[9 * n + c], (double)lvz * (double)(b1 + b2));
      if (gmask & (1u << 11)) gadd(&G[11 * n + c], (double)lvz * (double)vz);
    }
    Lo[2 * n + c] = lsxx;
    Lo[3 * n + c] = lszz;
    Lo[4 * n + c] = lsxz;
  }
  T E1 = 0, E2 = 0, E3 = 0, E4 = 0, F1 = 0, F2 = 0, F3 = 0, F4 = 0;
  const bool dos = !PML || (in && r <= nz - 2 && i >= 1), don = !PML || (in && r >= 1 && i <= nx - 2);
  // memory adjoints: the shear loop's own four if split, then the normal
  // loop's; one set for both loops otherwise
  const uint32_t xq = SPLIT ? 4 * SX : 0, zq = SPLIT ? 4 * SZ : 0;
  T q1 = 0, q2 = 0, q3 = 0, q4 = 0;
  if (inx) { q1 = Li[ox + xq]; q3 = Li[ox + xq + SX]; }
  if (inz) { q2 = Li[oz + zq]; q4 = Li[oz + zq + SZ]; }
  if (dos) {  // S^T
    const T mu = dt * lsxz;
    T g1 = (vx - vx_w) * idx, g2 = (L.u[1][wd][lane] - vz) * idz;
    T g3 = (vz - vz_w) * idx, g4 = (L.u[0][wd][lane] - vx) * idz;
    const T lg1 = s15 * mu, lg2 = s35 * mu, lg3 = s55 * mu;
    F1 = lg1; F2 = lg2; F3 = lg3; F4 = lg3;
    if (inx) {
      T l = q1 + lg1;
      F1 = ikxh * lg1 + axh * l;
      q1 = bxh * l;
      l = q3 + lg3;
      F3 = ikx * lg3 + ax * l;
      q3 = bx * l;
    }
    if (inz) {
      T l = q2 + lg2;
      F2 = ikz * lg2 + az * l;
      q2 = bz * l;
      l = q4 + lg3;
      F4 = ikzh * lg3 + azh * l;
      q4 = bzh * l;
    }
    if (own) {
      if (inx) {
        g1 = ikxh * g1 + u1[ox + xq];
        g3 = ikx * g3 + u1[ox + xq + SX];
      }
      if (inz) {
        g2 = ikz * g2 + u1[oz + zq];
        g4 = ikzh * g4 + u1[oz + zq + SZ];
      }
      if (gmask & (1u << 5)) gadd(&G[5 * n + c], (double)mu * (double)g1);
      if (gmask & (1u << 6)) gadd(&G[6 * n + c], (double)mu * (double)g2);
      if (gmask & (1u << 7)) gadd(&G[7 * n + c], (double)mu * ((double)g3 + (double)g4));
    }
  }
  if (SPLIT) {
    if (own && inx) { Lo[ox + xq] = q1; Lo[ox + xq + SX] = q3; }
    if (own && inz) { Lo[oz + zq] = q2; Lo[oz + zq + SZ] = q4; }
    if (inx) { q1 = Li[ox]; q3 = Li[ox + SX]; }
    if (inz) { q2 = Li[oz]; q4 = Li[oz + SZ]; }
  }
  if (don) {  // N^T
    const T mux = dt * lsxx, muz = dt * lszz;
    const T ld1 = n11 * mux + n13 * muz, ld2 = n13 * mux + n33 * muz, lsh = n15 * mux + n35 * muz;
    T d1 = (vx_e - vx) * idx, d2 = (vz - L.u[1][wu][lane]) * idz;
    T d3 = (vz_e - vz) * idx, d4 = (vx - L.u[0][wu][lane]) * idz;
    E1 = ld1; E2 = ld2; E3 = lsh; E4 = lsh;
    // (the legacy normal loop's decay of memory_dvx_dx: b_x_half by row, :255)
    T bxn = bxh;
    if (inx) {
      if (!SPLIT) bxn = cp<T>(M.aux)[rc];
      T l = q1 + ld1;
      E1 = ikxh * ld1 + axh * l;
      q1 = bxn * l;
      l = q3 + lsh;
      E3 = ikx * lsh + ax * l;
      q3 = bx * l;
    }
    if (inz) {
      T l = q2 + ld2;
      E2 = ikz * ld2 + az * l;
      q2 = bz * l;
      l = q4 + lsh;
      E4 = ikzh * lsh + azh * l;
      q4 = bzh * l;
    }
    if (own) {
      if (inx) {
        d1 = ikxh * d1 + (bxn * u0[ox] + axh * d1);
        d3 = ikx * d3 + (bx * u0[ox + SX] + ax * d3);
      }
      if (inz) {
        d2 = ikz * d2 + (bz * u0[oz] + az * d2);
        d4 = ikzh * d4 + (bzh * u0[oz + SZ] + azh * d4);
      }
      const double mx = (double)mux, mz = (double)muz, sh = (double)d3 + (double)d4;
      if (gmask & (1u << 0)) gadd(&G[c], mx * (double)d1);
      if (gmask & (1u << 1)) gadd(&G[n + c], mx * (double)d2 + mz * (double)d1);
      if (gmask & (1u << 2)) gadd(&G[2 * n + c], mx * sh);
      if (gmask & (1u << 3)) gadd(&G[3 * n + c], mz * (double)d2);
      if (gmask & (1u << 4)) gadd(&G[4 * n + c], mz * sh);
    }
  }
  if (own && inx) { Lo[ox] = q1; Lo[ox + SX] = q3; }
  if (own && inz) { Lo[oz] = q2; Lo[oz + SZ] = q4; }
  L.ef[0][w][lane] = E2;
  L.ef[1][w][lane] = E4;
  L.ef[2][w][lane] = F2;
  L.ef[3][w][lane] = F4;
  __syncthreads();

  // ---- velocities: gather of the stress-phase adjoints ----
  const T E1_w = dpp_prev(E1), E3_w = dpp_prev(E3), F1_e = dpp_next(F1), F3_e = dpp_next(F3);
  if (own) {
    Lo[c] = pvx + idx * (E1_w - E1) + idz * (E4 - L.ef[1][wd][lane]) + idx * (F1 - F1_e) +
            idz * (L.ef[3][wu][lane] - F4);
    Lo[n + c] = pvz + idz * (E2 - L.ef[0][wd][lane]) + idx * (E3_w - E3) + idz * (L.ef[2][wu][lane] - F2) +
                idx * (F3 - F3_e);
  }
}

// Whether the block at (x0, z0) avoids every slab and the grid's outer cells:
// it runs the body without memory variables and edge predicates.
__device__ __forceinline__ bool adj_interior(const DModel& M, int x0, int z0, int rows) {
  return x0 >= max(M.lx, 1) && x0 + 64 <= M.nx - max(M.lx, 2) && z0 >= max(M.lz, 1) &&
         z0 + rows <= M.nz - max(M.lz, 2);
}

template <typename T, bool SPLIT>
__global__ void __launch_bounds__((64 * AR<T, false>), sizeof(T) == 4 ? 8 : 4)
k_el2_adj(const DModel* __restrict__ models, const DShot* __restrict__ shots, const DAdj* __restrict__ adj,
          const int4* __restrict__ work, int nitems, const int* __restrict__ tbase, int k, unsigned gmask,
          const int* __restrict__ tsel) {
  __shared__ ElAdjLds<T> L;
  const int q = item8(nitems);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const int t0 = __builtin_amdgcn_readfirstlane(*tbase), tb = __builtin_amdgcn_readfirstlane(*tsel);
  const DModel& M = models[__builtin_amdgcn_readfirstlane(wv.w)];
  const int x0 = __builtin_amdgcn_readfirstlane(wv.y) - ElAdjOwn<T, SPLIT>::x0;
  const int z0 = __builtin_amdgcn_readfirstlane(wv.z) - 1;
  if (adj_interior(M, x0, z0, AR<T, false>))
    el2_adj_block<T, SPLIT, false>(M, shots[s], adj[s], x0, z0, t0 + k, t0, tb, gmask, L);
  else
    el2_adj_block<T, SPLIT, true>(M, shots[s], adj[s], x0, z0, t0 + k, t0, tb, gmask, L);
}

// ===========================================================================
// EM2: electromag2, legacy/fortran/electromagfdtd.f95:10-326, one pass per
// step.  psi slabs: x [nz][2lx]: dEz_dx dHy_dx ; z [2lz][nx]: dEx_dz dHy_dz.
// fields: Ex (nx-1 x nz), Ez (nx x nz-1), Hy (nx-1 x nz-1) stored nx*nz.
// A wavefront owns columns xo..xo+EW-1 (lanes 1..EW) of rows zo..zo+eh-1 and
// walks down z: at row r it updates Hy of row r from the old Ex of rows r and
// r+1 and the old Ez of columns i and i+1 (:249-266), then Ex and Ez of row r
// from the new Hy of rows r-1 and r and of columns i-1 and i (:273-295), then
// the source (:300-301) and the Dirichlet edges (:304-311).  The new Hy of
// row zo-1 is recomputed, so tiles are independent; the state ping-pongs
// between buffers A and B like the 2-D elastic one.  The Hy zeroing that ends
// each legacy step (:312-315) is applied by the next update, which reads a
// boundary Hy as 0, and by k_em2_edges at the end of a run.
// Every fused multiply-add is written out (contraction off).
// ===========================================================================
template <typename T, bool PML>
__device__ __forceinline__ void em2_tile(const DModel* __restrict__ models,
                                         const DShot* __restrict__ shots, const int4 wi, const int it,
                                         const int lane, const int eh, const int par) {
#pragma clang fp contract(off)
  const DShot& S = shots[wi.x];
  const DModel& M = models[S.model];
  const int nx = M.nx, nz = M.nz;
  const int xo = wi.y, zo = wi.z;
  const int i = xo - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);  // clamped column: every load stays in bounds
  const bool own = incol && lane >= 1 && lane <= EW;
  const int zend = min(zo + eh, nz);
  const bool has_rec = S.nrec > 0 && S.rrow[zend] > S.rrow[zo];  // receivers on own rows
  const long nn = (long)nx * nz;
  const A32<const T> exi(par ? S.g[0] : S.f[0]);
  const A32<const T> ezi(par ? S.g[1] : S.f[1]);
  const A32<const T> hyi(par ? S.g[2] : S.f[2]);
  const A32<T> exo(par ? S.f[0] : S.g[0]);
  const A32<T> ezo(par ? S.f[1] : S.g[1]);
  const A32<T> hyo(par ? S.f[2] : S.g[2]);
  const A32<const T> pin(par ? S.psi2 : S.psi);
  const A32<T> pout(par ? S.psi : S.psi2);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dbh = T(M.scal[0]);
  const int lx = M.lx, lz = M.lz;
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const bool inx = PML && incol && in_slab(i, nx, lx);
  const int xs = inx ? slab_pos(i, nx, lx) : 0;
  const Prof<T> P(&M.prof[0][0]);
  const T ikx = P[PK][ic], ax = P[PA][ic], bx = P[PB][ic];
  const T ikxh = P[PKH][ic], axh = P[PAH][ic], bxh = P[PBH][ic];
  const auto ikz = P[12 + PK], az = P[12 + PA], bz = P[12 + PB];
  const auto ikzh = P[12 + PKH], azh = P[12 + PAH], bzh = P[12 + PBH];
  const A32<const T> CAX(M.coef[0]), CBX(M.coef[1]), CAZ(M.coef[2]), CBZ(M.coef[3]);
  const bool hcol = incol && i <= nx - 2;                  // Hy, Ex columns
  const bool ezcol = incol && i >= 1 && i <= nx - 2;       // Ez columns
  const bool is_src_col = (i == S.isrc);
  const int ksrc = S.ksrc;
  const auto srcx = cp<T>(S.src[0]), srcz = cp<T>(S.src[2]);
  const T incx = (srcx != nullptr) ? srcx[it] : T(0);
  const T incz = (srcz != nullptr) ? srcz[it] : T(0);

  auto row = [&](int r) { return (uint32_t)(r < 0 ? 0 : (r >= nz ? nz - 1 : r)) * nx + ic; };
  auto valid = [&](int r) { return incol && r >= 0 && r < nz; };
  T ex_c = valid(zo - 1) ? exi[row(zo - 1)] : T(0);  // old Ex of row r
  T hy_p = 0;                                         // new Hy of row r-1
  for (int r = zo - 1; r < zend; ++r) {
    const uint32_t c = row(r);
    const bool rv = valid(r);
    const T ld_exn = exi[row(r + 1)], ld_ez = ezi[c], ld_hy = hyi[c];
    const T cax = CAX[c], cbx = CBX[c], caz = CAZ[c], cbz = CBZ[c];
    const int rs = r < 0 ? 0 : (r >= nz ? nz - 1 : r);
    const bool inz = PML && in_slab(rs, nz, lz), inzc = incol && inz;
    const uint32_t ox = (uint32_t)rs * 2 * lx + xs;
    const uint32_t oz = 2 * SX + (inz ? (uint32_t)slab_pos(rs, nz, lz) * nx + ic : 0);
    T m_ezx = inx ? pin[ox] : T(0);        // dEz_dx
    T m_hyx = inx ? pin[SX + ox] : T(0);   // dHy_dx
    T m_exz = inzc ? pin[oz] : T(0);       // dEx_dz
    T m_hyz = inzc ? pin[SZ + oz] : T(0);  // dHy_dz
    const T ex_n = valid(r + 1) ? ld_exn : T(0);
    const T ez_c = rv ? ld_ez : T(0);
    const T hy_o = rv ? ld_hy : T(0);

    // ---- Hy of row r (:249-266) ----
    const T ez_e = lane_next(ez_c);  // Ez(i+1, r)
    T hy = hy_o;
    if (rv && hcol && r <= nz - 2) {
      T a = (ex_n - ex_c) * idz;
      if (inz) {
        m_exz = fma(bz[rs], m_exz, az[rs] * a);
        a = fma(a, ikz[rs], m_exz);
      }
      T b = (ez_e - ez_c) * idx;
      if (inx) {
        m_ezx = fma(bx, m_ezx, ax * b);
        b = fma(b, ikx, m_ezx);
      }
      const bool edge = (i == 0 || i == nx - 2 || r == 0 || r == nz - 2);  // :312-315 of the last step
      hy = fma(dbh, b + a, edge ? T(0) : hy_o);
    }

    // ---- Ex, Ez of row r (:273-295), source, Dirichlet ----
    const T hy_w = lane_prev(hy);  // new Hy(i-1, r)
    T gex = 0, gez = 0;  // new E of the owned cells (receiver samples)
    if (own && rv && r >= zo) {
      T ex = ex_c, ez = ez_c;
      if (hcol && r >= 1 && r <= nz - 2) {
        T d = (hy - hy_p) * idz;
        if (inz) {
          m_hyz = fma(bzh[rs], m_hyz, azh[rs] * d);
          d = fma(d, ikzh[rs], m_hyz);
        }
        ex = fma(cax, ex, cbx * d);
      }
      if (ezcol && r <= nz - 2) {
        T d = (hy - hy_w) * idx;
        if (inx) {
          m_hyx = fma(bxh, m_hyx, axh * d);
          d = fma(d, ikxh, m_hyx);
        }
        ez = fma(caz, ez, cbz * d);
      }
      if (is_src_col && r == ksrc) { ex += incx; ez += incz; }
      if (i == 0 || i == nx - 2 || r == 0 || r == nz - 1) ex = 0;
      if (i == 0 || i == nx - 1 || r == 0 || r == nz - 2) ez = 0;
      if (i == nx - 1) ex = 0;  // outside the (nx-1) x nz Ex array
      if (r == nz - 1) ez = 0;  // outside the nx x (nz-1) Ez array
      check_blowup((double)ex * ex + (double)ez * ez, S.blowup, it);
      exo[c] = ex;
      ezo[c] = ez;
      hyo[c] = hy;
      gex = ex;
      gez = ez;
      if (inx) { pout[ox] = m_ezx; pout[SX + ox] = m_hyx; }
      if (inz) { pout[oz] = m_exz; pout[SZ + oz] = m_hyz; }
    }
    if (has_rec && r >= zo) gather_row<T>(S, r, it, lane, xo - 1, 1, EW, gex, gez);
    hy_p = hy;
    ex_c = ex_n;
  }
}

// Same work list and launch shape as k_el2_step, and the same buffer
// choice (prun: the single step that ends a run of two-step launches).
template <typename T, int WB>
__global__ void __launch_bounds__(64 * WB)
k_em2_step(const DModel* __restrict__ models, const DShot* __restrict__ shots,
           const int4* __restrict__ work, int nitems, const int* __restrict__ base, int rel,
           int eh, const int* __restrict__ prun) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = __builtin_amdgcn_readfirstlane(*base + rel);
  const int par = prun ? __builtin_amdgcn_readfirstlane(((it - *prun) >> 1) & 1) : (it & 1);
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const int4 wv = work[w];
    const int4 wi = make_int4(__builtin_amdgcn_readfirstlane(wv.x),
                              __builtin_amdgcn_readfirstlane(wv.y) + wave * EW,
                              __builtin_amdgcn_readfirstlane(wv.z), 0);
    if (wi.x < 0) continue;
    const DModel& M = models[shots[wi.x].model];
    if (wi.y >= M.nx) continue;
    // columns (halo included) and rows zo-1 .. zo+eh-1 clear of every slab
    const bool interior = wi.y - 1 >= M.lx && wi.y + 62 < M.nx - M.lx && wi.z - 1 >= M.lz &&
                          wi.z + eh <= M.nz - M.lz;
    if (interior)
      em2_tile<T, false>(models, shots, wi, it, threadIdx.x & 63, eh, par);
    else
      em2_tile<T, true>(models, shots, wi, it, threadIdx.x & 63, eh, par);
  }
}

// ===========================================================================
// EM2, two time steps per launch: the walk of k_em2_step with the second
// step one row behind the first.  At row r a wavefront computes
//   A  Hy of step it at row r        (E of it-1, rows r, r+1)
//   B  Ex, Ez of step it at row r     (Hy from A, rows r-1, r)
//   C  Hy of step it+1 at row r-1     (E from B, rows r-1, r)
//   D  Ex, Ez of step it+1 at row r-1 (Hy from C, rows r-2, r-1)
// so the state of step it lives only in registers.  One step makes a cell
// depend on columns i-1 .. i+1 and rows k-1 .. k+1 of the previous state,
// so lane l holds column xo - 2 + l, lanes 2 .. 2+EW2E-1 are exact after two
// steps, and rows zo-2 .. zo+eh read produce rows zo .. zo+eh-1.  The
// expressions are those of k_em2_step in the same order (identical bits),
// the Hy zeroing that ends step it is applied where step it+1 reads it, and
// the receiver samples of both steps are written here.  Buffers as in
// k_el2_step2.
// ===========================================================================
constexpr int EW2E = 60;

template <typename T, bool PML>
__device__ __forceinline__ void em2x2_tile(const DModel* __restrict__ models,
                                           const DShot* __restrict__ shots, const int4 wi, const int it,
                                           const int q, const int lane, const int eh) {
#pragma clang fp contract(off)
  // interior waves read only columns 1..nx-3 and rows 1..nz-3 outside the
  // C-PML slabs: every edge condition holds on every lane
  constexpr bool INT = !PML;
  const DShot& S = shots[wi.x];
  const DModel& M = models[S.model];
  const int nx = M.nx, nz = M.nz;
  const int xo = wi.y, zo = wi.z;
  const int i = xo - 2 + lane;
  const bool incol = INT || (i >= 0 && i < nx);
  const int ic = INT ? i : (incol ? i : (i < 0 ? 0 : nx - 1));  // clamped column
  const bool own = incol && lane >= 2 && lane < 2 + EW2E;
  const int ze = min(zo + eh, nz);
  const A32<const T> exi(q ? S.g[0] : S.f[0]);
  const A32<const T> ezi(q ? S.g[1] : S.f[1]);
  const A32<const T> hyi(q ? S.g[2] : S.f[2]);
  const A32<T> exo(q ? S.f[0] : S.g[0]);
  const A32<T> ezo(q ? S.f[1] : S.g[1]);
  const A32<T> hyo(q ? S.f[2] : S.g[2]);
  const A32<const T> pin(q ? S.psi2 : S.psi);
  const A32<T> pout(q ? S.psi : S.psi2);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dbh = T(M.scal[0]);
  const int lx = M.lx, lz = M.lz;
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const bool inx = PML && incol && in_slab(i, nx, lx);
  const int xs = inx ? slab_pos(i, nx, lx) : 0;
  const Prof<T> P(&M.prof[0][0]);
  const T ikx = P[PK][ic], ax = P[PA][ic], bx = P[PB][ic];
  const T ikxh = P[PKH][ic], axh = P[PAH][ic], bxh = P[PBH][ic];
  const auto ikz = kp<T>(M.prof[2][PK]), az = kp<T>(M.prof[2][PA]), bz = kp<T>(M.prof[2][PB]);
  const auto ikzh = kp<T>(M.prof[2][PKH]), azh = kp<T>(M.prof[2][PAH]), bzh = kp<T>(M.prof[2][PBH]);
  const A32<const T> CAX(M.coef[0]), CBX(M.coef[1]), CAZ(M.coef[2]), CBZ(M.coef[3]);
  const bool hcol = INT || (incol && i <= nx - 2);              // Hy, Ex columns
  const bool ezcol = INT || (incol && i >= 1 && i <= nx - 2);   // Ez columns
  const bool is_src_col = (i == S.isrc);
  const int ksrc = S.ksrc;
  const auto srcx = cp<T>(S.src[0]), srcz = cp<T>(S.src[2]);
  const T incx0 = srcx ? srcx[it] : T(0), incx1 = srcx ? srcx[it + 1] : T(0);
  const T incz0 = srcz ? srcz[it] : T(0), incz1 = srcz ? srcz[it + 1] : T(0);

  auto crow = [&](int r) { return r < 0 ? 0 : (r >= nz ? nz - 1 : r); };
  auto cell = [&](int r) { return (uint32_t)crow(r) * nx + ic; };
  auto valid = [&](int r) { return INT || (incol && r >= 0 && r < nz); };
  auto inzs = [&](int r) { return PML && in_slab(crow(r), nz, lz); };

  struct MX { T ezx, hyx, exz, hyz; };  // memory: dEz/dx, dHy/dx (x slab); dEx/dz, dHy/dz (z slab)
  struct CE { T cax, cbx, caz, cbz; };
  auto offx = [&](int r) { return inx ? (uint32_t)crow(r) * 2 * lx + xs : 0u; };
  auto offz = [&](int r) { return 2 * SX + (inzs(r) ? (uint32_t)slab_pos(crow(r), nz, lz) * nx + ic : 0u); };
  auto load_m = [&](int r) {
    MX m{};
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      const bool inzc = incol && inzs(r);
      m.ezx = inx ? pin[ox] : T(0);
      m.hyx = inx ? pin[SX + ox] : T(0);
      m.exz = inzc ? pin[oz] : T(0);
      m.hyz = inzc ? pin[SZ + oz] : T(0);
    }
    return m;
  };
  auto store_m = [&](int r, const MX& m) {  // own cells only
    if constexpr (PML) {
      const uint32_t ox = offx(r), oz = offz(r);
      if (inx) { pout[ox] = m.ezx; pout[SX + ox] = m.hyx; }
      if (inzs(r)) { pout[oz] = m.exz; pout[SZ + oz] = m.hyz; }
    }
  };
  // Hy of one step at row r (electromagfdtd.f95:249-266): the previous step's
  // Ex of rows r, r+1, Ez of row r (columns i, i+1) and Hy of row r
  auto hfield = [&](int r, T ex_c, T ex_n, T ez_c, T hy_o, MX& m) {
    const T ez_e = dpp_next(ez_c);  // Ez(i+1, r)
    const bool rv = valid(r);
    const int rs = crow(r);
    const bool inz = PML && in_slab(rs, nz, lz);
    T hy = hy_o;
    if (INT || (rv && hcol && r <= nz - 2)) {
      T a = (ex_n - ex_c) * idz;
      if (PML && inz) {
        m.exz = fma(bz[rs], m.exz, az[rs] * a);
        a = fma(a, ikz[rs], m.exz);
      }
      T b = (ez_e - ez_c) * idx;
      if (PML && inx) {
        m.ezx = fma(bx, m.ezx, ax * b);
        b = fma(b, ikx, m.ezx);
      }
      const bool edge = !INT && (i == 0 || i == nx - 2 || r == 0 || r == nz - 2);  // :312-315
      hy = fma(dbh, b + a, edge ? T(0) : hy_o);
    }
    return hy;
  };
  // Ex, Ez of one step at row r (:273-295), source, Dirichlet: the new Hy of
  // rows r-1, r (column i-1 for Ez)
  auto efield = [&](int r, T hy, T hy_p, T ex_c, T ez_c, const CE& k, MX& m, T ix, T iz, T& ex, T& ez) {
    const T hy_w = dpp_prev(hy);  // new Hy(i-1, r)
    const bool rv = valid(r);
    const int rs = crow(r);
    const bool inz = PML && in_slab(rs, nz, lz);
    ex = ex_c;
    ez = ez_c;
    if (INT || (rv && hcol && r >= 1 && r <= nz - 2)) {
      T d = (hy - hy_p) * idz;
      if (PML && inz) {
        m.hyz = fma(bzh[rs], m.hyz, azh[rs] * d);
        d = fma(d, ikzh[rs], m.hyz);
      }
      ex = fma(k.cax, ex, k.cbx * d);
    }
    if (INT || (rv && ezcol && r <= nz - 2)) {
      T d = (hy - hy_w) * idx;
      if (PML && inx) {
        m.hyx = fma(bxh, m.hyx, axh * d);
        d = fma(d, ikxh, m.hyx);
      }
      ez = fma(k.caz, ez, k.cbz * d);
    }
    if (r == ksrc && is_src_col) { ex += ix; ez += iz; }
    if (!INT) {
      if (i == 0 || i == nx - 2 || r == 0 || r == nz - 1) ex = 0;
      if (i == 0 || i == nx - 1 || r == 0 || r == nz - 2) ez = 0;
      if (i == nx - 1) ex = 0;  // outside the (nx-1) x nz Ex array
      if (r == nz - 1) ez = 0;  // outside the nx x (nz-1) Ez array
      if (!rv) { ex = 0; ez = 0; }
    }
  };
  const int nrec = S.nrec;
  auto gather = [&](int b, int itn, T ex, T ez) { gather_row<T>(S, b, itn, lane, xo - 2, 2, 1 + EW2E, ex, ez); };

  T ex0_c = valid(zo - 2) ? exi[cell(zo - 2)] : T(0);  // Ex of step it-1, row r
  T hy1_p = 0;                                          // Hy of step it, row r-1
  T ex1_p = 0, ez1_p = 0;                               // E of step it, row r-1
  T hy2_p = 0;                                          // Hy of step it+1, row r-2
  CE k_p{};                                             // coefficients of row r-1
  MX m_p{};                                             // memory of row r-1 after step it
  const bool has_rec = nrec > 0 && S.rrow[ze] > S.rrow[zo];  // receivers on own rows (per tile)
  bool bad0 = false, bad1 = false;

  // every load of row r (addresses clamped in bounds)
  struct Row { T exn, ez, hy; CE k; MX m; };
  auto load_row = [&](int r) {
    Row L;
    const uint32_t c = cell(r);
    L.exn = exi[cell(r + 1)];
    L.ez = ezi[c];
    L.hy = hyi[c];
    L.k.cax = CAX[c];
    L.k.cbx = CBX[c];
    L.k.caz = CAZ[c];
    L.k.cbz = CBZ[c];
    L.m = load_m(r);
    return L;
  };
  // row step r: A, B of step it at row r, then C, D of step it+1 at row r-1
  auto step_row = [&](const int r, const Row& L) {
    const bool actB = r >= zo - 1, actC = r >= zo, actD = r >= zo + 1;
    const T ld_exn = L.exn, ld_ez = L.ez, ld_hy = L.hy;
    const CE k = L.k;
    MX m = L.m;
    const bool rv = valid(r);
    const T ex0_n = valid(r + 1) ? ld_exn : T(0);
    const T ez0_c = rv ? ld_ez : T(0);
    const T hy0 = rv ? ld_hy : T(0);

    // A, B: step it at row r
    const T hy1_c = hfield(r, ex0_c, ex0_n, ez0_c, hy0, m);
    T ex1_c = 0, ez1_c = 0;
    if (actB) {
      efield(r, hy1_c, hy1_p, ex0_c, ez0_c, k, m, incx0, incz0, ex1_c, ez1_c);
      if (r >= zo && r < ze) {
        bad0 |= own && !((double)ex1_c * ex1_c + (double)ez1_c * ez1_c <= 1.0e50);
        if (has_rec) gather(r, it, ex1_c, ez1_c);
      }
    }
    // C, D: step it+1 at row r-1
    T hy2_c = 0;
    if (actC) {
      MX mc = m_p;
      hy2_c = hfield(r - 1, ex1_p, ex1_c, ez1_p, hy1_p, mc);
      if (actD && r - 1 < ze) {
        T ex2, ez2;
        efield(r - 1, hy2_c, hy2_p, ex1_p, ez1_p, k_p, mc, incx1, incz1, ex2, ez2);
        bad1 |= own && !((double)ex2 * ex2 + (double)ez2 * ez2 <= 1.0e50);
        if (own) {
          const uint32_t co = cell(r - 1);
          exo[co] = ex2;
          ezo[co] = ez2;
          hyo[co] = hy2_c;
          store_m(r - 1, mc);
        }
        if (has_rec) gather(r - 1, it + 1, ex2, ez2);
      }
    }
    ex0_c = ex0_n;
    hy1_p = hy1_c;
    ex1_p = ex1_c;
    ez1_p = ez1_c;
    hy2_p = hy2_c;
    k_p = k;
    m_p = m;
  };
  for (int r = zo - 2; r <= ze; ++r) step_row(r, load_row(r));
  if (bad0)
    check_blowup(HUGE_VAL, S.blowup, it);
  else if (bad1)
    check_blowup(HUGE_VAL, S.blowup, it + 1);
}

// Work: as k_em2_step, with EW2E owned columns per wavefront.
template <typename T, int WB>
__global__ void __launch_bounds__(64 * WB)
k_em2_step2(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const int4* __restrict__ work, int nitems, const int* __restrict__ base, int rel,
            const int* __restrict__ it0, int eh0) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int it = __builtin_amdgcn_readfirstlane(*base + rel);
  const int q = __builtin_amdgcn_readfirstlane(((it - *it0) >> 1) & 1);
  for (int w = blockIdx.x; w < nitems; w += gridDim.x) {
    const int4 wv = work[w];
    const int4 wi = make_int4(__builtin_amdgcn_readfirstlane(wv.x),
                              __builtin_amdgcn_readfirstlane(wv.y) + wave * EW2E,
                              __builtin_amdgcn_readfirstlane(wv.z), 0);
    if (wi.x < 0) continue;
    const DModel& M = models[shots[wi.x].model];
    if (wi.y >= M.nx) continue;
    const int eh = wv.w > 0 ? __builtin_amdgcn_readfirstlane(wv.w) : eh0;  // rows of this tile
    // every column (lanes) and row (zo-2 .. ze+1) the wave reads outside the
    // C-PML slabs and clear of the columns and rows the edge rules name
    const int ze = min(wi.z + eh, M.nz);
    const bool interior = wi.y - 2 >= M.lx + 1 && wi.y + 61 <= M.nx - M.lx - 3 &&
                          wi.z - 2 >= M.lz + 1 && ze + 1 <= M.nz - M.lz - 3;
    if (interior)
      em2x2_tile<T, false>(models, shots, wi, it, q, threadIdx.x & 63, eh);
    else
      em2x2_tile<T, true>(models, shots, wi, it, q, threadIdx.x & 63, eh);
  }
}

// Hy zeroed on its Dirichlet ring (:312-315) in buffer A at the end of a run,
// so the returned state equals the legacy state.
template <typename T>
__global__ void k_em2_edges(const DModel* __restrict__ models, const DShot* __restrict__ shots) {
  const DShot& S = shots[blockIdx.y];
  const DModel& M = models[S.model];
  const int nx = M.nx, nz = M.nz;
  auto hy = mp<T>(S.f[2]);
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < 2 * (nx + nz); q += gridDim.x * blockDim.x) {
    int i, j;
    if (q < nx) { i = q; j = 0; }
    else if (q < 2 * nx) { i = q - nx; j = nz - 2; }
    else if (q < 2 * nx + nz) { i = 0; j = q - 2 * nx; }
    else { i = nx - 2; j = q - 2 * nx - nz; }
    if (i >= 0 && j >= 0) hy[(long)j * nx + i] = T(0);
  }
}

// ===========================================================================
// ELASTIC25: seismic25, legacy/fortran/seismicfdtd.f95:388-949
// Two launches per step: stresses, then velocities.  A wavefront (a block of
// its own) takes one z plane k, 64 adjacent columns (lanes 1..EW25 are owned;
// lanes 0 and 63 only supply x neighbours, which travel by DPP lane shifts) and
// a chunk of rows in y (rows25), R rows at a time.  Chunks end at the y-slab
// edges, and a wavefront clear of every slab runs a body without memory
// variables.  z neighbours are plain loads of the adjacent planes.
// What bounds it: on large grids the bytes (the second pass re-reads what the
// first wrote; 832x96x432 FP32 moves 5.8 GB per step at 5.2 TB/s, a copy
// reaches 4.9 .. 5.3), on small ones the latency of a row's loads.  So the loads
// of a row group, C-PML memory included, are all issued before the first use,
// and the stress pass reads the 33 y-invariant coefficients of its column from
// LDS once per group.  Loading the memory variables after the wait for the
// fields, with the next row's fields prefetched only where there are none, and
// x neighbours by ds_bpermute, measured (us per step) 1302 against 1160 on
// 832x96x432 FP32, 2402 against 2179 in FP64, 433 against 342 on 332x72x182
// FP64, 177 against 135 in FP32, 86 against 68 on 171x57x95 FP64, 48 against 27
// on 112x56x82 FP32.
// psi slabs (per shot):
//   x [nz][ny][2lx]: dvx_dx dvy_dx dvz_dx dsxx_dx dsxy_dx dsxz_dx
//   y [nz][2ly][nx]: dvx_dy dvy_dy dvz_dy dsyy_dy dsxy_dy dsyz_dy
//   z [2lz][ny][nx]: dvx_dz dvy_dz dvz_dz dszz_dz dsxz_dz dsyz_dz
// ===========================================================================
// (56, which puts every row of stores on a 32-byte boundary, measured slower
// here: 1.319 against 1.309 ms per aniso25 step, 0.640 against 0.593 ms per
// gpr25 step; the lanes lost cost more than the aligned stores gain)
#ifndef SDT_EL25_EW
#define SDT_EL25_EW 62
#endif
constexpr int EW25 = SDT_EL25_EW;      // owned columns per wavefront
static_assert(EW25 >= 1 && EW25 <= 62, "2.5-D wavefront: one halo lane on each side");
constexpr int NT25 = 64;               // a block is one wavefront

// The y chunk [j0, j1) of a 2.5-D work item travels in one int as two
// unsigned 16-bit halves (ny <= 65535 is checked at plan creation); the
// decode shifts as unsigned so chunks ending at or above 32768 stay positive.
__host__ __device__ inline int ychunk_pack(int j0, int j1) {
  return (int)((unsigned)j0 | ((unsigned)j1 << 16));
}
__host__ __device__ inline int ychunk_j0(int w) { return (int)((unsigned)w & 0xffffu); }
__host__ __device__ inline int ychunk_j1(int w) { return (int)((unsigned)w >> 16); }

struct Slab3 {
  long SX, SY, SZ;       // elements per memory-variable array on each axis
  long bx, by, bz;       // base offsets of the x, y, z groups
  __device__ Slab3(int nx, int ny, int nz, int lx, int ly, int lz) {
    SX = (long)nz * ny * 2 * lx;
    SY = (long)nz * 2 * ly * nx;
    SZ = (long)2 * lz * ny * nx;
    bx = 0;
    by = 6 * SX;
    bz = 6 * SX + 6 * SY;
  }
};

// One z plane of a 3-D field: wave-uniform base, 32-bit offsets j * nx + i.
template <typename T>
__device__ __forceinline__ A32<T> plane(void* f, long nxy, int k) {
  return A32<T>(static_cast<T*>(f) + (long)k * nxy);
}
template <typename T>
__device__ __forceinline__ A32<const T> cplane(const void* f, long nxy, int k) {
  return A32<const T>(static_cast<const T*>(f) + (long)k * nxy);
}

// Rows whose loads a wavefront has in flight at once (stress, velocity), and
// the wavefronts per SIMD that the register budgets are sized for.  Measured on
// 832x96x432 (us per step): FP32 stress rows / waves 1 / 4 1160, 1 / 5 1187, 2 / 3
// 1166, 2 / 4 1167; FP32 velocity 2 / 5 and 2 / 6 1160, 4 / 4 (spills) 1210;
// FP64 stress 1 / 2 2213, 2 / 2 2179; FP64 velocity 1 / 4 2211, 2 / 3 2179, 2 / 4
// (spills) 2271.  On 112x56x82 FP32 one stress row 27.2, two 29.2.
template <typename T>
constexpr int RS25 = sizeof(T) == 4 ? 1 : 2;
constexpr int RV25 = 2;
template <typename T>
constexpr int WS25 = sizeof(T) == 4 ? 4 : 2;
template <typename T>
constexpr int WV25 = sizeof(T) == 4 ? 5 : 3;

// C-PML memory of an elastic 2.5-D pass on one plane: arrays q .. q + 2 of each
// axis (q = 0 stress, 3 velocity).  The bases are wave-uniform, the offsets
// 32-bit: x[j * 2lx + xs], y[slab row * nx + i], z[j * nx + i].
template <typename T>
struct PsiEl25 {
  const A32<T> x0, x1, x2, y0, y1, y2, z0, z1, z2;
  __device__ __forceinline__ PsiEl25(void* psi, const Slab3& L, int q, int nx, int ny, int lx, int ly, int k, int zs)
      : x0((T*)psi + L.bx + q * L.SX + (long)k * ny * 2 * lx), x1((T*)psi + L.bx + (q + 1) * L.SX + (long)k * ny * 2 * lx),
        x2((T*)psi + L.bx + (q + 2) * L.SX + (long)k * ny * 2 * lx),
        y0((T*)psi + L.by + q * L.SY + (long)k * 2 * ly * nx), y1((T*)psi + L.by + (q + 1) * L.SY + (long)k * 2 * ly * nx),
        y2((T*)psi + L.by + (q + 2) * L.SY + (long)k * 2 * ly * nx),
        z0((T*)psi + L.bz + q * L.SZ + (long)zs * ny * nx), z1((T*)psi + L.bz + (q + 1) * L.SZ + (long)zs * ny * nx),
        z2((T*)psi + L.bz + (q + 2) * L.SZ + (long)zs * ny * nx) {}
};

template <typename T, bool PML>
__device__ __forceinline__ void el25_stress_tile(const DModel* __restrict__ models,
                                              const DShot* __restrict__ shots, const int4 wv,
                                              const int it, T* __restrict__ cs) {
  constexpr int R = RS25<T>;
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const int nx = M.nx, ny = M.ny, nz = M.nz;
  const int k = __builtin_amdgcn_readfirstlane(wv.z);
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane(wv.y) - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);  // clamped column: loads stay in bounds
  const bool own = incol && lane >= 1 && lane <= EW25;
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  const long nxy = (long)nx * ny;
  const uint32_t p = (uint32_t)k * nx + ic;
  const T idx = T(1.0 / M.dx), idy = T(1.0 / M.dy), idz = T(1.0 / M.dz), dt = T(M.dt);
  const int lx = M.lx, ly = M.ly, lz = M.lz;
  // a chunk lies inside a y slab or outside both
  const bool inx = PML && incol && in_slab(i, nx, lx), inz = PML && in_slab(k, nz, lz);
  const bool iny = PML && in_slab(j0, ny, ly);
  const Prof<T> P(&M.prof[0][0]);
  const auto iky = kp<T>(M.prof[1][PK]), ay = kp<T>(M.prof[1][PA]), by = kp<T>(M.prof[1][PB]);
  const auto ikyh = kp<T>(M.prof[1][PKH]), ayh = kp<T>(M.prof[1][PAH]), byh = kp<T>(M.prof[1][PBH]);
  const T bx_i = P[PB][ic], ax_i = P[PA][ic], ikx_i = P[PK][ic];
  const T bxh_i = P[PBH][ic], axh_i = P[PAH][ic], ikxh_i = P[PKH][ic];
  const T bz_k = kp<T>(M.prof[2][PB])[k], az_k = kp<T>(M.prof[2][PA])[k], ikz_k = kp<T>(M.prof[2][PK])[k];
  const T bzh_k = kp<T>(M.prof[2][PBH])[k], azh_k = kp<T>(M.prof[2][PAH])[k], ikzh_k = kp<T>(M.prof[2][PKH])[k];
  // loop ranges of the four legacy stress loops (seismicfdtd.f95:617, :677, :728, :771)
  const bool p1 = own && k >= 1 && i <= nx - 2, p2 = own && k >= 1 && i >= 1;
  const bool p3 = own && k <= nz - 2 && i >= 1, p4 = own && k <= nz - 2 && i <= nx - 2;
  // The 33 coefficients of the four loops at this column and plane do not
  // change along y: they are loaded once per work item into LDS, one slot per
  // thread that only that thread reads back, and read once per row group where
  // each loop uses them (volatile, so they are not held in registers for the
  // whole walk).  cs: the block's 33 * NT25 LDS slots.
  {
    T* w = cs + threadIdx.x;
#pragma unroll
    for (int q = 0; q < 33; ++q) w[q * NT25] = A32<const T>(M.coef[q])[p];
  }
  // coefficient q at C[q * NT25], read through an LDS pointer (ds_read)
  const __attribute__((address_space(3))) volatile T* C =
      (const __attribute__((address_space(3))) volatile T*)(cs) + threadIdx.x;
  const int kd = k >= 1 ? k - 1 : 0, ku = k <= nz - 2 ? k + 1 : nz - 1;
  const A32<const T> VX = cplane<T>(S.f[0], nxy, k), VY = cplane<T>(S.f[1], nxy, k);
  const A32<const T> VZ = cplane<T>(S.f[2], nxy, k);
  const A32<const T> VXD = cplane<T>(S.f[0], nxy, kd), VYD = cplane<T>(S.f[1], nxy, kd);
  const A32<const T> VZD = cplane<T>(S.f[2], nxy, kd);
  const A32<const T> VXU = cplane<T>(S.f[0], nxy, ku), VYU = cplane<T>(S.f[1], nxy, ku);
  const A32<const T> VZU = cplane<T>(S.f[2], nxy, ku);
  const A32<T> SXX = plane<T>(S.f[3], nxy, k), SYY = plane<T>(S.f[4], nxy, k);
  const A32<T> SZZ = plane<T>(S.f[5], nxy, k), SXY = plane<T>(S.f[6], nxy, k);
  const A32<T> SXZ = plane<T>(S.f[7], nxy, k), SYZ = plane<T>(S.f[8], nxy, k);
  const int xs = inx ? slab_pos(i, nx, lx) : 0, zs = inz ? slab_pos(k, nz, lz) : 0;
  const PsiEl25<T> W(S.psi, Slab3(nx, ny, nz, lx, ly, lz), 0, nx, ny, lx, ly, k, zs);

  // velocity rows jb-1 .. jb+R: [0], [1] carried from group to group
  T vx[R + 2], vy[R + 2], vz[R + 2];
  {
    const uint32_t m = (uint32_t)max(j0 - 1, 0) * nx + ic, c = (uint32_t)j0 * nx + ic;
    vx[0] = VX[m]; vy[0] = VY[m]; vz[0] = VZ[m];
    vx[1] = VX[c]; vy[1] = VY[c]; vz[1] = VZ[c];
  }
#pragma unroll 1
  for (int jb = j0; jb < j1; jb += R) {
    T vxd[R], vyd[R], vzd[R], vxu[R], vyu[R], vzu[R];
    T sxx[R], syy[R], szz[R], sxy[R], sxz[R], syz[R];
    T mxx[R], myx[R], mzx[R], mxy[R], myy[R], mzy[R], mxz[R], myz[R], mzz[R];
    uint32_t c[R];
    // every load of the R rows before the first use (rows past the chunk
    // reload its last row; velocities the row below it)
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t n = (uint32_t)min(jb + q + 1, min(j1, ny - 1)) * nx + ic;
      c[q] = (uint32_t)min(jb + q, j1 - 1) * nx + ic;
      vx[q + 2] = VX[n]; vy[q + 2] = VY[n]; vz[q + 2] = VZ[n];
      vxd[q] = VXD[c[q]]; vyd[q] = VYD[c[q]]; vzd[q] = VZD[c[q]];
      vxu[q] = VXU[c[q]]; vyu[q] = VYU[c[q]]; vzu[q] = VZU[c[q]];
      sxx[q] = SXX[c[q]]; syy[q] = SYY[c[q]]; szz[q] = SZZ[c[q]];
      sxy[q] = SXY[c[q]]; sxz[q] = SXZ[c[q]]; syz[q] = SYZ[c[q]];
    }
    // velocity-derivative memory variables (shared by all four loops: A1)
    if (PML && iny) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)slab_pos(min(jb + q, j1 - 1), ny, ly) * nx + ic;
        mxy[q] = W.y0[o]; myy[q] = W.y1[o]; mzy[q] = W.y2[o];
      }
    }
    if (PML && inz) {
#pragma unroll
      for (int q = 0; q < R; ++q) { mxz[q] = W.z0[c[q]]; myz[q] = W.z1[c[q]]; mzz[q] = W.z2[c[q]]; }
    }
    if (PML && inx) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)min(jb + q, j1 - 1) * 2 * lx + xs;
        mxx[q] = W.x0[o]; myx[q] = W.x1[o]; mzx[q] = W.x2[o];
      }
    }
    // loop 1: sigma xx, yy, zz (seismicfdtd.f95:617-674)
    {
      const T c0 = C[0], c1 = C[1 * NT25], c2 = C[2 * NT25], c3 = C[3 * NT25], c4 = C[4 * NT25];
      const T c5 = C[5 * NT25], c6 = C[6 * NT25], c7 = C[7 * NT25], c8 = C[8 * NT25], c9 = C[9 * NT25];
      const T c10 = C[10 * NT25], c11 = C[11 * NT25], c12 = C[12 * NT25], c13 = C[13 * NT25];
      const T c14 = C[14 * NT25];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int j = jb + q;
        const T vxc = vx[q + 1], vyc = vy[q + 1], vzc = vz[q + 1];
        const T vxe = dpp_next(vxc), vye = dpp_next(vyc), vze = dpp_next(vzc);  // i+1
        if (p1 && j >= 1 && j < j1) {
          T dvx_dx = (vxe - vxc) * idx, dvy_dx = (vye - vyc) * idx, dvz_dx = (vze - vzc) * idx;
          T dvy_dy = (vyc - vy[q]) * idy, dvx_dy = (vxc - vx[q]) * idy, dvz_dy = (vzc - vz[q]) * idy;
          T dvz_dz = (vzc - vzd[q]) * idz, dvx_dz = (vxc - vxd[q]) * idz, dvy_dz = (vyc - vyd[q]) * idz;
          if (PML && inx) {
            mxx[q] = bxh_i * mxx[q] + axh_i * dvx_dx; myx[q] = bxh_i * myx[q] + axh_i * dvy_dx; mzx[q] = bxh_i * mzx[q] + axh_i * dvz_dx;
            dvx_dx = dvx_dx * ikxh_i + mxx[q]; dvy_dx = dvy_dx * ikxh_i + myx[q]; dvz_dx = dvz_dx * ikxh_i + mzx[q];
          }
          if (PML && iny) {
            const T b = by[j], a = ay[j], ik = iky[j];
            myy[q] = b * myy[q] + a * dvy_dy; mxy[q] = b * mxy[q] + a * dvx_dy; mzy[q] = b * mzy[q] + a * dvz_dy;
            dvy_dy = dvy_dy * ik + myy[q]; dvx_dy = dvx_dy * ik + mxy[q]; dvz_dy = dvz_dy * ik + mzy[q];
          }
          if (PML && inz) {
            mzz[q] = bz_k * mzz[q] + az_k * dvz_dz; mxz[q] = bz_k * mxz[q] + az_k * dvx_dz; myz[q] = bz_k * myz[q] + az_k * dvy_dz;
            dvz_dz = dvz_dz * ikz_k + mzz[q]; dvx_dz = dvx_dz * ikz_k + mxz[q]; dvy_dz = dvy_dz * ikz_k + myz[q];
          }
          SXX[c[q]] = sxx[q] + (c0 * dvx_dx + c1 * dvy_dy + c2 * dvz_dz + c3 * (dvy_dz + dvz_dy) +
                                c4 * (dvx_dz + dvz_dx) + c5 * (dvx_dy + dvz_dy)) * dt;  // A3 (c16)
          SYY[c[q]] = syy[q] + (c1 * dvx_dx + c6 * dvy_dy + c7 * dvz_dz + c8 * (dvy_dz + dvz_dy) +
                                c9 * (dvx_dz + dvz_dx) + c10 * (dvy_dx + dvx_dy)) * dt;
          SZZ[c[q]] = szz[q] + (c2 * dvx_dx + c7 * dvy_dy + c11 * dvz_dz + c12 * (dvy_dz + dvz_dy) +
                                c13 * (dvx_dz + dvz_dx) + c14 * (dvy_dx + dvx_dy)) * dt;
        }
      }
    }
    // loop 2: sigma xy (seismicfdtd.f95:677-725); dvz_dx and dvx_dz get no correction
    {
      const T c0 = C[15 * NT25], c1 = C[16 * NT25], c2 = C[17 * NT25], c3 = C[18 * NT25], c4 = C[19 * NT25], c5 = C[20 * NT25];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int j = jb + q;
        const T vxc = vx[q + 1], vyc = vy[q + 1], vzc = vz[q + 1];
        const T vxw = dpp_prev(vxc), vyw = dpp_prev(vyc), vzw = dpp_prev(vzc);  // i-1
        if (p2 && j <= ny - 2 && j < j1) {
          T dvx_dx = (vxc - vxw) * idx, dvy_dx = (vyc - vyw) * idx, dvz_dx = (vzc - vzw) * idx;
          T dvy_dy = (vy[q + 2] - vyc) * idy, dvx_dy = (vx[q + 2] - vxc) * idy, dvz_dy = (vz[q + 2] - vzc) * idy;
          T dvz_dz = (vzc - vzd[q]) * idz, dvx_dz = (vxc - vxd[q]) * idz, dvy_dz = (vyc - vyd[q]) * idz;
          if (PML && inx) {
            mxx[q] = bx_i * mxx[q] + ax_i * dvx_dx; myx[q] = bx_i * myx[q] + ax_i * dvy_dx; mzx[q] = bx_i * mzx[q] + ax_i * dvz_dx;
            dvx_dx = dvx_dx * ikx_i + mxx[q]; dvy_dx = dvy_dx * ikx_i + myx[q];
          }
          if (PML && iny) {
            const T b = byh[j], a = ayh[j], ik = ikyh[j];
            myy[q] = b * myy[q] + a * dvy_dy; mxy[q] = b * mxy[q] + a * dvx_dy; mzy[q] = b * mzy[q] + a * dvz_dy;
            dvy_dy = dvy_dy * ik + myy[q]; dvx_dy = dvx_dy * ik + mxy[q]; dvz_dy = dvz_dy * ik + mzy[q];
          }
          if (PML && inz) {
            mzz[q] = bzh_k * mzz[q] + azh_k * dvz_dz; mxz[q] = bzh_k * mxz[q] + azh_k * dvx_dz; myz[q] = bzh_k * myz[q] + azh_k * dvy_dz;
            dvz_dz = dvz_dz * ikzh_k + mzz[q]; dvy_dz = dvy_dz * ikzh_k + myz[q];
          }
          SXY[c[q]] = sxy[q] + (c0 * dvx_dx + c1 * dvy_dy + c2 * dvz_dz + c3 * (dvz_dy + dvy_dz) +
                                c4 * (dvz_dx + dvx_dz) + c5 * (dvy_dx + dvx_dy)) * dt;
        }
      }
    }
    // loop 3: sigma xz (seismicfdtd.f95:728-768)
    {
      const T c0 = C[21 * NT25], c1 = C[22 * NT25], c2 = C[23 * NT25], c3 = C[24 * NT25], c4 = C[25 * NT25], c5 = C[26 * NT25];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int j = jb + q;
        const T vxc = vx[q + 1], vyc = vy[q + 1], vzc = vz[q + 1];
        const T vxw = dpp_prev(vxc), vyw = dpp_prev(vyc), vzw = dpp_prev(vzc);
        if (p3 && j >= 1 && j < j1) {
          T dvx_dx = (vxc - vxw) * idx, dvy_dx = (vyc - vyw) * idx, dvz_dx = (vzc - vzw) * idx;
          T dvy_dy = (vyc - vy[q]) * idy, dvz_dy = (vzc - vz[q]) * idy, dvx_dy = (vxc - vx[q]) * idy;
          T dvz_dz = (vzu[q] - vzc) * idz, dvx_dz = (vxu[q] - vxc) * idz, dvy_dz = (vyu[q] - vyc) * idz;
          if (PML && inx) {
            mxx[q] = bx_i * mxx[q] + ax_i * dvx_dx; myx[q] = bx_i * myx[q] + ax_i * dvy_dx; mzx[q] = bx_i * mzx[q] + ax_i * dvz_dx;
            dvx_dx = dvx_dx * ikx_i + mxx[q]; dvy_dx = dvy_dx * ikx_i + myx[q]; dvz_dx = dvz_dx * ikx_i + mzx[q];
          }
          if (PML && iny) {
            const T b = by[j], a = ay[j], ik = iky[j];
            myy[q] = b * myy[q] + a * dvy_dy; mxy[q] = b * mxy[q] + a * dvx_dy; mzy[q] = b * mzy[q] + a * dvz_dy;
            dvy_dy = dvy_dy * ik + myy[q]; dvx_dy = dvx_dy * ik + mxy[q]; dvz_dy = dvz_dy * ik + mzy[q];
          }
          if (PML && inz) {
            mzz[q] = bzh_k * mzz[q] + azh_k * dvz_dz; mxz[q] = bzh_k * mxz[q] + azh_k * dvx_dz; myz[q] = bzh_k * myz[q] + azh_k * dvy_dz;
            dvz_dz = dvz_dz * ikzh_k + mzz[q]; dvx_dz = dvx_dz * ikzh_k + mxz[q]; dvy_dz = dvy_dz * ikzh_k + myz[q];
          }
          SXZ[c[q]] = sxz[q] + (c0 * dvx_dx + c1 * dvy_dy + c2 * dvz_dz + c3 * (dvx_dz + dvz_dx) +
                                c4 * (dvx_dz + dvz_dx) + c5 * (dvx_dy + dvy_dx)) * dt;  // A3 (c45)
        }
      }
    }
    // loop 4: sigma yz (seismicfdtd.f95:771-813)
    {
      const T c0 = C[27 * NT25], c1 = C[28 * NT25], c2 = C[29 * NT25], c3 = C[30 * NT25], c4 = C[31 * NT25], c5 = C[32 * NT25];
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int j = jb + q;
        const T vxc = vx[q + 1], vyc = vy[q + 1], vzc = vz[q + 1];
        const T vxe = dpp_next(vxc), vye = dpp_next(vyc), vze = dpp_next(vzc);
        if (p4 && j <= ny - 2 && j < j1) {
          T dvx_dx = (vxe - vxc) * idx, dvy_dx = (vye - vyc) * idx, dvz_dx = (vze - vzc) * idx;
          T dvy_dy = (vy[q + 2] - vyc) * idy, dvx_dy = (vx[q + 2] - vxc) * idy, dvz_dy = (vz[q + 2] - vzc) * idy;
          T dvz_dz = (vzu[q] - vzc) * idz, dvx_dz = (vxu[q] - vxc) * idz, dvy_dz = (vyu[q] - vyc) * idz;
          if (PML && inx) {
            mxx[q] = bxh_i * mxx[q] + axh_i * dvx_dx; myx[q] = bxh_i * myx[q] + axh_i * dvy_dx; mzx[q] = bxh_i * mzx[q] + axh_i * dvz_dx;
            dvx_dx = dvx_dx * ikxh_i + mxx[q]; dvy_dx = dvy_dx * ikxh_i + myx[q]; dvz_dx = dvz_dx * ikxh_i + mzx[q];
          }
          if (PML && iny) {
            const T b = byh[j], a = ayh[j], ik = ikyh[j];
            myy[q] = b * myy[q] + a * dvy_dy; mxy[q] = b * mxy[q] + a * dvx_dy; mzy[q] = b * mzy[q] + a * dvz_dy;
            dvy_dy = dvy_dy * ik + myy[q]; dvx_dy = dvx_dy * ik + mxy[q]; dvz_dy = dvz_dy * ik + mzy[q];
          }
          if (PML && inz) {
            mzz[q] = bzh_k * mzz[q] + azh_k * dvz_dz; mxz[q] = bzh_k * mxz[q] + azh_k * dvx_dz; myz[q] = bzh_k * myz[q] + azh_k * dvy_dz;
            dvz_dz = dvz_dz * ikzh_k + mzz[q]; dvx_dz = dvx_dz * ikzh_k + mxz[q]; dvy_dz = dvy_dz * ikzh_k + myz[q];
          }
          SYZ[c[q]] = syz[q] + (c0 * dvx_dx + c1 * dvy_dy + c2 * dvz_dz + c3 * (dvy_dz + dvz_dy) +
                                c4 * (dvx_dz + dvz_dx) + c5 * (dvy_dx + dvx_dy)) * dt;
        }
      }
    }
    if (own) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int j = jb + q;
        if (j >= j1) break;
        if (PML && inx) {
          const uint32_t o = (uint32_t)j * 2 * lx + xs;
          W.x0[o] = mxx[q]; W.x1[o] = myx[q]; W.x2[o] = mzx[q];
        }
        if (PML && iny) {
          const uint32_t o = (uint32_t)slab_pos(j, ny, ly) * nx + ic;
          W.y0[o] = mxy[q]; W.y1[o] = myy[q]; W.y2[o] = mzy[q];
        }
        if (PML && inz) { W.z0[c[q]] = mxz[q]; W.z1[c[q]] = myz[q]; W.z2[c[q]] = mzz[q]; }
        if (i == S.isrc && k == S.ksrc && j == S.jsrc) {  // stress-rate (moment-tensor) source
          if (S.msrc[0]) SXX[c[q]] = SXX[c[q]] + cp<T>(S.msrc[0])[it];
          if (S.msrc[1]) SYY[c[q]] = SYY[c[q]] + cp<T>(S.msrc[1])[it];
          if (S.msrc[2]) SZZ[c[q]] = SZZ[c[q]] + cp<T>(S.msrc[2])[it];
          if (S.msrc[3]) SXY[c[q]] = SXY[c[q]] + cp<T>(S.msrc[3])[it];
          if (S.msrc[4]) SXZ[c[q]] = SXZ[c[q]] + cp<T>(S.msrc[4])[it];
          if (S.msrc[5]) SYZ[c[q]] = SYZ[c[q]] + cp<T>(S.msrc[5])[it];
        }
      }
    }
    vx[0] = vx[R]; vy[0] = vy[R]; vz[0] = vz[R];
    vx[1] = vx[R + 1]; vy[1] = vy[R + 1]; vz[1] = vz[R + 1];
  }
}

// A wavefront whose columns, plane and rows all lie outside the C-PML slabs
// runs the body without memory variables.
template <typename T>
__global__ void __launch_bounds__(NT25, WS25<T>)
k_el25_stress(const DModel* __restrict__ models, const DShot* __restrict__ shots,
          const int4* __restrict__ work, int n, const int* __restrict__ base, int rel) {
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DModel& M = models[shots[s].model];
  const int xo = __builtin_amdgcn_readfirstlane(wv.y), k = __builtin_amdgcn_readfirstlane(wv.z);
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  const bool interior = xo - 1 >= M.lx && xo + 62 < M.nx - M.lx && k >= M.lz && k < M.nz - M.lz &&
                        j0 >= M.ly && j1 <= M.ny - M.ly;
  const int it = *base + rel;
  __shared__ T cs[33 * NT25];  // the y-invariant coefficients (el25_stress_tile)
  if (interior)
    el25_stress_tile<T, false>(models, shots, wv, it, cs);
  else
    el25_stress_tile<T, true>(models, shots, wv, it, cs);
}

template <typename T, bool PML>
__device__ __forceinline__ void el25_vel_tile(const DModel* __restrict__ models,
                                              const DShot* __restrict__ shots, const int4 wv, const int* __restrict__ base, int rel) {
  constexpr int R = RV25;
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const int nx = M.nx, ny = M.ny, nz = M.nz;
  const int k = __builtin_amdgcn_readfirstlane(wv.z);
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane(wv.y) - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);
  const bool own = incol && lane >= 1 && lane <= EW25;
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  const int it = *base + rel;
  const long nxy = (long)nx * ny;
  const uint32_t p = (uint32_t)k * nx + ic;
  const T idx = T(1.0 / M.dx), idy = T(1.0 / M.dy), idz = T(1.0 / M.dz);
  const int lx = M.lx, ly = M.ly, lz = M.lz;
  const bool inx = PML && incol && in_slab(i, nx, lx), inz = PML && in_slab(k, nz, lz);
  const bool iny = PML && in_slab(j0, ny, ly);
  const Prof<T> P(&M.prof[0][0]);
  const T bx_i = P[PB][ic], ax_i = P[PA][ic], ikx_i = P[PK][ic];
  const T bxh_i = P[PBH][ic], axh_i = P[PAH][ic], ikxh_i = P[PKH][ic];
  const T bz_k = kp<T>(M.prof[2][PB])[k], az_k = kp<T>(M.prof[2][PA])[k], ikz_k = kp<T>(M.prof[2][PK])[k];
  const T bzh_k = kp<T>(M.prof[2][PBH])[k], azh_k = kp<T>(M.prof[2][PAH])[k], ikzh_k = kp<T>(M.prof[2][PKH])[k];
  const auto iky = kp<T>(M.prof[1][PK]), ay = kp<T>(M.prof[1][PA]), by = kp<T>(M.prof[1][PB]);
  const auto ikyh = kp<T>(M.prof[1][PKH]), ayh = kp<T>(M.prof[1][PAH]), byh = kp<T>(M.prof[1][PBH]);
  // loop ranges of the legacy velocity loops (seismicfdtd.f95:821, :848, :873)
  const bool ux = own && k >= 1 && i >= 1, uy = own && k >= 1 && i <= nx - 2;
  const bool uz = own && k <= nz - 2 && i <= nx - 2;
  const T dtrx = A32<const T>(M.coef[33])[p], dtry = A32<const T>(M.coef[34])[p], dtrz = A32<const T>(M.coef[35])[p];
  const T omx = A32<const T>(M.coef[36])[p], omy = A32<const T>(M.coef[37])[p];
  const T omz = A32<const T>(M.coef[38])[p];
  const int kd = k >= 1 ? k - 1 : 0, ku = k <= nz - 2 ? k + 1 : nz - 1;
  const A32<const T> SXX = cplane<T>(S.f[3], nxy, k), SYY = cplane<T>(S.f[4], nxy, k);
  const A32<const T> SZZ = cplane<T>(S.f[5], nxy, k), SXY = cplane<T>(S.f[6], nxy, k);
  const A32<const T> SXZ = cplane<T>(S.f[7], nxy, k), SYZ = cplane<T>(S.f[8], nxy, k);
  const A32<const T> SXZD = cplane<T>(S.f[7], nxy, kd), SYZD = cplane<T>(S.f[8], nxy, kd);
  const A32<const T> SZZU = cplane<T>(S.f[5], nxy, ku);
  const A32<T> VX = plane<T>(S.f[0], nxy, k), VY = plane<T>(S.f[1], nxy, k), VZ = plane<T>(S.f[2], nxy, k);
  const int xs = inx ? slab_pos(i, nx, lx) : 0, zs = inz ? slab_pos(k, nz, lz) : 0;
  const PsiEl25<T> W(S.psi, Slab3(nx, ny, nz, lx, ly, lz), 3, nx, ny, lx, ly, k, zs);
  const bool kedge = (i == 0 || k == 0 || i == nx - 1 || k == nz - 1);
  const bool srccol = (i == S.isrc && k == S.ksrc);
  bool bad = false;

  // sxy, syz of rows jb-1 .. jb+R-1 and syy of rows jb .. jb+R: [0] carried
  T sxy[R + 1], syz[R + 1], syy[R + 1];
  {
    const uint32_t m = (uint32_t)max(j0 - 1, 0) * nx + ic;
    sxy[0] = SXY[m]; syz[0] = SYZ[m];
    syy[0] = SYY[(uint32_t)j0 * nx + ic];
  }
#pragma unroll 1
  for (int jb = j0; jb < j1; jb += R) {
    T sxx[R], sxz[R], szz[R], sxzd[R], syzd[R], szzu[R], vx[R], vy[R], vz[R];
    T x0[R], x1[R], x2[R], y0[R], y1[R], y2[R], z0[R], z1[R], z2[R];
    uint32_t c[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      c[q] = (uint32_t)min(jb + q, j1 - 1) * nx + ic;
      sxx[q] = SXX[c[q]]; sxz[q] = SXZ[c[q]]; szz[q] = SZZ[c[q]];
      sxy[q + 1] = SXY[c[q]]; syz[q + 1] = SYZ[c[q]];
      syy[q + 1] = SYY[(uint32_t)min(jb + q + 1, min(j1, ny - 1)) * nx + ic];
      sxzd[q] = SXZD[c[q]]; syzd[q] = SYZD[c[q]]; szzu[q] = SZZU[c[q]];
      vx[q] = VX[c[q]]; vy[q] = VY[c[q]]; vz[q] = VZ[c[q]];
    }
    if (PML && iny) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)slab_pos(min(jb + q, j1 - 1), ny, ly) * nx + ic;
        y0[q] = W.y0[o]; y1[q] = W.y1[o]; y2[q] = W.y2[o];
      }
    }
    if (PML && inz) {
#pragma unroll
      for (int q = 0; q < R; ++q) { z0[q] = W.z0[c[q]]; z1[q] = W.z1[c[q]]; z2[q] = W.z2[c[q]]; }
    }
    if (PML && inx) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)min(jb + q, j1 - 1) * 2 * lx + xs;
        x0[q] = W.x0[o]; x1[q] = W.x1[o]; x2[q] = W.x2[o];
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int j = jb + q;
      const T sxxw = dpp_prev(sxx[q]), sxye = dpp_next(sxy[q + 1]), sxze = dpp_next(sxz[q]);
      if (j >= j1) break;
      const uint32_t ox = (uint32_t)j * 2 * lx + xs;
      const uint32_t oy = PML && iny ? (uint32_t)slab_pos(j, ny, ly) * nx + ic : 0;
      T vxn = vx[q], vyn = vy[q], vzn = vz[q];
      // vx, seismicfdtd.f95:821-846
      if (ux && j >= 1) {
        T a = (sxx[q] - sxxw) * idx, b = (sxy[q + 1] - sxy[q]) * idy, d = (sxz[q] - sxzd[q]) * idz;
        if (PML && inx) { const T m = bx_i * x0[q] + ax_i * a; a = a * ikx_i + m; W.x0[ox] = m; }
        if (PML && iny) { const T m = by[j] * y1[q] + ay[j] * b; b = b * iky[j] + m; W.y1[oy] = m; }
        if (PML && inz) { const T m = bz_k * z1[q] + az_k * d; d = d * ikz_k + m; W.z1[c[q]] = m; }
        vxn = vxn * omx + (a + b + d) * dtrx;
      }
      // vy, seismicfdtd.f95:848-870
      if (uy && j <= ny - 2) {
        T a = (sxye - sxy[q + 1]) * idx, b = (syy[q + 1] - syy[q]) * idy, d = (syz[q + 1] - syzd[q]) * idz;
        if (PML && inx) { const T m = bxh_i * x1[q] + axh_i * a; a = a * ikxh_i + m; W.x1[ox] = m; }
        if (PML && iny) { const T m = byh[j] * y0[q] + ayh[j] * b; b = b * ikyh[j] + m; W.y0[oy] = m; }
        if (PML && inz) { const T m = bz_k * z2[q] + az_k * d; d = d * ikz_k + m; W.z2[c[q]] = m; }
        vyn = vyn * omy + (a + b + d) * dtry;
      }
      // vz, seismicfdtd.f95:873-896
      if (uz && j >= 1) {
        T a = (sxze - sxz[q]) * idx, b = (syz[q + 1] - syz[q]) * idy, d = (szzu[q] - szz[q]) * idz;
        if (PML && inx) { const T m = bxh_i * x2[q] + axh_i * a; a = a * ikxh_i + m; W.x2[ox] = m; }
        if (PML && iny) { const T m = by[j] * y2[q] + ay[j] * b; b = b * iky[j] + m; W.y2[oy] = m; }
        if (PML && inz) { const T m = bzh_k * z0[q] + azh_k * d; d = d * ikzh_k + m; W.z0[c[q]] = m; }
        vzn = vzn * omz + (a + b + d) * dtrz;
      }
      // source, seismicfdtd.f95:898-900
      if (srccol && j == S.jsrc) {
        if (S.src[0]) vxn += cp<T>(S.src[0])[it];
        if (S.src[1]) vyn += cp<T>(S.src[1])[it];
        if (S.src[2]) vzn += cp<T>(S.src[2])[it];
      }
      // Dirichlet faces, seismicfdtd.f95:903-925
      if (kedge || j == 0 || j == ny - 1) { vxn = 0; vyn = 0; vzn = 0; }
      if (own) {
        bad |= !((double)vxn * vxn + (double)vyn * vyn + (double)vzn * vzn <= 1.0e50);
        VX[c[q]] = vxn;
        VY[c[q]] = vyn;
        VZ[c[q]] = vzn;
      }
    }
    sxy[0] = sxy[R]; syz[0] = syz[R]; syy[0] = syy[R];
  }
  if (bad) atomicMin(S.blowup, it);
}

// A wavefront whose columns, plane and rows all lie outside the C-PML slabs
// runs the body without memory variables.
template <typename T>
__global__ void __launch_bounds__(NT25, WV25<T>)
k_el25_vel(const DModel* __restrict__ models, const DShot* __restrict__ shots,
          const int4* __restrict__ work, int n, const int* __restrict__ base, int rel) {
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DModel& M = models[shots[s].model];
  const int xo = __builtin_amdgcn_readfirstlane(wv.y), k = __builtin_amdgcn_readfirstlane(wv.z);
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  const bool interior = xo - 1 >= M.lx && xo + 62 < M.nx - M.lx && k >= M.lz && k < M.nz - M.lz &&
                        j0 >= M.ly && j1 <= M.ny - M.ly;
  if (interior)
    el25_vel_tile<T, false>(models, shots, wv, base, rel);
  else
    el25_vel_tile<T, true>(models, shots, wv, base, rel);
}

// ===========================================================================
// ELASTIC2 and EM2, several time steps per launch on regions.
//
// A block of 1024 threads holds a region of RM x RM cells of one shot, one cell
// per thread, with the state, the memory variables and the coefficients in
// registers, and takes up to tm steps: rows are exchanged through LDS, columns
// by DPP lane shifts (a wavefront is two rows of the region; what a shift
// carries across their ends reaches only halo columns).  One step makes a cell
// depend on one neighbour each way; with the legacy C-PML, whose shear loop uses
// the memory the normal loop has just updated, an elastic cell also on column
// i+2 (in an x slab) and row k-2 (in a z slab).  So after tm steps the middle of
// the region is exact (columns and rows tm .. RM-tm-1; where a legacy region
// touches an x slab columns tm .. RM-2tm-1, a z slab rows 2tm .. RM-tm-1; with
// that wider ring everywhere, us per step: FP32 48 shots of 39 M cells 350, now
// 248, 16 of 1064x552 77, 61, FP64 9 uneven shots 26, 21, 4 of 1064x808 67, 50):
// the block owns that and the neighbouring blocks recompute the rest.  Every
// expression is the one-step kernel's, in the same order: identical bits.  A
// launch reads state buffer par and writes the other.
// What bounds it: at most two blocks (four of the EM blocks of two rows per
// thread) share a CU, so a SIMD has 4 or 8 wavefronts
// whose instructions it issues one after the other (about 1.1 us per elastic
// step and block), and each launch waits once for its loads (5 to 7 us).
// Regions off the slabs and the outer rings run a body without memory
// variables and edge predicates (EM FP32 1064x808 5.6 -> 5.1 us per step with it).
// The budget of 8 wavefronts per SIMD (elastic FP64 4, at 110 registers) is what
// lets two blocks share a CU: EM FP64 1064x808 8.3 -> 6.5 us per step.  Letting
// the wavefronts whose rows no later step needs sit out measured 3 % slower.
// ===========================================================================
constexpr int RM = 32;       // region: RM x RM cells, one thread each
constexpr int TM_MAX = 8;    // most steps per launch

// Regions of tm steps, along one axis: rows above the owned cells (tm columns to
// their left), owned cells.  one: a step reaches one cell each way; otherwise
// the legacy elastic C-PML, on the axis whose slab the region touches.
__host__ __device__ constexpr int region_top(bool one, int tm) { return one ? tm : 2 * tm; }
__host__ __device__ constexpr int region_own(bool one, int tm) { return RM - (one ? 2 : 3) * tm; }
// Flags of a legacy elastic work item beside its model: the region keeps off
// the x slabs, off the z slabs.
constexpr int REGION_X1 = 1 << 30, REGION_Z1 = 1 << 29;

// The receivers of a thread's K cells (rows z0 + K * (threadIdx.x / RM) + k of
// the region at x0, z0): per cell the first index entry on it (INT_MAX: none),
// that receiver, and whether more follow.  The block owns ownx x ownz cells from
// column cx0, row cz0 on; mine: the thread's cell is one of them.  Called by
// every thread; slot: one entry per cell.
struct RegionRec {
  int e0, id0;
  bool more;
};
template <int K>
__device__ __forceinline__ void region_receivers(const DShot& S, int* slot, int x0, int z0, int nz, int cx0,
                                                 int cz0, int ownx, int ownz, const bool (&mine)[K],
                                                 RegionRec (&rec)[K]) {
  const int zr0 = z0 + cz0, zr1 = min(zr0 + ownz, nz);
  for (int k = 0; k < K; ++k) rec[k] = {INT_MAX, 0, false};
  if (S.nrec <= 0 || S.rrow[zr1] <= S.rrow[zr0]) return;  // block-uniform
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int tx = threadIdx.x % RM, ty = K * (int)(threadIdx.x / RM);
  for (int k = 0; k < K; ++k) slot[(ty + k) * RM + tx] = INT_MAX;
  __syncthreads();
  for (int h = 0; h < 2 * K; ++h) {  // a wavefront's own rows
    const int row = z0 + 2 * K * w + h;
    if (row < zr0 || row >= zr1) continue;
    const int q0 = S.rrow[row], q1 = S.rrow[row + 1];
    for (int e = q0 + lane; e < q1; e += 64) {
      const int cx = S.rxid[2 * e] - x0;
      if (cx >= cx0 && cx < cx0 + ownx) atomicMin(&slot[(2 * K * w + h) * RM + cx], e);
    }
  }
  __syncthreads();
  for (int k = 0; k < K; ++k) {
    const int e0 = slot[(ty + k) * RM + tx];
    if (!mine[k] || e0 == INT_MAX) continue;
    rec[k] = {e0, S.rxid[2 * e0 + 1], e0 + 1 < S.rrow[z0 + ty + k + 1] && S.rxid[2 * e0 + 2] == x0 + tx};
  }
}

// This step's samples a, b of the receivers on a cell of column i, row r.
template <typename T>
__device__ __forceinline__ void region_sample(const DShot& S, int it, int i, int r, const RegionRec& rec, T a,
                                              T b) {
  if (rec.e0 == INT_MAX) return;
  auto tr = mp<T>(S.trace) + (long)it * 2 * S.nrec;
  tr[rec.id0] = a;
  tr[S.nrec + rec.id0] = b;
  if (!rec.more) return;
  const int e1 = S.rrow[r + 1];
  for (int e = rec.e0 + 1; e < e1 && S.rxid[2 * e] == i; ++e) {
    const int id = S.rxid[2 * e + 1];
    tr[id] = a;
    tr[S.nrec + id] = b;
  }
}

template <typename T, bool SPLIT>
struct ElRegionLds {
  T v[2][RM][RM], s[2][RM][RM];  // vx, vz; sxz, szz
  T px[6][RM], pz[7][RM];        // C-PML profiles of the region's columns and rows
  T src[5][TM_MAX];              // source increments of the steps: vx vz sxx szz sxz
  // split C-PML, FP32: the shear loop's memory variables of each cell, used by
  // its own thread only (in registers two blocks would not fit on a CU; FP64,
  // whose single block has registers to spare, 709 -> 657 us per 300 steps of
  // a 139x113 plan without them here)
  static constexpr bool SH = SPLIT && sizeof(T) == 4;
  T sh[SH ? 4 : 1][SH ? RM : 1][SH ? RM : 1];
  int slot[RM * RM];
};

// PML false: no cell of the region lies in a C-PML slab or on the outer ring.
// TRAIL: the state is read from trail buffer ts.tb's slot ts.slot, every step's
// new one written to the next; no samples, no blow-up check (the forward has
// done both).
struct TrailSlot {
  const DAdj* adj;
  int tb, slot;
};

template <typename T, bool SPLIT, bool PML, bool TRAIL>
__device__ __forceinline__ void el2_region(const DModel& M, const DShot& S, const int x0, const int z0,
                                           const bool x1, const bool z1, const int it0, const int nsteps, const int tm, const int par,
                                           const TrailSlot ts, ElRegionLds<T, SPLIT>& L) {
#pragma clang fp contract(off)
  const int nx = M.nx, nz = M.nz;
  const int tx = threadIdx.x & (RM - 1), ty = threadIdx.x / RM;
  const int i = x0 + tx, r = z0 + ty;
  const int osx = region_own(x1, tm), osz = region_own(z1, tm), zt = region_top(z1, tm);
  const bool in = !PML || (i >= 0 && i < nx && r >= 0 && r < nz);
  const int ic = PML ? min(max(i, 0), nx - 1) : i, rc = PML ? min(max(r, 0), nz - 1) : r;
  const bool own = in && tx >= tm && tx < tm + osx && ty >= zt && ty < zt + osz;
  const uint32_t c = (uint32_t)rc * nx + ic;
  const long n = (long)nx * nz;
  T* const trail = TRAIL ? static_cast<T*>(ts.adj->trail[ts.tb]) + ts.slot * ts.adj->slot : nullptr;
  T vx = A32<const T>(TRAIL ? trail : par ? S.g[0] : S.f[0])[c];
  T vz = A32<const T>(TRAIL ? trail + n : par ? S.g[1] : S.f[1])[c];
  T sxx = A32<const T>(TRAIL ? trail + 2 * n : par ? S.g[2] : S.f[2])[c];
  T szz = A32<const T>(TRAIL ? trail + 3 * n : par ? S.g[3] : S.f[3])[c];
  T sxz = A32<const T>(TRAIL ? trail + 4 * n : par ? S.g[4] : S.f[4])[c];
  const A32<const T> pin(TRAIL ? trail + 5 * n : par ? S.psi2 : S.psi);
  const bool mono = M.coef[2] != nullptr, atten = M.coef[10] != nullptr;
  const T n11 = A32<const T>(M.coef[0])[c], n13 = A32<const T>(M.coef[1])[c], n33 = A32<const T>(M.coef[3])[c];
  const T s55 = A32<const T>(M.coef[7])[c];
  const T n15 = mono ? A32<const T>(M.coef[2])[c] : T(0), n35 = mono ? A32<const T>(M.coef[4])[c] : T(0);
  const T s15 = mono ? A32<const T>(M.coef[5])[c] : T(0), s35 = mono ? A32<const T>(M.coef[6])[c] : T(0);
  const T dtx = A32<const T>(M.coef[8])[c], dtz = A32<const T>(M.coef[9])[c];
  const T omx = atten ? A32<const T>(M.coef[10])[c] : T(1), omz = atten ? A32<const T>(M.coef[11])[c] : T(1);
  const int lx = M.lx, lz = M.lz;
  const bool inx = PML && in && in_slab(i, nx, lx), inz = PML && in && in_slab(r, nz, lz);
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx, ZB = (SPLIT ? 6 : 4) * SX;
  const uint32_t ox = inx ? (uint32_t)r * 2 * lx + slab_pos(i, nx, lx) : 0;
  const uint32_t oz = inz ? (uint32_t)slab_pos(r, nz, lz) * nx + i : 0;
  T m_vxx = 0, m_vzx = 0, m_sxx = 0, m_sxzx = 0, m_vzz = 0, m_vxz = 0, m_szz = 0, m_sxzz = 0;
  constexpr bool SH = ElRegionLds<T, SPLIT>::SH;
  T sh[4] = {0, 0, 0, 0};
  T& s_vxx = SH ? L.sh[0][ty][tx] : sh[0];
  T& s_vzx = SH ? L.sh[SH ? 1 : 0][ty][tx] : sh[1];
  T& s_vzz = SH ? L.sh[SH ? 2 : 0][ty][tx] : sh[2];
  T& s_vxz = SH ? L.sh[SH ? 3 : 0][ty][tx] : sh[3];
  if (inx) {
    m_vxx = pin[ox]; m_vzx = pin[SX + ox]; m_sxx = pin[2 * SX + ox]; m_sxzx = pin[3 * SX + ox];
    if (SPLIT) { s_vxx = pin[4 * SX + ox]; s_vzx = pin[5 * SX + ox]; }
  }
  if (inz) {
    const uint32_t q = ZB + oz;
    m_vzz = pin[q]; m_vxz = pin[SZ + q]; m_szz = pin[2 * SZ + q]; m_sxzz = pin[3 * SZ + q];
    if (SPLIT) { s_vzz = pin[4 * SZ + q]; s_vxz = pin[5 * SZ + q]; }
  }
  if (PML) {
    // (z entry 6: the legacy normal loop's decay of memory_dvx_dx, b_x_half by row)
    if (threadIdx.x < 6 * RM) {
      L.px[threadIdx.x / RM][tx] = cp<T>(M.prof[0][threadIdx.x / RM])[min(max(x0 + tx, 0), nx - 1)];
    } else if (threadIdx.x >= 256 && threadIdx.x < 256 + 7 * RM) {
      const int q = (threadIdx.x - 256) / RM, zr = min(max(z0 + tx, 0), nz - 1);
      L.pz[q][tx] = q < 6 ? cp<T>(M.prof[2][q])[zr] : SPLIT ? T(0) : cp<T>(M.aux)[zr];
    }
  }
  if (threadIdx.x >= 512 && threadIdx.x < 512 + 5 * TM_MAX) {  // (read after the first barrier)
    const int q = (threadIdx.x - 512) / TM_MAX, t = (threadIdx.x - 512) % TM_MAX;
    const void* a = q == 0 ? S.src[0] : q == 1 ? S.src[2] : S.msrc[q == 2 ? 0 : q == 3 ? 2 : 4];
    L.src[q][t] = a && t < nsteps ? cp<T>(a)[it0 + t] : T(0);
  }
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dt = T(M.dt);
  const bool issrc = in && i == S.isrc && r == S.ksrc;
  const bool msrc = S.msrc[0] || S.msrc[2] || S.msrc[4];
  RegionRec rec[1];
  if (!TRAIL) region_receivers<1>(S, L.slot, x0, z0, nz, tm, zt, osx, osz, {own}, rec);
  int bad = INT_MAX;
  auto store = [&](void* o0, void* o1, void* o2, void* o3, void* o4, void* o5) {
    A32<T>{o0}[c] = vx;
    A32<T>{o1}[c] = vz;
    A32<T>{o2}[c] = sxx;
    A32<T>{o3}[c] = szz;
    A32<T>{o4}[c] = sxz;
    // (array q by its scalar base: one offset register for all)
    T* const px = static_cast<T*>(o5);
    T* const pz = px + ZB;
    if (inx) {
      A32<T>{px}[ox] = m_vxx; A32<T>{px + SX}[ox] = m_vzx; A32<T>{px + 2 * SX}[ox] = m_sxx;
      A32<T>{px + 3 * SX}[ox] = m_sxzx;
      if (SPLIT) { A32<T>{px + 4 * SX}[ox] = s_vxx; A32<T>{px + 5 * SX}[ox] = s_vzx; }
    }
    if (inz) {
      A32<T>{pz}[oz] = m_vzz; A32<T>{pz + SZ}[oz] = m_vxz; A32<T>{pz + 2 * SZ}[oz] = m_szz;
      A32<T>{pz + 3 * SZ}[oz] = m_sxzz;
      if (SPLIT) { A32<T>{pz + 4 * SZ}[oz] = s_vzz; A32<T>{pz + 5 * SZ}[oz] = s_vxz; }
    }
  };
  const int tu = ty > 0 ? ty - 1 : 0, td = ty < RM - 1 ? ty + 1 : RM - 1;
  for (int t = 0; t < nsteps; ++t) {
    // ---- stresses (seismicfdtd.f95:247-312) ----
    L.v[0][ty][tx] = vx;
    L.v[1][ty][tx] = vz;
    __syncthreads();
    {
      const T vx_e = dpp_next(vx), vz_e = dpp_next(vz), vx_w = dpp_prev(vx), vz_w = dpp_prev(vz);
      const T vx_m = L.v[0][tu][tx], vz_m = L.v[1][tu][tx], vx_n = L.v[0][td][tx], vz_n = L.v[1][td][tx];
      if (!PML || (in && i <= nx - 2 && r >= 1)) {
        T dvx_dx = (vx_e - vx) * idx;
        T dvz_dz = (vz - vz_m) * idz;
        T dvz_dx = (vz_e - vz) * idx;
        T dvx_dz = (vx - vx_m) * idz;
        if (inx) {
          m_vxx = fma(SPLIT ? L.px[PBH][tx] : L.pz[6][ty], m_vxx, L.px[PAH][tx] * dvx_dx);  // :255
          m_vzx = fma(L.px[PB][tx], m_vzx, L.px[PA][tx] * dvz_dx);
          dvx_dx = fma(dvx_dx, L.px[PKH][tx], m_vxx);
          dvz_dx = fma(dvz_dx, L.px[PK][tx], m_vzx);
        }
        if (inz) {
          m_vzz = fma(L.pz[PB][ty], m_vzz, L.pz[PA][ty] * dvz_dz);
          m_vxz = fma(L.pz[PBH][ty], m_vxz, L.pz[PAH][ty] * dvx_dz);
          dvz_dz = fma(dvz_dz, L.pz[PK][ty], m_vzz);
          dvx_dz = fma(dvx_dz, L.pz[PKH][ty], m_vxz);
        }
        const T sh = dvz_dx + dvx_dz;
        sxx = fma(fma(n15, sh, fma(n13, dvz_dz, n11 * dvx_dx)), dt, sxx);
        szz = fma(fma(n35, sh, fma(n33, dvz_dz, n13 * dvx_dx)), dt, szz);
      }
      if (!PML || (in && i >= 1 && r <= nz - 2)) {  // same psi arrays (A1) unless split
        T& q_vxx = SPLIT ? s_vxx : m_vxx;
        T& q_vzx = SPLIT ? s_vzx : m_vzx;
        T& q_vzz = SPLIT ? s_vzz : m_vzz;
        T& q_vxz = SPLIT ? s_vxz : m_vxz;
        T dvx_dx = (vx - vx_w) * idx;
        T dvz_dz = (vz_n - vz) * idz;
        T dvz_dx = (vz - vz_w) * idx;
        T dvx_dz = (vx_n - vx) * idz;
        if (inx) {
          q_vxx = fma(L.px[PBH][tx], q_vxx, L.px[PAH][tx] * dvx_dx);
          q_vzx = fma(L.px[PB][tx], q_vzx, L.px[PA][tx] * dvz_dx);
          dvx_dx = fma(dvx_dx, L.px[PKH][tx], q_vxx);
          dvz_dx = fma(dvz_dx, L.px[PK][tx], q_vzx);
        }
        if (inz) {
          q_vzz = fma(L.pz[PB][ty], q_vzz, L.pz[PA][ty] * dvz_dz);
          q_vxz = fma(L.pz[PBH][ty], q_vxz, L.pz[PAH][ty] * dvx_dz);
          dvz_dz = fma(dvz_dz, L.pz[PK][ty], q_vzz);
          dvx_dz = fma(dvx_dz, L.pz[PKH][ty], q_vxz);
        }
        sxz = fma(fma(s55, dvz_dx + dvx_dz, fma(s35, dvz_dz, s15 * dvx_dx)), dt, sxz);
      }
      if (msrc && issrc) {
        sxx += L.src[2][t];
        szz += L.src[3][t];
        sxz += L.src[4][t];
      }
    }
    // ---- velocities (:317-375) ----
    L.s[0][ty][tx] = sxz;
    L.s[1][ty][tx] = szz;
    __syncthreads();
    {
      const T sxx_w = dpp_prev(sxx), sxz_e = dpp_next(sxz);
      const T sxz_u = L.s[0][tu][tx], szz_d = L.s[1][td][tx];
      if (!PML || (in && i >= 1 && r >= 1)) {
        T a = (sxx - sxx_w) * idx;
        T b = (sxz - sxz_u) * idz;
        if (inx) {
          m_sxx = fma(L.px[PB][tx], m_sxx, L.px[PA][tx] * a);
          a = fma(a, L.px[PK][tx], m_sxx);
        }
        if (inz) {
          m_sxzz = fma(L.pz[PB][ty], m_sxzz, L.pz[PA][ty] * b);
          b = fma(b, L.pz[PK][ty], m_sxzz);
        }
        vx = fma(vx, omx, (a + b) * dtx);
      }
      if (!PML || (in && i <= nx - 2 && r <= nz - 2)) {
        T a = (sxz_e - sxz) * idx;
        T b = (szz_d - szz) * idz;
        if (inx) {
          m_sxzx = fma(L.px[PBH][tx], m_sxzx, L.px[PAH][tx] * a);
          a = fma(a, L.px[PKH][tx], m_sxzx);
        }
        if (inz) {
          m_szz = fma(L.pz[PBH][ty], m_szz, L.pz[PAH][ty] * b);
          b = fma(b, L.pz[PKH][ty], m_szz);
        }
        vz = fma(vz, omz, (a + b) * dtz);
      }
      if (issrc) {  // :359-361
        vx += L.src[0][t];
        vz += L.src[1][t];
      }
      if (PML && (i <= 0 || i >= nx - 1 || r <= 0 || r >= nz - 1)) { vx = 0; vz = 0; }  // :365-375
      if (TRAIL && own) {
        T* const o = trail + (t + 1) * ts.adj->slot;
        store(o, o + n, o + 2 * n, o + 3 * n, o + 4 * n, o + 5 * n);
      } else if (own) {
        if (!((double)vx * vx + (double)vz * vz <= 1.0e50)) bad = min(bad, it0 + t);
        region_sample<T>(S, it0 + t, i, r, rec[0], vx, vz);
      }
    }
  }
  if (!TRAIL && own) {
    if (par)
      store(S.f[0], S.f[1], S.f[2], S.f[3], S.f[4], S.psi);
    else
      store(S.g[0], S.g[1], S.g[2], S.g[3], S.g[4], S.psi2);
    if (bad != INT_MAX) atomicMin(S.blowup, bad);
  }
}

// Whether no cell of the region at (x0, z0) lies in a slab or on the outer two
// rows or columns (the rings of the EM fields' shorter extents included).
__device__ __forceinline__ bool region_interior(const DModel& M, int x0, int z0) {
  return x0 >= max(M.lx, 1) && x0 + RM <= M.nx - max(M.lx, 2) && z0 >= max(M.lz, 1) &&
         z0 + RM <= M.nz - max(M.lz, 2);
}

template <typename T, bool SPLIT, bool TRAIL>
__global__ void __launch_bounds__(RM* RM, sizeof(T) == 4 ? 8 : 4)
k_el2_multi(const DModel* __restrict__ models, const DShot* __restrict__ shots, const int4* __restrict__ work,
            int n, const int* __restrict__ base, int rel, int nsteps, int tm, int par,
            const DAdj* __restrict__ adj, const int* __restrict__ tsel) {
  __shared__ ElRegionLds<T, SPLIT> L;
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const int mf = __builtin_amdgcn_readfirstlane(wv.w);
  const bool x1 = SPLIT || (mf & REGION_X1), z1 = SPLIT || (mf & REGION_Z1);
  const DModel& M = models[mf & (REGION_Z1 - 1)];
  const int it0 = __builtin_amdgcn_readfirstlane(*base + rel);
  const int x0 = __builtin_amdgcn_readfirstlane(wv.y) - tm;
  const int z0 = __builtin_amdgcn_readfirstlane(wv.z) - region_top(z1, tm);
  const TrailSlot ts{TRAIL ? adj + s : nullptr, TRAIL ? __builtin_amdgcn_readfirstlane(*tsel) : 0, rel};
  if (region_interior(M, x0, z0))
    el2_region<T, SPLIT, false, TRAIL>(M, S, x0, z0, x1, z1, it0, nsteps, tm, par, ts, L);
  else
    el2_region<T, SPLIT, true, TRAIL>(M, S, x0, z0, x1, z1, it0, nsteps, tm, par, ts, L);
}

// EK: rows per thread.  With two, the z neighbour of one of them is in the
// thread's own registers and four FP32 regions share a CU (59 registers), so
// that the loads of one run beside the steps of the others; a plan whose
// regions all run at once wants the wavefronts of one row per thread, and two
// FP64 rows take 84 registers.  Measured (us per step, EK 1 then 2): FP32 32
// shots of 1064x808 107 -> 87, 8 of 740x540 13.6 -> 11.4, 32 of 2088x1540 374 ->
// 313, 3 of 340x240 2.8 -> 3.0, 130x110 1.5 -> 2.0; FP64 1064x808 6.1 -> 6.5, 32 shots
// 156 -> 164; the recomputation, which its stores bound, 52 -> 52.
template <typename T, int EK>
struct EmRegionLds {
  T ex[RM / EK][RM], hy[RM / EK][RM];  // the threads' first rows' Ex, last rows' Hy
  T px[6][RM], pz[6][RM];
  T src[2][TM_MAX];  // source increments of the steps: Ex, Ez
  int slot[RM * RM];
};

// psi slabs and stages of k_em2_step.
template <typename T, bool PML, bool TRAIL, int EK>
__device__ __forceinline__ void em2_region(const DModel& M, const DShot& S, const int x0, const int z0,
                                           const int it0, const int nsteps, const int tm, const int par,
                                           const TrailSlot ts, EmRegionLds<T, EK>& L) {
#pragma clang fp contract(off)
  const int nx = M.nx, nz = M.nz, lx = M.lx, lz = M.lz;
  const int tx = threadIdx.x & (RM - 1), tq = threadIdx.x / RM;
  const int i = x0 + tx, osz = RM - 2 * tm;
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const long n = (long)nx * nz;
  T* const trail = TRAIL ? static_cast<T*>(ts.adj->trail[ts.tb]) + ts.slot * ts.adj->slot : nullptr;
  const A32<const T> exi(TRAIL ? trail : par ? S.g[0] : S.f[0]);
  const A32<const T> ezi(TRAIL ? trail + n : par ? S.g[1] : S.f[1]);
  const A32<const T> hyi(TRAIL ? trail + 2 * n : par ? S.g[2] : S.f[2]);
  const A32<const T> pin(TRAIL ? trail + 3 * n : par ? S.psi2 : S.psi);
  const A32<const T> CAX(M.coef[0]), CBX(M.coef[1]), CAZ(M.coef[2]), CBZ(M.coef[3]);
  bool in[EK], own[EK], inx[EK], inz[EK], issrc[EK];
  uint32_t c[EK], ox[EK], oz[EK];
  T ex[EK], ez[EK], hy[EK], cax[EK], cbx[EK], caz[EK], cbz[EK];
  T m_ezx[EK], m_hyx[EK], m_exz[EK], m_hyz[EK];
#pragma unroll
  for (int k = 0; k < EK; ++k) {
    const int ty = EK * tq + k, r = z0 + ty;
    in[k] = !PML || (i >= 0 && i < nx && r >= 0 && r < nz);
    const int ic = PML ? min(max(i, 0), nx - 1) : i, rc = PML ? min(max(r, 0), nz - 1) : r;
    own[k] = in[k] && tx >= tm && tx < tm + osz && ty >= tm && ty < tm + osz;
    issrc[k] = in[k] && i == S.isrc && r == S.ksrc;
    c[k] = (uint32_t)rc * nx + ic;
    ex[k] = exi[c[k]];
    ez[k] = ezi[c[k]];
    hy[k] = hyi[c[k]];
    cax[k] = CAX[c[k]];
    cbx[k] = CBX[c[k]];
    caz[k] = CAZ[c[k]];
    cbz[k] = CBZ[c[k]];
    inx[k] = PML && in[k] && in_slab(i, nx, lx);
    inz[k] = PML && in[k] && in_slab(r, nz, lz);
    ox[k] = inx[k] ? (uint32_t)r * 2 * lx + slab_pos(i, nx, lx) : 0;
    oz[k] = 2 * SX + (inz[k] ? (uint32_t)slab_pos(r, nz, lz) * nx + i : 0);
    m_ezx[k] = inx[k] ? pin[ox[k]] : T(0);
    m_hyx[k] = inx[k] ? pin[SX + ox[k]] : T(0);
    m_exz[k] = inz[k] ? pin[oz[k]] : T(0);
    m_hyz[k] = inz[k] ? pin[SZ + oz[k]] : T(0);
  }
  if (PML) {
    if (threadIdx.x < 6 * RM) {
      L.px[tq][tx] = cp<T>(M.prof[0][tq])[min(max(x0 + tx, 0), nx - 1)];
    } else if (threadIdx.x >= 256 && threadIdx.x < 256 + 6 * RM) {
      L.pz[tq - 8][tx] = cp<T>(M.prof[2][tq - 8])[min(max(z0 + tx, 0), nz - 1)];
    }
  }
  if (threadIdx.x >= 480 && threadIdx.x < 480 + 2 * TM_MAX) {  // (read after the first barrier)
    const int q = (threadIdx.x - 480) / TM_MAX, t = (threadIdx.x - 480) % TM_MAX;
    const void* a = q == 0 ? S.src[0] : S.src[2];
    L.src[q][t] = a && t < nsteps ? cp<T>(a)[it0 + t] : T(0);
  }
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dbh = T(M.scal[0]);
  RegionRec rec[EK];
  if (!TRAIL) region_receivers<EK>(S, L.slot, x0, z0, nz, tm, tm, osz, osz, own, rec);
  int bad = INT_MAX;
  auto store = [&](int k, void* o0, void* o1, void* o2, void* o3) {
    A32<T>{o0}[c[k]] = ex[k];
    A32<T>{o1}[c[k]] = ez[k];
    A32<T>{o2}[c[k]] = hy[k];
    const A32<T> pout(o3);
    if (inx[k]) { pout[ox[k]] = m_ezx[k]; pout[SX + ox[k]] = m_hyx[k]; }
    if (inz[k]) { pout[oz[k]] = m_exz[k]; pout[SZ + oz[k]] = m_hyz[k]; }
  };
  const int tu = tq > 0 ? tq - 1 : 0, td = tq < RM / EK - 1 ? tq + 1 : RM / EK - 1;
  for (int t = 0; t < nsteps; ++t) {
    // ---- Hy (electromagfdtd.f95:249-266) ----
    L.ex[tq][tx] = ex[0];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EK; ++k) {
      const int ty = EK * tq + k, r = z0 + ty;
      const T ez_e = dpp_next(ez[k]), ex_n = k + 1 < EK ? ex[(k + 1) % EK] : L.ex[td][tx];
      if (!PML || (in[k] && i <= nx - 2 && r <= nz - 2)) {
        T a = (ex_n - ex[k]) * idz;
        if (inz[k]) {
          m_exz[k] = fma(L.pz[PB][ty], m_exz[k], L.pz[PA][ty] * a);
          a = fma(a, L.pz[PK][ty], m_exz[k]);
        }
        T b = (ez_e - ez[k]) * idx;
        if (inx[k]) {
          m_ezx[k] = fma(L.px[PB][tx], m_ezx[k], L.px[PA][tx] * b);
          b = fma(b, L.px[PK][tx], m_ezx[k]);
        }
        // (the zeroing of the ring that ends the last step, :312-315)
        const bool edge = PML && (i == 0 || i == nx - 2 || r == 0 || r == nz - 2);
        hy[k] = fma(dbh, b + a, edge ? T(0) : hy[k]);
      }
    }
    // ---- Ex, Ez (:273-295), source, Dirichlet ----
    L.hy[tq][tx] = hy[EK - 1];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EK; ++k) {
      const int ty = EK * tq + k, r = z0 + ty;
      const T hy_w = dpp_prev(hy[k]), hy_p = k > 0 ? hy[(k + EK - 1) % EK] : L.hy[tu][tx];
      if (!PML || (in[k] && i <= nx - 2 && r >= 1 && r <= nz - 2)) {
        T d = (hy[k] - hy_p) * idz;
        if (inz[k]) {
          m_hyz[k] = fma(L.pz[PBH][ty], m_hyz[k], L.pz[PAH][ty] * d);
          d = fma(d, L.pz[PKH][ty], m_hyz[k]);
        }
        ex[k] = fma(cax[k], ex[k], cbx[k] * d);
      }
      if (!PML || (in[k] && i >= 1 && i <= nx - 2 && r <= nz - 2)) {
        T d = (hy[k] - hy_w) * idx;
        if (inx[k]) {
          m_hyx[k] = fma(L.px[PBH][tx], m_hyx[k], L.px[PAH][tx] * d);
          d = fma(d, L.px[PKH][tx], m_hyx[k]);
        }
        ez[k] = fma(caz[k], ez[k], cbz[k] * d);
      }
      if (issrc[k]) {
        ex[k] += L.src[0][t];
        ez[k] += L.src[1][t];
      }
      if (PML) {  // :304-311, and the cells outside the fields' extents
        if (i <= 0 || i >= nx - 2 || r <= 0 || r >= nz - 1) ex[k] = 0;
        if (i <= 0 || i >= nx - 1 || r <= 0 || r >= nz - 2) ez[k] = 0;
      }
      if (TRAIL && own[k]) {
        T* const o = trail + (t + 1) * ts.adj->slot;
        store(k, o, o + n, o + 2 * n, o + 3 * n);
      } else if (own[k]) {
        if (!((double)ex[k] * ex[k] + (double)ez[k] * ez[k] <= 1.0e50)) bad = min(bad, it0 + t);
        region_sample<T>(S, it0 + t, i, r, rec[k], ex[k], ez[k]);
      }
    }
  }
  if (TRAIL) return;
#pragma unroll
  for (int k = 0; k < EK; ++k)
    if (own[k]) {
      if (par)
        store(k, S.f[0], S.f[1], S.f[2], S.psi);
      else
        store(k, S.g[0], S.g[1], S.g[2], S.psi2);
    }
  if (bad != INT_MAX) atomicMin(S.blowup, bad);
}

template <typename T, bool TRAIL, int EK>
__global__ void __launch_bounds__(RM* RM / EK, 8)
k_em2_multi(const DModel* __restrict__ models, const DShot* __restrict__ shots, const int4* __restrict__ work,
            int n, const int* __restrict__ base, int rel, int nsteps, int tm, int par,
            const DAdj* __restrict__ adj, const int* __restrict__ tsel) {
  __shared__ EmRegionLds<T, EK> L;
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const DModel& M = models[__builtin_amdgcn_readfirstlane(wv.w)];
  const int it0 = __builtin_amdgcn_readfirstlane(*base + rel);
  const int x0 = __builtin_amdgcn_readfirstlane(wv.y) - tm, z0 = __builtin_amdgcn_readfirstlane(wv.z) - tm;
  const TrailSlot ts{TRAIL ? adj + s : nullptr, TRAIL ? __builtin_amdgcn_readfirstlane(*tsel) : 0, rel};
  if (region_interior(M, x0, z0))
    em2_region<T, false, TRAIL, EK>(M, S, x0, z0, it0, nsteps, tm, par, ts, L);
  else
    em2_region<T, true, TRAIL, EK>(M, S, x0, z0, it0, nsteps, tm, par, ts, L);
}

// ===========================================================================
// EM2 adjoint: the transpose of one EM2 step (k_em2_step), for gradients
// of a trace misfit with respect to the E-update coefficients (caEx cbEx
// caEz cbEz, from permittivity and conductivity).  No counterpart in the
// reference.  The step as the device runs it: Hy' = m * Hy + dbH (dEz_dx +
// dEx_dz) with m = 0 on the Hy Dirichlet ring (the legacy zeroes it at the
// end of the previous step, electromagfdtd.f95:312-315), then Ex, Ez from
// Hy' (:273-295), source, Dirichlet (:304-311).  Three launches, like the
// elastic reference kernels: E^T (scratch planes 0, 1: adjoints of dHy_dz
// at Ex nodes and of dHy_dx at Ez nodes), H^T (gathers them into lambda_Hy;
// planes 2, 3: adjoints of dEx_dz and dEz_dx), and the E gather.
// psi slabs: x [nz][2lx]: dEz_dx dHy_dx ; z [2lz][nx]: dEx_dz dHy_dz.
// ===========================================================================
template <typename T>
__global__ void __launch_bounds__(NT)
k_em2_adj_e(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k,
            const int* __restrict__ tsel, unsigned gmask) {
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const int t = *tbase + k;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  const int lx = M.lx, lz = M.lz;
  const long SX = (long)nz * 2 * lx, SZ = (long)2 * lz * nx;
  const auto Lin = cp<T>(A.lam[(t + 1) & 1]);
  auto Lout = mp<T>(A.lam[t & 1]);
  const auto u1 = cp<T>(A.trail[*tsel]) + (long)(k + 1) * A.slot;
  const auto u0 = cp<T>(A.trail[*tsel]) + (long)k * A.slot;
  auto W = mp<T>(A.work);
  auto G = GAcc<T>::of(A);
  const Prof<T> P(&M.prof[0][0]);
  const bool inx = in_slab(i, nx, lx), inz = in_slab(j, nz, lz);
  const long ox = 3 * n + (inx ? (long)j * 2 * lx + slab_pos(i, nx, lx) : 0);
  const long oz = 3 * n + 2 * SX + (inz ? (long)slab_pos(j, nz, lz) * nx + i : 0);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz);
  // Dirichlet ring of Ex and Ez (and cells outside their Fortran extent)
  const bool edx = (i == 0 || i >= nx - 2 || j == 0 || j == nz - 1);
  const bool edz = (i == 0 || i == nx - 1 || j == 0 || j >= nz - 2);
  const T lex = edx ? T(0) : Lin[c], lez = edz ? T(0) : Lin[n + c];
  if (A.gsrc && i == S.isrc && j == S.ksrc) {
    A.gsrc[3 * (long)t + 0] = (double)lex;
    A.gsrc[3 * (long)t + 2] = (double)lez;
  }
  T wx = 0, wz = 0;
  if (j >= 1 && j <= nz - 2 && i <= nx - 2) {  // Ex node, :273-283
    const T ld = cp<T>(M.coef[1])[c] * lex;
    const T d = (u1[2 * n + c] - u1[2 * n + c - nx]) * idz;
    T D = d;
    wx = ld;
    if (inz) {
      const T lr = Lin[oz + SZ] + ld;
      wx = P[12 + PKH][j] * ld + P[12 + PAH][j] * lr;
      Lout[oz + SZ] = P[12 + PBH][j] * lr;
      D = P[12 + PKH][j] * d + u1[oz + SZ];
    }
    if (gmask & 1u) gadd(G + c, (double)lex * (double)u0[c]);
    if (gmask & 2u) gadd(G + n + c, (double)lex * (double)D);
    Lout[c] = cp<T>(M.coef[0])[c] * lex;
  } else {
    if (inz) Lout[oz + SZ] = Lin[oz + SZ];
    Lout[c] = lex;
  }
  if (j <= nz - 2 && i >= 1 && i <= nx - 2) {  // Ez node, :285-295
    const T le = cp<T>(M.coef[3])[c] * lez;
    const T e = (u1[2 * n + c] - u1[2 * n + c - 1]) * idx;
    T E = e;
    wz = le;
    if (inx) {
      const T lr = Lin[ox + SX] + le;
      wz = P[PKH][i] * le + P[PAH][i] * lr;
      Lout[ox + SX] = P[PBH][i] * lr;
      E = P[PKH][i] * e + u1[ox + SX];
    }
    if (gmask & 4u) gadd(G + 2 * n + c, (double)lez * (double)u0[n + c]);
    if (gmask & 8u) gadd(G + 3 * n + c, (double)lez * (double)E);
    Lout[n + c] = cp<T>(M.coef[2])[c] * lez;
  } else {
    if (inx) Lout[ox + SX] = Lin[ox + SX];
    Lout[n + c] = lez;
  }
  W[c] = wx;
  W[n + c] = wz;
}

template <typename T>
__global__ void __launch_bounds__(NT)
k_em2_adj_h(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k) {
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const int t = *tbase + k;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  const int lx = M.lx, lz = M.lz;
  const long SX = (long)nz * 2 * lx;
  const auto Lin = cp<T>(A.lam[(t + 1) & 1]);
  auto Lout = mp<T>(A.lam[t & 1]);
  auto W = mp<T>(A.work);
  const Prof<T> P(&M.prof[0][0]);
  const bool inx = in_slab(i, nx, lx), inz = in_slab(j, nz, lz);
  const long ox = 3 * n + (inx ? (long)j * 2 * lx + slab_pos(i, nx, lx) : 0);
  const long oz = 3 * n + 2 * SX + (inz ? (long)slab_pos(j, nz, lz) * nx + i : 0);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz);
  // Hy' feeds the E updates through dHy_dz (Ex node c, c+nx) and dHy_dx (Ez node c, c+1)
  const T lh = Lin[2 * n + c] + idz * (W[c] - (j + 1 < nz ? W[c + nx] : T(0))) +
               idx * (W[n + c] - (i + 1 < nx ? W[n + c + 1] : T(0)));
  T la = 0, lb = 0;
  if (i <= nx - 2 && j <= nz - 2) {  // Hy node, :249-266
    const bool ring = (i == 0 || i == nx - 2 || j == 0 || j == nz - 2);
    Lout[2 * n + c] = ring ? T(0) : lh;
    const T w = T(M.scal[0]) * lh;
    la = w;
    lb = w;
    if (inz) {
      const T lr = Lin[oz] + w;
      la = P[12 + PK][j] * w + P[12 + PA][j] * lr;
      Lout[oz] = P[12 + PB][j] * lr;
    }
    if (inx) {
      const T lr = Lin[ox] + w;
      lb = P[PK][i] * w + P[PA][i] * lr;
      Lout[ox] = P[PB][i] * lr;
    }
  } else {
    Lout[2 * n + c] = lh;
    if (inz) Lout[oz] = Lin[oz];
    if (inx) Lout[ox] = Lin[ox];
  }
  W[2 * n + c] = la;  // adjoint of dEx_dz at the Hy node
  W[3 * n + c] = lb;  // adjoint of dEz_dx at the Hy node
}

template <typename T>
__global__ void __launch_bounds__(NT)
k_em2_adj_g(const DModel* __restrict__ models, const DShot* __restrict__ shots,
            const DAdj* __restrict__ adj, int nshots, const int* __restrict__ tbase, int k) {
  const int s = blockIdx.z;
  if (s >= nshots) return;
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const DAdj& A = adj[s];
  const int nx = M.nx, nz = M.nz;
  const int i = blockIdx.x * TX + threadIdx.x, j = blockIdx.y * TZ + threadIdx.y;
  if (i >= nx || j >= nz) return;
  const int t = *tbase + k;
  const long n = (long)nx * nz, c = (long)j * nx + i;
  auto Lout = mp<T>(A.lam[t & 1]);
  const auto W = cp<T>(A.work);
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz);
  Lout[c] = Lout[c] + idz * ((j >= 1 ? W[2 * n + c - nx] : T(0)) - W[2 * n + c]);
  Lout[n + c] = Lout[n + c] + idx * ((i >= 1 ? W[3 * n + c - 1] : T(0)) - W[3 * n + c]);
}

// ---------------------------------------------------------------------------
// Fused EM2 adjoint step: the transpose of k_em2_adj_{e,h,g} in one launch, on
// blocks of 64 columns x AR rows like k_el2_adj: E^T of every cell, H^T (which
// reads the E^T results of the cells to the east and south), the E gather
// (the H^T results of the cells to the west and north).  Blocks own all but a
// ring of one cell.
// ---------------------------------------------------------------------------
template <typename T>
struct EmAdjLds {
  static constexpr int R = AR<T, true>;
  T wx[R][64], hy[R][64], la[R][64];  // E^T's adjoint of dHy_dz; u_{t+1}'s Hy; H^T's of dEx_dz
  T rs[2][R][64];                     // adj_residual
};

template <typename T, bool PML>
__device__ __forceinline__ void em2_adj_block(const DModel& M, const DShot& S, const DAdj& A, const int x0,
                                              const int z0, const int t, const int t0, const int tb,
                                              const unsigned gmask, EmAdjLds<T>& L) {
  using Own = EmAdjOwn<T>;
  constexpr int R = AR<T, true>;
  const int nx = M.nx, nz = M.nz, lx = M.lx, lz = M.lz;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = x0 + lane, r = z0 + w;
  const bool in = !PML || (i >= 0 && i < nx && r >= 0 && r < nz);
  const int ic = PML ? min(max(i, 0), nx - 1) : i, rc = PML ? min(max(r, 0), nz - 1) : r;
  const bool own = in && lane >= Own::x0 && lane < Own::x0 + Own::w && w >= 1 && w <= Own::h;
  // 32-bit element offsets within one state / gradient array (checked at setup)
  const uint32_t n = (uint32_t)nx * nz, c = (uint32_t)rc * nx + ic;
  const A32<const T> Li(A.lam[(t + 1) & 1]);
  const A32<T> Lo(A.lam[t & 1]);
  const T* trail = static_cast<const T*>(A.trail[tb]);
  const A32<const T> u1(trail + (long)(t + 1 - t0) * A.slot), u0(trail + (long)(t - t0) * A.slot);
  T lex = Li[c], lez = Li[n + c], lh = Li[2 * n + c];
  const T hy = u1[2 * n + c];
  const T uex = u0[c], uez = u0[n + c];
  const T cax = A32<const T>(M.coef[0])[c], cbx = A32<const T>(M.coef[1])[c];
  const T caz = A32<const T>(M.coef[2])[c], cbz = A32<const T>(M.coef[3])[c];
  const bool inx = PML && in && in_slab(i, nx, lx), inz = PML && in && in_slab(r, nz, lz);
  const uint32_t SX = (uint32_t)nz * 2 * lx, SZ = (uint32_t)2 * lz * nx;
  const uint32_t ox = 3 * n + (inx ? (uint32_t)r * 2 * lx + slab_pos(i, nx, lx) : 0);
  const uint32_t oz = 3 * n + 2 * SX + (inz ? (uint32_t)slab_pos(r, nz, lz) * nx + i : 0);
  const Prof<T> P(&M.prof[0][0]);
  T ikx = 0, ax = 0, bx = 0, ikxh = 0, axh = 0, bxh = 0, ikz = 0, az = 0, bz = 0, ikzh = 0, azh = 0, bzh = 0;
  T lx0 = 0, lx1 = 0, lz0 = 0, lz1 = 0, ux1 = 0, uz1 = 0;
  if (inx) {
    ikx = P[PK][ic]; ax = P[PA][ic]; bx = P[PB][ic];
    ikxh = P[PKH][ic]; axh = P[PAH][ic]; bxh = P[PBH][ic];
    lx0 = Li[ox]; lx1 = Li[ox + SX]; ux1 = u1[ox + SX];
  }
  if (inz) {
    ikz = P[12 + PK][rc]; az = P[12 + PA][rc]; bz = P[12 + PB][rc];
    ikzh = P[12 + PKH][rc]; azh = P[12 + PAH][rc]; bzh = P[12 + PBH][rc];
    lz0 = Li[oz]; lz1 = Li[oz + SZ]; uz1 = u1[oz + SZ];
  }
  const T idx = T(1.0 / M.dx), idz = T(1.0 / M.dz), dbh = T(M.scal[0]);
  const A32<typename std::remove_pointer<decltype(GAcc<T>::of(A))>::type> G(GAcc<T>::of(A));
  if (S.nrec > 0 && A.resid && r >= 0 && r < nz)
    adj_residual<T>(S, A, t, r, x0, lane, L.rs[0][w], L.rs[1][w], lex, lez);

  // ---- E^T (k_em2_adj_e); the Dirichlet ring of Ex and Ez and the cells
  // outside their extent pass nothing on ----
  if (PML && (i <= 0 || i >= nx - 2 || r <= 0 || r >= nz - 1)) lex = 0;
  if (PML && (i <= 0 || i >= nx - 1 || r <= 0 || r >= nz - 2)) lez = 0;
  if (own && A.gsrc && i == S.isrc && r == S.ksrc) {
    A.gsrc[3 * (long)t + 0] = (double)lex;
    A.gsrc[3 * (long)t + 2] = (double)lez;
  }
  const bool dox = !PML || (in && r >= 1 && r <= nz - 2 && i <= nx - 2);            // Ex node, :273-283
  const bool doz = !PML || (in && r <= nz - 2 && i >= 1 && i <= nx - 2);            // Ez node, :285-295
  T wx = 0, wz = 0, exq = in ? lex : T(0), ezq = in ? lez : T(0);
  if (dox) {
    const T ld = cbx * lex;
    wx = ld;
    if (inz) {
      const T lr = lz1 + ld;
      wx = ikzh * ld + azh * lr;
      lz1 = bzh * lr;
    }
    exq = cax * lex;
  }
  if (doz) {
    const T le = cbz * lez;
    wz = le;
    if (inx) {
      const T lr = lx1 + le;
      wz = ikxh * le + axh * lr;
      lx1 = bxh * lr;
    }
    ezq = caz * lez;
  }
  L.wx[w][lane] = wx;
  L.hy[w][lane] = hy;
  __syncthreads();

  // ---- H^T (k_em2_adj_h): Hy' feeds the E updates through dHy_dz (Ex nodes
  // of this row and the next) and dHy_dx (Ez nodes of this column and the next) ----
  const int wu = w > 0 ? w - 1 : 0, wd = w < R - 1 ? w + 1 : R - 1;
  const T wz_e = dpp_next(wz), hy_w = dpp_prev(hy);
  lh += idz * (wx - L.wx[wd][lane]) + idx * (wz - wz_e);
  T la = 0, lb = 0, out = lh;
  if (!PML || (in && i <= nx - 2 && r <= nz - 2)) {  // Hy node, :249-266
    if (PML && (i == 0 || i == nx - 2 || r == 0 || r == nz - 2)) out = 0;
    const T q = dbh * lh;
    la = q;
    lb = q;
    if (inz) {
      const T lr = lz0 + q;
      la = ikz * q + az * lr;
      lz0 = bz * lr;
    }
    if (inx) {
      const T lr = lx0 + q;
      lb = ikx * q + ax * lr;
      lx0 = bx * lr;
    }
  }
  if (own) {
    if (dox) {
      T D = (hy - L.hy[wu][lane]) * idz;
      if (inz) D = ikzh * D + uz1;
      if (gmask & 1u) gadd(&G[c], (double)lex * (double)uex);
      if (gmask & 2u) gadd(&G[n + c], (double)lex * (double)D);
    }
    if (doz) {
      T E = (hy - hy_w) * idx;
      if (inx) E = ikxh * E + ux1;
      if (gmask & 4u) gadd(&G[2 * n + c], (double)lez * (double)uez);
      if (gmask & 8u) gadd(&G[3 * n + c], (double)lez * (double)E);
    }
    Lo[2 * n + c] = out;
    if (inx) { Lo[ox] = lx0; Lo[ox + SX] = lx1; }
    if (inz) { Lo[oz] = lz0; Lo[oz + SZ] = lz1; }
  }
  L.la[w][lane] = la;
  __syncthreads();

  // ---- E gather (k_em2_adj_g) ----
  const T lb_w = dpp_prev(lb);
  if (own) {
    Lo[c] = exq + idz * (L.la[wu][lane] - la);
    Lo[n + c] = ezq + idx * (lb_w - lb);
  }
}

template <typename T>
__global__ void __launch_bounds__((64 * AR<T, true>), sizeof(T) == 4 ? 8 : 6)
k_em2_adj(const DModel* __restrict__ models, const DShot* __restrict__ shots, const DAdj* __restrict__ adj,
          const int4* __restrict__ work, int nitems, const int* __restrict__ tbase, int k, unsigned gmask,
          const int* __restrict__ tsel) {
  __shared__ EmAdjLds<T> L;
  const int q = item8(nitems);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const int t0 = __builtin_amdgcn_readfirstlane(*tbase), tb = __builtin_amdgcn_readfirstlane(*tsel);
  const DModel& M = models[__builtin_amdgcn_readfirstlane(wv.w)];
  const int x0 = __builtin_amdgcn_readfirstlane(wv.y) - EmAdjOwn<T>::x0;
  const int z0 = __builtin_amdgcn_readfirstlane(wv.z) - 1;
  if (adj_interior(M, x0, z0, AR<T, true>))
    em2_adj_block<T, false>(M, shots[s], adj[s], x0, z0, t0 + k, t0, tb, gmask, L);
  else
    em2_adj_block<T, true>(M, shots[s], adj[s], x0, z0, t0 + k, t0, tb, gmask, L);
}

// ===========================================================================
// EM25: electromag25, legacy/fortran/electromagfdtd.f95:619-1092
// psi slabs: x [nz][ny][2lx]: dEz_dx dEy_dx dHz_dx dHy_dx
//            y [nz][2ly][nx]: dEz_dy dEx_dy dHz_dy dHx_dy
//            z [2lz][ny][nx]: dEy_dz dEx_dz dHy_dz dHx_dz
// H boundary zeroing (:1059-1078) is applied by the next H update.
// Two launches per step (H, then E): a wavefront takes one plane, 64 columns
// (62 owned; x neighbours by DPP lane shifts) and a chunk of rows, R = 4 (FP64
// 2) rows at a time; the z neighbours are loads of the adjacent plane.
// What bounds it is the latency of a row's loads, with the fields streaming
// from HBM on large grids: so all loads of the R rows, C-PML memory included,
// are issued before the first use (34 field loads per lane in flight in FP32),
// and the y neighbours among them come from registers.  A walk of one row at a
// time, whose memory variables were loaded after the wait for the row's fields,
// took (us per step, same chunks) 495 against 429 on 544x96x416 FP32 (3.8
// against 4.4 TB/s of traffic), 865 against 850 in FP64, 219 against 202 on
// 332x72x182 FP64, 37.6 against 30.7 on 133x57x79 FP64, 30 against 19.6 on
// 112x56x82 FP32.  Four rows in FP64 need 180 registers (two wavefronts per
// SIMD): 841 and 32.4 on the large and the small grid.
// ===========================================================================
struct Slab3e {
  long SX, SY, SZ, bx, by, bz;
  __device__ Slab3e(int nx, int ny, int nz, int lx, int ly, int lz) {
    SX = (long)nz * ny * 2 * lx;
    SY = (long)nz * 2 * ly * nx;
    SZ = (long)2 * lz * ny * nx;
    bx = 0;
    by = 4 * SX;
    bz = 4 * SX + 4 * SY;
  }
};

// rows whose loads an EM 2.5-D wavefront has in flight at once
template <typename T>
constexpr int RE25 = sizeof(T) == 4 ? 4 : 2;

// C-PML memory of the EM 2.5-D passes on one plane: arrays q and q + 1 of each
// axis (q = 0 for the H pass, 2 for the E pass).  The bases are wave-uniform,
// the offsets 32-bit: x[j * 2lx + xs], y[slab row * nx + i], z[j * nx + i].
template <typename T>
struct Psi25 {
  const A32<T> x0, x1, y0, y1, z0, z1;
  __device__ __forceinline__ Psi25(void* psi, const Slab3e& L, int q, int nx, int ny, int lx, int ly, int k, int zs)
      : x0((T*)psi + L.bx + q * L.SX + (long)k * ny * 2 * lx), x1((T*)psi + L.bx + (q + 1) * L.SX + (long)k * ny * 2 * lx),
        y0((T*)psi + L.by + q * L.SY + (long)k * 2 * ly * nx), y1((T*)psi + L.by + (q + 1) * L.SY + (long)k * 2 * ly * nx),
        z0((T*)psi + L.bz + q * L.SZ + (long)zs * ny * nx), z1((T*)psi + L.bz + (q + 1) * L.SZ + (long)zs * ny * nx) {}
};

template <typename T, bool PML>
__device__ __forceinline__ void em25_h_tile(const DModel* __restrict__ models,
                                           const DShot* __restrict__ shots, const int4 wv) {
  constexpr int R = RE25<T>;
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const int nx = M.nx, ny = M.ny, nz = M.nz;
  const int k = __builtin_amdgcn_readfirstlane(wv.z);
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane(wv.y) - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);
  // H lives on i <= nx-2, j <= ny-2, k <= nz-2 (the loop ranges of :901-962)
  const bool own = incol && lane >= 1 && lane <= EW25 && i <= nx - 2 && k <= nz - 2;
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w));
  const int j1 = min(ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w)), ny - 1);
  const long nxy = (long)nx * ny;
  const T idx = T(1.0 / M.dx), idy = T(1.0 / M.dy), idz = T(1.0 / M.dz), dbH = T(M.scal[0]);
  const int lx = M.lx, ly = M.ly, lz = M.lz;
  // a chunk lies inside a y slab or outside both
  const bool inx = PML && incol && in_slab(i, nx, lx), inz = PML && in_slab(k, nz, lz);
  const bool iny = PML && in_slab(j0, ny, ly);
  const Prof<T> P(&M.prof[0][0]);
  const T bx_i = P[PB][ic], ax_i = P[PA][ic], ikx_i = P[PK][ic];
  const auto pz = kp<T>(M.prof[2][PK]), pza = kp<T>(M.prof[2][PA]), pzb = kp<T>(M.prof[2][PB]);
  const T ikz_k = pz[k], az_k = pza[k], bz_k = pzb[k];
  const T ikzh_k = kp<T>(M.prof[2][PKH])[k], azh_k = kp<T>(M.prof[2][PAH])[k], bzh_k = kp<T>(M.prof[2][PBH])[k];
  const auto iky = kp<T>(M.prof[1][PK]), ay = kp<T>(M.prof[1][PA]), by = kp<T>(M.prof[1][PB]);
  const auto ikyh = kp<T>(M.prof[1][PKH]), ayh = kp<T>(M.prof[1][PAH]), byh = kp<T>(M.prof[1][PBH]);
  const int ku = k + 1 < nz ? k + 1 : k;
  const A32<const T> EX = cplane<T>(S.f[0], nxy, k), EY = cplane<T>(S.f[1], nxy, k);
  const A32<const T> EZ = cplane<T>(S.f[2], nxy, k);
  const A32<const T> EXU = cplane<T>(S.f[0], nxy, ku), EYU = cplane<T>(S.f[1], nxy, ku);
  const A32<T> HX = plane<T>(S.f[3], nxy, k), HY = plane<T>(S.f[4], nxy, k), HZ = plane<T>(S.f[5], nxy, k);
  const int xs = inx ? slab_pos(i, nx, lx) : 0, zs = inz ? slab_pos(k, nz, lz) : 0;
  const Psi25<T> W(S.psi, Slab3e(nx, ny, nz, lx, ly, lz), 0, nx, ny, lx, ly, k, zs);
#pragma unroll 1
  for (int jb = j0; jb < j1; jb += R) {
    // every load of the R rows before the first use; rows past the chunk
    // reload its last row (E: the row below it, j1 <= ny - 1)
    T ex[R + 1], ez[R + 1], ey[R], eyu[R], exu[R], hx[R], hy[R], hz[R];
    T mx0[R], mx1[R], my0[R], my1[R], mz0[R], mz1[R];
    uint32_t c[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const uint32_t ce = (uint32_t)min(jb + q, j1) * nx + ic;
      c[q] = (uint32_t)min(jb + q, j1 - 1) * nx + ic;
      ex[q] = EX[ce]; ez[q] = EZ[ce]; ey[q] = EY[c[q]];
      eyu[q] = EYU[c[q]]; exu[q] = EXU[c[q]];
      hx[q] = HX[c[q]]; hy[q] = HY[c[q]]; hz[q] = HZ[c[q]];
    }
    const uint32_t cl = (uint32_t)min(jb + R, j1) * nx + ic;
    ex[R] = EX[cl]; ez[R] = EZ[cl];
    if (PML && iny) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)slab_pos(min(jb + q, j1 - 1), ny, ly) * nx + ic;
        my0[q] = W.y0[o]; my1[q] = W.y1[o];
      }
    }
    if (PML && inz) {
#pragma unroll
      for (int q = 0; q < R; ++q) { mz0[q] = W.z0[c[q]]; mz1[q] = W.z1[c[q]]; }
    }
    if (PML && inx) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)min(jb + q, j1 - 1) * 2 * lx + xs;
        mx0[q] = W.x0[o]; mx1[q] = W.x1[o];
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int j = jb + q;
      if (j >= j1) break;
      const T exc = ex[q], ezc = ez[q], exn = ex[q + 1], ezn = ez[q + 1], eyc = ey[q];
      const T eze = dpp_next(ezc), eye = dpp_next(eyc);
      T ay_ = (ezc - ezn) * idy, bz_ = (eyu[q] - eyc) * idz;   // Hx: dEz_dy, dEy_dz (:901-920)
      T az_ = (exc - exu[q]) * idz, bx_ = (eze - ezc) * idx;   // Hy: dEx_dz, dEz_dx (:922-942)
      T cy_ = (exn - exc) * idy, cx_ = (eyc - eye) * idx;      // Hz: dEx_dy, dEy_dx (:944-962)
      if (PML && iny) {
        my0[q] = byh[j] * my0[q] + ayh[j] * ay_; ay_ = ay_ * ikyh[j] + my0[q];
        my1[q] = by[j] * my1[q] + ay[j] * cy_; cy_ = cy_ * iky[j] + my1[q];
      }
      if (PML && inz) {
        mz0[q] = bzh_k * mz0[q] + azh_k * bz_; bz_ = bz_ * ikzh_k + mz0[q];
        mz1[q] = bz_k * mz1[q] + az_k * az_; az_ = az_ * ikz_k + mz1[q];
      }
      if (PML && inx) {
        mx0[q] = bx_i * mx0[q] + ax_i * bx_; bx_ = bx_ * ikx_i + mx0[q];
        mx1[q] = bx_i * mx1[q] + ax_i * cx_; cx_ = cx_ * ikx_i + mx1[q];
      }
      if (own) {
        const bool lo = (i == 0 || j == 0 || k == 0);
        HX[c[q]] = (lo || i == nx - 1 || j == ny - 2 || k == nz - 2 ? T(0) : hx[q]) + dbH * (bz_ + ay_);
        HY[c[q]] = (lo || i == nx - 2 || j == ny - 1 || k == nz - 2 ? T(0) : hy[q]) + dbH * (bx_ + az_);
        if (k >= 1) HZ[c[q]] = (lo || i == nx - 2 || j == ny - 2 || k == nz - 1 ? T(0) : hz[q]) + dbH * (cx_ + cy_);
        if (PML && iny) {
          const uint32_t o = (uint32_t)slab_pos(j, ny, ly) * nx + ic;
          W.y0[o] = my0[q];
          if (k >= 1) W.y1[o] = my1[q];
        }
        if (PML && inz) { W.z0[c[q]] = mz0[q]; W.z1[c[q]] = mz1[q]; }
        if (PML && inx) {
          const uint32_t o = (uint32_t)j * 2 * lx + xs;
          W.x0[o] = mx0[q];
          if (k >= 1) W.x1[o] = mx1[q];
        }
      }
    }
  }
}

template <typename T, bool PML>
__device__ __forceinline__ void em25_e_tile(const DModel* __restrict__ models,
                                           const DShot* __restrict__ shots, const int4 wv,
                                           const int it) {
  constexpr int R = RE25<T>;
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DShot& S = shots[s];
  const DModel& M = models[S.model];
  const int nx = M.nx, ny = M.ny, nz = M.nz;
  const int k = __builtin_amdgcn_readfirstlane(wv.z);
  const int lane = threadIdx.x & 63;
  const int i = __builtin_amdgcn_readfirstlane(wv.y) - 1 + lane;
  const bool incol = (i >= 0 && i < nx);
  const int ic = incol ? i : (i < 0 ? 0 : nx - 1);
  const bool own = incol && lane >= 1 && lane <= EW25;
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w));
  const int j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  const long nxy = (long)nx * ny;
  const uint32_t p = (uint32_t)k * nx + ic;
  const T idx = T(1.0 / M.dx), idy = T(1.0 / M.dy), idz = T(1.0 / M.dz);
  const int lx = M.lx, ly = M.ly, lz = M.lz;
  const bool inx = PML && incol && in_slab(i, nx, lx), inz = PML && in_slab(k, nz, lz);
  const bool iny = PML && in_slab(j0, ny, ly);
  const Prof<T> P(&M.prof[0][0]);
  const T bxh_i = P[PBH][ic], axh_i = P[PAH][ic], ikxh_i = P[PKH][ic];
  const T ikz_k = kp<T>(M.prof[2][PK])[k], az_k = kp<T>(M.prof[2][PA])[k], bz_k = kp<T>(M.prof[2][PB])[k];
  const T ikzh_k = kp<T>(M.prof[2][PKH])[k], azh_k = kp<T>(M.prof[2][PAH])[k], bzh_k = kp<T>(M.prof[2][PBH])[k];
  const auto ikyh = kp<T>(M.prof[1][PKH]), ayh = kp<T>(M.prof[1][PAH]), byh = kp<T>(M.prof[1][PBH]);
  // loop ranges of :968-1029
  const bool ux = own && k >= 1 && k <= nz - 2 && i <= nx - 2;
  const bool uy = own && k >= 1 && k <= nz - 2 && i >= 1 && i <= nx - 2;
  const bool uz = own && k <= nz - 2 && i >= 1 && i <= nx - 2;
  const T cax = A32<const T>(M.coef[0])[p], cbx = A32<const T>(M.coef[1])[p];
  const T cay = A32<const T>(M.coef[2])[p], cby = A32<const T>(M.coef[3])[p];
  const T caz = A32<const T>(M.coef[4])[p], cbz = A32<const T>(M.coef[5])[p];
  const int kd = k >= 1 ? k - 1 : 0;
  const A32<const T> HX = cplane<T>(S.f[3], nxy, k), HY = cplane<T>(S.f[4], nxy, k);
  const A32<const T> HZ = cplane<T>(S.f[5], nxy, k);
  const A32<const T> HXD = cplane<T>(S.f[3], nxy, kd), HYD = cplane<T>(S.f[4], nxy, kd);
  const A32<T> EX = plane<T>(S.f[0], nxy, k), EY = plane<T>(S.f[1], nxy, k), EZ = plane<T>(S.f[2], nxy, k);
  const int xs = inx ? slab_pos(i, nx, lx) : 0, zs = inz ? slab_pos(k, nz, lz) : 0;
  const Psi25<T> W(S.psi, Slab3e(nx, ny, nz, lx, ly, lz), 2, nx, ny, lx, ly, k, zs);
  const bool srccol = (i == S.isrc && k == S.ksrc);
  bool bad = false;
#pragma unroll 1
  for (int jb = j0; jb < j1; jb += R) {
    T hx[R + 1], hz[R + 1], hy[R], hyd[R], hxd[R], ex[R], ey[R], ez[R];
    T mx0[R], mx1[R], my0[R], my1[R], mz0[R], mz1[R];
    uint32_t c[R];
    const uint32_t cm = (uint32_t)max(jb - 1, 0) * nx + ic;  // the row above (row 0 uses none)
    hx[0] = HX[cm]; hz[0] = HZ[cm];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      c[q] = (uint32_t)min(jb + q, j1 - 1) * nx + ic;
      hx[q + 1] = HX[c[q]]; hy[q] = HY[c[q]]; hz[q + 1] = HZ[c[q]];
      hyd[q] = HYD[c[q]]; hxd[q] = HXD[c[q]];
      ex[q] = EX[c[q]]; ey[q] = EY[c[q]]; ez[q] = EZ[c[q]];
    }
    if (PML && iny) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)slab_pos(min(jb + q, j1 - 1), ny, ly) * nx + ic;
        my0[q] = W.y0[o]; my1[q] = W.y1[o];
      }
    }
    if (PML && inz) {
#pragma unroll
      for (int q = 0; q < R; ++q) { mz0[q] = W.z0[c[q]]; mz1[q] = W.z1[c[q]]; }
    }
    if (PML && inx) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const uint32_t o = (uint32_t)min(jb + q, j1 - 1) * 2 * lx + xs;
        mx0[q] = W.x0[o]; mx1[q] = W.x1[o];
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int j = jb + q;
      if (j >= j1) break;
      const T hxc = hx[q + 1], hyc = hy[q], hzc = hz[q + 1], hxm = hx[q], hzm = hz[q];
      const T hzw = dpp_prev(hzc), hyw = dpp_prev(hyc);
      const bool jx = j >= 1 && j <= ny - 2, jy = j <= ny - 2;
      T exn = ex[q], eyn = ey[q], ezn = ez[q];
      if (ux && jx) {  // Ex, :968-985
        T a = (hzc - hzm) * idy, b = (hyd[q] - hyc) * idz;  // dHz_dy, dHy_dz
        if (PML && iny) {
          my0[q] = byh[j] * my0[q] + ayh[j] * a; a = a * ikyh[j] + my0[q];
          W.y0[(uint32_t)slab_pos(j, ny, ly) * nx + ic] = my0[q];
        }
        if (PML && inz) { mz0[q] = bz_k * mz0[q] + az_k * b; b = b * ikz_k + mz0[q]; W.z0[c[q]] = mz0[q]; }
        exn = cax * exn + cbx * (a + b);
      }
      if (uy && jy) {  // Ey, :988-1006
        T a = (hzw - hzc) * idx, b = (hxc - hxd[q]) * idz;  // dHz_dx, dHx_dz
        if (PML && inx) {
          mx0[q] = bxh_i * mx0[q] + axh_i * a; a = a * ikxh_i + mx0[q];
          W.x0[(uint32_t)j * 2 * lx + xs] = mx0[q];
        }
        if (PML && inz) { mz1[q] = bzh_k * mz1[q] + azh_k * b; b = b * ikzh_k + mz1[q]; W.z1[c[q]] = mz1[q]; }
        eyn = cay * eyn + cby * (a + b);
      }
      if (uz && jx) {  // Ez, :1011-1029
        T a = (hxm - hxc) * idy, b = (hyc - hyw) * idx;  // dHx_dy, dHy_dx
        if (PML && iny) {
          my1[q] = byh[j] * my1[q] + ayh[j] * a; a = a * ikyh[j] + my1[q];
          W.y1[(uint32_t)slab_pos(j, ny, ly) * nx + ic] = my1[q];
        }
        if (PML && inx) {
          mx1[q] = bxh_i * mx1[q] + axh_i * b; b = b * ikxh_i + mx1[q];
          W.x1[(uint32_t)j * 2 * lx + xs] = mx1[q];
        }
        ezn = caz * ezn + cbz * (a + b);
      }
      if (srccol && j == S.jsrc && own) {  // source, :1033-1035
        if (S.src[0]) exn += cp<T>(S.src[0])[it];
        if (S.src[1]) eyn += cp<T>(S.src[1])[it];
        if (S.src[2]) ezn += cp<T>(S.src[2])[it];
      }
      // Dirichlet faces, :1038-1057 (and cells outside each staggered field's extent)
      const bool lo = (i == 0 || j == 0 || k == 0);
      if (lo || i >= nx - 2 || j == ny - 1 || k == nz - 1) exn = 0;
      if (lo || i == nx - 1 || j >= ny - 2 || k == nz - 1) eyn = 0;
      if (lo || i == nx - 1 || j == ny - 1 || k >= nz - 2) ezn = 0;
      if (own) {
        bad |= !((double)exn * exn + (double)eyn * eyn + (double)ezn * ezn <= 1.0e50);
        EX[c[q]] = exn;
        EY[c[q]] = eyn;
        EZ[c[q]] = ezn;
      }
    }
  }
  if (bad) atomicMin(S.blowup, it);
}

// A wavefront whose columns, plane and rows (with the neighbours it reads)
// lie outside every C-PML slab runs the body without memory variables.
__device__ __forceinline__ bool em25_interior(const DModel& M, int xo, int k, int j0, int j1) {
  return xo - 1 >= M.lx && xo + 62 < M.nx - M.lx && k >= M.lz && k < M.nz - M.lz &&
         j0 >= M.ly && j1 <= M.ny - M.ly;
}

template <typename T>
__global__ void __launch_bounds__(64)
k_em25_h(const DModel* __restrict__ models, const DShot* __restrict__ shots,
         const int4* __restrict__ work, int n) {
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DModel& M = models[shots[s].model];
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  if (em25_interior(M, __builtin_amdgcn_readfirstlane(wv.y), __builtin_amdgcn_readfirstlane(wv.z), j0, j1))
    em25_h_tile<T, false>(models, shots, wv);
  else
    em25_h_tile<T, true>(models, shots, wv);
}

template <typename T>
__global__ void __launch_bounds__(64)
k_em25_e(const DModel* __restrict__ models, const DShot* __restrict__ shots,
         const int4* __restrict__ work, int n, const int* __restrict__ base, int rel) {
  const int q = item8(n);
  if (q < 0) return;
  const int4 wv = work[q];
  const int s = __builtin_amdgcn_readfirstlane(wv.x);
  const DModel& M = models[shots[s].model];
  const int it = *base + rel;
  const int j0 = ychunk_j0(__builtin_amdgcn_readfirstlane(wv.w)), j1 = ychunk_j1(__builtin_amdgcn_readfirstlane(wv.w));
  if (em25_interior(M, __builtin_amdgcn_readfirstlane(wv.y), __builtin_amdgcn_readfirstlane(wv.z), j0, j1))
    em25_e_tile<T, false>(models, shots, wv, it);
  else
    em25_e_tile<T, true>(models, shots, wv, it);
}

// ===========================================================================
// Receiver gather (replaces arraybuild.py:199-295 reading snapshot files):
// trace[it][comp][r] = field_comp[rec_r] after the step.
// ===========================================================================
template <typename T>
__global__ void k_gather(const DModel* __restrict__ models, const DShot* __restrict__ shots,
                         int s0, int ncomp, const int* __restrict__ base, int rel, int k0, int k1) {
  const DShot& S = shots[s0 + blockIdx.y];
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= S.nrec || S.trace == nullptr) return;
  const DModel& M = models[S.model];
  const int it = *base + rel;
  const auto q = cp<int>(S.rec) + 3 * r;
  if (q[2] < k0 || q[2] >= k1) return;  // only planes k0 .. k1-1 are at this step
  const long c = ((long)q[2] * M.ny + q[1]) * M.nx + q[0];
  auto tr = mp<T>(S.trace) + ((long)it * ncomp) * S.nrec + r;
  for (int f = 0; f < ncomp; ++f) tr[(long)f * S.nrec] = cp<T>(S.f[f])[c];
}

// The H zeroing that closes each legacy 2.5-D EM step (electromagfdtd.f95
// :1059-1078) is folded into the next H update; at the end of a run it is
// applied here (one wavefront per work item of the EM25 kernels) so the
// returned state equals the legacy state.
template <typename T>
__global__ void __launch_bounds__(64)
k_em25_edges(const DModel* __restrict__ models, const DShot* __restrict__ shots,
             const int4* __restrict__ work) {
  const int4 wv = work[blockIdx.x];
  const DShot& S = shots[wv.x];
  const DModel& M = models[S.model];
  const int nx = M.nx, ny = M.ny, nz = M.nz;
  const int lane = threadIdx.x & 63;
  const int i = wv.y - 1 + lane, k = wv.z;
  if (lane < 1 || lane > EW25 || i >= nx || k >= nz) return;
  auto Hx = mp<T>(S.f[3]);
  auto Hy = mp<T>(S.f[4]);
  auto Hz = mp<T>(S.f[5]);
  for (int j = ychunk_j0(wv.w); j < ychunk_j1(wv.w); ++j) {
    const long c = ((long)k * ny + j) * nx + i;
    const bool lo = (i == 0 || j == 0 || k == 0);
    if (lo || i == nx - 1 || j == ny - 2 || k == nz - 2) Hx[c] = T(0);
    if (lo || i == nx - 2 || j == ny - 1 || k == nz - 2) Hy[c] = T(0);
    if (lo || i == nx - 2 || j == ny - 2 || k == nz - 1) Hz[c] = T(0);
  }
}

__global__ void k_set_int(int* p, int v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = v;
}
__global__ void k_set_int2(int* p, int v, int* p2, int v2) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    *p = v;
    *p2 = v2;
  }
}
__global__ void k_add_int(int* p, int v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *p = *p + v;
}
__global__ void k_fill_int(int* p, int n, int v) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

// ===========================================================================
// HBM probe: a copy of known traffic (4 n bytes read, 4 n written) whose
// loads and stores are one 4-byte element per lane, consecutive lanes on
// consecutive addresses -- the access width of the stencil kernels' loads.
// Measurement only: it calibrates the byte counters the stencils' traffic
// is read from.
// ===========================================================================
__global__ void __launch_bounds__(256) k_hbm_probe(const float* __restrict__ src,
                                                   float* __restrict__ dst, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

// ===========================================================================
// Plan
// ===========================================================================
// A block of the 2.5-D schedule (set_blocks25): shots s0..s1-1, or of one shot
// the planes from the previous block's `top` to below this one's (INT_MAX: nz).
struct Block25 {
  int s0, s1, top;
};

struct Plan {
  int kind = 0, prec = 0, nmodels = 0, nshots = 0, nt = 0, ncomp = 2;
  bool split = false;  // SDT_SPLIT_CPML
  int maxrec = 0;
  std::vector<sdt_model> hmodels;
  std::vector<sdt_shot> hshots;
  DModel* dmodels = nullptr;
  DShot* dshots = nullptr;
  int4* dwork = nullptr;
  int nwork = 0;
  std::vector<int> item25;                // 2.5-D: first work item of each shot, and their number
  std::vector<Block25> blocks25;          // 2.5-D: schedule (set_blocks25)
  std::vector<std::pair<int, int>> reck;  // per shot: lowest and highest receiver plane
  int el2_grid = 0;  // persistent grid of the ELASTIC2 step kernel
  int el2_wb = SDT_EL2_WAVES_PER_BLOCK;  // tile: wavefronts per block
  int el2_eh = SDT_EL2_ROWS;             // tile: rows
  int el2_order = 0;  // work-list order: 0 tiles dealt to the XCDs in turn, 1 column strips per XCD
  int spl = 1;                 // steps per launch of the ELASTIC2 step kernel (1 or 2)
  int4* dwork2 = nullptr;      // work list of the two-step kernel: interior blocks first
  int nwork2 = 0, nwork2i = 0;
  int el2x2_grid = 0, el2x2_grid_i = 0;
  int* dit0 = nullptr;         // first step of the current run of two-step launches
  int* drec = nullptr;         // receivers by row of every shot (DShot::rrow, rxid)
  int graph_mode = 0;          // what the cached graph holds (run_mode)
  // several steps per launch on regions (default_regions, run_mode): whether the
  // plan has their list, and whether it may take them (no launch shape asked for)
  bool multi = false, regions = true;
  int4* dwmulti = nullptr;     // work list: (shot, x0, z0, model) per region
  int nmulti = 0, tm = 0;      // tm: most steps per launch, the width of the regions' halo
  bool b_holds = false;        // buffer B holds the current state too (ELASTIC2 / EM2)
  int* dflags = nullptr;  // per shot first unstable step (INT_MAX = none)
  int* dbase = nullptr;   // step index of rel = 0
  long* dnel = nullptr;   // per shot: field elements (ping-pong copy-back)
  long* dnpsi = nullptr;  // per shot: psi elements
  hipStream_t last = nullptr;
  hipStream_t cap = nullptr;  // capture stream
  int graph_block = 0;
  hipGraphExec_t gexec = nullptr;
  hipGraph_t graph = nullptr;
  DAdj* dadj = nullptr;          // adjoint descriptors (sdt_adjoint_setup)
  std::vector<DAdj> hadj;
  int4* dadjwork = nullptr;      // work list of the fused adjoint kernel
  int4* dtrwork = nullptr;       // work list of the trail recomputation (regions)
  int ntrwork = 0, tr_tm = 0;    // its length and its steps per launch
  int* dtbase = nullptr;         // first step of the trail (adjoint kernels)
  int* dtsel_trail = nullptr;    // trail buffer the recomputation writes
  int* dtsel_adj = nullptr;      // trail buffer the adjoint reads
  // captured segments: (kind 0 trail / 1 adjoint, key) -> graph; kept until
  // setup or destroy so a replay in flight is never freed
  struct SegGraph {
    int kind;
    long long key;
    hipGraph_t g;
    hipGraphExec_t e;
  };
  std::vector<SegGraph> seg_graphs;
  std::vector<float*> g32;       // FP32 gradient staging per distinct grad array
  DFlush* dflush = nullptr;
  int nflush = 0;
  int nadjwork = 0;
  unsigned gmask = 0xfffu;       // gradient slots to accumulate
  int adj_flags = 0;
  int maxnx = 0, maxnz = 0;
  long long maxel = 0;           // elements of the largest field or psi
};

int kind_fields(int kind) {
  switch (kind) {
    case SDT_ELASTIC2: return 5;
    case SDT_ELASTIC25: return 9;
    case SDT_EM2: return 3;
    case SDT_EM25: return 6;
  }
  return 0;
}
int kind_ncoef(int kind) {
  switch (kind) {
    case SDT_ELASTIC2: return 12;
    case SDT_ELASTIC25: return 39;
    case SDT_EM2: return 4;
    case SDT_EM25: return 6;
  }
  return 0;
}
bool kind_3d(int kind) { return kind == SDT_ELASTIC25 || kind == SDT_EM25; }
// kinds whose single-pass step reads state A or B and writes the other
bool pingpong(int kind) { return kind == SDT_ELASTIC2 || kind == SDT_EM2; }

// kind may carry SDT_SPLIT_CPML (ELASTIC2 only: two more memory arrays per slab)
long long psi_elems(int kind, long long nx, long long ny, long long nz, long long lx,
                    long long ly, long long lz) {
  if (kind & SDT_SPLIT_CPML) {
    if ((kind & ~SDT_SPLIT_CPML) != SDT_ELASTIC2) return -1;
    return 6 * nz * 2 * lx + 6 * 2 * lz * nx;
  }
  switch (kind) {
    case SDT_ELASTIC2: return 4 * nz * 2 * lx + 4 * 2 * lz * nx;
    case SDT_EM2: return 2 * nz * 2 * lx + 2 * 2 * lz * nx;
    case SDT_ELASTIC25: return 6 * (nz * ny * 2 * lx + nz * 2 * ly * nx + 2 * lz * ny * nx);
    case SDT_EM25: return 4 * (nz * ny * 2 * lx + nz * 2 * ly * nx + 2 * lz * ny * nx);
  }
  return -1;
}

// One launch of the single-pass ELASTIC2 step with the plan's tile shape.
template <typename T, bool SPLIT>
void launch_el2(Plan* p, hipStream_t st, int rel, const int* prun = nullptr) {
  const dim3 g(p->el2_grid);
  const int4* w = p->dwork;
  const int n = p->nwork, wb = p->el2_wb, eh = p->el2_eh;
  if (eh == 1) {  // tiles of one row: all loads at once
    switch (wb) {
      case 1:
        hipLaunchKernelGGL((k_el2_step<T, SPLIT, 1, true>), g, dim3(64), 0, st, p->dmodels,
                           p->dshots, w, n, p->dbase, rel, 1, prun);
        break;
      case 2:
        hipLaunchKernelGGL((k_el2_step<T, SPLIT, 2, true>), g, dim3(128), 0, st, p->dmodels,
                           p->dshots, w, n, p->dbase, rel, 1, prun);
        break;
      default:
        hipLaunchKernelGGL((k_el2_step<T, SPLIT, 4, true>), g, dim3(256), 0, st, p->dmodels,
                           p->dshots, w, n, p->dbase, rel, 1, prun);
        break;
    }
    return;
  }
  switch (wb) {
    case 1:
      hipLaunchKernelGGL((k_el2_step<T, SPLIT, 1>), g, dim3(64), 0, st, p->dmodels,
                         p->dshots, w, n, p->dbase, rel, eh, prun);
      break;
    case 2:
      hipLaunchKernelGGL((k_el2_step<T, SPLIT, 2>), g, dim3(128), 0, st, p->dmodels,
                         p->dshots, w, n, p->dbase, rel, eh, prun);
      break;
    default:
      hipLaunchKernelGGL((k_el2_step<T, SPLIT, 4>), g, dim3(256), 0, st, p->dmodels,
                         p->dshots, w, n, p->dbase, rel, eh, prun);
      break;
  }
}

// One two-step ELASTIC2 step pair (steps base+rel, base+rel+1): the
// interior blocks, then the blocks that touch a C-PML slab or the outer ring.
template <typename T, bool SPLIT, bool INT>
void launch_el2x2_list(Plan* p, hipStream_t st, int rel, const int4* work, int n, int grid) {
  if (n <= 0) return;
  const dim3 g(grid);
  switch (p->el2_wb) {
    case 1:
      hipLaunchKernelGGL((k_el2_step2<T, SPLIT, 1, INT>), g, dim3(64), 0, st, p->dmodels, p->dshots,
                         work, n, p->dbase, rel, p->dit0, p->el2_eh);
      break;
    case 2:
      hipLaunchKernelGGL((k_el2_step2<T, SPLIT, 2, INT>), g, dim3(128), 0, st, p->dmodels, p->dshots,
                         work, n, p->dbase, rel, p->dit0, p->el2_eh);
      break;
    default:
      hipLaunchKernelGGL((k_el2_step2<T, SPLIT, 4, INT>), g, dim3(256), 0, st, p->dmodels, p->dshots,
                         work, n, p->dbase, rel, p->dit0, p->el2_eh);
      break;
  }
}
template <typename T, bool SPLIT>
void launch_el2x2(Plan* p, hipStream_t st, int rel) {
  launch_el2x2_list<T, SPLIT, true>(p, st, rel, p->dwork2, p->nwork2i, p->el2x2_grid_i);
  launch_el2x2_list<T, SPLIT, false>(p, st, rel, p->dwork2 + p->nwork2i, p->nwork2 - p->nwork2i,
                                     p->el2x2_grid);
}

template <typename T>
void launch_em2(Plan* p, hipStream_t st, int rel, const int* prun = nullptr) {
  const dim3 g(p->el2_grid);
  const int4* w = p->dwork;
  const int n = p->nwork, wb = p->el2_wb, eh = p->el2_eh;
  switch (wb) {
    case 1:
      hipLaunchKernelGGL((k_em2_step<T, 1>), g, dim3(64), 0, st, p->dmodels, p->dshots,
                         w, n, p->dbase, rel, eh, prun);
      break;
    case 2:
      hipLaunchKernelGGL((k_em2_step<T, 2>), g, dim3(128), 0, st, p->dmodels, p->dshots,
                         w, n, p->dbase, rel, eh, prun);
      break;
    default:
      hipLaunchKernelGGL((k_em2_step<T, 4>), g, dim3(256), 0, st, p->dmodels, p->dshots,
                         w, n, p->dbase, rel, eh, prun);
      break;
  }
}

// One two-step EM2 launch (steps base+rel, base+rel+1).
template <typename T>
void launch_em2x2(Plan* p, hipStream_t st, int rel) {
  const dim3 g(p->el2x2_grid);
  const int4* w = p->dwork2;
  const int n = p->nwork2;
  switch (p->el2_wb) {
    case 1:
      hipLaunchKernelGGL((k_em2_step2<T, 1>), g, dim3(64), 0, st, p->dmodels, p->dshots, w, n, p->dbase,
                         rel, p->dit0, p->el2_eh);
      break;
    case 2:
      hipLaunchKernelGGL((k_em2_step2<T, 2>), g, dim3(128), 0, st, p->dmodels, p->dshots, w, n, p->dbase,
                         rel, p->dit0, p->el2_eh);
      break;
    default:
      hipLaunchKernelGGL((k_em2_step2<T, 4>), g, dim3(256), 0, st, p->dmodels, p->dshots, w, n, p->dbase,
                         rel, p->dit0, p->el2_eh);
      break;
  }
}

// Whether every wavefront of the two-step kernel's block at (x0, z0) takes
// the interior body (the test of k_el2_step2 for each of its wavefronts).
bool el2x2_interior(const sdt_model& M, int x0, int z0, int wb, int eh) {
  const int ze = std::min(z0 + eh, M.nz);
  if (!(z0 - 4 >= M.lz + 1 && ze + 1 <= M.nz - M.lz - 2)) return false;
  for (int w = 0; w < wb; ++w) {
    const int xw = x0 + w * EW2;
    if (xw >= M.nx) break;
    if (!(xw - 2 >= M.lx + 1 && xw + 61 <= M.nx - M.lx - 2)) return false;
  }
  return true;
}

// Wavefronts of a 2-D plan with ew owned columns each and tiles of `rows` rows.
long long waves2d(const Plan* p, int ew, int rows) {
  long long n = 0;
  for (const sdt_shot& S : p->hshots) {
    const sdt_model& M = p->hmodels[S.model];
    n += (long long)((M.nx + ew - 1) / ew) * ((M.nz + rows - 1) / rows);
  }
  return n;
}

// Where the regions of one axis of n cells with slabs of l start owning cells,
// and whether a step reaches one cell each way in them (region_own).
std::vector<std::pair<int, bool>> region_cuts(const Plan* p, int n, int l, int tm) {
  const bool legacy = p->kind == SDT_ELASTIC2 && !p->split;
  std::vector<std::pair<int, bool>> c;
  for (int o = 0; o < n; o += region_own(c.back().second, tm)) {
    const int a = o - region_top(true, tm);  // (first cell of the region)
    c.push_back({o, !legacy || (a >= l && a + RM <= n - l)});
  }
  return c;
}
// Regions of a 2-D plan whose halo is tm steps wide.
long long regions2d(const Plan* p, int tm) {
  std::vector<long long> per(p->nmodels);
  for (int m = 0; m < p->nmodels; ++m) {
    const sdt_model& M = p->hmodels[m];
    per[m] = (long long)(region_cuts(p, M.nx, M.lx, tm).size() * region_cuts(p, M.nz, M.lz, tm).size());
  }
  long long n = 0;
  for (const sdt_shot& S : p->hshots) n += per[S.model];
  return n;
}

// The most steps per launch of a 2-D plan on regions (k_el2_multi, k_em2_multi),
// its default at every size (short runs aside: regions_pay).  A region recomputes its halo: with five steps per
// launch 47 % of its cells are owned.  Measured (us per step, walking kernels in
// the shape of default_shape, then regions): elastic FP64 127x103 6.3 -> 2.4, 296^2
// 8.3 -> 3.0, 12 shots of 1064x808 158 -> 150, 8 of 2088x808 208 -> 196; FP32 1064x808
// 18.7 -> 7.0, x 32 shots 227 -> 160, 48 shots of 39 M cells 312 -> 248; EM FP64
// 127x103 3.5 -> 1.5, 1064x808 11.9 -> 6.1, x 32 shots 207 -> 156; EM FP32 1064x808 7.6
// -> 4.4, x 32 shots 123 -> 87.
// Where the regions run all at once (one block of elastic FP64 per CU, else two),
// the most steps: a launch costs 5 to 7 us beside its steps (127x103 elastic FP64
// 5.1 / 2.8 / 2.3 us per step with 2 / 4 / 7).  Larger plans: the steps with the
// fewest regions times launches in a block of 50 steps (an even number of
// launches): FP32 32 shots of 1064x808 3 / 4 / 5 steps 211 / 188 / 159 (18 / 14 / 10
// launches).  That leaves out what the steps of a region cost beside its loads,
// a tenth of them per step in FP32 and a seventh in elastic FP64 (regions_pay);
// 9 uneven elastic FP64 shots take 21.1 us per step with 4 steps, 22.7 with the 5
// that this picks.
void default_regions(Plan* p) {
  auto cost = [&](int t) {
    const int n = (50 + t - 1) / t;
    return regions2d(p, t) * (n + (n & 1));
  };
  const int room = p->kind == SDT_ELASTIC2 && p->prec == SDT_FP64 ? 256 : 512;
  p->tm = 5;
  long long best = cost(5);
  for (int t = 3; t <= TM_MAX; ++t) {
    const long long c = cost(t);
    if (c < best) { best = c; p->tm = t; }
  }
  for (int t = TM_MAX; t >= 3; --t)
    if (regions2d(p, t) <= room) {
      p->tm = t;
      break;
    }
  p->multi = true;
}

// Default launch shape of a 2-D plan's walking kernels, which take the runs that
// are too short for regions (regions_pay) and those of a plan taken off them:
// steps per launch, wavefronts per block, rows per tile and tile order, from how
// many wavefronts the plan has and whether its ping-pong fields fit the 256 MB
// last-level cache.  Fitted to the
// times of every shape on 30 plans (6 k to 27 M cells per step, 1 to 36 shots)
// per kind and precision: within 2 to 4 % of the fastest shape in the mean.
// Against tiles of 32 .. 2 rows for 1024 blocks of four wavefronts, one step
// per launch below 4 M cells and order 0 (us per step, then and now): elastic
// FP64 127x103 12.1 -> 7.1, 296^2 15.3 -> 9.0, 1064x808 40.5 -> 28.3, 640x440 x
// 12 shots 119 -> 74; EM FP64 296^2 8.9 -> 5.0, 1064x808 22.8 -> 12.3; EM FP32
// 1064x808 16.4 -> 8.4.
//  - EM2 always takes two steps per launch (also the smallest grid, 80x70:
//    4.1 against 5.9 us per step).  The elastic two-step walk reads six halo
//    rows per tile, so below 2000 (FP64) and 6000 (FP32) wavefronts of one row
//    the one-step kernel's one-row tiles win (296^2 FP64 9.0 against 12.4).
//  - Rows: the tallest of 8, 4, 2 (EM also 1) that still give 2000 (FP64) or
//    4000 (elastic FP32; EM 2800) wavefronts; 16 and 32 only with many of them
//    (1064x808 x 6 shots EM FP64 46.6 with 8, 51.4 with 16).  EM plans of up to
//    4096 regions, whose walking runs are of one step or blocks of two, halve 8
//    rows (FP64 also 4): the one-step kernel's walk is the longer one (5 shots of
//    670x330 FP64 24.3 us with 8 rows, 18.3 with 4; of 438x624 FP32 20.0, 18.1).
//  - Column strips per XCD (order 1) while the fields fit the cache, tiles
//    dealt in turn beyond (1064x808 x 12 shots elastic FP64 157 against 178).
//  - Wide blocks waste wavefronts at the edge of a narrow grid and take its
//    interior tiles for edge tiles: fewer wavefronts per block below 400
//    columns, and (but for EM FP64) where the fields do not fit the cache.
void default_shape(Plan* p) {
  const bool em = p->kind == SDT_EM2, f64 = p->prec == SDT_FP64;
  const int ew = em ? EW2E : EW2;
  long long cells = 0;
  int maxnx = 0;
  for (const sdt_shot& S : p->hshots) {
    const sdt_model& M = p->hmodels[S.model];
    cells += (long long)M.nx * M.nz;
    maxnx = std::max(maxnx, M.nx);
  }
  const bool big = cells * kind_fields(p->kind) * 2 * (f64 ? 8 : 4) >= 250000000LL;
  p->spl = 2;
  p->el2_order = big ? 0 : 1;
  if (!em && waves2d(p, EW, 1) <= (f64 ? 2000 : 6000)) {
    p->spl = 1;
    p->el2_wb = 2;
    p->el2_eh = 1;
  } else if (waves2d(p, ew, 32) >= 16000) {
    p->el2_wb = 4;
    p->el2_eh = 32;
  } else {
    const bool narrow = maxnx < 400;
    if (big)
      p->el2_wb = em ? (f64 ? 4 : 2) : (f64 ? 1 : 2);
    else
      p->el2_wb = !narrow ? 4 : em ? 1 : f64 ? 2 : 4;
    p->el2_eh = em ? 1 : 2;
    for (int rows : {2, 4, 8})
      if (waves2d(p, ew, rows) >= (f64 ? 2000 : em ? 2800 : 4000)) p->el2_eh = rows;
    if (waves2d(p, ew, 16) >= (em ? 12000 : 8000)) p->el2_eh = 16;
  }
  default_regions(p);
  if (em && p->el2_eh <= 8 && p->el2_eh >= (f64 ? 4 : 8) && regions2d(p, p->tm) <= 4096) p->el2_eh /= 2;
}

// Work list of the region kernels: the regions of a model row by row, so that
// the run an XCD takes (item8) is one part of the model and neighbours in x,
// which write parts of the same cache lines, run together (column by column:
// EM FP32 32 shots of 1064x808 118 us per step against 107, elastic FP32 16 of
// 1064x552 84 against 77, their recomputation 142 against 114).
std::vector<int4> multi_work(const Plan* p, int tm) {
  const bool legacy = p->kind == SDT_ELASTIC2 && !p->split;
  std::vector<int4> w;
  w.reserve(regions2d(p, tm));
  for (int s = 0; s < p->nshots; ++s) {
    const int m = p->hshots[s].model;
    const sdt_model& M = p->hmodels[m];
    const auto xs = region_cuts(p, M.nx, M.lx, tm), zs = region_cuts(p, M.nz, M.lz, tm);
    for (const auto& z : zs)
      for (const auto& x : xs)
        w.push_back(make_int4(s, x.first, z.first,
                              m | (legacy && x.second ? REGION_X1 : 0) | (legacy && z.second ? REGION_Z1 : 0)));
  }
  return w;
}

// Launches of one run or graph block of n steps on regions: at most tm steps
// each, an even number of them if `even` (a graph block must leave the state in
// the buffer it started from).
int region_launches(int n, int tm, bool even) {
  const int L = (n + tm - 1) / tm;
  return even ? L + (L & 1) : L;
}

// Items per launch of the kernels that take one item per block: a launch holds
// fewer than 2^32 threads, which 4.2 M blocks of 1024 reach (2 G cells per step
// on regions), so longer lists go in several launches.  At this length (0.13 G
// cells, 4 ms per elastic FP32 launch of five steps) a further launch costs nothing
// against the work.
constexpr int LAUNCH_ITEMS = 1 << 18;
template <typename F>
void in_slices(int n, F&& launch) {
  for (int o = 0; o < n; o += LAUNCH_ITEMS) launch(o, std::min(LAUNCH_ITEMS, n - o));
}

// k steps from step base + r on regions, reading state buffer par.
template <typename T, bool TRAIL = false>
void launch_region(Plan* p, hipStream_t st, int r, int k, int par) {
  const int tm = TRAIL ? p->tr_tm : p->tm, items = TRAIL ? p->ntrwork : p->nmulti;
  const dim3 b(RM * RM);
  in_slices(items, [&](int o, int nw) {
    const int4* w = (TRAIL ? p->dtrwork : p->dwmulti) + o;
    const dim3 g((nw + 7) / 8 * 8);
    if (p->kind == SDT_EM2 && !TRAIL && sizeof(T) == 4 && items > 512)  // (see EmRegionLds)
      hipLaunchKernelGGL((k_em2_multi<float, false, 2>), g, dim3(RM * RM / 2), 0, st, p->dmodels, p->dshots, w, nw,
                         p->dbase, r, k, tm, par, p->dadj, p->dtsel_trail);
    else if (p->kind == SDT_EM2)
      hipLaunchKernelGGL((k_em2_multi<T, TRAIL, 1>), g, b, 0, st, p->dmodels, p->dshots, w, nw, p->dbase, r, k, tm,
                         par, p->dadj, p->dtsel_trail);
    else if (p->split)
      hipLaunchKernelGGL((k_el2_multi<T, true, TRAIL>), g, b, 0, st, p->dmodels, p->dshots, w, nw, p->dbase, r, k,
                         tm, par, p->dadj, p->dtsel_trail);
    else
      hipLaunchKernelGGL((k_el2_multi<T, false, TRAIL>), g, b, 0, st, p->dmodels, p->dshots, w, nw, p->dbase, r, k,
                         tm, par, p->dadj, p->dtsel_trail);
  });
}

// Steps of one run or graph block on regions, in launches of nearly equal
// length.  Returns the number of launches.
template <typename T, bool TRAIL = false>
int launch_multi(Plan* p, hipStream_t st, int n, bool even) {
  const int L = region_launches(n, TRAIL ? p->tr_tm : p->tm, even);
  for (int l = 0; l < L; ++l) {
    const int r = (int)((long long)n * l / L);
    launch_region<T, TRAIL>(p, st, r, (int)((long long)n * (l + 1) / L) - r, l & 1);
  }
  return L;
}

// Row cuts of one model's tiles: rows of at most eh, and with zt < zb also
// cuts at zt and zb, so the tiles between (those the kernel can run with
// its interior body) start exactly where that first becomes possible.
std::vector<int> row_cuts(int nz, int eh, int zt, int zb) {
  std::vector<int> c = {0};
  auto run = [&](int a, int b) {
    for (int z = a + eh; z < b; z += eh) c.push_back(z);
    if (b > c.back()) c.push_back(b);
  };
  if (zt > 0 && zt < zb && zb < nz) {
    run(0, zt);
    run(zt, zb);
    run(zb, nz);
  } else {
    run(0, nz);
  }
  return c;
}

// which: 0 every block, 1 the interior blocks of the two-step kernel, 2 the
// others.  ew: owned columns per wavefront; two-step lists (ew = EW2, EW2E)
// cut their rows at the interior limits of their kernel and carry each
// tile's height in .w (0: the plan's rows); one-step lists (ew = EW) carry
// the shot's model index in .w.  Order: 0 deals a model's
// tiles to the XCDs in turn (tile k of the list on XCD k % 8), every XCD
// covering the whole model; 1 lists them column by column and gives each
// XCD a contiguous run, so a tile and the one below it, which share halo
// rows, run on one XCD one after the other, and each XCD keeps to one part
// of the model from step to step.  Either way all shots of a tile run on
// one XCD, one after another.
std::vector<int4> el2_work(const Plan* p, int wb, int eh, int order, int ew = EW, int which = 0) {
  std::vector<int4> work;
  const int bw = ew * wb;
  for (int m = 0; m < p->nmodels; ++m) {
    const sdt_model& M = p->hmodels[m];
    // first and last-plus-one interior rows of k_el2_step2 / k_em2_step2
    const int zt = ew == EW2 ? M.lz + 5 : ew == EW2E ? M.lz + 3 : 0;
    const int zb = ew == EW2 ? M.nz - M.lz - 3 : ew == EW2E ? M.nz - M.lz - 4 : 0;
    const std::vector<int> cuts = row_cuts(M.nz, eh, zt, zb);
    const int tx = (M.nx + bw - 1) / bw, tz = (int)cuts.size() - 1, ntile = tx * tz;
    std::vector<int> ms;
    for (int s = 0; s < p->nshots; ++s)
      if (p->hshots[s].model == m) ms.push_back(s);
    if (ms.empty()) continue;
    std::vector<int> tl;
    auto take = [&](int t) {
      const int z0 = cuts[t / tx], h = cuts[t / tx + 1] - z0;
      if (which == 0 || el2x2_interior(M, (t % tx) * bw, z0, wb, h) == (which == 1))
        tl.push_back(t);
    };
    if (order) {
      for (int x = 0; x < tx; ++x)
        for (int z = 0; z < tz; ++z) take(z * tx + x);
    } else {
      for (int t = 0; t < ntile; ++t) take(t);
    }
    const int nt = (int)tl.size();
    // tile of slot tg of XCD tt (-1: none)
    const int chunk = (nt + 7) / 8;
    auto tile_at = [&](int tg, int tt) {
      const int k = order ? tt * chunk + tg : tg * 8 + tt;
      return k < nt ? tl[k] : -1;
    };
    for (int tg = 0; tg < chunk; ++tg)
      for (int s : ms)
        for (int tt = 0; tt < 8; ++tt) {
          const int t = tile_at(tg, tt);
          if (t < 0) {
            work.push_back(make_int4(-1, 0, 0, 0));
            continue;
          }
          const int z0 = cuts[t / tx], h = cuts[t / tx + 1] - z0;
          work.push_back(make_int4(s, (t % tx) * bw, z0, ew == EW ? m : h));
        }
  }
  return work;
}

// Where the y chunks of at most `rows` rows of one model start, and ny: chunks
// end at the y-slab edges, so a chunk lies inside a slab or outside both.
std::vector<int> cuts25(const sdt_model& M, int rows) {
  std::vector<int> cuts = {0};
  const int ya = std::min(M.ly, M.ny), yb = std::max(ya, M.ny - M.ly);
  auto cut = [&](int a, int b) {  // rows a .. b-1 in chunks of nearly equal height
    const int nc = b > a ? (b - a + rows - 1) / rows : 0;
    for (int c = 1; c <= nc; ++c) cuts.push_back(a + (int)((long long)(b - a) * c / nc));
  };
  cut(0, ya);
  cut(ya, yb);
  cut(yb, M.ny);
  return cuts;
}

// Rows per y chunk of a 2.5-D plan.  A wavefront takes its rows in turn,
// waiting for their loads, so tall chunks leave a small grid bound by the
// latency of that walk with most of the device idle; short ones reload the
// row above and below, and, in the elastic passes, the column's 39
// coefficients, per chunk.  Measured per step (us):
//   EM, 8 / 4 / 2 rows: 332x72x182 FP32 90 / 84 / 86, FP64 207 / 202 / 203,
//   133x57x79 FP64 35 / 31 / 31, 544x96x416 FP32 439 / 428 / -;
//   elastic FP32, 16 / 8 / 4 / 2 rows: 832x96x432 1161 / 1160 / - / -, 332x72x182
//   160 / 148 / 135 / 136, 112x56x82 63 / 42 / 31 / 27; FP64: 832x96x432 2180 /
//   2179 / - / -, 332x72x182 357 / 342 / 347 / 374, 171x57x95 70 / 70 / 68 / 68.
int rows25(const Plan* p) {
  auto waves = [&](int rows) {
    long long n = 0;
    for (const sdt_shot& S : p->hshots) {
      const sdt_model& M = p->hmodels[S.model];
      n += (long long)(cuts25(M, rows).size() - 1) * ((M.nx + EW25 - 1) / EW25) * M.nz;
    }
    return n;
  };
  if (p->kind == SDT_EM25) return 4;
  if (waves(16) >= 20000) return 16;
  if (p->prec == SDT_FP64) return waves(8) >= 5000 ? 8 : 4;
  return waves(4) >= 2500 ? 4 : 2;
}

// Work list of the 2.5-D kernels: one item (shot, x0, k, j0 | j1 << 16) per
// wavefront of EW25 columns x0.. of plane k and one y chunk, plane by plane,
// chunk by chunk, x fastest.  The kernels give each XCD a contiguous run of
// them, so the wavefronts an XCD runs at a time cover whole rows of a few
// planes (long contiguous runs of addresses in each array).
// `least`: the fewest rows per chunk (a shorter list for the fixed scratch).
std::vector<int4> el25_work(Plan* p, int least) {
  std::vector<int4> all;
  p->item25.assign(1, 0);
  const int rows = std::max(rows25(p), least);
  for (int s = 0; s < p->nshots; ++s) {
    const sdt_model& M = p->hmodels[p->hshots[s].model];
    const std::vector<int> cuts = cuts25(M, rows);
    for (int k = 0; k < M.nz; ++k)
      for (size_t c = 0; c + 1 < cuts.size(); ++c)
        for (int x0 = 0; x0 < M.nx; x0 += EW25)
          all.push_back(make_int4(s, x0, k, ychunk_pack(cuts[c], cuts[c + 1])));
    p->item25.push_back((int)all.size());
  }
  return all;
}

// Bytes of a shot's state.
double shot_bytes(const Plan* p, int s) {
  const sdt_model& M = p->hmodels[p->hshots[s].model];
  const double n = kind_fields(p->kind) * (double)M.nx * M.ny * M.nz +
                   psi_elems(p->kind | (p->split ? SDT_SPLIT_CPML : 0), M.nx, M.ny, M.nz, M.lx, M.ly, M.lz);
  return n * (p->prec == SDT_FP64 ? 8 : 4);
}

// The schedule of the EM 2.5-D steps.  Each pass streams the whole state, so a
// plan larger than the 256 MB last-level cache reads everything from HBM twice
// per step.  Blocks of planes of at most 160 MB go through both passes of up to
// 16 time steps before the next block starts, and what the first pass of a
// block left in the cache the following ones find there.  Nothing is computed
// twice: the H pass reads E of the plane above, so a block's upper bound moves
// down by one plane per step, and the next block takes those planes.  Shots
// that fit the cache go in groups of at most 200 MB.  Same kernels and results.
// Measured per step (us, whole plan per pass, then blocks): 544x96x416 FP32 428
// -> 350, FP64 831 -> 744; 832x96x432 FP32 682 -> 582; 432x96x282 FP64 468 ->
// 409; 6 shots of 232x96x182 FP32 508 -> 476; 24 shots of 152x62x112 FP64 1156 ->
// 1064 (groups of 150 MB: 1257; a launch over four of them leaves the device
// half empty at its end).  100 and 200 MB for blocks of planes: 378 and 357 on
// the first grid, 600 and 613 on the third.  The elastic passes are not run so:
// before their row groups they lost by it (832x96x432 FP32 1281 whole, 1398 ..
// 1750 in blocks of 40 .. 140 planes); as they are (1160 whole) it has not been
// measured.
constexpr int STEPS25 = 16;
constexpr double PLANES25_BYTES = 160e6, SHOTS25_BYTES = 200e6;

void set_blocks25(Plan* p) {
  p->blocks25.clear();
  double total = 0;
  for (int s = 0; s < p->nshots; ++s) total += shot_bytes(p, s);
  if (p->kind != SDT_EM25 || total < 250e6) {
    p->blocks25.push_back({0, p->nshots, INT_MAX});
    return;
  }
  for (int s = 0; s < p->nshots;) {
    const int nz = p->hmodels[p->hshots[s].model].nz;
    // a block keeps more planes than its bounds move in STEPS25 steps
    const int nb = shot_bytes(p, s) < 250e6 ? 1
                   : (int)std::min((double)(nz / (2 * STEPS25)), std::ceil(shot_bytes(p, s) / PLANES25_BYTES));
    if (nb > 1) {
      for (int b = 0; b < nb; ++b)
        p->blocks25.push_back({s, s + 1, b == nb - 1 ? INT_MAX : (int)((long long)nz * (b + 1) / nb)});
      ++s;
      continue;
    }
    int e = s;
    for (double sum = 0; e < p->nshots && (e == s || sum + shot_bytes(p, e) <= SHOTS25_BYTES); ++e)
      sum += shot_bytes(p, e);
    p->blocks25.push_back({s, e, INT_MAX});
    s = e;
  }
}

// One pass (0 stress / H, 1 velocity / E) of step base + rel over n items of
// the 2.5-D work list from item `off`.
template <typename T>
void launch_pass25(Plan* p, hipStream_t st, int rel, int pass, int off, int n) {
  const dim3 grd((n + 7) / 8 * 8), blk(NT25);
  const int4* w = p->dwork + off;
  if (p->kind == SDT_ELASTIC25) {
    if (pass == 0)
      hipLaunchKernelGGL(k_el25_stress<T>, grd, blk, 0, st, p->dmodels, p->dshots, w, n, p->dbase, rel);
    else
      hipLaunchKernelGGL(k_el25_vel<T>, grd, blk, 0, st, p->dmodels, p->dshots, w, n, p->dbase, rel);
  } else if (pass == 0) {
    hipLaunchKernelGGL(k_em25_h<T>, grd, blk, 0, st, p->dmodels, p->dshots, w, n);
  } else {
    hipLaunchKernelGGL(k_em25_e<T>, grd, blk, 0, st, p->dmodels, p->dshots, w, n, p->dbase, rel);
  }
}

// Receiver samples of step base + rel of shots s0..s1-1 on planes k0..k1-1.
template <typename T>
void launch_gather25(Plan* p, hipStream_t st, int rel, int s0, int s1, int k0, int k1) {
  int nrec = 0;
  for (int s = s0; s < s1; ++s)
    if (p->reck[s].first < k1 && p->reck[s].second >= k0) nrec = std::max(nrec, p->hshots[s].nrec);
  if (nrec > 0)
    hipLaunchKernelGGL(k_gather<T>, dim3((nrec + 63) / 64, s1 - s0), dim3(64), 0, st, p->dmodels, p->dshots,
                       s0, p->ncomp, p->dbase, rel, k0, k1);
}

template <typename T>
void launch_steps25(Plan* p, hipStream_t st, int n) {
  const bool one = p->blocks25.size() == 1;
  const int runs = one ? 1 : (n + STEPS25 - 1) / STEPS25;  // of nearly equal length
  for (int q = 0; q < runs; ++q) {
    const int r0 = (int)((long long)n * q / runs), r1 = (int)((long long)n * (q + 1) / runs);
    for (size_t b = 0; b < p->blocks25.size(); ++b) {
      const Block25& B = p->blocks25[b];
      const int i0 = p->item25[B.s0], ni = p->item25[B.s1] - i0;
      const bool first = b == 0 || p->blocks25[b - 1].s1 <= B.s0;  // of its shots
      for (int r = r0; r < r1; ++r) {
        int off = i0, m = ni, k0 = 0, k1 = INT_MAX;
        if (!first || B.top != INT_MAX) {  // planes k0 .. k1-1 of one shot
          const int nz = p->hmodels[p->hshots[B.s0].model].nz, per = ni / nz;
          k0 = first ? 0 : p->blocks25[b - 1].top - (r - r0);
          k1 = B.top == INT_MAX ? nz : B.top - (r - r0);
          off += k0 * per;
          m = (k1 - k0) * per;
        }
        launch_pass25<T>(p, st, r, 0, off, m);
        launch_pass25<T>(p, st, r, 1, off, m);
        launch_gather25<T>(p, st, r, B.s0, B.s1, k0, k1);
      }
    }
  }
}

// Launch kernel `which` (0: first field update, 1: second field update,
// 2: receiver gather) of one step.
template <typename T>
void launch_one(Plan* p, hipStream_t st, int rel, int which) {
  if (kind_3d(p->kind)) {
    if (which == 2)
      launch_gather25<T>(p, st, rel, 0, p->nshots, 0, INT_MAX);
    else
      launch_pass25<T>(p, st, rel, which, 0, p->nwork);
    return;
  }
  if (which == 2) return;  // the 2-D step kernels write their receiver samples themselves
  switch (p->kind * 2 + which) {
    case SDT_ELASTIC2 * 2:
      if (p->split)
        launch_el2<T, true>(p, st, rel);
      else
        launch_el2<T, false>(p, st, rel);
      break;
    case SDT_ELASTIC2 * 2 + 1:
      break;  // the fused step kernel does both phases
    case SDT_EM2 * 2:
      launch_em2<T>(p, st, rel);
      break;
    case SDT_EM2 * 2 + 1:
      break;  // the fused step kernel does both phases
  }
}

template <typename T>
void launch_copy_back(Plan* p, hipStream_t st, int to_b = 0) {
  // four vectors per thread of the largest array
  const int nf = kind_fields(p->kind);
  const int blocks = (int)std::min<long long>(512, p->maxel * (long long)sizeof(T) / (16 * 256 * 4) + 1);
  hipLaunchKernelGGL(k_copy_back<T>, dim3(blocks, p->nshots, nf + 1), dim3(256), 0, st, p->dshots, nf, p->dnel,
                     p->dnpsi, to_b);
}

template <typename T>
void launch_finalize(Plan* p, hipStream_t st) {
  if (p->kind == SDT_EM2)
    hipLaunchKernelGGL(k_em2_edges<T>, dim3(16, p->nshots), dim3(256), 0, st, p->dmodels, p->dshots);
  if (p->kind == SDT_EM25)
    hipLaunchKernelGGL(k_em25_edges<T>, dim3(p->nwork), dim3(64), 0, st, p->dmodels, p->dshots,
                       p->dwork);
}

template <typename T>
void launch_step(Plan* p, hipStream_t st, int rel) {
  for (int w = 0; w < 3; ++w) launch_one<T>(p, st, rel, w);
}

void launch_steps(Plan* p, hipStream_t st, int n) {
  if (kind_3d(p->kind)) {
    if (p->prec == SDT_FP64)
      launch_steps25<double>(p, st, n);
    else
      launch_steps25<float>(p, st, n);
    return;
  }
  for (int r = 0; r < n; ++r) {
    if (p->prec == SDT_FP64)
      launch_step<double>(p, st, r);
    else
      launch_step<float>(p, st, r);
  }
}

// Launch `which` of a run of two-step launches from the base step: pair
// r/2 (steps r, r+1) for even r, or the single step r that ends an odd
// run (one-step kernel, reading the buffer the pairs left the state in).
template <typename T>
void launch_two(Plan* p, hipStream_t st, int r, bool single) {
  const bool em = p->kind == SDT_EM2;
  if (!single) {
    if (em)
      launch_em2x2<T>(p, st, r);
    else if (p->split)
      launch_el2x2<T, true>(p, st, r);
    else
      launch_el2x2<T, false>(p, st, r);
    return;
  }
  if (em)
    launch_em2<T>(p, st, r, p->dit0);
  else if (p->split)
    launch_el2<T, true>(p, st, r, p->dit0);
  else
    launch_el2<T, false>(p, st, r, p->dit0);
}

void launch_pairs(Plan* p, hipStream_t st, int n) {
  for (int r = 0; r < n; r += 2) {
    const bool single = r + 1 == n;
    if (p->prec == SDT_FP64)
      launch_two<double>(p, st, r, single);
    else
      launch_two<float>(p, st, r, single);
  }
}

// Whether a run of n steps in graph blocks of graph_block uses two-step
// launches (the blocks must hold whole pairs).
bool use_two(const Plan* p, int n, int graph_block) {
  return p->spl == 2 && n >= 2 && (graph_block <= 1 || n < graph_block || graph_block % 2 == 0);
}

// Whether runs of n steps are faster on regions than with the walking kernels.
// A region loads its whole halo however few steps it takes, and an odd number
// of launches ends in buffer B, from where the state is copied back (a run of
// one step on the walkers: every second time).  Small plans wait for launches
// most of the time and gain from two steps on (us per step, walkers then
// regions: elastic FP64 127x103 runs of 1 / 2 / 3 steps 10.6 / 8.1 / 8.4, 13.2 / 7.1 /
// 5.2; 1064x808 49 / 42 / 36, 62 / 34 / 25; EM FP32 21 / 15.4 / 10.4, 29 / 15.3 /
// 10.7; graph blocks of 2 / 3 / 4 steps 10.8 / 14.6 / 9.3, 16.2 / 11.4 / 9.0).  Plans
// of many regions (6 and 36 shots of 1064x808) compare what both ways cost in
// units of one pair of steps on the walkers, fitted to runs and blocks of 1 to 20
// steps: a launch of k steps on regions a + b k, the copy c, a single step s.  36
// elastic FP64 shots: runs of 1 / 2 / 4 / 5 / 6 / 8 / 12 steps 1212 / 809 / 538 / 726 / 628 /
// 537 / 538, on regions 2140 / 1151 / 661 / 564 / 644 / 526 / 571 (with copies of 541 us,
// now 496).
bool regions_pay(const Plan* p, int n, int graph_block) {
  const bool blocks = graph_block > 1 && n >= graph_block;
  const int k = blocks ? graph_block : n;
  if (p->nmulti <= 4096) return k >= (blocks ? 3 : 2);
  // a up to 32768 regions, a beyond, b, c, s: elastic FP64, FP32, EM FP64, FP32
  static const double cost[4][5] = {{1.15, 1.32, 0.155, 0.42, 0.85}, {0.90, 1.22, 0.09, 0.38, 0.83},
                                    {1.28, 1.46, 0.065, 0.55, 0.96}, {1.20, 1.38, 0.11, 0.48, 0.89}};
  const double* t = cost[(p->kind == SDT_EM2 ? 2 : 0) + (p->prec == SDT_FP32 ? 1 : 0)];
  const double a = t[p->nmulti > 32768], b = t[2], c = blocks ? 0 : t[3], s = t[4];
  const int L = region_launches(k, p->tm, blocks);
  const bool two = use_two(p, n, graph_block);
  const int W = two ? k / 2 + (k & 1) : k;
  const double walk = two ? k / 2 + (k & 1) * s + (W & 1) * c : k * s + (W & 1) * c / 2;
  return L * a + k * b + (L & 1) * c < walk;
}

// How a run of n steps goes: 0 one step per launch, 1 two, 2 several on regions
// (unless a launch shape was asked for).
int run_mode(const Plan* p, int n, int graph_block) {
  if (p->multi && p->regions && regions_pay(p, n, graph_block)) return 2;
  return use_two(p, n, graph_block) ? 1 : 0;
}

// Enqueue n steps in mode `mode`; whether the state is then in buffer B, or -1
// where the step index says so (mode 0).
int launch_run(Plan* p, hipStream_t st, int n, int mode, bool even) {
  if (mode == 2) return (p->prec == SDT_FP64 ? launch_multi<double>(p, st, n, even) : launch_multi<float>(p, st, n, even)) & 1;
  if (mode == 1) {
    launch_pairs(p, st, n);
    return (n / 2 + (n & 1)) & 1;
  }
  launch_steps(p, st, n);
  return -1;
}

int validate(int kind, bool split, int prec, const sdt_model* models, int nmodels,
             const sdt_shot* shots, int nshots, int nt) {
  const int kpsi = kind | (split ? SDT_SPLIT_CPML : 0);
  if (kind < 0 || kind > 3) return fail(SDT_EINVAL, "unknown kind");
  if (prec != SDT_FP64 && prec != SDT_FP32) return fail(SDT_EINVAL, "unknown precision");
  if (!models || nmodels <= 0 || !shots || nshots <= 0) return fail(SDT_EINVAL, "no models or shots");
  if (nt <= 0) return fail(SDT_EINVAL, "nt must be positive");
  const bool d3 = kind_3d(kind);
  for (int m = 0; m < nmodels; ++m) {
    const sdt_model& M = models[m];
    const std::string tag = "model " + std::to_string(m) + ": ";
    if (M.nx < 3 || M.nz < 3 || (d3 && M.ny < 3) || (!d3 && M.ny != 1))
      return fail(SDT_EINVAL, tag + "grid too small (nx, nz >= 3; ny >= 3 in 2.5-D, 1 in 2-D)");
    if ((long long)M.nx * M.ny * M.nz > (1LL << 40)) return fail(SDT_EINVAL, tag + "grid too large");
    if (M.lx < 0 || M.lz < 0 || M.lx > (M.nx + 1) / 2 || M.lz > (M.nz + 1) / 2 ||
        (d3 && (M.ly < 0 || M.ly > (M.ny + 1) / 2)))
      return fail(SDT_EINVAL, tag + "slab width out of range");
    if (!(M.dx > 0) || !(M.dz > 0) || (d3 && !(M.dy > 0)) || !(M.dt > 0))
      return fail(SDT_EINVAL, tag + "dx, dy, dz, dt must be positive");
    for (int q = 0; q < kind_ncoef(kind); ++q) {
      const bool optional = kind == SDT_ELASTIC2 && (q == 2 || q == 4 || q == 5 || q == 6 || q >= 10);
      if (!M.coef[q] && !optional)
        return fail(SDT_EINVAL, tag + "coefficient slot " + std::to_string(q) + " is null");
    }
    if (kind == SDT_ELASTIC2) {
      const bool m1 = M.coef[2] || M.coef[4] || M.coef[5] || M.coef[6];
      const bool m2 = M.coef[2] && M.coef[4] && M.coef[5] && M.coef[6];
      if (m1 != m2 || (!M.coef[10]) != (!M.coef[11]))
        return fail(SDT_EINVAL, tag + "ELASTIC2 slots 2,4,5,6 (and 10,11) must be all set or all null");
    }
    for (int a = 0; a < 3; ++a) {
      if (a == 1 && !d3) continue;
      for (int q = 0; q < 6; ++q)
        if (!M.prof[a][q]) return fail(SDT_EINVAL, tag + "C-PML profile missing");
    }
    if (kind == SDT_ELASTIC2 && !split && !M.aux)
      return fail(SDT_EINVAL, tag + "aux (b_x_half by row) missing");
    if (kind == SDT_ELASTIC2 || kind == SDT_EM2) {
      // the step kernel addresses each array with 32-bit byte offsets
      const long long es = prec == SDT_FP64 ? 8 : 4;
      const long long np = psi_elems(kpsi, M.nx, M.ny, M.nz, M.lx, M.ly, M.lz);
      if ((long long)M.nx * M.nz * es >= (1LL << 32) || np * es >= (1LL << 32))
        return fail(SDT_EINVAL, tag + "grid too large (every array must stay under 4 GiB)");
    }
    if (d3) {
      // the kernels address one z plane of a field or memory variable, and a
      // coefficient array, with 32-bit byte offsets (slabs that cover an odd
      // axis hold one cell more than it), and pack a y chunk in 16-bit halves
      const long long es = prec == SDT_FP64 ? 8 : 4;
      const long long wide = std::max(M.nx, 2 * M.lx), tall = std::max(M.ny, 2 * M.ly);
      if (std::max(wide * M.ny, M.nx * tall) * es >= (1LL << 32) || (long long)M.nx * M.nz * es >= (1LL << 32))
        return fail(SDT_EINVAL, tag + "grid too large (an x-y plane must stay under 4 GiB)");
      if (M.ny > 65535) return fail(SDT_EINVAL, tag + "ny above 65535");
    }
  }
  for (int s = 0; s < nshots; ++s) {
    const sdt_shot& S = shots[s];
    const std::string tag = "shot " + std::to_string(s) + ": ";
    if (S.model < 0 || S.model >= nmodels) return fail(SDT_EINVAL, tag + "bad model index");
    const sdt_model& M = models[S.model];
    for (int f = 0; f < kind_fields(kind); ++f)
      if (!S.field[f]) return fail(SDT_EINVAL, tag + "field pointer null");
    if (!S.psi && psi_elems(kpsi, M.nx, M.ny, M.nz, M.lx, M.ly, M.lz) > 0)
      return fail(SDT_EINVAL, tag + "psi workspace null");
    if (pingpong(kind)) {
      for (int f = 0; f < kind_fields(kind); ++f)
        if (!S.field_b[f]) return fail(SDT_EINVAL, tag + "field_b pointer null (ELASTIC2 and EM2 ping-pong)");
      if (!S.psi_b && psi_elems(kpsi, M.nx, M.ny, M.nz, M.lx, M.ly, M.lz) > 0)
        return fail(SDT_EINVAL, tag + "psi_b workspace null");
    }
    if (S.isrc < 0 || S.isrc >= M.nx || S.ksrc < 0 || S.ksrc >= M.nz ||
        (d3 && (S.jsrc < 0 || S.jsrc >= M.ny)))
      return fail(SDT_EINVAL, tag + "source outside the padded grid");
    if (S.nrec < 0 || (S.nrec > 0 && (!S.rec || !S.trace)))
      return fail(SDT_EINVAL, tag + "receivers need rec and trace buffers");
  }
  return SDT_OK;
}

// State after the last step of a run: EM H edges zeroed; ping-pong kinds
// copied back into buffer A when the last step wrote buffer B (one-step runs
// ending before an odd step; final_b: whether a run of two-step launches
// ended in B, else -1).  A always holds the state afterwards; b_holds
// records whether B does too (it did when the last step wrote B).
void end_of_run(Plan* p, hipStream_t st, int next_step, int final_b = -1) {
  const bool b = pingpong(p->kind) && (final_b < 0 ? (next_step & 1) != 0 : final_b != 0);
  p->b_holds = b;
  if (p->prec == SDT_FP64) {
    if (b) launch_copy_back<double>(p, st);
    launch_finalize<double>(p, st);
  } else {
    if (b) launch_copy_back<float>(p, st);
    launch_finalize<float>(p, st);
  }
}

// Before a run: the one-step kernels read the state of step it from buffer
// it & 1, so a one-step run that starts at an odd step needs the state in B.
// Copy A into B unless the previous run left it there (a run of two-step
// launches always starts from A and needs nothing).
void start_of_run(Plan* p, hipStream_t st, int it0, bool two) {
  if (!pingpong(p->kind) || two || !(it0 & 1) || p->b_holds) return;
  if (p->prec == SDT_FP64)
    launch_copy_back<double>(p, st, 1);
  else
    launch_copy_back<float>(p, st, 1);
  p->b_holds = true;
}

long long state_elems(int kind, long long nx, long long ny, long long nz, long long lx,
                      long long ly, long long lz) {
  const long long np = psi_elems(kind, nx, ny, nz, lx, ly, lz);
  return np < 0 ? -1 : kind_fields(kind & ~SDT_SPLIT_CPML) * nx * ny * nz + np;
}

// Adjoint steps t = tbase + k for k = khi-1 down to klo (tbase = the trail's
// first step, held on the device so a captured segment replays anywhere).
template <typename T, bool SPLIT>
void launch_adjoint_steps(Plan* p, hipStream_t st, int khi, int klo) {
  const dim3 blk(TX, TZ);
  const dim3 grd((p->maxnx + TX - 1) / TX, (p->maxnz + TZ - 1) / TZ, p->nshots);
  const int* tb = p->dtbase;
  for (int k = khi - 1; k >= klo; --k) {
    if (!(p->adj_flags & SDT_ADJ_REFERENCE)) {
      in_slices(p->nadjwork, [&](int o, int n) {
        hipLaunchKernelGGL((k_el2_adj<T, SPLIT>), dim3((n + 7) / 8 * 8), dim3(64 * AR<T, false>), 0, st, p->dmodels,
                           p->dshots, p->dadj, p->dadjwork + o, n, tb, k, p->gmask, p->dtsel_adj);
      });
      continue;
    }
    if (p->maxrec > 0)
      hipLaunchKernelGGL(k_el2_adj_inject<T>, dim3((p->maxrec + 63) / 64, p->nshots), dim3(64), 0,
                         st, p->dmodels, p->dshots, p->dadj, p->nshots, tb, k);
    hipLaunchKernelGGL((k_el2_adj_v<T, SPLIT>), grd, blk, 0, st, p->dmodels, p->dshots, p->dadj,
                       p->nshots, tb, k, p->dtsel_adj);
    hipLaunchKernelGGL((k_el2_adj_s<T, SPLIT>), grd, blk, 0, st, p->dmodels, p->dshots, p->dadj,
                       p->nshots, tb, k, p->dtsel_adj);
    hipLaunchKernelGGL(k_el2_adj_g<T>, grd, blk, 0, st, p->dmodels, p->dshots, p->dadj, p->nshots, tb, k);
  }
}

void launch_trail(Plan* p, hipStream_t st, int nsteps) {
  if (p->prec == SDT_FP64)
    launch_multi<double, true>(p, st, nsteps, false);
  else
    launch_multi<float, true>(p, st, nsteps, false);
}

template <typename T>
void launch_adjoint_em2(Plan* p, hipStream_t st, int khi, int klo) {
  const dim3 blk(TX, TZ);
  const dim3 grd((p->maxnx + TX - 1) / TX, (p->maxnz + TZ - 1) / TZ, p->nshots);
  const int* tb = p->dtbase;
  for (int k = khi - 1; k >= klo; --k) {
    if (!(p->adj_flags & SDT_ADJ_REFERENCE)) {
      in_slices(p->nadjwork, [&](int o, int n) {
        hipLaunchKernelGGL(k_em2_adj<T>, dim3((n + 7) / 8 * 8), dim3(64 * AR<T, true>), 0, st, p->dmodels, p->dshots,
                           p->dadj, p->dadjwork + o, n, tb, k, p->gmask, p->dtsel_adj);
      });
      continue;
    }
    if (p->maxrec > 0)
      hipLaunchKernelGGL(k_el2_adj_inject<T>, dim3((p->maxrec + 63) / 64, p->nshots), dim3(64), 0,
                         st, p->dmodels, p->dshots, p->dadj, p->nshots, tb, k);
    hipLaunchKernelGGL(k_em2_adj_e<T>, grd, blk, 0, st, p->dmodels, p->dshots, p->dadj, p->nshots,
                       tb, k, p->dtsel_adj, p->gmask);
    hipLaunchKernelGGL(k_em2_adj_h<T>, grd, blk, 0, st, p->dmodels, p->dshots, p->dadj, p->nshots,
                       tb, k);
    hipLaunchKernelGGL(k_em2_adj_g<T>, grd, blk, 0, st, p->dmodels, p->dshots, p->dadj, p->nshots,
                       tb, k);
  }
}

void launch_adjoint(Plan* p, hipStream_t st, int khi, int klo) {
  if (p->kind == SDT_EM2) {
    if (p->prec == SDT_FP64)
      launch_adjoint_em2<double>(p, st, khi, klo);
    else
      launch_adjoint_em2<float>(p, st, khi, klo);
  } else if (p->prec == SDT_FP64)
    p->split ? launch_adjoint_steps<double, true>(p, st, khi, klo)
             : launch_adjoint_steps<double, false>(p, st, khi, klo);
  else
    p->split ? launch_adjoint_steps<float, true>(p, st, khi, klo)
             : launch_adjoint_steps<float, false>(p, st, khi, klo);
  if (p->nflush > 0)
    hipLaunchKernelGGL(k_grad_flush, dim3(256, p->nflush), dim3(256), 0, st, p->dflush, p->gmask);
}

void drop_adjoint_graphs(Plan* p) {
  for (auto& x : p->seg_graphs) {
    (void)hipGraphExecDestroy(x.e);
    (void)hipGraphDestroy(x.g);
  }
  p->seg_graphs.clear();
}

// Work list of the two-step kernels for the plan's tile shape.  ELASTIC2:
// interior blocks first (their count in *ni), then the others; EM2: one list.
std::vector<int4> build_work2(const Plan* p, int* ni) {
  const bool em = p->kind == SDT_EM2;
  auto list = [&](int ew, int which) { return el2_work(p, p->el2_wb, p->el2_eh, p->el2_order, ew, which); };
  std::vector<int4> work = em ? std::vector<int4>() : list(EW2, 1);
  *ni = (int)work.size();
  const std::vector<int4> edge = em ? list(EW2E, 0) : list(EW2, 2);
  work.insert(work.end(), edge.begin(), edge.end());
  if (work.empty()) work.push_back(make_int4(-1, 0, 0, 0));
  return work;
}

// Grid sizes of the two-step launches for a list of nw items, ni interior.
void set_work2_grids(Plan* p, int nw, int ni) {
  p->nwork2 = nw;
  p->nwork2i = ni;
  p->el2x2_grid_i = std::max(8, std::min(ni, SDT_EL2_GRID) / 8 * 8);
  p->el2x2_grid = std::max(8, std::min(p->nwork2 - ni, SDT_EL2_GRID) / 8 * 8);
}

// Rebuild that list for the plan's tile shape.
int upload_work2(Plan* p) {
  int ni = 0;
  const std::vector<int4> work = build_work2(p, &ni);
  int4* dw = nullptr;
  HIP_TRY(hipMalloc(&dw, sizeof(int4) * work.size()));
  if (hipMemcpy(dw, work.data(), sizeof(int4) * work.size(), hipMemcpyHostToDevice) != hipSuccess) {
    (void)hipFree(dw);
    return fail(SDT_EDEVICE, "hipMemcpy failed (work list)");
  }
  if (p->dwork2) (void)hipFree(p->dwork2);
  p->dwork2 = dw;
  set_work2_grids(p, (int)work.size(), ni);
  return SDT_OK;
}

// Replay (capturing on first use) the segment graph (kind, key) on st.
template <typename F>
int replay_segment(Plan* p, int kind, long long key, hipStream_t st, F&& enqueue) {
  for (auto& x : p->seg_graphs)
    if (x.kind == kind && x.key == key) {
      HIP_TRY(hipGraphLaunch(x.e, st));
      return SDT_OK;
    }
  if (p->seg_graphs.size() >= 8) {  // many segment shapes: free the old ones once idle
    HIP_TRY(hipDeviceSynchronize());
    drop_adjoint_graphs(p);
  }
  Plan::SegGraph x{kind, key, nullptr, nullptr};
  HIP_TRY(hipStreamBeginCapture(p->cap, hipStreamCaptureModeThreadLocal));
  enqueue(p->cap);
  HIP_TRY(hipStreamEndCapture(p->cap, &x.g));
  HIP_TRY(hipGraphInstantiate(&x.e, x.g, nullptr, nullptr, 0));
  p->seg_graphs.push_back(x);
  HIP_TRY(hipGraphLaunch(x.e, st));
  return SDT_OK;
}

// What a plan's device arrays hold, built on the host: model and shot
// descriptors, work lists, the receivers-by-row index and the per-shot
// sizes.  The descriptors' pointers into the plan's own arrays (blowup,
// rrow, rxid) are set by stage_bind once those arrays have addresses.
struct Stage {
  std::vector<DModel> dm;
  std::vector<DShot> ds;
  std::vector<int4> work;       // one-step ELASTIC2 / EM2 list, or the 2.5-D list
  std::vector<int4> work2;      // two-step list (ELASTIC2, EM2)
  std::vector<int4> workm;      // region list (ELASTIC2, EM2)
  std::vector<int> rows_cols;   // receivers by row (ELASTIC2, EM2)
  std::vector<long> rec_off;    // per shot offset into rows_cols, -1 = none
  long long rows_cols_size = 0; // known before the receivers are read
  std::vector<long> nel, npsi;
};

// bytes of the fixed scratch of sdt_run_noalloc
#ifndef SDT_NOALLOC_SCRATCH_BYTES
#define SDT_NOALLOC_SCRATCH_BYTES (8u << 20)
#endif

// Host half of plan creation: validate the inputs and fill the plan's
// settings and everything of `S` except the receivers-by-row index.  Reads
// no device memory.  once: for one run of that many steps in the fixed scratch
// (0: any runs); least_rows > 0: with shorter lists, without regions and with
// tiles or chunks of at least that many rows.
int stage_host(Plan* p, int kind, int prec, const sdt_model* models, int nmodels,
               const sdt_shot* shots, int nshots, int nt, Stage& S, int once = 0, int least_rows = 0) {
  const bool split = (kind & SDT_SPLIT_CPML) != 0;
  kind &= ~SDT_SPLIT_CPML;
  if (split && kind != SDT_ELASTIC2) return fail(SDT_EINVAL, "SDT_SPLIT_CPML applies to ELASTIC2 only");
  int rc = validate(kind, split, prec, models, nmodels, shots, nshots, nt);
  if (rc) return rc;
  p->kind = kind;
  p->split = split;
  p->prec = prec;
  p->nmodels = nmodels;
  p->nshots = nshots;
  p->nt = nt;
  p->ncomp = kind_3d(kind) ? 3 : 2;
  p->hmodels.assign(models, models + nmodels);
  p->hshots.assign(shots, shots + nshots);
  S.rec_off.assign(nshots, -1);
  for (int s = 0; s < nshots; ++s) {
    p->maxrec = std::max(p->maxrec, shots[s].nrec);
    if (pingpong(kind) && shots[s].nrec > 0) {
      S.rec_off[s] = (long)S.rows_cols_size;
      S.rows_cols_size += models[shots[s].model].nz + 1 + 2LL * shots[s].nrec;
    }
  }
  S.dm.assign(nmodels, DModel());
  for (int m = 0; m < nmodels; ++m) {
    const sdt_model& M = models[m];
    DModel& D = S.dm[m];
    D.nx = M.nx; D.ny = M.ny; D.nz = M.nz;
    D.lx = M.lx; D.ly = kind_3d(kind) ? M.ly : 0; D.lz = M.lz;
    D.dx = M.dx; D.dy = M.dy; D.dz = M.dz; D.dt = M.dt;
    for (int q = 0; q < 4; ++q) D.scal[q] = M.scal[q];
    for (int q = 0; q < 40; ++q) D.coef[q] = M.coef[q];
    for (int a = 0; a < 3; ++a)
      for (int q = 0; q < 6; ++q) D.prof[a][q] = M.prof[a][q];
    D.aux = M.aux;
    p->maxnx = std::max(p->maxnx, M.nx);
    p->maxnz = std::max(p->maxnz, M.nz);
  }
  S.ds.assign(nshots, DShot());
  for (int s = 0; s < nshots; ++s) {
    const sdt_shot& H = shots[s];
    DShot& D = S.ds[s];
    D.model = H.model; D.isrc = H.isrc; D.jsrc = kind_3d(kind) ? H.jsrc : 0; D.ksrc = H.ksrc;
    for (int f = 0; f < 9; ++f) D.f[f] = H.field[f];
    D.psi = H.psi;
    for (int f = 0; f < 9; ++f) D.g[f] = H.field_b[f];
    D.psi2 = H.psi_b;
    for (int c = 0; c < 3; ++c) D.src[c] = H.src[c];
    for (int c = 0; c < 6; ++c) D.msrc[c] = (kind == SDT_ELASTIC2 || kind == SDT_ELASTIC25) ? H.msrc[c] : nullptr;
    D.nrec = H.nrec; D.rec = H.rec; D.trace = H.trace;
    D.blowup = nullptr;
    D.rrow = nullptr;
    D.rxid = nullptr;
  }
  // work lists: (shot, x0, z0); all shots of one tile share blockIdx % 8 (XCD)
  if (kind_3d(kind)) {
    S.work = el25_work(p, least_rows);
    set_blocks25(p);
  }
  if (pingpong(kind)) {
    default_shape(p);
    if (least_rows > 0) p->multi = false;
    if (least_rows > p->el2_eh) {
      p->el2_eh = least_rows;
      p->el2_wb = 4;
    }
    p->nmulti = (int)regions2d(p, p->tm);
    if (once > 0 && (run_mode(p, once, 0) != 2 || sizeof(int4) * p->nmulti > SDT_NOALLOC_SCRATCH_BYTES))
      p->multi = false;
    if (p->multi) S.workm = multi_work(p, p->tm);
    S.work = el2_work(p, p->el2_wb, p->el2_eh, p->el2_order);
    const int nblk = (int)S.work.size();
    p->el2_grid = std::max(8, std::min(nblk, SDT_EL2_GRID) / 8 * 8);
    int ni = 0;
    S.work2 = build_work2(p, &ni);
    set_work2_grids(p, (int)S.work2.size(), ni);
  }
  if (S.work.empty()) S.work.push_back(make_int4(-1, 0, 0, 0));
  p->nwork = (int)S.work.size();
  S.nel.resize(nshots);
  S.npsi.resize(nshots);
  for (int s = 0; s < nshots; ++s) {
    const sdt_model& M = models[shots[s].model];
    S.nel[s] = (long)M.nx * M.ny * M.nz;
    S.npsi[s] = (long)psi_elems(kind | (split ? SDT_SPLIT_CPML : 0), M.nx, M.ny, M.nz, M.lx,
                                kind_3d(kind) ? M.ly : 0, M.lz);
    p->maxel = std::max<long long>(p->maxel, std::max(S.nel[s], S.npsi[s]));
  }
  return SDT_OK;
}

// Read every shot's receivers back from the device (synchronous copies),
// check them against the grid, and build the receivers-by-row index of the
// 2-D kinds: per shot rrow[nz + 1] then (column, index) pairs sorted by
// (row, column).
int stage_receivers(Plan* p, Stage& S) {
  p->reck.assign(p->nshots, {INT_MAX, -1});
  S.rows_cols.clear();
  S.rows_cols.reserve((size_t)S.rows_cols_size);
  for (int s = 0; s < p->nshots; ++s) {
    const sdt_shot& H = p->hshots[s];
    if (H.nrec <= 0) continue;
    std::vector<int> rec(3 * (size_t)H.nrec);
    if (hipMemcpy(rec.data(), H.rec, rec.size() * sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
      return fail(SDT_EDEVICE, "cannot read receiver indices (not device memory?)");
    const sdt_model& M = p->hmodels[H.model];
    for (int r = 0; r < H.nrec; ++r) {
      const int i = rec[3 * r], j = rec[3 * r + 1], k = rec[3 * r + 2];
      if (i < 0 || i >= M.nx || k < 0 || k >= M.nz || j < 0 || j >= M.ny)
        return fail(SDT_EINVAL, "shot " + std::to_string(s) + ": receiver " + std::to_string(r) +
                                    " outside the padded grid");
      p->reck[s] = {std::min(p->reck[s].first, k), std::max(p->reck[s].second, k)};
    }
    if (S.rec_off[s] < 0) continue;
    std::vector<int> order(H.nrec);
    for (int r = 0; r < H.nrec; ++r) order[r] = r;
    std::sort(order.begin(), order.end(), [&](int a, int b) {
      return rec[3 * a + 2] != rec[3 * b + 2] ? rec[3 * a + 2] < rec[3 * b + 2] : rec[3 * a] < rec[3 * b];
    });
    std::vector<int> rrow(M.nz + 1, 0);
    for (int r = 0; r < H.nrec; ++r) rrow[rec[3 * r + 2] + 1]++;
    for (int k = 0; k < M.nz; ++k) rrow[k + 1] += rrow[k];
    S.rows_cols.insert(S.rows_cols.end(), rrow.begin(), rrow.end());
    for (int r : order) {
      S.rows_cols.push_back(rec[3 * r]);
      S.rows_cols.push_back(r);
    }
  }
  return SDT_OK;
}

// Point each shot descriptor at its flag and its part of the receiver index.
void stage_bind(const Plan* p, Stage& S) {
  for (int s = 0; s < p->nshots; ++s) {
    DShot& D = S.ds[s];
    D.blowup = p->dflags + s;
    D.rrow = S.rec_off[s] < 0 ? nullptr : p->drec + S.rec_off[s];
    D.rxid = S.rec_off[s] < 0 ? nullptr : p->drec + S.rec_off[s] + p->hmodels[p->hshots[s].model].nz + 1;
  }
}

// ---------------------------------------------------------------------------
// Fixed scratch of the allocation-free run (sdt_run_noalloc): descriptors,
// work lists, receiver index, flags and step counters of one call, carved
// from one static device array per GPU.  Host code never passes `scratch`
// itself to the device: it uses the address hipGetSymbolAddress returns for
// the current device (scratch_ptr).
// ---------------------------------------------------------------------------
__device__ __align__(256) unsigned char scratch[SDT_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch (looked up once per device).
int scratch_ptr(unsigned char** out) {
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(SDT_EDEVICE, "device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(SDT_EDEVICE, "hipGetSymbolAddress returned null for the scratch array");
    g_scratch_ptr[dev] = ptr;
  }
  *out = static_cast<unsigned char*>(g_scratch_ptr[dev]);
  return SDT_OK;
}

// Offsets of one call's arrays inside the scratch (256-byte aligned).
struct ScratchLayout {
  size_t models, shots, work, work2, workm, rec, flags, ints, nel, npsi, total;
};
ScratchLayout scratch_layout(const Plan* p, const Stage& S) {
  auto up = [](size_t v) { return (v + 255) & ~size_t(255); };
  ScratchLayout L;
  size_t o = 0;
  L.models = o; o = up(o + sizeof(DModel) * p->nmodels);
  L.shots = o;  o = up(o + sizeof(DShot) * p->nshots);
  L.work = o;   o = up(o + sizeof(int4) * S.work.size());
  L.work2 = o;  o = up(o + sizeof(int4) * S.work2.size());
  L.workm = o;  o = up(o + sizeof(int4) * S.workm.size());
  L.rec = o;    o = up(o + sizeof(int) * (size_t)S.rows_cols_size);
  L.flags = o;  o = up(o + sizeof(int) * p->nshots);
  L.ints = o;   o = up(o + 2 * sizeof(int));
  L.nel = o;    o = up(o + sizeof(long) * p->nshots);
  L.npsi = o;   o = up(o + sizeof(long) * p->nshots);
  L.total = o;
  return L;
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

const char* sdt_last_error(void) { return g_err.c_str(); }

const char* sdt_version(void) { return "seidart_hip 0.1 gfx950"; }

int sdt_psi_elems(int kind, int nx, int ny, int nz, int lx, int ly, int lz, long long* out) {
  if (!out) return fail(SDT_EINVAL, "out is null");
  const long long n = psi_elems(kind, nx, ny, nz, lx, ly, lz);
  if (n < 0) return fail(SDT_EINVAL, "unknown kind");
  *out = n;
  return SDT_OK;
}

int sdt_plan_create(int kind, int prec, const sdt_model* models, int nmodels,
                    const sdt_shot* shots, int nshots, int nt, void** out_plan) {
  if (!out_plan) return fail(SDT_EINVAL, "out_plan is null");
  *out_plan = nullptr;
  Plan* p = new Plan();
  auto bail = [&](int code) {
    sdt_plan_destroy(p);
    return code;
  };
  Stage S;
  int rc = stage_host(p, kind, prec, models, nmodels, shots, nshots, nt, S);
  if (rc) return bail(rc);
  rc = stage_receivers(p, S);
  if (rc) return bail(rc);
  if (!S.rows_cols.empty()) {
    if (hipMalloc(&p->drec, sizeof(int) * S.rows_cols.size()) != hipSuccess ||
        hipMemcpy(p->drec, S.rows_cols.data(), sizeof(int) * S.rows_cols.size(), hipMemcpyHostToDevice) !=
            hipSuccess)
      return bail(fail(SDT_EDEVICE, "hipMalloc/hipMemcpy failed (receivers by row)"));
  }
  if (hipMalloc(&p->dflags, sizeof(int) * nshots) != hipSuccess ||
      hipMalloc(&p->dbase, sizeof(int)) != hipSuccess || hipMalloc(&p->dit0, sizeof(int)) != hipSuccess)
    return bail(fail(SDT_EDEVICE, "hipMalloc failed (flags)"));
  stage_bind(p, S);
  if (hipMalloc(&p->dnel, sizeof(long) * nshots) != hipSuccess ||
      hipMalloc(&p->dnpsi, sizeof(long) * nshots) != hipSuccess ||
      hipMemcpy(p->dnel, S.nel.data(), sizeof(long) * nshots, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->dnpsi, S.npsi.data(), sizeof(long) * nshots, hipMemcpyHostToDevice) != hipSuccess)
    return bail(fail(SDT_EDEVICE, "hipMalloc/hipMemcpy failed (sizes)"));
  if (hipMalloc(&p->dmodels, sizeof(DModel) * nmodels) != hipSuccess ||
      hipMalloc(&p->dshots, sizeof(DShot) * nshots) != hipSuccess ||
      hipMalloc(&p->dwork, sizeof(int4) * S.work.size()) != hipSuccess)
    return bail(fail(SDT_EDEVICE, "hipMalloc failed (descriptors)"));
  if (hipMemcpy(p->dmodels, S.dm.data(), sizeof(DModel) * nmodels, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->dshots, S.ds.data(), sizeof(DShot) * nshots, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(p->dwork, S.work.data(), sizeof(int4) * S.work.size(), hipMemcpyHostToDevice) != hipSuccess)
    return bail(fail(SDT_EDEVICE, "hipMemcpy failed (descriptors)"));
  if (!S.work2.empty()) {
    if (hipMalloc(&p->dwork2, sizeof(int4) * S.work2.size()) != hipSuccess ||
        hipMemcpy(p->dwork2, S.work2.data(), sizeof(int4) * S.work2.size(), hipMemcpyHostToDevice) !=
            hipSuccess)
      return bail(fail(SDT_EDEVICE, "hipMalloc/hipMemcpy failed (work list)"));
  }
  if (!S.workm.empty()) {
    if (hipMalloc(&p->dwmulti, sizeof(int4) * S.workm.size()) != hipSuccess ||
        hipMemcpy(p->dwmulti, S.workm.data(), sizeof(int4) * S.workm.size(), hipMemcpyHostToDevice) !=
            hipSuccess)
      return bail(fail(SDT_EDEVICE, "hipMalloc/hipMemcpy failed (work list)"));
  }
  hipLaunchKernelGGL(k_fill_int, dim3((nshots + 255) / 256), dim3(256), 0, nullptr, p->dflags,
                     nshots, INT_MAX);
  hipLaunchKernelGGL(k_set_int2, dim3(1), dim3(1), 0, nullptr, p->dbase, 0, p->dit0, 0);
  if (hipDeviceSynchronize() != hipSuccess) return bail(fail(SDT_EDEVICE, "init kernels failed"));
  if (hipStreamCreateWithFlags(&p->cap, hipStreamNonBlocking) != hipSuccess)
    return bail(fail(SDT_EDEVICE, "hipStreamCreate failed"));
  *out_plan = p;
  return SDT_OK;
}

int sdt_plan_run(void* plan, int it0, int nsteps, int graph_block, void* stream) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (it0 < 0 || nsteps < 0 || (long long)it0 + nsteps > p->nt)
    return fail(SDT_EINVAL, "step range outside [0, nt)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  p->last = st;
  if (nsteps == 0) return SDT_OK;
  const int mode = run_mode(p, nsteps, graph_block);
  start_of_run(p, st, it0, mode != 0);
  hipLaunchKernelGGL(k_set_int2, dim3(1), dim3(1), 0, st, p->dbase, it0, p->dit0, it0);
  int done = 0;
  if (graph_block > 1 && nsteps >= graph_block) {
    if (p->graph_block != graph_block || !p->gexec || p->graph_mode != mode) {
      if (p->gexec) { (void)hipGraphExecDestroy(p->gexec); p->gexec = nullptr; }
      if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
      HIP_TRY(hipStreamBeginCapture(p->cap, hipStreamCaptureModeThreadLocal));
      launch_run(p, p->cap, graph_block, mode, true);
      hipLaunchKernelGGL(k_add_int, dim3(1), dim3(1), 0, p->cap, p->dbase, graph_block);
      HIP_TRY(hipStreamEndCapture(p->cap, &p->graph));
      HIP_TRY(hipGraphInstantiate(&p->gexec, p->graph, nullptr, nullptr, 0));
      p->graph_block = graph_block;
      p->graph_mode = mode;
    }
    for (; done + graph_block <= nsteps; done += graph_block) HIP_TRY(hipGraphLaunch(p->gexec, st));
  }
  int final_b = mode == 2 ? 0 : mode == 1 ? (nsteps / 2 + (nsteps & 1)) & 1 : -1;
  if (done < nsteps) {
    const int b = launch_run(p, st, nsteps - done, mode, false);
    if (mode == 2) final_b = b;
  }
  end_of_run(p, st, it0 + nsteps, final_b);
  HIP_TRY(hipGetLastError());
  return SDT_OK;
}

int sdt_plan_profile(void* plan, int it0, int nsteps, void* stream, double* out_ms) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !out_ms) return fail(SDT_EINVAL, "plan or out_ms is null");
  if (it0 < 0 || nsteps <= 0 || (long long)it0 + nsteps > p->nt)
    return fail(SDT_EINVAL, "step range outside [0, nt)");
  hipStream_t st = static_cast<hipStream_t>(stream);
  p->last = st;
  hipEvent_t ev[4];
  for (int q = 0; q < 4; ++q) HIP_TRY(hipEventCreate(&ev[q]));
  double acc[3] = {0, 0, 0};
  const int mode = run_mode(p, nsteps, 0);
  start_of_run(p, st, it0, mode != 0);
  hipLaunchKernelGGL(k_set_int2, dim3(1), dim3(1), 0, st, p->dbase, it0, p->dit0, it0);
  int rc = SDT_OK;
  if (mode != 0) {
    // several steps per launch: slot 0 is the mean per launch; the single
    // step that ends an odd run of pairs is not timed
    const int L = mode == 2 ? region_launches(nsteps, p->tm, false) : nsteps / 2 + (nsteps & 1);
    int timed = 0;
    for (int l = 0; l < L && rc == SDT_OK; ++l) {
      const bool single = mode == 1 && 2 * l + 1 == nsteps;
      const int r = (int)((long long)nsteps * l / L), k = (int)((long long)nsteps * (l + 1) / L) - r;
      if (hipEventRecord(ev[0], st) != hipSuccess) { rc = fail(SDT_EDEVICE, "hipEventRecord"); break; }
      if (mode == 2)
        p->prec == SDT_FP64 ? launch_region<double>(p, st, r, k, l & 1) : launch_region<float>(p, st, r, k, l & 1);
      else if (p->prec == SDT_FP64)
        launch_two<double>(p, st, 2 * l, single);
      else
        launch_two<float>(p, st, 2 * l, single);
      if (hipEventRecord(ev[1], st) != hipSuccess || hipEventSynchronize(ev[1]) != hipSuccess) {
        rc = fail(SDT_EDEVICE, "event sync failed");
        break;
      }
      if (single) break;
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, ev[0], ev[1]) != hipSuccess) { rc = fail(SDT_EDEVICE, "elapsed"); break; }
      acc[0] += ms;
      ++timed;
    }
    if (rc == SDT_OK) end_of_run(p, st, it0 + nsteps, L & 1);
    for (int q = 0; q < 4; ++q) (void)hipEventDestroy(ev[q]);
    if (rc) return rc;
    out_ms[0] = timed ? acc[0] / timed : 0.0;
    out_ms[1] = 0.0;
    out_ms[2] = 0.0;
    HIP_TRY(hipGetLastError());
    return SDT_OK;
  }
  for (int s = 0; s < nsteps && rc == SDT_OK; ++s) {
    for (int w = 0; w < 3; ++w) {
      if (hipEventRecord(ev[w], st) != hipSuccess) { rc = fail(SDT_EDEVICE, "hipEventRecord"); break; }
      if (p->prec == SDT_FP64)
        launch_one<double>(p, st, s, w);
      else
        launch_one<float>(p, st, s, w);
    }
    if (rc) break;
    if (hipEventRecord(ev[3], st) != hipSuccess || hipEventSynchronize(ev[3]) != hipSuccess) {
      rc = fail(SDT_EDEVICE, "event sync failed");
      break;
    }
    for (int w = 0; w < 3; ++w) {
      float ms = 0.f;
      if (hipEventElapsedTime(&ms, ev[w], ev[w + 1]) != hipSuccess) { rc = fail(SDT_EDEVICE, "elapsed"); break; }
      acc[w] += ms;
    }
  }
  if (rc == SDT_OK) end_of_run(p, st, it0 + nsteps);
  for (int q = 0; q < 4; ++q) (void)hipEventDestroy(ev[q]);
  if (rc) return rc;
  for (int w = 0; w < 3; ++w) out_ms[w] = acc[w] / nsteps;
  HIP_TRY(hipGetLastError());
  return SDT_OK;
}

int sdt_plan_check(void* plan, int* first_step, int* per_shot) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  HIP_TRY(hipStreamSynchronize(p->last));
  std::vector<int> f(p->nshots);
  HIP_TRY(hipMemcpy(f.data(), p->dflags, sizeof(int) * p->nshots, hipMemcpyDeviceToHost));
  int first = INT_MAX;
  for (int s = 0; s < p->nshots; ++s) {
    first = std::min(first, f[s]);
    if (per_shot) per_shot[s] = f[s] == INT_MAX ? -1 : f[s];
  }
  if (first_step) *first_step = first == INT_MAX ? -1 : first;
  if (first != INT_MAX)
    return fail(SDT_EUNSTABLE, "code became unstable and blew up at step " + std::to_string(first));
  return SDT_OK;
}

int sdt_run_noalloc(int kind, int prec, const sdt_model* models, int nmodels,
                    const sdt_shot* shots, int nshots, int nt, int it0, int nsteps, void* stream,
                    int* first_step, int* per_shot) {
  if (first_step) *first_step = -1;
  if (it0 < 0 || nsteps < 0 || (long long)it0 + nsteps > nt)
    return fail(SDT_EINVAL, "step range outside [0, nt)");
  // The plan lives on this stack frame; its device arrays point into the
  // scratch, so nothing of it is freed (sdt_plan_destroy is never called).
  Plan P;
  Plan* p = &P;
  Stage S;
  int rc = stage_host(p, kind, prec, models, nmodels, shots, nshots, nt, S, nsteps);
  if (rc) return rc;
  ScratchLayout L = scratch_layout(p, S);
  // work lists too long for the scratch: no regions, then taller tiles, as far as
  // that helps
  for (int rows = kind_3d(p->kind) ? 8 : 1; L.total > (size_t)SDT_NOALLOC_SCRATCH_BYTES && rows <= 65536; rows *= 2) {
    P = Plan();
    S = Stage();
    rc = stage_host(p, kind, prec, models, nmodels, shots, nshots, nt, S, nsteps, rows);
    if (rc) return rc;
    L = scratch_layout(p, S);
  }
  if (L.total > (size_t)SDT_NOALLOC_SCRATCH_BYTES)
    return fail(SDT_EINVAL, "sdt_run_noalloc: this run needs " + std::to_string(L.total) +
                                " bytes of scratch (descriptors, work lists, receiver index) but the "
                                "library holds " + std::to_string((size_t)SDT_NOALLOC_SCRATCH_BYTES) +
                                "; use sdt_plan_create / sdt_plan_run");
  unsigned char* base = nullptr;
  rc = scratch_ptr(&base);
  if (rc) return rc;
  rc = stage_receivers(p, S);
  if (rc) return rc;
  p->dmodels = reinterpret_cast<DModel*>(base + L.models);
  p->dshots = reinterpret_cast<DShot*>(base + L.shots);
  p->dwork = reinterpret_cast<int4*>(base + L.work);
  p->dwork2 = S.work2.empty() ? nullptr : reinterpret_cast<int4*>(base + L.work2);
  p->dwmulti = S.workm.empty() ? nullptr : reinterpret_cast<int4*>(base + L.workm);
  p->drec = S.rows_cols.empty() ? nullptr : reinterpret_cast<int*>(base + L.rec);
  p->dflags = reinterpret_cast<int*>(base + L.flags);
  p->dbase = reinterpret_cast<int*>(base + L.ints);
  p->dit0 = p->dbase + 1;
  p->dnel = reinterpret_cast<long*>(base + L.nel);
  p->dnpsi = reinterpret_cast<long*>(base + L.npsi);
  stage_bind(p, S);
  hipStream_t st = static_cast<hipStream_t>(stream);
  p->last = st;
  // the host vectors outlive the copies: the call ends with a stream sync
  HIP_TRY(hipMemcpyAsync(p->dmodels, S.dm.data(), sizeof(DModel) * nmodels, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(p->dshots, S.ds.data(), sizeof(DShot) * nshots, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(p->dwork, S.work.data(), sizeof(int4) * S.work.size(), hipMemcpyHostToDevice, st));
  if (p->dwork2)
    HIP_TRY(hipMemcpyAsync(p->dwork2, S.work2.data(), sizeof(int4) * S.work2.size(),
                           hipMemcpyHostToDevice, st));
  if (p->dwmulti)
    HIP_TRY(hipMemcpyAsync(p->dwmulti, S.workm.data(), sizeof(int4) * S.workm.size(),
                           hipMemcpyHostToDevice, st));
  if (p->drec)
    HIP_TRY(hipMemcpyAsync(p->drec, S.rows_cols.data(), sizeof(int) * S.rows_cols.size(),
                           hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(p->dnel, S.nel.data(), sizeof(long) * nshots, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(p->dnpsi, S.npsi.data(), sizeof(long) * nshots, hipMemcpyHostToDevice, st));
  // flags and step counters start fresh every call (the scratch keeps the
  // previous call's contents); cleared by kernels, not hipMemsetAsync
  hipLaunchKernelGGL(k_fill_int, dim3((nshots + 255) / 256), dim3(256), 0, st, p->dflags, nshots, INT_MAX);
  hipLaunchKernelGGL(k_set_int2, dim3(1), dim3(1), 0, st, p->dbase, it0, p->dit0, it0);
  if (nsteps > 0) {
    const int mode = run_mode(p, nsteps, 0);
    start_of_run(p, st, it0, mode != 0);
    end_of_run(p, st, it0 + nsteps, launch_run(p, st, nsteps, mode, false));
  }
  HIP_TRY(hipGetLastError());
  std::vector<int> f(nshots);
  HIP_TRY(hipMemcpyAsync(f.data(), p->dflags, sizeof(int) * nshots, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  int first = INT_MAX;
  for (int s = 0; s < nshots; ++s) {
    first = std::min(first, f[s]);
    if (per_shot) per_shot[s] = f[s] == INT_MAX ? -1 : f[s];
  }
  if (first_step) *first_step = first == INT_MAX ? -1 : first;
  if (first != INT_MAX)
    return fail(SDT_EUNSTABLE, "code became unstable and blew up at step " + std::to_string(first));
  return SDT_OK;
}

long long sdt_noalloc_scratch_bytes(void) { return (long long)SDT_NOALLOC_SCRATCH_BYTES; }

int sdt_hbm_probe(const void* src, void* dst, long long nfloat, void* stream) {
  if (!src || !dst || nfloat <= 0) return fail(SDT_EINVAL, "sdt_hbm_probe: null buffer or empty size");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_hbm_probe, dim3(256 * 8 * 4), dim3(256), 0, st, static_cast<const float*>(src),
                     static_cast<float*>(dst), nfloat);
  HIP_TRY(hipGetLastError());
  return SDT_OK;
}

// Rebuild the 2-D work lists for a tile shape and order (all or nothing: on
// a failure the plan keeps its tiles, order and work lists), dropping the
// graphs that bake in the old launch shape.
static int retile(Plan* p, int waves_per_block, int rows, int order) {
  // the old work list and the graphs that bake in the launch shape may be in flight
  HIP_TRY(hipDeviceSynchronize());
  const int owb = p->el2_wb, oeh = p->el2_eh, oord = p->el2_order;
  p->el2_wb = waves_per_block;
  p->el2_eh = rows;
  p->el2_order = order;
  const std::vector<int4> work = el2_work(p, p->el2_wb, p->el2_eh, p->el2_order);
  int4* dw = nullptr;
  int rc = SDT_OK;
  if (hipMalloc(&dw, sizeof(int4) * work.size()) != hipSuccess) {
    dw = nullptr;
    rc = fail(SDT_EDEVICE, "hipMalloc failed (work list)");
  } else if (hipMemcpy(dw, work.data(), sizeof(int4) * work.size(), hipMemcpyHostToDevice) !=
             hipSuccess) {
    rc = fail(SDT_EDEVICE, "hipMemcpy failed (work list)");
  } else if (p->dwork2) {
    rc = upload_work2(p);  // replaces the two-step list only when it succeeds
  }
  if (rc != SDT_OK) {
    if (dw) (void)hipFree(dw);
    p->el2_wb = owb;
    p->el2_eh = oeh;
    p->el2_order = oord;
    return rc;
  }
  (void)hipFree(p->dwork);
  p->dwork = dw;
  p->nwork = (int)work.size();
  p->el2_grid = std::max(8, std::min(p->nwork, SDT_EL2_GRID) / 8 * 8);
  if (p->gexec) { (void)hipGraphExecDestroy(p->gexec); p->gexec = nullptr; }
  if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
  drop_adjoint_graphs(p);
  return SDT_OK;
}

int sdt_plan_set_tiles(void* plan, int waves_per_block, int rows) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (!pingpong(p->kind)) return fail(SDT_EINVAL, "tile shapes apply to ELASTIC2 and EM2 plans");
  if (waves_per_block != 1 && waves_per_block != 2 && waves_per_block != 4)
    return fail(SDT_EINVAL, "waves_per_block must be 1, 2 or 4");
  if (rows < 1 || rows > 256) return fail(SDT_EINVAL, "rows must be in [1, 256]");
  if (waves_per_block != p->el2_wb || rows != p->el2_eh) {
    const int rc = retile(p, waves_per_block, rows, p->el2_order);
    if (rc) return rc;
  }
  p->regions = false;
  return SDT_OK;
}

int sdt_plan_set_tile_order(void* plan, int order) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (!pingpong(p->kind)) return fail(SDT_EINVAL, "tile orders apply to ELASTIC2 and EM2 plans");
  if (order != 0 && order != 1) return fail(SDT_EINVAL, "tile order must be 0 or 1");
  if (order != p->el2_order) {
    const int rc = retile(p, p->el2_wb, p->el2_eh, order);
    if (rc) return rc;
  }
  p->regions = false;
  return SDT_OK;
}

int sdt_plan_get_tile_order(void* plan, int* order) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !order) return fail(SDT_EINVAL, "null argument");
  *order = p->el2_order;
  return SDT_OK;
}

int sdt_plan_set_steps_per_launch(void* plan, int steps) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (steps != 1 && steps != 2) return fail(SDT_EINVAL, "steps per launch must be 1 or 2");
  if (steps == 2 && p->kind != SDT_ELASTIC2 && p->kind != SDT_EM2)
    return fail(SDT_EINVAL, "two steps per launch apply to ELASTIC2 and EM2 plans");
  p->spl = steps;
  p->regions = false;
  return SDT_OK;
}

int sdt_plan_set_regions(void* plan, int on) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (!pingpong(p->kind)) return fail(SDT_EINVAL, "regions apply to ELASTIC2 and EM2 plans");
  if (on != 0 && on != 1) return fail(SDT_EINVAL, "on must be 0 or 1");
  p->regions = on == 1;
  return SDT_OK;
}

int sdt_plan_get_regions(void* plan, int* on, int* most_steps, int* count) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !on) return fail(SDT_EINVAL, "null argument");
  *on = p->multi && p->regions;
  if (most_steps) *most_steps = p->tm;
  if (count) *count = p->nmulti;
  return SDT_OK;
}

int sdt_plan_get_run_mode(void* plan, int nsteps, int graph_block, int* mode) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !mode) return fail(SDT_EINVAL, "null argument");
  if (nsteps < 1) return fail(SDT_EINVAL, "nsteps must be positive");
  *mode = run_mode(p, nsteps, graph_block);
  return SDT_OK;
}

int sdt_plan_get_steps_per_launch(void* plan, int* steps) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !steps) return fail(SDT_EINVAL, "null argument");
  *steps = p->spl;
  return SDT_OK;
}

int sdt_plan_get_tiles(void* plan, int* waves_per_block, int* rows) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !waves_per_block || !rows) return fail(SDT_EINVAL, "null argument");
  *waves_per_block = p->el2_wb;
  *rows = p->el2_eh;
  return SDT_OK;
}

int sdt_state_elems(int kind, int nx, int ny, int nz, int lx, int ly, int lz, long long* out) {
  if (!out) return fail(SDT_EINVAL, "out is null");
  const long long n = state_elems(kind, nx, ny, nz, lx, ly, lz);
  if (n < 0) return fail(SDT_EINVAL, "unknown kind");
  *out = n;
  return SDT_OK;
}

int sdt_adjoint_work_elems(int kind, int nx, int ny, int nz, int lx, int ly, int lz,
                           long long* out) {
  (void)ny; (void)lx; (void)ly; (void)lz;
  if (!out) return fail(SDT_EINVAL, "out is null");
  const int base = kind & ~SDT_SPLIT_CPML;
  if (base != SDT_ELASTIC2 && base != SDT_EM2)
    return fail(SDT_EINVAL, "the adjoint is available for ELASTIC2 and EM2 only");
  *out = (base == SDT_ELASTIC2 ? 12LL : 4LL) * nx * nz;
  return SDT_OK;
}

int sdt_adjoint_setup(void* plan, const sdt_adj_shot* adj, int nshots, unsigned grad_mask,
                      int flags) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p || !adj) return fail(SDT_EINVAL, "plan or adj is null");
  if (grad_mask & ~0xfffu) return fail(SDT_EINVAL, "grad_mask has bits beyond the 12 slots");
  if (flags & ~SDT_ADJ_REFERENCE) return fail(SDT_EINVAL, "unknown adjoint flags");
  if (p->kind != SDT_ELASTIC2 && p->kind != SDT_EM2)
    return fail(SDT_EINVAL, "the adjoint is available for ELASTIC2 and EM2 only");
  if (nshots != p->nshots) return fail(SDT_EINVAL, "adj must hold one entry per shot of the plan");
  if (p->kind == SDT_EM2 && (grad_mask & ~0xfu))
    return fail(SDT_EINVAL, "EM2 has 4 coefficient slots (grad_mask <= 0xf)");
  std::vector<DAdj> h(nshots);
  for (int s = 0; s < nshots; ++s) {
    const sdt_adj_shot& a = adj[s];
    const std::string tag = "shot " + std::to_string(s) + ": ";
    if (!a.trail[0] || !a.lam[0] || !a.lam[1] || !a.work || !a.grad)
      return fail(SDT_EINVAL, tag + "trail[0], lam, work and grad must be set");
    if ((a.trail[1] != nullptr) != (adj[0].trail[1] != nullptr))
      return fail(SDT_EINVAL, tag + "trail[1] must be set for every shot or for none");
    if (a.trail_len < 2) return fail(SDT_EINVAL, tag + "trail_len must be at least 2");
    const sdt_model& M = p->hmodels[p->hshots[s].model];
    DAdj& D = h[s];
    if (p->kind == SDT_ELASTIC2 || p->kind == SDT_EM2) {
      // the fused kernels address a state and a gradient with 32-bit byte offsets
      const long long es = p->prec == SDT_FP64 ? 8 : 4;
      const long long st = state_elems(p->kind | (p->split ? SDT_SPLIT_CPML : 0), M.nx, M.ny, M.nz,
                                       M.lx, M.ly, M.lz);
      if (st * es >= (1LL << 32) || 12LL * M.nx * M.nz * es >= (1LL << 32))
        return fail(SDT_EINVAL, tag + "grid too large for the adjoint (state or gradient over 4 GiB)");
    }
    D.trail[0] = a.trail[0];
    D.trail[1] = a.trail[1];
    D.slot = (long)state_elems(p->kind | (p->split ? SDT_SPLIT_CPML : 0), M.nx, M.ny, M.nz, M.lx,
                               kind_3d(p->kind) ? M.ly : 0, M.lz);
    D.trail_len = a.trail_len;
    D.lam[0] = a.lam[0];
    D.lam[1] = a.lam[1];
    D.work = a.work;
    D.resid = a.resid;
    D.grad = a.grad;
    D.gsrc = a.gsrc;
  }
  // the previous descriptors may still be read by queued kernels
  HIP_TRY(hipDeviceSynchronize());
  if (!p->dadj) HIP_TRY(hipMalloc(&p->dadj, sizeof(DAdj) * nshots));
  p->gmask = grad_mask;
  p->adj_flags = flags;
  drop_adjoint_graphs(p);  // they bake in the options
  // FP32 staging of the gradient, one per distinct grad array (fused kernel)
  for (float* g : p->g32) (void)hipFree(g);
  p->g32.clear();
  if (p->dflush) { (void)hipFree(p->dflush); p->dflush = nullptr; }
  p->nflush = 0;
  // (the EM2 reference kernels stage in FP32 too; the elastic ones add in FP64)
  if (p->prec == SDT_FP32 && (p->kind == SDT_EM2 || !(flags & SDT_ADJ_REFERENCE))) {
    std::vector<DFlush> fl;
    for (int s = 0; s < nshots; ++s) {
      const sdt_model& M = p->hmodels[p->hshots[s].model];
      const long nel = (long)M.nx * M.nz;
      int f = 0;
      while (f < (int)fl.size() && fl[f].grad != h[s].grad) ++f;
      if (f == (int)fl.size()) {
        float* g = nullptr;
        HIP_TRY(hipMalloc(&g, sizeof(float) * 12 * nel));
        HIP_TRY(hipMemset(g, 0, sizeof(float) * 12 * nel));
        p->g32.push_back(g);
        fl.push_back(DFlush{h[s].grad, g, nel});
      } else if (fl[f].n != nel) {
        return fail(SDT_EINVAL, "shots sharing a grad array must have grids of one size");
      }
      h[s].g32 = fl[f].g32;
    }
    HIP_TRY(hipMalloc(&p->dflush, sizeof(DFlush) * fl.size()));
    HIP_TRY(hipMemcpy(p->dflush, fl.data(), sizeof(DFlush) * fl.size(), hipMemcpyHostToDevice));
    p->nflush = (int)fl.size();
  }
  HIP_TRY(hipMemcpy(p->dadj, h.data(), sizeof(DAdj) * nshots, hipMemcpyHostToDevice));
  p->hadj = h;
  if (!p->dtbase) HIP_TRY(hipMalloc(&p->dtbase, sizeof(int)));
  if (!p->dtsel_trail) HIP_TRY(hipMalloc(&p->dtsel_trail, sizeof(int)));
  if (!p->dtsel_adj) HIP_TRY(hipMalloc(&p->dtsel_adj, sizeof(int)));
  if (!p->dtrwork) {
    // The recomputation runs on regions at every size, at the plan's steps per
    // launch where those are six or more, else at 4.  It writes every
    // step's state, so that at the largest plans the writes bound it (elastic
    // FP32 16 shots of 1064x552: 188 MB, 40 us at 5 TB/s) and a wider ring costs
    // more than fewer reads give.  Measured (us per step, one launch of tiled
    // wavefronts per step, then regions of 2 / 3 / 4 / 5 steps): elastic FP32
    // 120x90 9.8, 3.9 / 3.2 / 2.8 / 2.6, 740x440 x 6 shots 41, 25 / 27 / 28 / 34,
    // 1064x552 x 16 shots 160, 140 / 121 / 138 / 164; FP64 64, 53 / 52 / 49 / 61 and 255,
    // 245 / 211 / 233 / 266; EM FP64 1064x808 x 2 shots 30, 22 / 21 / 20 / 22.
    p->tr_tm = p->tm > 5 ? p->tm : 4;
    const std::vector<int4> work = multi_work(p, p->tr_tm);
    int4* dw = nullptr;
    HIP_TRY(hipMalloc(&dw, sizeof(int4) * work.size()));
    if (hipMemcpy(dw, work.data(), sizeof(int4) * work.size(), hipMemcpyHostToDevice) != hipSuccess) {
      (void)hipFree(dw);
      return fail(SDT_EDEVICE, "hipMemcpy failed (work list)");
    }
    p->dtrwork = dw;
    p->ntrwork = (int)work.size();
  }
  if (!p->dadjwork) {
    // (shot, x0, z0, model) blocks of the fused adjoint kernel, shot by shot:
    // an XCD (item8) then works on one shot's states at a time, about 20 arrays
    // whose pages its translation caches hold.  Measured for 16 shots of 1064x552
    // elastic FP32 (us per step, blocks of 12 rows): 238, with the blocks of one
    // tile over all shots next to each other 283 (fewer coefficients and gradient
    // cells to fetch, but every array of 16 shots in use at once), shots in turn
    // dealt to all XCDs 245.
    const bool f32 = p->prec == SDT_FP32, em = p->kind == SDT_EM2;
    const int bw = em || p->split ? ElAdjOwn<float, true>::w : ElAdjOwn<float, false>::w;
    const int bh = em ? (f32 ? EmAdjOwn<float>::h : EmAdjOwn<double>::h)
                 : p->split ? (f32 ? ElAdjOwn<float, true>::h : ElAdjOwn<double, true>::h)
                            : (f32 ? ElAdjOwn<float, false>::h : ElAdjOwn<double, false>::h);
    std::vector<int4> work;
    for (int s = 0; s < p->nshots; ++s) {
      const int m = p->hshots[s].model;
      for (int z = 0; z < p->hmodels[m].nz; z += bh)
        for (int x = 0; x < p->hmodels[m].nx; x += bw) work.push_back(make_int4(s, x, z, m));
    }
    HIP_TRY(hipMalloc(&p->dadjwork, sizeof(int4) * work.size()));
    HIP_TRY(hipMemcpy(p->dadjwork, work.data(), sizeof(int4) * work.size(), hipMemcpyHostToDevice));
    p->nadjwork = (int)work.size();
  }

  return SDT_OK;
}

int sdt_plan_run_trail(void* plan, int it0, int nsteps, int buf, void* stream) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (!p->dadj) return fail(SDT_EINVAL, "call sdt_adjoint_setup first");
  if (buf < 0 || buf > 1 || !p->hadj[0].trail[buf]) return fail(SDT_EINVAL, "no such trail buffer");
  if (it0 < 0 || nsteps < 0 || (long long)it0 + nsteps > p->nt)
    return fail(SDT_EINVAL, "step range outside [0, nt)");
  for (const DAdj& a : p->hadj)
    if (nsteps + 1 > a.trail_len) return fail(SDT_EINVAL, "trail too short for nsteps + 1 states");
  hipStream_t st = static_cast<hipStream_t>(stream);
  p->last = st;
  if (nsteps == 0) return SDT_OK;
  hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p->dbase, it0);
  hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p->dtsel_trail, buf);
  if (nsteps < 2) {
    launch_trail(p, st, nsteps);
  } else {
    const int rc = replay_segment(p, 0, nsteps, st, [&](hipStream_t c) { launch_trail(p, c, nsteps); });
    if (rc) return rc;
  }
  HIP_TRY(hipGetLastError());
  return SDT_OK;
}

int sdt_adjoint_run(void* plan, int t_hi, int t_lo, int trail_t0, int buf, void* stream) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return fail(SDT_EINVAL, "plan is null");
  if (!p->dadj) return fail(SDT_EINVAL, "call sdt_adjoint_setup first");
  if (buf < 0 || buf > 1 || !p->hadj[0].trail[buf]) return fail(SDT_EINVAL, "no such trail buffer");
  if (t_lo < 0 || t_hi < t_lo || t_hi > p->nt || trail_t0 < 0 || trail_t0 > t_lo)
    return fail(SDT_EINVAL, "need 0 <= trail_t0 <= t_lo <= t_hi <= nt");
  for (const DAdj& a : p->hadj)
    if (t_hi - trail_t0 + 1 > a.trail_len)
      return fail(SDT_EINVAL, "trail does not hold the states up to t_hi");
  hipStream_t st = static_cast<hipStream_t>(stream);
  p->last = st;
  if (t_hi == t_lo) return SDT_OK;
  const int khi = t_hi - trail_t0, klo = t_lo - trail_t0;
  hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p->dtbase, trail_t0);
  hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p->dtsel_adj, buf);
  if (khi - klo < 2) {
    launch_adjoint(p, st, khi, klo);
  } else {
    const long long key = (long long)khi << 32 | (unsigned)klo;
    const int rc = replay_segment(p, 1, key, st, [&](hipStream_t c) { launch_adjoint(p, c, khi, klo); });
    if (rc) return rc;
  }
  HIP_TRY(hipGetLastError());
  return SDT_OK;
}

void sdt_plan_destroy(void* plan) {
  Plan* p = static_cast<Plan*>(plan);
  if (!p) return;
  (void)hipDeviceSynchronize();  // nothing of the plan may still be in flight
  if (p->gexec) (void)hipGraphExecDestroy(p->gexec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  if (p->cap) (void)hipStreamDestroy(p->cap);
  if (p->dmodels) (void)hipFree(p->dmodels);
  if (p->dshots) (void)hipFree(p->dshots);
  if (p->dwork) (void)hipFree(p->dwork);
  if (p->dwork2) (void)hipFree(p->dwork2);
  if (p->dwmulti) (void)hipFree(p->dwmulti);
  if (p->dit0) (void)hipFree(p->dit0);
  if (p->drec) (void)hipFree(p->drec);
  if (p->dflags) (void)hipFree(p->dflags);
  if (p->dbase) (void)hipFree(p->dbase);
  if (p->dnel) (void)hipFree(p->dnel);
  if (p->dnpsi) (void)hipFree(p->dnpsi);
  if (p->dadj) (void)hipFree(p->dadj);
  if (p->dadjwork) (void)hipFree(p->dadjwork);
  if (p->dtrwork) (void)hipFree(p->dtrwork);
  if (p->dtbase) (void)hipFree(p->dtbase);
  if (p->dtsel_trail) (void)hipFree(p->dtsel_trail);
  if (p->dtsel_adj) (void)hipFree(p->dtsel_adj);
  drop_adjoint_graphs(p);
  for (float* g : p->g32) (void)hipFree(g);
  if (p->dflush) (void)hipFree(p->dflush);
  delete p;
}

}  // extern "C"
