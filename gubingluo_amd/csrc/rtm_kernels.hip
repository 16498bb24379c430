// rtm_kernels.hip -- gfx950 kernels of the RTM hot path.
//
// One launch per time step.  A workgroup owns a tile of 64 columns (one
// wave64 row: every array is x-fastest, so a wave touches one contiguous
// 256-byte row segment) by TZ rows of one shot, and does the whole step for
// it: the velocity update (kernel.cu:430-500, 542-713 forward; 318-388
// reverse) of the tile and of the radius-10 halo that the pressure stencil
// reads, then the pressure update (kernel.cu:501-541, 714-1185 forward;
// 389-429 reverse) with source (kernel.cu:36-47), recording (48-71),
// receiver insertion (72-95), boundary strips (1186-1400) and imaging
// (1401-1416).  The halo velocities are computed again by the neighbouring
// tiles instead of being read back, so a step reads p, vx, vz once and
// writes them once per cell.  The model (1/rho and rho v^2) is read from one
// array shared by every shot of a launch (the resident model; clamped
// indices give each shot its padded window), which stays in the caches.  Fields have two time levels
// (step it reads level it&1 and writes level (it+1)&1), so a tile's reads of
// its neighbours' cells never race with their writes.
//
// LDS: the pressure of the tile and its halo (columns x0-20..x0+83 of the
// tile rows, rows z0-19..z0+TZ+18 of the tile columns), then -- reusing the
// same bytes -- the new velocities (vx: columns x0-12..x0+75; vz: rows
// z0-10..z0+TZ+8).  x-derivatives are taken four columns a lane from 16-byte
// LDS reads, z-derivatives from a register window of a lane's column.  In the
// reverse step a tile's receiver field and its source reconstruction are two
// workgroups; the reconstruction adds the imaging products of the step
// before, whose pressures both fields still read.
//
// Arithmetic follows the reference operation order with explicit fused
// multiply-adds (the oracle's canonical FP32 form), so every cell matches the
// CPU restatement bit for bit; the redundant halo velocities are the same
// operations on the same inputs.  Compiled with -ffp-contract=off; float
// division is IEEE as HIP compiles it.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <type_traits>

#include "rtm_dev.h"

#define NTHR 256   // threads of the auxiliary kernels

// Pointers read from the descriptor are generic to the compiler, which would
// then emit flat loads/stores (they count against the LDS wait counter too,
// so every LDS wait would also wait for outstanding memory loads).  All
// device-memory accesses go through these global-address-space views.
typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) int gint;
typedef __attribute__((address_space(1))) unsigned int guint;
typedef __attribute__((address_space(1))) unsigned short gushort;
#define GF(p) ((gfloat*)(p))
#define GCF(p) ((const gfloat*)(p))
// wave-uniform reads of arrays that no kernel writes while a step runs
// (damping, coefficients, wavelet, block scales): scalar loads
#define CCF(p) ((const __attribute__((address_space(4))) float*)(p))
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) f4 gf4;

namespace {

__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }

// The slot descriptor of a step kernel, read through the constant address
// space: no kernel writes a descriptor while a step runs (k_bump advances the
// time origin between launches), so its fields may come from scalar loads and
// be loaded again where needed.  A by-value copy instead has to stay live in
// scalar registers across the whole step (later stores could alias the
// source), which overflows them into vector lanes: about a thousand
// v_readlane reloads in the reverse step.
typedef __attribute__((address_space(4))) const ShotDev const_shot_t;
__device__ __forceinline__ const ShotDev& shot_of(const ShotDev* shots, int slot)
{
  return *(const ShotDev*)((const_shot_t*)shots + slot);
}

// The descriptor's cache lines, all fetched at once: its members are read a
// few at a time all along a step, and each line's first read would wait for
// memory by itself.
__device__ __forceinline__ void fetch_shot(const ShotDev* __restrict__ shots, int slot)
{
  typedef const __attribute__((address_space(4))) int const_int_t;
  constexpr int N = (sizeof(ShotDev) + 63) / 64;
  static_assert(N == 8, "one word of each line");
  const_int_t* p = (const_int_t*)((const_shot_t*)shots + slot);
  const int a = p[0], b = p[16], c = p[32], d = p[48], e = p[64], f = p[80], g = p[96], h = p[112];
  asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d), "s"(e), "s"(f), "s"(g), "s"(h));
}

// blockIdx -> tile: workgroups are dealt to the 8 XCDs round-robin, so give
// each XCD a contiguous run of the tile table (neighbouring tiles of one shot
// share their halos through that XCD's L2).
__device__ __forceinline__ int xcd_tile(int ntiles)
{
  const int per = gridDim.x >> 3;          // launched as a multiple of 8
  const int b = blockIdx.x;
  const int t = (b & 7) * per + (b >> 3);
  return t < ntiles ? t : -1;
}

// ---------------------------------------------------------------- strips --
// store offset of a vx strip cell (kernel.cu:1186-1293 packing), -1 off the
// strip (the halo columns of a reconstruction tile)
__device__ __forceinline__ int strip_vx(const ShotDev& s, int iz, int ix)
{
  if (iz < s.npml || iz >= s.nzp - s.npml) return -1;
  const int r = iz - s.npml;
  if (ix >= s.npml - RTM_R && ix < s.npml) return r * RTM_R + ix - (s.npml - RTM_R);
  const int c0 = s.nxp - s.npml - 1;
  if (ix >= c0 && ix < c0 + RTM_R) return RTM_R * s.nzi + r * RTM_R + ix - c0;
  return -1;
}
// The offsets of the other blocks split into a row part and a column part.
// column part of the p lr block, -1 off its columns
__device__ __forceinline__ int strip_col_plr(const ShotDev& s, int ix)
{
  const int n = s.npml, blr = 2 * RTM_R * s.nzi + 2 * RTM_R * s.nxl;
  if (ix >= n - RTM_R && ix < n) return blr + ix - (n - RTM_R);
  if (ix >= s.nxp - n && ix < s.nxp - n + RTM_R) return blr + RTM_R * s.nzi + ix - (s.nxp - n);
  return -1;
}
// row part of the vz block offset (rows n-10..n-1 and nzp-n-1..nzp-n+8), -1
__device__ __forceinline__ int strip_row_vz(const ShotDev& s, int iz)
{
  const int n = s.npml, b = 2 * RTM_R * s.nzi;
  if (iz >= n - RTM_R && iz < n) return b + (iz - (n - RTM_R)) * s.nxl;
  const int r0 = s.nzp - n - 1;
  if (iz >= r0 && iz < r0 + RTM_R) return b + RTM_R * s.nxl + (iz - r0) * s.nxl;
  return -1;
}
// row part of the lr blocks (rows n..nzp-n-1), -1
__device__ __forceinline__ int strip_row_lr(const ShotDev& s, int iz)
{
  return (iz >= s.npml && iz < s.nzp - s.npml) ? (iz - s.npml) * RTM_R : -1;
}
// row part of the p tb block (rows n-10..n-1 and nzp-n..nzp-n+9), -1
__device__ __forceinline__ int strip_row_ptb(const ShotDev& s, int iz)
{
  const int n = s.npml, b = 4 * RTM_R * s.nzi + 2 * RTM_R * s.nxl;
  if (iz >= n - RTM_R && iz < n) return b + (iz - (n - RTM_R)) * s.nxl;
  const int r0 = s.nzp - n;
  if (iz >= r0 && iz < r0 + RTM_R) return b + RTM_R * s.nxl + (iz - r0) * s.nxl;
  return -1;
}
// after the nt x 4 scales: the wavefield guard word (k_guard), then the
// largest |value| of the four strip blocks (16-bit store) of even and of odd
// steps, as float bits
__device__ __forceinline__ unsigned int* guard_word(const ShotDev& s) { return (unsigned int*)(s.sscale + (size_t)s.nt * 4); }
__device__ __forceinline__ unsigned int* strip_max(const ShotDev& s, int it) { return guard_word(s) + 4 + 4 * (it & 1); }

// ------------------------------------------------------------ tile shape --
// G waves of 64 lanes; each thread owns RPT consecutive rows of one column.
template <int G_, int RPT_, bool CACHED, bool S16_>
struct Geo {
  static constexpr int G = G_, RPT = RPT_;
  static constexpr bool S16 = S16_;                    // the boundary store is 16-bit
  static constexpr int ST = CACHED ? 0 : 2;            // cache policy of the field stores (bst)
  static constexpr int TZ = G * RPT;                   // tile rows
  static constexpr int SPLIT = TZ < 16 ? 16 / TZ : 1;  // workgroups that share a tile of the table (16 rows or more)
  static constexpr int NT = 64 * G;                    // threads
  static constexpr int PW = 108;                       // p row: column x at float x - x0 + 21 (x0-20..x0+83 held):
                                                       // a quad's window x-9..x+14 starts on 16 bytes
  static constexpr int VXW = 88;                       // vx row: columns x0-12 .. x0+75
  static constexpr int ZR = TZ + 19;                   // vz rows z0-10 .. z0+TZ+8
  static constexpr int KZ = (ZR + G - 1) / G;          // vz rows per wave (consecutive)
  static constexpr int PZR = G * KZ + 19;              // p rows held (>= TZ + 38; the last
                                                       // wave's window may run past TZ+38)
  static constexpr int KQ = (RPT * 22 + 63) / 64;      // vx quads per lane (16 own and 6 halo quads a row)
  static constexpr int KO = (RPT * 16 + 63) / 64;      // own quads per lane
  static constexpr int LDS_A = PZR * PW;               // p rows z0-19..
  static constexpr int LDS_B = 4 + TZ * VXW + ZR * 64; // new vx | new vz
  static constexpr int LDS = LDS_A > LDS_B ? LDS_A : LDS_B;
  static constexpr int LDS_D = 2 * VXW + 128 + 2 * TZ; // damping factors (after LDS): of vx at columns x0-12..x0+75,
                                                       // of p at the tile's columns and rows
  static_assert(RPT == 2 || RPT % 4 == 0, "own quads fill whole waves, or half of one");
};

// ------------------------------------------------------- buffer access --
// Every field of a slot is one allocation of frows x pitch floats.  Tile
// accesses are raw buffer loads / stores with the row offset in a scalar
// register and the lane's column offset in a vector register, so the
// addressing costs no vector instructions per access.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t field_rsrc(const float* f00, const ShotDev& s)
{
  return __builtin_amdgcn_make_buffer_rsrc((void*)(f00 - s.forg), (short)0, s.frows * s.pitch * 4, 0x00020000);
}
// imaging accumulators: nzi x nxl, pitch nxl, addressed from interior cell (0,0)
__device__ __forceinline__ rsrc_t image_rsrc(float* a, const ShotDev& s)
{
  return __builtin_amdgcn_make_buffer_rsrc((void*)a, (short)0, s.nzi * s.nxl * 4, 0x00020000);
}
// the model a slot reads (mzn rows of mpitch floats)
__device__ __forceinline__ rsrc_t model_rsrc(const float* m, const ShotDev& s)
{
  return __builtin_amdgcn_make_buffer_rsrc((void*)m, (short)0, s.mzn * s.mpitch * 4, 0x00020000);
}
// byte offsets into the model of padded row iz (wave-uniform) and column ix:
// the window cut with edge replication (extractvel1 + extendvel1,
// Velocity_function.cpp:2011-2073) as a clamp
__device__ __forceinline__ int model_row(const ShotDev& s, int iz)
{
  return imin(imax(iz - s.mz0, 0), s.mzn - 1) * s.mpitch * 4;
}
__device__ __forceinline__ int model_col(const ShotDev& s, int ix)
{
  return (s.mx0 + imin(imax(ix - s.mxs, 0), s.mxn - 1)) * 4;
}
// A load offset past any buffer's end: a buffer load whose lane offset is
// out of range returns 0 for that lane without fetching memory (the same
// holds for the loads that write LDS).  Field cells outside the grid's
// columns -- the margins, and the lanes of a window's last tile column past
// nxp-1 -- are never written and hold 0, so their loads take this offset:
// same values, and the part of the last tile column's lines past the window
// is not fetched.
#define RTM_OOB ((int)0x80000000)
__device__ __forceinline__ int col_load(int voff, int col, int nxp)
{
  return (unsigned)col < (unsigned)nxp ? voff : (voff | RTM_OOB);
}
// a lane's offset, or the out-of-range one where the lane takes no part:
// its load returns 0 and its store is dropped, with no exec-mask branch
__device__ __forceinline__ int pred_off(int voff, bool on) { return on ? voff : (voff | RTM_OOB); }
__device__ __forceinline__ float bld(rsrc_t r, int voff, int soff)
{
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
// Cache policy ST of the field stores: 2 is the non-temporal hint ("nt" on
// gfx950), 0 an ordinary store.  A value written in one step is next read in
// the following step.  Where the launches in flight work on more than the
// 256 MB Infinity Cache holds, it is gone by then, and the hint keeps the
// stores from pushing out lines that neighbouring tiles still read; where
// they work on less, an ordinary store leaves the value there for the next
// step.  Survey shots, us per reverse step, nt against ordinary: 64 shots
// (0.9 GB) 268 / 277, 32 shots 139 / 143, 16 shots (220 MB) 75 / 68, 8 shots
// 44 / 36, 4 shots 26 / 23.  rtm_launch.h's `cached` says which.
template <int ST>
__device__ __forceinline__ void bst(rsrc_t r, float v, int voff, int soff)
{
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, voff, soff, ST);
}
__device__ __forceinline__ f4 bld4(rsrc_t r, int voff, int soff)
{
  return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
template <int ST>
__device__ __forceinline__ void bst4(rsrc_t r, f4 v, int voff, int soff)
{
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, voff, soff, ST);
}
// The boundary strips of step `it` as a buffer.  It starts 16 bytes before the
// record and ends 16 after it (both inside the slot): a quad that holds the
// first or last columns of a strip loads four values at the strip's own
// offsets, of which the ones past the strip are not used.
template <bool S16>
__device__ __forceinline__ rsrc_t strip_rsrc(const ShotDev& s, int it)
{
  constexpr int es = S16 ? 2 : 4;
  return __builtin_amdgcn_make_buffer_rsrc((char*)s.store + (long long)it * s.strip_len * es - 16, (short)0,
                                           (int)s.strip_len * es + 32, 0x00020000);
}
// raw stored values (the fp32 value, or the 16-bit code in the low bits) at
// offset off (a row offset row and a lane's col), and the value of one with
// the scale of its block and step
template <bool S16>
__device__ __forceinline__ float strip1(rsrc_t r, int col, int row, bool on)
{
  if (!S16) return bld(r, pred_off(col * 4 + 16, on), row * 4);
  return __uint_as_float((unsigned int)__builtin_amdgcn_raw_buffer_load_b16(r, pred_off(col * 2 + 16, on), row * 2, 0));
}
template <bool S16>
__device__ __forceinline__ f4 strip4(rsrc_t r, int off, bool on)
{
  if (!S16) return bld4(r, pred_off(off * 4 + 16, on), 0);
  return f4{strip1<S16>(r, off, 0, on), strip1<S16>(r, off + 1, 0, on), strip1<S16>(r, off + 2, 0, on),
            strip1<S16>(r, off + 3, 0, on)};
}
template <bool S16>
__device__ __forceinline__ float strip_value(const ShotDev& s, float sc, float raw)
{
  if (!S16) return raw;
  const unsigned int h = __float_as_uint(raw);
  const float f = __half2float(__ushort_as_half((unsigned short)h)), b = __uint_as_float(h << 16);
  return (s.store_fmt == ST_F16 ? f : b) * sc;
}

// load one dword per lane into LDS: lane i writes lds_row[i] (lds_row is
// wave-uniform)
typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void bld_lds(rsrc_t r, float* lds_row, int voff, int soff)
{
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds_row, 4, voff, soff, 0, 0);
}

// true for every lane of the wave if any active lane has c: branches on it
// are uniform, so the rare cases (reduced radius near the grid edge, damped
// cells) cost their instructions only in the waves that hold them
__device__ __forceinline__ bool any_lane(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }

// keeps the instructions of one part of a step from being moved into another:
// left free, the scheduler fetches the operands of every part first and needs
// 256 registers for them
__device__ __forceinline__ void part() { __builtin_amdgcn_sched_barrier(0); }

// the value is computed here: a result that is first used in a later part
// would otherwise be computed there, and its whole window held until then
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }

// lane k's value (k < 64 known at compile time) as a scalar
__device__ __forceinline__ float lane_value(float v, int k)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// sum of the staggered differences w[h + i] - w[h + 1 - i], i = 1..10, as the
// reference loops (kernel.cu:459-460), one fused multiply-add a tap
template <class W, class Cf>
__device__ __forceinline__ float taps(const W& w, int h, const Cf& c)
{
  float acc = 0.0f;
#pragma unroll
  for (int i = 1; i <= RTM_R; i++) acc = __builtin_fmaf(c[i - 1], w[h + i] - w[h + 1 - i], acc);
  return acc;
}
// The same with the coefficient row of order 2 r from the LDS table (rows of
// CTW floats, zero beyond their order): a reduced-radius cell runs the same
// ten steps with its own row and no predicate, the extra steps add
// 0*(a-b) = +-0, which leaves the sum unchanged (the operands past the radius
// are finite cells of the staged halo or the zero margins), and row 9 gives
// the radius-10 sum bit for bit.
constexpr int CTW = 12;
struct CoefRow {
  f4 a, b;
  f2 d;
  __device__ __forceinline__ CoefRow(const float* ctab, int r)
  {
    const f4* cr = (const f4*)(ctab + (r - 1) * CTW);
    a = cr[0];
    b = cr[1];
    d = *(const f2*)(cr + 2);
  }
};
template <class W>
__device__ __forceinline__ float taps_r(const W& w, int h, const CoefRow& r)
{
  const float c[RTM_R] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w, r.d.x, r.d.y};
  // (the difference as -(b - a), the same value: the compiler would hoist the
  // differences it shares with the full-radius branch and hold them)
  float acc = 0.0f;
#pragma unroll
  for (int i = 1; i <= RTM_R; i++) acc = __builtin_fmaf(c[i - 1], -(w[h + 1 - i] - w[h + i]), acc);
  return acc;
}
template <class W>
__device__ __forceinline__ float taps_r(const W& w, int h, const float* ctab, int r)
{
  return taps_r(w, h, CoefRow(ctab, r));
}
// entry t of that table
__device__ __forceinline__ float ctab_entry(const ShotDev& s, int t)
{
  const int r = t / CTW, i = t - r * CTW;
  return i <= r && i < RTM_R ? GCF(s.coef)[r * RTM_R + i] : 0.0f;
}

// field kinds of one pass
enum : int { FK_SRC = 0, FK_RCV = 1, FK_RCN = 2 };
// tile classes: interior (no damping, no strips), general (absorbing layer or
// strips), edge (general with cells of reduced radius)
enum : int { TC_IN = 0, TC_GEN = 1, TC_EDGE = 2 };

// One field through one time step on a tile: p of the current level pc (with
// velocities vxc, vzc) to the next level (pn, vxn, vzn).  A reconstruction
// pass with `img` also adds the imaging products of the PREVIOUS reverse step,
// of the pressure levels both fields read (pr: the receiver field's), so that
// the two fields of a reverse step need not wait for each other.
//
// What bounds it: instruction issue and the chain of a workgroup's phases,
// then HBM.  So the classes are compiled apart (straight-line code; one body
// with per-cell tests issued three instructions for each stencil operation),
// and everything but the z-differences is mapped to quads of four columns:
//   p staging   rows g + G m of the tile (LDS-writing loads, no registers)
//   z-derivatives (columns): lane = column, a wave takes consecutive rows and
//               reads their window of rows once; row offsets, the damping of a
//               row and its radius are wave-uniform (scalar registers)
//   x-derivatives (quads): a wave's own RPT rows as 16 quads of a row and the
//               6 quads of its halo columns x0-12.., x0+64..; a quad reads its
//               window of 24 values as six 16-byte LDS loads instead of 20
//               loads per cell, and its operands and results move as 16-byte
//               accesses (a quarter of the memory instructions)
// The rows of the new vx are written and read by the same wave, so only the
// new vz crosses waves (one exchange), and the z-differences reach the quads
// through the wave's own vx rows once those are consumed.
// A forward step keeps its own boundary strips (`save`): it writes them to the
// fp32 store from the registers that hold them, or takes the largest |value|
// of each 16-bit block for k_quant16, which scales and stores them.  Only tiles
// that hold strip cells (TF_SAVE) have the code run.  A launch of its own that
// read the strips back from the new fields cost 2.4 us a step on a 480 x 280
// shot (11.6 -> 9.1 us), 15.7 us on three survey shots in turn (43.9 ->
// 28.1), 3.7 of 79 us on 48 of them.
template <class Q, int FK, int TC>
__device__ __forceinline__ void tile_step(float* __restrict__ lds, const float* __restrict__ ctab, const ShotDev& s,
                                          const Tile& tl, int it, const float* pc, const float* vxc, const float* vzc,
                                          float* pn, float* vxn, float* vzn, const float* pr, bool img, bool save_,
                                          unsigned char* actw)
{
  constexpr int G = Q::G, RPT = Q::RPT, TZ = Q::TZ, KZ = Q::KZ, PW = Q::PW, VXW = Q::VXW, ZR = Q::ZR;
  constexpr int KQ = Q::KQ, KO = Q::KO;
  constexpr bool S16 = Q::S16;
  constexpr bool RCN = FK == FK_RCN, GEN = TC != TC_IN, EDGE = TC == TC_EDGE;
  // the OR of the bit patterns of the lane's stored field values (-0 counts
  // as non-zero): written to actw[wave] at the end for the zero-tile skip
  unsigned int nzb = 0u;
  float* PS = lds;                                     // p rows z0-19.., columns x0-20..x0+83 from float 1 of a row
  float* DMP = lds + Q::LDS;                           // a, b of vx at columns x0-12.. (88 each)
  float* DPX = DMP + 2 * VXW;                          // a, b of p at the tile's columns (64 each)
  float* DPZ = DPX + 128;                              // a, b of p at the tile's rows
  float* VXL = lds + 4;                                // (after the pressure is consumed) column x at x - x0 + 10
  float* VZL = lds + 4 + TZ * VXW;                     // new vz rows z0-10.., 64 columns
  const int lane = threadIdx.x & 63;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x0 = tl.x0, z0 = tl.z0, nxp = s.nxp, nzp = s.nzp, npml = s.npml;
  const int ix = x0 + lane;                            // the lane's column (column mapping)
  const int zw = z0 + g * RPT;                         // the wave's first own row
  const bool strips = RCN && GEN && (tl.kind & TF_STRIP) != 0;
  const bool save = FK == FK_SRC && GEN && save_ && (tl.kind & TF_SAVE);
  float smax[4] = {0.0f, 0.0f, 0.0f, 0.0f};            // (16-bit store) largest |value| of the strip blocks
  // a strip value of block b at offset off, where `on`: no branch per lane
  auto put = [&](rsrc_t r, int b, int off, float v, bool on) {
    if (!S16) bst<2>(r, v, pred_off(off * 4 + 16, on), 0);
    else smax[b] = fmaxf(smax[b], on ? fabsf(v) : 0.0f);
  };
  const int pr4 = s.pitch * 4;
  const int srow0 = (z0 + RTM_MZT) * pr4;              // byte offset of tile row 0
  const int vcol = (ix + RTM_MXL) * 4;                 // byte offset of the lane's column
  const int vld = GEN ? col_load(vcol, ix, nxp) : vcol;
  const rsrc_t Rp = field_rsrc(pc, s), Rvx = field_rsrc(vxc, s), Rvz = field_rsrc(vzc, s);
  const rsrc_t Rib = model_rsrc(s.mib, s), Rkk = model_rsrc(s.mkk, s);
  const float dtx = s.dtx, dtz = s.dtz;
  // (per-lane conditions are combined with & and |: a short-circuit operator
  // would branch on the lanes)
  auto inner_row = [&](int z) { return (unsigned)(z - npml) < (unsigned)(nzp - 2 * npml); };
  auto inner_col = [&](int x) { return (unsigned)(x - npml) < (unsigned)(nxp - 2 * npml); };
  // the strips' columns beside the interior: vx and p left, vx right, p right
  // (kernel.cu:1186-1293), and whether the tile's own and halo quads reach them
  auto left = [&](int x) { return (unsigned)(x - npml + RTM_R) < (unsigned)RTM_R; };
  auto rightv = [&](int x) { return (unsigned)(x - nxp + npml + 1) < (unsigned)RTM_R; };
  auto rightp = [&](int x) { return (unsigned)(x - nxp + npml) < (unsigned)RTM_R; };
  const bool hasL = x0 - 12 < npml && x0 + 75 >= npml - RTM_R;
  const bool hasR = x0 - 12 < nxp - npml + RTM_R && x0 + 75 >= nxp - npml - 1;
  const int blr = 2 * RTM_R * (s.nzi + s.nxl);         // the p lr block
  // rows of the wave that hold cells of this pass (a partial last tile row,
  // the absorbing rows beyond the reconstruction's strips)
  const bool live = !GEN || (RCN ? zw + RPT > npml - RTM_R && zw < nzp - npml + RTM_R : zw < nzp);
  // columns near the left or right edge; columns that no window edge clamps
  const bool edge_x = EDGE && (x0 - 12 <= 9 || x0 + 75 >= nxp - 10);
  const bool mfree = !GEN || (x0 - 12 >= s.mxs && x0 + 76 <= s.mxs + s.mxn);
  const bool inner_cols = !GEN || (x0 >= npml && x0 + 64 <= nxp - npml);
  // ---- 1. the pressure and its halo into LDS (buffer loads with the lds
  //         modifier: lane i of a wave writes its dword to base + 4 i): tile
  //         rows as two full-wave loads (x0-20..x0+43, x0+20..x0+83; the
  //         middle 24 columns arrive twice with the same values), halo rows
  //         the tile's columns; old vz and its 1/rho into registers
  {
    int ca = (x0 - 20 + lane + RTM_MXL) * 4, cb = (x0 + 20 + lane + RTM_MXL) * 4;
    if (GEN) {
      ca = col_load(ca, x0 - 20 + lane, nxp);
      cb = col_load(cb, x0 + 20 + lane, nxp);
    }
    const int sw = srow0 + g * RPT * pr4;
#pragma unroll
    for (int m = 0; m < RPT; m++) {
      bld_lds(Rp, PS + (g * RPT + m + 19) * PW + 1, ca, sw + m * pr4);
      bld_lds(Rp, PS + (g * RPT + m + 19) * PW + 41, cb, sw + m * pr4);
    }
#pragma unroll
    for (int m = 0; m < (38 + G - 1) / G; m++) {       // 19 rows above the tile, 19 below
      const int h = g + G * m;
      if (G * (m + 1) <= 38 || h < 38) {
        const int k = h < 19 ? h : h + TZ;
        bld_lds(Rp, PS + k * PW + 21, vld, srow0 + (k - 19) * pr4);
      }
    }
  }
  part();                                              // (nothing waits before these loads are on their way)
  float c10[RTM_R];
#pragma unroll
  for (int i = 0; i < RTM_R; i++) c10[i] = CCF(s.coef)[90 + i];
  // rows of the z phase that exist for every wave need no test
  auto zrow = [&](int k) { return k < ZR - (G - 1) * KZ || g * KZ + k < ZR; };
  const int mcol = model_col(s, ix);
  const bool zcol = inner_col(ix);                     // interior columns
  float vzo[KZ], ibz[KZ];
#pragma unroll
  for (int k = 0; k < KZ; k++) {
    const int kz = g * KZ + k, iz = z0 - 10 + kz;
    vzo[k] = 0.0f;
    ibz[k] = 1.0f;
    if (zrow(k)) {
      vzo[k] = bld(Rvz, vld, srow0 + (kz - 10) * pr4);
      if (strips) {                                    // a strip row: the stored value of step it+1 (raw)
        const int st = strip_row_vz(s, iz);
        if (st >= 0) vzo[k] = strip1<S16>(strip_rsrc<S16>(s, it + 1), ix - npml, st, zcol);
      }
      ibz[k] = bld(Rib, mcol, GEN ? model_row(s, iz) : (iz - s.mz0) * s.mpitch * 4);
    }
  }
  // quads of the x phase.  Own quads: lane n of quad round k has row
  // n / 16 + 4 k, columns 4 (n % 16), so that the rounds differ by a scalar
  // row offset.  The last round holds the halo quads, 6 a row (two rows a
  // wave: in the lanes past the 32 own quads)
  const bool oq = RPT >= 4 || lane < 32;               // the lane has own quads
  const int hn = RPT >= 4 ? lane : lane - 32;          // its halo quad
  const bool hon = hn >= 0 && hn < RPT * 6;
  const int hr = hn / 6, hq = hn - hr * 6;
  const int hcol = hq < 3 ? -12 + 4 * hq : 52 + 4 * hq;
  const int orow = RPT >= 4 ? lane >> 4 : (oq ? lane >> 4 : (hon ? hr : 0));
  const int ocol = RPT >= 4 ? 4 * (lane & 15) : (oq ? 4 * (lane & 15) : (hon ? hcol : 0));
  const int xrow = hon ? hr : 0, xcol = hon ? hcol : 0;   // the halo round's (RPT >= 4)
  const int ooff = ((zw + orow + RTM_MZT) * s.pitch + x0 + ocol + RTM_MXL) * 4;
  const int xoff = ((zw + xrow + RTM_MZT) * s.pitch + x0 + xcol + RTM_MXL) * 4;
  auto qrow = [&](int k) { return k < KO ? orow + 4 * k : xrow; };
  auto qcol = [&](int k) { return k < KO ? ocol : xcol; };
  auto qx = [&](int k) { return x0 + qcol(k); };       // first column of a quad
  auto qsoff = [&](int k) { return k < KO ? 4 * k * pr4 : 0; };
  // load offset of a quad: quads off the grid's columns fetch nothing
  const int old_ = GEN ? pred_off(ooff, (unsigned)(x0 + ocol) < (unsigned)nxp) : ooff;
  const int xld_ = GEN ? pred_off(xoff, (unsigned)(x0 + xcol) < (unsigned)nxp) : xoff;
  auto qld = [&](int k) { return k < KO ? old_ : xld_; };
  if (!RCN && GEN) {                                   // vx damping of the columns x0-12..x0+75
    for (int t = threadIdx.x; t < 22; t += 64 * G) {
      ((f4*)DMP)[t] = *(const gf4*)(GCF(s.axv) + x0 - 12 + 4 * t);
      ((f4*)DMP)[22 + t] = *(const gf4*)(GCF(s.bxv) + x0 - 12 + 4 * t);
    }
    for (int t = threadIdx.x; t < 128 + 2 * TZ; t += 64 * G) {
      const gfloat* src = t < 64 ? GCF(s.ax) + x0 : t < 128 ? GCF(s.bx) + x0 - 64
                         : t < 128 + TZ ? GCF(s.az) + z0 - 128 : GCF(s.bz) + z0 - 128 - TZ;
      DPX[t] = src[t];
    }
  }
  // (damping of the wave's vz rows: lane k holds row k's, so that a row reads
  // it as a scalar with no memory access)
  float azl = 1.0f, bzl = 0.0f;
  if (!RCN && GEN) {
    const int r = z0 - 10 + imin(g * KZ + lane, ZR - 1);
    azl = GCF(s.azv)[r];
    bzl = GCF(s.bzv)[r];
  }
  __builtin_amdgcn_s_waitcnt(0);                       // the LDS writes of the staging loads
  __syncthreads();                                     // p staged

  // operands of the x phase: they arrive while the z phase computes.  Four
  // model values of a quad: one 16-byte load where no column is clamped
  auto model4 = [&](rsrc_t r, int k) -> f4 {
    if (!GEN) {
      const int o = ((zw + (k < KO ? orow : xrow) - s.mz0) * s.mpitch + s.mx0 + qx(k) - s.mxs) * 4;
      return bld4(r, o, k < KO ? 16 * k * s.mpitch : 0);
    }
    const int ro = model_row(s, zw + qrow(k)), x = qx(k);
    if (mfree) return bld4(r, ro + (s.mx0 + x - s.mxs) * 4, 0);
    return f4{bld(r, ro + model_col(s, x), 0), bld(r, ro + model_col(s, x + 1), 0), bld(r, ro + model_col(s, x + 2), 0),
              bld(r, ro + model_col(s, x + 3), 0)};
  };
  f4 vxo[KQ], ibx[KQ], sxr[KQ];                        // (sxr: stored vx of a quad's strip cells, raw)
  float scv[4] = {1.0f, 1.0f, 1.0f, 1.0f};             // 16-bit block scales: vx, vz of step it+1, p-lr, p-tb of step it
  if (live) {
#pragma unroll
    for (int k = 0; k < KQ; k++) {
      vxo[k] = bld4(Rvx, qld(k), qsoff(k));
      ibx[k] = model4(Rib, k);
    }
    if (strips) {
      if (S16)
#pragma unroll
        for (int b = 0; b < 4; b++) scv[b] = CCF(s.sscale)[(long long)(b < 2 ? it + 1 : it) * 4 + b];
      const rsrc_t R = strip_rsrc<S16>(s, it + 1);
#pragma unroll
      for (int k = 0; k < KQ; k++) {
        const int x = qx(k), r = zw + qrow(k) - npml;
        const bool in = inner_row(zw + qrow(k));
        sxr[k] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (hasL) sxr[k] = strip4<S16>(R, r * RTM_R + x - npml + RTM_R, in & (x + 3 >= npml - RTM_R) & (x < npml));
        if (hasR) {
          const f4 u = strip4<S16>(R, RTM_R * s.nzi + r * RTM_R + x - nxp + npml + 1,
                              in & (x + 3 >= nxp - npml - 1) & (x < nxp - npml - 1 + RTM_R));
          if (!hasL) sxr[k] = u;
          else                                         // a window narrower than the tile
#pragma unroll
            for (int c = 0; c < 4; c++) sxr[k][c] = rightv(x + c) ? u[c] : sxr[k][c];
        }
      }
    }
  }

  part();
  // ---- 2. new vz (rows z0-10 + g KZ + k of the lane's column).  Forward
  //         fields: v = (c1*v - u)/c2, u = (sum * dt/h) / rho
  //         (kernel.cu:588-594) as u = (s*dt/h)*ib, v = fma(a, v, -(u*b)) with
  //         a = c1/c2, b = 1/c2 (off the layer v - u, kernel.cu:462), radius
  //         min(10, distance to the grid edge) (cuda_norderx/z,
  //         kernel.cu:299-317); off the grid b = 0, so the value stays +0.
  //         Reconstruction: v + u as fma(s*dt/h, ib, v) (kernel.cu:318-388),
  //         stored strip values (kernel.cu:1294-1347), 0 elsewhere
  float vzn_[KZ];
  const float scz = S16 && strips ? CCF(s.sscale)[(long long)(it + 1) * 4 + 1] : 1.0f;
  {
    float cw[KZ + 19];                                 // p rows z0-19 + g KZ + m of the column
#pragma unroll
    for (int m = 0; m < KZ + 19; m++) cw[m] = PS[(g * KZ + m) * PW + 21 + lane];
#pragma unroll
    for (int k = 0; k < KZ; k++) {
      if (k % 3 == 0) part();
      vzn_[k] = 0.0f;
      if (zrow(k)) {
        const int kz = g * KZ + k, iz = z0 - 10 + kz;  // wave-uniform
        if (RCN) {
          if (!GEN) {
            vzn_[k] = __builtin_fmaf(taps(cw, k + 9, c10) * dtz, ibz[k], vzo[k]);
          } else {
            // every row is computed and then selected, with no branch
            const float v = __builtin_fmaf(taps(cw, k + 9, c10) * dtz, ibz[k], vzo[k]);
            vzn_[k] = zcol & (iz >= npml) & (iz <= nzp - npml - 2) ? v : 0.0f;
            if (strips) vzn_[k] = zcol & (strip_row_vz(s, iz) >= 0) ? strip_value<S16>(s, scz, vzo[k]) : vzn_[k];
          }
        } else if (!EDGE || (iz >= 0 && iz <= nzp - 2)) {   // (rows off the grid stay +0)
          float sum;
          if (EDGE) {
            const int rad = imin(RTM_R, imin(iz + 1, nzp - 1 - iz));
            sum = rad == RTM_R ? taps(cw, k + 9, c10) : taps_r(cw, k + 9, ctab, rad);
          } else {
            sum = taps(cw, k + 9, c10);
          }
          const float u = (sum * dtz) * ibz[k];
          vzn_[k] = GEN ? __builtin_fmaf(lane_value(azl, k), vzo[k], -(u * lane_value(bzl, k))) : vzo[k] - u;
        }
      }
      pin(vzn_[k]);
    }
  }

  // ---- 3. new vx of the own and the halo quads; the quad's own pressure is
  //         in its window
  f4 hv[KQ], po[KO];
  if (live) {
  if (S16 && strips)
#pragma unroll
    for (int k = 0; k < KQ; k++)
#pragma unroll
      for (int c = 0; c < 4; c++) sxr[k][c] = strip_value<S16>(s, scv[0], sxr[k][c]);
#pragma unroll
  for (int k = 0; k < KQ; k++) {
    part();
    float w[24];                                       // p at columns x-9 .. x+14
    const f4* row = (const f4*)(PS + (g * RPT + qrow(k) + 19) * PW + qcol(k) + 12);
#pragma unroll
    for (int m = 0; m < 6; m++) {
      const f4 v = row[m];
      w[4 * m] = v.x; w[4 * m + 1] = v.y; w[4 * m + 2] = v.z; w[4 * m + 3] = v.w;
    }
    if (k < KO) po[k < KO ? k : 0] = f4{w[9], w[10], w[11], w[12]};
    f4 av, bv;
    if (!RCN && GEN) {
      av = *(const f4*)(DMP + qcol(k) + 12);
      bv = *(const f4*)(DMP + VXW + qcol(k) + 12);
    }
    int rad[4] = {RTM_R, RTM_R, RTM_R, RTM_R};
    bool red = false;
    if (edge_x && !RCN) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int x = qx(k) + c;
        if ((unsigned)x <= (unsigned)(nxp - 2)) rad[c] = imin(RTM_R, imin(x + 1, nxp - 1 - x));
        red = red | (rad[c] != RTM_R);
      }
      red = any_lane(red);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      float sum;
      if (EDGE && !RCN && red) sum = taps_r(w, 9 + c, ctab, rad[c]);
      else sum = taps(w, 9 + c, c10);
      if (RCN) {
        float v = __builtin_fmaf(sum * dtx, ibx[k][c], vxo[k][c]);
        if (GEN) {
          const int x = qx(k) + c;
          const bool in = inner_row(zw + qrow(k));
          v = in & (x >= npml) & (x <= nxp - npml - 2) ? v : 0.0f;
          if (strips) v = in & (left(x) | rightv(x)) ? sxr[k][c] : v;
        }
        hv[k][c] = v;
      } else {
        const float u = (sum * dtx) * ibx[k][c];
        hv[k][c] = GEN ? __builtin_fmaf(av[c], vxo[k][c], -(u * bv[c])) : vxo[k][c] - u;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
      float v = hv[k][c];
      pin(v);
      hv[k][c] = v;
    }
    if (k < KO) {                                      // own quads to memory
      const bool on = oq & (!GEN | ((qx(k) < nxp) & (zw + qrow(k) < nzp)));
      bst4<Q::ST>(field_rsrc(vxn, s), hv[k], pred_off(ooff, on), qsoff(k));
      if (oq)
#pragma unroll
        for (int c = 0; c < 4; c++) nzb |= __float_as_uint(hv[k][c]);
      if (save) {
        const rsrc_t R = strip_rsrc<S16>(s, it);
        const int x = qx(k), r = zw + qrow(k) - npml;
        const bool in = oq & inner_row(zw + qrow(k));
        if (hasL)
#pragma unroll
          for (int c = 0; c < 4; c++) put(R, 0, r * RTM_R + x + c - npml + RTM_R, hv[k][c], in & left(x + c));
        if (hasR)
#pragma unroll
          for (int c = 0; c < 4; c++)
            put(R, 0, RTM_R * s.nzi + r * RTM_R + x + c - nxp + npml + 1, hv[k][c], in & rightv(x + c));
      }
    }
  }
  }
  part();
  // operands of the pressure phase, fetched now so that the round trip
  // overlaps the exchange and the differences below: rho v^2 of the own quads, and the PML split pair
  // (forward-type passes, quads with a damped cell) or, in the
  // reconstruction, the imaging accumulators and the receiver pressure
  f4 kk[KO], qa[KO], qb[KO], qc[KO], spr[KO];          // (spr: stored p of a quad's strip cells, raw)
  // split cells: the absorbing layer within the ring
  auto split = [&](int z, int x) {
    return ((unsigned)(z - 1) < (unsigned)(nzp - 2)) & ((unsigned)(x - 1) < (unsigned)(nxp - 2)) &
           !(inner_row(z) & inner_col(x));
  };
  auto split_q = [&](int z, int x) { return oq & (split(z, x) | split(z, x + 1) | split(z, x + 2) | split(z, x + 3)); };
  if (live) {
#pragma unroll
    for (int h = 0; h < KO; h++) {
      const int z = zw + qrow(h), x = qx(h);
      kk[h] = model4(Rkk, h);
      qa[h] = qb[h] = qc[h] = spr[h] = f4{0.0f, 0.0f, 0.0f, 0.0f};
      if (!RCN && GEN && any_lane(split_q(z, x))) {
        const int o = pred_off(ooff, split_q(z, x));
        qa[h] = bld4(field_rsrc(s.q1, s), o, qsoff(h));
        qb[h] = bld4(field_rsrc(s.q2, s), o, qsoff(h));
      }
      if (RCN && img) {
        qc[h] = bld4(field_rsrc(pr, s), old_, qsoff(h));
        const int o = ((z - npml) * s.nxl + x - npml) * 4;
        if (inner_cols) {
          const int oo = GEN ? pred_off(o, inner_row(z)) : o;
          qa[h] = bld4(image_rsrc(s.g1, s), oo, 0);
          qb[h] = bld4(image_rsrc(s.illum, s), oo, 0);
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const int oc = pred_off(o + 4 * c, inner_row(z) & inner_col(x + c) & oq);
            qa[h][c] = bld(image_rsrc(s.g1, s), oc, 0);
            qb[h][c] = bld(image_rsrc(s.illum, s), oc, 0);
          }
        }
      }
      if (strips) {
        const rsrc_t R = strip_rsrc<S16>(s, it);
        const int r = (z - npml) * RTM_R, tb = strip_row_ptb(s, z);
        const bool in = inner_row(z);
        if (hasL) spr[h] = strip4<S16>(R, blr + r + x - npml + RTM_R, in & (x + 3 >= npml - RTM_R) & (x < npml));
        if (hasR) {
          const f4 u = strip4<S16>(R, blr + RTM_R * s.nzi + r + x - nxp + npml,
                              in & (x + 3 >= nxp - npml) & (x < nxp - npml + RTM_R));
          if (!hasL) spr[h] = u;
          else
#pragma unroll
            for (int c = 0; c < 4; c++) spr[h][c] = rightp(x + c) ? u[c] : spr[h][c];
        }
        if (any_lane(tb >= 0)) {
          const f4 u = strip4<S16>(R, tb + x - npml, (tb >= 0) & (x + 3 >= npml) & (x < nxp - npml));
#pragma unroll
          for (int c = 0; c < 4; c++) spr[h][c] = tb >= 0 ? u[c] : spr[h][c];
        }
      }
    }
  }

  __syncthreads();                                     // PS consumed
#pragma unroll
  for (int k = 0; k < KZ; k++)
    if (zrow(k)) VZL[(g * KZ + k) * 64 + lane] = vzn_[k];
  if (live)
#pragma unroll
  for (int k = 0; k < KQ; k++)
    if ((k < KO && oq) || ((k >= KO || RPT < 4) && hon)) {
      f2* d = (f2*)(VXL + (g * RPT + qrow(k)) * VXW + qcol(k) + 10);
      d[0] = f2{hv[k].x, hv[k].y};
      d[1] = f2{hv[k].z, hv[k].w};
    }
  __syncthreads();                                     // new velocities staged

  // ---- 4. differences of the new velocities (kernel.cu:520-534): in x by
  //         own quads, in z by columns, the latter handed to the quads
  //         through the wave's vx rows.  Radius of a cell: min(10, distance
  //         to the nearest grid edge); cells off the grid or on its ring are
  //         computed with radius 10 and dropped
  if (live) {
  f4 dx_[KO], dz_[KO];
#pragma unroll
  for (int h = 0; h < KO; h++) {
    part();
    float w[24];                                       // vx at columns x-10 .. x+13
    const f4* row = (const f4*)(VXL + (g * RPT + qrow(h)) * VXW + (oq ? ocol : 0));
#pragma unroll
    for (int m = 0; m < 6; m++) {
      const f4 v = row[m];
      w[4 * m] = v.x; w[4 * m + 1] = v.y; w[4 * m + 2] = v.z; w[4 * m + 3] = v.w;
    }
    int rad[4] = {RTM_R, RTM_R, RTM_R, RTM_R};
    bool red = false, mixed = false;
    if (EDGE && !RCN) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int x = qx(h) + c, z = zw + qrow(h);
        if (((unsigned)(z - 1) < (unsigned)(nzp - 2)) & ((unsigned)(x - 1) < (unsigned)(nxp - 2)))
          rad[c] = imin(imin(RTM_R, imin(x, nxp - 1 - x)), imin(z, nzp - 1 - z));
        red = red | (rad[c] != RTM_R);
        mixed = mixed | (rad[c] != rad[0]);
      }
      red = any_lane(red);
      mixed = any_lane(mixed);
    }
    if (EDGE && !RCN && red && !mixed) {               // (away from the left and right edge: one row of coefficients)
      const CoefRow cr(ctab, rad[0]);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        float v = taps_r(w, 9 + c, cr);
        pin(v);
        dx_[h][c] = v;
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        float v;
        if (EDGE && !RCN && red) v = taps_r(w, 9 + c, ctab, rad[c]);
        else v = taps(w, 9 + c, c10);
        pin(v);
        dx_[h][c] = v;
      }
    }
  }
  part();
  {
    float cz[RPT + 19];                                // new vz rows zw-10 + m of the column
#pragma unroll
    for (int m = 0; m < RPT + 19; m++) cz[m] = VZL[(g * RPT + m) * 64 + lane];
    const rsrc_t Rvzn = field_rsrc(vzn, s);
    float* T = VXL + g * RPT * VXW;                    // the wave's vx rows, consumed above
    float szc[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) {
      if (r % 2 == 0) part();
      const int iz = zw + r;
      bst<Q::ST>(Rvzn, cz[r + 10], GEN ? pred_off(vcol, (ix < nxp) & (iz < nzp)) : vcol, srow0 + (g * RPT + r) * pr4);
      nzb |= __float_as_uint(cz[r + 10]);
      if (save) {
        const int st = strip_row_vz(s, iz);            // wave-uniform
        if (st >= 0) put(strip_rsrc<S16>(s, it), 1, st + ix - npml, cz[r + 10], zcol);
      }
      if (EDGE && !RCN) {
        int rad = RTM_R;
        if (iz > 0 && iz < nzp - 1 && ix > 0 && ix < nxp - 1)
          rad = imin(imin(RTM_R, imin(ix, nxp - 1 - ix)), imin(iz, nzp - 1 - iz));
        szc[r] = any_lane(rad != RTM_R) ? taps_r(cz, r + 9, ctab, rad) : taps(cz, r + 9, c10);
      } else {
        szc[r] = taps(cz, r + 9, c10);
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < RPT; r++) T[r * 64 + lane] = szc[r];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < KO; h++) dz_[h] = *(const f4*)(T + (oq ? qrow(h) * 64 + ocol : 0));
  }

  // ---- 5. new pressure of the own quads
  const rsrc_t Rpn = field_rsrc(pn, s);
  auto strip_p = [&](int z, int x) {
    const bool in = inner_row(z);
    return strips && ((in & (left(x) | rightp(x))) | (!in & (strip_row_ptb(s, z) >= 0) & inner_col(x)));
  };
#pragma unroll
  for (int h = 0; h < KO; h++) {
    part();
    const int z = zw + qrow(h), x = qx(h);
    const bool on = oq;
    f4 p = po[h];
    if (RCN) {
      if (img) {                                       // imaging of the step before (kernel.cu:1401-1416)
        const int o = ((z - npml) * s.nxl + x - npml) * 4;
        f4 gi, ii;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          gi[c] = __builtin_fmaf(po[h][c], qc[h][c], qa[h][c]);
          ii[c] = __builtin_fmaf(po[h][c], po[h][c], qb[h][c]);
        }
        if (inner_cols) {
          const int oo = pred_off(o, on & (!GEN | inner_row(z)));
          bst4<Q::ST>(image_rsrc(s.g1, s), gi, oo, 0);
          bst4<Q::ST>(image_rsrc(s.illum, s), ii, oo, 0);
        } else {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const int oc = pred_off(o + 4 * c, inner_row(z) & inner_col(x + c) & on);
            bst<Q::ST>(image_rsrc(s.g1, s), gi[c], oc, 0);
            bst<Q::ST>(image_rsrc(s.illum, s), ii[c], oc, 0);
          }
        }
      }
      if (S16 && strips)
#pragma unroll
        for (int c = 0; c < 4; c++) spr[h][c] = strip_value<S16>(s, inner_row(z) ? scv[2] : scv[3], spr[h][c]);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float sum = __builtin_fmaf(dx_[h][c], dtx, dz_[h][c] * dtz);
        float v = __builtin_fmaf(kk[h][c], sum, po[h][c]);   // kernel.cu:389-429
        bool wr = true;
        if (GEN) {
          wr = inner_row(z) & inner_col(x + c);
          v = wr ? v : 0.0f;                           // cells the reconstruction does not hold
          v = strip_p(z, x + c) ? spr[h][c] : v;       // kernel.cu:1348-1400
        }
        p[c] = v;
      }
      if (tl.kind & TF_SRC) {                          // source removal (rtm_model.cu:437)
        const float wv = CCF(s.wav)[it];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const bool wr = !GEN | (inner_row(z) & inner_col(x + c)) | strip_p(z, x + c);
          if (wr && on && z >= s.sz0 && z <= s.sz1 && x + c >= s.sx0 && x + c <= s.sx1)
            p[c] = __builtin_fmaf(-GCF(s.sa)[(z - s.sz0) * (s.sx1 - s.sx0 + 1) + x + c - s.sx0], wv, p[c]);
        }
      }
      bst4<Q::ST>(Rpn, p, pred_off(ooff, on & (!GEN | ((x < nxp) & (z < nzp)))), qsoff(h));
      continue;
    }
    f4 pu;
#pragma unroll
    for (int c = 0; c < 4; c++)                        // p - rho v^2 (sx dt/dx + sz dt/dz) (kernel.cu:536-539)
      pu[c] = __builtin_fmaf(-kk[h][c], __builtin_fmaf(dx_[h][c], dtx, dz_[h][c] * dtz), po[h][c]);
    if (!GEN) {
      p = pu;
    } else {
      // the outer ring and the cells off the grid keep their value
#pragma unroll
      for (int c = 0; c < 4; c++) p[c] = inner_row(z) & inner_col(x + c) ? pu[c] : po[h][c];
      if (any_lane(split_q(z, x))) {                   // split pair, p = p1 + p2 (kernel.cu:774-783)
        const f4 ax = *(const f4*)(DPX + (oq ? ocol : 0));
        const f4 bx = *(const f4*)(DPX + 64 + (oq ? ocol : 0));
        const float az = DPZ[g * RPT + qrow(h)], bz = DPZ[TZ + g * RPT + qrow(h)];
        f4 q1, q2;
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const float dxv = (dx_[h][c] * dtx) * kk[h][c], dzv = (dz_[h][c] * dtz) * kk[h][c];
          const bool sp = split(z, x + c);
          q1[c] = sp ? __builtin_fmaf(ax[c], qa[h][c], -(dxv * bx[c])) : qa[h][c];   // (c1 q - d)/c2
          q2[c] = sp ? __builtin_fmaf(az, qb[h][c], -(dzv * bz)) : qb[h][c];
          p[c] = sp ? q1[c] + q2[c] : p[c];
          if (on) nzb |= __float_as_uint(q1[c]) | __float_as_uint(q2[c]);
        }
        const int o = pred_off(ooff, split_q(z, x));
        bst4<Q::ST>(field_rsrc(s.q1, s), q1, o, qsoff(h));
        bst4<Q::ST>(field_rsrc(s.q2, s), q2, o, qsoff(h));
      }
    }
    if (FK == FK_SRC && (tl.kind & TF_SRC)) {          // kernel.cu:36-47
      const float wv = CCF(s.wav)[it];
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (on && z >= s.sz0 && z <= s.sz1 && x + c >= s.sx0 && x + c <= s.sx1)
          p[c] = __builtin_fmaf(GCF(s.sa)[(z - s.sz0) * (s.sx1 - s.sx0 + 1) + x + c - s.sx0], wv, p[c]);
    }
    if (tl.kind & TF_REC) {
      if (on && z == npml && (FK == FK_RCV || s.record)) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const int ir = x + c - s.rcol0;
          if (ir >= 0 && ir < s.nrec) {
            if (FK == FK_SRC) {                        // kernel.cu:48-71
              GF(s.rec)[(size_t)it * s.nrec + ir] = p[c];
            } else {                                   // Dirichlet insertion (kernel.cu:72-95)
              const float rv = (it <= ((const gint*)s.cut)[ir]) ? 0.0f : GCF(s.rec)[(size_t)it * s.nrec + ir];
              p[c] = s.dt * rv;
            }
          }
        }
      }
    }
    if (on)
#pragma unroll
      for (int c = 0; c < 4; c++) nzb |= __float_as_uint(p[c]);
    if (save) {
      const rsrc_t R = strip_rsrc<S16>(s, it);
      const int r = (z - npml) * RTM_R, tb = strip_row_ptb(s, z);
      const bool in = on & inner_row(z);
      if (hasL)
#pragma unroll
        for (int c = 0; c < 4; c++) put(R, 2, blr + r + x + c - npml + RTM_R, p[c], in & left(x + c));
      if (hasR)
#pragma unroll
        for (int c = 0; c < 4; c++) put(R, 2, blr + RTM_R * s.nzi + r + x + c - nxp + npml, p[c], in & rightp(x + c));
      if (any_lane(tb >= 0))
#pragma unroll
        for (int c = 0; c < 4; c++) put(R, 3, tb + x + c - npml, p[c], on & (tb >= 0) & inner_col(x + c));
    }
    bst4<Q::ST>(Rpn, p, pred_off(ooff, on & (!GEN | ((x < nxp) & (z < nzp)))), qsoff(h));
  }
  }
  if (S16 && save) {
#pragma unroll
    for (int b = 0; b < 4; b++) {
      if (!any_lane(smax[b] > 0.0f)) continue;
      float m = smax[b];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      if (lane == 0) atomicMax(strip_max(s, it) + b, __float_as_uint(m));
    }
  }
  if (FK == FK_SRC && actw) {
    const bool any = any_lane(nzb != 0u);
    // (a word is 8 bytes whatever the wave count: its bytes start non-zero)
    if (lane == 0) {
      if (G == 4) ((unsigned short*)actw)[g] = any ? 1 : 0;
      else actw[g] = any ? 1 : 0;
    }
  }
}

template <class Q, int FK>
__device__ __forceinline__ void field_step(float* __restrict__ lds, float* __restrict__ ctab, const ShotDev& s,
                                           const Tile& tl, int it, const float* pc, const float* vxc,
                                           const float* vzc, float* pn, float* vxn, float* vzn,
                                           const float* pr = nullptr, bool img = false, bool save = false,
                                           unsigned char* actw = nullptr)
{
  if (!(tl.kind & TF_GEN)) {
    tile_step<Q, FK, TC_IN>(lds, ctab, s, tl, it, pc, vxc, vzc, pn, vxn, vzn, pr, img, save, actw);
  } else if (FK == FK_RCN || !(tl.kind & TF_EDGE)) {
    tile_step<Q, FK, TC_GEN>(lds, ctab, s, tl, it, pc, vxc, vzc, pn, vxn, vzn, pr, img, save, actw);
  } else {
    for (int t = threadIdx.x; t < RTM_R * CTW; t += Q::NT) ctab[t] = ctab_entry(s, t);   // read after the first barrier
    tile_step<Q, FK, TC_EDGE>(lds, ctab, s, tl, it, pc, vxc, vzc, pn, vxn, vzn, pr, img, save, actw);
  }
}

// Zero-tile skip of the forward step: a tile skips the step when the forward
// field is zero at the level the step reads, on the tile and its 8
// neighbours (all the step's inputs are then +0 and so would be its
// outputs: the step reads 19 rows and columns out, within the adjacent
// tiles for tiles of 32 or 64 rows; the host passes no words for 16-row
// tiles), and at the level it writes, on the tile itself (the buffer
// already holds those +0).  The wavefield starts at +0 and spreads from the
// source, so far tiles skip until it comes near.  Words of both levels are
// fetched beside the tile's other first loads; `it` picks the level.  (The
// same skip of the reverse step's receiver field cost more than it saved:
// that field rarely has a zero neighbourhood.)
struct SkipWords { unsigned long long self0, self1, nb0, nb1; };   // (no arrays: a runtime index would spill)
__device__ __forceinline__ SkipWords skip_words(const unsigned long long* act, int ntiles, int t, const Tile& tl)
{
  SkipWords w{act[t], act[ntiles + t], 0ull, 0ull};
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (tl.nbr[j] >= 0) {
      w.nb0 |= act[tl.nbr[j]];
      w.nb1 |= act[ntiles + tl.nbr[j]];
    }
  return w;
}
__device__ __forceinline__ bool skip_of(const SkipWords& w, int it)
{
  const bool odd = it & 1;
  const unsigned long long in = odd ? (w.self1 | w.nb1) : (w.self0 | w.nb0);
  const unsigned long long out = odd ? w.self0 : w.self1;
  return (in | out) == 0ull;
}

// the strip values of a tile that skips its step: all +0
template <class Q>
__device__ __forceinline__ void save_zeros(const ShotDev& s, const Tile& tl, int it)
{
  gfloat* rec = GF(s.store) + (long long)it * s.strip_len;
  for (int e = threadIdx.x; e < 64 * Q::TZ; e += Q::NT) {
    const int z = tl.z0 + (e >> 6), x = tl.x0 + (e & 63);
    const bool in = x >= s.npml && x < s.nxp - s.npml;
    const int vx = strip_vx(s, z, x), vz = strip_row_vz(s, z), lr = strip_row_lr(s, z), tb = strip_row_ptb(s, z);
    const int pl = lr >= 0 ? strip_col_plr(s, x) : -1;
    if (vx >= 0) rec[vx] = 0.0f;
    if (vz >= 0 && in) rec[vz + x - s.npml] = 0.0f;
    if (pl >= 0) rec[lr + pl] = 0.0f;
    else if (tb >= 0 && in) rec[tb + x - s.npml] = 0.0f;
  }
}

// index of the snapshot of step k (below: decimated snapshots), -1 if none
__device__ __forceinline__ int snap_index(const ShotDev& s, int k)
{
  if (!s.snap || k < 0 || k % s.snap_every != 0) return -1;
  const int q = k / s.snap_every - s.snap_k0;
  return (q >= 0 && q < s.nsnap) ? q : -1;
}

}  // namespace

// ================================================================ kernels ==
// forward time step of the source wavefield (modelling, recording, strips)
template <int G, int RPT, bool C, bool S16>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_fwd(LaunchArgs a)
{
  using Q = Geo<G, RPT, C, S16>;
  __shared__ __attribute__((aligned(16))) float lds[Q::LDS + Q::LDS_D];
  __shared__ __attribute__((aligned(16))) float ctab[RTM_R * CTW];   // coefficient table (reduced radii near the edges)
  const int v = xcd_tile(a.ntiles * Q::SPLIT);
  if (v < 0) return;
  const int t = v / Q::SPLIT;
  Tile tl = a.tiles[t];
  if (tl.slot < 0) return;                             // padding of a shorter XCD run
  tl.z0 += v % Q::SPLIT * Q::TZ;
  const bool track = a.act && !(tl.kind & (TF_SRC | TF_REC));
  SkipWords sw{};
  if (track) sw = skip_words(a.act, a.ntiles, t, tl);
  fetch_shot(a.shots, tl.slot);
  const ShotDev& s = shot_of(a.shots, tl.slot);
  const int it = s.it_off + s.it_dir * a.step;
  if (track && skip_of(sw, it)) {                      // the forward field is +0 around the tile
    if (!S16 && a.save && (tl.kind & TF_SAVE)) save_zeros<Q>(s, tl, it);
    return;
  }
  const bool odd = it & 1;                             // (a runtime index into s would spill it to scratch)
  unsigned char* actw = a.act ? (unsigned char*)(a.act + (size_t)((it + 1) & 1) * a.ntiles + t) : nullptr;
  field_step<Q, FK_SRC>(lds, ctab, s, tl, it, odd ? s.sp[1] : s.sp[0], odd ? s.svx[1] : s.svx[0],
                        odd ? s.svz[1] : s.svz[0], odd ? s.sp[0] : s.sp[1], odd ? s.svx[0] : s.svx[1],
                        odd ? s.svz[0] : s.svz[1], nullptr, false, a.save != 0, actw);
}

// tiles whose receiver halves, then reconstruction halves, follow each other
// on an XCD: workgroups go to its shader engines in turn, so alternating the
// two kinds one by one gave half of the engines the shorter kind only (10.3 of
// 16 waves resident per CU, 634 us a reverse step of 128 survey shots; in
// groups of 8, 16 or 32: 13.5 waves, 519 us)
constexpr int RGRP = 16;

// reverse time step: two workgroups per tile, close together on one XCD, one
// for the receiver wavefield and one for the source reconstruction with the
// imaging products.  The reconstruction images the step before (both fields'
// old levels: its own pressure is staged anyway, the receiver pressure is in
// L2 from the other workgroup), so the two run at the same time; the last
// step's products are added by k_image after the pass, those of a step whose
// snapshot is restored by k_snap_load before it overwrites the field.
template <int G, int RPT, bool C, bool S16>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_rev(LaunchArgs a)
{
  using Q = Geo<G, RPT, C, S16>;
  __shared__ __attribute__((aligned(16))) float lds[Q::LDS + Q::LDS_D];
  __shared__ __attribute__((aligned(16))) float ctab[RTM_R * CTW];
  // XCD c's workgroups take its run of the table RGRP tiles at a time, their
  // receiver halves and then their reconstruction halves
  const int n = a.ntiles * Q::SPLIT, per = (n + 7) >> 3, b = blockIdx.x >> 3, r = b % (2 * RGRP);
  const int i = b / (2 * RGRP) * RGRP + r % RGRP;
  if (i >= per) return;
  const int v = (blockIdx.x & 7) * per + i;
  if (v >= n) return;
  Tile tl = a.tiles[v / Q::SPLIT];
  if (tl.slot < 0) return;                             // padding of a shorter XCD run
  tl.z0 += v % Q::SPLIT * Q::TZ;
  fetch_shot(a.shots, tl.slot);
  const ShotDev& s = shot_of(a.shots, tl.slot);
  const int it = s.it_off + s.it_dir * a.step;
  const bool odd = it & 1;
  if (r >= RGRP) {
    if (!(tl.kind & TF_INT)) return;
    const bool img = it < s.nt - 2 && snap_index(s, it + 1) < 0;
    field_step<Q, FK_RCN>(lds, ctab, s, tl, it, odd ? s.sp[1] : s.sp[0], odd ? s.svx[1] : s.svx[0],
                          odd ? s.svz[1] : s.svz[0], odd ? s.sp[0] : s.sp[1], odd ? s.svx[0] : s.svx[1],
                          odd ? s.svz[0] : s.svz[1], odd ? s.rp[1] : s.rp[0], img);
  } else {
    field_step<Q, FK_RCV>(lds, ctab, s, tl, it, odd ? s.rp[1] : s.rp[0], odd ? s.rvx[1] : s.rvx[0],
                          odd ? s.rvz[1] : s.rvz[0], odd ? s.rp[0] : s.rp[1], odd ? s.rvx[0] : s.rvx[1],
                          odd ? s.rvz[0] : s.rvz[1]);
  }
}

// imaging products of reverse step `it` of the listed slots from the levels
// it wrote (kernel.cu:1401-1416): the last step of a pass, which no later
// step images.  Grid (slots, GY), one wave per row.
__global__ __launch_bounds__(NTHR) void k_image(const ShotDev* __restrict__ shots, const int* __restrict__ slots, int it)
{
  const ShotDev& s = shot_of(shots, slots[blockIdx.x]);
  const bool lev = (it + 1) & 1;
  const float* fs = lev ? s.sp[1] : s.sp[0];
  const float* fr = lev ? s.rp[1] : s.rp[0];
  const int nxl = s.nxl, lane = threadIdx.x & 63;
  for (int r = blockIdx.y * (NTHR / 64) + (threadIdx.x >> 6); r < s.nzi; r += gridDim.y * (NTHR / 64)) {
    const long long o = (long long)(s.npml + r) * s.pitch + s.npml;
    for (int c = lane; c < nxl; c += 64) {
      const float ps = GCF(fs)[o + c], p = GCF(fr)[o + c];
      const long long e = (long long)r * nxl + c;
      GF(s.g1)[e] = __builtin_fmaf(ps, p, GCF(s.g1)[e]);
      GF(s.illum)[e] = __builtin_fmaf(ps, ps, GCF(s.illum)[e]);
    }
  }
}

// Boundary strips of forward step `it` -- the new fields of that step -- in
// the store, packed as kernel.cu:1186-1293 per step:
//   vx lr [2][nzi][10] | vz tb [2][10][nxl] | p lr [2][nzi][10] | p tb [2][10][nxl]
// The step kernel writes the fp32 ones itself; the 16-bit forms store each
// block with a scale of its own, known only once every tile has stepped
// (k_quant16).
struct StripBlock {
  const float* f;    // field (cell (0,0)), new level
  int lr;            // 1: [2][nzi][10] column strips, 0: [2][10][nxl] row strips
  int lo, n;         // offset of the block in the step's record, element count
  int a0, a1;        // first column (lr) / row (tb) of side 0 and side 1
};
__device__ __forceinline__ StripBlock strip_block_of(const ShotDev& s, int b, int lev)
{
  const int n = s.npml, e1 = 2 * RTM_R * s.nzi, e2 = e1 + 2 * RTM_R * s.nxl, e3 = e2 + 2 * RTM_R * s.nzi;
  // (levels selected, not indexed: a run-time index would put s in scratch)
  const float* vx = lev ? s.svx[1] : s.svx[0];
  const float* vz = lev ? s.svz[1] : s.svz[0];
  const float* p = lev ? s.sp[1] : s.sp[0];
  StripBlock k;
  if (b == 0) k = {vx, 1, 0, e1, n - RTM_R, s.nxp - n - 1};                  // strip_vx
  else if (b == 1) k = {vz, 0, e1, e2 - e1, n - RTM_R, s.nzp - n - 1};        // strip_vz
  else if (b == 2) k = {p, 1, e2, e3 - e2, n - RTM_R, s.nxp - n};             // strip_p lr
  else k = {p, 0, e3, (int)s.strip_len - e3, n - RTM_R, s.nzp - n};            // strip_p tb
  return k;
}
// element e of a block: its field value
__device__ __forceinline__ float strip_elem(const ShotDev& s, const StripBlock& k, int e)
{
  if (k.lr) {                                          // e = (side*nzi + r)*10 + c
    const int q = e / RTM_R, c = e - q * RTM_R;
    const int side = q >= s.nzi, r = q - side * s.nzi;
    return GCF(k.f)[(size_t)(s.npml + r) * s.pitch + (side ? k.a1 : k.a0) + c];
  }
  const int q = e / s.nxl, c = e - q * s.nxl;          // e = (side*10 + r)*nxl + c
  const int side = q >= RTM_R, r = q - side * RTM_R;
  return GCF(k.f)[(size_t)((side ? k.a1 : k.a0) + r) * s.pitch + s.npml + c];
}

// 16-bit store of step `step`'s strips: block b of a slot with the scale
// max(maxabs / 32768, FLT_MIN) (1 for an all-zero block; a denormal max-abs,
// e.g. source tails before the wave arrives, must not underflow the scale to
// zero: |x| <= 32768 * FLT_MIN then anyway), x / scale rounded to nearest
// even.  The step's tiles have left the block's max-abs (strip_max), so a
// block is spread over gridDim.y workgroups, SV loads in flight a thread, and
// the words of the next step are cleared here.  Latency-bound: one workgroup
// of 1024 threads per block, which also took the max-abs, needed 18.7 us a
// step on 4 slots of 2148 x 1124 (16 workgroups on 256 CUs).
constexpr int SV = 4;
__global__ __launch_bounds__(NTHR) void k_quant16(const ShotDev* __restrict__ shots, const int* __restrict__ slots,
                                                   int nslots, int step)
{
  const int k = blockIdx.x >> 2, b = blockIdx.x & 3;
  if (k >= nslots) return;
  const ShotDev& s = shot_of(shots, slots[k]);
  const int it = s.it_off + s.it_dir * step;
  const StripBlock blk = strip_block_of(s, b, (it + 1) & 1);
  const long long base = (long long)it * s.strip_len + blk.lo;
  const float m = __uint_as_float(strip_max(s, it)[b]);
  const float sc = m > 0.0f ? fmaxf(m * (1.0f / 32768.0f), 1.17549435e-38f) : 1.0f;
  if (blockIdx.y == 0 && threadIdx.x == 0) {
    s.sscale[(long long)it * 4 + b] = sc;
    strip_max(s, it + 1)[b] = 0u;
  }
  const int stride = gridDim.y * NTHR * SV;
  for (int e0 = blockIdx.y * NTHR * SV + threadIdx.x; e0 < blk.n; e0 += stride) {
    float v[SV];
#pragma unroll
    for (int u = 0; u < SV; u++) v[u] = e0 + u * NTHR < blk.n ? strip_elem(s, blk, e0 + u * NTHR) : 0.0f;
#pragma unroll
    for (int u = 0; u < SV; u++) {
      const int e = e0 + u * NTHR;
      if (e >= blk.n) continue;
      const float q = v[u] / sc;
      unsigned short h;
      if (s.store_fmt == ST_F16) {
        h = __half_as_ushort(__float2half_rn(q));
      } else {
        unsigned int w = __float_as_uint(q);           // bf16, round to nearest even
        w += 0x7FFFu + ((w >> 16) & 1u);
        h = (unsigned short)(w >> 16);
      }
      __builtin_nontemporal_store(h, (gushort*)s.store + base + e);
    }
  }
}

// 1/rho and rho v^2 of a model, rounded once (the factors the step kernels
// read): the resident model at its creation, a shot's smoothed window
// (pmlvelsmooth1d / velsmooth1d) whenever it changes
__global__ __launch_bounds__(NTHR) void k_model_prep(const float* __restrict__ rho, const float* __restrict__ vv,
                                                      float* __restrict__ ib, float* __restrict__ kk, long long n)
{
  for (long long e = (long long)blockIdx.x * NTHR + threadIdx.x; e < n; e += (long long)gridDim.x * NTHR) {
    const float rh = rho[e];
    ib[e] = 1.0f / rh;
    kk[e] = rh * vv[e];
  }
}

// ------------------------------------------------------------ snapshots --
// Decimated snapshots of the source wavefield.  The reverse pass runs the
// leapfrog backwards, velocities first: after reverse step k it holds the
// pressure of forward step k and the velocities of forward step k+1 (its
// strips are read the same way, rtm_model.cu:424-434).  Snapshot k (k =
// snap_every * (snap_k0 + q)) therefore keeps the interior of p as forward
// step k leaves it and of vx, vz as forward step k+1 leaves them, and the
// reverse pass writes them back after its step k, so that the steps below k
// start from the stored field.  Block (q, f), f = 0 p, 1 vx, 2 vz: nzi x nxl
// codes; 16-bit forms with one max-abs scale per block (the strips' rule:
// max(maxabs / 32768, FLT_MIN), 1 for an all-zero block).
// the snapshot a forward step `it` contributes field f to: p of step k = it,
// velocities of step it = k + 1
__device__ __forceinline__ int snap_of_fwd(const ShotDev& s, int it, int f)
{
  return snap_index(s, f == 0 ? it : it - 1);
}
__device__ __forceinline__ const float* snap_field(const ShotDev& s, int f, bool lev)
{
  return f == 0 ? (lev ? s.sp[1] : s.sp[0]) : (f == 1 ? (lev ? s.svx[1] : s.svx[0]) : (lev ? s.svz[1] : s.svz[0]));
}
__device__ __forceinline__ unsigned int* snap_acc(const ShotDev& s) { return (unsigned int*)(s.snap_scale + 3 * s.nsnap); }

// The snapshot kernels run after every step of a pass (a captured graph
// holds the same launches for every step) and return at once unless the step
// takes or restores a snapshot.  When it does, a block is the nz x nxl
// interior of one field: one wave per row, rows dealt over the waves of
// gridDim.y workgroups, a lane taking SU columns 64 apart per iteration
// (independent loads in flight, no index division).
constexpr int SU = 4, SWB = NTHR / 64;

// forward, pass 1 (16-bit forms): max-abs of the workgroup's share of block
// (q, f) after forward step `step` (its new level).  Grid (3 slots, GY).
__global__ __launch_bounds__(NTHR) void k_snap_max(const ShotDev* __restrict__ shots, const int* __restrict__ slots,
                                                    int step)
{
  __shared__ float red[NTHR / 64];
  const ShotDev& s = shot_of(shots, slots[blockIdx.x / 3]);
  const int it = s.it_off + s.it_dir * step, f = blockIdx.x % 3;
  const int q = snap_of_fwd(s, it, f);
  if (q < 0) return;
  const float* fld = snap_field(s, f, (it + 1) & 1);
  const int nxl = s.nxl, lane = threadIdx.x & 63;
  float m = 0.0f;
  for (int r = blockIdx.y * SWB + (threadIdx.x >> 6); r < s.nzi; r += gridDim.y * SWB) {
    const gfloat* row = GCF(fld) + (long long)(s.npml + r) * s.pitch + s.npml;
    for (int c0 = lane; c0 < nxl; c0 += SU * 64) {
      float a[SU];
#pragma unroll
      for (int u = 0; u < SU; u++) a[u] = c0 + u * 64 < nxl ? fabsf(row[c0 + u * 64]) : 0.0f;
#pragma unroll
      for (int u = 0; u < SU; u++) m = fmaxf(m, a[u]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NTHR / 64; w++) m = fmaxf(m, red[w]);
    atomicMax(snap_acc(s) + q * 3 + f, __float_as_uint(m));
  }
}

// forward, pass 2: block (q, f) stored as codes (fp32: a copy) with its scale
__global__ __launch_bounds__(NTHR) void k_snap_q(const ShotDev* __restrict__ shots, const int* __restrict__ slots,
                                                  int step)
{
  const ShotDev& s = shot_of(shots, slots[blockIdx.x / 3]);
  const int it = s.it_off + s.it_dir * step, f = blockIdx.x % 3;
  const int q = snap_of_fwd(s, it, f);
  if (q < 0) return;
  const float* fld = snap_field(s, f, (it + 1) & 1);
  const int nxl = s.nxl, n = s.nzi * nxl, lane = threadIdx.x & 63;
  const long long base = (long long)(q * 3 + f) * n;
  float sc = 1.0f;
  if (s.snap_fmt != ST_F32) {
    const float m = __uint_as_float(snap_acc(s)[q * 3 + f]);
    sc = m > 0.0f ? fmaxf(m * (1.0f / 32768.0f), 1.17549435e-38f) : 1.0f;
  }
  if (blockIdx.y == 0 && threadIdx.x == 0) s.snap_scale[q * 3 + f] = sc;
  for (int r = blockIdx.y * SWB + (threadIdx.x >> 6); r < s.nzi; r += gridDim.y * SWB) {
    const gfloat* row = GCF(fld) + (long long)(s.npml + r) * s.pitch + s.npml;
    const long long ob = base + (long long)r * nxl;
    for (int c0 = lane; c0 < nxl; c0 += SU * 64) {
      float v[SU];
#pragma unroll
      for (int u = 0; u < SU; u++) v[u] = c0 + u * 64 < nxl ? row[c0 + u * 64] : 0.0f;
#pragma unroll
      for (int u = 0; u < SU; u++) {
        const int c = c0 + u * 64;
        if (c >= nxl) continue;
        if (s.snap_fmt == ST_F32) {
          GF(s.snap)[ob + c] = v[u];
        } else if (s.snap_fmt == ST_F16) {
          ((__half*)s.snap)[ob + c] = __float2half_rn(v[u] / sc);
        } else {
          unsigned int w = __float_as_uint(v[u] / sc);   // bf16, round to nearest even
          w += 0x7FFFu + ((w >> 16) & 1u);
          ((unsigned short*)s.snap)[ob + c] = (unsigned short)(w >> 16);
        }
      }
    }
  }
}

// reverse: after reverse step `step` = k (its new level (k+1)&1), snapshot
// k replaces the reconstructed interior cells: p on the
// interior, vx on its columns npml..nxp-npml-2, vz on its rows
// npml..nzp-npml-2 (the cells the reconstruction computes; the strips come
// from the boundary store as on every step).  The step's imaging products are
// added first: they take the reconstructed pressure
__global__ __launch_bounds__(NTHR) void k_snap_load(const ShotDev* __restrict__ shots, const int* __restrict__ slots,
                                                     int step)
{
  const ShotDev& s = shot_of(shots, slots[blockIdx.x / 3]);
  const int it = s.it_off + s.it_dir * step;
  const int q = snap_index(s, it);
  if (q < 0) return;
  const int f = blockIdx.x % 3;
  float* fld = (float*)snap_field(s, f, (it + 1) & 1);
  const int nxl = s.nxl, n = s.nzi * nxl, lane = threadIdx.x & 63;
  const int ncol = f == 1 ? nxl - 1 : nxl, nrow = f == 2 ? s.nzi - 1 : s.nzi;
  const long long base = (long long)(q * 3 + f) * n;
  const float sc = s.snap_scale[q * 3 + f];
  const float* fr = (it + 1) & 1 ? s.rp[1] : s.rp[0];
  for (int r = blockIdx.y * SWB + (threadIdx.x >> 6); r < nrow; r += gridDim.y * SWB) {
    gfloat* row = GF(fld) + (long long)(s.npml + r) * s.pitch + s.npml;
    const long long ib = base + (long long)r * nxl;
    if (f == 0) {                                      // the step's imaging products, before its field is replaced
      const gfloat* rr = GCF(fr) + (long long)(s.npml + r) * s.pitch + s.npml;
      for (int c = lane; c < nxl; c += 64) {
        const float ps = row[c], p = rr[c];
        const long long e = (long long)r * nxl + c;
        GF(s.g1)[e] = __builtin_fmaf(ps, p, GCF(s.g1)[e]);
        GF(s.illum)[e] = __builtin_fmaf(ps, ps, GCF(s.illum)[e]);
      }
    }
    for (int c0 = lane; c0 < ncol; c0 += SU * 64) {
      float v[SU];
#pragma unroll
      for (int u = 0; u < SU; u++) {
        const int c = c0 + u * 64;
        v[u] = 0.0f;
        if (c >= ncol) continue;
        if (s.snap_fmt == ST_F32) v[u] = GCF(s.snap)[ib + c];
        else if (s.snap_fmt == ST_F16) v[u] = __half2float(((const __half*)s.snap)[ib + c]) * sc;
        else v[u] = __uint_as_float((unsigned int)((const unsigned short*)s.snap)[ib + c] << 16) * sc;
      }
#pragma unroll
      for (int u = 0; u < SU; u++)
        if (c0 + u * 64 < ncol) row[c0 + u * 64] = v[u];
    }
  }
}

// ------------------------------------------------------- model smoothing --
// velsmooth1d (Velocity_function.cpp:199-313) of an nz x nx window: every
// output cell is the sum over the (2 nsp + 1)^2 window around it of
// weight x value, in double, rows then columns as the reference loops, on
// the window extended by its edge values (a clamp), rounded to float and
// then divided (in double) by the sum of the weights.  The weights are
// tabulated on the host with the reference's expression (wt, row-major),
// so every term is the reference's.
__global__ __launch_bounds__(NTHR) void k_gauss_smooth(const float* __restrict__ in, float* __restrict__ out, int nz,
                                                        int nx, int nsp, const double* __restrict__ wt, double norm)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e >= (long long)nz * nx) return;
  const int iz = (int)(e / nx), ix = (int)(e - (long long)iz * nx);
  const int k = 2 * nsp + 1;
  double acc = 0.0;
  for (int i = 0; i < k; i++) {
    const float* row = in + (size_t)imin(imax(iz + i - nsp, 0), nz - 1) * nx;
    const double* w = wt + (size_t)i * k;
    for (int j = 0; j < k; j++) acc += w[j] * (double)row[imin(imax(ix + j - nsp, 0), nx - 1)];
  }
  out[e] = (float)((double)(float)acc / norm);
}

// pmlvelsmooth1d (Velocity_function.cpp:9-103) of one nz x nx window per
// workgroup (wins[blockIdx.x]: the window w, in place, and a scratch window
// v of the same size).  The reference mirrors the interior into the
// absorbing layer, then relaxes the layer in place -- each cell becomes the
// average of its four neighbours, taking those already updated in the sweep
// as updated -- until a sweep changes no cell by more than 5e-4 (relative)
// or 1001 sweeps ran.  The in-place order is kept exactly:
//   * left and right layers (columns 1..npml-1, rows 1..nz-2 in order, the
//     reference's ix-outer / iz-inner loop), one wave each (smooth_front);
//   * top and bottom layers (rows 1..npml-1, columns 1..nx-2) the same with
//     lanes over rows;
//   * the edge columns and rows: four independent recurrences, one lane
//     each, from sums formed beforehand; then the four corners.
// Each sweep ends with the largest relative change over the layer ring (the
// rest of the window never changes) and copies the ring back into w.  Sums
// are formed in the reference's operand order, as floats, scaled by the
// double literal 0.25 (a power of two: the float product is the same value).
// What bounds it is the serial chain: about nz + nx + 2 npml dependent steps
// a sweep and up to 1001 sweeps, on the few CUs that hold windows.  So a
// step's operands are read ahead, its neighbours come by lane shifts in the
// VALU, and the ring with one interior line beside it stays in LDS where it
// fits (SMOOTH_LDS floats); a larger one is read through the caches.  The 16
// waves are for the comparison of the ring (512 threads: within 10 % at rings
// in LDS, 15 % slower in memory; 256: 50 % slower).  One window with its
// transfers, against every operand loaded when needed and shuffled through
// LDS: 265 x 320, npml 32, 20.0 -> 7.0 ms; 401 x 612, npml 50, 55.5 -> 24.8;
// 2148 x 1124, npml 50, 162 -> 74.5.
// Needs npml - 1 <= 64, nx, nz >= 3 npml (the mirrors read only interior
// cells) and nx, nz <= RTM_SMOOTH_MAXN.
#define RTM_SMOOTH_MAXN 4096
struct SmoothWin { float* w; float* v; int nx, nz, npml, _pad; };
constexpr int SMT = 1024, SMOOTH_LDS = 40000;

__device__ __forceinline__ float avg4(float a, float b, float c, float d) { return 0.25f * (((a + b) + c) + d); }

// Where the cells of the ring are (byte offsets).  A line of a front is a
// column, at base + row * pitch, or a row, whose columns start at l, c and r in
// the left layer, the centre and the right layer (less the column itself).
struct RowAt { int l, c, r; };
// the full window in memory ...
struct RingMem {
  typedef __attribute__((address_space(1))) char gchar;
  gfloat* p;
  int nx;
  __device__ __forceinline__ gfloat* cell(int a) const { return (gfloat*)((gchar*)p + (unsigned)a); }
  __device__ __forceinline__ float get(int a) const { return *cell(a); }
  __device__ __forceinline__ void set(int a, float x) const { *cell(a) = x; }
  __device__ __forceinline__ int pitch() const { return 4 * nx; }
  __device__ __forceinline__ int column(int c) const { return 4 * c; }
  __device__ __forceinline__ RowAt row(int r) const { return RowAt{4 * r * nx, 4 * r * nx, 4 * r * nx}; }
  __device__ __forceinline__ int in_row(const RowAt& w, int c) const { return w.c + 4 * c; }
  __device__ __forceinline__ bool straight(int, int) const { return true; }
  __device__ __forceinline__ int at(int r, int c) const { return 4 * (r * nx + c); }
};
// ... or the ring and one line beside it (m = npml + 1 deep) in LDS: the first
// and last m columns of every row, 2 m to a row, then the centre columns of
// the first and last m rows.  Both pitches are even, so that a front, whose
// lanes are a pitch less one apart, meets every bank.
typedef __attribute__((address_space(3))) float lds_float_t;
typedef __attribute__((address_space(3))) char lds_char_t;
struct RingLds {
  lds_float_t* p;
  int nx, nz, m, P;                                    // P: pitch of the centre columns
  __device__ __forceinline__ lds_float_t* cell(int a) const { return (lds_float_t*)((lds_char_t*)p + a); }
  __device__ __forceinline__ float get(int a) const { return *cell(a); }
  __device__ __forceinline__ void set(int a, float x) const { *cell(a) = x; }
  __device__ __forceinline__ int pitch() const { return 8 * m; }
  __device__ __forceinline__ int column(int c) const { return 4 * (c < m ? c : c - nx + 2 * m); }
  __device__ __forceinline__ RowAt row(int r) const
  {
    const int k = r < m ? r : r - nz + 2 * m;          // its place among the first and last m rows
    return RowAt{8 * r * m, 4 * (2 * nz * m + k * P - m), 4 * (2 * r * m - nx + 2 * m)};
  }
  __device__ __forceinline__ int in_row(const RowAt& w, int c) const { return 4 * c + (c < m ? w.l : c < nx - m ? w.c : w.r); }
  __device__ __forceinline__ bool straight(int c0, int c1) const { return c0 >= m && c1 < nx - m; }
  __device__ __forceinline__ int at(int r, int c) const { return in_row(row(r), c); }
  static __device__ __forceinline__ int floats(int nx, int nz, int npml)
  {
    const int m = npml + 1, P = (nx - 2 * m + 1) & ~1;
    return 2 * m * (nz + P);
  }
};

// lane l's value from lane l-1 (lane 0: `first`) and from lane l+1
__device__ __forceinline__ float from_before(float first, float x)
{
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(x), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_after(float x)
{
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x130, 0xf, 0xf, true));
}

// One side of the layer, one wave: `lanes` lines from line0, positions 1..len
// along each, as a front in which lane t (of line line0 + t) runs one position
// behind lane t-1.  LR: lines are columns and positions rows; otherwise lines
// are rows and positions columns.  A step of a lane at position j = 1 + k - t
// needs four values: the old one at j+1 of its own line (read FB steps ahead:
// no lane has updated it yet), the old one at j of the next line (what lane
// t+1 reads in the same step; lane `lanes` reads the line beside for that, or,
// FULL, the last lane does where all 64 are lines), the new one at j of the
// line before (the result of lane t-1 in the step before; for lane 0 the line
// beside) and its own result at j-1.  While every line is under way and no
// address changes its stride (most of the front), a step is three adds, one
// multiplication, two lane shifts, two reads and one write.
template <bool LR, bool FULL, class A>
__device__ __forceinline__ void smooth_front(const A acc, int line0, int lanes, int len)
{
  constexpr int FB = 8;
  const int t = threadIdx.x & 63;
  const int tl = imin(t, lanes);
  const bool real = t < lanes;
  // a line's place, and the address of a position (0..len+1) on it
  struct Line { int base; RowAt row; };
  auto line_of = [&](int ln) { return LR ? Line{acc.column(ln), RowAt{}} : Line{0, acc.row(ln)}; };
  auto at = [&](const Line& ln, int pos) {
    const int q = imin(imax(pos, 0), len + 1);
    return LR ? ln.base + q * acc.pitch() : acc.in_row(ln.row, q);
  };
  const Line own = line_of(line0 + tl), before = line_of(line0 - 1), beside = line_of(line0 + lanes);
  // operands of the steps k0 .. k0+FB-1: own line at 2 + k - t, the line
  // before lane 0's at 1 + k, the line after the last one's at 2 + k - lanes;
  // ad: the own line's addresses, the positions updated one step later
  struct Block { float v[FB], first[FB], last[FB]; int ad[FB]; };
  auto read = [&](int k0, Block& b) {
    const int lo = 2 + k0 - lanes, hi = 1 + k0 + FB;   // positions of all lanes
    if (lo >= 0 && hi <= len + 1 && (LR || acc.straight(lo, hi))) {
      const int step = LR ? acc.pitch() : 4;
      const int a = at(own, 2 + k0 - tl), f = at(before, 1 + k0);
#pragma unroll
      for (int u = 0; u < FB; u++) {
        b.ad[u] = LR ? a + u * step : a + 4 * u;
        b.first[u] = acc.get(LR ? f + u * step : f + 4 * u);
      }
    } else {
#pragma unroll
      for (int u = 0; u < FB; u++) {
        b.ad[u] = at(own, 2 + k0 + u - tl);
        b.first[u] = acc.get(at(before, 1 + k0 + u));
      }
    }
#pragma unroll
    for (int u = 0; u < FB; u++) b.v[u] = acc.get(b.ad[u]);
    if (FULL)
#pragma unroll
      for (int u = 0; u < FB; u++) b.last[u] = acc.get(at(beside, 2 + k0 + u - lanes));
  };
  int ab = at(own, 1 - t);                             // address of the position a lane updates
  float prev = acc.get(at(own, 0));
  const int K = len + lanes - 1;
  auto steps = [&](int k0, const Block& cur) {
    float after[FB];
#pragma unroll
    for (int u = 0; u < FB; u++) {
      after[u] = from_after(cur.v[u]);
      if (FULL) after[u] = t == 63 ? cur.last[u] : after[u];
    }
    auto step = [&](int u) {
      const float c = from_before(cur.first[u], prev);
      return LR ? avg4(after[u], c, cur.v[u], prev) : avg4(cur.v[u], prev, after[u], c);
    };
    if (k0 >= lanes - 1 && k0 + FB <= len) {           // every line under way for the whole block
      if (FULL || real)
#pragma unroll
        for (int u = 0; u < FB; u++) {
          prev = step(u);
          acc.set(u ? cur.ad[u - 1] : ab, prev);
        }
    } else {
#pragma unroll
      for (int u = 0; u < FB; u++) {
        const float x = step(u);
        const bool act = real & ((unsigned)(k0 + u - t) < (unsigned)len);
        prev = act ? x : prev;
        if (act) acc.set(u ? cur.ad[u - 1] : ab, x);
      }
    }
    ab = cur.ad[FB - 1];
  };
  Block p, q;
  read(0, p);
  for (int k0 = 0; k0 < K; k0 += 2 * FB) {             // (a block past the end reads clamped positions)
    read(k0 + FB, q);
    steps(k0, p);
    read(k0 + 2 * FB, p);
    steps(k0 + FB, q);
  }
}

// One edge line's recurrence, one lane: x(i) = ((s(i) + x(i-1)) [+ e(i)]) / 4
// for i = 1..n-2 from x(0), in place of s
template <bool COL, class E>
__device__ void smooth_edge(lds_float_t* s, int n, float x, E e)
{
  constexpr int EB = 8;
  float a[EB], b[EB];
  auto read = [&](int i0) {
#pragma unroll
    for (int u = 0; u < EB; u++) {
      a[u] = s[imin(i0 + u, n - 1)];
      b[u] = COL ? 0.0f : e(imin(i0 + u, n - 2));
    }
  };
  read(1);
  for (int i0 = 1; i0 < n - 1; i0 += EB) {
    float ca[EB], cb[EB];
#pragma unroll
    for (int u = 0; u < EB; u++) { ca[u] = a[u]; cb[u] = b[u]; }
    read(i0 + EB);
#pragma unroll
    for (int u = 0; u < EB; u++) {
      x = COL ? 0.25f * (ca[u] + x) : 0.25f * ((ca[u] + x) + cb[u]);
      if (i0 + u < n - 1) s[i0 + u] = x;
    }
  }
}

// The change of one cell, a the value before the sweep and b after it.  The
// reference's test is max |a-b| / |a| > 5e-4 in float division; a change
// clearly past the bound is found by a multiplication (`far`), and only a
// sweep without any divides.
struct Change {
  float far = -1.0e+5f, ratio = -1.0e+5f;
  __device__ __forceinline__ void add(float a, float b) { far = fmaxf(far, __builtin_fmaf(-5.1e-4f, fabsf(a), fabsf(a - b))); }
  __device__ __forceinline__ void divide(float a, float b) { ratio = fmaxf(ratio, fabsf(a - b) / fabsf(a)); }
};
__device__ __forceinline__ float block_max(float m, float* red)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int i = 1; i < SMT / 64; i++) m = fmaxf(m, red[i]);
  return m;
}

// the cells of the ring a thread compares: those of the LDS ring at tid + u
// SMT (with the line beside, which never changes), kept in registers ...
struct OldLds {
  static constexpr int N = (SMOOTH_LDS + SMT - 1) / SMT;
  lds_float_t* p;
  int n;
  float old[N];
  __device__ __forceinline__ void take()
  {
#pragma unroll
    for (int u = 0; u < N; u++) old[u] = (int)threadIdx.x + u * SMT < n ? p[threadIdx.x + u * SMT] : 0.0f;
  }
  template <bool DIVIDE>
  __device__ __forceinline__ void compare(Change& c) const
  {
#pragma unroll
    for (int u = 0; u < N; u++)
      if ((int)threadIdx.x + u * SMT < n) {
        const float b = p[threadIdx.x + u * SMT];
        if (DIVIDE) c.divide(old[u], b);
        else c.add(old[u], b);
      }
  }
};
// ... or the ring in memory against w: a wave per row, 4 loads in flight
struct OldMem {
  gfloat* v;
  gfloat* w;
  int nx, nz, npml;
  template <class F>
  __device__ __forceinline__ void rows(F f) const
  {
    for (int r = threadIdx.x >> 6; r < nz; r += SMT / 64) {
      const bool mid = r >= npml && r < nz - npml;
      const int n = mid ? 2 * npml : nx;
      for (int c0 = threadIdx.x & 63; c0 < n; c0 += 4 * 64) {
        int o[4];
        float a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int c = c0 + 64 * u;
          o[u] = c < n ? r * nx + (mid && c >= npml ? c + nx - 2 * npml : c) : -1;
          a[u] = o[u] >= 0 ? w[o[u]] : 1.0f;
          b[u] = o[u] >= 0 ? v[o[u]] : 1.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) f(o[u], a[u], b[u]);
      }
    }
  }
  __device__ __forceinline__ void take() { rows([&](int o, float, float b) { if (o >= 0) w[o] = b; }); }
  template <bool DIVIDE>
  __device__ __forceinline__ void compare(Change& c) const
  {
    rows([&](int, float a, float b) { if (DIVIDE) c.divide(a, b); else c.add(a, b); });
  }
};

template <bool FULL, class A, class O>
__device__ __forceinline__ void smooth_sweeps(const A acc, O& old, lds_float_t* T, float* red, int nx, int nz, int npml)
{
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  lds_float_t* c0 = T;                                 // columns 0 and nx-1 (nz each), rows 0 and nz-1 (nx each)
  lds_float_t* cN = T + nz;
  lds_float_t* r0 = T + 2 * nz;
  lds_float_t* rN = r0 + nx;
  auto g = [&](int r, int c) { return acc.get(acc.at(r, c)); };
  old.take();
  for (int num = 0; num <= 1000; num++) {
    // left and right layers, then top and bottom layers
    if (wave < 2) smooth_front<true, FULL>(acc, wave ? nx - npml : 1, npml - 1, nz - 2);
    __syncthreads();
    if (wave < 2) smooth_front<false, FULL>(acc, wave ? nz - npml : 1, npml - 1, nx - 2);
    __syncthreads();
    // edges.  Columns: C + E + S + N, rows: C + S + W + E, N and W being the
    // recurrence's own last value
    for (int i = 1 + tid; i < nz - 1; i += SMT) {
      c0[i] = (g(i, 0) + g(i, 1)) + g(i + 1, 0);
      cN[i] = (g(i, nx - 1) + g(i, nx - 2)) + g(i + 1, nx - 1);
    }
    for (int i = 1 + tid; i < nx - 1; i += SMT) {
      r0[i] = g(0, i) + g(1, i);
      rN[i] = g(nz - 1, i) + g(nz - 2, i);
    }
    __syncthreads();
    if (tid == 0) smooth_edge<true>(c0, nz, g(0, 0), [](int) { return 0.0f; });
    else if (tid == 64) smooth_edge<true>(cN, nz, g(0, nx - 1), [](int) { return 0.0f; });
    else if (tid == 128) smooth_edge<false>(r0, nx, g(0, 0), [&](int i) { return g(0, i + 1); });
    else if (tid == 192) smooth_edge<false>(rN, nx, g(nz - 1, 0), [&](int i) { return g(nz - 1, i + 1); });
    __syncthreads();
    for (int i = 1 + tid; i < nz - 1; i += SMT) { acc.set(acc.at(i, 0), c0[i]); acc.set(acc.at(i, nx - 1), cN[i]); }
    for (int i = 1 + tid; i < nx - 1; i += SMT) { acc.set(acc.at(0, i), r0[i]); acc.set(acc.at(nz - 1, i), rN[i]); }
    __syncthreads();
    if (tid == 0) {                                    // corners (none reads another)
      const float a = avg4(g(0, 0), g(1, 0), g(0, 1), g(1, 1));
      const float b = avg4(g(nz - 1, 0), g(nz - 2, 0), g(nz - 1, 1), g(nz - 2, 1));
      const float c = avg4(g(0, nx - 1), g(0, nx - 2), g(1, nx - 1), g(1, nx - 2));
      const float d = avg4(g(nz - 1, nx - 1), g(nz - 2, nx - 1), g(nz - 1, nx - 2), g(nz - 2, nx - 2));
      acc.set(acc.at(0, 0), a); acc.set(acc.at(nz - 1, 0), b);
      acc.set(acc.at(0, nx - 1), c); acc.set(acc.at(nz - 1, nx - 1), d);
    }
    __syncthreads();
    // the largest change against the sweep before, whose values then go
    Change ch;
    old.template compare<false>(ch);
    bool more = block_max(ch.far, red) > 0.0f;
    if (!more) {
      old.template compare<true>(ch);
      more = (double)block_max(ch.ratio, red) > 0.0005;
    }
    old.take();
    if (!more) break;
    __syncthreads();
  }
  __syncthreads();
}

__global__ __launch_bounds__(SMT) void k_pml_smooth(const SmoothWin* __restrict__ wins)
{
  __shared__ float S[SMOOTH_LDS];
  __shared__ float red[SMT / 64];
  const SmoothWin sw = wins[blockIdx.x];
  gfloat* w = GF(sw.w);
  const int nx = sw.nx, nz = sw.nz, npml = sw.npml, tid = threadIdx.x;
  // mirror the interior into the layer: columns (rows 1..nz-2), then rows
  // (columns 1..nx-2, which include the mirrored columns)
  for (int e = tid; e < npml * (nz - 2); e += SMT) {
    const int ix = e % npml, iz = 1 + e / npml;
    w[iz * nx + ix] = w[iz * nx + 2 * npml - ix - 1];
    w[iz * nx + nx - npml + ix] = w[iz * nx + nx - npml - ix - 1];
  }
  __syncthreads();
  for (int e = tid; e < npml * (nx - 2); e += SMT) {
    const int iz = e / (nx - 2), ix = 1 + e % (nx - 2);
    w[iz * nx + ix] = w[(2 * npml - iz - 1) * nx + ix];
    w[(nz - npml + iz) * nx + ix] = w[(nz - npml - iz - 1) * nx + ix];
  }
  __syncthreads();
  lds_float_t* L = (lds_float_t*)S;
  const int rf = RingLds::floats(nx, nz, npml);
  if (rf + 2 * (nx + nz) <= SMOOTH_LDS && npml <= 64) {
    const int m = npml + 1;
    const RingLds acc{L, nx, nz, m, (nx - 2 * m + 1) & ~1};
    for (int e = tid; e < nx * nz; e += SMT) {
      const int r = e / nx, c = e - r * nx;
      if (r < m || r >= nz - m || c < m || c >= nx - m) acc.set(acc.at(r, c), w[e]);
    }
    if (tid < 2 * m && acc.P > nx - 2 * m) L[2 * nz * m + tid * acc.P + nx - 2 * m] = 1.0f;   // the centre's pad
    __syncthreads();
    OldLds old{L, rf};
    smooth_sweeps<false>(acc, old, L + rf, red, nx, nz, npml);
    for (int e = tid; e < nx * nz; e += SMT) {
      const int r = e / nx, c = e - r * nx;
      if (r < npml || r >= nz - npml || c < npml || c >= nx - npml) w[e] = acc.get(acc.at(r, c));
    }
  } else {
    gfloat* v = GF(sw.v);
    for (int e = tid; e < nx * nz; e += SMT) v[e] = w[e];
    __syncthreads();
    OldMem old{v, w, nx, nz, npml};
    if (npml <= 64) smooth_sweeps<false>(RingMem{v, nx}, old, L, red, nx, nz, npml);
    else smooth_sweeps<true>(RingMem{v, nx}, old, L, red, nx, nz, npml);
  }
}

// Phase start of one slot.  FWD: zero both levels of both wavefields and the
// PML pair.  REV: zero both levels of the source velocities (rtm_model.cu:
// 366-372), the receiver set, the PML pair and the imaging accumulators.
__global__ __launch_bounds__(NTHR) void k_phase_init(const ShotDev* __restrict__ shots, int slot, int phase)
{
  const ShotDev s = shots[slot];
  const long long n = (long long)s.frows * s.pitch;
  const long long ni = (long long)s.nzi * s.nxl;
  const long long g0 = (long long)blockIdx.x * NTHR + threadIdx.x, gs = (long long)gridDim.x * NTHR;
  float* f[14] = {s.sp[0], s.sp[1], s.svx[0], s.svx[1], s.svz[0], s.svz[1], s.rp[0], s.rp[1],
                  s.rvx[0], s.rvx[1], s.rvz[0], s.rvz[1], s.q1, s.q2};
  const int first = phase == PH_FWD ? 0 : 2;
  for (long long e = g0; e < n; e += gs)
#pragma unroll
    for (int k = 0; k < 14; k++)
      if (k >= first) (f[k] - s.forg)[e] = 0.0f;
  if (phase == PH_FWD) {
    if (g0 < 12) guard_word(s)[g0] = 0u;               // ... and the strips' max-abs words
    if (s.snap)
      for (long long e = g0; e < 3LL * s.nsnap; e += gs) snap_acc(s)[e] = 0u;   // snapshot max-abs words
  } else {
    for (long long e = g0; e < ni; e += gs) { s.g1[e] = 0.f; s.illum[e] = 0.f; }
    if (s.ic)
      for (long long e = g0; e < ni * (5 + 2 * 61); e += gs) s.ic[e] = 0.f;
  }
}

// receiver wavefield at it = nt-1 (rtm_model.cu:366-372 with the insertion
// of kernel.cu:72-95), written to the level the first reverse step reads
__global__ __launch_bounds__(NTHR) void k_seed_receivers(const ShotDev* __restrict__ shots, int slot)
{
  const ShotDev s = shots[slot];
  const int ir = blockIdx.x * NTHR + threadIdx.x;
  if (ir >= s.nrec) return;
  const int it = s.nt - 1;
  const float rv = (it <= s.cut[ir]) ? 0.0f : s.rec[(size_t)it * s.nrec + ir];
  float* rp = ((s.nt - 2) & 1) ? s.rp[1] : s.rp[0];
  rp[(size_t)s.npml * s.pitch + s.rcol0 + ir] = s.dt * rv;
}

// taper and stack shots into the FP64 images, one image cell per thread,
// shots in the given order (kernel.cu:1556-1615, rtm_model.cu:462-488)
struct StackShot { const float* g1; const float* illum; const float* taper; int nx1, nxl; };

__global__ __launch_bounds__(NTHR) void k_stack(const StackShot* __restrict__ sh, int nsh, int nx, int nz,
                                                 double* __restrict__ img1, double* __restrict__ img2s,
                                                 double* __restrict__ ill)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e >= (long long)nx * nz) return;
  const int iz = (int)(e / nx), ix = (int)(e - (long long)iz * nx);
  double a1 = img1[e], a2 = img2s[e], a3 = ill[e];
  for (int k = 0; k < nsh; k++) {
    const StackShot q = sh[k];
    const int c = ix - q.nx1;
    if (c < 0 || c >= q.nxl) continue;
    const float t = q.taper[c];
    const float g = q.g1[(size_t)iz * q.nxl + c] * t;
    const float il = q.illum[(size_t)iz * q.nxl + c] * t;
    a2 += (double)g / ((double)il + 1.0e-6);
    a1 += (double)g;
    a3 += (double)il;
  }
  img1[e] = a1; img2s[e] = a2; ill[e] = a3;
}

// ------------------------------------------------- other imaging conditions --
// After reverse step `step` (kernel.cu:1417-1529, one thread per interior
// cell of a slot): wavefield decomposition, Poynting-vector angle bins and the
// energy norm, from the new fields (level (it+1)&1) and the fields before the
// step (level it&1).  The reference's quirks are kept: vx and vxs are read at
// the p index (stride nxp in an array of rows nxp-1, kernel.cu:1431,1468) and
// the source Poynting vector takes the receiver's vz (kernel.cu:1469).  Each
// expression is evaluated as nvcc contracts it by default (a*b + c*d ->
// fma(a, b, c*d); accumulations -> fma), with the float / double mixing of
// the reference's double literals.  Off the hot path: launched only when the
// job asks for these images.
__global__ __launch_bounds__(NTHR) void k_ic(const ShotDev* __restrict__ shots, const int* __restrict__ slots, int step)
{
  const ShotDev& s = shot_of(shots, slots[blockIdx.y]);
  if (!s.ic) return;
  const int nxl = s.nxl, nn = s.nzi * nxl;
  const int e = blockIdx.x * NTHR + threadIdx.x;
  if (e >= nn) return;
  const int iz = e / nxl + s.npml, ix = e - (e / nxl) * nxl + s.npml;   // padded cell
  const int nxp = s.nxp, pitch = s.pitch;
  const int it = s.it_off + s.it_dir * step;
  const bool odd = it & 1;                              // the step read level it&1, wrote the other
  const float* psn = odd ? s.sp[0] : s.sp[1];
  const float* pso = odd ? s.sp[1] : s.sp[0];
  const float* prn = odd ? s.rp[0] : s.rp[1];
  const float* pro = odd ? s.rp[1] : s.rp[0];
  const float* vxs_f = odd ? s.svx[0] : s.svx[1];
  const float* vzs_f = odd ? s.svz[0] : s.svz[1];
  const float* vxr_f = odd ? s.rvx[0] : s.rvx[1];
  const float* vzr_f = odd ? s.rvz[0] : s.rvz[1];
  const long long id = (long long)iz * pitch + ix;
  // the p index read in an array of rows nxp-1: row q/(nxp-1), column
  // q%(nxp-1); past that array's end (windows taller than about npml*nxp, where
  // the reference reads out of bounds) the value is taken as 0
  const int q = iz * nxp + ix, qr = q / (nxp - 1), qc = q - qr * (nxp - 1);
  const bool qin = qr < s.nzp;
  const long long iq = qin ? (long long)qr * pitch + qc : 0;
  const float ps = psn[id], p = prn[id];
  const float vxs = qin ? vxs_f[iq] : 0.0f, vzs = vzs_f[id], vxr = qin ? vxr_f[iq] : 0.0f, vzr = vzr_f[id];
  const int mr = imin(imax(iz - s.mz0, 0), s.mzn - 1), mc = s.mx0 + imin(imax(ix - s.mxs, 0), s.mxn - 1);
  const float vv = s.vv[(size_t)mr * s.mpitch + mc];
  float* ic = s.ic;
  // cuda_wavefield_decomposition (kernel.cu:1417-1450)
  const float vtxs = -ps * vxs, vtzs = -ps * vzs, vtxr = -p * vxr, vtzr = -p * vzr;
  const float psu = vtzs < 0 ? ps : 0.0f, psd = vtzs > 0 ? ps : 0.0f, psl = vtxs < 0 ? ps : 0.0f, psr = vtxs > 0 ? ps : 0.0f;
  const float pu = vtzr < 0 ? p : 0.0f, pd = vtzr > 0 ? p : 0.0f, pl = vtxr < 0 ? p : 0.0f, pr = vtxr > 0 ? p : 0.0f;
  // An accumulator plane is read and written only where neither factor of its
  // product is zero.  There the reference's fma(a, b, c) adds +-0 and returns
  // c unchanged, except that it can turn a -0 into +0.  A plane holds -0 only
  // after an fma whose exact product was a negative value too small for a
  // float, so the skipped form can differ from the reference's only in the
  // sign of a zero.  The stacks sum the planes in FP64 from +0
  // (+0 + -0 = +0), so the images are the same bit for bit.  The up/down
  // (left/right) conditions exclude each other, and a wave travelling one way
  // keeps them constant over a region, so whole cache lines are skipped.
  if (psu != 0.0f && pd != 0.0f) ic[e] = __builtin_fmaf(psu, pd, ic[e]);
  if (psd != 0.0f && pu != 0.0f) ic[nn + e] = __builtin_fmaf(psd, pu, ic[nn + e]);
  if (psl != 0.0f && pr != 0.0f) ic[2 * nn + e] = __builtin_fmaf(psl, pr, ic[2 * nn + e]);
  if (psr != 0.0f && pl != 0.0f) ic[3 * nn + e] = __builtin_fmaf(psr, pl, ic[3 * nn + e]);
  // cuda_poynting (kernel.cu:1452-1488).  Both bins add a multiple of ps*p:
  // where that product is zero (either wavefield zero, or the product
  // underflows) they add +-0, so the bins keep their value up to the sign of
  // a zero, as above.  The angle, its cosine and sine and the FP64 quotient
  // are then not needed.
  const float ksx = ps * vxs, ksz = ps * vzr, krx = p * vxr, krz = p * vzr;
  if (ps * p != 0.0f) {
    const float qd = sqrtf(__builtin_fmaf(ksx, ksx, ksz * ksz) * __builtin_fmaf(krx, krx, krz * krz));
    float w = (float)((double)__builtin_fmaf(ksx, krx, ksz * krz) / (qd > 0 ? (double)qd : 1.0e-6));
    if (w >= -1.0 && w <= 1.0) {
      const double pi = 3.1415926535897932;
      w = (float)(0.5 * (double)acosf(w));
      w = (float)(pi / 2.0 - (double)w);
      if (w > 0 && w <= pi / 3.0) {
        const float dw = (float)(pi / 180);
        const size_t ib = (size_t)(int)(w / dw) * nn + e;
        float* g31 = ic + 5 * (size_t)nn;
        float* g32 = ic + 66 * (size_t)nn;
        g31[ib] = __builtin_fmaf(ps * p, cosf(w), g31[ib]);
        g32[ib] = (float)((double)g32[ib] + (double)(ps * p) * 16.0 * pi * (double)sqrtf(vv) / (double)sinf(w));
      }
    }
  }
  // cuda_energynorm (kernel.cu:1489-1529)
  const float psx = (float)(0.5 * (double)(psn[id + 1] - psn[id - 1]) / (double)s.dx);
  const float psz = (float)(0.5 * (double)(psn[id + pitch] - psn[id - pitch]) / (double)s.dz);
  const float px = (float)(0.5 * (double)(prn[id + 1] - prn[id - 1]) / (double)s.dx);
  const float pz = (float)(0.5 * (double)(prn[id + pitch] - prn[id - pitch]) / (double)s.dz);
  const float t = -(ps - pso[id]) * (p - pro[id]) / (s.dt * s.dt * vv);
  const float en = __builtin_fmaf(psz, pz, __builtin_fmaf(psx, px, t));
  // a sum of floats is +0 on exact cancellation and never underflows to 0,
  // so this plane never holds -0 and adding +-0 leaves it bit for bit
  if (en != 0.0f) ic[4 * nn + e] = ic[4 * nn + e] + en;
}

// one shot's other images into the FP64 stacks (kernel.cu:1530-1579): g2 as
// the four decomposed products summed, g3 / g3_true as the 61 bins summed,
// each tapered, then normalised by the tapered illumination (image3s..5s)
// or not (image3m..5m, imagetrue)
struct StackIc { const float* ic; const float* illum; const float* taper; int nx1, nxl; };
__global__ __launch_bounds__(NTHR) void k_stack_ic(const StackIc* __restrict__ sh, int nx, int nz, double* __restrict__ i7)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e >= (long long)nx * nz) return;
  const int iz = (int)(e / nx), ix = (int)(e - (long long)iz * nx);
  const StackIc q = *sh;
  const int c = ix - q.nx1;
  if (c < 0 || c >= q.nxl) return;
  const size_t nn = (size_t)nz * q.nxl, ip = (size_t)iz * q.nxl + c;
  const float* ic = q.ic;
  const float t = q.taper[c];
  float g3 = 0.0f, g3t = 0.0f;
  for (int iw = 0; iw <= 60; iw++) { g3 += ic[(5 + iw) * nn + ip]; g3t += ic[(66 + iw) * nn + ip]; }
  const float g2 = ((ic[ip] + ic[nn + ip]) + ic[2 * nn + ip]) + ic[3 * nn + ip];
  const float il = q.illum[ip] * t;
  const float g[3] = {g2 * t, g3 * t, ic[4 * nn + ip] * t};
  const size_t n = (size_t)nx * nz;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    i7[k * n + e] += (double)g[k] / ((double)il + 1.0e-6);
    i7[(3 + k) * n + e] += (double)g[k];
  }
  i7[6 * n + e] += (double)(g3t * t);
}

// final products: fp32 images from the FP64 stacks, the Laplacian-filtered
// image (laplacefd1d, image_function.cpp:44-79, integer spacings) and the
// multi-shot normalised image (kernel.cu:1580-1590)
__global__ __launch_bounds__(NTHR) void k_round(const double* __restrict__ a, float* __restrict__ o, long long n)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e < n) o[e] = (float)a[e];
}

__global__ __launch_bounds__(NTHR) void k_laplace(const float* __restrict__ im, float* __restrict__ out, int nx, int nz,
                                                   int dxi, int dzi)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e >= (long long)nx * nz) return;
  const int iz = (int)(e / nx), ix = (int)(e - (long long)iz * nx);
  if (ix == 0 || iz == 0 || ix == nx - 1 || iz == nz - 1) { out[e] = 0.0f; return; }
  const float c = im[e];
  const float t1 = (float)(((double)(im[e + 1] + im[e - 1]) - 2.0 * (double)c) / (double)(dxi * dxi));
  const float t2 = (float)(((double)(im[e + nx] + im[e - nx]) - 2.0 * (double)c) / (double)(dzi * dzi));
  out[e] = t1 + t2;
}

__global__ __launch_bounds__(NTHR) void k_norm_multi(const float* __restrict__ sg, const float* __restrict__ ss,
                                                      float* __restrict__ out, long long n)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e < n) out[e] = (float)((double)sg[e] / ((double)ss[e] + 1.0e-6));
}

__global__ __launch_bounds__(NTHR) void k_zero_f64(double* __restrict__ a, long long n)
{
  const long long e = (long long)blockIdx.x * NTHR + threadIdx.x;
  if (e < n) a[e] = 0.0;
}

// one wave that lasts `ticks` of the constant 100 MHz clock (and ends after a
// bounded number of reads of it whatever the clock does): t[0], t[1] = its
// start and end
__global__ void k_clock(long long* __restrict__ t, long long ticks)
{
  const long long b = wall_clock64();
  long long e = b;
  for (int i = 0; i < 100000 && e - b < ticks; i++) e = wall_clock64();
  if (threadIdx.x == 0) {
    t[0] = b;
    t[1] = e;
  }
}

// Wavefield guard: the device form of the reference's max|p| print every
// ntsnap steps (rtm_model.cu:271-273, 324, 415).  The largest |p| of each
// listed slot's pressure as written by step `step` (it = it_off + it_dir *
// step wrote level (it+1)&1; the source field, and in the reverse phase also
// the receiver field) goes into the slot's guard word and into *flag as float
// bits: non-negative floats order as their bits, and an infinity (0x7F800000)
// or a NaN (0x7FC00000 and up) compares above every finite value, so the host
// detects a blow-up (unstable dt, bad model) from one word.  Grid: (slots, GW).
__global__ __launch_bounds__(NTHR) void k_guard(const ShotDev* __restrict__ shots, const int* __restrict__ slots,
                                                 int step, unsigned int* __restrict__ flag)
{
  __shared__ unsigned int red[NTHR / 64];
  const ShotDev& s = shot_of(shots, slots[blockIdx.x]);
  const int it = s.it_off + s.it_dir * step;
  const bool lev = (it + 1) & 1;
  const float* ps = lev ? s.sp[1] : s.sp[0];
  const float* pr = lev ? s.rp[1] : s.rp[0];
  const bool rev = s.phase == PH_REV;
  // one wave per row, rows dealt over the waves of gridDim.y workgroups; a
  // lane takes GU columns 64 apart per iteration (independent loads in
  // flight, no index division, lanes busy on windows of any width)
  constexpr int GU = 4, WPB = NTHR / 64;
  const int lane = threadIdx.x & 63, nxp = s.nxp;
  unsigned int m = 0u;
  for (int iz = blockIdx.y * WPB + (threadIdx.x >> 6); iz < s.nzp; iz += gridDim.y * WPB) {
    const gfloat* rs = GCF(ps) + (long long)iz * s.pitch;
    const gfloat* rr = GCF(pr) + (long long)iz * s.pitch;
    for (int x0 = lane; x0 < nxp; x0 += GU * 64) {
      unsigned int a[GU];
#pragma unroll
      for (int u = 0; u < GU; u++) {
        const int ix = x0 + u * 64;
        a[u] = ix < nxp ? __float_as_uint(rs[ix]) & 0x7FFFFFFFu : 0u;
        if (rev && ix < nxp) a[u] = max(a[u], __float_as_uint(rr[ix]) & 0x7FFFFFFFu);
      }
#pragma unroll
      for (int u = 0; u < GU; u++) m = max(m, a[u]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned int)__shfl_xor((int)m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NTHR / 64; w++) m = max(m, red[w]);
    atomicMax(guard_word(s), m);
    if (flag) atomicMax(flag, m);
  }
}

// advance the time origin of the slots of a captured chunk of `k` steps so
// that replaying the same graph continues where the last replay stopped
__global__ void k_bump(ShotDev* __restrict__ shots, const int* __restrict__ slots, int nslots, int k)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nslots) {
    ShotDev* s = &shots[slots[i]];
    s->it_off += s->it_dir * k;
  }
}

// =========================================================== launchers ==
#include "rtm_launch.h"

static inline int grid8(int ntiles) { return ((ntiles + 7) / 8) * 8; }

template <int G, int RPT>
static hipError_t launch_step_t(const LaunchArgs& a, int phase, hipStream_t st)
{
  const int n = a.ntiles * Geo<G, RPT, false, false>::SPLIT;
  const dim3 b(64 * G), gf(grid8(n)), gr(16 * (((n + 7) / 8 + RGRP - 1) / RGRP * RGRP));
  auto go = [&](auto cached, auto s16) {
    if (phase == PH_FWD) hipLaunchKernelGGL((k_fwd<G, RPT, cached.value, s16.value>), gf, b, 0, st, a);
    else hipLaunchKernelGGL((k_rev<G, RPT, cached.value, s16.value>), gr, b, 0, st, a);
  };
  if (a.cached && a.s16) go(std::true_type{}, std::true_type{});
  else if (a.cached) go(std::true_type{}, std::false_type{});
  else if (a.s16) go(std::false_type{}, std::true_type{});
  else go(std::false_type{}, std::false_type{});
  return hipGetLastError();
}

hipError_t rtm_launch_step(const LaunchArgs& a, int phase, int tz, hipStream_t st)
{
  if (a.ntiles <= 0) return hipSuccess;
  switch (tz) {
    // 16 rows are the height of the smallest launches, whose time is a
    // workgroup's own chain of phases (about 6 of 8 us a step).  Up to one
    // tile per CU two workgroups of 8 rows share a tile: a reverse step has two
    // fields, so whole tiles leave some CUs with two workgroups and others idle.
    // Up to one and a half, 8 waves of 2 rows; past that the 4 x 4 form does
    // less halo work a wave.  us per forward / reverse step, halves against 8 x
    // 2: one 184 x 124 window (24 tiles) 7.5 / 7.7 against 7.8 / 8.3, 480 x 280
    // (144) 7.8 / 10.4 against 8.0 / 11.8, two of 265 x 320 a launch (200) 9.0 /
    // 11.7 against 8.9 / 13.2, 401 x 612 (273) 8.6 / 11.2 against 8.4 / 10.7;
    // 8 x 2 against 4 x 4 (with a strip save of its own): 273 tiles 14.3 /
    // 10.9 against 15.4 / 12.3, 546 15.9 / 18.2 against 16.0 / 15.1
    case 16:
      if (a.ntiles <= 256) return launch_step_t<4, 2>(a, phase, st);
      return a.ntiles <= 384 ? launch_step_t<8, 2>(a, phase, st) : launch_step_t<4, 4>(a, phase, st);
    case 32: return launch_step_t<4, 8>(a, phase, st);
    case 64: return launch_step_t<8, 8>(a, phase, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t rtm_launch_clock(long long* t, long long ticks, hipStream_t st)
{
  hipLaunchKernelGGL(k_clock, dim3(1), dim3(64), 0, st, t, ticks);
  return hipGetLastError();
}

hipError_t rtm_launch_image(const ShotDev* shots, const int* slots, int nslots, int it, hipStream_t st)
{
  if (nslots <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_image, dim3(nslots, std::min(64, std::max(8, 2048 / nslots))), dim3(NTHR), 0, st, shots, slots, it);
  return hipGetLastError();
}

hipError_t rtm_launch_quant16(const ShotDev* shots, const int* slots, int nslots, int step, hipStream_t st)
{
  if (nslots <= 0) return hipSuccess;
  // about 1024 workgroups in all, at most 32 per block (a block of the widest
  // windows holds 41 K values)
  hipLaunchKernelGGL(k_quant16, dim3(4 * nslots, std::min(32, std::max(4, 256 / nslots))), dim3(NTHR), 0, st, shots,
                     slots, nslots, step);
  return hipGetLastError();
}

hipError_t rtm_launch_phase_init(const ShotDev* shots, int slot, int phase, int nblocks, hipStream_t st)
{
  hipLaunchKernelGGL(k_phase_init, dim3(nblocks), dim3(NTHR), 0, st, shots, slot, phase);
  return hipGetLastError();
}

hipError_t rtm_launch_model_prep(const float* rho, const float* vv, float* ib, float* kk, long long n, hipStream_t st)
{
  const long long nb = (n + NTHR - 1) / NTHR;
  hipLaunchKernelGGL(k_model_prep, dim3((unsigned)(nb < 4096 ? nb : 4096)), dim3(NTHR), 0, st, rho, vv, ib, kk, n);
  return hipGetLastError();
}

hipError_t rtm_launch_seed(const ShotDev* shots, int slot, int nrec, hipStream_t st)
{
  if (nrec <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_seed_receivers, dim3((nrec + NTHR - 1) / NTHR), dim3(NTHR), 0, st, shots, slot);
  return hipGetLastError();
}

hipError_t rtm_launch_ic(const ShotDev* shots, const int* slots, int nslots, int step, int max_cells, hipStream_t st)
{
  if (nslots <= 0 || max_cells <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ic, dim3((unsigned)((max_cells + NTHR - 1) / NTHR), (unsigned)nslots), dim3(NTHR), 0, st,
                     shots, slots, step);
  return hipGetLastError();
}

hipError_t rtm_launch_stack_ic(const void* sh, int nx, int nz, double* i7, hipStream_t st)
{
  const long long n = (long long)nx * nz;
  hipLaunchKernelGGL(k_stack_ic, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, (const StackIc*)sh, nx, nz, i7);
  return hipGetLastError();
}

hipError_t rtm_launch_stack(const void* sh, int nsh, int nx, int nz, double* i1, double* i2, double* il, hipStream_t st)
{
  const long long n = (long long)nx * nz;
  hipLaunchKernelGGL(k_stack, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st,
                     (const StackShot*)sh, nsh, nx, nz, i1, i2, il);
  return hipGetLastError();
}

hipError_t rtm_launch_round(const double* a, float* o, long long n, hipStream_t st)
{
  hipLaunchKernelGGL(k_round, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, a, o, n);
  return hipGetLastError();
}

hipError_t rtm_launch_laplace(const float* im, float* out, int nx, int nz, int dxi, int dzi, hipStream_t st)
{
  const long long n = (long long)nx * nz;
  hipLaunchKernelGGL(k_laplace, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, im, out, nx, nz, dxi, dzi);
  return hipGetLastError();
}

hipError_t rtm_launch_norm_multi(const float* sg, const float* ss, float* out, long long n, hipStream_t st)
{
  hipLaunchKernelGGL(k_norm_multi, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, sg, ss, out, n);
  return hipGetLastError();
}

hipError_t rtm_launch_zero_f64(double* a, long long n, hipStream_t st)
{
  hipLaunchKernelGGL(k_zero_f64, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, a, n);
  return hipGetLastError();
}

hipError_t rtm_launch_snap(const ShotDev* shots, const int* slots, int nslots, int phase, int step, int snap_fmt,
                           hipStream_t st)
{
  if (nslots <= 0) return hipSuccess;
  // about 2048 workgroups when a snapshot is taken (each returns at once on
  // the other steps): 42 per block for 16 slots, 8 for 200
  const int gy = std::min(64, std::max(8, 2048 / (3 * nslots)));
  const dim3 g(3 * nslots, gy), b(NTHR);
  if (phase == PH_FWD) {
    if (snap_fmt != ST_F32) hipLaunchKernelGGL(k_snap_max, g, b, 0, st, shots, slots, step);
    hipLaunchKernelGGL(k_snap_q, g, b, 0, st, shots, slots, step);
  } else {
    hipLaunchKernelGGL(k_snap_load, g, b, 0, st, shots, slots, step);
  }
  return hipGetLastError();
}

hipError_t rtm_launch_gauss_smooth(const float* in, float* out, int nz, int nx, int nsp, const double* wt, double norm,
                                   hipStream_t st)
{
  const long long n = (long long)nz * nx;
  hipLaunchKernelGGL(k_gauss_smooth, dim3((unsigned)((n + NTHR - 1) / NTHR)), dim3(NTHR), 0, st, in, out, nz, nx, nsp,
                     wt, norm);
  return hipGetLastError();
}

hipError_t rtm_launch_pml_smooth(const void* wins, int n, hipStream_t st)
{
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pml_smooth, dim3(n), dim3(SMT), 0, st, (const SmoothWin*)wins);
  return hipGetLastError();
}

hipError_t rtm_launch_guard(const ShotDev* shots, const int* slots, int nslots, int step, unsigned int* flag,
                            hipStream_t st)
{
  if (nslots <= 0) return hipSuccess;
  // about 2048 workgroups in all: 10 per slot for 200 survey slots, 64 for
  // a few wide ones
  const int gy = nslots >= 256 ? 8 : std::min(64, std::max(8, 2048 / nslots));
  hipLaunchKernelGGL(k_guard, dim3(nslots, gy), dim3(NTHR), 0, st, shots, slots, step, flag);
  return hipGetLastError();
}

hipError_t rtm_launch_bump(ShotDev* shots, const int* slots, int nslots, int k, hipStream_t st)
{
  hipLaunchKernelGGL(k_bump, dim3((nslots + 63) / 64), dim3(64), 0, st, shots, slots, nslots, k);
  return hipGetLastError();
}
