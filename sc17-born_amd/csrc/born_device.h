// Device-side building blocks of the Born propagator on CDNA4 (gfx950).
//
// march_kernel advances one or two pressure fields by one leapfrog step of
// the 8th-order constant-density acoustic operator.  A block owns a tile of
// the xy plane and a chunk of z planes, which it marches.  z neighbours live
// in a 9-deep register queue per cell; x/y neighbours of the current plane
// come from an LDS tile with a 4-cell halo.  The loop is software pipelined:
// the loads of plane z+1 (the queue's new leading plane, the LDS halo and the
// op's pointwise inputs) are issued before plane z is computed.
//
// What bounds it (MI355X, FP32).  At 304^3 memory: with the arithmetic and the
// LDS exchange left out a launch takes as long.  At 160^3 (fields that fit
// the 256 MB memory-side cache) a plane's loads and its arithmetic take about
// as long as each other, and the 8 planes that a chunk shares with its
// neighbours weigh.  At 64^3 latency: the launch, the chunk's first loads and
// the planes marched one after the other.
//   - A plane needs one barrier, not two: the LDS tile is double, and the halo
//     loaded kH planes ahead waits in the loading thread's own LDS place.
//   - Addresses are a scalar base that moves by a plane plus a lane offset
//     that does not change over the march: one addition per load.
//   - Chunks are marched up and down in turn, and turned round from one step
//     to the next (Grid::back): neighbours read the planes they share
//     together, and a step starts with the planes the last one ended with.
//   - Four cells per lane (16-byte loads) where nx allows; the smallest tiles
//     are one wavefront, whose barrier waits for nobody.
//   - The Laplacians go row by row and field by field where registers bound
//     the wavefronts (Op::LEAN).
// Together, fastest shape, us per step: 304^3 adjoint state 142.8 -> 130.9,
// reference adjoint 233 -> 200, source propagation 79.9 -> 72.0, 24-bit
// forward 194 -> 158; 160^3 forward 32.6 -> 30.0, adjoint state 24.9 -> 21.1,
// source propagation 15.7 -> 12.6.
//
// What the step does with the Laplacian is supplied by an immutable "op"
// functor inlined into the kernel: sponge, source injection, Born scatter,
// receiver extraction/injection and imaging are fused into the same pass.
// Ops are passed by value as kernel arguments and never written, so their
// pointers stay in the global address space (global_load/store, not flat).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace born {

constexpr int kTX = 64;  // x cells per tile (one wavefront)
constexpr int kH = 4;    // stencil half-width

// Stencil taps in the reference's order and axis convention
// (base/cpu_prop.cc:6-18, 233-248, 298-326): cx = fast axis, cy = middle,
// cz = slow.
struct Taps {
  float c0;
  float cx[4], cy[4], cz[4];
};

struct Grid {
  int nx, ny, nz;
  int ntx, nty, ntz;  // tiles along x, y and z chunks
  int zc;             // planes per z chunk
  uint32_t plane;     // nx*ny
  int back;           // 1: every z chunk is marched the other way; 2: all are marched up
};

// Per-axis sponge factors: bound[min(edge_x, edge_y, edge_z)] equals
// min(bx[x], by[y], bz[z]) because the table grows with the edge distance.
struct Sponge {
  const float *bx, *by, *bz;
};

// Point sources: (x, y, z, 0) per point in device memory.
struct Points {
  const int4 *p;
  int n;
};

// Receivers: every receiver plane z has a slot; rmap[slot][y][x] is the first
// receiver at that cell (or -1), rnext[] chains receivers sharing a cell.
//
// A step touches one value per receiver cell, indexed by the cell's first
// receiver: the forward leaves the new r there (the receivers' samples of a
// window of steps are added to the traces afterwards, rec_accum_kernel), the
// adjoints take from there what is injected (computed for a window of steps
// beforehand, rec_inject_kernel).  Reading and writing the eight trace
// samples of a receiver inside the step was a chain of three dependent loads
// and a store per cell of a lane that the whole launch waited for.
struct RecMap {
  const int *plane_slot;  // [nz], -1 when the plane has no receiver
  const int *rmap;        // [nslots][ny][nx]
  const int *rnext;       // [nrec]
  int nrec;
  int ntb;                // trace length (nt_big)
  int shared;             // some cell holds more than one receiver
};

// The address `b` bytes (uniform, a scalar addition) past p, and the T at byte
// offset o (a lane's, 32 bits) from a base: one load with a scalar base and
// a vector offset.
__device__ __forceinline__ const char *adv(const void *p, uint64_t b) {
  return (const char *)p + b;
}
template <class T>
__device__ __forceinline__ const T &ldb(const char *p, uint32_t o) {
  return *(const T *)(p + (uint64_t)o);
}
// element at 32-bit element offset o (fields are < 2^30 cells)
template <class T>
__device__ __forceinline__ T &at(T *p, uint32_t o) {
  return *(T *)((char *)p + (uint64_t)(o * (uint32_t)sizeof(T)));
}
template <class T>
__device__ __forceinline__ const T &at(const T *p, uint32_t o) {
  return *(const T *)((const char *)p + (uint64_t)(o * (uint32_t)sizeof(T)));
}

// ---- Stores the compiler's wait-counter model does not see.  Loads and
// stores share one counter (vmcnt) on this architecture and the compiler
// takes a counter with both pending as unordered, so any wait for a load
// would drain every load in flight.  As inline asm the step kernels' stores
// are invisible to it: a wait for a load issued two steps earlier can leave
// the previous step's loads in flight.  That wait stays exact because a
// wavefront's loads return in order, so a vmcnt that counts only the loads
// issued after the one waited for covers it (pending stores only make the
// wait longer).  No step kernel reads what it stores before the launch ends,
// and a store of at most 8 bytes reads its data registers at issue.  The
// base is a wave-uniform pointer (scalar registers), off a byte offset.
// A vector memory instruction that reads a scalar register written by a
// vector instruction (v_readlane, as in a reload of a spilled scalar) needs
// 5 wait states before it, which the compiler does not insert for inline
// asm: each store starts with s_nop 4.  NT adds the non-temporal hint (where
// it pays is measured at the ops).
template <bool NT>
__device__ __forceinline__ void st_b8(void *p, uint32_t off, unsigned char v) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_store_byte %0, %1, %2 nt"
                 : : "v"(off), "v"((uint32_t)v), "s"(p) : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_store_byte %0, %1, %2"
                 : : "v"(off), "v"((uint32_t)v), "s"(p) : "memory");
}
template <bool NT>
__device__ __forceinline__ void st_b16(void *p, uint32_t off, unsigned short v) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_store_short %0, %1, %2 nt"
                 : : "v"(off), "v"((uint32_t)v), "s"(p) : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_store_short %0, %1, %2"
                 : : "v"(off), "v"((uint32_t)v), "s"(p) : "memory");
}
template <bool NT>
__device__ __forceinline__ void st_b32(void *p, uint32_t off, uint32_t v) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_store_dword %0, %1, %2 nt"
                 : : "v"(off), "v"(v), "s"(p) : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_store_dword %0, %1, %2"
                 : : "v"(off), "v"(v), "s"(p) : "memory");
}
template <bool NT>
__device__ __forceinline__ void st_b64(void *p, uint32_t off, uint64_t v) {
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2 nt"
                 : : "v"(off), "v"(v), "s"(p) : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2"
                 : : "v"(off), "v"(v), "s"(p) : "memory");
}

// A store of more than 8 bytes reads its data registers over more than one
// cycle: one wait state before they may be written again.
template <bool NT>
__device__ __forceinline__ void st_b128(void *p, uint32_t off, uint4 v) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 w = {v.x, v.y, v.z, v.w};
  if constexpr (NT)
    asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 nt\n\ts_nop 1"
                 : : "v"(off), "v"(w), "s"(p) : "memory");
  else
    asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2\n\ts_nop 1"
                 : : "v"(off), "v"(w), "s"(p) : "memory");
}

// VX consecutive floats in LDS (VX = 2, 4: aligned to all of them)
template <int VX>
__device__ __forceinline__ void ld_lds(const float *p, float (&v)[VX]) {
  if constexpr (VX == 1) {
    v[0] = p[0];
  } else {
    typedef float vec __attribute__((ext_vector_type(VX)));
    const vec w = *(const vec *)p;
#pragma unroll
    for (int i = 0; i < VX; i++) v[i] = w[i];
  }
}
template <int VX>
__device__ __forceinline__ void st_lds(float *p, const float (&v)[VX]) {
  if constexpr (VX == 1) {
    p[0] = v[0];
  } else {
    typedef float vec __attribute__((ext_vector_type(VX)));
    vec w;
#pragma unroll
    for (int i = 0; i < VX; i++) w[i] = v[i];
    *(vec *)p = w;
  }
}

// Block barrier for LDS: the block's LDS accesses complete, then s_barrier.
// __syncthreads also fences global memory, which waits for every load in
// flight; the step kernels share nothing through global memory in a launch.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

// Scale for a level whose magnitude is at most bound: a power of two that
// maps bound to [8192, 16384), 4x below the FP16 maximum.  Relative precision
// of FP16 does not depend on the scale; the scale only keeps the level inside
// the normal range (a value 2^28 below the bound is still normal).
__device__ __forceinline__ float level_scale(float bound) {
  if (!(bound > 0.f)) return 1.f;
  int e;
  frexpf(bound, &e);  // bound < 2^e
  e = min(max(14 - e, -120), 120);
  return ldexpf(1.f, e);
}

// Scales of the stored levels of one FP16 field.  Level k lives in slot k % 4:
// scale[s] (stored = value * scale) and maxb[s], the largest |value| of the
// level as float bits (non-negative floats order like their bits).  The step
// that reads levels k (cur) and k-1 (old) and writes k+1 (nxt) derives the
// scale of k+1 from a bound on |level k+1| (gain * max k + max k-1 +
// injections), accumulates max |level k+1| with atomics, and clears slot
// k+2, which the following step fills.
struct Ring {
  float *scale;
  unsigned *maxb;
};
struct Slots {
  int cur, old, nxt, clr;
};
__device__ __forceinline__ float ring_max(const Ring &r, int s) {
  return __uint_as_float(r.maxb[s]);
}

// Read-only tables indexed by a uniform value (sponge factor of a plane, the
// receiver slot of a plane, source points): read through the constant
// address space, so they become scalar loads, tracked apart from the vector
// loads of the wavefields.  A vector load issued after the next plane's
// prefetch would otherwise make the wait for it a wait for the prefetch too.
template <class T>
__device__ __forceinline__ T ldc(const T *p, long long i) {
  static_assert(sizeof(T) % 4 == 0, "32-bit words");
  typedef const __attribute__((address_space(4))) uint32_t *cwords;
  const cwords w = (cwords)(p + i);
  uint32_t u[sizeof(T) / 4];
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 4); k++) u[k] = w[k];
  T v;
  __builtin_memcpy(&v, u, sizeof(T));
  return v;
}

// The hardware hands block h to XCD h % 8.  Give every XCD a contiguous range
// of logical tiles so that tiles sharing halo rows share an L2.
__device__ __forceinline__ int xcd_remap(int h, int nb) {
  const int q = nb / 8, r = nb % 8;
  const int xcd = h % 8, k = h / 8;
  return xcd * q + (xcd < r ? xcd : r) + k;
}

// Arithmetic with its rounding fixed.  The compiler fuses a product into a
// following sum where it can; these products and sums are never fused, and
// fma_r always is, so every kernel that computes a cell in the same terms
// gets the same bits.
__device__ __forceinline__ float add_r(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
__device__ __forceinline__ float mul_r(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ double add_r(double a, double b) {
#pragma clang fp contract(off)
  return a + b;
}
__device__ __forceinline__ double mul_r(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float fma_r(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// One leapfrog update b * (V lap + 2 cur - b old) (cpu_prop.cc:31-53 with
// the damping of cpu_prop.cc:141-165), as fma(V, lap, cur) + cur - b old.
__device__ __forceinline__ float leap(float b, float v, float lap, float cur, float old) {
  return mul_r(b, fma_r(-b, old, add_r(fma_r(v, lap, cur), cur)));
}

// The Born source term of a forward step and the scatter operand kept for
// the exact adjoint.  Scatter 0 (image): r += 1e-6 s m in double, the
// reference's double literal (cpu_prop.cc:220); scatter 1 (dV): sigma =
// b L(s), r += m sigma.
template <int SCATTER>
__device__ __forceinline__ void born_scatter(float bb, float lap_s, float sn, float m,
                                             float &rn, float &sig) {
  if (SCATTER == 0) {
    rn = (float)add_r((double)rn, mul_r(mul_r(.000001, (double)sn), (double)m));
    sig = sn;
  } else {
    sig = mul_r(bb, lap_s);
    rn = fma_r(m, sig, rn);
  }
}

// Eight-tap sinc interpolation with the reference's rounding: products and
// sums rounded separately, left to right (base/cpu_prop.cc:169-176).
__device__ __forceinline__ float sinc8(const float *t, const float *v,
                                       long long stride) {
  float s = mul_r(t[0], v[0]);
#pragma unroll
  for (int k = 1; k < 8; k++) s = add_r(s, mul_r(t[k], v[k * stride]));
  return s;
}

// Uniform per-block mask of the source points inside the block's cells.
__device__ __forceinline__ uint32_t points_in_block(const Points &pts, int x0,
                                                   int x1, int y0, int y1,
                                                   int z0, int z1) {
  uint32_t m = 0;
  for (int i = 0; i < pts.n; i++) {
    const int4 q = ldc(pts.p, i);
    if (q.x >= x0 && q.x < x1 && q.y >= y0 && q.y < y1 && q.z >= z0 && q.z < z1)
      m |= 1u << i;
  }
  return m;
}

__device__ __forceinline__ uint32_t points_on_plane(const Points &pts,
                                                    uint32_t mask, int z) {
  uint32_t m = 0;
  for (uint32_t b = mask; b; b &= b - 1) {
    const int i = __builtin_ctz(b);
    if (ldc(pts.p, i).z == z) m |= 1u << i;
  }
  return m;
}

// The source points of a block: the mask of those inside and the range of
// their z planes, so that the test of a plane off that range loads nothing
// (a loop of dependent scalar loads per plane cost the block that holds a
// 9-point source about 8 us of a 160 us step at 304^3).
struct PtsBlk {
  uint32_t m;
  int zlo, zhi;
};
__device__ __forceinline__ PtsBlk points_of_block(const Points &pts, int x0, int x1, int y0,
                                                  int y1, int z0, int z1) {
  PtsBlk b{0u, 1, 0};
  for (int i = 0; i < pts.n; i++) {
    const int4 q = ldc(pts.p, i);
    if (q.x >= x0 && q.x < x1 && q.y >= y0 && q.y < y1 && q.z >= z0 && q.z < z1) {
      b.zlo = b.m ? min(b.zlo, q.z) : q.z;
      b.zhi = b.m ? max(b.zhi, q.z) : q.z;
      b.m |= 1u << i;
    }
  }
  return b;
}
__device__ __forceinline__ uint32_t points_on_plane(const Points &pts, const PtsBlk &b,
                                                    int z) {
  return z < b.zlo || z > b.zhi ? 0u : points_on_plane(pts, b.m, z);
}

// v plus, in list order, amp[i] of the points at (x, y) among plane mask m
__device__ __forceinline__ float add_points(const Points &pts, uint32_t m, int x,
                                            int y, float v, const float *amp) {
  for (uint32_t b = m; b; b &= b - 1) {
    const int i = __builtin_ctz(b);
    const int4 q = ldc(pts.p, i);
    if (q.x == x && q.y == y) v = add_r(v, ldc(amp, i));
  }
  return v;
}

// Receiver injection of the adjoint-state step: u + V b g, g the sum over
// the receivers at (x, y) of their time-sinc interpolated residual
// (born_abi.hip, exact adjoint).  Rounding fixed as in leap().
__device__ __forceinline__ float lam_inject(const RecMap &rm, int slot, int x, int y, int nx,
                                            int ny, const float *tr, const float *tab, int id,
                                            float v, float b, float u) {
  float g = 0.f;
  for (int i = rm.rmap[((long long)slot * ny + y) * nx + x]; i >= 0; i = rm.rnext[i])
    g = add_r(g, sinc8(tab, tr + (long long)id * rm.nrec + i, rm.nrec));
  return fma_r(mul_r(v, b), g, u);
}

struct CellArgs {
  int x, y, z;
  float b;     // sponge factor (1 outside the sponge)
  int rs;      // receiver slot of the plane, or -1 (then ri and rg are not set)
  int ri;      // first receiver at the cell, or -1
  float rg;    // what is injected there
};

__device__ __forceinline__ float sat_half(float v) { return fminf(fmaxf(v, -65504.f), 65504.f); }

// ---- VX consecutive cells of a row (VX = 1, 2 or 4): the cells at plane
// offset po (uniform) and lane offset o, in elements.  A lane's first cell is
// at a multiple of VX (x tiles start at a multiple of it and nx is one), so
// the accesses are naturally aligned.

// stored words (T: uint16_t, uint32_t) at byte base b and byte offset o;
// NT: the non-temporal hint, for inputs a launch reads once
template <class T, int N, bool NT = false>
__device__ __forceinline__ void ld_words(const char *b, uint32_t o, T (&u)[N]) {
  if constexpr (N == 1) {
    const T *q = (const T *)(b + (uint64_t)o);
    u[0] = NT ? __builtin_nontemporal_load(q) : *q;
  } else {
    // (the instructions need no more than 4-byte alignment)
    typedef T vec __attribute__((ext_vector_type(N), aligned(4)));
    const vec *q = (const vec *)(b + (uint64_t)o);
    const vec w = NT ? __builtin_nontemporal_load(q) : *q;
#pragma unroll
    for (int i = 0; i < N; i++) u[i] = w[i];
  }
}
// N 32-bit words (1, 2 or 4)
template <bool NT, int N>
__device__ __forceinline__ void st_words(const char *b, uint32_t o, const uint32_t (&u)[N]) {
  if constexpr (N == 1)
    st_b32<NT>((void *)b, o, u[0]);
  else if constexpr (N == 2)
    st_b64<NT>((void *)b, o, (uint64_t)u[1] << 32 | u[0]);
  else
    st_b128<NT>((void *)b, o, make_uint4(u[0], u[1], u[2], u[3]));
}
__device__ __forceinline__ __half2 as_half2(uint32_t u) {
  __half2 h;
  __builtin_memcpy(&h, &u, 4);
  return h;
}
__device__ __forceinline__ uint32_t half2_bits(float a, float b) {
  const __half2 h = __floats2half2_rn(a, b);
  uint32_t u;
  __builtin_memcpy(&u, &h, 4);
  return u;
}

// ---- Two FP16 fields stored as one __half2 per cell (first field in the
// low half): one 4-byte load brings both, half the load instructions of two
// separate FP16 arrays.  inv = 1/scale of each field.
template <int VX>
__device__ __forceinline__ void ld_pair(const __half2 *p, uint32_t po, uint32_t o,
                                        const float (&inv)[2], float (&v)[2][VX],
                                        uint32_t = 0) {
  uint32_t u[VX];
  ld_words(adv(p, (uint64_t)po * 4u), o * 4u, u);
#pragma unroll
  for (int i = 0; i < VX; i++) {
    v[0][i] = __low2float(as_half2(u[i])) * inv[0];
    v[1][i] = __high2float(as_half2(u[i])) * inv[1];
  }
}
template <int VX, bool NT = true>
__device__ __forceinline__ void st_pair(__half2 *p, uint32_t po, uint32_t o,
                                        const float (&a)[VX], const float (&b)[VX],
                                        const float (&scale)[2], uint32_t = 0) {
  uint32_t u[VX];
#pragma unroll
  for (int i = 0; i < VX; i++)
    u[i] = half2_bits(sat_half(a[i] * scale[0]), sat_half(b[i] * scale[1]));
  st_words<NT>(adv(p, (uint64_t)po * 4u), o * 4u, u);
}

// ---- 24-bit storage: an FP32 value rounded to 24 bits per cell (sign, the
// 8 exponent bits and 15 significand bits; relative precision 2^-16, the
// whole FP32 range, no scale).  hi holds the top 16 bits of the rounded
// FP32 word and lo the 8 bits below them; the value's FP32 bits are
// hi << 16 | lo << 8.  Rounding adds 0x80 to the word and truncates: half
// way cases go away from zero, a finite value past the largest 24-bit one
// becomes an infinity as in FP32 rounding, infinities stay infinities.
//
// Layout of a level of n cells: the n hi halves, then the n lo bytes; for
// two fields stored together (s, r), n hi pairs then n lo byte pairs.  So
// a cell's hi and lo addresses are a shift of its offset, lo's plus the
// uniform 2n (4n) bytes.  A pointer to Split (SplitPair) advances by 3 (6)
// bytes per cell: the levels of a history and the shots of a batch are
// whole regions of 3n (6n) bytes.  The scale arguments of the loads and
// stores below are those of the scaled FP16 storage and are not used.
struct Split {
  unsigned char b[3];
};
struct SplitPair {
  unsigned char b[6];
};
static_assert(sizeof(Split) == 3 && sizeof(SplitPair) == 6, "packed split types");

// the rounded FP32 word of v
__device__ __forceinline__ uint32_t split_word(float v) { return __float_as_uint(v) + 0x80u; }
// value of a stored cell from hi (in the low 16 bits) and lo (low 8 bits)
__device__ __forceinline__ float split_val(uint32_t hi, uint32_t lo) {
  return __uint_as_float(hi << 16 | (lo & 0xffu) << 8);
}

// hi words of two cells a and b (a in the low half), and their lo bytes in
// the two lowest bytes of a word
__device__ __forceinline__ uint32_t split_hi(uint32_t qa, uint32_t qb) {
  return qa >> 16 | (qb & 0xffff0000u);
}
__device__ __forceinline__ uint32_t split_lo(uint32_t qa, uint32_t qb) {
  return (qa >> 8 & 0xffu) | (qb & 0xff00u);
}
// the two cells of hi word h whose lo bytes are the two lowest of l
__device__ __forceinline__ void split_two(uint32_t h, uint32_t l, float &a, float &b) {
  a = __uint_as_float(h << 16 | (l & 0xffu) << 8);
  b = __uint_as_float((h & 0xffff0000u) | (l & 0xff00u));
}

// (n a multiple of VX: the lo bytes of VX cells are aligned to VX bytes)
template <int VX, bool = false>
__device__ __forceinline__ void ld_vec(const Split *p, uint32_t po, uint32_t o, float,
                                       float (&v)[VX], uint32_t n) {
  const char *bh = adv(p, (uint64_t)po * 2u), *bl = adv(p, (uint64_t)n * 2u + po);
  if constexpr (VX == 1) {
    v[0] = split_val(ldb<unsigned short>(bh, o * 2u), ldb<unsigned char>(bl, o));
  } else {
    uint32_t h[VX / 2], l;
    ld_words(bh, o * 2u, h);
    l = VX == 2 ? ldb<unsigned short>(bl, o) : ldb<uint32_t>(bl, o);
    split_two(h[0], l, v[0], v[1]);
    if constexpr (VX == 4) split_two(h[1], l >> 16, v[2], v[3]);
  }
}
template <int VX, bool NT = true>
__device__ __forceinline__ void st_vec(Split *p, uint32_t po, uint32_t o,
                                       const float (&v)[VX], float, uint32_t n) {
  const char *bh = adv(p, (uint64_t)po * 2u), *bl = adv(p, (uint64_t)n * 2u + po);
  if constexpr (VX == 1) {
    const uint32_t q0 = split_word(v[0]);
    st_b16<NT>((void *)bh, o * 2u, (unsigned short)(q0 >> 16));
    st_b8<NT>((void *)bl, o, (unsigned char)(q0 >> 8));
  } else {
    uint32_t h[VX / 2], l[VX / 2];
#pragma unroll
    for (int i = 0; i < VX / 2; i++) {
      const uint32_t a = split_word(v[2 * i]), b = split_word(v[2 * i + 1]);
      h[i] = split_hi(a, b);
      l[i] = split_lo(a, b);
    }
    st_words<NT>(bh, o * 2u, h);
    if constexpr (VX == 2)
      st_b16<NT>((void *)bl, o, (unsigned short)l[0]);
    else
      st_b32<NT>((void *)bl, o, l[0] | l[1] << 16);
  }
}
// two fields stored together: first field in the low half of each pair
template <int VX>
__device__ __forceinline__ void ld_pair(const SplitPair *p, uint32_t po, uint32_t o,
                                        const float (&)[2], float (&v)[2][VX], uint32_t n) {
  const char *bh = adv(p, (uint64_t)po * 4u), *bl = adv(p, (uint64_t)n * 4u + (uint64_t)po * 2u);
  uint32_t h[VX];
  ld_words(bh, o * 4u, h);
  if constexpr (VX == 1) {
    split_two(h[0], ldb<unsigned short>(bl, o * 2u), v[0][0], v[1][0]);
  } else {
    uint32_t l[VX / 2];
    ld_words(bl, o * 2u, l);
#pragma unroll
    for (int i = 0; i < VX / 2; i++) {
      split_two(h[2 * i], l[i], v[0][2 * i], v[1][2 * i]);
      split_two(h[2 * i + 1], l[i] >> 16, v[0][2 * i + 1], v[1][2 * i + 1]);
    }
  }
}
template <int VX, bool NT = true>
__device__ __forceinline__ void st_pair(SplitPair *p, uint32_t po, uint32_t o,
                                        const float (&a)[VX], const float (&b)[VX],
                                        const float (&)[2], uint32_t n) {
  const char *bh = adv(p, (uint64_t)po * 4u), *bl = adv(p, (uint64_t)n * 4u + (uint64_t)po * 2u);
  uint32_t h[VX], l[VX];
#pragma unroll
  for (int i = 0; i < VX; i++) {
    const uint32_t qa = split_word(a[i]), qb = split_word(b[i]);
    h[i] = split_hi(qa, qb);
    l[i] = split_lo(qa, qb);
  }
  st_words<NT>(bh, o * 4u, h);
  if constexpr (VX == 1) {
    st_b16<NT>((void *)bl, o * 2u, (unsigned short)l[0]);
  } else {
    uint32_t w[VX / 2];
#pragma unroll
    for (int i = 0; i < VX / 2; i++) w[i] = l[2 * i] | l[2 * i + 1] << 16;
    st_words<NT>(bl, o * 2u, w);
  }
}

// ---- one field per array, FP32 (NT: with the non-temporal hint) or FP16
template <int VX, bool NT = false>
__device__ __forceinline__ void ld_vec(const float *p, uint32_t po, uint32_t o, float,
                                       float (&v)[VX], uint32_t = 0) {
  uint32_t u[VX];
  ld_words<uint32_t, VX, NT>(adv(p, (uint64_t)po * 4u), o * 4u, u);
#pragma unroll
  for (int i = 0; i < VX; i++) v[i] = __uint_as_float(u[i]);
}
template <int VX, bool = false>
__device__ __forceinline__ void ld_vec(const __half *p, uint32_t po, uint32_t o, float inv,
                                       float (&v)[VX], uint32_t = 0) {
  const char *b = adv(p, (uint64_t)po * 2u);
  if constexpr (VX == 1) {
    v[0] = __half2float(ldb<__half>(b, o * 2u)) * inv;
  } else {
    uint32_t u[VX / 2];
    ld_words(b, o * 2u, u);
#pragma unroll
    for (int i = 0; i < VX / 2; i++) {
      v[2 * i] = __low2float(as_half2(u[i])) * inv;
      v[2 * i + 1] = __high2float(as_half2(u[i])) * inv;
    }
  }
}
// two FP32 fields interleaved cell by cell
template <int VX, bool NT = false>
__device__ __forceinline__ void ld_vec2(const float2 *p, uint32_t po, uint32_t o,
                                           float (&a)[VX], float (&b)[VX]) {
  const char *q = adv(p, (uint64_t)po * 8u);
#pragma unroll
  for (int h = 0; h < (VX + 1) / 2; h++) {
    constexpr int N = VX == 1 ? 2 : 4;
    uint32_t u[N];
    ld_words<uint32_t, N, NT>(q + 16 * h, o * 8u, u);
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
      a[2 * h + i] = __uint_as_float(u[2 * i]);
      b[2 * h + i] = __uint_as_float(u[2 * i + 1]);
    }
  }
}

template <int VX>
__device__ __forceinline__ void ld_pair(const float2 *p, uint32_t po, uint32_t o,
                                        const float (&)[2], float (&v)[2][VX], uint32_t = 0) {
  ld_vec2<VX>(p, po, o, v[0], v[1]);
}
template <int VX, bool NT = true>
__device__ __forceinline__ void st_pair(float2 *p, uint32_t po, uint32_t o, const float (&a)[VX],
                                        const float (&b)[VX], const float (&)[2], uint32_t = 0) {
  const char *q = adv(p, (uint64_t)po * 8u);
#pragma unroll
  for (int h = 0; h < (VX + 1) / 2; h++) {
    constexpr int N = VX == 1 ? 2 : 4;
    uint32_t u[N];
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
      u[2 * i] = __float_as_uint(a[2 * h + i]);
      u[2 * i + 1] = __float_as_uint(b[2 * h + i]);
    }
    st_words<NT>(q + 16 * h, o * 8u, u);
  }
}

template <int VX, bool NT = true>
__device__ __forceinline__ void st_vec(float *p, uint32_t po, uint32_t o, const float (&v)[VX],
                                       float, uint32_t = 0) {
  uint32_t u[VX];
#pragma unroll
  for (int i = 0; i < VX; i++) u[i] = __float_as_uint(v[i]);
  st_words<NT>(adv(p, (uint64_t)po * 4u), o * 4u, u);
}
template <int VX, bool NT = true>
__device__ __forceinline__ void st_vec(__half *p, uint32_t po, uint32_t o,
                                       const float (&v)[VX], float scale, uint32_t = 0) {
  const char *b = adv(p, (uint64_t)po * 2u);
  if constexpr (VX == 1) {
    st_b16<NT>((void *)b, o * 2u, __half_as_ushort(__float2half_rn(sat_half(v[0] * scale))));
  } else {
    uint32_t u[VX / 2];
#pragma unroll
    for (int i = 0; i < VX / 2; i++)
      u[i] = half2_bits(sat_half(v[2 * i] * scale), sat_half(v[2 * i + 1] * scale));
    st_words<NT>(b, o * 2u, u);
  }
}

// Generic z-marching leapfrog tile: LX*VX x RY*(64*WY/LX) cells of the xy
// plane.  Op supplies (all const):
//   static constexpr int NF, NPRE, NOUT, NMAX; static constexpr bool DAMP;
//   static constexpr int REC;                   receivers: 0 none, 1 read, 2 injected
//   static constexpr bool LEAN;                 Laplacians row by row, field by field
//   Blk block(x0, x1, y0, y1, z0, z1);          uniform per-block state
//   void first(const Blk&);                     (NMAX > 0) once per launch
//   ldv<VX>(const Blk&, int f, uint32_t po, uint32_t o, float (&v)[VX])
//     the current level at plane offset po and lane offset o
//   (PAIRED ops instead: ldv2<VX>(const Blk&, uint32_t po, uint32_t o,
//   float (&v)[NF][VX]) loads every field of the current level at once)
//   Pln plane(const Blk&, int z);               uniform per-plane state
//   prefetchv<VX>(const Blk&, float (&p)[NPRE][VX], uint32_t po, uint32_t o)
//   int rec_slot(const Pln&);                   (REC) receiver slot of the plane, or -1
//   const int *rec_map(int slot);               (REC) its [ny][nx] first receivers
//   float rec_value(int i);                     (REC 2) what receiver cell i injects
//   void cell(const Blk&, const Pln&, const CellArgs&, const float *lap,
//             const float *ctr, const float *pre, float (&out)[NOUT],
//             float (&tmax)[NF]);                the new values of one cell
//   storev<VX>(const Blk&, uint32_t po, uint32_t o, const float (&out)[NOUT][VX])
//   void publish_max(int f, float m);           (NMAX > 0) block max of |new|
template <int B>
struct StepSet {
  static constexpr int value = B;
};

template <class Op, int RY, int WY, int VX, int LX, int D>
__device__ __forceinline__ void march_tile(const Grid &g, const Taps &t, const Sponge &sp,
                                           const Op &op, const int L) {
  constexpr int NF = Op::NF;
  constexpr int NP = Op::NPRE > 0 ? Op::NPRE : 1;
  constexpr int NO = Op::NOUT;
  // LX lanes per row (64: a wavefront per row; 32, 16, 8: it covers 2, 4, 8
  // rows), NG row groups per block of NT threads
  constexpr int NT = kTX * WY;
  constexpr int NG = NT / LX;
  constexpr int TW = LX * VX;
  constexpr int TY = RY * NG;
  constexpr int LW = TW + 2 * kH;
  constexpr int LH = TY + 2 * kH;
  // Ops that ask for it (Op::Q2, the FP16 ops: their steps ran 7-8 %
  // faster, the FP32 forward 2.5 % slower) with one step of lookahead unroll
  // the loop over pairs of steps: the z queue holds one plane more and moves
  // by two planes every second step (half the register moves), and the
  // pointwise inputs of the two steps sit in two buffers that the steps
  // refill alternately (no copy).
  constexpr bool Q2 = Op::Q2 && D == 1;
  constexpr int NB = Q2 ? 2 : D;  // buffer sets of loads in flight
  // queue: planes z - kH .. z + kH (Q2: one more)
  constexpr int NQ = 2 * kH + 1 + (Q2 ? 1 : 0);

  const int bx = L % g.ntx;
  const int rest = L / g.ntx;
  const int by = rest % g.nty;
  const int bz = rest / g.nty;
  const int tx = (int)threadIdx.x % LX;
  const int ty = (int)threadIdx.x / LX;
  // x tiles start at the row start so that a wavefront's row maps onto whole
  // cache lines; the 4-cell shell at either end is masked
  const int x0 = bx * TW, y0 = kH + by * TY;
  // The chunk's planes z0 .. z1 - 1.  Chunks are marched up and down in turn,
  // so that two neighbours read the planes they share at about the same time,
  // and a time loop turns every chunk round from one step to the next
  // (g.back), so that a step starts with the planes the last one ended with
  // (back 2: all are marched up, see batch_sweep() in born_abi.hip).  z is the count of a marched plane, zp its plane in the fields.
  const int z0 = kH + bz * g.zc;
  const int z1 = min(z0 + g.zc, g.nz - kH);
  const bool down = g.back < 2 && ((bz & 1) ^ g.back) != 0;
  const int zb = down ? z0 + z1 - 1 : 0, zs = down ? -1 : 1;
  auto zp = [&](int z) { return zb + zs * z; };
  auto zoff = [&](int z) { return (uint32_t)zp(z) * g.plane; };
  const int x = x0 + VX * tx;
  const bool xin = x >= kH && x < g.nx - kH;  // with VX > 1 a lane's cells are in or out
  const int xc = min(x, g.nx - VX);

  const auto blk = op.block(max(x0, kH), min(x0 + TW, g.nx - kH), y0,
                            min(y0 + TY, g.ny - kH), z0, z1);
  if constexpr (Op::NMAX > 0)
    if (L == 0 && threadIdx.x == 0) op.first(blk);

  // Cells are addressed by the plane's offset, uniform and added to the
  // arrays' scalar base addresses, plus a lane's offset in the plane, which
  // does not change over the march.  (The compiler adds the two as 64-bit values
  // at each load; made to use the scalar-base form of the loads, 9 registers
  // fewer, the 24-bit adjoint ran 3 % slower and the rest the same.)
  int yy[RY];
  bool in[RY];
  uint32_t row[RY];
  float bxy[RY][VX];
#pragma unroll
  for (int j = 0; j < RY; j++) {
    yy[j] = y0 + RY * ty + j;  // a thread's rows are consecutive
    in[j] = xin && yy[j] < g.ny - kH;
    const int yc = min(yy[j], g.ny - 1);
    row[j] = (uint32_t)yc * g.nx + xc;
#pragma unroll
    for (int v = 0; v < VX; v++) bxy[j][v] = Op::DAMP ? fminf(sp.bx[xc + v], sp.by[yc]) : 1.f;
  }

  // LDS halo in units of VX cells: 8 y-halo rows of LX units and, per row,
  // kH/VX units on either side, spread over the block's threads
  constexpr int XU = kH / VX;
  constexpr int NYH = 2 * kH * LX;
  constexpr int NXH = 2 * XU * TY;
  constexpr int NHALO = NYH + NXH;
  constexpr int HPT = (NHALO + NT - 1) / NT;
  uint32_t hoff[HPT];
  int ht[HPT];  // the unit's place in an LDS tile
  bool hv[HPT];
#pragma unroll
  for (int k = 0; k < HPT; k++) {
    const int h = (int)threadIdx.x + k * NT;
    hv[k] = (k + 1) * NT <= NHALO || h < NHALO;
    int lr, lc;
    if (h < NYH) {  // rows 0..3 and TY+4..TY+7
      const int r = h / LX;
      lr = r < kH ? r : TY + r;
      lc = kH + VX * (h % LX);
    } else {  // columns 0..3 and TW+4..TW+7 of rows 4..TY+3
      const int hh = min(h - NYH, NXH - 1);
      const int c = hh % (2 * XU);
      lr = kH + hh / (2 * XU);
      lc = c < XU ? VX * c : kH + TW + VX * (c - XU);
    }
    ht[k] = lr * LW + lc;
    const int gy = min(max(y0 - kH + lr, 0), g.ny - 1);
    const int gx = min(max(x0 - kH + lc, 0), g.nx - VX);
    hoff[k] = (uint32_t)gy * g.nx + gx;
  }

  // The loads of step z + D (queue leads, LDS halos, pointwise inputs) are
  // issued before step z is computed: with D = 2 a load has two steps'
  // compute to arrive, and the wait at a step's start leaves the previous
  // step's loads in flight (the stores are invisible to the compiler's wait
  // model and the barriers do not fence global memory, see st_b32 and
  // lds_barrier).  Loads past the chunk's last step are clamped to planes the
  // chunk reads anyway.
  //
  // The LDS halo of a plane is loaded together with the plane's centre rows
  // (when the plane enters the z queue as a lead), not kH planes later: the
  // neighbouring tiles read those rows at about the same time, so they come
  // from L2.  It waits kH planes in the loading thread's own place of stage
  // (slot = plane mod kH), not in registers; hl holds the halos of the leads
  // in flight.  tile holds the plane computed, in two buffers that the steps
  // take in turn: a step writes one while slower wavefronts still read the
  // other, so a step has a single barrier.
  __shared__ __align__(16) float tile[2][NF][LH][LW];
  __shared__ __align__(16) float stage[kH][NF][NHALO][VX];
  float q[NF][RY][VX][NQ];
  float lead[NB][NF][RY][VX];
  float hl[NB][NF][HPT][VX];
  // pointwise inputs of the steps in flight, and of the step computed
  float pre[NB][RY][NP][VX], cur[RY][NP][VX];
  float tmax[NF];
  // every field of the current level at plane offset po, lane offset o
  auto ld_all = [&](uint32_t po, uint32_t o, float (&v)[NF][VX]) {
    if constexpr (Op::PAIRED) {
      op.template ldv2<VX>(blk, po, o, v);
    } else {
#pragma unroll
      for (int f = 0; f < NF; f++) op.template ldv<VX>(blk, f, po, o, v[f]);
    }
  };
  // the loads of the step at plane zs into buffer set b
  auto issue = [&](int zs, int b) {
    const uint32_t zl = zoff(min(zs + kH, z1 - 1 + kH));
    const uint32_t zn = zoff(min(zs, z1 - 1));
#pragma unroll
    for (int j = 0; j < RY; j++) {
      float w[NF][VX];
      ld_all(zl, row[j], w);
#pragma unroll
      for (int f = 0; f < NF; f++)
#pragma unroll
        for (int v = 0; v < VX; v++) lead[b][f][j][v] = w[f][v];
    }
#pragma unroll
    for (int k = 0; k < HPT; k++) {
      float w[NF][VX];
      ld_all(zl, hoff[k], w);
#pragma unroll
      for (int f = 0; f < NF; f++)
#pragma unroll
        for (int v = 0; v < VX; v++) hl[b][f][k][v] = w[f][v];
    }
#pragma unroll
    for (int j = 0; j < RY; j++) op.template prefetchv<VX>(blk, pre[b][j], zn, row[j]);
  };
#pragma unroll
  for (int f = 0; f < NF; f++) tmax[f] = 0.f;
  // all of the chunk's first loads are in flight together
#pragma unroll
  for (int j = 0; j < RY; j++) {
#pragma unroll
    for (int k = 0; k < 2 * kH; k++) {
      float w[NF][VX];
      ld_all(zoff(z0 - kH + k), row[j], w);
#pragma unroll
      for (int f = 0; f < NF; f++)
#pragma unroll
        for (int v = 0; v < VX; v++) q[f][j][v][k] = w[f][v];
    }
  }
  {
    float h[kH][HPT][NF][VX];
#pragma unroll
    for (int p = 0; p < kH; p++)
#pragma unroll
      for (int k = 0; k < HPT; k++) ld_all(zoff(z0 + p), hoff[k], h[p][k]);
#pragma unroll
    for (int b = 0; b < D; b++) issue(z0 + b, b);
#pragma unroll
    for (int p = 0; p < kH; p++)
#pragma unroll
      for (int k = 0; k < HPT; k++)
#pragma unroll
        for (int f = 0; f < NF; f++)
          if (hv[k]) st_lds<VX>(stage[p][f][(int)threadIdx.x + k * NT], h[p][k][f]);
  }

  // The new values of a step are stored at the start of the next step,
  // after its wait and before its loads: the wait for a step's inputs then
  // finds stores and loads that were issued a whole step earlier.
  float pend[RY][NO][VX];
  int pend_z = -1;
  auto flush = [&]() {
    if (pend_z >= 0) {
      // (in a scalar register: the stores' base addresses have to be)
      const uint32_t po = __builtin_amdgcn_readfirstlane(zoff(pend_z));
#pragma unroll
      for (int j = 0; j < RY; j++)
        if (in[j]) op.template storev<VX>(blk, po, row[j], pend[j]);
    }
  };

  // One step at plane z from buffer set b; its loads go to set bn.  R = 1
  // for the second step of a Q2 pair, whose queue entries are one register
  // further on.  b and R are compile-time constants.
  auto step = [&](const int z, auto bc, auto rc) {
    constexpr int b = decltype(bc)::value;
    constexpr int R = decltype(rc)::value;
    constexpr int bn = Q2 ? 1 - b : b;
    // the pointwise inputs are copied out of a buffer that this step's loads
    // refill
    constexpr bool COPY = bn == b;
    const int sl = (z - z0) % 2, ss = (z - z0) % kH;
    // plane z to LDS: the centre rows from the queue, the halo from stage
#pragma unroll
    for (int f = 0; f < NF; f++) {
#pragma unroll
      for (int k = 0; k < HPT; k++) {
        float h[VX];
        if (hv[k]) {
          ld_lds<VX>(stage[ss][f][(int)threadIdx.x + k * NT], h);
          st_lds<VX>(&tile[sl][f][0][0] + ht[k], h);
        }
      }
#pragma unroll
      for (int j = 0; j < RY; j++) {
        float c[VX];
#pragma unroll
        for (int v = 0; v < VX; v++) c[v] = q[f][j][v][kH + R];
        st_lds<VX>(&tile[sl][f][kH + RY * ty + j][kH + VX * tx], c);
      }
    }
    // the loads of this step: leads to the queue, their halo to stage
    float(&pw)[RY][NP][VX] = COPY ? cur : pre[b];
    if constexpr (COPY) {
#pragma unroll
      for (int j = 0; j < RY; j++)
#pragma unroll
        for (int k = 0; k < NP; k++)
#pragma unroll
          for (int v = 0; v < VX; v++) cur[j][k][v] = pre[b][j][k][v];
    }
#pragma unroll
    for (int f = 0; f < NF; f++) {
#pragma unroll
      for (int j = 0; j < RY; j++)
#pragma unroll
        for (int v = 0; v < VX; v++) q[f][j][v][2 * kH + R] = lead[b][f][j][v];
#pragma unroll
      for (int k = 0; k < HPT; k++)
        if (hv[k]) st_lds<VX>(stage[ss][f][(int)threadIdx.x + k * NT], hl[b][f][k]);
    }
    flush();
    issue(z + D, bn);
    lds_barrier();
    const auto pl = op.plane(blk, zp(z));
    const float bzv = Op::DAMP ? ldc(sp.bz, zp(z)) : 1.f;
    // the receivers of the cells of a plane that has some (rs >= 0), loaded
    // while the Laplacians are computed; not set on the other planes
    int ri[RY][VX];
    float rg[RY][VX];
    int rs = -1;
    if constexpr (Op::REC > 0) {
      rs = op.rec_slot(pl);
      if (rs >= 0) {
        const int *rmap = op.rec_map(rs);
#pragma unroll
        for (int j = 0; j < RY; j++) ld_words<int, VX>((const char *)rmap, row[j] * 4u, ri[j]);
        if constexpr (Op::REC == 2) {
#pragma unroll
          for (int j = 0; j < RY; j++)
#pragma unroll
            for (int v = 0; v < VX; v++) rg[j][v] = op.rec_value(max(ri[j][v], 0));
        }
      }
    }
    // Laplacians field by field.  The column above and below this
    // thread's RY consecutive rows is read from LDS once per field (kH
    // rows either side; the thread's own rows come from its z queues) and
    // shared by the RY cells.
    // LEAN ops skip the rows outside the domain and finish a field before the
    // next: left to itself the compiler issues the LDS reads of every row and
    // field together and holds them all.  Registers of a lane and wavefronts of
    // a SIMD, without -> with: FP32 forward with s and r apart, 2 x 4, 152 and 3
    // -> 113 and 4; FP16 forward, 2 x 8 with two planes of lookahead, 162 and 3
    // -> 127 and 4; 25 of 50 kernels that spilled no longer do.  us per step:
    // FP32 forward 304^3, 1000 levels kept, 159 -> 154; FP16 forward 304^3 124
    // -> 114, 480x448x416 411 -> 380.
    const int lr0 = kH + RY * ty, lc = kH + VX * tx;
    float lap[RY][VX][NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
      if (Op::LEAN && f > 0) __builtin_amdgcn_sched_barrier(0);
      float col[RY + 2 * kH][VX];
#pragma unroll
      for (int i = 0; i < kH; i++) {
        ld_lds<VX>(&tile[sl][f][lr0 - kH + i][lc], col[i]);
        ld_lds<VX>(&tile[sl][f][lr0 + RY + i][lc], col[kH + RY + i]);
      }
#pragma unroll
      for (int j = 0; j < RY; j++)
#pragma unroll
        for (int v = 0; v < VX; v++) col[kH + j][v] = q[f][j][v][kH + R];
#pragma unroll
      for (int j = 0; j < RY; j++) {
        if (Op::LEAN && !in[j]) continue;
        // the row from lc - 4 to lc + VX + 3
        float xs[2 * kH + VX];
#pragma unroll
        for (int i = 0; i < kH; i += VX) {
          float w[VX];
          ld_lds<VX>(&tile[sl][f][lr0 + j][lc - kH + i], w);
#pragma unroll
          for (int v = 0; v < VX; v++) xs[i + v] = w[v];
          ld_lds<VX>(&tile[sl][f][lr0 + j][lc + VX + i], w);
#pragma unroll
          for (int v = 0; v < VX; v++) xs[kH + VX + i + v] = w[v];
        }
#pragma unroll
        for (int v = 0; v < VX; v++) xs[kH + v] = q[f][j][v][kH + R];
#pragma unroll
        for (int v = 0; v < VX; v++) {
          // centre, then the x, y and z pairs, each pair summed first
          float a = mul_r(t.c0, q[f][j][v][kH + R]);
#pragma unroll
          for (int k = 1; k <= kH; k++)
            a = fma_r(t.cx[k - 1], add_r(xs[kH + v - k], xs[kH + v + k]), a);
#pragma unroll
          for (int k = 1; k <= kH; k++)
            a = fma_r(t.cy[k - 1], add_r(col[kH + j - k][v], col[kH + j + k][v]), a);
#pragma unroll
          for (int k = 1; k <= kH; k++)
            a = fma_r(t.cz[k - 1], add_r(q[f][j][v][kH - k + R], q[f][j][v][kH + k + R]), a);
          lap[j][v][f] = a;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < RY; j++) {
      if (!in[j]) continue;
#pragma unroll
      for (int v = 0; v < VX; v++) {
        float ctr[NF];
#pragma unroll
        for (int f = 0; f < NF; f++) ctr[f] = q[f][j][v][kH + R];
        CellArgs c;
        c.x = x + v;
        c.y = yy[j];
        c.z = zp(z);
        c.b = fminf(bxy[j][v], bzv);
        c.rs = rs;
        if constexpr (Op::REC > 0) c.ri = ri[j][v];
        if constexpr (Op::REC == 2) c.rg = rg[j][v];
        float pv[NP], o[NO];
#pragma unroll
        for (int k = 0; k < NP; k++) pv[k] = pw[j][k][v];
        op.cell(blk, pl, c, lap[j][v], ctr, pv, o, tmax);
#pragma unroll
        for (int k = 0; k < NO; k++) pend[j][k][v] = o[k];
      }
    }
    pend_z = z;
    // the queue moves by a plane a step, or by two after a Q2 pair
    constexpr int MV = Q2 ? (R == 1 ? 2 : 0) : 1;
    if constexpr (MV > 0) {
#pragma unroll
      for (int f = 0; f < NF; f++)
#pragma unroll
        for (int j = 0; j < RY; j++)
#pragma unroll
          for (int v = 0; v < VX; v++)
#pragma unroll
            for (int k = 0; k < 2 * kH; k++) q[f][j][v][k] = q[f][j][v][k + MV];
    }
  };

  if constexpr (Q2) {
    for (int z = z0; z < z1; z += 2) {
      step(z, StepSet<0>{}, StepSet<0>{});
      if (z + 1 >= z1) break;
      step(z + 1, StepSet<1>{}, StepSet<1>{});
    }
  } else {
    for (int z = z0; z < z1; z += D) {
      step(z, StepSet<0>{}, StepSet<0>{});
      if constexpr (D == 2) {
        if (z + 1 >= z1) break;
        step(z + 1, StepSet<1>{}, StepSet<0>{});
      }
    }
  }
  flush();
  // block maxima of |new level| for the next step's FP16 scales
  if constexpr (Op::NMAX > 0) {
    __shared__ float red[NF][WY];
#pragma unroll
    for (int f = 0; f < NF; f++) {
      float m = tmax[f];
      for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
      if (threadIdx.x % kTX == 0) red[f][threadIdx.x / kTX] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int f = 0; f < NF; f++) {
        float m = 0.f;
        for (int w = 0; w < WY; w++) m = fmaxf(m, red[f][w]);
        op.publish_max(f, m);
      }
    }
  }
}

// The step kernels take one plane per step; LA steps of load lookahead.
template <class Op, int RY, int WY, int VX, int LA, int LX>
__global__ void __launch_bounds__(kTX *WY)
    march_kernel(const Grid g, const Taps t, const Sponge sp, const Op op) {
  march_tile<Op, RY, WY, VX, LX, LA>(g, t, sp, op,
                                        xcd_remap((int)blockIdx.x, (int)gridDim.x));
}

// Tiles of a batch of shots with their own grids: shot s owns the logical
// tiles [tile0[s], tile0[s + 1]).
constexpr int kMaxBatch = 64;
struct BatchTiles {
  int n;
  int zc;
  int back;  // Grid::back of every shot
  int tile0[kMaxBatch + 1];
};

// Tile grid of a domain for tiles of tw x ty cells and z chunk zc.
__host__ __device__ inline Grid tile_grid(int nx, int ny, int nz, int tw, int ty, int zc) {
  Grid g;
  g.nx = nx;
  g.ny = ny;
  g.nz = nz;
  g.plane = (uint32_t)nx * ny;
  g.back = 0;
  g.ntx = (nx - kH + tw - 1) / tw;
  g.nty = (ny - 2 * kH + ty - 1) / ty;
  g.zc = zc;
  g.ntz = (nz - 2 * kH + zc - 1) / zc;
  return g;
}

// One launch advances every shot of a batch by one step.  BOp::shot(s, tw,
// ty, zc) returns {Grid, Sponge, Op} of shot s with the op's pointers moved to
// the shot's part of the batch arrays.
template <class BOp, int RY, int WY, int VX, int LA, int LX>
__global__ void __launch_bounds__(kTX *WY)
    march_batch_kernel(const BatchTiles bt, const Taps t, const BOp bop) {
  const int Lg = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  int s = 0;
  while (s + 1 < bt.n && Lg >= bt.tile0[s + 1]) s++;
  auto sh = bop.shot(s, LX * VX, RY * (kTX * WY / LX), bt.zc);
  sh.g.back = bt.back;
  march_tile<typename BOp::Op, RY, WY, VX, LX, LA>(sh.g, t, sh.sp, sh.op, Lg - bt.tile0[s]);
}

}  // namespace born
