// Fused time-step ops of the Born propagator (gfx950) and the templates
// that launch them; the launchers are instantiated in the born_k_*.hip
// translation units (compiled in parallel) and dispatched in born_kernels.hip.
//
// Each op below is one time step of one of the reference's loops
// (base/cpu_prop.cc), with every per-cell pass of that step fused into the
// single z-marching sweep of march_kernel:
//   FwdOp     rtmForward step (cpu_prop.cc:31-53): prop s, prop r, damp both,
//             inject source, Born scatter, extract receivers.
//   SrcOp     sourceProp step (cpu_prop.cc:112-122): undamped, inject source.
//   RadjOp    rtmAdjoint step (cpu_prop.cc:71-95): reverse s (vel1), r (vel2),
//             damp r, inject receivers, imaging condition.
//   SrecOp    background step of the exact adjoint (the s half of FwdOp) that
//             also stores the scatter operand of the step.
//   LamOp     adjoint-state step of the exact adjoint (see born_abi.hip).
//
// Storage convention: a field buffer holds each level exactly as the
// reference holds it right after that level was produced (damped, injected).
// The reference additionally damps the current level in place after the
// update (cpu_prop.cc:141-165 on p1); that value is only ever read back as the
// "old" level of the next step, so it is recomputed there as fl(b * old)
// instead of being written: same arithmetic, one HBM write less per field.
#pragma once
#include <type_traits>

#include "born_device.h"
#include "born_launch.h"

namespace born {

struct NoBlk {};
struct RecPln {
  int slot;
};
struct SrcPln {
  uint32_t pm;
  int slot;
};

__device__ __forceinline__ const int *rec_plane(const RecMap &rm, int slot, int nx, int ny) {
  return rm.rmap + (long long)slot * ny * nx;
}

// Scaled storage (FP16) shares the state of the ops (unused with float and
// 24-bit storage): each stored level has a power-of-two scale derived from a
// bound on |new level|, gain * max|cur| + max|old| + injections, with
// gain = 2 + max(V) * tapsum and tapsum >= |L u| / max|u|.
template <class T>
constexpr bool kScaled = std::is_same<T, __half>::value;
// 24-bit storage (FP32 rounded to 24 bits)
template <class T>
constexpr bool kSplit = std::is_same<T, Split>::value;
// levels narrower than FP32 (FP16 or 24-bit): the forward stores s and r
// together, the steps run in pairs, the streams take the FP16 cache hints
template <class T>
constexpr bool kNarrow = !std::is_same<T, float>::value;
// two fields stored together: FP32 as float2, FP16 as __half2, 24-bit as
// SplitPair
template <class T>
using PairOf = typename std::conditional<
    kNarrow<T>, typename std::conditional<kSplit<T>, SplitPair, __half2>::type, float2>::type;

struct Blk1 {  // one stored field
  PtsBlk pb;
  float ic, io, sn, sh;  // 1/scale of cur and old, scale of new and of sigma
};
struct Blk2 {  // two stored fields
  PtsBlk pb;
  float ic[2], io[2], sn[2], sh;
};

__device__ __forceinline__ float amp_sum(const Points &pts, const float *amp) {
  float a = 0.f;
  for (int i = 0; i < pts.n; i++) a += fabsf(ldc(amp, i));
  return a;
}

// ---------------------------------------------------------------- forward
// NT: the single-shot forward: velocity and model as one stream, the
// non-temporal hint on the stores of levels apart and of the history (the shot
// batch: see BatchFwd).  The other accesses take no hint (but see s0 and HINT):
// what a step reads the next one reads or overwrites, and an access with the
// hint leaves nothing in the 256 MB memory-side cache.  FP32, us per step with
// the hint on the pointwise loads -> without: 160^3 31.6 -> 26.4 (dV scatter 35.5
// -> 26.1), 224^3 73.7 -> 63.9 (83.7 -> 61.7).  Levels apart are those of large
// grids: 304^3 172.4 with the hint on their stores, 177.9 without.  No step reads
// the history again.  FP16 levels with the hint -> without: 160^3 38.1 -> 36.1,
// 224^3 72.8 -> 66.9, 304^3 127.9 -> 128.9.
//
// PAIR: s and r together per cell.  Half as many streams, twice as long: rows
// of a level are seldom whole cache lines, and each tile's row ends in two
// partial ones per stream.  FP32, us per step apart -> together: 160^3 25.2 ->
// 22.9, 224^3 61.5 -> 51.8, 304^3 173.7 -> 162.9, 203^3 54.6 -> 52.8, 64^3 7.8 ->
// 7.7; 16 shots of 114-144 x 114-152 x 112 222 -> 188.  FP32 levels stay apart
// where s levels are wanted by themselves (born_dev_forward).
//
// HINT: FP32 levels together with the non-temporal hint on the old level,
// velocity and model, and on the stores: for grids whose levels, velocity and
// model (24 bytes per cell) are past the 256 MB memory-side cache, where what a
// step leaves there is gone before the next one comes to it, and accesses
// without the hint only evict the halo rows.  us per step without -> with: 224^3
// 52 -> 63, 240^3 78.0 -> 78.3, 256^3 92.6 -> 87.4, 304^3 163 -> 146, 384 x 384 x
// 352 340 -> 306, 448 x 448 x 400 524 -> 469, 640 x 640 x 500 1484 -> 1402 (1394
// with s and r apart and hints throughout); dV term with its history 240^3 89.4
// -> 89.0, 256^3 101.9 -> 103.1, 272^3 129.8 -> 126.5, 304^3 187 -> 167.  Narrow
// levels do without: FP16 gains 1 % from 448^3 on; 24-bit 256^3 80 -> 77, 272 x
// 288 x 320 (pair) 30.7 -> 31.3 ms, 448 x 448 x 400 445 -> 440.
template <int SCATTER, class T, bool NT = true, bool PAIR = kNarrow<T>, bool HINT = false>
struct FwdOp {
  static constexpr bool H = kScaled<T>;
  static constexpr int NF = 2, NPRE = 4, NOUT = 3, NMAX = H ? 2 : 0, REC = 1;
  // s and r together per cell: sr1 level k, sr0 level k-1, srn level k+1, the
  // same buffer as sr0 in place
  static constexpr bool PAIRED = PAIR;
  static constexpr bool Q2 = kNarrow<T>;  // steps in pairs (march_tile)
  // (FP32, s and r together: 22.8 us per step without, 23.4 with, at 160^3,
  // where the registers are not what limits the wavefronts)
  static constexpr bool LEAN = kNarrow<T> || !PAIR || HINT;
  static constexpr bool DAMP = true;
  const T *__restrict__ s1;
  const T *__restrict__ r1;
  // old s level (read) and new s level (written): the same buffer (in
  // place), or with scatter 0 and a kept history two levels of the history,
  // whose level k is s of level k+1
  const T *s0;
  T *s_new;
  T *__restrict__ r0;
  const PairOf<T> *sr1;
  const PairOf<T> *sr0;
  PairOf<T> *srn;
  const float *__restrict__ vel;  // vel and model: the shot batch
  const float *__restrict__ model;
  // NT (the single-shot forward): vel and model interleaved per cell, one
  // load and one stream for both
  const float2 *__restrict__ vm;
  T *__restrict__ hist;  // optional scatter-operand history
  Points pts;
  const float *__restrict__ amp;  // source amplitudes of this step [npts]
  RecMap rm;
  float *rv;  // the new r at the receiver cells (nullptr: not wanted)
  int nx, ny;
  uint32_t nlev;  // cells of a level (24-bit storage: the lo bytes follow the hi values)
  // FP16 scale state in as few scalar registers as possible (the loop needs
  // none of it, but kernel arguments stay live in scalar registers, and
  // too many of them spill into vector lanes that every use reloads): the
  // ring block rg holds the s ring at 0, the r ring at 8 and max |model| at
  // 16 (float bits); slots packs cur, old, nxt, clr in its four bytes.
  float *rg;
  int slots;
  float gain, tapsum;
  float *hscale;  // FP16: scale of this step's history level

  __device__ Ring ring(int f) const { return {rg + 8 * f, (unsigned *)(rg + 8 * f + 4)}; }
  __device__ int slot(int i) const { return (slots >> (8 * i)) & 0xff; }

  __device__ Blk2 block(int x0, int x1, int y0, int y1, int z0, int z1) const {
    Blk2 b;
    b.pb = points_of_block(pts, x0, x1, y0, y1, z0, z1);
    for (int f = 0; f < 2; f++) b.ic[f] = b.io[f] = b.sn[f] = 1.f;
    b.sh = 1.f;
    if constexpr (H) {
      const int cur = slot(0), old = slot(1);
      for (int f = 0; f < 2; f++) {
        b.ic[f] = 1.f / ring(f).scale[cur];
        b.io[f] = 1.f / ring(f).scale[old];
      }
      const float ms = ring_max(ring(0), cur);
      const float bs = gain * ms + ring_max(ring(0), old) + amp_sum(pts, amp);
      const float mm = __uint_as_float(*(const unsigned *)(rg + 16));
      const float sig = SCATTER == 0 ? bs : tapsum * ms;
      const float br = gain * ring_max(ring(1), cur) + ring_max(ring(1), old) +
                       (SCATTER == 0 ? 1e-6f * bs * mm : mm * sig);
      b.sn[0] = level_scale(bs);
      b.sn[1] = level_scale(br);
      b.sh = SCATTER == 0 ? b.sn[0] : level_scale(sig);
    }
    return b;
  }
  __device__ void first(const Blk2 &b) const {
    for (int f = 0; f < 2; f++) {
      ring(f).scale[slot(2)] = b.sn[f];
      ring(f).maxb[slot(3)] = 0u;
    }
    if (hscale) *hscale = b.sh;
  }
  __device__ void publish_max(int f, float m) const {
    atomicMax(&ring(f).maxb[slot(2)], __float_as_uint(m));
  }
  template <int VX>
  __device__ void ldv(const Blk2 &b, int f, uint32_t po, uint32_t o, float (&v)[VX]) const {
    ld_vec<VX>(f == 0 ? s1 : r1, po, o, b.ic[f], v, nlev);
  }
  template <int VX>
  __device__ void ldv2(const Blk2 &b, uint32_t po, uint32_t o, float (&v)[2][VX]) const {
    ld_pair<VX>(sr1, po, o, b.ic, v, nlev);
  }
  __device__ SrcPln plane(const Blk2 &b, int z) const {
    return {points_on_plane(pts, b.pb, z), ldc(rm.plane_slot, z)};
  }
  __device__ int rec_slot(const SrcPln &pl) const { return rv ? pl.slot : -1; }
  __device__ const int *rec_map(int slot) const { return rec_plane(rm, slot, nx, ny); }
  template <int VX>
  __device__ void prefetchv(const Blk2 &b, float (&p)[NPRE][VX], uint32_t po,
                            uint32_t o) const {
    if constexpr (PAIRED) {
      float sr[2][VX];
      if constexpr (HINT)
        ld_vec2<VX, true>(sr0, po, o, sr[0], sr[1]);
      else
        ld_pair<VX>(sr0, po, o, b.io, sr, nlev);
#pragma unroll
      for (int v = 0; v < VX; v++) {
        p[0][v] = sr[0][v];
        p[1][v] = sr[1][v];
      }
    } else {
      // s0 alone takes the hint: levels apart are those of a kept history, whose
      // oldest one no step reads again (304^3 169.9 -> 167.7 us, 352^3 266.1 ->
      // 260.9)
      ld_vec<VX, true>(s0, po, o, b.io[0], p[0], nlev);
      ld_vec<VX>(r0, po, o, b.io[1], p[1], nlev);
    }
    if constexpr (NT) {
      ld_vec2<VX, HINT>(vm, po, o, p[2], p[3]);
    } else {
      ld_vec<VX>(vel, po, o, 1.f, p[2]);
      ld_vec<VX>(model, po, o, 1.f, p[3]);
    }
  }
  template <int VX>
  __device__ void storev(const Blk2 &b, uint32_t po, uint32_t o,
                         const float (&out)[NOUT][VX]) const {
    if constexpr (PAIRED) {
      st_pair<VX, HINT>(srn, po, o, out[0], out[1], b.sn, nlev);
    } else {
      st_vec<VX, NT>(s_new, po, o, out[0], b.sn[0], nlev);
      st_vec<VX, NT>(r0, po, o, out[1], b.sn[1], nlev);
    }
    if (hist) st_vec<VX, NT>(hist, po, o, out[2], b.sh, nlev);
  }
  __device__ void cell(const Blk2 &b, const SrcPln &pl, const CellArgs &c,
                       const float *lap, const float *ctr, const float *p,
                       float (&out)[NOUT], float (&tmax)[NF]) const {
    const float v = p[2], bb = c.b;
    float sn = leap(bb, v, lap[0], ctr[0], p[0]);
    if (pl.pm) sn = add_points(pts, pl.pm, c.x, c.y, sn, amp);
    float rn = leap(bb, v, lap[1], ctr[1], p[1]);
    float sig;
    if constexpr (kNarrow<T> && SCATTER == 0) {
      // FP16 and 24-bit levels: the 1e-6 s m term in FP32.  FP32 levels
      // round it in FP64 as the reference does (bitwise parity); the
      // narrow levels' own rounding (2^-11, 2^-16) is far above FP32's.
      rn = fma_r(mul_r(1e-6f, sn), p[3], rn);
      sig = sn;
    } else {
      born_scatter<SCATTER>(bb, lap[0], sn, p[3], rn, sig);
    }
    out[0] = sn;
    out[1] = rn;
    out[2] = sig;
    if constexpr (H) {
      tmax[0] = fmaxf(tmax[0], fabsf(sn));
      tmax[1] = fmaxf(tmax[1], fabsf(rn));
    }
    if (c.rs >= 0 && c.ri >= 0) st_b32<false>(rv, (uint32_t)c.ri * 4u, __float_as_uint(rn));
  }
};

// ------------------------------------------------------------- sourceProp
struct SrcOp {
  static constexpr int NF = 1, NPRE = 2, NOUT = 1, NMAX = 0, REC = 0;
  static constexpr bool PAIRED = false;
  static constexpr bool Q2 = false;
  static constexpr bool LEAN = true;
  static constexpr bool DAMP = false;
  const float *__restrict__ s1;
  float *__restrict__ s0;
  const float *__restrict__ vel;
  Points pts;
  const float *__restrict__ amp;
  __device__ PtsBlk block(int x0, int x1, int y0, int y1, int z0, int z1) const {
    return points_of_block(pts, x0, x1, y0, y1, z0, z1);
  }
  template <int VX>
  __device__ void ldv(const PtsBlk &, int, uint32_t po, uint32_t o, float (&v)[VX]) const {
    ld_vec<VX>(s1, po, o, 1.f, v);
  }
  __device__ uint32_t plane(const PtsBlk &blk, int z) const {
    return points_on_plane(pts, blk, z);
  }
  template <int VX>
  __device__ void prefetchv(const PtsBlk &, float (&p)[NPRE][VX], uint32_t po,
                            uint32_t o) const {
    ld_vec<VX>(s0, po, o, 1.f, p[0]);
    ld_vec<VX>(vel, po, o, 1.f, p[1]);
  }
  template <int VX>
  __device__ void storev(const PtsBlk &, uint32_t po, uint32_t o,
                         const float (&out)[NOUT][VX]) const {
    st_vec<VX>(s0, po, o, out[0], 1.f);
  }
  __device__ void cell(const PtsBlk &, uint32_t pm, const CellArgs &c, const float *lap,
                       const float *ctr, const float *p, float (&out)[NOUT],
                       float (&)[NF]) const {
    float sn = p[1] * lap[0] + ctr[0] + ctr[0] - p[0];
    if (pm) sn = add_points(pts, pm, c.x, c.y, sn, amp);
    out[0] = sn;
  }
};

// ------------------------------------------------------ reference adjoint
// PAIR: s and r together per cell in s1 and s0, as in the forward (FP32, us per
// step apart -> together: 160^3 27.9 -> 26.8, 224^3 86.5 -> 77.3, 304^3 223.6 ->
// 210.6, 203^3 59.7 -> 57.5; 64^3 7.0 -> 7.6).
template <bool PAIR>
struct RadjOp {
  static constexpr int NF = 2, NPRE = 5, NOUT = 3, NMAX = 0, REC = 2;
  static constexpr bool PAIRED = PAIR;
  static constexpr bool Q2 = false;
  static constexpr bool LEAN = !PAIR;  // (80 steps of 304^3, both loops: 23.2 ms without, 23.45 with)
  static constexpr bool DAMP = true;
  const float *__restrict__ s1;
  const float *__restrict__ r1;
  float *__restrict__ s0;
  float *__restrict__ r0;
  const float *__restrict__ vel1;
  const float *__restrict__ vel2;
  float *__restrict__ img;
  int s_prop, r_prop;
  // source amplitude injected into the current level by the previous
  // iteration (cpu_prop.cc:89-92), applied here to the old level it became
  Points pts;
  const float *__restrict__ amp_pre;
  int pre;
  RecMap rm;
  const float *__restrict__ gin;  // injected per receiver (nullptr: nothing)
  int nx, ny;

  __device__ int rec_slot(const SrcPln &pl) const { return gin ? pl.slot : -1; }
  __device__ const int *rec_map(int slot) const { return rec_plane(rm, slot, nx, ny); }
  __device__ float rec_value(int i) const { return gin[i]; }
  __device__ PtsBlk block(int x0, int x1, int y0, int y1, int z0, int z1) const {
    return pre ? points_of_block(pts, x0, x1, y0, y1, z0, z1) : PtsBlk{0u, 1, 0};
  }
  template <int VX>
  __device__ void ldv(const PtsBlk &, int f, uint32_t po, uint32_t o, float (&v)[VX]) const {
    ld_vec<VX>(f == 0 ? s1 : r1, po, o, 1.f, v);
  }
  template <int VX>
  __device__ void ldv2(const PtsBlk &, uint32_t po, uint32_t o, float (&v)[2][VX]) const {
    ld_vec2<VX>((const float2 *)s1, po, o, v[0], v[1]);
  }
  __device__ SrcPln plane(const PtsBlk &blk, int z) const {
    return {points_on_plane(pts, blk, z), ldc(rm.plane_slot, z)};
  }
  template <int VX>
  __device__ void prefetchv(const PtsBlk &, float (&p)[NPRE][VX], uint32_t po,
                            uint32_t o) const {
    if constexpr (PAIRED) {
      ld_vec2<VX>((const float2 *)s0, po, o, p[0], p[1]);
    } else {
      ld_vec<VX>(s0, po, o, 1.f, p[0]);
      ld_vec<VX>(r0, po, o, 1.f, p[1]);
    }
    ld_vec<VX>(vel1, po, o, 1.f, p[2]);
    ld_vec<VX>(vel2, po, o, 1.f, p[3]);
    ld_vec<VX>(img, po, o, 1.f, p[4]);
  }
  template <int VX>
  __device__ void storev(const PtsBlk &, uint32_t po, uint32_t o,
                         const float (&out)[NOUT][VX]) const {
    // no hint: every array here is read again by the next step (304^3 227.9 ->
    // 223.4 us, 160^3 29.4 -> 27.9; with the hint on the loads too, 160^3 35)
    if constexpr (PAIRED) {  // out[0] is the old s when s stands still
      const float one[2] = {1.f, 1.f};
      st_pair<VX, false>((float2 *)s0, po, o, out[0], out[1], one);
    } else {
      if (s_prop) st_vec<VX, false>(s0, po, o, out[0], 1.f);
      st_vec<VX, false>(r0, po, o, out[1], 1.f);
    }
    st_vec<VX, false>(img, po, o, out[2], 1.f);
  }
  __device__ void cell(const PtsBlk &, const SrcPln &pl, const CellArgs &c, const float *lap,
                       const float *ctr, const float *p, float (&out)[NOUT],
                       float (&)[NF]) const {
    float sn;
    if (s_prop) {
      float so = p[0];
      if (pl.pm) so = add_points(pts, pl.pm, c.x, c.y, so, amp_pre);
      sn = p[2] * lap[0] + ctr[0] + ctr[0] - so;
    } else {
      sn = p[0];
    }
    const float b = c.b;
    float rn = r_prop ? leap(b, p[3], lap[1], ctr[1], p[1]) : mul_r(b, mul_r(b, p[1]));
    if (c.rs >= 0) {
      // the receivers of a cell one after the other, as the reference adds them
      if (c.ri >= 0) rn = add_r(rn, c.rg);
      if (rm.shared && c.ri >= 0)
        for (int i = rm.rnext[c.ri]; i >= 0; i = rm.rnext[i]) rn = add_r(rn, gin[i]);
    }
    out[0] = sn;
    out[1] = rn;
    out[2] = p[4] + sn * rn;
  }
};

// ------------------------------------- exact adjoint: background recompute
// HINT: narrow levels with the non-temporal hint on the stores and the
// velocity, for grids past the memory-side cache; the same bit of LamOp, where
// the image takes it too.  us per step of both without -> with: FP16 304^3 172 ->
// 185, 384 x 384 x 352 308 -> 291, 448 x 448 x 400 489 -> 463, 640 x 640 x 500 1464
// -> 1350; 24-bit 304^3 233 -> 244, 384 x 384 x 352 409 -> 409, 448 x 448 x 400 674
// -> 642, 640 x 640 x 500 1875 -> 1744.
template <int SCATTER, class T, bool HINT = false>
struct SrecOp {
  static constexpr bool H = kScaled<T>;
  static constexpr int NF = 1, NPRE = 2, NOUT = 2, NMAX = H ? 1 : 0, REC = 0;
  static constexpr bool PAIRED = false;
  static constexpr bool Q2 = kNarrow<T>;  // steps in pairs (march_tile)
  static constexpr bool LEAN = true;
  static constexpr bool DAMP = true;
  const T *__restrict__ s1;
  // old s level (read) and new s level (written): the same buffer, or with
  // scatter 0 two levels of the segment history (level k of s is sigma of
  // step k-1)
  const T *s0;
  T *s_new;
  const float *__restrict__ vel;
  T *__restrict__ sig;  // scatter operand of this step (nullptr: none)
  Points pts;
  const float *__restrict__ amp;
  Ring ring;
  Slots sl;
  float gain, tapsum;
  float *hscale;  // FP16: scale of this step's sigma
  uint32_t nlev;  // cells of a level

  __device__ Blk1 block(int x0, int x1, int y0, int y1, int z0, int z1) const {
    Blk1 b;
    b.pb = points_of_block(pts, x0, x1, y0, y1, z0, z1);
    b.ic = b.io = b.sn = b.sh = 1.f;
    if constexpr (H) {
      b.ic = 1.f / ring.scale[sl.cur];
      b.io = 1.f / ring.scale[sl.old];
      const float ms = ring_max(ring, sl.cur);
      const float bs = gain * ms + ring_max(ring, sl.old) + amp_sum(pts, amp);
      b.sn = level_scale(bs);
      b.sh = SCATTER == 0 ? b.sn : level_scale(tapsum * ms);
    }
    return b;
  }
  __device__ void first(const Blk1 &b) const {
    ring.scale[sl.nxt] = b.sn;
    ring.maxb[sl.clr] = 0u;
    if (hscale) *hscale = b.sh;
  }
  __device__ void publish_max(int, float m) const {
    atomicMax(&ring.maxb[sl.nxt], __float_as_uint(m));
  }
  template <int VX>
  __device__ void ldv(const Blk1 &b, int, uint32_t po, uint32_t o, float (&v)[VX]) const {
    ld_vec<VX>(s1, po, o, b.ic, v, nlev);
  }
  __device__ uint32_t plane(const Blk1 &b, int z) const {
    return points_on_plane(pts, b.pb, z);
  }
  template <int VX>
  __device__ void prefetchv(const Blk1 &b, float (&p)[NPRE][VX], uint32_t po,
                            uint32_t o) const {
    // FP32: the old level and the stores with the non-temporal hint; narrow
    // levels without any, but see HINT (FP16 background and adjoint state, us per step of
    // each together: 304^3 196.9 -> 184.9, 160^3 49.7 -> 47.1)
    ld_vec<VX, !kNarrow<T>>(s0, po, o, b.io, p[0], nlev);
    ld_vec<VX, HINT>(vel, po, o, 1.f, p[1]);
  }
  template <int VX>
  __device__ void storev(const Blk1 &b, uint32_t po, uint32_t o,
                         const float (&out)[NOUT][VX]) const {
    st_vec<VX, !kNarrow<T> || HINT>(s_new, po, o, out[0], b.sn, nlev);
    if (sig) st_vec<VX, !kNarrow<T> || HINT>(sig, po, o, out[1], b.sh, nlev);
  }
  __device__ void cell(const Blk1 &, uint32_t pm, const CellArgs &c, const float *lap,
                       const float *ctr, const float *p, float (&out)[NOUT],
                       float (&tmax)[NF]) const {
    const float bb = c.b;
    float sn = leap(bb, p[1], lap[0], ctr[0], p[0]);
    if (pm) sn = add_points(pts, pm, c.x, c.y, sn, amp);
    if constexpr (H) tmax[0] = fmaxf(tmax[0], fabsf(sn));
    out[0] = sn;
    out[1] = SCATTER == 0 ? sn : mul_r(bb, lap[0]);
  }
};

// ---------------------------------------- exact adjoint: adjoint-state step
// nu = V B lambda obeys the forward recursion with V B-weighted receiver
// injection; the image accumulates sigma * nu and is divided by V B at the end.
template <class T, bool HINT = false>
struct LamOp {
  static constexpr bool H = kScaled<T>;
  static constexpr int NF = 1, NPRE = 4, NOUT = 2, NMAX = H ? 1 : 0, REC = 2;
  static constexpr bool PAIRED = false;
  static constexpr bool Q2 = kNarrow<T>;  // steps in pairs (march_tile)
  static constexpr bool LEAN = true;
  static constexpr bool DAMP = true;
  const T *__restrict__ u1;
  T *__restrict__ u0;
  const float *__restrict__ vel;
  const T *__restrict__ sig;
  float *__restrict__ acc;
  RecMap rm;
  const float *__restrict__ gin;  // injected per receiver cell (nullptr: nothing)
  int nx, ny;
  Ring ring;
  Slots sl;
  float gain;
  float inj;                // bound of |V B P^T w| per unit of max |trace|
  const unsigned *trmax;    // max |trace| as float bits
  const float *hscale;      // FP16: scale of sigma
  uint32_t nlev;            // cells of a level

  __device__ Blk1 block(int, int, int, int, int, int) const {
    Blk1 b;
    b.pb = PtsBlk{0u, 1, 0};
    b.ic = b.io = b.sn = b.sh = 1.f;
    if constexpr (H) {
      b.ic = 1.f / ring.scale[sl.cur];
      b.io = 1.f / ring.scale[sl.old];
      const float bu = gain * ring_max(ring, sl.cur) + ring_max(ring, sl.old) +
                       (gin ? inj * __uint_as_float(*trmax) : 0.f);
      b.sn = level_scale(bu);
      b.sh = 1.f / *hscale;
    }
    return b;
  }
  __device__ void first(const Blk1 &b) const {
    ring.scale[sl.nxt] = b.sn;
    ring.maxb[sl.clr] = 0u;
  }
  __device__ void publish_max(int, float m) const {
    atomicMax(&ring.maxb[sl.nxt], __float_as_uint(m));
  }
  template <int VX>
  __device__ void ldv(const Blk1 &b, int, uint32_t po, uint32_t o, float (&v)[VX]) const {
    ld_vec<VX>(u1, po, o, b.ic, v, nlev);
  }
  __device__ int plane(const Blk1 &, int z) const { return ldc(rm.plane_slot, z); }
  __device__ int rec_slot(int slot) const { return gin ? slot : -1; }
  __device__ const int *rec_map(int slot) const { return rec_plane(rm, slot, nx, ny); }
  __device__ float rec_value(int i) const { return gin[i]; }
  template <int VX>
  __device__ void prefetchv(const Blk1 &b, float (&p)[NPRE][VX], uint32_t po,
                            uint32_t o) const {
    // FP32: the non-temporal hint on the levels, not on velocity and image
    // (304^3 134.8 us; without any 143.5); narrow levels without any, but see
    // HINT at SrecOp (24-bit 224^3 61.7 -> 58.4)
    ld_vec<VX, !kNarrow<T>>(u0, po, o, b.io, p[0], nlev);
    ld_vec<VX, !kNarrow<T>>(sig, po, o, b.sh, p[2], nlev);
    ld_vec<VX, HINT>(vel, po, o, 1.f, p[1]);
    ld_vec<VX, HINT>(acc, po, o, 1.f, p[3]);
  }
  template <int VX>
  __device__ void storev(const Blk1 &b, uint32_t po, uint32_t o,
                         const float (&out)[NOUT][VX]) const {
    st_vec<VX, !kNarrow<T> || HINT>(u0, po, o, out[0], b.sn, nlev);
    st_vec<VX, HINT>(acc, po, o, out[1], 1.f);
  }
  __device__ void cell(const Blk1 &, int slot, const CellArgs &c, const float *lap,
                       const float *ctr, const float *p, float (&out)[NOUT],
                       float (&tmax)[NF]) const {
    const float bb = c.b, v = p[1];
    float un = leap(bb, v, lap[0], ctr[0], p[0]);
    if (c.rs >= 0 && c.ri >= 0) un = fma_r(mul_r(v, bb), c.rg, un);
    if constexpr (H) tmax[0] = fmaxf(tmax[0], fabsf(un));
    out[0] = un;
    out[1] = fma_r(p[2], un, p[3]);
  }
};

// ------------------------------------------------------------ shot batches
// The forward op of every shot of a batch: the op's arrays start at the
// batch's first shot and are moved by the shot's descriptor.
template <int SCATTER, class T>
struct BatchFwd {
  // without the non-temporal hint: it slowed the batch (32 windowed shots)
  // by about 5 % where it sped up single shots
  using Op = FwdOp<SCATTER, T, false, true>;
  Op base;
  const float *sponge;
  float *rings;
  const ShotDesc *__restrict__ desc;
  int step, npts_total;
  struct Shot {
    Grid g;
    Sponge sp;
    Op op;
  };
  __device__ Shot shot(int s, int tw, int ty, int zc) const {
    const ShotDesc d = desc[s];
    Shot r;
    r.g = tile_grid(d.nx, d.ny, d.nz, tw, ty, zc);
    r.sp.bx = sponge + d.sp0;
    r.sp.by = sponge + d.sp0 + d.nx;
    r.sp.bz = sponge + d.sp0 + d.nx + d.ny;
    Op &o = r.op;
    o = base;
    o.sr1 = base.sr1 + d.cell0;
    o.sr0 = base.sr0 + d.cell0;
    o.srn = base.srn + d.cell0;
    o.vel = base.vel + d.cell0;
    o.model = base.model + d.cell0;
    o.hist = nullptr;
    o.pts.p = base.pts.p + d.pts0;
    o.pts.n = d.npts;
    o.amp = base.amp + (long long)step * npts_total + d.pts0;
    o.rm.plane_slot = base.rm.plane_slot + d.slot0;
    o.rm.rmap = base.rm.rmap + d.rmap0;
    o.rm.rnext = base.rm.rnext + d.rnext0;
    o.rm.nrec = d.nrec;
    o.rv = base.rv ? base.rv + d.rnext0 : nullptr;
    o.nx = d.nx;
    o.ny = d.ny;
    o.rg = rings + d.ring0;
    o.gain = d.gain;
    o.nlev = (uint32_t)d.nx * d.ny * d.nz;
    return r;
  }
};

// The exact adjoint's ops for every shot of a batch, moved per shot as
// BatchFwd: the background recompute and the adjoint-state step, with each
// shot's scale rings, bound gain, receiver tables and traces.
template <int SCATTER, class T>
struct BatchSrec {
  using Op = SrecOp<SCATTER, T>;
  Op base;
  const float *sponge;
  float *rings;
  const ShotDesc *__restrict__ desc;
  int step, npts_total;
  struct Shot {
    Grid g;
    Sponge sp;
    Op op;
  };
  __device__ Shot shot(int s, int tw, int ty, int zc) const {
    const ShotDesc d = desc[s];
    Shot r;
    r.g = tile_grid(d.nx, d.ny, d.nz, tw, ty, zc);
    r.sp.bx = sponge + d.sp0;
    r.sp.by = sponge + d.sp0 + d.nx;
    r.sp.bz = sponge + d.sp0 + d.nx + d.ny;
    Op &o = r.op;
    o = base;
    o.s1 = base.s1 + d.cell0;
    o.s0 = base.s0 + d.cell0;
    o.s_new = base.s_new + d.cell0;
    o.vel = base.vel + d.cell0;
    o.sig = base.sig ? base.sig + d.cell0 : nullptr;
    o.pts.p = base.pts.p + d.pts0;
    o.pts.n = d.npts;
    o.amp = base.amp + (long long)step * npts_total + d.pts0;
    o.ring = {rings + d.ring0 + BR_S, (unsigned *)(rings + d.ring0 + BR_S + 4)};
    o.gain = d.gain;
    o.hscale = base.hscale ? base.hscale + s : nullptr;
    o.nlev = (uint32_t)d.nx * d.ny * d.nz;
    return r;
  }
};

template <class T>
struct BatchLam {
  using Op = LamOp<T>;
  Op base;
  const float *sponge;
  float *rings;
  const ShotDesc *__restrict__ desc;
  int step, npts_total;
  struct Shot {
    Grid g;
    Sponge sp;
    Op op;
  };
  __device__ Shot shot(int s, int tw, int ty, int zc) const {
    const ShotDesc d = desc[s];
    Shot r;
    r.g = tile_grid(d.nx, d.ny, d.nz, tw, ty, zc);
    r.sp.bx = sponge + d.sp0;
    r.sp.by = sponge + d.sp0 + d.nx;
    r.sp.bz = sponge + d.sp0 + d.nx + d.ny;
    Op &o = r.op;
    o = base;
    o.u1 = base.u1 + d.cell0;
    o.u0 = base.u0 + d.cell0;
    o.vel = base.vel + d.cell0;
    o.sig = base.sig + d.cell0;
    o.acc = base.acc + d.cell0;
    o.rm.plane_slot = base.rm.plane_slot + d.slot0;
    o.rm.rmap = base.rm.rmap + d.rmap0;
    o.rm.rnext = base.rm.rnext + d.rnext0;
    o.rm.nrec = d.nrec;
    o.gin = base.gin ? base.gin + d.rnext0 : nullptr;
    o.nx = d.nx;
    o.ny = d.ny;
    o.ring = {rings + d.ring0 + BR_U, (unsigned *)(rings + d.ring0 + BR_U + 4)};
    o.gain = d.gain;
    // the single-shot bound's factors in its order: (max(V) |tab|) per cell
    o.inj = d.vmax * base.inj * (float)d.per_cell;
    o.trmax = (const unsigned *)(rings + d.ring0 + BR_MAXTR);
    o.hscale = base.hscale ? base.hscale + s : nullptr;
    o.nlev = (uint32_t)d.nx * d.ny * d.nz;
    return r;
  }
};

// ------------------------------------------------------------- launchers

// switch (shape) { case i: return F<..., RY, WY, VX, LA, LX>(ARGS); } over kShapes
#define BORN_SHAPE_CASES(F, OP, ...)                         \
  case 0: return F<OP, 2, 4, 1, 1, 64>(__VA_ARGS__);         \
  case 1: return F<OP, 4, 4, 1, 1, 64>(__VA_ARGS__);         \
  case 2: return F<OP, 2, 8, 1, 1, 64>(__VA_ARGS__);         \
  case 3: return F<OP, 2, 16, 1, 1, 64>(__VA_ARGS__);        \
  case 4: return F<OP, 1, 8, 1, 1, 64>(__VA_ARGS__);         \
  case 5: return F<OP, 1, 16, 1, 1, 64>(__VA_ARGS__);        \
  case 6: return F<OP, 1, 4, 2, 1, 32>(__VA_ARGS__);         \
  case 7: return F<OP, 2, 4, 2, 1, 32>(__VA_ARGS__);         \
  case 8: return F<OP, 1, 8, 2, 1, 32>(__VA_ARGS__);         \
  case 9: return F<OP, 2, 8, 2, 1, 32>(__VA_ARGS__);         \
  case 10: return F<OP, 1, 12, 2, 1, 32>(__VA_ARGS__);       \
  case 11: return F<OP, 2, 2, 2, 1, 32>(__VA_ARGS__);        \
  case 12: return F<OP, 2, 4, 1, 2, 64>(__VA_ARGS__);        \
  case 13: return F<OP, 4, 4, 1, 2, 64>(__VA_ARGS__);        \
  case 14: return F<OP, 2, 8, 1, 2, 64>(__VA_ARGS__);        \
  case 15: return F<OP, 2, 16, 1, 2, 64>(__VA_ARGS__);       \
  case 16: return F<OP, 1, 8, 1, 2, 64>(__VA_ARGS__);        \
  case 17: return F<OP, 1, 16, 1, 2, 64>(__VA_ARGS__);       \
  case 18: return F<OP, 1, 4, 2, 2, 32>(__VA_ARGS__);        \
  case 19: return F<OP, 2, 4, 2, 2, 32>(__VA_ARGS__);        \
  case 20: return F<OP, 1, 8, 2, 2, 32>(__VA_ARGS__);        \
  case 21: return F<OP, 2, 8, 2, 2, 32>(__VA_ARGS__);        \
  case 22: return F<OP, 1, 12, 2, 2, 32>(__VA_ARGS__);       \
  case 23: return F<OP, 2, 2, 2, 2, 32>(__VA_ARGS__);        \
  case 24: return F<OP, 1, 4, 4, 1, 16>(__VA_ARGS__);        \
  case 25: return F<OP, 1, 2, 4, 1, 16>(__VA_ARGS__);        \
  case 26: return F<OP, 2, 2, 4, 1, 16>(__VA_ARGS__);        \
  case 27: return F<OP, 1, 8, 4, 1, 16>(__VA_ARGS__);        \
  case 28: return F<OP, 1, 1, 4, 1, 8>(__VA_ARGS__);         \
  case 29: return F<OP, 1, 3, 4, 1, 8>(__VA_ARGS__);         \
  case 30: return F<OP, 1, 4, 4, 2, 16>(__VA_ARGS__);        \
  case 31: return F<OP, 1, 2, 4, 2, 16>(__VA_ARGS__);        \
  case 32: return F<OP, 1, 2, 2, 1, 16>(__VA_ARGS__);        \
  case 33: return F<OP, 2, 1, 2, 1, 16>(__VA_ARGS__);


inline Grid make_grid(const Geometry &geo, const TileShape &ts, int zc) {
  return tile_grid(geo.nx, geo.ny, geo.nz, ts.lx * ts.vx, ts.ry * (kTX * ts.wy / ts.lx),
                   zc > 0 ? zc : 32);
}

template <class Op, int RY, int WY, int VX, int LA, int LX>
hipError_t launch_shape(const Geometry &geo, const Tune &tu, const Op &op, hipStream_t st) {
  if (geo.nx % VX) return hipErrorInvalidValue;
  Grid g = make_grid(geo, {RY, WY, VX, LA, LX}, tu.zchunk);
  g.back = tu.back;
  const int nb = g.ntx * g.nty * g.ntz;
  hipLaunchKernelGGL((march_kernel<Op, RY, WY, VX, LA, LX>), dim3(nb), dim3(kTX * WY), 0, st,
                     g, geo.taps, geo.sponge, op);
  return hipGetLastError();
}

template <class Op>
hipError_t launch(const Geometry &geo, const Tune &tu, const Op &op, hipStream_t st) {
  switch (tu.shape) {
    BORN_SHAPE_CASES(launch_shape, Op, geo, tu, op, st)
    default: return hipErrorInvalidValue;
  }
}

inline Points to_points(const SrcPts &s) { return {(const int4 *)s.p, s.n}; }
inline int pack_slots(const Slots &s) { return s.cur | s.old << 8 | s.nxt << 16 | s.clr << 24; }

template <class T>
T *as(const void *p) {
  return (T *)p;
}

template <class BOp, int RY, int WY, int VX, int LA, int LX>
hipError_t launch_batch_shape(const Taps &taps, const Tune &tu, const BatchCommon &b,
                              const BOp &op, hipStream_t st) {
  if (b.nshots < 1 || b.nshots > kMaxBatch) return hipErrorInvalidValue;
  BatchTiles bt{};
  bt.n = b.nshots;
  bt.zc = tu.zchunk > 0 ? tu.zchunk : 32;
  bt.back = tu.back;
  int tiles = 0;
  for (int s = 0; s < b.nshots; s++) {
    const ShotDesc &d = b.host_desc[s];
    if (d.nx % VX) return hipErrorInvalidValue;
    const Grid g = tile_grid(d.nx, d.ny, d.nz, LX * VX, RY * (kTX * WY / LX), bt.zc);
    bt.tile0[s] = tiles;
    tiles += g.ntx * g.nty * g.ntz;
  }
  bt.tile0[b.nshots] = tiles;
  hipLaunchKernelGGL((march_batch_kernel<BOp, RY, WY, VX, LA, LX>), dim3(tiles),
                     dim3(kTX * WY), 0, st, bt, taps, op);
  return hipGetLastError();
}

template <class BOp>
hipError_t launch_batch(const Taps &taps, const Tune &tu, const BatchCommon &b,
                               const BOp &op, hipStream_t st) {
  switch (tu.shape) {
    BORN_SHAPE_CASES(launch_batch_shape, BOp, taps, tu, b, op, st)
    default: return hipErrorInvalidValue;
  }
}

// ---- the launchers of each op type.  They are templates here and are
// instantiated explicitly, each in one translation unit (born_k_*.hip, built
// in parallel); born_kernels.hip declares them extern and dispatches.

template <int SCATTER, class T, bool PAIR, bool HINT>
hipError_t fwd_step(const Geometry &geo, const Tune &tu, const FwdStep &a, hipStream_t st) {
  FwdOp<SCATTER, T, true, PAIR, HINT> op{};
  op.s1 = as<T>(a.s1); op.r1 = as<T>(a.r1); op.s0 = as<T>(a.s0); op.r0 = as<T>(a.r0);
  op.s_new = as<T>(a.s_new ? a.s_new : a.s0);
  op.sr1 = (const PairOf<T> *)a.s1; op.sr0 = (const PairOf<T> *)a.s0;
  op.srn = (PairOf<T> *)(a.s_new ? a.s_new : a.s0);
  op.vm = (const float2 *)a.vm; op.hist = as<T>(a.hist);
  if (!a.vm) return hipErrorInvalidValue;
  op.pts = to_points(a.src); op.amp = a.amp;
  op.rm = a.rec; op.rv = a.rv; op.nx = geo.nx; op.ny = geo.ny;
  op.rg = a.rg; op.slots = pack_slots(a.h.sl);
  op.gain = a.h.gain; op.tapsum = a.h.tapsum; op.hscale = a.hscale;
  op.nlev = (uint32_t)geo.nx * geo.ny * geo.nz;
  return launch(geo, tu, op, st);
}

template <bool PAIR>
hipError_t radj_step(const Geometry &geo, const Tune &tu, const RadjStep &a, hipStream_t st) {
  RadjOp<PAIR> op{};
  op.s1 = a.s1; op.r1 = a.r1; op.s0 = a.s0; op.r0 = a.r0;
  op.vel1 = a.vel1; op.vel2 = a.vel2; op.img = a.img;
  op.s_prop = a.s_prop; op.r_prop = a.r_prop;
  op.pts = to_points(a.src); op.amp_pre = a.amp_pre; op.pre = a.pre;
  op.rm = a.rec; op.gin = a.gin; op.nx = geo.nx; op.ny = geo.ny;
  return launch(geo, tu, op, st);
}

template <int SCATTER, class T, bool HINT>
hipError_t srec_step(const Geometry &geo, const Tune &tu, const SrecStep &a, hipStream_t st) {
  SrecOp<SCATTER, T, HINT> op{};
  op.s1 = as<T>(a.s1); op.s0 = as<T>(a.s0); op.vel = a.vel; op.sig = as<T>(a.sig);
  op.s_new = as<T>(a.s_new ? a.s_new : a.s0);
  op.pts = to_points(a.src); op.amp = a.amp;
  op.ring = a.ring; op.sl = a.h.sl; op.gain = a.h.gain; op.tapsum = a.h.tapsum;
  op.hscale = a.hscale;
  op.nlev = (uint32_t)geo.nx * geo.ny * geo.nz;
  return launch(geo, tu, op, st);
}

template <class T, bool HINT>
hipError_t lam_step(const Geometry &geo, const Tune &tu, const LamStep &a, hipStream_t st) {
  LamOp<T, HINT> op{};
  op.u1 = as<T>(a.u1); op.u0 = as<T>(a.u0); op.vel = a.vel; op.sig = as<T>(a.sig);
  op.acc = a.acc; op.rm = a.rec; op.gin = a.gin; op.nx = geo.nx; op.ny = geo.ny;
  op.ring = a.ring; op.sl = a.h.sl; op.gain = a.h.gain; op.inj = a.inj;
  op.trmax = a.trmax; op.hscale = a.hscale;
  op.nlev = (uint32_t)geo.nx * geo.ny * geo.nz;
  return launch(geo, tu, op, st);
}

template <int SCATTER, class T>
hipError_t batch_fwd_step(const Taps &taps, const Tune &tu, const BatchFwdStep &b,
                          hipStream_t st) {
  const FwdStep &a = b.a;
  BatchFwd<SCATTER, T> bop{};
  auto &op = bop.base;
  op.sr1 = (const PairOf<T> *)a.s1; op.sr0 = (const PairOf<T> *)a.s0;
  op.srn = (PairOf<T> *)a.s0;
  op.vel = a.vel; op.model = a.model; op.hist = nullptr;
  op.pts = to_points(a.src); op.amp = a.amp;
  op.rm = a.rec; op.rv = a.rv;
  op.slots = pack_slots(a.h.sl); op.tapsum = a.h.tapsum; op.hscale = nullptr;
  bop.sponge = b.sponge; bop.rings = b.rings; bop.desc = b.desc; bop.step = b.step;
  bop.npts_total = b.npts_total;
  return launch_batch(taps, tu, b, bop, st);
}

template <int SCATTER, class T>
hipError_t batch_srec_step(const Taps &taps, const Tune &tu, const BatchSrecStep &b,
                           hipStream_t st) {
  const SrecStep &a = b.a;
  BatchSrec<SCATTER, T> bop{};
  auto &op = bop.base;
  op.s1 = as<T>(a.s1); op.s0 = as<T>(a.s0); op.vel = a.vel; op.sig = as<T>(a.sig);
  op.s_new = as<T>(a.s_new ? a.s_new : a.s0);
  op.pts = to_points(a.src); op.amp = a.amp;
  op.sl = a.h.sl; op.tapsum = a.h.tapsum; op.hscale = a.hscale;
  bop.sponge = b.sponge; bop.rings = b.rings; bop.desc = b.desc; bop.step = b.step;
  bop.npts_total = b.npts_total;
  return launch_batch(taps, tu, b, bop, st);
}

template <class T>
hipError_t batch_lam_step(const Taps &taps, const Tune &tu, const BatchLamStep &b,
                          hipStream_t st) {
  const LamStep &a = b.a;
  BatchLam<T> bop{};
  auto &op = bop.base;
  op.u1 = as<T>(a.u1); op.u0 = as<T>(a.u0); op.vel = a.vel; op.sig = as<T>(a.sig);
  op.acc = a.acc; op.rm = a.rec; op.gin = a.gin; op.sl = a.h.sl; op.inj = a.inj; op.hscale = a.hscale;
  bop.sponge = b.sponge; bop.rings = b.rings; bop.desc = b.desc; bop.step = b.step;
  bop.npts_total = b.npts_total;
  return launch_batch(taps, tu, b, bop, st);
}

// the instantiations, one translation unit each (F: template or extern template)
#define BORN_FWD_STEP(F, S, T)                                                          \
  F hipError_t fwd_step<S, T, kNarrow<T>, false>(const Geometry &, const Tune &,         \
                                                 const FwdStep &, hipStream_t)
// FP32 levels of s and r together
#define BORN_FWD_STEP_SR(F, S) \
  F hipError_t fwd_step<S, float, true, false>(const Geometry &, const Tune &,           \
                                               const FwdStep &, hipStream_t)
// the same with the non-temporal hint
#define BORN_FWD_STEP_HINT(F, S)                                                        \
  F hipError_t fwd_step<S, float, true, true>(const Geometry &, const Tune &,            \
                                              const FwdStep &, hipStream_t)
#define BORN_RADJ_STEP(F, PAIR) \
  F hipError_t radj_step<PAIR>(const Geometry &, const Tune &, const RadjStep &, hipStream_t)
#define BORN_SREC_STEP(F, S, T) \
  F hipError_t srec_step<S, T, false>(const Geometry &, const Tune &, const SrecStep &, hipStream_t)
// narrow levels with the hint
#define BORN_SREC_STEP_HINT(F, S, T) \
  F hipError_t srec_step<S, T, true>(const Geometry &, const Tune &, const SrecStep &, hipStream_t)
#define BORN_LAM_STEP(F, T) \
  F hipError_t lam_step<T, false>(const Geometry &, const Tune &, const LamStep &, hipStream_t)
#define BORN_LAM_STEP_HINT(F, T) \
  F hipError_t lam_step<T, true>(const Geometry &, const Tune &, const LamStep &, hipStream_t)
#define BORN_BATCH_SREC_STEP(F, S, T)                                                   \
  F hipError_t batch_srec_step<S, T>(const Taps &, const Tune &, const BatchSrecStep &, \
                                     hipStream_t)
#define BORN_BATCH_LAM_STEP(F, T) \
  F hipError_t batch_lam_step<T>(const Taps &, const Tune &, const BatchLamStep &, hipStream_t)
#define BORN_BATCH_FWD_STEP(F, S, T)                                                     \
  F hipError_t batch_fwd_step<S, T>(const Taps &, const Tune &, const BatchFwdStep &, \
                                    hipStream_t)

}  // namespace born
