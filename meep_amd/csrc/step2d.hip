// step2d.hip — several FDTD steps of a 2D chunk in one launch.
//
// A 2D chunk is small: 320 x 160 cells are 4 MB of FP64 state, and a step of it was six
// launches of 6.9 us that each waited for memory once (47 us a step, 0.07 TB/s).  Here a block
// loads a tile of S2_ROWS x 64 points into registers, steps it `nsteps` times and stores the
// core of the tile: every step spoils one more point on each side, so a tile's core is the tile
// less its margin of S2_STEPS points (and one more above, for the monitors' centring), and
// neighbouring tiles recompute each other's margins from the same old values.  Arrays are
// double-buffered, so no block waits for another.
//
// A lane owns one column (the stride-1 direction) and a wave K consecutive rows of it: the
// stride-1 neighbour of a curl is a lane shift, the other neighbour a register of the same
// thread, and only the wave's first row of E and last row of H go through LDS.  The update of
// each point is that of k_fast (kernels.hip), branch by branch: the curl with its four uPML
// forms, currents, walls, E = chi1inv (D - P - dipoles) or H = B with the f_w branch, and the
// poles; the uPML branches run only in tiles that meet a profile (uniform per block).
//
// What bounds it: instruction issue in the tiles that meet a uPML corner (about three times a
// plain tile's time), then the load of a tile before its first step (4 us).  Per step with its
// monitors, one-step kernels -> here: 320 x 160 FP64 (88 tiles) 47 us -> 5.2 us; 401 x 263 FP32
// TE with a Drude pole and a field map over the cell 61 us -> 14.2 us; 64 squares of 128 to
// 512 cells together 181 us -> 75 us.  A plain tile pays for the registers of a uPML tile: 113 to
// 128 VGPRs, with spills of 0 to 34 of them in FP32 (20 to 140 bytes of scratch a lane from TM with
// two poles on) and 16 (TM, no pole) to 153 (TE, two poles; 400 bytes) in FP64, and 83 to 185
// SGPRs in every form.  Rows x columns 32 x 64 with 16 waves of 2 rows each: 4 rows a
// thread and 8 waves have more neighbours in the same wave but half the waves to issue from
// (32 us against 19 for up to 8 steps of a 400 x 300 FP32 cell).
#include "engine.hpp"
#include "stencil.hpp"

#include <hip/hip_runtime.h>

namespace mx {

// the next / previous lane's value (0 past the wave's ends)
__device__ __forceinline__ float lane_next(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_prev(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_next(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_prev(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// A pointer read from device memory, as one into global memory: through a plain pointer the
// compiler emits flat accesses, which wait for the LDS counter too.
template <class T> using Glob = __attribute__((address_space(1))) T *;
template <class T> __device__ __forceinline__ Glob<T> global(T *p) { return (Glob<T>)p; }

// a value that is the same in every lane of the wave, in scalar registers
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ bool uni(bool v) { return __builtin_amdgcn_readfirstlane(int(v)) != 0; }
template <class T> __device__ __forceinline__ Glob<T> uni(T *p) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = uint32_t(uni(int(uint32_t(u)))), hi = uint32_t(uni(int(uint32_t(u >> 32))));
  return (Glob<T>)(T *)((uint64_t(hi) << 32) | lo);
}

// one axis's uPML coefficients at a point; on: the profile is active there (0, 1, 1 where not)
template <class R> struct S2Prof {
  R sig, kap, sinv;
  bool on;
};
template <class R> __device__ __forceinline__ S2Prof<R> s2_prof(Glob<const R> sig, Glob<const R> kap, Glob<const R> siginv, int j, int ysh, int n) {
  S2Prof<R> p{R(0), R(1), R(1), false};
  if (j < 0 || j > n) return p;
  const int k = 2 * j + ysh;
  p.sig = sig[k];
  p.kap = kap[k];
  p.sinv = siginv[k];
  p.on = p.sig != R(0) || p.kap != R(1);
  return p;
}

// Yee shift of the component of slot C along axis A in the B (mag) or D phase: the component's
// own axis is shifted for E and D, the others for H and B (slot 2, along Z, is never shifted
// along X or Y as E, always as H)
template <bool MAG, int C, int A> constexpr int s2_ysh() { return MAG ? (C == A ? 0 : 1) : (C == A ? 1 : 0); }

// NW waves of K rows each; TM: B has X and Y components, D and E one along Z; else the reverse
template <class R, bool TM, int NP, int NW, int K> struct Tile2d {
  static constexpr int RX = NW * K;
  static constexpr int NPA = NP > 0 ? NP : 1;
  const Step2dArgs<R> &a;
  const Step2dLaunch<R> &l;
  R *bE, *bH;     // boundary rows: the first E row of wave w at w, the last H row of wave w at w + 1
  R (*px)[3][RX]; // the X profile of the tile's rows, by Yee shift: sig, kap, siginv
  double *vals;   // the launch's source values, a row per step
  SrcSet *set;    // the sources of the two phases
  int lane, wave, x0, y, X0, Y0;
  R dtdx;
  bool srcs[2], mu[3];
  bool polar[NPA][3];       // pole p polarises slot c (P and sigma exist)
  uint64_t tmask[3];        // per list, SRC_TAB bits per row: entries on the point
  unsigned tcomp[3][3];     // per list and slot: its entries
  // A property of points that is a product of one of the row (the same in the whole wave: scalar
  // bits) and one of the column (a lane condition): inside the grid, updated by slot c, zeroed by
  // a wall (either), inside pole p's box (none where the tile does not meet it)
  unsigned rin, rown[3], rzero[3], rpin[NPA];
  bool cin, cown[3], czero[3], cpin[NPA];
  unsigned rowx[2]; // rows where the X profile is active, by Yee shift
  bool pmly;        // the tile meets an active profile of Y
  S2Prof<R> py[2];          // the Y profile at the lane, by Yee shift
  R f[3][K], e[3][K], chi[3][K]; // chi: of the E components
  double fuY[K], fuZ[K], fwX[K], fwY[K];
  R P[TM ? 1 : 2][NPA][K], Pp[TM ? 1 : 2][NPA][K];
  __device__ Tile2d(const Step2dArgs<R> &args, const Step2dLaunch<R> &launch) : a(args), l(launch) {}

  __device__ __forceinline__ uint32_t index(int k) const { return uint32_t(x0 + k) * a.sx + uint32_t(y); }
  __device__ __forceinline__ S2Prof<R> profx(int ysh, int k) const {
    const int r = wave * K + k;
    S2Prof<R> p;
    p.sig = px[ysh][0][r];
    p.kap = px[ysh][1][r];
    p.sinv = px[ysh][2][r];
    p.on = p.sig != R(0) || p.kap != R(1);
    return p;
  }
  static constexpr int pslot(int C) { return TM ? 0 : C; }

  __device__ __forceinline__ bool in(int k) const { return ((rin >> k) & 1) && cin; }
  template <int C> __device__ __forceinline__ bool own(int k) const { return ((rown[C] >> k) & 1) && cown[C]; }
  template <int C> __device__ __forceinline__ bool wall(int k) const { return ((rzero[C] >> k) & 1) || czero[C]; }
  __device__ __forceinline__ bool pin(int p, int k) const { return ((rpin[p] >> k) & 1) && cpin[p]; }

  // D or B of slot C, row k, from its curl term.  FULL: the tile meets a uPML profile or the
  // chunk's edge.  The X profile is that of the row, so its branches are scalar; where the tile
  // meets the Y profile, its branch is evaluated in every lane and selected (lane branches per
  // point and component left two waves per SIMD waiting: 63 us for 8 steps of a 320 x 160 FP64
  // cell).
  template <bool MAG, int C, bool FULL> __device__ __forceinline__ void curl(int k, R cu) {
    const R f0 = f[C][k];
    R fv = f0 - dtdx * cu;
    if (FULL && C == 0) { // uPML of Y on f (dsig = Y, no f_u: its direction Z is absent)
      if (pmly) {
        // selected although an inactive profile (0, 1, 1) gives the plain update too: the two
        // contract to differently rounded fused multiply-adds
        const S2Prof<R> &s = py[s2_ysh<MAG, 0, 1>()];
        const R fp = ((s.kap - s.sig) * f0 - dtdx * cu) * s.sinv;
        fv = s.on ? fp : fv;
      }
    }
    if (FULL && C == 1) { // uPML of X through f_u
      if ((rowx[s2_ysh<MAG, 1, 0>()] >> k) & 1) {
        const S2Prof<R> u = profx(s2_ysh<MAG, 1, 0>(), k);
        const double fprev = fuY[k], d = dtdx, cud = cu;
        const double fun = fprev - d * cud;
        fuY[k] = own<1>(k) ? fun : fprev;
        fv = R(double(u.sinv) * ((double(u.kap) - double(u.sig)) * double(f0) + fun - fprev));
      }
    }
    if (FULL && C == 2) { // uPML of X on f, of Y through f_u
      const bool xon = (rowx[s2_ysh<MAG, 2, 0>()] >> k) & 1;
      S2Prof<R> s{R(0), R(1), R(1), false};
      if (xon) {
        s = profx(s2_ysh<MAG, 2, 0>(), k);
        fv = ((s.kap - s.sig) * f0 - dtdx * cu) * s.sinv;
      }
      if (pmly) {
        const S2Prof<R> &u = py[s2_ysh<MAG, 2, 1>()];
        const double fprev = fuZ[k], d = dtdx, cud = cu;
        double fun = fprev - d * cud;
        if (xon) fun = ((double(s.kap) - double(s.sig)) * fprev - d * cud) * double(s.sinv);
        const R fp = R(double(u.sinv) * ((double(u.kap) - double(u.sig)) * double(f0) + fun - fprev));
        fuZ[k] = u.on && own<2>(k) ? fun : fprev;
        fv = u.on ? fp : fv;
      }
    }
    f[C][k] = !FULL || own<C>(k) ? fv : f0;
  }

  // The sources a tile meets are found once: which entries of the three short lists (B currents,
  // D currents, D dipoles) fall on each of the thread's points, and the step values of the whole
  // launch, so that a step finds them without waiting for memory (the tile with the source was
  // the slowest of a launch by far: 59 us with its lists read every step).
  __device__ __forceinline__ void find_sources() {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      tmask[q] = 0;
#pragma unroll
      for (int c = 0; c < 3; ++c) tcomp[q][c] = 0;
    }
    if (!(srcs[0] || srcs[1])) return;
#pragma unroll
    for (int ph = 0; ph < 2; ++ph) {
      static_assert(sizeof(SrcSet) % 8 == 0 && sizeof(SrcSet) / 8 <= NW * 64, "one word per thread");
      if (srcs[ph] && threadIdx.x < sizeof(SrcSet) / 8)
        reinterpret_cast<uint64_t *>(set + ph)[threadIdx.x] = ((Glob<const uint64_t>)uni(a.src[ph]))[threadIdx.x];
    }
    const int rl = uni(a.rl);
    for (int q = int(threadIdx.x); q < l.nsteps * rl; q += NW * 64) vals[q] = l.vrow[a.vofs + int64_t(q / rl) * l.stride + q % rl];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const int ph = q ? 1 : 0;
      if (!srcs[ph]) continue;
      const SrcTab &t = q == 2 ? set[ph].dip : set[ph].cur;
      const int n = uni(min(t.n, SRC_TAB));
      int pos = -1, comp = 0;
      if (lane < n) {
        const uint32_t i = uint32_t(t.idx[lane]), x = i / a.sx;
        const int lx = int(x) - X0, ly = int(i - x * a.sx) - Y0;
        if (lx >= 0 && lx < RX && ly >= 0 && ly < S2_COLS) pos = lx * S2_COLS + ly;
        comp = t.comp[lane];
      }
      for (int j = 0; j < n; ++j) {
        const int p = __builtin_amdgcn_readlane(pos, j), c = __builtin_amdgcn_readlane(comp, j);
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (c == d) tcomp[q][d] |= 1u << j;
        const int d = (p >> 6) - wave * K;
        if (p >= 0 && (p & 63) == lane && d >= 0 && d < K) tmask[q] |= uint64_t(1) << (SRC_TAB * d + j);
      }
    }
  }
  // currents (L 0: B, 1: D) or integrated dipoles (L 2) of slot C at step s subtracted from v
  template <int C, int L> __device__ __forceinline__ void sources(R (&v)[K], int s) {
    static_assert(SRC_TAB * K <= 64, "a bit per list entry and row");
    const SrcTab &t = L == 2 ? set[1].dip : set[L ? 1 : 0].cur;
    const SrcBoxes &b = L == 2 ? set[1].dipb : set[L ? 1 : 0].curb;
    const double *val = vals + s * a.rl;
    if (tmask[L]) {
      const int vb = t.vbase;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        unsigned m = unsigned(tmask[L] >> (SRC_TAB * k)) & tcomp[L][C];
        while (m) {
          v[k] = R(double(v[k]) - val[vb + __builtin_ctz(m)]);
          m &= m - 1;
        }
      }
    }
    const int nb = uni(b.n);
#pragma unroll 1
    for (int q = 0; q < nb; ++q) {
      if (uni(b.comp[q]) != C) continue;
      // the thread's amplitudes, loaded together (from the box's edge where a row is outside)
      const int lx = b.lo[q][1], hx = b.hi[q][1], ly = b.lo[q][2], hy = b.hi[q][2];
      const Glob<const double> am = (Glob<const double>)uni(b.amp[q]);
      const int64_t sx = b.bst[q][1], col = int64_t(min(max(y, ly), hy) - ly) * b.bst[q][2];
      double re[K], im[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int64_t j = int64_t(min(max(x0 + k, lx), hx) - lx) * sx + col;
        re[k] = am[2 * j];
        im[k] = am[2 * j + 1];
      }
      const double vx = val[b.vbase + 2 * q], vy = val[b.vbase + 2 * q + 1], mult = b.mult[q];
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (y >= ly && y <= hy && x0 + k >= lx && x0 + k <= hx) v[k] = R(double(v[k]) - boxed(re[k], im[k], vx, vy, mult));
    }
  }
  // a box source's value, rounded as the host forms it (box_value in stencil.hpp)
  __device__ __forceinline__ double boxed(double ax, double ay, double vx, double vy, double mult) const {
#pragma clang fp contract(off)
    const double re = ax * vx - ay * vy, im = ax * vy + ay * vx;
    return a.cmp ? im * mult : re * mult;
  }

  // the sources and walls of slot C's D or B, then its E or H and the poles
  template <bool MAG, int C, bool FULL> __device__ __forceinline__ void finish(int s) {
    constexpr int PH = MAG ? 0 : 1;
    if (srcs[PH]) sources<C, PH>(f[C], s);
    R gv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (FULL) f[C][k] = wall<C>(k) ? R(0) : f[C][k];
      gv[k] = f[C][k];
      if (!MAG && NP > 0) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
          if (((rpin[p] >> k) & 1)) gv[k] = cpin[p] ? gv[k] - P[pslot(C)][p][k] : gv[k];
      }
    }
    if (!MAG && srcs[PH]) sources<C, 2>(gv, s);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      R ev = gv[k];
      if (!MAG)
        ev = gv[k] * chi[C][k];
      else if (mu[C])
        ev = gv[k] * (in(k) ? global(a.c[C].chi)[index(k)] : R(1));
      const R wv = ev;
      const bool mine = !FULL || own<C>(k);
      if (FULL && C == 0) { // f_w: along the component's own axis
        if ((rowx[s2_ysh<MAG, 0, 0>()] >> k) & 1) {
          const S2Prof<R> w = profx(s2_ysh<MAG, 0, 0>(), k);
          const double fwprev = fwX[k], fwn = ev, kw = w.kap, sw = w.sig;
          ev = R(double(e[C][k]) + ((kw + sw) * fwn - (kw - sw) * fwprev));
          fwX[k] = mine ? fwn : fwprev;
        }
      }
      if (FULL && C == 1) {
        if (pmly) {
          const S2Prof<R> &w = py[s2_ysh<MAG, 1, 1>()];
          const double fwprev = fwY[k], fwn = ev, kw = w.kap, sw = w.sig;
          const R ew = R(double(e[C][k]) + ((kw + sw) * fwn - (kw - sw) * fwprev));
          fwY[k] = w.on && mine ? fwn : fwprev;
          ev = w.on ? ew : ev;
        }
      }
      if (!MAG && NP > 0) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
          if (((rpin[p] >> k) & 1) && polar[p][C]) {
            const PoleCoef<R> &q = a.pole[p];
            const bool lp = cpin[p] && mine;
            const R sg = ((a.c[C].sigone >> p) & 1) ? a.c[C].sigval[p] : (lp ? R(global(a.c[C].sigma[p])[index(k)]) : R(0));
            const R pc = P[pslot(C)][p][k], po = Pp[pslot(C)][p][k];
            const R pn = q.gamma1inv * (pc * (R(2) - q.omega0dtsqr_denom) - q.gamma1 * po + q.omega0dtsqr * (sg * wv));
            P[pslot(C)][p][k] = lp ? pn : pc;
            Pp[pslot(C)][p][k] = lp ? pc : po;
          }
      }
      if (FULL) ev = wall<C>(k) ? R(0) : ev;
      e[C][k] = mine ? ev : e[C][k];
    }
  }

  // the phase whose X and Y components take the Z partner's differences (forward for B)
  template <bool MAG, bool FULL> __device__ __forceinline__ void pair_phase(int s) {
    const R beyond = MAG ? bE[(wave + 1) * S2_COLS + lane] : bH[wave * S2_COLS + lane];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const R c = e[2][k];
      const R cx = MAG ? (k + 1 < K ? e[2][k + 1 < K ? k + 1 : 0] : beyond) : (k > 0 ? e[2][k > 0 ? k - 1 : 0] : beyond);
      const R cy = MAG ? lane_next(c) : lane_prev(c);
      curl<MAG, 0, FULL>(k, cy - c);
      curl<MAG, 1, FULL>(k, c - cx);
    }
    finish<MAG, 0, FULL>(s);
    finish<MAG, 1, FULL>(s);
  }
  // the phase whose Z component takes the X and Y partners' differences
  template <bool MAG, bool FULL> __device__ __forceinline__ void single_phase(int s) {
    const R beyond = MAG ? bE[(wave + 1) * S2_COLS + lane] : bH[wave * S2_COLS + lane];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const R gy = e[1][k], gx = e[0][k];
      const R gyn = MAG ? (k + 1 < K ? e[1][k + 1 < K ? k + 1 : 0] : beyond) : (k > 0 ? e[1][k > 0 ? k - 1 : 0] : beyond);
      const R gxn = MAG ? lane_next(gx) : lane_prev(gx);
      curl<MAG, 2, FULL>(k, gyn - gy + gx - gxn);
    }
    finish<MAG, 2, FULL>(s);
  }

  // Monitors: the tile's points and the chunks' facts are brought to LDS once per launch.
  struct Mons {
    R *field;                // the fields read, whole
    S2Entry *entry;          // the first S2_ENTRIES points
    int *slot;               // per chunk: this step's slot of its ring, or -1
    int *off;                // per chunk: its field's place in `field`, and the two centring offsets
    uint32_t first, last;    // the tile's points
    int nchunk;
  };
  __device__ __forceinline__ void load_mons(Mons &m) const {
    const int n = int(min(m.last - m.first, uint32_t(S2_ENTRIES)));
    const Glob<const uint64_t> src = (Glob<const uint64_t>)(uni(a.mon) + m.first);
    for (int q = int(threadIdx.x); q < 2 * n; q += NW * 64) reinterpret_cast<uint64_t *>(m.entry)[q] = src[q];
    if (int(threadIdx.x) < m.nchunk) {
      const Glob<const S2Mon<R>> c = global(a.mons) + threadIdx.x;
      m.off[3 * threadIdx.x] = __popc(a.monmask & ((1 << c->fld) - 1)) * RX * S2_COLS;
      m.off[3 * threadIdx.x + 1] = c->o1;
      m.off[3 * threadIdx.x + 2] = c->o2;
    }
  }
  // the tile's points at step tt: the fields go to LDS whole, then each point's average to the
  // centred grid as avg_value forms it (the next step's first barrier follows every read)
  __device__ __forceinline__ void monitor(const Mons &m, int tt) {
    const int mask = uni(a.monmask);
    int slot = 0;
#pragma unroll
    for (int q = 0; q < 6; ++q)
      if ((mask >> q) & 1) {
#pragma unroll
        for (int k = 0; k < K; ++k)
          m.field[(slot * RX + wave * K + k) * S2_COLS + lane] = q < 3 ? R(e[q < 3 ? q : 0][k]) : R(f[q < 3 ? 0 : q - 3][k]);
        ++slot;
      }
    if (int(threadIdx.x) < m.nchunk) { // step counts fit 32 bits (checked on the host)
      const int dec = (global(a.mons) + threadIdx.x)->dec, tq = tt / dec;
      m.slot[threadIdx.x] = tq * dec == tt ? tq - int(a.t0 + l.w) / dec - 1 : -1;
    }
    __syncthreads();
    const int n = int(m.last - m.first);
    for (int q = int(threadIdx.x); q < n; q += NW * 64) {
      double w;
      uint32_t kk;
      int pos, ch;
      if (q < S2_ENTRIES) {
        const S2Entry &en = m.entry[q];
        w = en.w, kk = en.k, pos = en.pos, ch = en.chunk;
      }
      else {
        const Glob<const S2Entry> en = global(a.mon) + (m.first + q);
        w = en->w, kk = en->k, pos = en->pos, ch = en->chunk;
      }
      const int sl = m.slot[ch];
      if (sl < 0) continue;
      const int o1 = m.off[3 * ch + 1], o2 = m.off[3 * ch + 2];
      const R *F = m.field + (m.off[3 * ch] + pos);
      R v;
      if (o2)
        v = R((w * 0.25) * double(F[0] + F[o1] + F[o2] + F[o1 + o2]));
      else if (o1)
        v = R((w * 0.5) * double(F[0] + F[o1]));
      else
        v = R(w * double(F[0]));
      const Glob<const S2Mon<R>> c = global(a.mons) + ch;
      global(c->snap)[size_t(sl) * c->npts + kk] = v;
    }
  }
  // one of two register values; kept from becoming a choice between their addresses, which would
  // put the whole tile into scratch memory
  static __device__ __forceinline__ R pick(bool second, R u, R v) {
    asm volatile("" : "+v"(u));
    asm volatile("" : "+v"(v));
    return second ? v : u;
  }
  // the step's D on the reverse mode's design box
  __device__ __forceinline__ void record(int s) {
    const int n2 = l.rec_hi[1] - l.rec_lo[1] + 1, cl = a.margin;
    R *dst = l.rec + size_t(s) * size_t(l.rec_hi[0] - l.rec_lo[0] + 1) * size_t(n2);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int x = x0 + k, lx = wave * K + k;
      if (lx >= cl && lx < cl + a.cx && lane >= cl && lane < cl + a.cy && x >= l.rec_lo[0] && x <= l.rec_hi[0] && y >= l.rec_lo[1] &&
          y <= l.rec_hi[1])
        dst[size_t(x - l.rec_lo[0]) * n2 + (y - l.rec_lo[1])] = TM ? f[2][k] : pick(l.rec_c == 1, f[0][k], f[1][k]);
    }
  }

  // the launch's steps on the tile in registers
  template <bool FULL> __device__ __forceinline__ void steps(const Mons &mons) {
    constexpr int EC = TM ? 2 : 1, HC = TM ? 1 : 2; // the partners whose row neighbour crosses waves
    for (int s = 0; s < l.nsteps; ++s) {
      if constexpr (TM)
        pair_phase<true, FULL>(s);
      else
        single_phase<true, FULL>(s);
      bH[(wave + 1) * S2_COLS + lane] = e[HC][K - 1];
      __syncthreads();
      if constexpr (TM)
        single_phase<false, FULL>(s);
      else
        pair_phase<false, FULL>(s);
      bE[wave * S2_COLS + lane] = e[EC][0];
      if (mons.first < mons.last) monitor(mons, int(a.t0 + l.s) + s + 1);
      if (l.rec) record(s);
      __syncthreads();
    }
  }

  __device__ __forceinline__ void run(uint32_t tile, unsigned char *dyn) {
    const int tx = uni(int(tile / uint32_t(a.nty))), ty = uni(int(tile) - tx * a.nty);
    X0 = uni(tx * a.cx - a.margin);
    Y0 = uni(ty * a.cy - a.margin);
    x0 = X0 + wave * K;
    y = Y0 + lane;
    dtdx = a.dtdx;
    const bool pmlx = uni(a.sig[0] && (X0 < a.qlo[0] || X0 + RX - 1 > a.qhi[0]));
    pmly = uni(a.sig[1] && (Y0 < a.qlo[1] || Y0 + S2_COLS - 1 > a.qhi[1]));
    const bool edge = uni(X0 < 1 || X0 + RX - 1 > a.nx - 1 || Y0 < 1 || Y0 + S2_COLS - 1 > a.ny - 1);
    cin = y >= 0 && y <= a.ny;
    rin = 0;
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (x0 + k >= 0 && x0 + k <= a.nx) rin |= 1u << k;
    rin = unsigned(uni(int(rin)));
    // ---- load ----
    // Every load is unconditional, from the nearest point of the grid where the tile reaches past
    // it (no update reads such a point: an owned point's neighbours are all in the grid), so that
    // a thread's loads are in flight together; one predicated load after another cost 12 us a
    // launch.
    uint32_t at[K];
#pragma unroll
    for (int k = 0; k < K; ++k) at[k] = uint32_t(min(max(x0 + k, 0), a.nx)) * a.sx + uint32_t(min(max(y, 0), a.ny));
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const S2Comp<R> &q = a.c[c];
      const bool electric = TM ? c == 2 : c != 2;
      mu[c] = uni(!electric && q.chi);
      const Glob<const R> fp = uni(q.f), ep = uni(q.e ? q.e : q.f);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        f[c][k] = fp[at[k]];
        e[c][k] = ep[at[k]];
        chi[c][k] = R(1);
      }
      if (electric && uni(q.chi != nullptr)) {
        const Glob<const R> up = uni(q.chi);
#pragma unroll
        for (int k = 0; k < K; ++k) chi[c][k] = up[at[k]];
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) fuY[k] = fuZ[k] = fwX[k] = fwY[k] = 0.0;
    if (pmlx) {
      const Glob<const double> u = uni(a.c[1].fu), w = uni(a.c[0].fw);
#pragma unroll
      for (int k = 0; k < K; ++k) fuY[k] = u[at[k]], fwX[k] = w[at[k]];
    }
    if (pmly) {
      const Glob<const double> u = uni(a.c[2].fu), w = uni(a.c[1].fw);
#pragma unroll
      for (int k = 0; k < K; ++k) fuZ[k] = u[at[k]], fwY[k] = w[at[k]];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      py[q] = S2Prof<R>{R(0), R(1), R(1), false};
      if (pmly) py[q] = s2_prof(global(a.sig[1]), global(a.kap[1]), global(a.siginv[1]), y, q, a.ny);
    }
    if (pmlx || pmly || edge)
      for (int q = int(threadIdx.x); q < 2 * RX; q += NW * 64) {
        const int ysh = q / RX, r = q - ysh * RX;
        S2Prof<R> p{R(0), R(1), R(1), false};
        if (pmlx) p = s2_prof(global(a.sig[0]), global(a.kap[0]), global(a.siginv[0]), X0 + r, ysh, a.nx);
        px[ysh][0][r] = p.sig;
        px[ysh][1][r] = p.kap;
        px[ysh][2][r] = p.sinv;
      }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const S2Comp<R> &q = a.c[c];
      unsigned o = 0, z = 0;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int x = x0 + k;
        if (x >= q.lo[0] && x <= q.hi[0]) o |= 1u << k;
        if (x == q.mhi[0] || x == q.mlo[0]) z |= 1u << k;
      }
      rown[c] = unsigned(uni(int(o)));
      rzero[c] = unsigned(uni(int(z)));
      cown[c] = y >= q.lo[1] && y <= q.hi[1];
      czero[c] = y == q.mhi[1] || y == q.mlo[1];
    }
    rowx[0] = rowx[1] = 0;
    if (pmlx) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        unsigned o = 0;
#pragma unroll
        for (int k = 0; k < K; ++k)
          if (s2_prof(uni(a.sig[0]), uni(a.kap[0]), uni(a.siginv[0]), x0 + k, q, a.nx).on) o |= 1u << k;
        rowx[q] = unsigned(uni(int(o)));
      }
    }
#pragma unroll
    for (int ph = 0; ph < 2; ++ph)
      srcs[ph] = uni(a.src[ph] && X0 <= a.sbox_hi[ph][0] && X0 + RX - 1 >= a.sbox_lo[ph][0] && Y0 <= a.sbox_hi[ph][1] &&
                 Y0 + S2_COLS - 1 >= a.sbox_lo[ph][1]);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const PoleCoef<R> &q = a.pole[p]; // loop axes 1 and 2 are X and Y
      unsigned o = 0;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (p < a.npole && x0 + k >= q.lo[1] && x0 + k <= q.hi[1] && Y0 <= q.hi[2] && Y0 + S2_COLS - 1 >= q.lo[2]) o |= 1u << k;
      rpin[p] = unsigned(uni(int(o))) & rin;
      cpin[p] = cin && y >= q.lo[2] && y <= q.hi[2];
#pragma unroll
      for (int c = 0; c < 3; ++c) polar[p][c] = uni(a.c[c].P[p] && a.c[c].sigma[p]);
#pragma unroll
      for (int q2 = 0; q2 < (TM ? 1 : 2); ++q2) {
        const S2Comp<R> &c = a.c[TM ? 2 : q2];
#pragma unroll
        for (int k = 0; k < K; ++k) P[q2][p][k] = Pp[q2][p][k] = R(0);
        if (uni(p < a.npole && c.P[p] && X0 <= q.hi[1] && X0 + RX - 1 >= q.lo[1] && Y0 <= q.hi[2] && Y0 + S2_COLS - 1 >= q.lo[2])) {
          const Glob<const R> pp = uni(c.P[p]), qp = uni(c.Pp[p]);
#pragma unroll
          for (int k = 0; k < K; ++k) P[q2][p][k] = pp[at[k]], Pp[q2][p][k] = qp[at[k]];
        }
      }
    }
    find_sources();
    Mons mons;
    mons.first = mons.last = 0;
    mons.nchunk = 0;
    if (l.hits && uni(a.mon_first != nullptr)) {
      mons.first = uint32_t(uni(int(uni(a.mon_first)[tile])));
      mons.last = uint32_t(uni(int(uni(a.mon_first)[tile + 1])));
      mons.nchunk = uni(a.nmon);
    }
    mons.entry = reinterpret_cast<S2Entry *>(dyn);
    mons.slot = reinterpret_cast<int *>(dyn + S2_ENTRIES * sizeof(S2Entry));
    mons.off = mons.slot + S2_MONS;
    mons.field = reinterpret_cast<R *>(dyn + S2_ENTRIES * sizeof(S2Entry) + 4 * S2_MONS * sizeof(int));
    if (mons.first < mons.last) load_mons(mons);
    if (threadIdx.x < S2_COLS) bE[NW * S2_COLS + lane] = bH[lane] = R(0);
    bE[wave * S2_COLS + lane] = e[TM ? 2 : 1][0];
    __syncthreads();
    if (pmlx || pmly || edge)
      steps<true>(mons);
    else
      steps<false>(mons);
    // ---- store the core ----
    const int cl = a.margin;
    Glob<R> fo[3], eo[3];
    bool own_e[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      fo[c] = uni(a.c[c].fo);
      eo[c] = uni(a.c[c].eo);
      own_e[c] = uni(a.c[c].e != nullptr);
    }
    const bool coly = cin && lane >= cl && lane < cl + a.cy;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int lx = wave * K + k;
      if (!(coly && ((rin >> k) & 1) && lx >= cl && lx < cl + a.cx)) continue;
      const uint32_t i = index(k);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        fo[c][i] = f[c][k];
        if (own_e[c]) eo[c][i] = e[c][k];
      }
      if (pmlx) uni(a.c[1].fuo)[i] = fuY[k], uni(a.c[0].fwo)[i] = fwX[k];
      if (pmly) uni(a.c[2].fuo)[i] = fuZ[k], uni(a.c[1].fwo)[i] = fwY[k];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int q = 0; q < (TM ? 1 : 2); ++q) {
          const S2Comp<R> &c = a.c[TM ? 2 : q];
          if (pin(p, k) && uni(c.P[p] != nullptr)) {
            global(c.Po[p])[i] = P[q][p][k];
            global(c.Ppo[p])[i] = Pp[q][p][k];
          }
        }
    }
  }
};

template <class R, bool TM, int NP, int NW, int K>
__global__ __launch_bounds__(NW * 64) void k_step2d(const Step2dLaunch<R> l) {
  constexpr int RX = NW * K;
  static_assert(RX == S2_ROWS, "the host plans tiles of S2_ROWS rows");
  __shared__ R bE[(NW + 1) * S2_COLS], bH[(NW + 1) * S2_COLS], px[2][3][RX];
  __shared__ double vals[S2_STEPS * S2_VALS];
  extern __shared__ __align__(16) unsigned char dyn[];
  const uint32_t lb = xcd_block();
  if (lb >= l.ntile) return;
  // The arguments come to LDS in one go: read from memory field by field, each first touch of a
  // cache line behind a branch was a wait of its own (8.5 us before a tile's first step).
  __shared__ Step2dArgs<R> args;
  __shared__ SrcSet set[2];
  {
    static_assert(sizeof(Step2dArgs<R>) % 8 == 0 && sizeof(Step2dArgs<R>) / 8 <= NW * 64, "one word per thread");
    const uint64_t *w = reinterpret_cast<const uint64_t *>(l.items + (l.blk_item ? l.blk_item[lb] : 0));
    if (threadIdx.x < sizeof(Step2dArgs<R>) / 8) reinterpret_cast<uint64_t *>(&args)[threadIdx.x] = w[threadIdx.x];
    __syncthreads();
  }
  const Step2dArgs<R> &a = args;
  Tile2d<R, TM, NP, NW, K> T(a, l);
  T.bE = bE;
  T.bH = bH;
  T.px = px;
  T.vals = vals;
  T.set = set;
  T.lane = int(threadIdx.x) & 63;
  T.wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  T.run(l.blk_tile ? l.blk_tile[lb] : lb, dyn);
}

template <class R, bool TM, int NP> static void launch_s2(const Step2dLaunch<R> &l, int monmask, hipStream_t s) {
  // two rows a thread: four waves on a SIMD hide each other's waits (against four rows and two
  // waves: 32 / 19 us for up to 8 steps of a 400 x 300 FP32 cell, and less in FP64, where some
  // registers then spill)
  constexpr int NW = 16, K = S2_ROWS / NW;
  const unsigned nb = (l.ntile + 7u) / 8u * 8u;
  const size_t lds = l.hits ? S2_ENTRIES * sizeof(S2Entry) + 4 * S2_MONS * sizeof(int) +
                                  size_t(__builtin_popcount(unsigned(monmask))) * S2_ROWS * S2_COLS * sizeof(R)
                            : 0;
  hipLaunchKernelGGL((k_step2d<R, TM, NP, NW, K>), dim3(nb), dim3(NW * 64), lds, s, l);
}
template <class R> void launch_step2d(const Step2dLaunch<R> &l, bool tm, int npole, int monmask, hipStream_t s) {
  if (!l.ntile) return;
  if (tm)
    switch (npole) {
      case 0: launch_s2<R, true, 0>(l, monmask, s); break;
      case 1: launch_s2<R, true, 1>(l, monmask, s); break;
      default: launch_s2<R, true, 2>(l, monmask, s); break;
    }
  else
    switch (npole) {
      case 0: launch_s2<R, false, 0>(l, monmask, s); break;
      case 1: launch_s2<R, false, 1>(l, monmask, s); break;
      default: launch_s2<R, false, 2>(l, monmask, s); break;
    }
}

#define INSTANTIATE_S2(R) template void launch_step2d<R>(const Step2dLaunch<R> &, bool, int, int, hipStream_t);
#ifdef MX_REAL
INSTANTIATE_S2(MX_REAL)
#else
INSTANTIATE_S2(float)
INSTANTIATE_S2(double)
#endif

} // namespace mx
