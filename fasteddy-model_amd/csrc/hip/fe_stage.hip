/*
 * fe_stage.hip -- fused RK3 stage kernels of the FastEddy compressible LES for gfx950.
 *
 * One launch evaluates the complete tendency of every prognostic field at
 * every cell and applies the RK3-WS2002 stage update (or, in emit mode, stores
 * the tendency).  A 64x8 work-group owns a tile of columns and marches up the
 * column:
 *   - each thread keeps its own column's 7-deep window (z-3..z+3) of every
 *     field in registers (vertical stencils, z face fluxes computed once and
 *     carried to the next level);
 *   - the tile's xy plane at level z, with a 3-cell halo loaded with periodic
 *     wrap-around, is staged in LDS for the horizontal stencils;
 *   - x and y face quantities (advective fluxes, SGS stresses) are computed
 *     once per face into LDS and differenced by the two cells that share them.
 * Reference path replaced: SRC/HYDRO_CORE/CUDA/cuda_hydroCoreDevice.cu:246-947
 * (tendency build, one launch per phase there) and
 * SRC/TIME_INTEGRATION/CUDA/cuda_RKschemes.cu:21-157 (stage update).
 *
 * Arithmetic is FP32 throughout.  The perturbation pressure uses the
 * well-conditioned form p' = p_BS((1+r)^gamma - 1), r = rho*theta/(rho*theta)_BS - 1
 * (a binomial series for |r| < 1/8) instead of the difference of two ~1e5 Pa
 * powers; amd_pressureForm = 0 selects the reference's difference form.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>
#include "fe_kernels.h"

namespace fe {

/* Work-group tile: TX x TY columns, one thread per column, thread t at (t % TX, t / TX); a
 * 64-lane wave covers 64 / TX whole rows.  The build uses 64 x 8 (eight waves, one work-group
 * per compute unit).  16 x 16 (-DFE_TILE_X=16 -DFE_TILE_Y=16: four waves and about half the
 * LDS, two work-groups per compute unit) computes the same tendencies but measured slower on
 * the 512 x 512 x 128 dry step (plain stage 0.97 vs 0.66 ms, physics 1.32 vs 1.14 ms): a ring
 * row costs a whole wave's issue whatever its length, so the ring work per cell doubles, and
 * two rows of a half-wave fall on the same LDS banks at a 22-float row pitch.  32 x 16 (eight
 * waves, a third less halo and ring work per cell) measured 0.73 / 1.18 ms on that step, but
 * 5% faster on the 48-member ensemble, whose 96- and 160-wide members it tiles without
 * padding. */
#ifndef FE_TILE_X
#define FE_TILE_X 64
#endif
#ifndef FE_TILE_Y
#define FE_TILE_Y 8
#endif
constexpr int TX = FE_TILE_X, TY = FE_TILE_Y, NT = TX * TY, HH = 3, NW = NT / 64;
constexpr int RW = TX + 2 * HH, RH = TY + 2 * HH;      /* raw plane with 3-cell halo          */
constexpr int DW = TX + 2, DH = TY + 2;                /* ring-1 region [-1,TX] x [-1,TY]     */
constexpr int NHALO = RW * RH - TX * TY;               /* halo cells of the raw plane (<= NT) */
constexpr int NR1 = DW * DH - TX * TY;                 /* ring-1 cells, listed first          */
constexpr int NFP = 8;                                 /* fields per row of the ring column's fluxes (16-byte rows) */
/* third word of a raw (stride 0) buffer resource on CDNA: 32-bit data format, no swizzle */
constexpr int FE_RSRC_W3 = 0x00020000;
static_assert(NHALO <= NT, "one halo cell per thread");
static_assert(64 % TX == 0 && NT % 64 == 0, "waves cover whole rows of the tile");

/* A row of the tile's extra work per level (ring faces, ring stresses, ring TKE fluxes):
 * lanes [l0, l0 + n) of wave w, item i = lane - l0.  Where these rows and the ring-1 cells
 * land decides how evenly a level's extra work spreads over the SIMDs (on the 64 x 8 tile
 * waves w and w + 4 share SIMD w); the placements were chosen by measurement. */
struct Job { int w, l0, n; };
__device__ __forceinline__ bool on_job(Job j, int wave, int lane, int &i) {
  i = lane - j.l0;
  return wave == j.w && (unsigned)i < (unsigned)j.n;
}
/* Ring-1 cells (whose derived planes the owning threads build): thread ranges [a, a+na),
 * [b, b+nb), [c, c+nc), all below NHALO; the other halo cells go to the remaining threads. */
struct R1Layout { int a, na, b, nb, c, nc; };
struct RingPlan {
  R1Layout r1;
  bool split;          /* advective ring faces: half of the fields per job row (rfy[1], rfx[1]) */
  Job rfy[2], rfx[2];  /* advective ring faces: the y row y = TY, the x column x = TX */
  Job sty, stx;        /* SGS stresses on the ring faces (physics stage) */
  Job qy0, qxs, qy1;   /* TKE transport fluxes of the ring cells y = -1, x = -1 and TX, y = TY */
};
#if FE_TILE_X == 64 && FE_TILE_Y == 8
constexpr RingPlan PLAN_PLAIN = {{128, 64, 192, 64, 384, 20}, false, {{0, 0, TX}, {}}, {{1, 0, TY}, {}},
                                 {}, {}, {}, {}, {}};
constexpr RingPlan PLAN_PHYS = {{128, 64, 192, 64, 384, 20}, true, {{0, 0, TX}, {1, 0, TX}}, {{4, 0, TY}, {5, 0, TY}},
                                {7, 0, TX}, {2, 0, TY}, {3, 0, TX}, {3, 0, 2 * TY}, {6, 0, TX}};
#elif FE_TILE_X == 32 && FE_TILE_Y == 16
constexpr RingPlan PLAN_PLAIN = {{128, 64, 192, 36, 0, 0}, false, {{0, 0, TX}, {}}, {{1, 0, TY}, {}},
                                 {}, {}, {}, {}, {}};
constexpr RingPlan PLAN_PHYS = {{128, 64, 192, 36, 0, 0}, true, {{0, 0, TX}, {1, 0, TX}}, {{4, 0, TY}, {5, 0, TY}},
                                {7, 0, TX}, {2, 0, TY}, {3, 0, TX}, {3, 0, 2 * TY}, {6, 0, TX}};
#elif FE_TILE_X == 16 && FE_TILE_Y == 16
constexpr RingPlan PLAN_PLAIN = {{128, 64, 192, 4, 0, 0}, false, {{0, 0, TX}, {}}, {{1, 0, TY}, {}},
                                 {}, {}, {}, {}, {}};
constexpr RingPlan PLAN_PHYS = {{128, 64, 192, 4, 0, 0}, false, {{0, 0, TX}, {}}, {{1, 0, TY}, {}},
                                {2, 0, TX}, {2, 16, TY}, {3, 0, TX}, {3, 16, 2 * TY}, {3, 48, TX}};
#else
#error "tile geometry without a ring plan"
#endif
static_assert(PLAN_PLAIN.r1.na + PLAN_PLAIN.r1.nb + PLAN_PLAIN.r1.nc == NR1, "every ring-1 cell has a thread");
static_assert(PLAN_PHYS.sty.w != PLAN_PHYS.stx.w || PLAN_PHYS.sty.l0 + PLAN_PHYS.sty.n <= PLAN_PHYS.stx.l0 ||
                  PLAN_PHYS.stx.l0 + PLAN_PHYS.stx.n <= PLAN_PHYS.sty.l0,
              "a lane holds at most one ring stress face");
static_assert(PLAN_PHYS.r1.na + PLAN_PHYS.r1.nb + PLAN_PHYS.r1.nc == NR1, "every ring-1 cell has a thread");
static_assert(PLAN_PLAIN.r1.c + PLAN_PLAIN.r1.nc <= NHALO && PLAN_PHYS.r1.c + PLAN_PHYS.r1.nc <= NHALO &&
              PLAN_PLAIN.r1.b + PLAN_PLAIN.r1.nb <= NHALO && PLAN_PHYS.r1.b + PLAN_PHYS.r1.nb <= NHALO,
              "ring-1 threads hold halo cells");

__device__ __forceinline__ int wrapi(int v, int n) {
  v %= n;
  return v < 0 ? v + n : v;
}

/* Column (row) of the lateral position v, -3 <= v < N + 3, of a tile's neighbourhood.  A
 * periodic grid wraps v into [0, N).  With lateral halo storage the grid is one block of a
 * larger domain: its planes are padded to P >= Nx + 6 columns and NyS = Ny + 6 rows, the three
 * positions past each edge are stored after the block (v >= N) and in the last three columns
 * (rows) of the plane (v < 0), and a separate step fills them (from the neighbouring blocks, or
 * from the block's own periodic images on one device). */
__device__ __forceinline__ int colx(const StepArgs &a, int v) { return a.halo ? (v < 0 ? v + a.P : v) : wrapi(v, a.Nx); }
__device__ __forceinline__ int rowy(const StepArgs &a, int v) { return a.halo ? (v < 0 ? v + a.NyS : v) : wrapi(v, a.Ny); }

/* hardware reciprocal (1 ulp): rho^-1 and the WENO weights */
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

/* Profiles are read-only for the whole step and indexed by wave-uniform (p, z):
 * reading them through the constant address space makes them scalar loads,
 * which wait on their own counter instead of behind the prefetched vector loads. */
typedef const __attribute__((address_space(4))) float cfloat;
__device__ __forceinline__ float prof(const StepArgs &a, int p, int z) { return ((cfloat *)a.prof)[(z + 3) * PROW + p]; }
/* Row p at level z of the column at plane offset col (y P + x, wrapped): on a terrain-following
 * grid the metrics and the base state vary from column to column and come from the per-column
 * table [PROW][np][Ny][P]; the flat kernels read the shared level table (col unused). */
template <class C>
__device__ __forceinline__ float cprof(const StepArgs &a, int p, int z, unsigned col) {
  if constexpr (C::TERR) return a.tprof[((size_t)p * (size_t)a.np + (size_t)(z + 3)) * (size_t)a.ps + col];
  else return prof(a, p, z);
}

/* ---- advective face fluxes: u * f(face) from phi[i-3..i+2] (cuda_advectionDevice.cu:123-926) ---- */
__device__ __forceinline__ float weno5_side(float a, float b, float c, float d, float e) {
  const float tol = 1e-6f;
  float fh1 = (1.f / 3.f) * a - (7.f / 6.f) * b + (11.f / 6.f) * c;
  float fh2 = -(1.f / 6.f) * b + (5.f / 6.f) * c + (1.f / 3.f) * d;
  float fh3 = (1.f / 3.f) * c + (5.f / 6.f) * d - (1.f / 6.f) * e;
  float t1 = a - 2.f * b + c, t2 = a - 4.f * b + 3.f * c;
  float t3 = b - 2.f * c + d, t4 = b - d;
  float t5 = c - 2.f * d + e, t6 = 3.f * c - 4.f * d + e;
  float b1 = (13.f / 12.f) * t1 * t1 + 0.25f * t2 * t2;
  float b2 = (13.f / 12.f) * t3 * t3 + 0.25f * t4 * t4;
  float b3 = (13.f / 12.f) * t5 * t5 + 0.25f * t6 * t6;
  /* weights with the hardware reciprocal instead of IEEE divisions (smoothness weights: their
   * last bit does not matter; 0.1/inf = 0 and 1/0 = inf behave as the divisions do) */
  float w1 = 0.1f * frcp((tol + b1) * (tol + b1));
  float w2 = 0.6f * frcp((tol + b2) * (tol + b2));
  float w3 = 0.3f * frcp((tol + b3) * (tol + b3));
  float inv = frcp(w1 + w2 + w3);
  return (w1 * fh1 + w2 * fh2 + w3 * fh3) * inv;
}
__device__ __forceinline__ float weno3_side(float a, float b, float c) {
  const float tol = 1e-6f;
  float fh1 = -0.5f * a + 1.5f * b, fh2 = 0.5f * b + 0.5f * c;
  float b1 = (b - a) * (b - a), b2 = (c - b) * (c - b);
  float w1 = (1.f / 3.f) * frcp((tol + b1) * (tol + b1)), w2 = (2.f / 3.f) * frcp((tol + b2) * (tol + b2));
  return (w1 * fh1 + w2 * fh2) * frcp(w1 + w2);
}

template <int S, bool SEL = false>
__device__ __forceinline__ float face_flux(float U, float omb, float m3, float m2, float m1, float c0, float p1, float p2) {
  if constexpr (S == 3) {        /* hybrid 5th/6th: b=0 is 5th-order upwind (WS2002) */
    /* 37(c0+m1) - 8(p1+m2) + (p2+m3) - s[10(c0-m1) - 5(p1-m2) + (p2-m3)], s = (1-b) sgn(U),
     * as one 6-point stencil whose weights depend only on s: they are shared by every
     * field advected through the face, leaving one multiply and five FMAs per field */
    const float sg = copysignf(omb, U);
    const float w0 = fmaf(-10.f, sg, 37.f), w1 = fmaf(10.f, sg, 37.f);
    const float w2 = fmaf(5.f, sg, -8.f), w3 = fmaf(-5.f, sg, -8.f);
    const float w4 = 1.f - sg, w5 = 1.f + sg;
    float t = w0 * c0;
    t = fmaf(w1, m1, t);
    t = fmaf(w2, p1, t);
    t = fmaf(w3, m2, t);
    t = fmaf(w4, p2, t);
    t = fmaf(w5, m3, t);
    return (U * (1.f / 60.f)) * t;
  } else if constexpr (S == 2) { /* hybrid 3rd/4th */
    float cen = fmaf(7.f, c0 + m1, -(p1 + m2));
    float upw = fmaf(-3.f, c0 - m1, p1 - m2);
    float sg = copysignf(omb, U);
    return U * ((cen + sg * upw) * (1.f / 12.f));
  } else if constexpr (S == 1) { /* QUICK */
    return 0.125f * (fmaxf(0.f, U) * (6.f * m1 + 3.f * c0 - m2) + fminf(0.f, U) * (6.f * c0 + 3.f * m1 - p1));
  } else if constexpr (S == 4) { /* WENO3 */
    /* The upwind side is evaluated once per lane either way (the compiler merges the two
     * identical side evaluations of the ternary into one on selected inputs).  SEL writes the
     * selection out, which gives the physics stage a better register allocation (moist
     * 256x256x160: 0.555 -> 0.532 ms) and the plain stage a worse one (a spill: 0.347 ->
     * 0.358 ms); the two forms give the same bits. */
    if constexpr (SEL) {
      const bool neg = signbit(U);
      return U * weno3_side(neg ? p1 : m2, neg ? c0 : m1, neg ? m1 : c0);
    } else {
      return signbit(U) ? U * weno3_side(p1, c0, m1) : U * weno3_side(m2, m1, c0);
    }
  } else if constexpr (S == 5) { /* WENO5, the two forms as for WENO3 */
    if constexpr (SEL) {
      const bool neg = signbit(U);
      return U * weno5_side(neg ? p2 : m3, neg ? p1 : m2, neg ? c0 : m1, neg ? m1 : c0, neg ? m2 : p1);
    } else {
      return signbit(U) ? U * weno5_side(p2, p1, c0, m1, m2) : U * weno5_side(m3, m2, m1, c0, p1);
    }
  } else if constexpr (S == 6) { /* centred 2nd order */
    return U * (0.5f * (c0 + m1));
  } else {                       /* 1st-order upstream */
    return fmaxf(0.f, U) * m1 + fminf(0.f, U) * c0;
  }
}

/* ---- perturbation pressure (cuda_pressureDevice.cu:53-113) of rho*theta*(1 + mf), with
 *      mf = (R_v/R) q_v the moisture factor (0 when dry).  r = rho*theta_m/(rho*theta)_BS - 1 is
 *      formed from the small parts, (rho*theta - (rho*theta)_BS) and mf, so that it keeps
 *      full relative precision even where moisture makes theta_m differ from the base state
 *      by a few percent. ---- */
/* the base-state rows p' reads at (z, col): (rho*theta)_BS, its inverse and p_BS, or the
 * reference form's base pressure term (as DynRows, loaded ahead of use on terrain) */
struct PRows { float pbs, rth, irth, pbsraw; };
template <class C>
__device__ __forceinline__ PRows p_rows(const StepArgs &a, int z, unsigned col) {
  PRows r{0.f, 0.f, 0.f, 0.f};
  if (a.pform == 0) {
    r.pbsraw = cprof<C>(a, PR_PBSRAW, z, col);
  } else {
    r.pbs = cprof<C>(a, PR_PBS, z, col);
    r.rth = cprof<C>(a, PR_RTH, z, col);
    r.irth = cprof<C>(a, PR_IRTH, z, col);
  }
  return r;
}
template <class C>
__device__ __forceinline__ float pprime_r(const StepArgs &a, float rth, float mf, const PRows &R) {
  if (a.pform == 0) return powf(rth * (1.f + mf) * a.c1p, a.gam) - R.pbsraw;
  const float ib = R.irth;
  float r = fmaf(rth * ib, mf, (rth - R.rth) * ib);
  float s;
  if (fabsf(r) < 0.125f) {
    s = fmaf(r, a.pc[7], a.pc[6]);
    s = fmaf(r, s, a.pc[5]); s = fmaf(r, s, a.pc[4]); s = fmaf(r, s, a.pc[3]);
    s = fmaf(r, s, a.pc[2]); s = fmaf(r, s, a.pc[1]); s = fmaf(r, s, a.pc[0]);
    s = r * s;
  } else {
    s = expm1f(a.gam * log1pf(r));
  }
  return R.pbs * s;
}
template <class C>
__device__ __forceinline__ float pprime(const StepArgs &a, float rth, float mf, int z, unsigned col) {
  return pprime_r<C>(a, rth, mf, p_rows<C>(a, z, col));
}


template <bool TKE_, int NM_, int SH_, int SE_, int SQV_, int SQL_, bool PHYS_, bool TERR_ = false, bool SB_ = false>
struct Cfg {
  static constexpr bool SB = SB_;             /* one blending weight b of the hybrid schemes for every field */
  static constexpr bool TKE = TKE_;
  static constexpr bool TERR = TERR_;         /* terrain-following grid: per-column metrics and base state */
  static constexpr int NM = NM_;
  static constexpr int NF = 5 + (TKE_ ? 1 : 0) + NM_;
  static constexpr int IE = 5;
  static constexpr int IQV = 5 + (TKE_ ? 1 : 0);
  static constexpr int IQL = IQV + 1;
  static constexpr int IQV_SAFE = NM_ > 0 ? IQV : 0;  /* in-range index for reads behind NM > 0 */
  static constexpr int IE_SAFE = TKE_ ? IE : 0;
  static constexpr int SH = SH_, SE = SE_, SQV = SQV_, SQL = SQL_;
  static constexpr bool PHYS = PHYS_;
  /* own cell and x fluxes in registers (own_faces); through LDS (own_faces_lds) where the kernel has
   * no registers left for them.  256 x 256 x 160, us a launch, registers -> LDS: moist over a hill
   * plain stage 500 (29 VGPRs spilled) -> 383 (none), physics stage 722 (24) -> 692 (20); dry WENO5
   * plain stage 584 (21) -> 465 (none).  Nothing spills and registers are faster in the WENO5 physics
   * stage (528, LDS 556) and in the others (dry plain 192, LDS 255; moist flat plain 310, LDS 321). */
  static constexpr bool REG = !(NM_ > 0 && TERR_) && (PHYS_ || SH_ != 5);
  static constexpr int NV = 4 + NM_;          /* u, v, w, theta, q/rho ... */
  static constexpr int NB = 4 + NM_;          /* face stress components per face family */
  template <int F> static constexpr int sch() {
    return F < 5 ? SH_ : (TKE_ && F == 5 ? SE_ : (F == IQV ? SQV_ : SQL_));
  }
};

/* LDS-qualified float: stencil reads through it compile to ds_read (paired where the offsets
 * allow) rather than flat loads whose address space the compiler would have to prove */
typedef __attribute__((address_space(3))) float SRD;
/* LDS address p + K floats, added where the compiler cannot see it: reads at small constant
 * offsets from the result share it as their base.  Left alone, the compiler folds every constant
 * into each read and then adds a base of its own per paired read (whose offsets reach 255 floats):
 * 40 adds per level and wave of the plain stage. */
template <int K>
__device__ __forceinline__ const SRD *lds_at(const SRD *p) {
  unsigned r;
  asm("v_add_u32 %0, %2, %1" : "=v"(r) : "v"((unsigned)(unsigned long)p), "n"(K * 4));
  return (const SRD *)(unsigned long)r;
}
/* v of the next lane in x (a wave holds whole tile rows); the last lane of a row gets edge */
__device__ __forceinline__ float lane_up(float v, float edge, int tx) {
  constexpr int WAVE_SHL1 = 0x130;         /* DPP: lane i takes lane i + 1; the last lane keeps 'old' */
  const int r = __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge), __builtin_bit_cast(int, v), WAVE_SHL1, 0xf, 0xf, false);
  if constexpr (TX == 64) return __builtin_bit_cast(float, r);
  else return tx == TX - 1 ? edge : __builtin_bit_cast(float, r);
}
/* x fluxes in LDS: those of the ring column x = TX (16-byte rows), or of every face of the tile */
template <class C, bool REG = C::REG>
struct XFaces {
  float g[TY][NFP];
  __device__ __forceinline__ float &at(int f, int fy, int) { return g[fy][f]; }
};
template <class C>
struct XFaces<C, false> {
  float g[C::NF][TY][TX + 1];
  __device__ __forceinline__ float &at(int f, int fy, int fx) { return g[f][fy][fx]; }
};
template <class C, int F, int FE = C::NF>
struct FaceLoop {
  __device__ __forceinline__ static void xf(float (*raw)[RH][RW], XFaces<C> &gx, int fy, int fx, float U, const float *omb) {
    if constexpr (F < FE) {
      const SRD *o = (const SRD *)&raw[0][fy + HH][fx], *r;
      if constexpr (C::REG) r = lds_at<F * RH * RW>(o);
      else r = o + F * RH * RW;
      gx.at(F, fy, fx) = face_flux<C::template sch<F>(), C::PHYS>(U, omb[F], r[0], r[1], r[2], r[3], r[4], r[5]);
      FaceLoop<C, F + 1, FE>::xf(raw, gx, fy, fx, U, omb);
    }
  }
  __device__ __forceinline__ static void yf(float (*raw)[RH][RW], float (*gy)[TY + 1][TX], int fy, int fx, float V, const float *omb) {
    if constexpr (F < FE) {
      const SRD *o = (const SRD *)&raw[0][fy][fx + HH], *r;
      if constexpr (C::REG) r = lds_at<F * RH * RW>(o);
      else r = o + F * RH * RW;
      gy[F][fy][fx] = face_flux<C::template sch<F>(), C::PHYS>(V, omb[F], r[0], r[RW], r[2 * RW], r[3 * RW],
                                                               o[F * RH * RW + 4 * RW], o[F * RH * RW + 5 * RW]);
      FaceLoop<C, F + 1, FE>::yf(raw, gy, fy, fx, V, omb);
    }
  }
  /* z face below level z0 + J0 + 3, win[f][j] holding level z0 + j */
  template <int WD, int J0>
  __device__ __forceinline__ static void zf(float (*win)[WD], float *gz, float W, const float *omb) {
    if constexpr (F < FE) {
      gz[F] = face_flux<C::template sch<F>(), C::PHYS>(W, omb[F], win[F][J0], win[F][J0 + 1], win[F][J0 + 2], win[F][J0 + 3],
                                                       win[F][J0 + 4], win[F][J0 + 5]);
      FaceLoop<C, F + 1, FE>::template zf<WD, J0>(win, gz, W, omb);
    }
  }
};

/* The own cell's x and y neighbours in the planes, i-3, i-2, i-1, i+1, i+2 of fields [F0, F1)
 * (the cell itself, c, is in its register window), and the fluxes through its low faces. */
template <class C, int F0, int F1>
struct OwnStencil {
  float x[F1 - F0][5], y[F1 - F0][5];
  template <int F = F0>
  __device__ __forceinline__ void load(const SRD *o) {    /* o = &raw[0][ty][tx] */
    if constexpr (F < F1) {
      const SRD *r = lds_at<F * RH * RW>(o);
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const int d = j < 3 ? j : j + 1;
        x[F - F0][j] = r[HH * RW + d];
        y[F - F0][j] = d < 5 ? r[d * RW + HH] : o[F * RH * RW + d * RW + HH];
      }
      load<F + 1>(o);
    }
  }
  template <int F = F0>
  __device__ __forceinline__ void flux(const float *c, float U, float V, const float *omb, float *fx, float *fy) const {
    if constexpr (F < F1) {
      constexpr int SC = C::template sch<F>(), N = F - F0;
      fx[F] = face_flux<SC, C::PHYS>(U, omb[F], x[N][0], x[N][1], x[N][2], c[F], x[N][3], x[N][4]);
      fy[F] = face_flux<SC, C::PHYS>(V, omb[F], y[N][0], y[N][1], y[N][2], c[F], y[N][3], y[N][4]);
      flux<F + 1>(c, U, V, omb, fx, fy);
    }
  }
};
/* Advective fluxes of every field through the own cell's low x and y faces; dr: the rho^-1 plane
 * (terrain: D rho^-1) around the cell, rc its value at the cell, hxD, hyD: 0.5 D/dx, 0.5 D/dy (0.5/dx, 0.5/dy).
 * The stages issue about one vector instruction in two cycles of their two waves per SIMD, and
 * every other instruction takes an issue slot of the wave too, so what counts here is their number:
 * the cell's own values come from registers, five neighbours per field and direction from LDS at
 * one base per field, the x flux of the next cell from the neighbouring lane (lane_up), and only
 * the y fluxes go through LDS.  512 x 512 x 128 dry: 391 -> 336 vector and 81 -> 71 LDS
 * instructions per level and wave of the plain stage, 0.643 -> 0.606 ms (3.7 TB/s of its HBM
 * traffic); physics stage 1.099 -> 1.061 ms; over a hill (256 x 256 x 128) 0.249 -> 0.215 ms. */
template <class C>
__device__ __forceinline__ void own_faces(float (*raw)[RH][RW], const float (*dr)[DW], int ty, int tx, const float *c,
                                          float rc, float hxD, float hyD, const float *omb, float *fx, float *fy) {
  const SRD *o = (const SRD *)&raw[0][ty][tx];
  constexpr int FH = C::NM > 0 ? 4 : C::NF;    /* moist: in two halves, which keeps the second's neighbours out of registers */
  OwnStencil<C, 0, FH> n;
  n.load(o);
  const float U = hxD * (n.x[1][2] * dr[ty + 1][tx] + c[1] * rc);
  const float V = hyD * (n.y[2][2] * dr[ty][tx + 1] + c[2] * rc);
  n.flux(c, U, V, omb, fx, fy);
  if constexpr (FH < C::NF) {
    __builtin_amdgcn_sched_barrier(0);
    OwnStencil<C, FH, C::NF> m;
    m.load(o);
    m.flux(c, U, V, omb, fx, fy);
  }
}

/* The same through LDS (C::REG off): the own cell read there as its neighbours are, fluxes to gx and gy. */
template <class C>
__device__ __forceinline__ void own_faces_lds(float (*raw)[RH][RW], const float (*dr)[DW], int ty, int tx, float hxD, float hyD,
                                              const float *omb, XFaces<C> &gx, float (*gy)[TY + 1][TX]) {
  const float U = hxD * (raw[1][ty + HH][tx + HH - 1] * dr[ty + 1][tx] + raw[1][ty + HH][tx + HH] * dr[ty + 1][tx + 1]);
  FaceLoop<C, 0>::xf(raw, gx, ty, tx, U, omb);
  const float V = hyD * (raw[2][ty + HH - 1][tx + HH] * dr[ty][tx + 1] + raw[2][ty + HH][tx + HH] * dr[ty + 1][tx + 1]);
  FaceLoop<C, 0>::yf(raw, gy, ty, tx, V, omb);
}

/* Advective fluxes of fields [F0, F1) through the tile's ring faces: face i of the y face
 * row y = TY and face i of the x face column x = TX. */
template <class C, int F0, int F1>
__device__ __forceinline__ void ring_faces_y(float (*raw)[RH][RW], float (*gy)[TY + 1][TX], const float (*dr)[DW], int i,
                                             float hyD, const float *omb) {
  const int fx = i, fy = TY;
  const float V = hyD * (raw[2][fy + HH - 1][fx + HH] * dr[fy][fx + 1] + raw[2][fy + HH][fx + HH] * dr[fy + 1][fx + 1]);
  FaceLoop<C, F0, F1>::yf(raw, gy, fy, fx, V, omb);
}
template <class C, int F0, int F1>
__device__ __forceinline__ void ring_faces_x(float (*raw)[RH][RW], XFaces<C> &gx, const float (*dr)[DW], int i,
                                             float hxD, const float *omb) {
  const int fx = TX, fy = i;
  const float U = hxD * (raw[1][fy + HH][fx + HH - 1] * dr[fy + 1][fx] + raw[1][fy + HH][fx + HH] * dr[fy + 1][fx + 1]);
  FaceLoop<C, F0, F1>::xf(raw, gx, fy, fx, U, omb);
}

/* SGS stress pieces on a face-located cell (cuda_sgsTurbDevice.cu:60-367).  All
 * arguments are velocities (momentum * rho^-1) around the staggered location. */
struct KmCell { float A, B, E; };   /* rho*Km, rho*Km*invPr, (2/3)*rho*e */

/* Surface-layer scheme for one column (cuda_surfaceLayerDevice.cu:112-521). */
__device__ __forceinline__ void surface_column(const StepArgs &a, long c2, float rho, float ru, float rv, float rth, float rqv, bool moist, float z1) {
  const SurfArgs &s = a.s;
  float z0 = s.z0m[c2], z0t = s.z0t[c2];
  float z1oz0 = (z1 + z0) / z0, z1ozt0 = (z1 + z0t) / z0t;
  float u1 = ru / rho, v1 = rv / rho;
  float U1 = sqrtf(u1 * u1 + v1 * v1);
  float th1 = rth / rho;
  float q1 = moist ? rqv / rho : 0.f;
  const float kap2 = a.kappa * a.kappa;
  const float pi = 3.14159265358979f;
  float cd = s.cd[c2], ch = s.ch[c2], cq = moist ? s.cq[c2] : 0.f;
  float hf = s.hf[c2], qf = moist ? s.qf[c2] : 0.f, tsk = s.tsk[c2], qsk = moist ? s.qsk[c2] : 0.f;
  const float qsk_in = qsk;
  float ust = s.ust[c2];
  float th0;
  const float pfac = powf(a.refP / a.presg, a.R_cp);
  if (a.step_it == a.step_itR && a.step_it == 0) {
    float l0 = logf(z1oz0), l1 = logf(z1ozt0);
    cd = kap2 / (l0 * l0);
    ch = kap2 / (l1 * l1);
    cq = kap2 / (l1 * l1);
  } else if (a.step_it == a.step_itR) {
    cd = (ust * ust) / (U1 * U1);
    th0 = tsk * pfac;
    ch = hf / (U1 * (th0 - th1));
    if (moist) cq = qf / (U1 * (qsk - q1));
  }
  if (a.slSel == 1) {
    if (a.slIdeal == 1) {
      float t = a.simTime;
      hf = (t > a.slTs && t <= a.slTe) ? (float)(a.slWth + a.slAmp * sin((double)pi * (t - a.slTs) / (a.slTe - a.slTs))) : a.slWth;
      if (moist) qf = (t > a.slQts && t <= a.slQte) ? (float)(a.slQamp * sin((double)pi * (t - a.slQts) / (a.slQte - a.slQts))) : a.slWq;
    }
  } else if (a.slSel == 2) {
    int tf = (int)roundf(10.0f / a.dt);
    float tff = (float)tf;
    float tskc = tsk, qskc = qsk;
    if ((a.step_it % tf) == 0 && a.stage == 2) {
      float t = a.simTime;
      if (a.slIdeal == 1 && t > a.slTs && t < a.slTe + a.dt * tff) {
        float prev = fmaxf(t - tff * a.dt, a.slTs);
        tskc = tsk + (float)(a.slAmp * (sin((double)pi * (t - a.slTs) / (a.slTe - a.slTs)) - sin((double)pi * (prev - a.slTs) / (a.slTe - a.slTs))));
        if (moist) qskc = qsk + (float)(a.slQamp * (sin((double)pi * (t - a.slQts) / (a.slQte - a.slQts)) - sin((double)pi * (prev - a.slQts) / (a.slQte - a.slQts))));
      } else {
        tskc = (float)(tsk + a.slTr * a.dt * tff / 3600.0);
        if (moist) qskc = (float)(qsk + a.slQr * a.dt * tff / 3600.0);
      }
      tsk = tskc;
      qsk = qskc;
    }
    th0 = tskc * pfac;
    hf = ch * U1 * (th0 - th1);
    if (moist) qf = cq * U1 * (qskc - q1);
    /* input-qskin option (cuda_surfaceLayerDevice.cu:313-315): the incremented skin humidity
     * feeds this call's flux only; the stored value, and the q0 of the Monin-Obukhov pass,
     * stay at the entry value */
    if (moist && a.slQin) qsk = qsk_in;
  }
  /* Monin-Obukhov iteration: it_max+1 passes */
  th0 = tsk * pfac;
  const float q0 = qsk;
  const int itmax = (a.slStab == 0) ? 5 : 1;
  float cd0 = cd, cdi = cd, chi = ch, cqi = cq, iol = 0.f;
  const float lz = logf(z1oz0), lzt = logf(z1ozt0);
  for (int it = 0; it <= itmax; ++it) {
    float tx = -cd0 * U1 * u1, ty = -cd0 * U1 * v1;
    ust = sqrtf(sqrtf(tx * tx + ty * ty));
    if (a.slStab == 0) {
      if (ust > 0.f) {
        iol = -(a.kappa * a.g * hf) / (ust * ust * ust * th1);
        iol = fmaxf(fminf(iol, 1.f), -1.f);
      } else {
        iol = -1.f;
      }
    } else {
      iol = 0.f;
    }
    float zol = iol * (z1 + z0);
    float pm, ph;
    if (zol < 0.f) {
      float xi = sqrtf(sqrtf(1.f - 16.f * zol));
      float h = 0.5f * (1.f + xi);
      pm = logf(0.5f * (1.f + xi * xi) * h * h) - 2.f * atanf(xi) + 0.5f * pi;
      ph = 2.f * logf(0.5f * (1.f + xi * xi));
    } else {
      pm = -5.f * zol;
      ph = -5.f * zol;
    }
    cdi = kap2 / ((lz - pm) * (lz - pm));
    chi = kap2 / ((lzt - pm) * (lzt - ph));
    cqi = chi;
    if (a.slSel > 1) {
      hf = chi * U1 * (th0 - th1);
      if (moist) qf = cqi * U1 * (q0 - q1);
    }
    cd0 = cdi;
  }
  float Um = sqrtf(u1 * u1 + v1 * v1);
  float t13 = -cdi * Um * ru, t23 = -cdi * Um * rv;
  ust = sqrtf(sqrtf(t13 * t13 + t23 * t23));
  iol = -(a.kappa * a.g * hf) / (ust * ust * ust * th1);
  s.cd[c2] = cdi; s.ch[c2] = chi; s.ust[c2] = ust; s.iol[c2] = iol; s.hf[c2] = hf; s.tsk[c2] = tsk;
  s.t13[c2] = t13; s.t23[c2] = t23; s.th3[c2] = hf * rho;
  if (moist) { s.cq[c2] = cqi; s.qf[c2] = qf; s.qsk[c2] = qsk; s.tq3[c2] = qf * rho; }
}

/* Surface-layer pre-pass of the physics stage (cuda_surfaceLayerDevice.cu:112-521):
 * one thread per column at the lowest level; writes the surface stresses and
 * fluxes the stage kernel applies at z = 0, and the 2-D surface state. */
template <class C>
__device__ __forceinline__ void surface_cell(const StepArgs &a, int x, int y) {
  const long col = (long)y * a.P + x;
  float z1 = 0.5f / (a.dZi * cprof<C>(a, PR_J33, 0, (unsigned)col));
  float rho = a.in[col], ru = a.in[a.fs + col], rv = a.in[2 * a.fs + col], rth = a.in[4 * a.fs + col];
  float rqv = C::NM > 0 ? a.in[C::IQV * a.fs + col] : 0.f;
  surface_column(a, col, rho, ru, rv, rth, rqv, C::NM > 0, z1);
}
/* One thread per column.  With lateral halo storage the pass also covers the two columns and
 * rows past the block's high edges, with those columns' own metrics and state, as the reference's
 * surface layer covers iMax and iMax + 1 (cuda_hydroCoreDevice.cu:907-908): the stage kernels'
 * ring faces read the surface stresses there. */
template <class C>
__global__ void __launch_bounds__(256) surface_kernel(StepArgs a) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y;
  const int ext = a.halo ? 2 : 0;
  if (x >= a.Nx + ext || y >= a.Ny + ext) return;
  surface_cell<C>(a, x, y);
}

/* Dynamics part of the own-cell tendency at level z (both stage kernels):
 * flux-form advection from the x/y face-flux differences dxy and the z face
 * fluxes (the upper one computed here from the register window, the lower one
 * carried), pressure gradient (cuda_pressureDevice.cu:118-194), Rayleigh damping
 * (cuda_rayleighDampingDevice.cu:49-79), buoyancy (cuda_buoyancyDevice.cu:48-67),
 * Coriolis with the geostrophic term (cuda_coriolisDevice.cu:50-58) and the
 * 6th-order filter on rho*w (cuda_filtersDevice.cu:46-122).  win[f][j] holds
 * level z-3+j; pzm/pzp are p' at z-1 and z+1; pgx/pgy the horizontal p'
 * differences. */
/* The metric and base-state rows dyn_tendency reads for the cell (z, col).  On a terrain-following
 * grid they are vector loads from the per-column table, which the stage kernels issue at the start
 * of the level, ahead of the state prefetches: vector-memory loads complete in order, so a row
 * loaded where it is used would wait for every prefetch issued before it.  Flat grids read the
 * shared level table through scalar loads, which wait on their own counter. */
struct DynRows { float Dz, Dp, J33z, J33p, invD, damp, rho, ug, vg; };
template <class C>
__device__ __forceinline__ DynRows dyn_rows(const StepArgs &a, int z, unsigned col) {
  DynRows r;
  r.Dz = cprof<C>(a, PR_D, z, col);
  r.Dp = cprof<C>(a, PR_D, z + 1, col);
  r.J33z = cprof<C>(a, PR_J33, z, col);
  r.J33p = cprof<C>(a, PR_J33, z + 1, col);
  r.invD = cprof<C>(a, PR_INVD, z, col);
  r.damp = a.damp ? cprof<C>(a, PR_DAMP, z, col) : 0.f;
  r.rho = cprof<C>(a, PR_RHO, z, col);
  r.ug = cprof<C>(a, PR_UG, z, col);
  r.vg = cprof<C>(a, PR_VG, z, col);
  return r;
}

/* The rows of level z with D and J33 of the level itself taken from the level below's Dp and
 * J33p (the level loops run upward, so those were loaded one level earlier): two loads fewer
 * per level on terrain-following grids. */
template <class C>
__device__ __forceinline__ DynRows dyn_rows_up(const StepArgs &a, int z, unsigned col, float Dz, float J33z) {
  DynRows r;
  r.Dz = Dz;
  r.J33z = J33z;
  r.Dp = cprof<C>(a, PR_D, z + 1, col);
  r.J33p = cprof<C>(a, PR_J33, z + 1, col);
  r.invD = cprof<C>(a, PR_INVD, z, col);
  r.damp = a.damp ? cprof<C>(a, PR_DAMP, z, col) : 0.f;
  r.rho = cprof<C>(a, PR_RHO, z, col);
  r.ug = cprof<C>(a, PR_UG, z, col);
  r.vg = cprof<C>(a, PR_VG, z, col);
  return r;
}

/* Velocity through the z face between levels z and z + 1 (0 at the lid): D, J33, rho*w and rho^-1 of both. */
__device__ __forceinline__ float zface_vel(const StepArgs &a, int z, float Dz, float J33z, float w, float rin, float Dp,
                                           float J33p, float wp, float rinp) {
  return (z + 1 >= a.Nz) ? 0.f : 0.5f * a.dZi * (Dp * J33p * wp * rinp + Dz * J33z * w * rin);
}

template <class C, int WD>
__device__ __forceinline__ void dyn_tendency(const StepArgs &a, int z, const DynRows &R, float (*win)[WD], float rin, float rinp,
                                             float pzm, float pzp, float pgx, float pgy, const float *dxy,
                                             const float *gzlo, float *gzhi, const float *omb, float *F) {
  constexpr int NF = C::NF;
  const float Dz = R.Dz, Dp = R.Dp, J33z = R.J33z, J33p = R.J33p, invD = R.invD;
  const float W = zface_vel(a, z, Dz, J33z, win[3][3], rin, Dp, J33p, win[3][4], rinp);
  FaceLoop<C, 0>::template zf<WD, 1>(win, gzhi, W, omb);
#pragma unroll
  for (int f = 0; f < NF; ++f) F[f] = -invD * (dxy[f] + (gzhi[f] - gzlo[f]));
  const float rho = win[0][3];
  {
    float fac = a.pgf;
    if constexpr (C::NM > 0) {
      float qs = 0.f;
#pragma unroll
      for (int m = 0; m < C::NM; ++m) qs += win[C::IQV + m][3];
      fac = a.pgf * frcp(1.f + qs * rin * 1e-3f);
    }
    F[1] -= fac * pgx;
    F[2] -= fac * pgy;
    F[3] -= fac * 0.5f * a.dZi * J33z * (pzp - pzm);
  }
  if (a.damp) F[3] -= R.damp * win[3][3];
  if constexpr (C::NM == 0) {
    F[3] -= a.gb * (rho - R.rho);
  } else {
    float rt = rho;
#pragma unroll
    for (int m = 0; m < C::NM; ++m) rt += win[C::IQV + m][3] * 1e-3f;
    F[3] -= (rho * frcp(rt)) * a.gb * (rt - R.rho);
  }
  {
    float u = win[1][3] * rin, v = win[2][3] * rin, w = win[3][3] * rin;
    F[1] += a.fH * (v - R.vg) - a.fV * w;
    F[2] -= a.fH * (u - R.ug);
    F[3] += a.fV * (u - R.ug);
  }
  if (a.filt != 0.f) {
    const float *w = win[3];
    float gm = w[3] - w[2], gp = w[4] - w[3];
    float fm = 10.f * (w[3] - w[2]) - 5.f * (w[4] - w[1]) + (w[5] - w[0]);
    float fp = 10.f * (w[4] - w[3]) - 5.f * (w[5] - w[2]) + (w[6] - w[1]);
    fm = signbit(gm * fm) ? 0.f : fm;
    fp = signbit(gp * fp) ? 0.f : fp;
    F[3] += a.filt * (fp - fm);
  }
}

/* RK3-WS2002 stage update of the own cell (cuda_RKschemes.cu:113-157, positivity of
 * rho*e and moisture), or the tendency itself in emit mode. */
template <class C, bool EMIT, class TL>
__device__ __forceinline__ void rk_store(const StepArgs &a, const TL &T, unsigned oz, const float *F,
                                         const float *base) {
  if (EMIT && a.fem) {
#pragma unroll
    for (int f = 0; f < C::NF; ++f) *(float *)((char *)(a.fem + (long)f * a.fs) + oz) = F[f];
  }
  if (a.emitF) {
#pragma unroll
    for (int f = 0; f < C::NF; ++f) T.st_out(f, oz, F[f]);
  } else {
#pragma unroll
    for (int f = 0; f < C::NF; ++f) {
      float v = fmaf(a.coefdt, F[f], base[f]);
      if (C::TKE && f == C::IE) v = fmaxf(v, 1e-10f);
      if (C::NM > 0 && f >= C::IQV) v = fmaxf(v, 0.f);
      T.st_out(f, oz, v);
    }
  }
}

/* =============================================================================== */
/* Halo cell h of a tile, in tile-local coordinates: the ring-1 cells (the ring
 * around the tile that the derived planes need) come first, then the rest of
 * the 3-cell halo of the raw plane. */
__device__ __forceinline__ void halo_cell(int h, int &lx, int &ly) {
  if (h < NR1) {
    if (h < DW) { ly = -1; lx = h - 1; }
    else if (h < 2 * DW) { ly = TY; lx = h - DW - 1; }
    else if (h < 2 * DW + TY) { lx = -1; ly = h - 2 * DW; }
    else { lx = TX; ly = h - 2 * DW - TY; }
  } else {
    int q = h - NR1;
    if (q < 2 * RW) { ly = -3 + q / RW; lx = -3 + q % RW; }
    else if (q < 4 * RW) { q -= 2 * RW; ly = TY + 1 + q / RW; lx = -3 + q % RW; }
    else { q -= 4 * RW; ly = -1 + q / 4; int c = q % 4; lx = c < 2 ? -3 + c : TX + 1 + (c - 2); }
  }
}

#ifndef FE_PLAIN_WPE
#define FE_PLAIN_WPE 2   /* occupancy hint (waves per SIMD) of the stage kernel without SGS physics */
#endif


/* SGS length scale (cuda_sgstkeDevice.cu:96-151) at level z from theta at z-1, z, z+1 and
 * e = rho*e/rho at z: N^2 = g/theta dtheta/dz (centred); l = Delta, or
 * max(min(0.76 sqrt(e)/N, Delta), 0.01) where N^2 > 0.  Returns l and q = l sqrt(e);
 * the Lilly eddy viscosity is Km(z) = c_k/2 (q(z) + q(z-1)) (cuda_sgsTurbDevice.cu:202-254). */
__device__ __forceinline__ void sgs_lq_v(const StepArgs &a, float J33, float delta, float thm, float th0, float thp, float e,
                                         float &l, float &q) {
  const float dthdz = 0.5f * J33 * a.dZi * (thp - thm);
  const float N2 = a.g * frcp(th0) * dthdz;
  const float se = sqrtf(e);
  l = delta;
  if (N2 > 0.f) l = fmaxf(fminf(0.76f * se * rsqrtf(N2), delta), 1e-2f);
  q = l * se;
}
/* the same at (z, col), the metric rows read there (J33 and Delta given: sgs_lq_v) */
template <class C>
__device__ __forceinline__ void sgs_lq(const StepArgs &a, int z, unsigned col, float thm, float th0, float thp, float e,
                                       float &l, float &q) {
  sgs_lq_v(a, cprof<C>(a, PR_J33, z, col), cprof<C>(a, PR_DELTA, z, col), thm, th0, thp, e, l, q);
}

/* Position of a work-group's tile: tile index b in the model's grid of nbx tiles per row
 * (row-major), and its z segment bz.  Uniform over the work-group. */
struct TilePos { int b, nbx, bz; };

/* The tile of a plain (one model per launch) stage launch, from the work-group's grid
 * position.  XCD-aware tile order: the hardware deals work-groups round-robin over the 8
 * XCDs, so each XCD gets a contiguous run of tiles (neighbours then share an L2). */
__device__ __forceinline__ TilePos grid_tile() {
  const int nbt = gridDim.x * gridDim.y;
  int b = blockIdx.x + gridDim.x * blockIdx.y;
  if ((nbt & 7) == 0) b = (b & 7) * (nbt >> 3) + (b >> 3);
  return TilePos{b, (int)gridDim.x, (int)blockIdx.z};
}

/* Per-thread set-up shared by the stage kernels: tile position, own column, this
 * thread's halo cell, buffer resources of the state arrays and the upwind weights. */
template <class C>
struct Tile {
  static constexpr int NF = C::NF;
  int tid, tx, ty, wave, lane, x0, y0, cx, cy, col;
  int zs, ze;                  /* levels [zs, ze) of this work-group's z segment */
  bool active, baseIn, hasH, hasR1;
  int hlx, hly, hcol, hslot, hd, od;
  unsigned pb, colb, hcolb;
  /* Global accesses go through one buffer resource per array (stage input, RK
   * base, stage output) with the field's byte offset f*fsb in the instruction's
   * scalar offset and one 32-bit column offset per thread: three descriptors and
   * one stride in scalar registers instead of a 64-bit pointer per field and
   * array (all fields of an array span < 4 GiB, checked at set-up). */
  __amdgpu_buffer_rsrc_t rin, rbs, rout;
  unsigned fsb;
  float omb[NF];               /* (1 - b) of the hybrid schemes, 0 for the others */

  __device__ __forceinline__ Tile(const StepArgs &a, TilePos tp, R1Layout L1) {
    tid = threadIdx.x;
    tx = tid % TX;
    ty = tid / TX;
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    x0 = (tp.b % tp.nbx) * TX;
    y0 = (tp.b / tp.nbx) * TY;
    zs = tp.bz * a.zseg;
    ze = min(a.Nz, zs + a.zseg);
    active = (x0 + tx < a.Nx) && (y0 + ty < a.Ny);
    cx = colx(a, x0 + tx);
    cy = rowy(a, y0 + ty);
    col = cy * a.P + cx;
    baseIn = (a.base == a.in);             /* first RK stage: phi^n is the stage input */
    rin = __builtin_amdgcn_make_buffer_rsrc((void *)a.in, 0, -1, FE_RSRC_W3);
    rbs = __builtin_amdgcn_make_buffer_rsrc((void *)a.base, 0, -1, FE_RSRC_W3);
    rout = __builtin_amdgcn_make_buffer_rsrc((void *)a.out, 0, -1, FE_RSRC_W3);
    fsb = (unsigned)a.fs * 4u;
    pb = (unsigned)a.ps * 4u;              /* bytes per xy plane */
    /* this thread's halo cell h: the ring-1 cells (h < NR1) go to the thread ranges of L1,
     * the other halo cells to the remaining threads below NHALO in thread order */
    hlx = 0; hly = 0; hcol = 0; hslot = -1;
    hasH = tid < NHALO;
    int h;
    {
      const int ia = tid - L1.a, ib = tid - L1.b, ic = tid - L1.c;
      if ((unsigned)ia < (unsigned)L1.na) h = ia;
      else if ((unsigned)ib < (unsigned)L1.nb) h = L1.na + ib;
      else if ((unsigned)ic < (unsigned)L1.nc) h = L1.na + L1.nb + ic;
      else {
        const int below = min(max(ia, 0), L1.na) + min(max(ib, 0), L1.nb) + min(max(ic, 0), L1.nc);
        h = NR1 + tid - below;
      }
    }
    hasR1 = hasH && h < NR1;
    if (hasH) {
      halo_cell(h, hlx, hly);
      hslot = (hly + HH) * RW + (hlx + HH);
      hcol = rowy(a, y0 + hly) * a.P + colx(a, x0 + hlx);
    }
    hd = (hly + 1) * DW + (hlx + 1);       /* ring-1 slot (valid when hasR1) */
    od = (ty + 1) * DW + (tx + 1);         /* own slot in the ring-1 region  */
    colb = (unsigned)col * 4u;
    hcolb = (unsigned)hcol * 4u;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      int s = (f < 5) ? C::SH : ((C::TKE && f == C::IE) ? C::SE : (f == C::IQV ? C::SQV : C::SQL));
      float bb = (C::SB || f < 5) ? a.bh : ((C::TKE && f == C::IE) ? a.be : a.bqv);
      omb[f] = (s == 3 || s == 2) ? bb : 0.f;
    }
  }

  __device__ __forceinline__ float ld_in(int f, unsigned o) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rin, o, (unsigned)f * fsb, 0));
  }
  __device__ __forceinline__ float ld_bs(int f, unsigned o) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rbs, o, (unsigned)f * fsb, 0));
  }
  __device__ __forceinline__ void st_out(int f, unsigned o, float v) const {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rout, o, (unsigned)f * fsb, 0);
  }

  /* every field of level zz of the column at byte offset cb, with the vertical
   * boundary rules applied for levels outside [0, Nz) (one uniform branch) */
  __device__ __forceinline__ void lvl(const StepArgs &a, float (&v)[NF], int zz, unsigned cb) const {
    if (zz >= 0 && zz < a.Nz) {
      const unsigned o = (unsigned)zz * pb + cb;
#pragma unroll
      for (int f = 0; f < NF; ++f) v[f] = ld_in(f, o);
    } else {
      const bool top = zz >= a.Nz;
      const unsigned o = top ? (unsigned)(a.Nz - 1) * pb + cb : cb;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if (f == 0) v[f] = cprof<C>(a, PR_RHO, zz, cb >> 2);
        else if (f == 4) v[f] = cprof<C>(a, PR_RTH, zz, cb >> 2);
        else if (top && f == 1) v[f] = C::TERR ? cprof<C>(a, PR_UTOP, 0, cb >> 2) : a.uTop;
        else if (top && f == 2) v[f] = C::TERR ? cprof<C>(a, PR_VTOP, 0, cb >> 2) : a.vTop;
        else if (top && (f == 3 || (C::TKE && f == C::IE))) v[f] = 0.f;
        else v[f] = ld_in(f, o);
      }
    }
  }
  /* moisture factor of theta_m: (R_v/R) q_v */
  __device__ __forceinline__ float mfac(const StepArgs &a, float rho, float qv) const {
    if constexpr (C::NM > 0) return a.Rv_Rg * qv * frcp(rho) * 1e-3f;
    else return 0.f;
  }
};

/* The RK stage that carries the SGS physics (the third stage when the physics
 * runs once per step; every stage otherwise).  The stages without it use
 * stage_plain_kernel below; this kernel is instantiated with C::PHYS only, and
 * its !PHYS branches are the same algorithm without the SGS parts.  Per level z,
 * with two work-group barriers:
 *   P1  write the xy plane of level z (own cell from the register window,
 *       halo from registers prefetched two levels earlier), rho^-1 and p' on
 *       the ring-1 region, velocities of level z+1 and rho*Km terms of level z
 *       on the ring-1 region;
 *   P2  x and y face fluxes (each face once), SGS stresses on x and y faces,
 *       cell-centred TKE transport fluxes;
 *   P3  own-cell tendency (flux differences, z faces from registers, pressure
 *       gradient, buoyancy, damping, Coriolis, filter, SGS divergence, TKE
 *       sources, microphysics) and the RK update.
 * The p' plane is consumed in P2 (own-cell horizontal differences go to
 * registers), so one copy suffices; velocity planes read in P3 and written in
 * the next P1 rotate over four levels (u, v, w: levels z-1..z+1 are live) or
 * three (theta and moisture: z, z+1). */
template <class C, bool EMIT = false, bool MP = true>
__device__ __forceinline__ void stage_body(const StepArgs &a, TilePos tp) {
  constexpr int NF = C::NF;
  constexpr bool PH = C::PHYS;
  /* Prefetch distances in levels: the own column's level z+3 (first read at the end of
   * level z) and the halo's level z+PD are loaded at the start of level z (the
   * register-bound physics stage keeps the halo two levels ahead).  MP = false compiles
   * the microphysics out: the steps between its calls run without its registers. */
  constexpr int PD = PH ? 2 : 3;
  constexpr int NV = PH ? C::NV : 1;
  constexpr int NB = PH ? C::NB : 1;
  __shared__ float raw[NF][RH][RW];
  __shared__ float dvr[DH][DW];          /* rho^-1 of the ring-1 region (terrain-following grids: D rho^-1) */
  __shared__ float dvp[DH][DW];
  __shared__ __align__(16) XFaces<C> gx;
  __shared__ float gy[NF][TY + 1][TX];
  /* velocities u,v,w rotate over four levels, theta and moisture over three */
  __shared__ float velm[PH ? 4 : 1][PH ? 3 : 1][DH][DW];
  __shared__ float vels[PH ? 3 : 1][PH ? NV - 3 : 1][DH][DW];
  __shared__ float kmp[PH ? 2 : 1][PH ? DH : 1][PH ? DW : 1];
  __shared__ float tb1[NB][PH ? TY : 1][PH ? TX + 1 : 1];
  __shared__ float tb2[NB][PH ? TY + 1 : 1][PH ? TX : 1];
  __shared__ float qx[PH ? TY : 1][PH ? TX + 2 : 1];
  __shared__ float qy[PH ? TY + 2 : 1][PH ? TX : 1];

  typedef float Plane[DH][DW];
  auto VL = [&](int lev, int q) -> Plane & { return q < 3 ? velm[lev & 3][q] : vels[(lev + 3) % 3][q - 3]; };
  /* Smagorinsky eddy viscosity (cuda_sgsTurbDevice.cu:238-248, strain rates :60-197) of the
   * cell at plane position (X, Y) of level lev (X, Y >= 1: its strain needs the cells below
   * and to its low sides):
   *   K_m = (c_s Delta)^2 sqrt(max(0, S11^2/2 + S22^2/2 + S33^2/2 + S21^2 + S31^2 + S32^2
   *                                    - max(0, 3 N^2))),  N^2 = g/theta dtheta/dz */
  auto smag = [&](int lev, int X, int Y, unsigned scol) -> float {
    const Plane &u = VL(lev, 0), &v = VL(lev, 1), &w = VL(lev, 2), &th = VL(lev, 3);
    const Plane &um = VL(lev - 1, 0), &vm = VL(lev - 1, 1), &wm = VL(lev - 1, 2), &thm = VL(lev - 1, 3);
    const float J33 = cprof<C>(a, PR_J33, lev, scol), dz = J33 * a.dZi;
    const float s11 = a.dXi * (u[Y][X] - u[Y][X - 1]);
    const float s22 = a.dYi * (v[Y][X] - v[Y - 1][X]);
    const float s33 = dz * (w[Y][X] - wm[Y][X]);
    const float s21 = 0.25f * (a.dXi * ((v[Y][X] - v[Y][X - 1]) + (v[Y - 1][X] - v[Y - 1][X - 1]))
                             + a.dYi * ((u[Y][X] - u[Y - 1][X]) + (u[Y][X - 1] - u[Y - 1][X - 1])));
    const float s31 = 0.25f * (a.dXi * ((w[Y][X] - w[Y][X - 1]) + (wm[Y][X] - wm[Y][X - 1]))
                             + dz * ((u[Y][X] - um[Y][X]) + (u[Y][X - 1] - um[Y][X - 1])));
    const float s32 = 0.25f * (a.dYi * ((w[Y][X] - w[Y - 1][X]) + (wm[Y][X] - wm[Y - 1][X]))
                             + dz * ((v[Y][X] - vm[Y][X]) + (v[Y - 1][X] - vm[Y - 1][X])));
    const float t1 = 0.5f * (s11 * s11 + s22 * s22 + s33 * s33) + s21 * s21 + s31 * s31 + s32 * s32;
    const float N2 = a.g / th[Y][X] * (dz * (th[Y][X] - thm[Y][X]));
    const float cd = a.c_s * cprof<C>(a, PR_DELTA, lev, scol);
    return cd * cd * sqrtf(fmaxf(0.f, t1 - fmaxf(0.f, N2 * 3.f)));
  };

  /* SGS fluxes (tau_31, tau_32, tau_33, tau_theta3, moisture) through the own cell's (plane
   * position X, Y) lower face of level lev, from its planes and those below: A = rho*Km, l, Delta, E = (2/3) rho*e and J33
   * of level lev (cuda_sgsTurbDevice.cu:60-442) */
  auto zflux = [&](int lev, int X, int Y, float A, float l, float delta, float E, float J33, float *zn) {
    auto vp = [&](int q) -> Plane & { return VL(lev, q); };
    auto vz = [&](int q) -> Plane & { return VL(lev - 1, q); };
    const float Bv = A * fmaf(2.f * l, frcp(delta), 1.f);
    float s33 = J33 * a.dZi * (vp(2)[Y][X] - vz(2)[Y][X]);
    float s11 = a.dXi * (vp(0)[Y][X] - vp(0)[Y][X - 1]);
    float s22 = a.dYi * (vp(1)[Y][X] - vp(1)[Y - 1][X]);
    float s31 = 0.25f * (a.dXi * ((vp(2)[Y][X] - vp(2)[Y][X - 1]) + (vz(2)[Y][X] - vz(2)[Y][X - 1]))
                       + J33 * a.dZi * ((vp(0)[Y][X] - vz(0)[Y][X]) + (vp(0)[Y][X - 1] - vz(0)[Y][X - 1])));
    float s32 = 0.25f * (a.dYi * ((vp(2)[Y][X] - vp(2)[Y - 1][X]) + (vz(2)[Y][X] - vz(2)[Y - 1][X]))
                       + J33 * a.dZi * ((vp(1)[Y][X] - vz(1)[Y][X]) + (vp(1)[Y - 1][X] - vz(1)[Y - 1][X])));
    zn[0] = -2.f * A * s31;
    zn[1] = -2.f * A * s32;
    zn[2] = -2.f * A * s33 + (C::TKE ? (2.f / 3.f) * A * (s11 + s22 + s33) : 0.f) + E;
    zn[3] = -Bv * J33 * a.dZi * (vp(3)[Y][X] - vz(3)[Y][X]);
#pragma unroll
    for (int m = 0; m < C::NM; ++m) zn[4 + m] = -Bv * J33 * a.dZi * (vp(4 + m)[Y][X] - vz(4 + m)[Y][X]);
  };

  constexpr RingPlan PL = PLAN_PHYS;
  const Tile<C> T(a, tp, PL.r1);
  const int tid = T.tid, tx = T.tx, ty = T.ty, wave = T.wave, lane = T.lane;
  const int x0 = T.x0, y0 = T.y0, col = T.col, Nz = a.Nz;
  const bool active = T.active, baseIn = T.baseIn, hasH = T.hasH, hasR1 = T.hasR1;
  const int hslot = T.hslot, hd = T.hd, od = T.od;
  const unsigned pb = T.pb, colb = T.colb, hcolb = T.hcolb;
  const float *omb = T.omb;
  auto lvl = [&](float (&v)[NF], int zz, unsigned cb) { T.lvl(a, v, zz, cb); };
  auto mfac = [&](float rho, float qv) { return T.mfac(a, rho, qv); };

  /* The loop starts at the segment's first level z0.  What a level takes over from the one below
   * (z fluxes through its lower face, rho*Km below, eddy viscosities) is formed by the set-up with
   * the loop's own expressions, so a segment costs no level of its own (two levels run below the
   * segment without output instead cost a 16-level segment 10%). */
  const int z0 = T.zs, ze = T.ze;

  /* register window of the own column, z-3..z+3 */
  float win[NF][7];
#pragma unroll
  for (int j = 0; j < 6; ++j) {                    /* slot 6 (z+3) is loaded in the loop */
    float t[NF];
    lvl(t, z0 + j - 3, colb);
#pragma unroll
    for (int f = 0; f < NF; ++f) win[f][j] = t[f];
  }
  /* halo values of levels z .. z+PD */
  float hv[PD + 1][NF];
#pragma unroll
  for (int l = 0; l < PD; ++l) {
    if (hasH) lvl(hv[l], z0 + l, hcolb);
    else {
#pragma unroll
      for (int f = 0; f < NF; ++f) hv[l][f] = 0.f;
    }
  }

  float pz[3];
  {
    float q2 = C::NM > 0 ? win[C::IQV][2] : 0.f;
    float q3 = C::NM > 0 ? win[C::IQV][3] : 0.f, q4 = C::NM > 0 ? win[C::IQV][4] : 0.f;
    pz[1] = pprime<C>(a, win[4][3], mfac(win[0][3], q3), z0, (unsigned)col);
    pz[0] = (z0 > 0) ? pprime<C>(a, win[4][2], mfac(win[0][2], q2), z0 - 1, (unsigned)col) : pz[1];
    pz[2] = (z0 + 1 < Nz) ? pprime<C>(a, win[4][4], mfac(win[0][4], q4), z0 + 1, (unsigned)col) : pz[1];
  }
  float gzlo[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) gzlo[f] = 0.f;
  float rin = frcp(win[0][3]);
  if (z0 > 0) {                                    /* z fluxes through the segment's lower face */
    const float W = zface_vel(a, z0 - 1, cprof<C>(a, PR_D, z0 - 1, (unsigned)col), cprof<C>(a, PR_J33, z0 - 1, (unsigned)col),
                              win[3][2], frcp(win[0][2]), cprof<C>(a, PR_D, z0, (unsigned)col),
                              cprof<C>(a, PR_J33, z0, (unsigned)col), win[3][3], rin);
    FaceLoop<C, 0>::template zf<7, 0>(win, gzlo, W, omb);
  }

  /* ---- physics-stage carried state ---- */
  float zc[PH ? 4 + C::NM : 1];
  float Aown[3] = {0.f, 0.f, 0.f};     /* rho*Km own column at z-1, z, z+1 */
  float riz[5];                         /* rho^-1 own column at z-2..z+2    */
  float kmo = 0.f, lso = 0.f;           /* own Km, l at level z             */
  float kmo1 = 0.f, lso1 = 0.f;         /* own Km, l at level z+1           */
  float qo1 = 0.f;                      /* own l sqrt(e) at level z+1       */
  float kh = 0.f, lh = 0.f, qh = 0.f;   /* ring-1 cell: Km, l, l sqrt(e) at level z */
  if constexpr (PH) {
#pragma unroll
    for (int j = 0; j < 5; ++j) riz[j] = frcp(win[0][j + 1]);
    /* l and Km of levels 0 and 1 (own column) and of level 0 (ring-1 cell); Km(0)
     * takes l sqrt(e) of level -1, evaluated with the boundary values */
    if constexpr (C::TKE) {
      float th[5];
#pragma unroll
      for (int j = 0; j < 5; ++j) th[j] = win[4][j + 1] * riz[j];     /* levels -2..2 */
      float lm, qm, l0, q0, l1, q1;
      sgs_lq<C>(a, z0 - 1, (unsigned)col, th[0], th[1], th[2], win[C::IE][2] * riz[1], lm, qm);
      sgs_lq<C>(a, z0, (unsigned)col, th[1], th[2], th[3], win[C::IE][3] * riz[2], l0, q0);
      sgs_lq<C>(a, z0 + 1, (unsigned)col, th[2], th[3], th[4], win[C::IE][4] * riz[3], l1, q1);
      kmo = a.c_k * 0.5f * (q0 + qm); lso = l0;
      kmo1 = a.c_k * 0.5f * (q1 + q0); lso1 = l1; qo1 = q1;
      if (z0 > 0) {                                /* rho*Km of the level below the segment */
        float l2, q2;
        sgs_lq<C>(a, z0 - 2, (unsigned)col, win[4][0] * frcp(win[0][0]), th[0], th[1], win[C::IE][1] * riz[0], l2, q2);
        const float km = a.c_k * 0.5f * (qm + q2);
        Aown[0] = km * win[0][2];
      }
      if (hasR1) {
        float t2[NF], t1[NF];
        lvl(t2, z0 - 2, hcolb);
        lvl(t1, z0 - 1, hcolb);
        const float r2 = frcp(t2[0]), r1 = frcp(t1[0]), r0 = frcp(hv[0][0]), rp = frcp(hv[1][0]);
        float lq, qq, l0h, q0h;
        sgs_lq<C>(a, z0 - 1, (unsigned)T.hcol, t2[4] * r2, t1[4] * r1, hv[0][4] * r0, t1[C::IE] * r1, lq, qq);
        sgs_lq<C>(a, z0, (unsigned)T.hcol, t1[4] * r1, hv[0][4] * r0, hv[1][4] * rp, hv[0][C::IE] * r0, l0h, q0h);
        kh = a.c_k * 0.5f * (q0h + qq); lh = l0h; qh = q0h;
      }
    }
    /* u,v,w of levels z0-1 and z0, theta and moisture of level z0, on the ring-1 region */
    for (int i = tid; i < DW * DH; i += NT) {
      int dx = i % DW - 1, dy = i / DW - 1;
      int c = rowy(a, y0 + dy) * a.P + colx(a, x0 + dx);
#pragma unroll
      for (int lev = -1; lev <= 0; ++lev) {
        float t[NF];
        lvl(t, z0 + lev, (unsigned)c * 4u);
        float r = frcp(t[0]);
        VL(z0 + lev, 0)[dy + 1][dx + 1] = t[1] * r;
        VL(z0 + lev, 1)[dy + 1][dx + 1] = t[2] * r;
        VL(z0 + lev, 2)[dy + 1][dx + 1] = t[3] * r;
        VL(z0 + lev, 3)[dy + 1][dx + 1] = t[4] * r;       /* level z0-1: the Smagorinsky N^2 */
#pragma unroll
        for (int m = 0; m < C::NM; ++m) VL(z0 + lev, 4 + m)[dy + 1][dx + 1] = t[C::IQV + m] * r;
      }
    }
    __syncthreads();
    if constexpr (!C::TKE) {                        /* Smagorinsky: K_m of level z0 from the planes */
      kmo = smag(z0, tx + 1, ty + 1, (unsigned)col);
      lso = cprof<C>(a, PR_DELTA, z0, (unsigned)col);
    }
    Aown[1] = kmo * win[0][3];
    if (z0 > 0) {
      /* SGS fluxes through the lower face of a later segment: the loop's (zflux) */
      zflux(z0, tx + 1, ty + 1, kmo * win[0][3], lso, cprof<C>(a, PR_DELTA, z0, (unsigned)col),
            C::TKE ? (2.f / 3.f) * win[C::IE_SAFE][3] : 0.f, cprof<C>(a, PR_J33, z0, (unsigned)col), zc);
    } else {
      /* SGS fluxes through the ground: the surface layer's */
      auto v0 = [&](int q) -> Plane & { return VL(z0, q); };
      const int Y = ty + 1, X = tx + 1;
      float A = Aown[1];
      float Bv = A * (1.f + 2.f * lso / cprof<C>(a, PR_DELTA, z0, (unsigned)col));
      float E = C::TKE ? (2.f / 3.f) * win[C::IE][3] : 0.f;
      float s33 = cprof<C>(a, PR_J33, z0, (unsigned)col) * a.dZi * (win[3][3] * riz[2] - win[3][2] * riz[1]);
      float s11 = a.dXi * (v0(0)[Y][X] - v0(0)[Y][X - 1]);
      float s22 = a.dYi * (v0(1)[Y][X] - v0(1)[Y - 1][X]);
      zc[2] = -2.f * A * s33 + (C::TKE ? (2.f / 3.f) * A * (s11 + s22 + s33) : 0.f) + E;
      if (a.slSel > 0) {
        zc[0] = a.s.t13[col];
        zc[1] = a.s.t23[col];
        zc[3] = a.s.th3[col];
      } else {
        /* no surface layer: the interior forms across the lower face, level z0-1 from the
         * vertical boundary rules (the reference's gradients at kMin use its halo level,
         * cuda_sgsTurbDevice.cu:60-197, 390-397) */
        auto vm0 = [&](int q) -> Plane & { return VL(z0 - 1, q); };
        const float J33 = cprof<C>(a, PR_J33, z0, (unsigned)col);
        const float s31 = 0.25f * (a.dXi * ((v0(2)[Y][X] - v0(2)[Y][X - 1]) + (vm0(2)[Y][X] - vm0(2)[Y][X - 1]))
                                 + J33 * a.dZi * ((v0(0)[Y][X] - vm0(0)[Y][X]) + (v0(0)[Y][X - 1] - vm0(0)[Y][X - 1])));
        const float s32 = 0.25f * (a.dYi * ((v0(2)[Y][X] - v0(2)[Y - 1][X]) + (vm0(2)[Y][X] - vm0(2)[Y - 1][X]))
                                 + J33 * a.dZi * ((v0(1)[Y][X] - vm0(1)[Y][X]) + (v0(1)[Y - 1][X] - vm0(1)[Y - 1][X])));
        zc[0] = -2.f * A * s31;
        zc[1] = -2.f * A * s32;
        zc[3] = -Bv * J33 * a.dZi * (v0(3)[Y][X] - vm0(3)[Y][X]);
      }
#pragma unroll
      for (int m = 0; m < C::NM; ++m)
        zc[4 + m] = (m == 0 && a.slSel > 0)
                        ? a.s.tq3[col]
                        : -Bv * cprof<C>(a, PR_J33, z0, (unsigned)col) * a.dZi * (win[C::IQV + m][3] * riz[2] - win[C::IQV + m][2] * riz[1]);
    }
  }

  float bse[NF];                       /* RK base of level z */
#pragma unroll
  for (int f = 0; f < NF; ++f) bse[f] = 0.f;

  /* the column of this lane's ring stress face (the cell past the tile edge): its surface
   * stresses at the lowest level and, on terrain-following grids, its J33 (loaded with the
   * level's other rows) */
  unsigned tfc = 0;
  {
    int i;
    if (on_job(PL.sty, wave, lane, i)) tfc = (unsigned)(rowy(a, y0 + TY) * a.P + colx(a, x0 + i));
    else if (on_job(PL.stx, wave, lane, i)) tfc = (unsigned)(rowy(a, y0 + i) * a.P + colx(a, x0 + TX));
  }
  /* terrain-following grids: rows of the coming level that an earlier level loaded, carried up
   * the column: D(z), J33(z-1), J33(z), J33(z+1), Delta(z), Delta(z+1) of the own column and
   * Delta(z) of the ring-1 cell */
  float cD = 0.f, cJm = 0.f, cJ = 0.f, cJ2 = 0.f, cDl = 0.f, cDlp = 0.f, cDlH = 0.f;
  if constexpr (C::TERR) {
    cD = cprof<C>(a, PR_D, z0, (unsigned)col);
    cJm = cprof<C>(a, PR_J33, z0 - 1, (unsigned)col);
    cJ = cprof<C>(a, PR_J33, z0, (unsigned)col);
    cJ2 = cprof<C>(a, PR_J33, z0 + 1, (unsigned)col);
    cDl = cprof<C>(a, PR_DELTA, z0, (unsigned)col);
    cDlp = cprof<C>(a, PR_DELTA, z0 + 1, (unsigned)col);
    if (hasR1) cDlH = cprof<C>(a, PR_DELTA, z0, (unsigned)T.hcol);
  }
  for (int z = z0; z < ze; ++z) {
    /* always the same as active: a mask formed in each level leaves the compiler a better order
     * of the level than the loop-invariant one (512 x 512 x 128 dry: 1080 -> 1060 us) */
    const bool out = active && z >= T.zs;
    /* ---- loads (vector-memory waits are in order): the RK base of this level first, so
     *      that P3's wait for it leaves the prefetches in flight (two barrier phases cover
     *      its latency, and only one level of it is held in registers); then own level z+3
     *      (read at the end of this level) and the halo of level z+PD ---- */
    const unsigned oz = (unsigned)z * pb + colb;
    /* terrain-following grids: the per-column rows of this level that P1 and P3 read, loaded
     * first (vector-memory loads complete in order, so that P1's waits leave the prefetches
     * in flight); the rows read at the end of the level follow the prefetches */
    DynRows trow{};
    float tdO = 0.f, tdelO = 0.f, tdH = 0.f, tdelH = 0.f, tj33F = 0.f;
    PRows tprH{0.f, 0.f, 0.f, 0.f};
    if constexpr (C::TERR) {
      trow.Dz = cD;
      trow.J33z = cJ;
      trow.J33p = cJ2;
      trow.Dp = cprof<C>(a, PR_D, z + 1, (unsigned)col);
      trow.invD = cprof<C>(a, PR_INVD, z, (unsigned)col);
      trow.damp = a.damp ? cprof<C>(a, PR_DAMP, z, (unsigned)col) : 0.f;
      trow.rho = cprof<C>(a, PR_RHO, z, (unsigned)col);
      trow.ug = cprof<C>(a, PR_UG, z, (unsigned)col);
      trow.vg = cprof<C>(a, PR_VG, z, (unsigned)col);
      tj33F = cprof<C>(a, PR_J33, z, tfc);
      tdO = trow.Dz;
      tdelO = cDl;
      if (hasR1) {
        tdH = cprof<C>(a, PR_D, z, (unsigned)T.hcol);
        tdelH = cDlH;
        tprH = p_rows<C>(a, z, (unsigned)T.hcol);
      }
    }
    if (!a.emitF && !baseIn) {
#pragma unroll
      for (int f = 0; f < NF; ++f) bse[f] = T.ld_bs(f, oz);
    }
    {
      float nxt[NF];
      lvl(nxt, z + 3, colb);
#pragma unroll
      for (int f = 0; f < NF; ++f) win[f][6] = nxt[f];
    }
    if (hasH) lvl(hv[PD], z + PD, hcolb);
    float tdelP = 0.f, tj33M = 0.f, tj33O2 = 0.f, tdelO2 = 0.f, tj33H1 = 0.f, tdelH1 = 0.f;
    PRows tprO2{0.f, 0.f, 0.f, 0.f};
    if constexpr (C::TERR) {
      tdelP = cDlp;
      tj33M = cJm;
      tj33O2 = cprof<C>(a, PR_J33, z + 2, (unsigned)col);
      tdelO2 = cprof<C>(a, PR_DELTA, z + 2, (unsigned)col);
      tprO2 = p_rows<C>(a, z + 2, (unsigned)col);
      if (hasR1) {
        tj33H1 = cprof<C>(a, PR_J33, z + 1, (unsigned)T.hcol);
        tdelH1 = cprof<C>(a, PR_DELTA, z + 1, (unsigned)T.hcol);
      }
      /* the carries for level z + 1 */
      cD = trow.Dp;
      cJm = cJ;
      cJ = cJ2;
      cJ2 = tj33O2;
      cDl = cDlp;
      cDlp = tdelO2;
      cDlH = tdelH1;
    }

    /* ---- P1 ---- */
#pragma unroll
    for (int f = 0; f < NF; ++f) raw[f][ty + HH][tx + HH] = win[f][3];
    if (hasH) {
#pragma unroll
      for (int f = 0; f < NF; ++f) (&raw[f][0][0])[hslot] = hv[0][f];
    }
    (&dvr[0][0])[od] = C::TERR ? tdO * rin : rin;
    (&dvp[0][0])[od] = pz[1];
    if (hasR1) {
      float q = C::NM > 0 ? hv[0][C::IQV] : 0.f;
      (&dvr[0][0])[hd] = C::TERR ? tdH * frcp(hv[0][0]) : frcp(hv[0][0]);
      (&dvp[0][0])[hd] = C::TERR ? pprime_r<C>(a, hv[0][4], mfac(hv[0][0], q), tprH)
                                 : pprime<C>(a, hv[0][4], mfac(hv[0][0], q), z, (unsigned)T.hcol);
    }
    if constexpr (PH) {
      auto vb = [&](int q) -> Plane & { return VL(z + 1, q); };
      {
        float r = frcp(win[0][4]);
        (&vb(0)[0][0])[od] = win[1][4] * r;
        (&vb(1)[0][0])[od] = win[2][4] * r;
        (&vb(2)[0][0])[od] = win[3][4] * r;
        (&vb(3)[0][0])[od] = win[4][4] * r;
#pragma unroll
        for (int m = 0; m < C::NM; ++m) (&vb(4 + m)[0][0])[od] = win[C::IQV + m][4] * r;
      }
      if (hasR1) {
        float r = frcp(hv[1][0]);
        (&vb(0)[0][0])[hd] = hv[1][1] * r;
        (&vb(1)[0][0])[hd] = hv[1][2] * r;
        (&vb(2)[0][0])[hd] = hv[1][3] * r;
        (&vb(3)[0][0])[hd] = hv[1][4] * r;
#pragma unroll
        for (int m = 0; m < C::NM; ++m) (&vb(4 + m)[0][0])[hd] = hv[1][C::IQV + m] * r;
      }
      const float idl = 2.f * frcp(C::TERR ? tdelO : cprof<C>(a, PR_DELTA, z, (unsigned)col));
      const float idlh = C::TERR ? 2.f * frcp(tdelH) : idl;   /* ring-1 cell */
      if constexpr (!C::TKE) {
        /* Smagorinsky: the ring-1 cells whose faces the tile uses (x = TX, y = TY; the
         * low-side ring cells take no stress here) from the planes of levels z, z-1; the own
         * cell's K_m of level z was formed one level earlier */
        kh = (hasR1 && T.hlx >= 0 && T.hly >= 0) ? smag(z, T.hlx + 1, T.hly + 1, (unsigned)T.hcol) : 0.f;
        lh = C::TERR ? cprof<C>(a, PR_DELTA, z, (unsigned)T.hcol) : lso;
      }
      {
        float A = win[0][3] * kmo;
        (&kmp[0][0][0])[od] = A;
        (&kmp[1][0][0])[od] = A * (1.f + lso * idl);
      }
      if (hasR1) {
        float A = hv[0][0] * kh;
        (&kmp[0][0][0])[hd] = A;
        (&kmp[1][0][0])[hd] = A * (1.f + lh * idlh);
      }
    }
    __syncthreads();

    /* ---- P2: faces ---- */
    /* horizontal p' differences of the own cell, read here so that the p' plane
     * is free to be rewritten in the next level's first phase */
    float t11 = 0.f, t21 = 0.f, t22 = 0.f;          /* own-cell SGS stresses, P2 -> P3 */
    float fx[NF], fy[NF];                           /* fluxes through the own cell's low faces, P2 -> P3 */
    const float pgx = 0.5f * a.dXi * (dvp[ty + 1][tx + 2] - dvp[ty + 1][tx]);
    const float pgy = 0.5f * a.dYi * (dvp[ty + 2][tx + 1] - dvp[ty][tx + 1]);
    {
      /* face velocities: 0.5 dXi (D/rho u)|i-1 + (D/rho u)|i); flat grids factor the level's D out
       * of the rho^-1 plane, on terrain-following ones the plane holds D rho^-1 */
      const float Dz = C::TERR ? 1.f : prof(a, PR_D, z);
      const float hxD = 0.5f * a.dXi * Dz, hyD = 0.5f * a.dYi * Dz;
      const float (*dr)[DW] = dvr;
      const float (*dfv)[DW] = dvr;
      /* own x face (low face of the own cell) and own y face */
      {
        if constexpr (C::REG) {
          float c[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) c[f] = win[f][3];
          own_faces<C>(raw, dfv, ty, tx, c, C::TERR ? dfv[ty + 1][tx + 1] : rin, hxD, hyD, omb, fx, fy);
#pragma unroll
          for (int f = 0; f < NF; ++f) gy[f][ty][tx] = fy[f];
        } else {
          own_faces_lds<C>(raw, dfv, ty, tx, hxD, hyD, omb, gx, gy);
        }
      }
      /* ring faces (on the 64 x 8 tile half of the fields per job row) */
      {
        constexpr int HF = PL.split ? NF / 2 : NF;
        int i;
        if (on_job(PL.rfy[0], wave, lane, i)) ring_faces_y<C, 0, HF>(raw, gy, dfv, i, hyD, omb);
        if (on_job(PL.rfx[0], wave, lane, i)) ring_faces_x<C, 0, HF>(raw, gx, dfv, i, hxD, omb);
        if constexpr (PL.split) {
          if (on_job(PL.rfy[1], wave, lane, i)) ring_faces_y<C, HF, NF>(raw, gy, dfv, i, hyD, omb);
          if (on_job(PL.rfx[1], wave, lane, i)) ring_faces_x<C, HF, NF>(raw, gx, dfv, i, hxD, omb);
        }
      }
      if constexpr (PH) {
        const float J33z = C::TERR ? trow.J33z : cprof<C>(a, PR_J33, z, (unsigned)col);
        auto vz = [&](int q) -> const Plane & { return VL(z, q); };
        auto vm = [&](int q) -> const Plane & { return VL(z - 1, q); };
        /* face-located SGS stresses (cuda_sgsTurbDevice.cu:60-367) at the cell (fx,fy), whose
         * column's J33 at level z is J33f */
        auto xface = [&](int fx, int fy, int c2, float J33f) {
          const int X = fx + 1, Y = fy + 1;
          float A = kmp[0][Y][X], Bv = kmp[1][Y][X], E = C::TKE ? (2.f / 3.f) * raw[C::IE][fy + HH][fx + HH] : 0.f;
          float s11 = a.dXi * (vz(0)[Y][X] - vz(0)[Y][X - 1]);
          float s22 = a.dYi * (vz(1)[Y][X] - vz(1)[Y - 1][X]);
          float s33 = J33f * a.dZi * (vz(2)[Y][X] - vm(2)[Y][X]);
          float s21 = 0.25f * (a.dXi * ((vz(1)[Y][X] - vz(1)[Y][X - 1]) + (vz(1)[Y - 1][X] - vz(1)[Y - 1][X - 1]))
                             + a.dYi * ((vz(0)[Y][X] - vz(0)[Y - 1][X]) + (vz(0)[Y][X - 1] - vz(0)[Y - 1][X - 1])));
          float s31 = 0.25f * (a.dXi * ((vz(2)[Y][X] - vz(2)[Y][X - 1]) + (vm(2)[Y][X] - vm(2)[Y][X - 1]))
                             + J33f * a.dZi * ((vz(0)[Y][X] - vm(0)[Y][X]) + (vz(0)[Y][X - 1] - vm(0)[Y][X - 1])));
          tb1[0][fy][fx] = -2.f * A * s11 + (C::TKE ? (2.f / 3.f) * A * (s11 + s22 + s33) : 0.f) + E;
          tb1[1][fy][fx] = -2.f * A * s21;
          tb1[2][fy][fx] = (z == 0) ? a.s.t13[c2] : -2.f * A * s31;
          tb1[3][fy][fx] = -Bv * a.dXi * (vz(3)[Y][X] - vz(3)[Y][X - 1]);
#pragma unroll
          for (int m = 0; m < C::NM; ++m) tb1[4 + m][fy][fx] = -Bv * a.dXi * (vz(4 + m)[Y][X] - vz(4 + m)[Y][X - 1]);
        };
        auto yface = [&](int fx, int fy, int c2, float J33f) {
          const int X = fx + 1, Y = fy + 1;
          float A = kmp[0][Y][X], Bv = kmp[1][Y][X], E = C::TKE ? (2.f / 3.f) * raw[C::IE][fy + HH][fx + HH] : 0.f;
          float s11 = a.dXi * (vz(0)[Y][X] - vz(0)[Y][X - 1]);
          float s22 = a.dYi * (vz(1)[Y][X] - vz(1)[Y - 1][X]);
          float s33 = J33f * a.dZi * (vz(2)[Y][X] - vm(2)[Y][X]);
          float s21 = 0.25f * (a.dXi * ((vz(1)[Y][X] - vz(1)[Y][X - 1]) + (vz(1)[Y - 1][X] - vz(1)[Y - 1][X - 1]))
                             + a.dYi * ((vz(0)[Y][X] - vz(0)[Y - 1][X]) + (vz(0)[Y][X - 1] - vz(0)[Y - 1][X - 1])));
          float s32 = 0.25f * (a.dYi * ((vz(2)[Y][X] - vz(2)[Y - 1][X]) + (vm(2)[Y][X] - vm(2)[Y - 1][X]))
                             + J33f * a.dZi * ((vz(1)[Y][X] - vm(1)[Y][X]) + (vz(1)[Y - 1][X] - vm(1)[Y - 1][X])));
          tb2[0][fy][fx] = -2.f * A * s21;
          tb2[1][fy][fx] = -2.f * A * s22 + (C::TKE ? (2.f / 3.f) * A * (s11 + s22 + s33) : 0.f) + E;
          tb2[2][fy][fx] = (z == 0) ? a.s.t23[c2] : -2.f * A * s32;
          tb2[3][fy][fx] = -Bv * a.dYi * (vz(3)[Y][X] - vz(3)[Y - 1][X]);
#pragma unroll
          for (int m = 0; m < C::NM; ++m) tb2[4 + m][fy][fx] = -Bv * a.dYi * (vz(4 + m)[Y][X] - vz(4 + m)[Y - 1][X]);
        };
        /* own cell: the strain terms shared by its x and y faces once; tau_31 and tau_32 of
         * the own column at level z are the z-face stresses carried from the previous level */
        {
          const int X = tx + 1, Y = ty + 1;
          float A = kmp[0][Y][X], Bv = kmp[1][Y][X], E = C::TKE ? (2.f / 3.f) * raw[C::IE][ty + HH][tx + HH] : 0.f;
          float s11 = a.dXi * (vz(0)[Y][X] - vz(0)[Y][X - 1]);
          float s22 = a.dYi * (vz(1)[Y][X] - vz(1)[Y - 1][X]);
          float s33 = J33z * a.dZi * (vz(2)[Y][X] - vm(2)[Y][X]);
          float s21 = 0.25f * (a.dXi * ((vz(1)[Y][X] - vz(1)[Y][X - 1]) + (vz(1)[Y - 1][X] - vz(1)[Y - 1][X - 1]))
                             + a.dYi * ((vz(0)[Y][X] - vz(0)[Y - 1][X]) + (vz(0)[Y][X - 1] - vz(0)[Y - 1][X - 1])));
          const float iso = C::TKE ? (2.f / 3.f) * A * (s11 + s22 + s33) : 0.f;
          t11 = -2.f * A * s11 + iso + E;
          t22 = -2.f * A * s22 + iso + E;
          t21 = -2.f * A * s21;
          tb1[0][ty][tx] = t11;
          tb1[1][ty][tx] = t21;
          tb1[2][ty][tx] = zc[0];
          tb1[3][ty][tx] = -Bv * a.dXi * (vz(3)[Y][X] - vz(3)[Y][X - 1]);
          tb2[0][ty][tx] = t21;
          tb2[1][ty][tx] = t22;
          tb2[2][ty][tx] = zc[1];
          tb2[3][ty][tx] = -Bv * a.dYi * (vz(3)[Y][X] - vz(3)[Y - 1][X]);
#pragma unroll
          for (int m = 0; m < C::NM; ++m) {
            tb1[4 + m][ty][tx] = -Bv * a.dXi * (vz(4 + m)[Y][X] - vz(4 + m)[Y][X - 1]);
            tb2[4 + m][ty][tx] = -Bv * a.dYi * (vz(4 + m)[Y][X] - vz(4 + m)[Y - 1][X]);
          }
        }
        {
          int i;
          if (on_job(PL.sty, wave, lane, i)) yface(i, TY, z == 0 ? (int)tfc : 0, C::TERR ? tj33F : J33z);
          if (on_job(PL.stx, wave, lane, i)) xface(TX, i, z == 0 ? (int)tfc : 0, C::TERR ? tj33F : J33z);
        }
        if constexpr (C::TKE) {
          /* cell-centred TKE transport fluxes rho*Km*de/dx, rho*Km*de/dy (cuda_sgstkeDevice.cu:309-397) */
          auto ecell = [&](int lx, int ly) { return raw[C::IE][ly + HH][lx + HH] * frcp(raw[0][ly + HH][lx + HH]); };
          auto qxf = [&](int lx, int ly) { return 0.5f * a.dXi * (ecell(lx + 1, ly) - ecell(lx - 1, ly)) * kmp[0][ly + 1][lx + 1]; };
          auto qyf = [&](int lx, int ly) { return 0.5f * a.dYi * (ecell(lx, ly + 1) - ecell(lx, ly - 1)) * kmp[0][ly + 1][lx + 1]; };
          /* own cell: e of the four neighbours with rho^-1 from the ring-1 plane (terrain-following
           * grids: from the raw plane, the same reciprocal) */
          auto eown = [&](int lx, int ly) {
            return C::TERR ? ecell(lx, ly) : raw[C::IE][ly + HH][lx + HH] * dr[ly + 1][lx + 1];
          };
          qx[ty][tx + 1] = 0.5f * a.dXi * (eown(tx + 1, ty) - eown(tx - 1, ty)) * kmp[0][ty + 1][tx + 1];
          qy[ty + 1][tx] = 0.5f * a.dYi * (eown(tx, ty + 1) - eown(tx, ty - 1)) * kmp[0][ty + 1][tx + 1];
          int i;
          if (on_job(PL.qy0, wave, lane, i)) qy[0][i] = qyf(i, -1);
          if (on_job(PL.qxs, wave, lane, i)) {
            const int ly = i % TY, side = i / TY;
            if (side == 0) qx[ly][0] = qxf(-1, ly);
            else qx[ly][TX + 1] = qxf(TX, ly);
          }
          if (on_job(PL.qy1, wave, lane, i)) qy[TY + 1][i] = qyf(i, TY);
        }
      }
    }
    __syncthreads();

    /* ---- P3: own cell ---- */
    {
      const float J33z = C::TERR ? trow.J33z : cprof<C>(a, PR_J33, z, (unsigned)col);
      const float J33p = C::TERR ? trow.J33p : cprof<C>(a, PR_J33, z + 1, (unsigned)col);
      const float rinp = frcp(win[0][4]);
      float dxy[NF], gzhi[NF], F[NF];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if constexpr (C::REG)
          dxy[f] = (lane_up(fx[f], ((const SRD *)gx.g[ty])[f], tx) - fx[f]) + (((const SRD *)&gy[f][ty][tx])[TX] - fy[f]);
        else
          dxy[f] = (gx.at(f, ty, tx + 1) - gx.at(f, ty, tx)) + (gy[f][ty + 1][tx] - gy[f][ty][tx]);
      }
      dyn_tendency<C, 7>(a, z, C::TERR ? trow : dyn_rows<C>(a, z, (unsigned)col), win, rin, rinp, pz[0], pz[2], pgx, pgy, dxy,
                         gzlo, gzhi, omb, F);
      const float rho = win[0][3];
      const int X = tx + 1, Y = ty + 1;

      if constexpr (PH) {
        auto vz = [&](int q) -> const Plane & { return VL(z, q); };
        auto vp = [&](int q) -> const Plane & { return VL(z + 1, q); };
        auto vm = [&](int q) -> const Plane & { return VL(z - 1, q); };
        float zn[4 + C::NM];
        if constexpr (!C::TKE) {
          kmo1 = smag(z + 1, X, Y, (unsigned)col);
          lso1 = cprof<C>(a, PR_DELTA, z + 1, (unsigned)col);
        }
        Aown[2] = kmo1 * win[0][4];
        zflux(z + 1, X, Y, Aown[2], lso1, C::TERR ? tdelP : cprof<C>(a, PR_DELTA, z + 1, (unsigned)col),
              C::TKE ? (2.f / 3.f) * win[C::IE_SAFE][4] : 0.f, J33p, zn);
        const float zdz = J33z * a.dZi;
        F[1] -= a.dXi * (tb1[0][ty][tx + 1] - tb1[0][ty][tx]) + a.dYi * (tb2[0][ty + 1][tx] - tb2[0][ty][tx]) + zdz * (zn[0] - zc[0]);
        F[2] -= a.dXi * (tb1[1][ty][tx + 1] - tb1[1][ty][tx]) + a.dYi * (tb2[1][ty + 1][tx] - tb2[1][ty][tx]) + zdz * (zn[1] - zc[1]);
        F[3] -= a.dXi * (tb1[2][ty][tx + 1] - tb1[2][ty][tx]) + a.dYi * (tb2[2][ty + 1][tx] - tb2[2][ty][tx]) + zdz * (zn[2] - zc[2]);
        F[4] -= a.dXi * (tb1[3][ty][tx + 1] - tb1[3][ty][tx]) + a.dYi * (tb2[3][ty + 1][tx] - tb2[3][ty][tx]) + zdz * (zn[3] - zc[3]);
        if (a.mSGS) {
#pragma unroll
          for (int m = 0; m < C::NM; ++m)
            F[C::IQV + m] -= a.dXi * (tb1[4 + m][ty][tx + 1] - tb1[4 + m][ty][tx]) + a.dYi * (tb2[4 + m][ty + 1][tx] - tb2[4 + m][ty][tx])
                            + zdz * (zn[4 + m] - zc[4 + m]);
        }
        if constexpr (C::TKE) {
          const float rhoe = win[C::IE][3];
          const float e = rhoe * rin;
          const float th = win[4][3] * rin;
          float src = a.g * frcp(th) * zc[3];
          {
            const float ils = frcp(lso);
            float ce = 1.9f * a.c_k + (0.93f - 1.9f * a.c_k) * lso * frcp(C::TERR ? tdelO : cprof<C>(a, PR_DELTA, z, (unsigned)col));
            src += -ce * rhoe * sqrtf(e) * ils;
          }
          {
            float gxu = 0.5f * a.dXi * (vz(0)[Y][X + 1] - vz(0)[Y][X - 1]);
            float gyu = 0.5f * a.dYi * (vz(0)[Y + 1][X] - vz(0)[Y - 1][X]);
            float gzu = 0.5f * zdz * (vp(0)[Y][X] - vm(0)[Y][X]);
            float gxv = 0.5f * a.dXi * (vz(1)[Y][X + 1] - vz(1)[Y][X - 1]);
            float gyv = 0.5f * a.dYi * (vz(1)[Y + 1][X] - vz(1)[Y - 1][X]);
            float gzv = 0.5f * zdz * (vp(1)[Y][X] - vm(1)[Y][X]);
            float gxw = 0.5f * a.dXi * (vz(2)[Y][X + 1] - vz(2)[Y][X - 1]);
            float gyw = 0.5f * a.dYi * (vz(2)[Y + 1][X] - vz(2)[Y - 1][X]);
            float gzw = 0.5f * zdz * (vp(2)[Y][X] - vm(2)[Y][X]);
            const float t31 = zc[0], t32 = zc[1], t33 = zc[2];
            src -= t11 * gxu + t21 * gyu + t31 * gzu + t21 * gxv + t22 * gyv + t32 * gzv + t31 * gxw + t32 * gyw + t33 * gzw;
          }
          {
            float ezp2 = win[C::IE][5] * riz[4], ezm2 = win[C::IE][1] * riz[0];
            float dezp = 0.5f * J33p * a.dZi * (ezp2 - e);
            float dezm = 0.5f * (C::TERR ? tj33M : cprof<C>(a, PR_J33, z - 1, (unsigned)col)) * a.dZi * (e - ezm2);
            src += a.dXi * (qx[ty][tx + 2] - qx[ty][tx]) + a.dYi * (qy[ty + 2][tx] - qy[ty][tx])
                 + zdz * (dezp * Aown[2] - dezm * Aown[0]);
          }
          F[C::IE] += src;
        }
        if constexpr (C::NM > 1 && MP) {
          if (a.mpActive) {
            const float rth = win[4][3];
            const float thd = rth * rin;
            const float c1 = a.c1p;
            /* pressure and Exner factor of the cell (the thermal-forcing temperature below);
             * with the base-pressure option the condensation uses the level's base-state
             * pressure and its Exner factor, tabulated per level */
            const float prf = powf(rth * c1, a.gam);
            const float exf = powf(prf / a.refP, a.R_cp);
            float pr = a.condBase ? cprof<C>(a, PR_PBSRAW, z, (unsigned)col) : prf;
            float Td = thd * (a.condBase ? cprof<C>(a, PR_EXB, z, (unsigned)col) : exf);
            float Tc = fmaxf(-80.f, Td - 273.16f);
            float pvs;
            if (Td >= 273.15f)
              pvs = (6.11239921f + Tc * (0.443987641f + Tc * (0.142986287e-1f + Tc * (0.264847430e-3f + Tc * (0.302950461e-5f
                    + Tc * (0.206739458e-7f + Tc * (0.640689451e-10f + Tc * (-0.952447341e-13f + -0.976195544e-15f * Tc)))))))) * 100.f;
            else
              pvs = (6.11147274f + Tc * (0.503160820f + Tc * (0.188439774e-1f + Tc * (0.420895665e-3f + Tc * (0.615021634e-5f
                    + Tc * (0.602588177e-7f + Tc * (0.385852041e-9f + Tc * (0.146898966e-11f + 0.252751365e-14f * Tc)))))))) * 100.f;
            pvs = fminf(0.99f * pr, pvs);
            const float qv = win[C::IQV][3], ql = win[C::IQL][3];
            float ffor = 0.f, flim = ql * 1e-3f;
            if (a.condSel == 1) {
              ffor = qv * 1e-3f - pvs / (a.R_vapor * Td);
            } else {
              float rvs = (a.condSel == 2) ? pvs / (a.R_vapor * Td) : (pvs / (pr - pvs) / a.Rv_Rg) * rho;
              ffor = (qv * 1e-3f - rvs) / (1.f + (a.L_v * a.L_v * rvs * rin / (a.cp * a.R_vapor * Td * Td)));
            }
            float fc = (fmaxf(ffor, 0.f) - fmaxf(fminf(flim, -ffor), 0.f)) / a.condTs;
            F[C::IQV] -= fc * 1e3f;
            F[C::IQL] += fc * 1e3f;
            float Tf = thd * exf;
            F[4] += ((thd * a.L_v) / (Tf * a.cp)) * fc;
          }
        }
        if (EMIT && out && a.tau) {
          /* SGS stresses of the own cell at level z, in the reference's field order
           * (11, 21, 31, 32, 22, 33, theta 1..3; moisture x, y, z per species) */
          const float tv[9] = {t11, t21, zc[0], zc[1], t22, zc[2], tb1[3][ty][tx], tb2[3][ty][tx], zc[3]};
#pragma unroll
          for (int k = 0; k < 9; ++k) *(float *)((char *)(a.tau + (long)k * a.fs) + oz) = tv[k];
          if (C::NM > 0 && a.mtau && a.mSGS) {
#pragma unroll
            for (int m = 0; m < C::NM; ++m) {
              *(float *)((char *)(a.mtau + (long)(3 * m) * a.fs) + oz) = tb1[4 + m][ty][tx];
              *(float *)((char *)(a.mtau + (long)(3 * m + 1) * a.fs) + oz) = tb2[4 + m][ty][tx];
              *(float *)((char *)(a.mtau + (long)(3 * m + 2) * a.fs) + oz) = zc[4 + m];
            }
          }
        }
#pragma unroll
        for (int q = 0; q < 4 + C::NM; ++q) zc[q] = zn[q];
        Aown[0] = Aown[1];
        Aown[1] = Aown[2];
      }

      if (out) {
        float b0[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) b0[f] = baseIn ? win[f][3] : bse[f];
        rk_store<C, EMIT>(a, T, oz, F, b0);
        if (a.pout) *(float *)((char *)a.pout + oz) = pz[1];
      }
#pragma unroll
      for (int f = 0; f < NF; ++f) gzlo[f] = gzhi[f];
      rin = rinp;
    }

    /* ---- SGS length scale and eddy viscosity one level ahead (loads of this level are
     *      consumed here, at the end, so that their latency is hidden) ---- */
    float r3 = 0.f;
    if constexpr (PH) {
      r3 = frcp(win[0][6]);                             /* rho^-1 at z+3 */
      if constexpr (C::TKE) {
        /* own column: l, Km of level z+2 (theta at z+1..z+3, e at z+2) */
        float l2, q2;
        if constexpr (C::TERR)
          sgs_lq_v(a, tj33O2, tdelO2, win[4][4] * riz[3], win[4][5] * riz[4], win[4][6] * r3, win[C::IE][5] * riz[4], l2, q2);
        else
          sgs_lq<C>(a, z + 2, (unsigned)col, win[4][4] * riz[3], win[4][5] * riz[4], win[4][6] * r3, win[C::IE][5] * riz[4], l2, q2);
        kmo = kmo1; lso = lso1;
        kmo1 = a.c_k * 0.5f * (q2 + qo1); lso1 = l2; qo1 = q2;
        /* ring-1 cell: l, Km of level z+1 (halo levels z..z+2) */
        if (hasR1) {
          const float h0 = frcp(hv[0][0]), h1 = frcp(hv[1][0]), h2 = frcp(hv[2][0]);
          float l1h, q1h;
          if constexpr (C::TERR)
            sgs_lq_v(a, tj33H1, tdelH1, hv[0][4] * h0, hv[1][4] * h1, hv[2][4] * h2, hv[1][C::IE] * h1, l1h, q1h);
          else
            sgs_lq<C>(a, z + 1, (unsigned)T.hcol, hv[0][4] * h0, hv[1][4] * h1, hv[2][4] * h2, hv[1][C::IE] * h1, l1h, q1h);
          kh = a.c_k * 0.5f * (q1h + qh); lh = l1h; qh = q1h;
        }
      } else {
        kmo = kmo1; lso = lso1;
      }
    }

    /* ---- advance the pipelines ---- */
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < 6; ++j) win[f][j] = win[f][j + 1];
    }
#pragma unroll
    for (int l = 0; l < PD; ++l)
#pragma unroll
      for (int f = 0; f < NF; ++f) hv[l][f] = hv[l + 1][f];
    if constexpr (PH) {
#pragma unroll
      for (int j = 0; j < 4; ++j) riz[j] = riz[j + 1];
      riz[4] = r3;
    }
    pz[0] = pz[1];
    pz[1] = pz[2];
    if (z + 2 < Nz) {
      float q = C::NM > 0 ? win[C::IQV][4] : 0.f;
      pz[2] = C::TERR ? pprime_r<C>(a, win[4][4], mfac(win[0][4], q), tprO2)
                      : pprime<C>(a, win[4][4], mfac(win[0][4], q), z + 2, (unsigned)col);
    }
  }
}

/* The stage without SGS physics (the first two RK stages when the physics runs once
 * per step), software-pipelined over levels with one work-group barrier per level:
 * iteration it writes the xy plane of level it (P1), computes the x/y face fluxes of
 * level it-1 (P2) and the own-cell tendency and RK update of level it-2 (P3).  The
 * plane, rho^-1, p' and face-flux buffers have two copies selected by level parity,
 * so the three phases of one iteration never touch the same copy, and the barrier at
 * the end of an iteration orders each copy's writes before its reads.  Every global
 * load is issued one iteration before the iteration that first uses it; the own
 * column and the halo cell are both loaded two levels ahead of P1, so a tile fetches
 * its halo lines while its neighbours fetch the same lines as their own columns. */
template <class C, bool EMIT = false>
__device__ __forceinline__ void stage_plain_body(const StepArgs &a, TilePos tp) {
  constexpr int NF = C::NF;
  __shared__ float raw[2][NF][RH][RW];
  __shared__ float dvr[2][DH][DW];       /* rho^-1 of the ring-1 region (terrain-following grids: D rho^-1) */
  __shared__ float dvp[2][DH][DW];
  __shared__ __align__(16) XFaces<C> gx[2];
  __shared__ float gy[2][NF][TY + 1][TX];
  /* x fluxes through the own cells' low faces (C::REG): carried in registers from P2 to the next
   * iteration's P3, or through LDS when moist (two more fields, and no registers left) */
  constexpr bool FXR = C::REG && C::NM == 0, FXL = C::REG && !FXR;
  /* RK base of P3's level loaded one iteration ahead, or (own cell in registers and moist, for
   * registers) at the start of its own; moist over a hill 383 us a launch ahead, 397 at its own */
  constexpr bool BSA = C::NM == 0 || !C::REG;
  __shared__ float gxo[FXL ? 2 : 1][FXL ? NF : 1][FXL ? TY : 1][FXL ? TX : 1];

  constexpr RingPlan PL = PLAN_PLAIN;
  const Tile<C> T(a, tp, PL.r1);
  const int tx = T.tx, ty = T.ty, wave = T.wave, lane = T.lane, Nz = a.Nz;
  const unsigned pb = T.pb, colb = T.colb, hcolb = T.hcolb;

  /* Loop-carried values live in small register arrays that the body indexes with a
   * compile-time slot offset S: the loop runs two levels per trip (S = 0, 1) and
   * rotates the arrays by two slots at the end of the trip, instead of shifting
   * every array by one slot per level.
   *   win[f][j+S]: own column, level it-5+j (P3's level it-2 at j = 3, P1's level it
   *                at j = 5, j = 7 in flight);
   *   hv[l+S]: halo cell, level it+l;  bs[S]: RK base of level it-2 (bs[S+1] in flight);
   *   pp[S..S+3]: own p' of levels it-3..it;  ri[S..S+2]: own rho^-1 of levels it-2..it;
   *   pg[S]: horizontal p' differences of level it-2 (pg[S+1] written for it-1);
   *   gz[0]: z flux through the lower face of level it-2 (GZS: gz[S], gz[S+1] its upper face);
   *   fx[S]: x flux through the own cell's low face at level it-2 (fx[S+1] written for it-1). */
  /* The pipeline starts at the segment's first level it0 and computes no plane or face outside
   * [it0, ze): p' below the segment and the z flux through its lower face come from the set-up,
   * formed with the loop's own expressions (64 x 64 x 48 in 12 segments of 4 levels: six
   * iterations where two levels below the segment run without output made eight). */
  const int it0 = T.zs, ze = T.ze;
  /* the face's flux in slots that the rotation renames, or copied down in each iteration: WENO5 465 us
   * in slots, 510 copied; moist over a hill 398 and 383 */
  constexpr bool GZS = C::SH == 5;
  float gz[GZS ? 3 : 1][NF], pp[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int l = 0; l < (GZS ? 3 : 1); ++l)
#pragma unroll
    for (int f = 0; f < NF; ++f) gz[l][f] = 0.f;
  /* from levels it0-3 .. it0+2: moist flat grids form it before the window is held (256 x 256 x 160:
   * 331 us after it, 307 before), the others from the window (terrain-following 256 x 256 x 128:
   * 227 us before, 215 from it; 64 x 64 x 48: 16.0 and 15.3) */
  auto below = [&](float (&w6)[NF][6]) {
    const float W = zface_vel(a, it0 - 1, cprof<C>(a, PR_D, it0 - 1, (unsigned)T.col), cprof<C>(a, PR_J33, it0 - 1, (unsigned)T.col),
                              w6[3][2], frcp(w6[0][2]), cprof<C>(a, PR_D, it0, (unsigned)T.col),
                              cprof<C>(a, PR_J33, it0, (unsigned)T.col), w6[3][3], frcp(w6[0][3]));
    FaceLoop<C, 0>::template zf<6, 0>(w6, gz[0], W, T.omb);
    pp[2] = pprime<C>(a, w6[4][2], T.mfac(a, w6[0][2], C::NM > 0 ? w6[C::IQV_SAFE][2] : 0.f), it0 - 1, (unsigned)T.col);
  };
  if (C::NM > 0 && !C::TERR && it0 > 0) {
    float w6[NF][6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      float t[NF];
      T.lvl(a, t, it0 + j - 3, colb);
#pragma unroll
      for (int f = 0; f < NF; ++f) w6[f][j] = t[f];
    }
    below(w6);
  }
  float win[NF][9];
  float hv[4][NF];
  /* the first segment's levels are compile-time constants (their boundary rules fold) */
  auto init = [&](int base) {
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      float t[NF];
      if (j >= 2 && j < 7) {
        T.lvl(a, t, base + j - 5, colb);
      } else {
#pragma unroll
        for (int f = 0; f < NF; ++f) t[f] = 0.f;    /* levels base-5, base-4: never read; 7, 8: loaded */
      }
#pragma unroll
      for (int f = 0; f < NF; ++f) win[f][j] = t[f];
    }
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (T.hasH && l < 2) {
        T.lvl(a, hv[l], base + l, hcolb);
      } else {
#pragma unroll
        for (int f = 0; f < NF; ++f) hv[l][f] = 0.f;
      }
    }
  };
  if (it0 == 0) init(0);
  else init(it0);
  float bs[BSA ? 3 : 1][NF], fx[FXR ? 3 : 1][FXR ? NF : 1];
#pragma unroll
  for (int f = 0; f < NF; ++f)
    for (int l = 0; l < (BSA ? 3 : 1); ++l) bs[l][f] = 0.f;
  if constexpr (FXR)
#pragma unroll
    for (int f = 0; f < NF; ++f) fx[0][f] = fx[1][f] = fx[2][f] = 0.f;
  float ri[4] = {0.f, 0.f, 0.f, 0.f};
  /* terrain-following grids: P1's base-state rows and D of level it (own column and ring-1
   * cell) in slot S, loaded one iteration ahead (slot S+1 for level it+1) */
  PRows pr1[C::TERR ? 3 : 1], prh[C::TERR ? 3 : 1];
  float d1[C::TERR ? 3 : 1], dh[C::TERR ? 3 : 1];
  if (!(C::NM > 0 && !C::TERR) && it0 > 0) {
    float w6[NF][6], t[NF];
    T.lvl(a, t, it0 + 2, colb);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < 5; ++j) w6[f][j] = win[f][j + 2];
      w6[f][5] = t[f];
    }
    below(w6);
  }
  if constexpr (C::TERR) {
    pr1[0] = p_rows<C>(a, it0, (unsigned)T.col);
    d1[0] = cprof<C>(a, PR_D, it0, (unsigned)T.col);
    prh[0] = PRows{0.f, 0.f, 0.f, 0.f};
    dh[0] = 0.f;
    if (T.hasR1) {
      prh[0] = p_rows<C>(a, it0, (unsigned)T.hcol);
      dh[0] = cprof<C>(a, PR_D, it0, (unsigned)T.hcol);
    }
  }
  float pg[3][2] = {{0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}};
  /* terrain-following grids: D and J33 of P3's level, carried up from the level below */
  float cD = 0.f, cJ = 0.f;
  if constexpr (C::TERR) {
    cD = cprof<C>(a, PR_D, it0 - 2, (unsigned)T.col);
    cJ = cprof<C>(a, PR_J33, it0 - 2, (unsigned)T.col);
  }

  auto step = [&](auto slot, int it) {
    constexpr int S = decltype(slot)::value;
    const int z1 = it, z2 = it - 1, z3 = it - 2;
    constexpr int b1 = S, b2 = S ^ 1;                /* copies of levels it (and it-2) and it-1; it has parity S */
    const unsigned o3 = (unsigned)z3 * pb + colb;

    /* ---- terrain-following grids: the metric and base-state rows of P3's level (it-2), issued
     *      before this iteration's prefetches (DynRows) ---- */
    DynRows trow{};
    if constexpr (C::TERR) {
      trow = dyn_rows_up<C>(a, z3, (unsigned)T.col, cD, cJ);
      cD = trow.Dp;
      cJ = trow.J33p;
      pr1[S + 1] = p_rows<C>(a, it + 1, (unsigned)T.col);
      d1[S + 1] = cprof<C>(a, PR_D, it + 1, (unsigned)T.col);
      prh[S + 1] = PRows{0.f, 0.f, 0.f, 0.f};
      dh[S + 1] = 0.f;
      if (T.hasR1) {
        prh[S + 1] = p_rows<C>(a, it + 1, (unsigned)T.hcol);
        dh[S + 1] = cprof<C>(a, PR_D, it + 1, (unsigned)T.hcol);
      }
    }
    /* ---- loads for the next level: RK base of level it-1, own level it+2, halo level it+2 ---- */
    if constexpr (BSA) {
      if (z2 >= it0 && z2 < ze && !a.emitF && !T.baseIn) {
        const unsigned o2 = (unsigned)z2 * pb + colb;
#pragma unroll
        for (int f = 0; f < NF; ++f) bs[S + 1][f] = T.ld_bs(f, o2);
      }
    } else if (z3 >= it0 && !a.emitF && !T.baseIn) {
#pragma unroll
      for (int f = 0; f < NF; ++f) bs[0][f] = T.ld_bs(f, o3);
    }
    {
      float t[NF];
      T.lvl(a, t, it + 2, colb);
#pragma unroll
      for (int f = 0; f < NF; ++f) win[f][7 + S] = t[f];
    }
    if (T.hasH && it + 2 < ze) T.lvl(a, hv[S + 2], it + 2, hcolb);

    /* ---- P1: plane, rho^-1 and p' of level it (above the segment rho^-1 and p' only) ---- */
    ri[S + 2] = frcp(win[0][5 + S]);
    auto plane = [&]() {
#pragma unroll
      for (int f = 0; f < NF; ++f) raw[b1][f][ty + HH][tx + HH] = win[f][5 + S];
      if (T.hasH) {
#pragma unroll
        for (int f = 0; f < NF; ++f) (&raw[b1][f][0][0])[T.hslot] = hv[S][f];
      }
    };
    auto pown = [&]() {
      const float q = C::NM > 0 ? win[C::IQV_SAFE][5 + S] : 0.f;
      pp[S + 3] = C::TERR ? pprime_r<C>(a, win[4][5 + S], T.mfac(a, win[0][5 + S], q), pr1[S])
                          : pprime<C>(a, win[4][5 + S], T.mfac(a, win[0][5 + S], q), z1, (unsigned)T.col);
      if (it == 0) pp[S + 2] = pp[S + 3];            /* p'(-1) = p'(0) */
    };
    auto ring1 = [&]() {
      (&dvr[b1][0][0])[T.od] = C::TERR ? d1[S] * ri[S + 2] : ri[S + 2];
      (&dvp[b1][0][0])[T.od] = pp[S + 3];
      if (T.hasR1) {
        const float qh = C::NM > 0 ? hv[S][C::IQV_SAFE] : 0.f;
        (&dvr[b1][0][0])[T.hd] = C::TERR ? dh[S] * frcp(hv[S][0]) : frcp(hv[S][0]);
        (&dvp[b1][0][0])[T.hd] = C::TERR ? pprime_r<C>(a, hv[S][4], T.mfac(a, hv[S][0], qh), prh[S])
                                         : pprime<C>(a, hv[S][4], T.mfac(a, hv[S][0], qh), z1, (unsigned)T.hcol);
      }
    };
    if (z1 >= Nz) pp[S + 3] = pp[S + 2];             /* p'(Nz) = p'(Nz-1) */
    if constexpr (C::NM > 0 || C::TERR) {
      if (z1 < Nz) pown();
      if (z1 < ze) {
        plane();
        ring1();
      }
    } else if (z1 < Nz) {                            /* one block: level ze's plane is written too and never read */
      plane();
      pown();
      ring1();
    }

    /* ---- P2: x and y face fluxes of level it-1 ---- */
    if (z2 >= it0 && z2 < ze) {
      float (*rw)[RH][RW] = raw[b2];
      /* face velocities: the rho^-1 plane with the level's D factored out, or (terrain) the
       * plane of D rho^-1 */
      const float (*dr)[DW] = dvr[b2];
      pg[S + 1][0] = 0.5f * a.dXi * (dvp[b2][ty + 1][tx + 2] - dvp[b2][ty + 1][tx]);
      pg[S + 1][1] = 0.5f * a.dYi * (dvp[b2][ty + 2][tx + 1] - dvp[b2][ty][tx + 1]);
      const float Dz = C::TERR ? 1.f : prof(a, PR_D, z2);
      const float hxD = 0.5f * a.dXi * Dz, hyD = 0.5f * a.dYi * Dz;
      {
        if constexpr (C::REG) {
          float c[NF], fxn[NF], fy[NF];
#pragma unroll
          for (int f = 0; f < NF; ++f) c[f] = win[f][4 + S];
          own_faces<C>(rw, dr, ty, tx, c, C::TERR ? dr[ty + 1][tx + 1] : ri[S + 1], hxD, hyD, T.omb, fxn, fy);
#pragma unroll
          for (int f = 0; f < NF; ++f) {
            gy[b2][f][ty][tx] = fy[f];
            if constexpr (FXR) fx[S + 1][f] = fxn[f];
            else gxo[b2][f][ty][tx] = fxn[f];
          }
        } else {
          own_faces_lds<C>(rw, dr, ty, tx, hxD, hyD, T.omb, gx[b2], gy[b2]);
        }
      }
      /* ring faces, all fields per job row (splitting them over more waves costs more issue
       * slots than it saves in barrier wait) */
      {
        int i;
        if (on_job(PL.rfy[0], wave, lane, i)) ring_faces_y<C, 0, NF>(rw, gy[b2], dr, i, hyD, T.omb);
        if (on_job(PL.rfx[0], wave, lane, i)) ring_faces_x<C, 0, NF>(rw, gx[b2], dr, i, hxD, T.omb);
      }
    }

    /* ---- P3: own cell of level it-2 ---- */
    if (z3 >= it0) {
      float dxy[NF], gzhi[NF], F[NF];
      float (*wv)[9] = win;
      float w7[NF][7];
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int j = 0; j < 7; ++j) w7[f][j] = wv[f][j + S];
      float xr[NFP];
      if constexpr (C::REG)
#pragma unroll
        for (int f = 0; f < NFP; ++f) xr[f] = f < NF ? ((const SRD *)gx[b1].g[ty])[f] : 0.f;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const SRD *py = (const SRD *)&gy[b1][f][ty][tx];
        if constexpr (C::REG) {
          float px;
          if constexpr (FXR) px = fx[S][f];
          else px = ((const SRD *)&gxo[b1][f][ty][tx])[0];
          dxy[f] = (lane_up(px, xr[f], tx) - px) + (py[TX] - py[0]);
        } else {
          const SRD *px = (const SRD *)&gx[b1].g[f][ty][tx];
          dxy[f] = (px[1] - px[0]) + (py[TX] - py[0]);
        }
      }
      dyn_tendency<C, 7>(a, z3, C::TERR ? trow : dyn_rows<C>(a, z3, (unsigned)T.col), w7, ri[S], ri[S + 1], pp[S], pp[S + 2], pg[S][0], pg[S][1],
                         dxy, gz[GZS ? S : 0], GZS ? gz[GZS ? S + 1 : 0] : gzhi, T.omb, F);
      if constexpr (!GZS)
#pragma unroll
        for (int f = 0; f < NF; ++f) gz[0][f] = gzhi[f];
      if (T.active) {
        float b0[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) b0[f] = T.baseIn ? win[f][3 + S] : bs[BSA ? S : 0][f];
        rk_store<C, EMIT>(a, T, o3, F, b0);
        if (a.pout) *(float *)((char *)a.pout + o3) = pp[S + 1];
      }
    } else if constexpr (GZS) {
#pragma unroll
      for (int f = 0; f < NF; ++f) gz[S + 1][f] = gz[S][f];
    }
    __syncthreads();
  };

  for (int it = it0; it < ze + 2; it += 2) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 >= ze + 2) break;
    step(std::integral_constant<int, 1>{}, it + 1);
    /* ---- rotate the carried arrays by two slots ---- */
#pragma unroll
    for (int f = 0; f < NF; ++f) {
#pragma unroll
      for (int j = 0; j < 7; ++j) win[f][j] = win[f][j + 2];
      hv[0][f] = hv[2][f];
      hv[1][f] = hv[3][f];
      if constexpr (BSA) bs[0][f] = bs[2][f];
      if constexpr (GZS) gz[0][f] = gz[2][f];
      if constexpr (FXR) fx[0][f] = fx[2][f];
    }
    pp[0] = pp[2]; pp[1] = pp[3]; pp[2] = pp[4];
    ri[0] = ri[2]; ri[1] = ri[3];
    pg[0][0] = pg[2][0]; pg[0][1] = pg[2][1];
    if constexpr (C::TERR) {
      pr1[0] = pr1[2]; prh[0] = prh[2];
      d1[0] = d1[2]; dh[0] = dh[2];
    }
  }
}


/* One model per launch: a grid of (tiles in x, tiles in y, z segments) work-groups.  MP =
 * false: the physics stage without the microphysics, for the steps between its calls. */
template <class C, bool EMIT = false, bool MP = true>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(C::PHYS ? 2 : FE_PLAIN_WPE, 8))) stage_kernel(StepArgs a) {
  stage_body<C, EMIT, MP>(a, grid_tile());
}
template <class C, bool EMIT = false>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(FE_PLAIN_WPE, 8))) stage_plain_kernel(StepArgs a) {
  stage_plain_body<C, EMIT>(a, grid_tile());
}

}  // namespace fe
