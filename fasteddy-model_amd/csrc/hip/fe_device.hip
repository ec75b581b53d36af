/*
 * fe_device.hip -- the C-ABI device layer of the FastEddy time step on MI355X.
 *
 * Replaces the reference's CUDA modules behind their own entry points
 * (include/fasteddy_amd.h): SRC/FECUDA/fecuda.c, SRC/GRID/CUDA/cuda_grid.c,
 * SRC/HYDRO_CORE/CUDA/cuda_hydroCore.c and SRC/TIME_INTEGRATION/CUDA/cuda_timeInt.c.
 * Inputs are the host modules' globals and halo-inclusive host arrays; the
 * device keeps interior-only fields in [field][z][y][x] order plus 1-D
 * profiles of the (flat-terrain) metric and base state.
 *
 * One RK3 step is three fused stage launches with out-of-place buffers:
 *   stage 1: S0 -> S1, stage 2: (S1, S0) -> S2, stage 3: (S2, S0) -> S0,
 * the physics stage preceded by a surface-layer pass over the lowest level.
 * All launches go to one non-blocking stream; the host synchronises once per
 * batch.
 */
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <limits.h>
#include <stdint.h>
#include <math.h>
#include <algorithm>
#include <array>
#include <functional>
#include <map>
#include <random>
#include <string>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <vector>
#include "../host/fe_host.h"
#include "../../../include/fasteddy_amd.h"
#include "fe_kernels.h"
#include "fe_stage.hip"
#include "fe_ensemble_kernels.hip"
#include "fe_sgs_kernels.hip"

using namespace fe;

/* The one host global this layer reads that the reference's host modules do not
 * define.  This weak default (the well-conditioned p' form) applies when the
 * layer is linked under those modules; the host module here overrides it. */
extern "C" __attribute__((weak)) int amd_pressureForm = 1;
/* z segments per stage launch: 0 chooses them from the grid (see choose_segments) */
extern "C" __attribute__((weak)) int amd_zSegments = 0;
/* 1: lateral halo storage (the grid as one block of a larger domain, see cuda_gridInit) */
extern "C" __attribute__((weak)) int amd_haloBuffer = 0;

/* The FECUDA module's own globals and parameter query (SRC/FECUDA/fecuda.c:29-47), defined
 * here so that this object alone replaces the reference's FECUDA objects: the launch block
 * shape stays a mandatory key; the fused kernels choose their own tile shapes, so tBx/tBy/tBz
 * are validated and recorded. */
extern "C" {
int tBx, tBy, tBz;
int fecuda_GetParams(void) {
  int rc = 0, r;
  r = queryIntegerParameter("tBx", &tBx, 1, INT_MAX, PARAM_MANDATORY); if (r) rc = r;
  r = queryIntegerParameter("tBy", &tBy, 1, INT_MAX, PARAM_MANDATORY); if (r) rc = r;
  r = queryIntegerParameter("tBz", &tBz, 1, INT_MAX, PARAM_MANDATORY); if (r) rc = r;
  return rc;
}
}

#define HIPCHK(x)                                                                               \
  do {                                                                                          \
    hipError_t e_ = (x);                                                                        \
    if (e_ != hipSuccess) {                                                                     \
      fprintf(stderr, "HIP error %s at %s:%d: %s\n", hipGetErrorName(e_), __FILE__, __LINE__,  \
              hipGetErrorString(e_));                                                           \
      return FE_ERR_HIP;                                                                        \
    }                                                                                           \
  } while (0)

namespace {

struct Dev {
  int fecuda = 0, grid = 0, hydro = 0, timeint = 0;
  hipStream_t stream = nullptr;
  int Nx = 0, Ny = 0, Nz = 0, Nh = 0, P = 0, NF = 0, nTKE = 0, nM = 0;
  int halo = 0, NyS = 0;           /* lateral halo storage; rows per plane (Ny, or Ny + 6 with it) */
  int terrain_np = 0;              /* terrain not periodic at the lateral boundaries (halo storage only) */
  int nseg = 1, zseg = 0;          /* z segments of the stage launches and their length */
  float *lsfM = nullptr;           /* slab means of rho, rho*u, rho*v, rho*theta, rho*q_v, levels -1..Nz */
  float *lsfR = nullptr;           /* large-scale forcing rows, LSF_ROW per level */
  double *lsfP = nullptr;          /* partial slab sums, [part][level -1..Nz][5] */
  double *stat = nullptr;          /* workspace of the statistics reductions, kept from call to call */
  size_t stat_n = 0;
  bool lsfNow = false;             /* the current step's last stage carries the forcing */
  long fs = 0, ps = 0;
  int np = 0;
  std::vector<float> hprof;
  float *prof = nullptr;
  /* terrain-following grids: per-column table [PROW][np][Ny][P] (metric rows from cuda_gridInit,
   * base-state rows from cuda_hydroCoreInit) */
  int terrain = 0;
  std::vector<float> htprof;
  float *tprof = nullptr;
  float *S[3] = {nullptr, nullptr, nullptr};
  float *pout = nullptr;
  /* batch-end emissions (allocated when the host asks for them): SGS stresses
   * (hydroSubGridWrite), SGS moisture fluxes, tendencies (hydroForcingWrite/Log) */
  float *tau = nullptr, *mtau = nullptr, *fem = nullptr;
  float *surf = nullptr;           /* 15 planes of [NyS][P] */
  float *stg = nullptr;            /* halo-inclusive staging, one 3-D field */
  long n3h = 0, n2h = 0;
  float uTop = 0, vTop = 0;
  float ms_per_step = 0;
  int gridBlocks[3] = {0, 0, 0};
  int tb[3] = {0, 0, 0};
  /* per-kernel HIP-event timing on the launch stream: class 0 surface-layer pass, 1 plain stage, 2 physics stage,
   * 3 lateral halo fill */
  int timing = 0;
  std::vector<hipEvent_t> ev;
  std::vector<int> evcls;
  size_t evn = 0;
  float *probe = nullptr;
  long probe_n = 0;
} D;

}  // namespace

#include "fe_segments.h"
#include "fe_transfer.hip"

namespace {

/* A launch on the model's stream, timed as class cls while the event pool has room: the launch
 * carries its pair of events itself (hipExtLaunchKernelGGL takes them from the kernel's own
 * dispatch), where event records of their own between the launches would add about 7 us of wall
 * time per launch. */
template <typename F, typename... A>
void launch_timed(int cls, F kernel, dim3 grid, dim3 block, A... args) {
  if (D.timing && D.evn + 2 <= D.ev.size()) {
    D.evcls[D.evn / 2] = cls;
    hipExtLaunchKernelGGL(kernel, grid, block, 0, D.stream, D.ev[D.evn], D.ev[D.evn + 1], 0, args...);
    D.evn += 2;
  } else {
    hipLaunchKernelGGL(kernel, grid, block, 0, D.stream, args...);
  }
}

enum { SF_CD = 0, SF_CH, SF_CQ, SF_UST, SF_HF, SF_TSK, SF_IOL, SF_Z0M, SF_Z0T, SF_QF, SF_QSK, SF_T13, SF_T23, SF_TH3, SF_TQ3, SF_N };

inline float *surfp(int i) { return D.surf + (long)i * D.ps; }
/* plane offset of the lateral position (x, y), -3 <= x < Nx + 3 and -3 <= y < Ny + 3 with
 * lateral halo storage (as colx/rowy in the stage kernels), 0 <= x < Nx, 0 <= y < Ny otherwise */
inline size_t padded_col(int x, int y) {
  return (size_t)(y < 0 ? y + D.NyS : y) * D.P + (size_t)(x < 0 ? x + D.P : x);
}

/* --------------------------------------------------------------------------- */
/* layout conversion kernels                                                    */
/* The host arrays are z fastest, the device planes x fastest: both conversions go through a 64 x 64
 * tile of (x, z) at one y in LDS, so that either side is read and written in 256-byte runs
 * (without it each lane touched a line of its own: 512 x 512 x 128, one field, 265 us up and
 * 352 us down -> 76 and 99 us). */
constexpr int TT = 64;
__global__ void __launch_bounds__(256) k_host_to_dev(const float *src, float *dst, int Nx, int Ny, int Nz, int Nh, int P, long ps) {
  __shared__ float t[TT][TT + 1];
  const long NYH = Ny + 2 * Nh, NZH = Nz + 2 * Nh;
  const int l = threadIdx.x % TT, r = threadIdx.x / TT, x0 = blockIdx.x * TT, z0 = blockIdx.z * TT, y = blockIdx.y;
  for (int i = r; i < TT; i += 256 / TT)
    if (x0 + i < Nx && z0 + l < Nz) t[i][l] = src[((long)(x0 + i + Nh) * NYH + (y + Nh)) * NZH + (z0 + l + Nh)];
  __syncthreads();
  for (int i = r; i < TT; i += 256 / TT)
    if (x0 + l < Nx && z0 + i < Nz) dst[(long)(z0 + i) * ps + (long)y * P + x0 + l] = t[l][i];
}

/* rule: 0 rho, 1 rho*u, 2 rho*v, 3 rho*w, 4 rho*theta, 5 sgs tke, 6 moisture (and other fields with
 * zero-gradient halos), 7 pressure, 8 interior only (zero halos) */
__global__ void __launch_bounds__(256) k_dev_to_host(const float *src, float *dst, int Nx, int Ny, int Nz, int Nh, int P, long ps,
                                                     int rule, const float *prof, int np, float uTop, float vTop,
                                                     const float *tprof, int NyS) {
  __shared__ float t[TT][TT + 1];
  const int NXH = Nx + 2 * Nh, NZH = Nz + 2 * Nh;
  const long NYH = Ny + 2 * Nh;
  const int l = threadIdx.x % TT, r = threadIdx.x / TT, i0 = blockIdx.x * TT, k0 = blockIdx.z * TT, j = blockIdx.y;
  const int i = i0 + l;
  int x = i - Nh, y = j - Nh;
  x = ((x % Nx) + Nx) % Nx;
  y = ((y % Ny) + Ny) % Ny;
  const long col = (long)y * P + x;
  auto value = [&](int k) -> float {
    const int z = k - Nh;
    float v;
    if (rule == 8 && (i < Nh || i >= Nx + Nh || j < Nh || j >= Ny + Nh || z < 0 || z >= Nz)) v = 0.f;
    else if (z >= 0 && z < Nz) v = src[z * ps + col];
    else if (tprof && (rule == 0 || rule == 4 || (z >= Nz && (rule == 1 || rule == 2)))) {
      /* terrain-following grid: the column's own base state and top-halo momentum (with lateral
       * halo storage, NyS > Ny, the table holds the lateral halo columns' own rows) */
      const int row = rule == 0 ? PR_RHO : (rule == 4 ? PR_RTH : (rule == 1 ? PR_UTOP : PR_VTOP));
      const int hx = i - Nh, hy = j - Nh;
      const long tcol = (NyS > Ny && hx >= -3 && hx < Nx + 3 && hy >= -3 && hy < Ny + 3)
                            ? (long)(hy < 0 ? hy + NyS : hy) * P + (hx < 0 ? hx + P : hx)
                            : col;
      v = tprof[((long)row * np + (z + 3)) * ps + tcol];
    }
    else if (rule == 0) v = prof[(z + 3) * PROW + PR_RHO];
    else if (rule == 4) v = prof[(z + 3) * PROW + PR_RTH];
    else if (rule == 7) v = (k == 0) ? 0.f : src[(z < 0 ? 0 : Nz - 1) * ps + col];
    else if (z < 0) v = src[col];
    else if (rule == 1) v = uTop;
    else if (rule == 2) v = vTop;
    else if (rule == 3 || rule == 5) v = 0.f;
    else v = src[(long)(Nz - 1) * ps + col];
    return v;
  };
  for (int k = r; k < TT; k += 256 / TT)
    if (i < NXH && k0 + k < NZH) t[k][l] = value(k0 + k);
  __syncthreads();
  for (int n = r; n < TT; n += 256 / TT)
    if (i0 + n < NXH && k0 + l < NZH) dst[((long)(i0 + n) * NYH + j) * NZH + k0 + l] = t[l][n];
}

/* Lateral halo of a block with lateral halo storage (see cuda_gridInit) from the block's own
 * periodic images -- the cells a decomposed run receives from its neighbours before every stage
 * (cuda_hydroCoreDevice.cu:276-315, fecuda_Utils.cu:205-418) -- for every plane blockIdx.y (plane stride ps) of every field blockIdx.z (field
 * stride fs); one thread per halo cell.  The first nbx work-groups copy the three columns past
 * each x edge over the block's rows (six consecutive threads per row); the others, six per
 * 256-column chunk, one row each of the three past each y edge, over the block's columns and
 * the x halo (the corners).  Sources are interior cells and destinations halo cells, so the
 * copies are independent. */
constexpr int HALO_NT = 256;
__global__ void __launch_bounds__(HALO_NT) k_halo_fill(float *S, long fs, long ps, int Nx, int Ny, int P, int NyS) {
  const int nbx = (2 * HH * Ny + HALO_NT - 1) / HALO_NT;
  float *pl = S + (long)blockIdx.z * fs + (long)blockIdx.y * ps;
  int x, y, sx, sy;
  if ((int)blockIdx.x < nbx) {
    const int h = blockIdx.x * HALO_NT + threadIdx.x;
    if (h >= 2 * HH * Ny) return;
    const int k = h % (2 * HH);
    y = h / (2 * HH);
    x = k < HH ? k - HH : Nx + k - HH;
    sx = k < HH ? x + Nx : x - Nx;
    sy = y;
  } else {
    const int b = blockIdx.x - nbx, k = b % (2 * HH), c = (b / (2 * HH)) * HALO_NT + threadIdx.x;
    if (c >= Nx + 2 * HH) return;
    x = c - HH;
    y = k < HH ? k - HH : Ny + k - HH;
    sx = x < 0 ? x + Nx : (x >= Nx ? x - Nx : x);
    sy = k < HH ? y + Ny : y - Ny;
  }
  const int dx = x < 0 ? x + P : x, dy = y < 0 ? y + NyS : y;
  pl[(long)dy * P + dx] = pl[(long)sy * P + sx];
}

__global__ void k_2d_to_dev(const float *src, float *dst, int Nx, int Ny, int Nh, int P) {
  int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
  if (x >= Nx) return;
  dst[(long)y * P + x] = src[(long)(x + Nh) * (Ny + 2 * Nh) + (y + Nh)];
}
__global__ void k_2d_to_host(const float *src, float *dst, int Nx, int Ny, int Nh, int P) {
  int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
  if (j >= Ny + 2 * Nh) return;
  int x = (((i - Nh) % Nx) + Nx) % Nx, y = (((j - Nh) % Ny) + Ny) % Ny;
  dst[(long)i * (Ny + 2 * Nh) + j] = src[(long)y * P + x];
}

/* --------------------------------------------------------------------------- */
/* kernel variant table                                                         */
typedef void (*stage_fn)(StepArgs);
typedef void (*surface_fn)(StepArgs);
typedef void (*ens_fn)(EnsQueues, int);
typedef void (*ens_surface_fn)(const StepArgs *, int);

struct Variant {
  stage_fn plain, phys, plain_emit, phys_emit;   /* *_emit: the batch's last stage, with emissions */
  stage_fn phys_nomp;                            /* physics stage without the microphysics (its off steps) */
  surface_fn surface;
  ens_fn ens_plain, ens_phys;                    /* persistent ensemble stage kernels (null: no ensemble) */
  ens_surface_fn ens_surface;
  bool sb;                                       /* compiled for one blending weight of the hybrid schemes */
  const char *name;
};

/* SB: compiled for equal blending weights b of the hybrid schemes.  A face's six stencil weights
 * depend on the wind's sign and b only, so they are then formed once per face for all fields, not
 * once per field group (20 of 390 vector instructions per level and wave of the plain stage); the
 * results are the same bits. */
template <bool TKE, int NM, int SH, int SE, int SQV, int SQL, bool ENS, bool TERR, bool SB>
Variant make_variant(const char *name) {
  Variant v;
  v.sb = SB;
  v.plain = stage_plain_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, false, TERR, SB>, false>;
  v.plain_emit = stage_plain_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, false, TERR, SB>, true>;
  v.phys = stage_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, TERR, SB>, false>;
  v.phys_emit = stage_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, TERR, SB>, true>;
  if constexpr (NM > 1) v.phys_nomp = stage_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, TERR, SB>, false, false>;
  else v.phys_nomp = v.phys;
  v.surface = surface_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, TERR, SB>>;
  v.ens_plain = nullptr;
  v.ens_phys = nullptr;
  v.ens_surface = nullptr;
  if constexpr (ENS) {
    v.ens_plain = ens_stage_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, false, false, SB>, false>;
    v.ens_phys = ens_stage_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, false, SB>, true>;
    v.ens_surface = ens_surface_kernel<Cfg<TKE, NM, SH, SE, SQV, SQL, true, false, SB>>;
  }
  v.name = name;
  return v;
}

Variant g_var;      /* the model's kernels, for any blending weights */
Variant g_var_sb;   /* the same for one weight of every field; g_var where the schemes have no weight to share */
int g_var_ok = 0;

template <bool TKE, int NM, int SH, int SE, int SQV, int SQL, bool ENS = false, bool TERR = false>
void set_variants(const char *name) {
  g_var = g_var_sb = make_variant<TKE, NM, SH, SE, SQV, SQL, ENS, TERR, false>(name);
  constexpr bool hyb = SH == 2 || SH == 3;                 /* schemes with a blending weight */
  if constexpr (hyb && (TKE || NM > 0)) g_var_sb = make_variant<TKE, NM, SH, SE, SQV, SQL, ENS, TERR, true>(name);
}

/* The kernels for the weights that a launch carries: they are the program's variables, read for every
 * launch (for an ensemble member when it is added), and need not be those of the set-up. */
const Variant &variant_of(const StepArgs &a) {
  const bool one = (D.nTKE == 0 || a.be == a.bh) && (D.nM == 0 || a.bqv == a.bh);
  return one ? g_var_sb : g_var;
}

int select_variant(void) {
  const int tke = (turbulenceSelector > 0 && TKESelector > 0);
  const int nm = (moistureSelector > 0) ? moistureNvars : 0;
  const int sh = advectionSelector, se = tke ? TKEAdvSelector : 3;
  const int sqv = nm > 0 ? moistureAdvSelectorQv : 3;
  const int sql = nm > 1 ? (moistureAdvSelectorQi == 0 ? 0 : (moistureAdvSelectorQi == 1 ? 4 : 5)) : 5;
  g_var_ok = 0;
  if (D.terrain) {
    /* terrain-following grids: per-column metrics and base state, compiled for HYB56
     * advection with the prognostic-TKE closure (dry, and the shallow-cumulus q_v/q_l set with
     * WENO5 liquid) and with the Smagorinsky closure (dry) */
    if (tke && nm == 0 && sh == 3 && se == 3) {
      set_variants<true, 0, 3, 3, 3, 5, false, true>("dry+tke hyb56/hyb56 terrain-following");
    } else if (tke && nm == 2 && sh == 3 && se == 3 && sqv == 3 && sql == 5) {
      set_variants<true, 2, 3, 3, 3, 5, false, true>("moist2+tke hyb56/hyb56/hyb56/weno5 terrain-following");
    } else if (!tke && turbulenceSelector > 0 && nm == 0 && sh == 3) {
      set_variants<false, 0, 3, 3, 3, 5, false, true>("dry smagorinsky hyb56 terrain-following");
    } else {
      fprintf(stderr, "select_variant: terrain-following grids run HYB56 advection with the prognostic-TKE closure "
                      "(dry, or q_v/q_l with WENO5 liquid) or the dry Smagorinsky closure\n");
      return FE_ERR_TERRAIN;
    }
    g_var_ok = 1;
    return FE_OK;
  }
  if (tke && nm == 0 && sh == 3 && se == 3) { set_variants<true, 0, 3, 3, 3, 5, true>("dry+tke hyb56/hyb56"); g_var_ok = 1; }
  else if (tke && nm == 2 && sh == 3 && se == 3 && sqv == 3 && sql == 5) { set_variants<true, 2, 3, 3, 3, 5, true>("moist2+tke hyb56/hyb56/hyb56/weno5"); g_var_ok = 1; }
  else if (tke && nm == 2 && sh == 3 && se == 3 && sqv == 2 && sql == 5) { set_variants<true, 2, 3, 3, 2, 5>("moist2+tke hyb56/hyb56/hyb34/weno5"); g_var_ok = 1; }
  else if (tke && nm == 2 && sh == 3 && se == 3 && sqv == 3 && sql == 0) { set_variants<true, 2, 3, 3, 3, 0>("moist2+tke hyb56/.../upstream"); g_var_ok = 1; }
  else if (tke && nm == 1 && sh == 3 && se == 3 && sqv == 3) { set_variants<true, 1, 3, 3, 3, 5>("moist1+tke hyb56"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 5 && se == 5) { set_variants<true, 0, 5, 5, 3, 5>("dry+tke weno5/weno5"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 2 && se == 2) { set_variants<true, 0, 2, 2, 3, 5>("dry+tke hyb34/hyb34"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 1 && se == 1) { set_variants<true, 0, 1, 1, 3, 5>("dry+tke quick/quick"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 0 && se == 0) { set_variants<true, 0, 0, 0, 3, 5>("dry+tke upstream"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 6 && se == 6) { set_variants<true, 0, 6, 6, 3, 5>("dry+tke centred2"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 4 && se == 4) { set_variants<true, 0, 4, 4, 3, 5>("dry+tke weno3"); g_var_ok = 1; }
  else if (tke && nm == 0 && sh == 3 && se == 0) { set_variants<true, 0, 3, 0, 3, 5>("dry+tke hyb56/upstream"); g_var_ok = 1; }
  else if (!tke && turbulenceSelector == 0 && nm == 0 && sh == 3) { set_variants<false, 0, 3, 3, 3, 5>("dry inviscid hyb56"); g_var_ok = 1; }
  else if (!tke && turbulenceSelector > 0 && nm == 0 && sh == 3) { set_variants<false, 0, 3, 3, 3, 5, true>("dry smagorinsky hyb56"); g_var_ok = 1; }
  else if (!tke && turbulenceSelector > 0 && nm == 2 && sh == 3 && sqv == 3 && sql == 5) { set_variants<false, 2, 3, 3, 3, 5>("moist2 smagorinsky hyb56/hyb56/weno5"); g_var_ok = 1; }
  return g_var_ok ? FE_OK : FE_ERR_UNSUPPORTED;
}

void fill_args(StepArgs &a, int stage, const float *in, const float *base, float *out, int emitF, float *pout) {
  memset(&a, 0, sizeof a);
  a.in = in; a.base = base; a.out = out; a.prof = D.prof; a.pout = pout;
  a.tprof = D.terrain ? D.tprof : nullptr;
  if (pout) {                      /* the last stage of a batch also emits what the host will read */
    a.tau = D.tau; a.mtau = D.mtau; a.fem = D.fem;
  }
  a.s.cd = surfp(SF_CD); a.s.ch = surfp(SF_CH); a.s.cq = surfp(SF_CQ); a.s.ust = surfp(SF_UST); a.s.hf = surfp(SF_HF);
  a.s.tsk = surfp(SF_TSK); a.s.iol = surfp(SF_IOL); a.s.z0m = surfp(SF_Z0M); a.s.z0t = surfp(SF_Z0T); a.s.qf = surfp(SF_QF);
  a.s.qsk = surfp(SF_QSK); a.s.t13 = surfp(SF_T13); a.s.t23 = surfp(SF_T23); a.s.th3 = surfp(SF_TH3); a.s.tq3 = surfp(SF_TQ3);
  a.Nx = D.Nx; a.Ny = D.Ny; a.Nz = D.Nz; a.P = D.P; a.fs = D.fs; a.ps = D.ps; a.np = D.np;
  a.halo = D.halo; a.NyS = D.NyS;
  a.dXi = dXi; a.dYi = dYi; a.dZi = dZi;
  static const float coef[3] = {1.0f / 3.0f, 0.5f, 1.0f};
  a.coefdt = coef[stage] * dt;
  a.bh = 1.f - b_hyb; a.be = 1.f - TKEAdvSelector_b_hyb; a.bqv = 1.f - moistureAdvSelectorQv_b;
  a.g = accel_g; a.fH = corioConstHorz; a.fV = corioConstVert;
  a.pgf = pgfSelector > 0 ? 1.f : 0.f; a.gb = buoyancySelector > 0 ? accel_g : 0.f;
  a.Rv_Rg = Rv_Rg; a.c1p = R_gas / powf(refPressure, R_cp); a.gam = cp_cv;
  {
    double c = 1.0, gm = (double)cp_cv;
    for (int n = 1; n <= 8; ++n) { c = c * (gm - (n - 1)) / n; a.pc[n - 1] = (float)c; }
  }
  a.pform = amd_pressureForm;
  a.filt = filterSelector > 0 ? (float)(0.015625 * filter_6th_coeff / (1.0 * dt)) : 0.f;
  a.damp = dampingLayerSelector > 0;
  a.uTop = D.uTop; a.vTop = D.vTop;
  a.c_k = c_k; a.kappa = kappa; a.refP = refPressure; a.presg = pres_grnd; a.R_cp = R_cp; a.L_v = L_v; a.cp = cp_gas;
  a.R_vapor = R_vapor; a.condTs = moistureCondTscale; a.condSel = moistureCond; a.condBase = moistureCondBasePres;
  a.mSGS = moistureSGSturb > 0;
  /* Smagorinsky constant of the non-TKE closure; 0 without turbulence, so that the
   * closure's K_m, and with it every SGS stress, is zero in the inviscid form */
  a.c_s = (turbulenceSelector > 0 && TKESelector == 0) ? c_s : 0.f;
  a.step_it = simTime_it; a.step_itR = simTime_itRestart; a.simTime = simTime; a.dt = dt;
  a.slSel = surflayerSelector; a.slIdeal = surflayer_idealsine; a.slStab = surflayer_stab;
  a.slQin = surflayer_qskin_input == 1;
  a.slWth = surflayer_wth; a.slWq = surflayer_wq; a.slTr = surflayer_tr; a.slQr = surflayer_qr;
  a.slTs = surflayer_ideal_ts; a.slTe = surflayer_ideal_te; a.slAmp = surflayer_ideal_amp;
  a.slQts = surflayer_ideal_qts; a.slQte = surflayer_ideal_qte; a.slQamp = surflayer_ideal_qamp;
  a.stage = stage;
  a.emitF = emitF;
  a.zseg = D.zseg;
  if (moistureSelector > 0 && moistureCond > 0 && moistureNvars > 1) {
    int tf = (int)roundf(fmaxf(moistureMPcallTscale, dt) / dt);
    a.mpActive = (simTime_it % tf) == 0;
  }
}

inline int physics_stage(int stage) { return (physics_oneRKonly == 0) || (stage == numRKstages); }

/* Work-groups of a stage launch that run at once on one compute unit (LDS and registers
 * decide: one on the 64 x 8 tile, two on the 16 x 16 tile), the lower of the variant's
 * two stage kernels. */
static int stage_wg_per_cu(const Variant &v) {
  int o1 = 0, o2 = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&o1, v.phys, NT, 0) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&o2, v.plain, NT, 0) != hipSuccess)
    return 1;
  return std::max(1, std::min(o1, o2));
}

/* Split the column into z segments, one work-group per tile and segment, when the
 * tiles alone leave compute units idle: a stage work-group holds one compute unit
 * (its LDS), so fewer than 256 tiles (e.g. 256 x 256 cells = 128 tiles) would run
 * the chip at tiles/256.  Segments are even; amd_zSegments > 0 sets the count.
 * A launch runs in rounds of (work-groups per CU) x CUs work-groups; a segment also loads its
 * window and fills its pipeline (about 2 levels' worth of set-up).  The count minimises rounds x
 * (segment length + 2) over segments of at least 4 levels (fewest segments on ties): a count
 * whose work-groups overflow the slots by a few would add a nearly empty round, and a small grid
 * gets enough work-groups to spread over the CUs. */
void choose_segments() {
  const int tiles = ((D.Nx + TX - 1) / TX) * ((D.Ny + TY - 1) / TY);
  static int ncu = 0;
  if (ncu <= 0) {
    int dev = 0;
    hipDeviceProp_t pr;
    ncu = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&pr, dev) == hipSuccess && pr.multiProcessorCount > 0)
              ? pr.multiProcessorCount : 256;
  }
  const int slots = ncu * stage_wg_per_cu(g_var);
  int n = amd_zSegments;
  if (n <= 0) {
    long best = -1;
    n = 1;
    for (int c = 1; c <= D.Nz; ++c) {
      int len, nseg;
      seg_shape(D.Nz, c, len, nseg);
      if (c > 1 && len < 4) break;
      const long rounds = ((long)tiles * nseg + slots - 1) / slots;
      const long cost = rounds * (len + (nseg > 1 ? 2 : 0));
      if (best < 0 || cost < best) { best = cost; n = c; }
    }
  }
  n = std::max(1, std::min(n, (D.Nz + 1) / 2));
  seg_shape(D.Nz, n, D.zseg, D.nseg);
}

/* learned SGS closure (fe_sgs.hip) */
bool sgs_active();
int sgs_infer(const float *Sin);
int sgs_correct(float *Sout, float coefdt);

/* launch one RK stage (surface-layer pass first when the stage carries the physics); with the
 * learned SGS closure on, its network runs on the stage input first, the physics stage emits
 * the TKE closure's stresses, and the learned stresses replace them where the cells pass */
/* lateral halo storage: the halo of nf fields (field stride fs) of nz planes each from S */
void halo_fill(float *S, long fs, int nf, int nz) {
  const int nbx = (2 * HH * D.Ny + HALO_NT - 1) / HALO_NT, nby = 2 * HH * ((D.Nx + 2 * HH + HALO_NT - 1) / HALO_NT);
  launch_timed(3, k_halo_fill, dim3(nbx + nby, nz, nf), dim3(HALO_NT), S, fs, D.ps, D.Nx, D.Ny, D.P, D.NyS);
}

int launch_stage(int stage, const float *in, const float *base, float *out, int emitF, float *pout) {
  StepArgs a;
  fill_args(a, stage, in, base, out, emitF, pout);
  const Variant &var = variant_of(a);
  /* the stage reads its input's lateral halo (the exchange of a decomposed run) */
  if (D.halo) halo_fill(const_cast<float *>(in), D.fs, D.NF, D.Nz);
  const int phys = physics_stage(stage) && turbulenceSelector > 0;
  const bool learned = phys && sgs_active();
  if (learned) {
    int rc;
    a.tau = D.tau;
    if ((rc = sgs_infer(in))) return rc;
  }
  if (physics_stage(stage) && surflayerSelector > 0) {
    /* lateral halo storage: the surface pass covers the columns past the high edges too (the
     * ring faces of the lowest level read their stresses); their surface parameters and
     * previous surface state come from the periodic images, filled first */
    const int ext = D.halo ? 2 : 0;
    if (D.halo) halo_fill(D.surf, D.ps, SF_N, 1);
    dim3 cg((D.Nx + ext + 255) / 256, D.Ny + ext);
    launch_timed(0, var.surface, cg, dim3(256), a);
  }
  dim3 grid((D.Nx + TX - 1) / TX, (D.Ny + TY - 1) / TY, D.nseg);
  /* the batch's last stage also emits the SGS stresses and tendencies the host will read */
  const bool emit = a.tau || a.mtau || a.fem;
  /* the microphysics runs every few steps (a.mpActive); the steps between use the physics
   * kernel compiled without it, which has the registers to spare (no spill when moist) */
  stage_fn k = phys ? (emit ? var.phys_emit : (a.mpActive ? var.phys : var.phys_nomp))
                    : (emit ? var.plain_emit : var.plain);
  launch_timed(phys ? 2 : 1, k, grid, dim3(NT), a);
  HIPCHK(hipGetLastError());
  if (learned) return sgs_correct(out, emitF ? 1.f : a.coefdt);
  return FE_OK;
}

/* Work-groups per level of a plane reduction over n4 groups of four cells: about 1024 in all (four
 * per compute unit, which keeps enough loads in flight for the copy rate; one per level left most
 * of the chip idle and ran at the latency of one wave's loads), at least 256 groups each, at most
 * `most`. */
constexpr int STAT_NT = 256;
static int stat_parts(int nlev, long n4, long most) {
  return (int)std::max<long>(1, std::min<long>({(1024 + nlev - 1) / nlev, n4 / STAT_NT, most}));
}

/* Sums each of v[0..N) over the work-group's STAT_NT threads; thread k < N returns its total in v[0]. */
template <int N, typename T>
__device__ __forceinline__ void block_sums(T (&v)[N], T (*part)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off);
  if (threadIdx.x % 64 == 0)
#pragma unroll
    for (int k = 0; k < N; ++k) part[threadIdx.x / 64][k] = v[k];
  __syncthreads();
  if (threadIdx.x < N) {
    T t = part[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < STAT_NT / 64; ++w) t += part[w][threadIdx.x];
    v[0] = t;
  }
}

/* Slab means over the halo-inclusive plane (fecuda_PlugIns.cu:25-45 reduces the
 * halo-inclusive extents and divides by their product), levels -1..Nz; halo values follow the
 * boundary rules of the state (periodic sides: a column counts as often as the halo-inclusive
 * plane holds its images; at the bottom and lid: rho, rho*theta from the base state, rho*u, rho*v
 * zero-gradient below and geostrophic above, q_v zero-gradient).  FP64 sums of work-group
 * (part, level) into part, [part][level][5]; k_lsf_mean adds the parts in order.  Bound by the
 * loads of five fields: 152 x 146 x 122, one work-group per level 113 us, parts 19 us. */
__global__ void __launch_bounds__(STAT_NT) k_lsf_sums(const float *S, long fs, long ps, int Nx, int Ny, int Nz, int P, int Nh,
                                                      int iqv, const float *prof, float uTop, float vTop, long chunk,
                                                      double *out) {
  const int z = (int)blockIdx.x - 1;
  const int g = (Nx + 3) / 4;
  const long n4 = (long)g * Ny, i1 = min(n4, (long)(blockIdx.y + 1) * chunk);
  /* halo-inclusive positions -Nh .. N+Nh-1 that wrap to v */
  auto images = [&](int v, int N) { return (N + Nh - 1 - v) / N + (v + Nh) / N + 1; };
  const int zc = z < 0 ? 0 : (z >= Nz ? Nz - 1 : z);
  const bool in = (z >= 0 && z < Nz);
  const float r0 = prof[(z + 3) * PROW + PR_RHO], t0 = prof[(z + 3) * PROW + PR_RTH];
  double acc[5] = {0, 0, 0, 0, 0};
  for (long i = (long)blockIdx.y * chunk + threadIdx.x; i < i1; i += STAT_NT) {
    const int y = (int)(i / g), x = 4 * (int)(i - (long)y * g);
    const long o = (long)zc * ps + (long)y * P + x;
    const float4 a = *(const float4 *)(S + o), b = *(const float4 *)(S + fs + o), c = *(const float4 *)(S + 2 * fs + o),
                 d = *(const float4 *)(S + 4 * fs + o);
    const float4 q = iqv >= 0 ? *(const float4 *)(S + (long)iqv * fs + o) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float va[4] = {a.x, a.y, a.z, a.w}, vb[4] = {b.x, b.y, b.z, b.w}, vc[4] = {c.x, c.y, c.z, c.w},
                vd[4] = {d.x, d.y, d.z, d.w}, vq[4] = {q.x, q.y, q.z, q.w};
    const double wy = images(y, Ny);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (x + j >= Nx) continue;                     /* the row's padding */
      const double w = wy * images(x + j, Nx);
      acc[0] += w * (in ? va[j] : r0);
      acc[1] += w * (in || z < 0 ? vb[j] : uTop);
      acc[2] += w * (in || z < 0 ? vc[j] : vTop);
      acc[3] += w * (in ? vd[j] : t0);
      acc[4] += w * vq[j];                           /* iqv < 0: no q_v field */
    }
  }
  __shared__ double part[STAT_NT / 64][5];
  block_sums(acc, part);
  if (threadIdx.x < 5) out[((long)blockIdx.y * (Nz + 2) + blockIdx.x) * 5 + threadIdx.x] = acc[0];
}
__global__ void k_lsf_mean(const double *part, int parts, int nlev, double cells, float *M) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;   /* (level, field) */
  if (i >= nlev * 5) return;
  double s = 0.0;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) s += part[(long)p * nlev * 5 + i];
  M[(i % 5) * nlev + i / 5] = (float)(s / cells);
}

struct LsfPar { float p[3][5]; int horMn, moist; float fac; };

__device__ __forceinline__ float lsf_piece(const float *pp, float z, float rho) {
  if (z <= pp[3]) return (pp[0] + ((pp[1] - pp[0]) / pp[3]) * z) * rho;
  if (z <= pp[4]) return (pp[1] + ((pp[2] - pp[1]) / (pp[4] - pp[3])) * (z - pp[3])) * rho;
  return pp[2] * rho;
}

/* Forcing rows per level (cudaDevice_lsfRHS, cuda_largeScaleForcingsDevice.cu:141-250): the
 * density is the base state's, values are per hour times the step factor, and the
 * subsidence term carries the density twice, as the reference writes it. */
__global__ void k_lsf_rows(LsfPar q, const float *prof, const float *M, int Nz, float *R) {
  const int z = blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= Nz) return;
  const float rho = prof[(z + 3) * PROW + PR_RHO], zz = prof[(z + 3) * PROW + PR_Z];
  float *r = R + (long)z * LSF_ROW;
  for (int k = 0; k < LSF_ROW; ++k) r[k] = 0.f;
  r[2] = (float)((double)(lsf_piece(q.p[1], zz, rho) * q.fac) / 3600.0);
  if (q.moist) r[4] = (float)((double)(lsf_piece(q.p[2], zz, rho) * q.fac) / 3600.0);
  if (q.horMn) {
    const float fw = (float)((double)(lsf_piece(q.p[0], zz, rho) * q.fac) / 3600.0);
    const float dz = prof[(z + 4) * PROW + PR_Z] - prof[(z + 2) * PROW + PR_Z];
    const int n = Nz + 2, kp = z + 2, km = z;        /* rows of levels z+1 and z-1 */
    auto sub = [&](int f) { return fw * rho * (M[f * n + kp] / M[kp] - M[f * n + km] / M[km]) / dz; };
    r[0] = -sub(1);
    r[1] = -sub(2);
    r[3] = -sub(3);
    r[5] = -sub(4);
  }
}

/* The forcing enters the last stage's update phi = phi^n + dt (F + F_lsf) through its RK
 * base: phi^n += dt F_lsf before that stage (phi^n is read there by the update only), so the
 * stage kernels carry no forcing code and the positivity clip acts on the total as in
 * cuda_RKschemes.cu:140-157.  The emitted tendencies of such a step leave F_lsf out. */
__global__ void k_lsf_base(float *S, long fs, long ps, int Nx, int Ny, int Nz, int P, int iqv, int moist, float dt,
                           const float *R) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
  if (x >= Nx) return;
  const long o = (long)z * ps + (long)y * P + x;
  const float *r = R + (long)z * LSF_ROW;
  S[fs + o] += dt * r[0];
  S[2 * fs + o] += dt * r[1];
  S[4 * fs + o] += dt * (r[2] + r[3]);
  if (moist) S[(long)iqv * fs + o] += dt * (r[4] + r[5]);
}

/* Large-scale forcing of the step starting at simTime_it: slab means of the step's input
 * when the subsidence terms are on (cuda_timeIntDevice.cu:125-127) and the rows for the
 * last stage when the forcing is due (cuda_hydroCoreDevice.cu:401-406). */
int lsf_prepare() {
  D.lsfNow = false;
  if (lsfSelector != 1) return FE_OK;
  const int itn = (int)roundf(lsf_freq / dt);
  if (!(simTime_it > simTime_itRestart && itn > 0 && simTime_it % itn == 0)) return FE_OK;
  if (lsf_horMnSubTerms == 1) {
    const long n4 = (long)((D.Nx + 3) / 4) * D.Ny;
    const int parts = stat_parts(D.Nz + 2, n4, LONG_MAX);
    hipLaunchKernelGGL(k_lsf_sums, dim3(D.Nz + 2, parts), dim3(STAT_NT), 0, D.stream, D.S[0], D.fs, D.ps, D.Nx, D.Ny, D.Nz, D.P,
                       D.Nh, D.nM > 0 ? 5 + D.nTKE : -1, D.prof, D.uTop, D.vTop, (n4 + parts - 1) / parts, D.lsfP);
    hipLaunchKernelGGL(k_lsf_mean, dim3((5 * (D.Nz + 2) + 63) / 64), dim3(64), 0, D.stream, (const double *)D.lsfP, parts, D.Nz + 2,
                       (double)(D.Nx + 2 * D.Nh) * (double)(D.Ny + 2 * D.Nh), D.lsfM);
    HIPCHK(hipGetLastError());
  }
  if (simTime_it - simTime_itRestart < itn) return FE_OK;
  LsfPar q;
  const float pw[5] = {lsf_w_surf, lsf_w_lev1, lsf_w_lev2, lsf_w_zlev1, lsf_w_zlev2};
  const float pt[5] = {lsf_th_surf, lsf_th_lev1, lsf_th_lev2, lsf_th_zlev1, lsf_th_zlev2};
  const float pq[5] = {lsf_qv_surf, lsf_qv_lev1, lsf_qv_lev2, lsf_qv_zlev1, lsf_qv_zlev2};
  for (int k = 0; k < 5; ++k) { q.p[0][k] = pw[k]; q.p[1][k] = pt[k]; q.p[2][k] = pq[k]; }
  q.horMn = lsf_horMnSubTerms == 1;
  q.moist = D.nM > 0;
  q.fac = (float)itn;
  hipLaunchKernelGGL(k_lsf_rows, dim3((D.Nz + 63) / 64), dim3(64), 0, D.stream, q, D.prof, D.lsfM, D.Nz, D.lsfR);
  HIPCHK(hipGetLastError());
  D.lsfNow = true;
  return FE_OK;
}

int one_step(float *pout_last) {
  int rc;
  if ((rc = lsf_prepare())) return rc;
  if ((rc = launch_stage(0, D.S[0], D.S[0], D.S[1], 0, nullptr))) return rc;
  if ((rc = launch_stage(1, D.S[1], D.S[0], D.S[2], 0, nullptr))) return rc;
  if (D.lsfNow) {
    hipLaunchKernelGGL(k_lsf_base, dim3((D.Nx + 63) / 64, D.Ny, D.Nz), dim3(64), 0, D.stream, D.S[0], D.fs, D.ps, D.Nx,
                       D.Ny, D.Nz, D.P, 5 + D.nTKE, D.nM > 0 ? 1 : 0, dt, D.lsfR);
    HIPCHK(hipGetLastError());
  }
  if ((rc = launch_stage(2, D.S[2], D.S[0], D.S[0], 0, pout_last))) return rc;
  return FE_OK;
}

int upload_field(const float *host, float *dev) {
  int rc;
  if ((rc = xfer_up(D.stream, D.stg, host, D.n3h * sizeof(float)))) return rc;
  dim3 g((D.Nx + TT - 1) / TT, D.Ny, (D.Nz + TT - 1) / TT);
  hipLaunchKernelGGL(k_host_to_dev, g, dim3(256), 0, D.stream, D.stg, dev, D.Nx, D.Ny, D.Nz, D.Nh, D.P, D.ps);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

int download_field(const float *dev, float *host, int rule) {
  dim3 g((D.Nx + 2 * D.Nh + TT - 1) / TT, D.Ny + 2 * D.Nh, (D.Nz + 2 * D.Nh + TT - 1) / TT);
  hipLaunchKernelGGL(k_dev_to_host, g, dim3(256), 0, D.stream, dev, D.stg, D.Nx, D.Ny, D.Nz, D.Nh, D.P, D.ps, rule, D.prof, D.np, D.uTop, D.vTop,
                     (const float *)(D.terrain ? D.tprof : nullptr), D.NyS);
  HIPCHK(hipGetLastError());
  return xfer_down(D.stream, host, D.stg, D.n3h * sizeof(float));
}

int upload_2d(const float *host, float *dev) {
  if (!host) return FE_OK;
  int rc;
  if ((rc = xfer_up(D.stream, D.stg, host, D.n2h * sizeof(float)))) return rc;
  dim3 g((D.Nx + 63) / 64, D.Ny);
  hipLaunchKernelGGL(k_2d_to_dev, g, dim3(64), 0, D.stream, D.stg, dev, D.Nx, D.Ny, D.Nh, D.P);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

int download_2d(const float *dev, float *host) {
  if (!host) return FE_OK;
  dim3 g((D.Ny + 2 * D.Nh + 63) / 64, D.Nx + 2 * D.Nh);
  hipLaunchKernelGGL(k_2d_to_host, g, dim3(64), 0, D.stream, dev, D.stg, D.Nx, D.Ny, D.Nh, D.P);
  HIPCHK(hipGetLastError());
  return xfer_down(D.stream, host, D.stg, D.n2h * sizeof(float));
}

float *field_ptr(float *S, int f) { return S + (long)f * D.fs; }

int upload_state(void) {
  int rc;
  const long n3 = D.n3h;
  if ((rc = xfer_reserve(n3 * sizeof(float)))) return rc;
  XferScope scope;
  for (int f = 0; f < 5; ++f)
    if ((rc = upload_field(hydroFlds + f * n3, field_ptr(D.S[0], f)))) return rc;
  for (int f = 0; f < D.nTKE; ++f)
    if ((rc = upload_field(sgstkeScalars + f * n3, field_ptr(D.S[0], 5 + f)))) return rc;
  for (int f = 0; f < D.nM; ++f)
    if ((rc = upload_field(moistScalars + f * n3, field_ptr(D.S[0], 5 + D.nTKE + f)))) return rc;
  if (surflayerSelector > 0) {
    if ((rc = upload_2d(tskin, surfp(SF_TSK)))) return rc;
    if ((rc = upload_2d(fricVel, surfp(SF_UST)))) return rc;
    if ((rc = upload_2d(htFlux, surfp(SF_HF)))) return rc;
    if ((rc = upload_2d(z0m, surfp(SF_Z0M)))) return rc;
    if ((rc = upload_2d(z0t, surfp(SF_Z0T)))) return rc;
    if (moistureSelector > 0) {
      if ((rc = upload_2d(qskin, surfp(SF_QSK)))) return rc;
      if ((rc = upload_2d(qFlux, surfp(SF_QF)))) return rc;
    }
  }
  return xfer_finish(D.stream);
}

int download_state(int with_pres) {
  int rc;
  const long n3 = D.n3h;
  if ((rc = xfer_reserve(n3 * sizeof(float)))) return rc;
  XferScope scope;
  for (int f = 0; f < 5; ++f)
    if ((rc = download_field(field_ptr(D.S[0], f), hydroFlds + f * n3, f))) return rc;
  for (int f = 0; f < D.nTKE; ++f)
    if ((rc = download_field(field_ptr(D.S[0], 5 + f), sgstkeScalars + f * n3, 5))) return rc;
  for (int f = 0; f < D.nM; ++f)
    if ((rc = download_field(field_ptr(D.S[0], 5 + D.nTKE + f), moistScalars + f * n3, 6))) return rc;
  if (with_pres && hydroPres)
    if ((rc = download_field(D.pout, hydroPres, 7))) return rc;
  /* batch-end emissions (cuda_timeIntDevice.cu:210-247): tendencies with zero halos,
   * SGS stresses and moisture fluxes with periodic and zero-gradient halos */
  if (with_pres && D.fem) {
    for (int f = 0; f < 5; ++f)
      if ((rc = download_field(D.fem + (long)f * D.fs, hydroFldsFrhs + f * n3, 8))) return rc;
    for (int f = 0; f < D.nTKE; ++f)
      if ((rc = download_field(D.fem + (long)(5 + f) * D.fs, sgstkeScalarsFrhs + f * n3, 8))) return rc;
    for (int f = 0; f < D.nM; ++f)
      if ((rc = download_field(D.fem + (long)(5 + D.nTKE + f) * D.fs, moistScalarsFrhs + f * n3, 8))) return rc;
  }
  if (with_pres && D.tau)
    for (int f = 0; f < 9; ++f)
      if ((rc = download_field(D.tau + (long)f * D.fs, hydroTauFlds + f * n3, 6))) return rc;
  if (with_pres && D.mtau)
    for (int f = 0; f < 3 * D.nM; ++f)
      if ((rc = download_field(D.mtau + (long)f * D.fs, moistTauFlds + f * n3, 6))) return rc;
  if (surflayerSelector > 0) {
    if ((rc = download_2d(surfp(SF_UST), fricVel))) return rc;
    if ((rc = download_2d(surfp(SF_HF), htFlux))) return rc;
    if ((rc = download_2d(surfp(SF_TSK), tskin))) return rc;
    if ((rc = download_2d(surfp(SF_IOL), invOblen))) return rc;
    if ((rc = download_2d(surfp(SF_Z0M), z0m))) return rc;
    if ((rc = download_2d(surfp(SF_Z0T), z0t))) return rc;
    if ((rc = download_2d(surfp(SF_CD), cdFld))) return rc;
    if ((rc = download_2d(surfp(SF_CH), chFld))) return rc;
    if (moistureSelector > 0) {
      if ((rc = download_2d(surfp(SF_CQ), cqFld))) return rc;
      if ((rc = download_2d(surfp(SF_QF), qFlux))) return rc;
      if ((rc = download_2d(surfp(SF_QSK), qskin))) return rc;
    }
  }
  return xfer_finish(D.stream);
}

long idx3(int i, int j, int k) { return ((long)i * (Nyp + 2 * Nh) + j) * (Nzp + 2 * Nh) + k; }

}  // namespace

/* =========================================================================== */
extern "C" {

/* device address of the no-allocation scratch array on the current device (fe_profiles_noalloc) */
static int scratch_lookup();

int fecuda_Init(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
    fprintf(stderr, "fecuda_Init: no HIP device found\n");
    return FE_ERR_NO_DEVICE;
  }
  if (numProcsX * numProcsY != 1) return FE_ERR_RANKS;
  HIPCHK(hipSetDevice(mpi_rank_world % n));
  {
    int rc = scratch_lookup();
    if (rc) return rc;
  }
  if (!D.stream) HIPCHK(hipStreamCreateWithFlags(&D.stream, hipStreamNonBlocking));
  D.tb[0] = tBx; D.tb[1] = tBy; D.tb[2] = tBz;
  D.fecuda = 1;
  return FE_OK;
}

int fecuda_Cleanup(void) {
  /* the pinned slots go with the model, unless an ensemble is being put together from models */
  if (fe_ens_count() == 0) xfer_release();
  if (D.stream) { (void)hipStreamDestroy(D.stream); D.stream = nullptr; }
  D.fecuda = 0;
  return FE_OK;
}

int fecuda_SetBlocksPerGrid(int Nx_, int Ny_, int Nz_) {
  /* recorded for reporting; the tile shape of the fused kernels is fixed at 64x8 columns */
  D.gridBlocks[0] = Nx_; D.gridBlocks[1] = Ny_; D.gridBlocks[2] = Nz_;
  return FE_OK;
}

int fecuda_AllocateHaloBuffers(int, int, int, int) { return FE_OK; }
int fecuda_DeallocateHaloBuffers(void) { return FE_OK; }

/* cuda_gridInit: metric profiles.  J31 = J32 = 0 everywhere (the reference's cofactors vanish on
 * its terrain-following grids, grid.c:634-636).  A flat grid (zPos, J33, D_Jac horizontally
 * uniform) uses one level table; a terrain-following grid a table per column, and its lateral
 * halo columns must hold their periodic images' coordinates and metrics: the host gives a halo
 * column the nearest interior column's (grid.c:480-540, 665-741) while the state there is the
 * periodic image's, and the two agree only for terrain that is periodic at the lateral
 * boundaries (e.g. flat within Nh cells of every edge) -- other terrain is refused. */
int cuda_gridInit(void) {
  if (!D.fecuda) return FE_ERR_STATE;
  D.Nx = Nxp; D.Ny = Nyp; D.Nz = Nzp; D.Nh = Nh;
  /* lateral halo storage (amd_haloBuffer = 1): the grid is one block of a larger x-y
   * decomposition; each plane is padded to P >= Nx + 6 columns and Ny + 6 rows, the 3-cell
   * lateral halo of the block lives in the padding (positions -3..-1 in the last three columns
   * and rows, Nx..Nx+2 and Ny..Ny+2 after the block), and the stage kernels read it there
   * instead of wrapping.  Here a fill kernel copies the block's own periodic images into it
   * before every stage (the exchange with the neighbouring blocks in a decomposed run).  The
   * block holds whole 64 x 8 tiles. */
  D.halo = amd_haloBuffer ? 1 : 0;
  if (D.halo && Nh < HH) {
    fprintf(stderr, "cuda_gridInit: lateral halo storage needs Nh >= %d (Nh = %d)\n", HH, Nh);
    return FE_ERR_UNSUPPORTED;
  }
  if (D.halo && (Nxp % TX || Nyp % TY)) {
    fprintf(stderr, "cuda_gridInit: lateral halo storage needs Nx a multiple of %d and Ny of %d (%d x %d)\n", TX, TY, Nxp,
            Nyp);
    return FE_ERR_UNSUPPORTED;
  }
  D.P = D.halo ? (Nxp + 2 * HH + 31) / 32 * 32 : (Nxp + 31) / 32 * 32;
  D.NyS = D.halo ? Nyp + 2 * HH : Nyp;
  D.ps = (long)D.NyS * D.P;
  D.fs = D.ps * D.Nz;
  D.np = Nzp + 10;
  /* the kernels address within one field with 32-bit byte offsets */
  if (D.Nz * D.ps * (long)sizeof(float) > 0xFFFFFFFFL) {
    fprintf(stderr, "cuda_gridInit: %d x %d x %d exceeds 4 GiB per field\n", Nxp, Nyp, Nzp);
    return FE_ERR_UNSUPPORTED;
  }
  D.n3h = (long)(Nxp + 2 * Nh) * (Nyp + 2 * Nh) * (Nzp + 2 * Nh);
  D.n2h = (long)(Nxp + 2 * Nh) * (Nyp + 2 * Nh);
  const int i0 = iMin, j0 = jMin;
  bool flat = true;
  for (int i = iMin - Nh; i < iMax + Nh; ++i)
    for (int j = jMin - Nh; j < jMax + Nh; ++j)
      for (int k = 0; k < Nzp + 2 * Nh; ++k) {
        long n = idx3(i, j, k), r = idx3(i0, j0, k);
        if (J31[n] != 0.f || J32[n] != 0.f) {
          fprintf(stderr, "cuda_gridInit: J31/J32 != 0 (a non-terrain-following transform) is not supported\n");
          return FE_ERR_TERRAIN;
        }
        if (J33[n] != J33[r] || D_Jac[n] != D_Jac[r] || zPos[n] != zPos[r]) flat = false;
      }
  auto wrapc = [](int i, int lo, int n) { return lo + ((i - lo) % n + n) % n; };
  /* With lateral halo storage the per-column table holds the halo columns' own metrics (the
   * host's, as the reference reads them); the wrapped layout reads a halo column's metrics at
   * its periodic image and so needs the two to agree. */
  D.terrain_np = 0;
  if (!flat) {
    for (int i = iMin - Nh; i < iMax + Nh && !D.terrain_np; ++i)
      for (int j = jMin - Nh; j < jMax + Nh; ++j) {
        if (i >= iMin && i < iMax && j >= jMin && j < jMax) continue;
        const int iw = wrapc(i, iMin, Nxp), jw = wrapc(j, jMin, Nyp);
        for (int k = 0; k < Nzp + 2 * Nh; ++k) {
          long n = idx3(i, j, k), w = idx3(iw, jw, k);
          if (zPos[n] != zPos[w] || J33[n] != J33[w] || D_Jac[n] != D_Jac[w] || invD_Jac[n] != invD_Jac[w]) {
            if (D.halo) {
              D.terrain_np = 1;
              break;
            }
            fprintf(stderr, "cuda_gridInit: terrain not periodic at the lateral boundaries (halo column %d,%d differs "
                    "from its periodic image); make the topography flat within %d cells of every edge, or run with "
                    "lateral halo storage (amd_haloBuffer = 1)\n", i - Nh, j - Nh, Nh);
            return FE_ERR_TERRAIN;
          }
        }
      }
  }
  D.terrain = flat ? 0 : 1;
  auto metric_rows = [&](float *base, size_t stride, int i, int j) {
    for (int z = -3; z < D.Nz + 7; ++z) {
      int k = z + Nh;
      int kc = k < 0 ? 0 : (k >= Nzp + 2 * Nh ? Nzp + 2 * Nh - 1 : k);
      long r = idx3(i, j, kc);
      float *q = base + (size_t)(z + 3) * stride;
      q[(size_t)PR_Z * stride * D.np] = zPos[r];
      q[(size_t)PR_J33 * stride * D.np] = J33[r];
      q[(size_t)PR_D * stride * D.np] = D_Jac[r];
      q[(size_t)PR_INVD * stride * D.np] = invD_Jac[r];
      q[(size_t)PR_DELTA * stride * D.np] = powf(dX * dY * dZ * D_Jac[r], (float)(1.0 / 3.0));
    }
  };
  D.htprof.clear();
  if (D.terrain) {
    D.htprof.assign((size_t)PROW * D.np * D.ps, 0.f);
    const int hh = D.halo ? HH : 0;      /* lateral halo storage: the halo columns' rows too */
    for (int y = -hh; y < D.Ny + hh; ++y)
      for (int x = -hh; x < D.Nx + hh; ++x)
        metric_rows(D.htprof.data() + padded_col(x, y), (size_t)D.ps, x + iMin, y + jMin);
  }
  D.hprof.assign((size_t)PROW * D.np, 0.f);
  auto P = [&](int row, int z) -> float & { return D.hprof[(size_t)(z + 3) * PROW + row]; };
  for (int z = -3; z < D.Nz + 7; ++z) {
    int k = z + Nh;
    int kc = k < 0 ? 0 : (k >= Nzp + 2 * Nh ? Nzp + 2 * Nh - 1 : k);
    long r = idx3(i0, j0, kc);
    P(PR_Z, z) = zPos[r];
    P(PR_J33, z) = J33[r];
    P(PR_D, z) = D_Jac[r];
    P(PR_INVD, z) = invD_Jac[r];
    P(PR_DELTA, z) = powf(dX * dY * dZ * D_Jac[r], (float)(1.0 / 3.0));
  }
  if (D.prof) (void)hipFree(D.prof);
  HIPCHK(hipMalloc(&D.prof, D.hprof.size() * sizeof(float)));
  HIPCHK(hipMemcpy(D.prof, D.hprof.data(), D.hprof.size() * sizeof(float), hipMemcpyHostToDevice));
  D.grid = 1;
  return FE_OK;
}

int cuda_gridCleanup(void) {
  if (D.prof) { (void)hipFree(D.prof); D.prof = nullptr; }
  D.grid = 0;
  return FE_OK;
}

/* cuda_hydroCoreInit: base-state and forcing profiles, device fields. */
int cuda_hydroCoreInit(void) {
  if (!D.grid) return FE_ERR_STATE;
  if (select_variant() != FE_OK) {
    fprintf(stderr, "cuda_hydroCoreInit: unsupported selector combination (advection %d, TKE adv %d, turbulence %d/%d, moisture %d/%d)\n",
            advectionSelector, TKEAdvSelector, turbulenceSelector, TKESelector, moistureSelector, moistureNvars);
    return FE_ERR_UNSUPPORTED;
  }
  if (hydroBCs != 2) return FE_ERR_UNSUPPORTED;
  if (D.terrain_np && moistureSelector > 0) {
    /* the moisture SGS fluxes at the lateral seam of such terrain differ from the reference's
     * by more than FP32 rounding; the dry closures match it */
    fprintf(stderr, "cuda_hydroCoreInit: terrain that is not periodic at the lateral boundaries runs the dry closures only\n");
    return FE_ERR_UNSUPPORTED;
  }
  D.nTKE = (turbulenceSelector > 0 && TKESelector > 0) ? 1 : 0;
  D.nM = moistureSelector > 0 ? moistureNvars : 0;
  D.NF = 5 + D.nTKE + D.nM;
  /* the subsidence terms average and force q_v (cuda_largeScaleForcingsDevice.cu:100-252) */
  if (lsfSelector == 1 && lsf_horMnSubTerms == 1 && D.nM == 0) {
    fprintf(stderr, "cuda_hydroCoreInit: lsf_horMnSubTerms = 1 needs moisture (q_v)\n");
    return FE_ERR_UNSUPPORTED;
  }
  choose_segments();
  /* the stage kernels address all fields of a state array through one buffer
   * resource with 32-bit offsets */
  if ((long)D.NF * D.fs * (long)sizeof(float) > 0xFFFFFFFFL) {
    fprintf(stderr, "cuda_hydroCoreInit: %d fields of %d x %d x %d exceed 4 GiB per state array\n", D.NF, D.Nx, D.Ny,
            D.Nz);
    return FE_ERR_UNSUPPORTED;
  }
  const long fsH = D.n3h;
  const float *rbs = hydroBaseStateFlds, *tbs = hydroBaseStateFlds + fsH;
  const int i0 = iMin, j0 = jMin;
  if (!D.terrain) {
    for (int i = iMin - Nh; i < iMax + Nh; ++i)
      for (int j = jMin - Nh; j < jMax + Nh; ++j)
        for (int k = 0; k < Nzp + 2 * Nh; ++k) {
          long n = idx3(i, j, k), r = idx3(i0, j0, k);
          if (rbs[n] != rbs[r] || tbs[n] != tbs[r]) {
            fprintf(stderr, "cuda_hydroCoreInit: base state must be horizontally uniform on a flat grid\n");
            return FE_ERR_TERRAIN;
          }
        }
  } else {
    if (lsfSelector == 1) {
      fprintf(stderr, "cuda_hydroCoreInit: large-scale forcing (slab means) is not supported on terrain-following grids\n");
      return FE_ERR_UNSUPPORTED;
    }
    /* the halo columns' base state must be their periodic images' (see cuda_gridInit), unless
     * the table holds the halo columns' own (lateral halo storage) */
    auto wrapc = [](int i, int lo, int n) { return lo + ((i - lo) % n + n) % n; };
    for (int i = iMin - Nh; i < iMax + Nh && !D.halo; ++i)
      for (int j = jMin - Nh; j < jMax + Nh; ++j) {
        if (i >= iMin && i < iMax && j >= jMin && j < jMax) continue;
        const long iw = wrapc(i, iMin, Nxp), jw = wrapc(j, jMin, Nyp);
        for (int k = 0; k < Nzp + 2 * Nh; ++k) {
          long n = idx3(i, j, k), w = idx3((int)iw, (int)jw, k);
          if (rbs[n] != rbs[w] || tbs[n] != tbs[w] || hydroBaseStatePres[n] != hydroBaseStatePres[w]) {
            fprintf(stderr, "cuda_hydroCoreInit: base state not periodic at the lateral boundaries\n");
            return FE_ERR_TERRAIN;
          }
        }
      }
  }
  const float c1 = R_gas / powf(refPressure, R_cp);
  const float pio2 = (float)(0.5 * acos(-1.0));
  /* base-state, forcing and damping rows of the column (i, j) through the accessor P(row, z);
   * the damping layer hangs from the column's own top cell, the top-halo momentum is the
   * column's geostrophic base state there (cuda_BCsDevice.cu:183-211) */
  auto bs_rows = [&](auto &&P, int i, int j) {
    const long rtop = idx3(i, j, kMax - 1);
    const float ztop = zPos[rtop];
    for (int z = -3; z < D.Nz + 7; ++z) {
      int k = z + Nh;
      int kc = k < 0 ? 0 : (k >= Nzp + 2 * Nh ? Nzp + 2 * Nh - 1 : k);
      long r = idx3(i, j, kc);
      P(PR_RHO, z) = rbs[r];
      P(PR_RTH, z) = tbs[r];
      P(PR_IRTH, z) = 1.0f / tbs[r];
      P(PR_PBS, z) = hydroBaseStatePres[r];
      P(PR_PBSRAW, z) = powf(tbs[r] * c1, cp_cv);
      P(PR_EXB, z) = powf(P(PR_PBSRAW, z) / refPressure, R_cp);
      float zz = zPos[r];
      float ubs = (zz < z_Ug) ? U_g * rbs[r] : (U_g + Ug_grad * (zz - z_Ug)) * rbs[r];
      float vbs = (zz < z_Vg) ? V_g * rbs[r] : (V_g + Vg_grad * (zz - z_Vg)) * rbs[r];
      P(PR_UG, z) = corioLS_fact * ubs / rbs[r];
      P(PR_VG, z) = corioLS_fact * vbs / rbs[r];
      float dmp = 0.f;
      if (dampingLayerSelector > 0 && zz >= ztop - dampingLayerDepth) {
        float s = sinf((float)(pio2 * (1.0 - (ztop - zz) / dampingLayerDepth)));
        dmp = (float)(0.2 * pow((double)s, 2));
      }
      P(PR_DAMP, z) = dmp;
    }
    const float zt = zPos[rtop], rt = rbs[rtop];
    const float ut = (zt < z_Ug) ? U_g * rt : (U_g + Ug_grad * (zt - z_Ug)) * rt;
    const float vt = (zt < z_Vg) ? V_g * rt : (V_g + Vg_grad * (zt - z_Vg)) * rt;
    for (int z = -3; z < D.Nz + 7; ++z) {
      P(PR_UTOP, z) = ut;
      P(PR_VTOP, z) = vt;
    }
  };
  bs_rows([&](int row, int z) -> float & { return D.hprof[(size_t)(z + 3) * PROW + row]; }, i0, j0);
  D.uTop = D.hprof[(size_t)3 * PROW + PR_UTOP];
  D.vTop = D.hprof[(size_t)3 * PROW + PR_VTOP];
  if (D.terrain) {
    const int hh = D.halo ? HH : 0;      /* lateral halo storage: the halo columns' rows too */
    for (int y = -hh; y < D.Ny + hh; ++y)
      for (int x = -hh; x < D.Nx + hh; ++x) {
        const size_t col = padded_col(x, y);
        bs_rows([&](int row, int z) -> float & { return D.htprof[((size_t)row * D.np + (z + 3)) * D.ps + col]; }, x + iMin,
                y + jMin);
      }
    if (D.tprof) (void)hipFree(D.tprof);
    D.tprof = nullptr;
    HIPCHK(hipMalloc(&D.tprof, D.htprof.size() * sizeof(float)));
    HIPCHK(hipMemcpy(D.tprof, D.htprof.data(), D.htprof.size() * sizeof(float), hipMemcpyHostToDevice));
  }
  HIPCHK(hipMemcpy(D.prof, D.hprof.data(), D.hprof.size() * sizeof(float), hipMemcpyHostToDevice));
  for (int s = 0; s < 3; ++s) {
    if (D.S[s]) (void)hipFree(D.S[s]);
    HIPCHK(hipMalloc(&D.S[s], (size_t)D.NF * D.fs * sizeof(float)));
    HIPCHK(hipMemset(D.S[s], 0, (size_t)D.NF * D.fs * sizeof(float)));
  }
  HIPCHK(hipMalloc(&D.pout, (size_t)D.fs * sizeof(float)));
  HIPCHK(hipMemset(D.pout, 0, (size_t)D.fs * sizeof(float)));
  if (hydroSubGridWrite == 1 && turbulenceSelector > 0 && hydroTauFlds) {
    HIPCHK(hipMalloc(&D.tau, (size_t)9 * D.fs * sizeof(float)));
    HIPCHK(hipMemset(D.tau, 0, (size_t)9 * D.fs * sizeof(float)));
  }
  if (hydroSubGridWrite == 1 && moistureSGSturb == 1 && D.nM > 0 && moistTauFlds) {
    HIPCHK(hipMalloc(&D.mtau, (size_t)3 * D.nM * D.fs * sizeof(float)));
    HIPCHK(hipMemset(D.mtau, 0, (size_t)3 * D.nM * D.fs * sizeof(float)));
  }
  if (hydroForcingWrite == 1 || hydroForcingLog == 1) {
    HIPCHK(hipMalloc(&D.fem, (size_t)D.NF * D.fs * sizeof(float)));
    HIPCHK(hipMemset(D.fem, 0, (size_t)D.NF * D.fs * sizeof(float)));
  }
  HIPCHK(hipMalloc(&D.surf, (size_t)SF_N * D.ps * sizeof(float)));
  HIPCHK(hipMemset(D.surf, 0, (size_t)SF_N * D.ps * sizeof(float)));
  HIPCHK(hipMalloc(&D.stg, (size_t)D.n3h * sizeof(float)));
  if (lsfSelector == 1) {
    HIPCHK(hipMalloc(&D.lsfM, (size_t)5 * (D.Nz + 2) * sizeof(float)));
    HIPCHK(hipMemset(D.lsfM, 0, (size_t)5 * (D.Nz + 2) * sizeof(float)));
    HIPCHK(hipMalloc(&D.lsfP, (size_t)stat_parts(D.Nz + 2, (long)((D.Nx + 3) / 4) * D.Ny, LONG_MAX) * (D.Nz + 2) * 5 * sizeof(double)));
    HIPCHK(hipMalloc(&D.lsfR, (size_t)LSF_ROW * D.Nz * sizeof(float)));
    HIPCHK(hipMemset(D.lsfR, 0, (size_t)LSF_ROW * D.Nz * sizeof(float)));
  }
  D.hydro = 1;
  return FE_OK;
}

int cuda_hydroCoreCleanup(void) {
  for (int s = 0; s < 3; ++s) if (D.S[s]) { (void)hipFree(D.S[s]); D.S[s] = nullptr; }
  float **p[] = {&D.pout, &D.tau, &D.mtau, &D.fem, &D.surf, &D.stg, &D.lsfM, &D.lsfR, &D.tprof};
  for (auto q : p) if (*q) { (void)hipFree(*q); *q = nullptr; }
  double **pd[] = {&D.lsfP, &D.stat};
  for (auto q : pd) if (*q) { (void)hipFree(*q); *q = nullptr; }
  D.stat_n = 0;
  D.hydro = 0;
  return FE_OK;
}

int cuda_timeIntInit(void) {
  if (!D.hydro) return FE_ERR_STATE;
  if (timeMethod != 0) return FE_ERR_UNSUPPORTED;
  int rc = upload_state();
  if (rc) return rc;
  D.timeint = 1;
  return FE_OK;
}

int cuda_timeIntCommence(int it) {
  if (!D.timeint) return FE_ERR_STATE;
  int rc;
  if (it == simTime_itRestart)
    if ((rc = upload_state())) return rc;
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  HIPCHK(hipEventRecord(e0, D.stream));
  for (int s = 0; s < NtBatch; ++s) {
    if ((rc = one_step(s == NtBatch - 1 ? D.pout : nullptr))) return rc;
    simTime = simTime + dt;
    simTime_it = simTime_it + 1;
  }
  HIPCHK(hipEventRecord(e1, D.stream));
  HIPCHK(hipEventSynchronize(e1));
  float ms = 0.f;
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  D.ms_per_step = ms / NtBatch;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return download_state(1);
}

int cuda_timeIntCleanup(void) {
  D.timeint = 0;
  return FE_OK;
}

int fe_upload_state(void) { return D.hydro ? upload_state() : FE_ERR_STATE; }
int fe_download_state(void) { return D.hydro ? download_state(0) : FE_ERR_STATE; }
float fe_last_ms_per_step(void) { return D.ms_per_step; }
const char *fe_kernel_info(void) {
  static char buf[224];
  if (!g_var_ok) return "none";
  int n = D.nseg > 1 ? snprintf(buf, sizeof(buf), "%s, %d z-segments of %d levels", g_var.name, D.nseg, D.zseg)
                     : snprintf(buf, sizeof(buf), "%s", g_var.name);
  if (D.halo && n > 0 && n < (int)sizeof(buf))
    snprintf(buf + n, sizeof(buf) - n, ", lateral halo storage (%d x %d planes)", D.P, D.NyS);
  return buf;
}

int fe_device_steps(int nsteps) {
  if (!D.timeint) return FE_ERR_STATE;
  int rc;
  for (int s = 0; s < nsteps; ++s) {
    if ((rc = one_step(nullptr))) return rc;
    simTime = simTime + dt;
    simTime_it = simTime_it + 1;
  }
  HIPCHK(hipStreamSynchronize(D.stream));
  return FE_OK;
}

/* Per-kernel timing: enable with a pool for npairs launches; read the summed
 * milliseconds and launch counts per kernel class after a synchronising call. */
int fe_timing_enable(int npairs) {
  for (auto e : D.ev) (void)hipEventDestroy(e);
  D.ev.clear();
  D.evcls.clear();
  D.evn = 0;
  D.timing = npairs > 0;
  if (!D.timing) return FE_OK;
  D.ev.resize((size_t)2 * npairs);
  D.evcls.assign((size_t)npairs, -1);
  for (auto &e : D.ev) HIPCHK(hipEventCreate(&e));
  return FE_OK;
}

int fe_timing_read(double *ms, int *count, int ncls) {
  for (int c = 0; c < ncls; ++c) { ms[c] = 0; count[c] = 0; }
  HIPCHK(hipStreamSynchronize(D.stream));
  for (size_t i = 0; i + 1 < D.evn; i += 2) {
    float t = 0.f;
    HIPCHK(hipEventElapsedTime(&t, D.ev[i], D.ev[i + 1]));
    int c = D.evcls[i / 2];
    if (c >= 0 && c < ncls) { ms[c] += t; count[c] += 1; }
  }
  D.evn = 0;
  return FE_OK;
}

__global__ void k_copy_probe(const float4 *__restrict__ a, float4 *__restrict__ b, long n4) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long stride = (long)gridDim.x * blockDim.x;
  for (; i < n4; i += stride) b[i] = a[i];
}

/* Streaming copy of nfloats floats, reps times, timed with HIP events; returns GB/s
 * (read + write bytes).  Used to calibrate the HBM byte counters and to report the
 * box's measured copy bandwidth. */
double fe_copy_probe(long nfloats, int reps) {
  nfloats = (nfloats + 3) / 4 * 4;
  if (nfloats <= 0 || reps <= 0) return -1;
  if (D.probe_n < nfloats) {
    if (D.probe) (void)hipFree(D.probe);
    D.probe = nullptr;
    D.probe_n = 0;
    if (hipMalloc(&D.probe, (size_t)2 * nfloats * sizeof(float)) != hipSuccess) return -1;
    if (hipMemset(D.probe, 0, (size_t)2 * nfloats * sizeof(float)) != hipSuccess) return -1;
    D.probe_n = nfloats;
  }
  if (!D.stream && hipStreamCreateWithFlags(&D.stream, hipStreamNonBlocking) != hipSuccess) return -1;
  const long n4 = nfloats / 4;
  const float4 *a = (const float4 *)D.probe;
  float4 *b = (float4 *)(D.probe + nfloats);
  int blocks = 256 * 8;
  hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, D.stream, a, b, n4);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return -1;
  if (hipEventCreate(&e1) != hipSuccess) { (void)hipEventDestroy(e0); return -1; }
  float ms = 0.f;
  bool ok = hipEventRecord(e0, D.stream) == hipSuccess;
  for (int r = 0; r < reps && ok; ++r) hipLaunchKernelGGL(k_copy_probe, dim3(blocks), dim3(256), 0, D.stream, a, b, n4);
  ok = ok && hipGetLastError() == hipSuccess && hipEventRecord(e1, D.stream) == hipSuccess &&
       hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess && ms > 0.f;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (!ok) return -1;
  return (double)2 * nfloats * sizeof(float) * reps / (ms * 1e-3) / 1e9;
}

/* Horizontal-mean profile statistics of the device state in FP64, the on-device
 * counterpart of the reference's post-processing of an output state
 * (tutorials/notebooks/fetutorialfunctions.py:55-83,344-431).  The work-groups of a
 * level accumulate the sums of u, v, w, theta (rho-weighted fields over
 * rho), their products, and the SGS TKE and moisture per unit mass over their
 * part of its cells, four cells per thread and load; each
 * wavefront reduces its lanes with cross-lane shuffles, the wavefronts'
 * partial sums meet in LDS, and k_profiles_final adds a level's parts in order.
 * 256 x 256 x 96, eight fields (201 MB): one work-group per level 324 us, parts 52 us.
 * Output columns, per level:
 *   0 <u> 1 <v> 2 <w> 3 <theta> 4 <u'u'> 5 <u'w'> 6 <v'v'> 7 <v'w'> 8 <w'w'>
 *   9 resolved TKE 10 <theta'w'> 11 <e> 12 <q_v> 13 <q_l>
 *   14 (<tau13>^2 + <tau23>^2)^1/2, 15 <tau33>, 16 <tau_theta3> (level means of the SGS
 *   stresses emitted by the last batch; moved to cell centres on the host)
 * (covariances from FP64 first and second moments). */
constexpr int PROF_NSTAT = 17, PROF_NSUM = 17;
__global__ void __launch_bounds__(STAT_NT) k_profiles(const float *S, long fs, long ps, int Nx, int Ny, int P, int nTKE,
                                                      int nM, const float *tau, long chunk, double *out) {
  const int z = blockIdx.x, g = (Nx + 3) / 4;
  const long n4 = (long)g * Ny, i1 = min(n4, (long)(blockIdx.y + 1) * chunk);
  double acc[PROF_NSUM];
#pragma unroll
  for (int k = 0; k < PROF_NSUM; ++k) acc[k] = 0.0;
  for (long i = (long)blockIdx.y * chunk + threadIdx.x; i < i1; i += STAT_NT) {
    const int y = (int)(i / g), x = 4 * (int)(i - (long)y * g);
    const long o = (long)z * ps + (long)y * P + x;
    /* rows are padded to whole 128-byte lines, so the last group of a row stays inside its row */
    auto ld = [&](const float *p, float (&v)[4]) {
      const float4 t = *(const float4 *)(p + o);
      v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    };
    float r[4], a[4], b[4], c[4], d[4], e[4] = {0.f, 0.f, 0.f, 0.f}, q[4] = {0.f, 0.f, 0.f, 0.f}, l[4] = {0.f, 0.f, 0.f, 0.f};
    float t1[4] = {0.f, 0.f, 0.f, 0.f}, t2[4] = {0.f, 0.f, 0.f, 0.f}, t3[4] = {0.f, 0.f, 0.f, 0.f}, t4[4] = {0.f, 0.f, 0.f, 0.f};
    ld(S, r); ld(S + fs, a); ld(S + 2 * fs, b); ld(S + 3 * fs, c); ld(S + 4 * fs, d);
    if (nTKE > 0) ld(S + 5 * fs, e);
    if (nM > 0) ld(S + (long)(5 + nTKE) * fs, q);
    if (nM > 1) ld(S + (long)(6 + nTKE) * fs, l);
    if (tau) { ld(tau + 2 * fs, t1); ld(tau + 3 * fs, t2); ld(tau + 5 * fs, t3); ld(tau + 8 * fs, t4); }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (x + j >= Nx) continue;
      const double rho = r[j];
      const double u = a[j] / rho, v = b[j] / rho, w = c[j] / rho, th = d[j] / rho;
      acc[0] += u; acc[1] += v; acc[2] += w; acc[3] += th;
      acc[4] += u * u; acc[5] += u * w; acc[6] += v * v; acc[7] += v * w; acc[8] += w * w; acc[9] += th * w;
      if (nTKE > 0) acc[10] += e[j] / rho;
      if (nM > 0) acc[11] += q[j] / rho;
      if (nM > 1) acc[12] += l[j] / rho;
      if (tau) { acc[13] += t1[j]; acc[14] += t2[j]; acc[15] += t3[j]; acc[16] += t4[j]; }
    }
  }
  __shared__ double part[STAT_NT / 64][PROF_NSUM];
  block_sums(acc, part);
  if (threadIdx.x < PROF_NSUM) out[((long)blockIdx.y * gridDim.x + z) * PROF_NSTAT + threadIdx.x] = acc[0];
}
/* Level z's sums over its parts, then its profile row, in place of part 0's row. */
__global__ void __launch_bounds__(64) k_profiles_final(double *out, int parts, int nlev, double n) {
  const int z = blockIdx.x, k = threadIdx.x;
  __shared__ double s[PROF_NSUM];
  if (k < PROF_NSUM) {
    double t = 0.0;
    for (int p = 0; p < parts; ++p) t += out[((long)p * nlev + z) * PROF_NSTAT + k];
    s[k] = t / n;
  }
  __syncthreads();
  if (k == 0) {
    double *r = out + (long)z * PROF_NSTAT;
    r[0] = s[0]; r[1] = s[1]; r[2] = s[2]; r[3] = s[3];
    r[4] = s[4] - s[0] * s[0];
    r[5] = s[5] - s[0] * s[2];
    r[6] = s[6] - s[1] * s[1];
    r[7] = s[7] - s[1] * s[2];
    r[8] = s[8] - s[2] * s[2];
    r[9] = 0.5 * (r[4] + r[6] + r[8]);
    r[10] = s[9] - s[3] * s[2];
    r[11] = s[10]; r[12] = s[11]; r[13] = s[12];
    r[14] = sqrt(s[13] * s[13] + s[14] * s[14]);
    r[15] = s[15];
    r[16] = s[16];
  }
}

/* The no-allocation variant's partial results: per-level profile rows of at most
 * FE_NOALLOC_MAX_LEVELS levels, in a file-scope device array (each GPU the library runs
 * on holds its own copy until the process ends).  Host code never names the array in a
 * kernel argument or copy: its device address, per device, comes from
 * hipGetSymbolAddress at set-up (fecuda_Init, or the entry point's first call on a
 * device). */
constexpr int FE_NOALLOC_MAX_LEVELS = 2048;
static __device__ __align__(256) double scratch[FE_NOALLOC_MAX_LEVELS * PROF_NSTAT];
constexpr int FE_MAX_DEVICES = 64;
static double *g_scratch_ptr[FE_MAX_DEVICES];

static int scratch_lookup() {
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= FE_MAX_DEVICES) return FE_ERR_UNSUPPORTED;
  if (g_scratch_ptr[dev]) return FE_OK;
  void *p = nullptr;
  HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[dev] = (double *)p;
  return FE_OK;
}

/* cell-centred SGS columns, as fetutorialfunctions.py:426-429 (the top level stays 0) */
static void profiles_centre_sgs(double *out, int nz) {
  for (int c = 14; c < 17; ++c) {
    for (int k = 0; k + 1 < nz; ++k) out[k * PROF_NSTAT + c] = 0.5 * (out[k * PROF_NSTAT + c] + out[(k + 1) * PROF_NSTAT + c]);
    out[(nz - 1) * PROF_NSTAT + c] = 0.0;
  }
}

/* The profile rows of the current state into d[0 .. Nz), which has room for every part's rows:
 * parts x Nz <= FE_NOALLOC_MAX_LEVELS (or one part), the same for both entry points, so that they
 * give the same bits; then to out. */
static int profiles_parts(void) {
  return stat_parts(D.Nz, (long)((D.Nx + 3) / 4) * D.Ny, std::max(1, FE_NOALLOC_MAX_LEVELS / D.Nz));
}
static int profiles_run(double *d, double *out) {
  const int parts = profiles_parts();
  const long n4 = (long)((D.Nx + 3) / 4) * D.Ny;
  hipLaunchKernelGGL(k_profiles, dim3(D.Nz, parts), dim3(STAT_NT), 0, D.stream, D.S[0], D.fs, D.ps, D.Nx, D.Ny, D.P, D.nTKE, D.nM,
                     D.tau, (n4 + parts - 1) / parts, d);
  hipLaunchKernelGGL(k_profiles_final, dim3(D.Nz), dim3(64), 0, D.stream, d, parts, D.Nz, (double)D.Nx * D.Ny);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(out, d, (size_t)D.Nz * PROF_NSTAT * sizeof(double), hipMemcpyDeviceToHost, D.stream));
  HIPCHK(hipStreamSynchronize(D.stream));
  profiles_centre_sgs(out, D.Nz);
  return FE_OK;
}

/* n doubles of the model's statistics workspace (kept until cuda_hydroCoreCleanup) */
static int stat_space(size_t n) {
  if (n <= D.stat_n) return FE_OK;
  if (D.stat) HIPCHK(hipFree(D.stat));
  D.stat = nullptr;
  D.stat_n = 0;
  HIPCHK(hipMalloc(&D.stat, n * sizeof(double)));
  D.stat_n = n;
  return FE_OK;
}

int fe_profiles(double *out, int nstat) {
  if (!D.hydro) return FE_ERR_STATE;
  if (nstat != PROF_NSTAT || !out) return FE_ERR_UNSUPPORTED;
  int rc;
  if ((rc = stat_space((size_t)profiles_parts() * D.Nz * PROF_NSTAT))) return rc;
  return profiles_run(D.stat, out);
}

/* fe_profiles without any device allocation: the per-level rows go to the library's
 * static scratch array (no hipMalloc/hipFree; the only device memory touched besides the
 * state is that array).  Grids of more than FE_NOALLOC_MAX_LEVELS levels are rejected.
 * Every row the kernels read they have written in the same call, so nothing needs clearing; calls
 * that overlap on one GPU share the array and race. */
int fe_profiles_noalloc(double *out, int nstat) {
  if (!D.hydro) return FE_ERR_STATE;
  if (nstat != PROF_NSTAT || !out) return FE_ERR_UNSUPPORTED;
  if (D.Nz > FE_NOALLOC_MAX_LEVELS) {
    fprintf(stderr, "fe_profiles_noalloc: %d levels exceed the static scratch of %d levels\n", D.Nz, FE_NOALLOC_MAX_LEVELS);
    return FE_ERR_UNSUPPORTED;
  }
  int rc, dev = 0;
  if ((rc = scratch_lookup())) return rc;
  HIPCHK(hipGetDevice(&dev));
  return profiles_run(g_scratch_ptr[dev], out);
}

/* Per-field state summary of the device state, the on-device counterpart of the
 * reference's host scan hydro_coreStateLogDump / hydro_coreFldStateLogEntry
 * (SRC/HYDRO_CORE/hydro_core.c:1282-1525): over the interior cells, the maximum
 * and minimum with their first location in the reference's (i, j, k) loop order,
 * the mean over all cells of the finite values, and the NaN and Inf counts, of
 * rho, u, v, w, theta (rho-weighted fields times float(1/rho), as the reference
 * forms them), p', the SGS TKE and the moisture species per unit mass; plus the
 * horizontal sum of the raw (rho-weighted) field, from which the host forms its
 * volume integral (mass, rho*theta, ... budgets).  Several work-groups per level, four cells
 * per thread and load; the FP64 sums and the (value, location) extremes are reduced with
 * cross-lane shuffles, then across the wavefronts in LDS, then over the level's parts; the host
 * combines the levels.  256 x 256 x 96, nine rows (226 MB): one work-group per level 1186 us,
 * parts 165 us (an extremes-of-four fast path for finite cells measured 440 us: registers). */
constexpr int SUM_NCOL = 12, SUM_LV = 8, SUM_MAXF = 9;
constexpr unsigned SUM_NONE = 0xffffffffu;      /* no location (a plane has fewer columns: fields are below 4 GiB) */
__device__ __forceinline__ void sum_pick(float &v, unsigned &k, float v2, unsigned k2, bool is_max) {
  const bool take = is_max ? (v2 > v || (v2 == v && k2 < k)) : (v2 < v || (v2 == v && k2 < k));
  if (take) { v = v2; k = k2; }
}
/* Joins n partial rows, stride doubles apart, into one at to (which may be the first of them). */
__device__ __forceinline__ void summary_join(const double *q, long stride, int n, double *to) {
  float vx = (float)q[0], vn = (float)q[2];
  unsigned kx = (unsigned)q[1], kn = (unsigned)q[3];
  double a4 = q[4], a5 = q[5], a6 = q[6], a7 = q[7];
  for (int i = 1; i < n; ++i) {
    const double *p = q + (long)i * stride;
    sum_pick(vx, kx, (float)p[0], (unsigned)p[1], true);
    sum_pick(vn, kn, (float)p[2], (unsigned)p[3], false);
    a4 += p[4]; a5 += p[5]; a6 += p[6]; a7 += p[7];
  }
  to[0] = vx; to[1] = (double)kx; to[2] = vn; to[3] = (double)kn; to[4] = a4; to[5] = a5; to[6] = a6; to[7] = a7;
}
/* Partial rows of work-group (part, level): [part][level][row][SUM_LV] = max, its column x Ny + y,
 * min, its column, sum of the finite values, NaN count, Inf count, sum of the raw field. */
__global__ void __launch_bounds__(STAT_NT) k_summary(const float *S, const float *pres, long fs, long ps, int Nx, int Ny,
                                                      int P, int ns, long chunk, double *out, const float *dcol) {
  const int z = blockIdx.x, g = (Nx + 3) / 4;
  const long n4 = (long)g * Ny, i1 = min(n4, (long)(blockIdx.y + 1) * chunk);
  float mx[SUM_MAXF], mn[SUM_MAXF];
  unsigned kx[SUM_MAXF], kn[SUM_MAXF], nnan[SUM_MAXF], ninf[SUM_MAXF];
  double sm[SUM_MAXF], raw[SUM_MAXF];
#pragma unroll
  for (int f = 0; f < SUM_MAXF; ++f) {
    mx[f] = -1.0e16f; mn[f] = 1.0e16f; kx[f] = kn[f] = SUM_NONE; sm[f] = raw[f] = 0.0; nnan[f] = ninf[f] = 0;
  }
  for (long i = (long)blockIdx.y * chunk + threadIdx.x; i < i1; i += STAT_NT) {
    const int y = (int)(i / g), x = 4 * (int)(i - (long)y * g);
    const long o = (long)z * ps + (long)y * P + x;
    float rinv[4];
    double dc[4] = {1.0, 1.0, 1.0, 1.0};
    if (dcol) {                                 /* terrain: D per cell */
      const float4 t = *(const float4 *)(dcol + (long)(z + 3) * ps + (long)y * P + x);
      dc[0] = t.x; dc[1] = t.y; dc[2] = t.z; dc[3] = t.w;
    }
#pragma unroll
    for (int f = 0; f < SUM_MAXF; ++f) {
      if (f >= ns) break;
      /* rows: rho, u, v, w, theta, p', TKE..., moisture... */
      float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
      if (f < 5) t = *(const float4 *)(S + (long)f * fs + o);
      else if (f == 5) { if (pres) t = *(const float4 *)(pres + o); }
      else t = *(const float4 *)(S + (long)(f - 1) * fs + o);
      const float fr[4] = {t.x, t.y, t.z, t.w};
      const bool cons = (f != 0 && f != 5);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (f == 0) rinv[j] = (float)(1.0 / (double)fr[j]);
        if (x + j >= Nx) continue;              /* the row's padding */
        const float v = cons ? fr[j] * rinv[j] : fr[j];
        raw[f] += dcol ? (double)fr[j] * dc[j] : (double)fr[j];
        if (isnan(v)) { nnan[f]++; continue; }
        if (isinf(v)) { ninf[f]++; continue; }
        const unsigned key = (unsigned)(x + j) * (unsigned)Ny + (unsigned)y;
        sum_pick(mx[f], kx[f], v, key, true);
        sum_pick(mn[f], kn[f], v, key, false);
        sm[f] += (double)v;
      }
    }
  }
  /* wavefront reduction */
#pragma unroll
  for (int f = 0; f < SUM_MAXF; ++f) {
    if (f >= ns) break;
    for (int off = 32; off > 0; off >>= 1) {
      sum_pick(mx[f], kx[f], __shfl_xor(mx[f], off), __shfl_xor(kx[f], off), true);
      sum_pick(mn[f], kn[f], __shfl_xor(mn[f], off), __shfl_xor(kn[f], off), false);
      sm[f] += __shfl_xor(sm[f], off);
      raw[f] += __shfl_xor(raw[f], off);
      nnan[f] += __shfl_xor(nnan[f], off);
      ninf[f] += __shfl_xor(ninf[f], off);
    }
  }
  __shared__ double part[STAT_NT / 64][SUM_MAXF][SUM_LV];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  if (lane == 0) {
#pragma unroll
    for (int f = 0; f < SUM_MAXF; ++f) {
      double *q = part[wave][f];
      q[0] = mx[f]; q[1] = (double)kx[f]; q[2] = mn[f]; q[3] = (double)kn[f];
      q[4] = sm[f]; q[5] = nnan[f]; q[6] = ninf[f]; q[7] = raw[f];
    }
  }
  __syncthreads();
  if (threadIdx.x < ns)
    summary_join(&part[0][threadIdx.x][0], SUM_MAXF * SUM_LV, STAT_NT / 64,
                 out + (((long)blockIdx.y * gridDim.x + z) * ns + threadIdx.x) * SUM_LV);
}
/* A level's parts joined into part 0's row, in place. */
__global__ void __launch_bounds__(64) k_summary_final(double *out, int parts, int nlev, int ns) {
  if (threadIdx.x >= ns) return;
  double *r = out + ((long)blockIdx.x * ns + threadIdx.x) * SUM_LV;
  summary_join(r, (long)nlev * ns * SUM_LV, parts, r);
}

int fe_state_summary(double *out, int nrow) {
  if (!D.hydro) return FE_ERR_STATE;
  const int ns = 6 + D.nTKE + D.nM;
  if (nrow != ns || !out || ns > SUM_MAXF) return FE_ERR_UNSUPPORTED;
  std::vector<double> lv((size_t)D.Nz * ns * SUM_LV);
  const long n4 = (long)((D.Nx + 3) / 4) * D.Ny;
  const int parts = stat_parts(D.Nz, n4, LONG_MAX);
  int rc;
  if ((rc = stat_space((size_t)parts * lv.size()))) return rc;
  /* on a terrain-following grid the kernel weights each cell by its own D (row PR_D of the
   * per-column table); on a flat one the host multiplies the level sums by the level's D */
  const float *dcol = D.terrain ? D.tprof + (size_t)PR_D * D.np * D.ps : nullptr;
  hipLaunchKernelGGL(k_summary, dim3(D.Nz, parts), dim3(STAT_NT), 0, D.stream, D.S[0], D.pout, D.fs, D.ps, D.Nx, D.Ny, D.P, ns,
                     (n4 + parts - 1) / parts, D.stat, dcol);
  if (parts > 1) hipLaunchKernelGGL(k_summary_final, dim3(D.Nz), dim3(64), 0, D.stream, D.stat, parts, D.Nz, ns);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(lv.data(), D.stat, lv.size() * sizeof(double), hipMemcpyDeviceToHost, D.stream));
  HIPCHK(hipStreamSynchronize(D.stream));
  const double NONE = (double)0x7fffffffffffffffLL;
  const double ncell = (double)D.Nx * D.Ny * D.Nz;
  const double dV = (double)dX * dY * dZ;
  for (int f = 0; f < ns; ++f) {
    float vx = -1.0e16f, vn = 1.0e16f;
    long long qx = 0x7fffffffffffffffLL, qn = qx;
    double sum = 0, nn = 0, ni = 0, integ = 0;
    for (int z = 0; z < D.Nz; ++z) {
      const double *r = &lv[((size_t)z * ns + f) * SUM_LV];
      const float v1 = (float)r[0], v2 = (float)r[2];
      /* column x Ny + y of the level -> the reference's loop order over the grid */
      const long long none = 0x7fffffffffffffffLL;
      const long long k1 = r[1] >= (double)SUM_NONE ? none : (long long)r[1] * D.Nz + z;
      const long long k2 = r[3] >= (double)SUM_NONE ? none : (long long)r[3] * D.Nz + z;
      if (v1 > vx || (v1 == vx && k1 < qx)) { vx = v1; qx = k1; }
      if (v2 < vn || (v2 == vn && k2 < qn)) { vn = v2; qn = k2; }
      sum += r[4]; nn += r[5]; ni += r[6];
      integ += r[7] * (D.terrain ? 1.0 : (double)D_Jac[idx3(Nh, Nh, z + Nh)]) * dV;
    }
    double *o = out + (long)f * SUM_NCOL;
    auto loc = [&](long long q, double *ijk) {
      if ((double)q >= NONE) { ijk[0] = ijk[1] = ijk[2] = 0; return; }
      const long long zk = q % D.Nz, rest = q / D.Nz, yj = rest % D.Ny, xi = rest / D.Ny;
      ijk[0] = (double)(xi + Nh); ijk[1] = (double)(yj + Nh); ijk[2] = (double)(zk + Nh);
    };
    o[0] = vx; loc(qx, o + 1);
    o[4] = vn; loc(qn, o + 5);
    o[8] = sum / ncell; o[9] = nn; o[10] = ni; o[11] = integ;
  }
  return FE_OK;
}

int fe_debug_build_frhs(int stage) {
  if (!D.hydro) return FE_ERR_STATE;
  int rc;
  /* F of the stage evaluated on the current device state S0, into S1 */
  if ((rc = launch_stage(stage, D.S[0], D.S[0], D.S[1], 1, nullptr))) return rc;
  HIPCHK(hipStreamSynchronize(D.stream));
  const long n3 = D.n3h;
  std::vector<float> tmp((size_t)D.NF * D.fs);
  HIPCHK(hipMemcpy(tmp.data(), D.S[1], tmp.size() * sizeof(float), hipMemcpyDeviceToHost));
  auto put = [&](float *host, int f) {
    if (!host) return;
    memset(host, 0, n3 * sizeof(float));
    for (int z = 0; z < D.Nz; ++z)
      for (int y = 0; y < D.Ny; ++y)
        for (int x = 0; x < D.Nx; ++x)
          host[idx3(x + Nh, y + Nh, z + Nh)] = tmp[(size_t)f * D.fs + (size_t)z * D.ps + (size_t)y * D.P + x];
  };
  for (int f = 0; f < 5; ++f) put(hydroFldsFrhs + f * n3, f);
  for (int f = 0; f < D.nTKE; ++f) put(sgstkeScalarsFrhs + f * n3, 5 + f);
  for (int f = 0; f < D.nM; ++f) put(moistScalarsFrhs + f * n3, 5 + D.nTKE + f);
  /* surface-layer state was advanced by a physics stage; bring it back too */
  if (physics_stage(stage) && surflayerSelector > 0) {
    if ((rc = xfer_reserve(D.n3h * sizeof(float)))) return rc;
    XferScope scope;
    if ((rc = download_2d(surfp(SF_CD), cdFld))) return rc;
    if ((rc = download_2d(surfp(SF_CH), chFld))) return rc;
    if ((rc = download_2d(surfp(SF_UST), fricVel))) return rc;
    if ((rc = download_2d(surfp(SF_IOL), invOblen))) return rc;
    if ((rc = download_2d(surfp(SF_HF), htFlux))) return rc;
    return xfer_finish(D.stream);
  }
  return FE_OK;
}

}  // extern "C"

#include "fe_ensemble.hip"
#include "fe_sgs.hip"
#include "fe_checkpoint.hip"
