/*
 * fe_sgs_kernels.hip -- device side of the learned SGS closure.
 *
 * The closure it stands beside is the prognostic-TKE eddy-viscosity closure of the
 * physics stage (SRC/HYDRO_CORE/CUDA/cuda_sgsTurbDevice.cu:202-367,
 * cuda_sgstkeDevice.cu:68-397).  A small MLP maps the local resolved-gradient stencil of a
 * cell to its SGS stresses and heat fluxes:
 *   inputs (250): the nine centred velocity gradients du_i/dx_j at the 27 cells of the
 *     3x3x3 stencil around the cell (243; stencil order z, y, x from -1 to +1, components
 *     u_x u_y u_z v_x v_y v_z w_x w_y w_z), then dtheta/dz at the cell and its six face
 *     neighbours (x-, x+, y-, y+, z-, z+); lateral neighbours wrap periodically, vertical
 *     ones are clamped to the column, and d/dz carries the level's J33; each feature is
 *     normalised by its training mean and standard deviation (padded to 256 columns);
 *   network: 256 -> 64 -> 64 -> 64 (GELU) -> 9 (linear), weights [in][out] row-major;
 *   outputs (9): the kinematic SGS stresses tau_11, tau_22, tau_33, tau_12, tau_13,
 *     tau_23 and heat fluxes tau_theta1..3 at the cell centre, normalised likewise.
 * Every product runs on the matrix cores: a BF16 MFMA GEMM (operands rounded to BF16 when
 * staged in LDS, FP32 accumulation), with FP32 activations, gradients and master weights.
 */

namespace fe {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int SGS_NIN = 250, SGS_KIN = 256, SGS_H = 64, SGS_NOUT = 9, SGS_KOUT = 16;
/* parameter vector: W1 [256][64], b1 [64], W2 [64][64], b2, W3 [64][64], b3, W4 [64][16], b4 [16] */
constexpr long OW1_ = 0, OB1_ = OW1_ + (long)SGS_KIN * SGS_H, OW2_ = OB1_ + SGS_H, OB2_ = OW2_ + SGS_H * SGS_H,
               OW3_ = OB2_ + SGS_H, OB3_ = OW3_ + SGS_H * SGS_H, OW4_ = OB3_ + SGS_H, OB4_ = OW4_ + SGS_H * SGS_KOUT,
               NPARAM_ = OB4_ + SGS_KOUT;

/* FP32 -> BF16, round to nearest even (the hardware conversion, v_cvt_pk_bf16_f32) */
__device__ __forceinline__ unsigned short f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }

enum { GEMM_PLAIN = 0, GEMM_BIAS, GEMM_BIAS_GELU, GEMM_GELU_BACK };

struct GemmArgs {
  const float *A; long sam, sak;   /* A(m, k) = A[m*sam + k*sak], one of the strides 1 */
  const float *B; long sbk, sbn;   /* B(k, n) = B[k*sbk + n*sbn], one of the strides 1 */
  float *C; long ldc;              /* C(m, n) = C[m*ldc + n] */
  int M, N, K;
  int kchunk;                      /* rows of k per work-group z (a multiple of GK) */
  long zstride;                    /* C (and csum) of work-group z start z*zstride further on */
  float *csum;                     /* sum over k of B(k, n) in FP32 (null: none; needs sbn = 1) */
  int epi;                         /* GEMM_*: what is applied to the product */
  const float *bias;               /* GEMM_BIAS*: C = A B + bias (row broadcast) */
  float *act;                      /* GEMM_BIAS_GELU: GELU(C), same layout as C */
  const float *Z;                  /* GEMM_GELU_BACK: C = (A B) GELU'(Z), same layout as C */
};

constexpr int GT = 64, GK = 32, GKP = GK + 4;

/* GELU(z) = z Phi(z) without transcendentals: Phi(z) = 1/2 + zc Q(zc^2), zc = z clamped to
 * [-4, 4], Q a degree-7 polynomial (in zc^2) fitted to the normal CDF on [0, 4] in the
 * weighted least-squares sense with Q(16) = 1/8 imposed, so that Phi = 0 and 1 beyond the
 * clamp (to 5e-9): |GELU - z Phi_exact(z)| <= 1.4e-4 for all z (largest at |z| = 4, where the exact
 * tail 4 Phi(-4) = 1.3e-4 is dropped), below half a BF16 step of any activation above 0.035,
 * and 11 instructions against two quarter-rate transcendentals and 16 instructions of an
 * erf-based form.  Q(s) = sum_j c_j s^j; c_0 = 0.39881 ~ 1/sqrt(2 pi). */
__device__ __forceinline__ float gelu_q(float s) {
  float q = fmaf(-1.288297990e-09f, s, 1.050534689e-07f);
  q = fmaf(q, s, -3.724001524e-06f);
  q = fmaf(q, s, 7.636147270e-05f);
  q = fmaf(q, s, -1.022127353e-03f);
  q = fmaf(q, s, 9.584851178e-03f);
  q = fmaf(q, s, -6.606890165e-02f);
  return fmaf(q, s, 3.988074278e-01f);
}
__device__ __forceinline__ float gelu(float z) {
  const float zc = fminf(fmaxf(z, -4.f), 4.f);
  return z * fmaf(zc, gelu_q(zc * zc), 0.5f);
}
/* its derivative Phi(z) + z Phi'(z): Phi' = d/dz [zc Q(zc^2)] = sum_j (2j+1) c_j zc^2j inside
 * the clamp and 0 outside, so that the training gradient is that of the function evaluated */
__device__ __forceinline__ float gelu_d(float z) {
  const float zc = fminf(fmaxf(z, -4.f), 4.f), s = zc * zc;
  float d = fmaf(-1.932446985e-08f, s, 1.365695096e-06f);
  d = fmaf(d, s, -4.096401676e-05f);
  d = fmaf(d, s, 6.872532543e-04f);
  d = fmaf(d, s, -7.154891471e-03f);
  d = fmaf(d, s, 4.792425589e-02f);
  d = fmaf(d, s, -1.982067049e-01f);
  d = fmaf(d, s, 3.988074278e-01f);
  return fmaf(zc, gelu_q(s), 0.5f) + (fabsf(z) < 4.f ? z * d : 0.f);
}

/* Four consecutive values of an operand tile: element (r, c) at p + r*ld + c, c the unit-stride
 * index; columns at or past nc and rows at or past nr are 0.  vec: 16-byte loads are aligned. */
__device__ __forceinline__ f32x4 tile4(const float *p, long ld, long r, long c, long nr, long nc, bool vec) {
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
  if (r < nr) {
    const float *q = p + r * ld + c;
    if (vec && c + 3 < nc) v = *(const f32x4 *)q;
    else
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (c + i < nc) v[i] = q[i];
  }
  return v;
}

/* C = A B on 64 x 64 output tiles, four waves of 32 x 32, v_mfma_f32_16x16x16_bf16 over
 * K steps of 32 staged in LDS (k contiguous per row and per column, so each lane's four
 * operand values are adjacent).  Operand layout of the instruction: lane l holds
 * A[l % 16][4 (l / 16) + v] and B[4 (l / 16) + v][l % 16], v = 0..3, and receives
 * D[4 (l / 16) + v][l % 16].
 * The network's products are small: what bounds them is the latency of a K step (load, stage,
 * multiply) and the launches around them.  So the next step's operands are loaded (16 bytes per
 * lane where alignment allows) before the current step is multiplied, LDS has two buffers (one
 * barrier per step), bias, GELU and GELU' are applied to the accumulators instead of in passes of
 * their own, and a product over the rows of a batch (the weight gradients: 64 or 256 x 64 outputs,
 * thousands of k) is split over k into work-groups whose partial sums k_gemm_reduce adds in order;
 * the bias gradient is the column sum of B, formed from the same loads.  8192 rows, forward and
 * backward: first layer 50 -> 21 us, a weight gradient 1350 us (1 or 4 work-groups) -> 14 us. */
__global__ void __launch_bounds__(256) k_gemm_bf16(GemmArgs g) {
  __shared__ __align__(16) unsigned short As[2][GT][GKP];
  __shared__ __align__(16) unsigned short Bs[2][GT][GKP];
  __shared__ __align__(16) float cs[16][GT];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m0 = blockIdx.x * GT, n0 = blockIdx.y * GT;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  const int kbeg = blockIdx.z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
  float *C = g.C + (long)blockIdx.z * g.zstride;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool a_krow = (g.sak == 1), b_ncol = (g.sbn == 1);
  const long lda = a_krow ? g.sam : g.sak, ldb = b_ncol ? g.sbk : g.sbn;
  const bool va = ((unsigned long)g.A & 15) == 0 && (lda & 3) == 0, vb = ((unsigned long)g.B & 15) == 0 && (ldb & 3) == 0;
  /* element e of a tile, four values wide: (row e / 8, k 4 (e % 8)) where k is the unit-stride
   * index, (k e / 16, row 4 (e % 16)) where the row is */
  auto loads = [&](int k0, f32x4 (&ra)[2], f32x4 (&rb)[2]) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int e = tid + 256 * q;
      ra[q] = a_krow ? tile4(g.A, lda, m0 + (e >> 3), k0 + 4 * (e & 7), g.M, kend, va)
                     : tile4(g.A, lda, k0 + (e >> 4), m0 + 4 * (e & 15), kend, g.M, va);
      rb[q] = b_ncol ? tile4(g.B, ldb, k0 + (e >> 4), n0 + 4 * (e & 15), kend, g.N, vb)
                     : tile4(g.B, ldb, n0 + (e >> 3), k0 + 4 * (e & 7), g.N, kend, vb);
    }
  };
  auto stage = [&](unsigned short (*T)[GKP], const f32x4 &v, int e, bool krow) {
    if (krow) {
      *(bf16x4 *)&T[e >> 3][4 * (e & 7)] = bf16x4{(short)f2bf(v[0]), (short)f2bf(v[1]), (short)f2bf(v[2]), (short)f2bf(v[3])};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) T[4 * (e & 15) + i][e >> 4] = f2bf(v[i]);
    }
  };
  const bool do_cs = g.csum && blockIdx.x == 0;
  f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 ra[2], rb[2];
  loads(kbeg, ra, rb);
  int buf = 0;
  for (int k0 = kbeg; k0 < kend; k0 += GK, buf ^= 1) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      stage(As[buf], ra[q], tid + 256 * q, a_krow);
      stage(Bs[buf], rb[q], tid + 256 * q, !b_ncol);
      if (do_cs) sum += rb[q];
    }
    if (k0 + GK < kend) loads(k0 + GK, ra, rb);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < GK; ks += 16) {
      bf16x4 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = *(const bf16x4 *)&As[buf][wm + 16 * i + (lane & 15)][ks + 4 * (lane >> 4)];
        b[i] = *(const bf16x4 *)&Bs[buf][wn + 16 * i + (lane & 15)][ks + 4 * (lane >> 4)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + v, n = n0 + wn + 16 * j + (lane & 15);
        if (m < g.M && n < g.N) {
          const long o = (long)m * g.ldc + n;
          float c = acc[i][j][v];
          if (g.epi == GEMM_BIAS || g.epi == GEMM_BIAS_GELU) c = c + g.bias[n];
          if (g.epi == GEMM_GELU_BACK) c = c * gelu_d(g.Z[o]);
          C[o] = c;
          if (g.epi == GEMM_BIAS_GELU) g.act[o] = gelu(c);
        }
      }
  if (do_cs) {                     /* uniform over the work-group */
    *(f32x4 *)&cs[tid >> 4][4 * (tid & 15)] = sum;
    __syncthreads();
    if (tid < GT && n0 + tid < g.N) {
      float t = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) t += cs[r][tid];
      g.csum[(long)blockIdx.z * g.zstride + n0 + tid] = t;
    }
  }
}

/* out[i] = sum over z of part[z*n + i], in order of z */
__global__ void __launch_bounds__(256) k_gemm_reduce(const float *part, int nz, long n, float *out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
#pragma unroll 8
  for (int z = 0; z < nz; ++z) s += part[(long)z * n + i];
  out[i] = s;
}

/* mean-squared-error gradient over the first nout of N columns: dY = 2 (Y - T) / (M nout);
 * the loss sum (FP64) goes to loss[0] */
__global__ void __launch_bounds__(256) k_loss_grad(const float *Y, const float *T, long M, int N, int nout, float *dY,
                                                   double *loss) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (i < M * N) {
    const int c = (int)(i % N);
    const float d = (c < nout) ? Y[i] - T[i] : 0.f;
    dY[i] = 2.f * d / (float)(M * nout);
    l = (double)d * d;
  }
  for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
  __shared__ double part[4];       /* one atomic per work-group: they queue up on the one address */
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0) {
    l = (part[0] + part[1]) + (part[2] + part[3]);
    if (l != 0.0) atomicAdd(loss, l);
  }
}

/* Adam (Kingma & Ba 2015) on FP32 master weights; bc1, bc2 = 1 - beta^t */
__global__ void k_adam(float *w, const float *g, float *m, float *v, long n, float lr, float b1, float b2, float eps,
                       float bc1, float bc2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

/* rows idx[r] of src (N columns) to row r of dst */
__global__ void k_gather_rows(const float *src, const int *idx, long rows, int N, float *dst) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * N) return;
  const long r = i / N;
  dst[i] = src[(long)idx[r] * N + (i % N)];
}

/* ---- features ---------------------------------------------------------------------------- */
struct FeatArgs {
  const float *S;        /* state [field][z][y][x] (row pitch P): rho, rho*u, rho*v, rho*w, rho*theta */
  long fs, ps;
  int Nx, Ny, Nz, P;
  float dXi, dYi, dZi;
  const float *j33;      /* J33 per level */
  const float *mu, *isd; /* normalisation (null: raw features); isd = 1/std */
  float *X;              /* [cells][256] */
  float *gmax;           /* max |normalised feature| per cell (null: none) */
  long c0, nc;           /* cells [c0, c0 + nc) of the x-fastest interior index */
};

/* (x, y, z) of the x-fastest interior index c, in 32-bit arithmetic (the host keeps the learned
 * closure's grids below 2^31 cells, and 12 x cells below 2^32) */
__device__ __forceinline__ void cell_xyz(long c, int Nx, int Ny, int &x, int &y, int &z) {
  const unsigned u = (unsigned)c, q = u / (unsigned)Nx, zz = q / (unsigned)Ny;
  x = (int)(u - q * (unsigned)Nx);
  y = (int)(q - zz * (unsigned)Ny);
  z = (int)zz;
}

__device__ __forceinline__ float fvel(const FeatArgs &a, int f, int x, int y, int z) {
  x = x < 0 ? x + a.Nx : (x >= a.Nx ? x - a.Nx : x);
  y = y < 0 ? y + a.Ny : (y >= a.Ny ? y - a.Ny : y);
  z = z < 0 ? 0 : (z >= a.Nz ? a.Nz - 1 : z);
  const long o = (long)z * a.ps + (long)y * a.P + x;
  return a.S[f * a.fs + o] / a.S[o];
}

/* The nine centred velocity gradients du_i/dx_j of cell (x, y, z), ordered u_x u_y u_z v_x
 * v_y v_z w_x w_y w_z, and dtheta/dz (g[9]); lateral neighbours wrap (x, y may lie one cell
 * outside the grid), vertical ones are clamped to the column, d/dz carries the level's J33.
 * Shared by the feature kernel and the gradient pass of the fused inference, so that both
 * produce the same bits. */
__device__ __forceinline__ void sgs_grad_cell(const FeatArgs &a, int x, int y, int z, float g[10]) {
  const float hz = 0.5f * a.j33[z] * a.dZi;
  int q = 0;
#pragma unroll
  for (int f = 1; f <= 3; ++f) {
    g[q++] = 0.5f * a.dXi * (fvel(a, f, x + 1, y, z) - fvel(a, f, x - 1, y, z));
    g[q++] = 0.5f * a.dYi * (fvel(a, f, x, y + 1, z) - fvel(a, f, x, y - 1, z));
    g[q++] = hz * (fvel(a, f, x, y, z + 1) - fvel(a, f, x, y, z - 1));
  }
  g[9] = hz * (fvel(a, 4, x, y, z + 1) - fvel(a, 4, x, y, z - 1));
}

/* The seven neighbours whose dtheta/dz are features 243..249: the cell, x-, x+, y-, y+, z-, z+. */
__constant__ int c_sgs_tnb[7][3] = {{0, 0, 0}, {-1, 0, 0}, {1, 0, 0}, {0, -1, 0}, {0, 1, 0}, {0, 0, -1}, {0, 0, 1}};

/* one thread per cell: the 250 features, normalised, and their largest magnitude */
__global__ void __launch_bounds__(256) k_sgs_features(FeatArgs a) {
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= a.nc) return;
  const long c = a.c0 + r;
  int x, y, z;
  cell_xyz(c, a.Nx, a.Ny, x, y, z);
  float *X = a.X + r * SGS_KIN;
  float gm = 0.f;
  int q = 0;
  auto put = [&](float v) {
    if (a.mu) v = (v - a.mu[q]) * a.isd[q];
    gm = fmaxf(gm, fabsf(v));
    X[q++] = v;
  };
  float g[10];
  for (int dz = -1; dz <= 1; ++dz) {
    const int zz = z + dz < 0 ? 0 : (z + dz >= a.Nz ? a.Nz - 1 : z + dz);
    for (int dy = -1; dy <= 1; ++dy)
      for (int dx = -1; dx <= 1; ++dx) {
        sgs_grad_cell(a, x + dx, y + dy, zz, g);
        for (int k = 0; k < 9; ++k) put(g[k]);
      }
  }
  for (int n = 0; n < 7; ++n) {
    const int zz = z + c_sgs_tnb[n][2] < 0 ? 0 : (z + c_sgs_tnb[n][2] >= a.Nz ? a.Nz - 1 : z + c_sgs_tnb[n][2]);
    sgs_grad_cell(a, x + c_sgs_tnb[n][0], y + c_sgs_tnb[n][1], zz, g);
    put(g[9]);
  }
  for (; q < SGS_KIN; ++q) X[q] = 0.f;
  if (a.gmax) a.gmax[c] = gm;
}

/* Gradient pass of the fused inference: one thread per cell of [c0, c0 + nc), the ten values
 * of sgs_grad_cell into G: [cells][4], [cells][4], [cells], [cells] (a wave's gathers there are
 * contiguous; in records of 12 floats a cell each spread over three times the lines). */
__global__ void __launch_bounds__(256) k_sgs_grad(FeatArgs a, float *G) {
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= a.nc) return;
  const long c = a.c0 + r;
  int x, y, z;
  cell_xyz(c, a.Nx, a.Ny, x, y, z);
  float g[10];
  sgs_grad_cell(a, x, y, z, g);
  const long n = (long)a.Nx * a.Ny * a.Nz;
  ((float4 *)G)[c] = make_float4(g[0], g[1], g[2], g[3]);
  ((float4 *)(G + 4 * n))[c] = make_float4(g[4], g[5], g[6], g[7]);
  G[8 * n + c] = g[8];
  G[9 * n + c] = g[9];
}

/* ---- training data: box filter of a fine state ------------------------------------------- */
/* One thread per coarse cell of fac^3 fine cells: the filtered state (rho and the
 * rho-weighted fields averaged) into Sc ([5][zc][yc][xc]), and the Favre-filtered SGS
 * fluxes per unit mass, tau_ij = <rho u_i u_j>/<rho> - u~_i u~_j + <tau_f,ij>/<rho> (the fine
 * run's own SGS stresses tau_f included), in the output order 11, 22, 33, 12, 13, 23,
 * theta1..3, into T ([cells][16]); sums in FP64. */
__global__ void __launch_bounds__(256) k_sgs_filter(const float *S, const float *tau, long fs, long ps, int P, int nxc,
                                                    int nyc, int nzc, int fac, float *Sc, float *T) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ncell = (long)nxc * nyc * nzc;
  if (c >= ncell) return;
  int xc, yc, zc;
  cell_xyz(c, nxc, nyc, xc, yc, zc);
  double s[5] = {0, 0, 0, 0, 0}, p[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, t[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  /* emitted stress fields: 11, 21, 31, 32, 22, 33, theta1, theta2, theta3 -> output order */
  const int tmap[9] = {0, 4, 5, 1, 2, 3, 6, 7, 8};
  for (int kz = 0; kz < fac; ++kz)
    for (int ky = 0; ky < fac; ++ky)
      for (int kx = 0; kx < fac; ++kx) {
        const long o = (long)(zc * fac + kz) * ps + (long)(yc * fac + ky) * P + (xc * fac + kx);
        const double r = S[o], ru = S[fs + o], rv = S[2 * fs + o], rw = S[3 * fs + o], rt = S[4 * fs + o];
        s[0] += r; s[1] += ru; s[2] += rv; s[3] += rw; s[4] += rt;
        const double u = ru / r, v = rv / r, w = rw / r, th = rt / r;
        p[0] += ru * u; p[1] += rv * v; p[2] += rw * w; p[3] += ru * v; p[4] += ru * w; p[5] += rv * w;
        p[6] += ru * th; p[7] += rv * th; p[8] += rw * th;
        if (tau)
          for (int q = 0; q < 9; ++q) t[q] += tau[(long)tmap[q] * fs + o];
      }
  const double n = (double)fac * fac * fac;
  const long psc = (long)nxc * nyc, fsc = psc * nzc, oc = (long)zc * psc + (long)yc * nxc + xc;
  for (int f = 0; f < 5; ++f) Sc[f * fsc + oc] = (float)(s[f] / n);
  const double u = s[1] / s[0], v = s[2] / s[0], w = s[3] / s[0], th = s[4] / s[0];
  const double mean[9] = {u * u, v * v, w * w, u * v, u * w, v * w, u * th, v * th, w * th};
  float *Tr = T + c * SGS_KOUT;
  for (int q = 0; q < 9; ++q) Tr[q] = (float)((p[q] + t[q]) / s[0] - mean[q]);
  for (int q = 9; q < SGS_KOUT; ++q) Tr[q] = 0.f;
}

/* column mean and sum of squared deviations (FP64), one work-group per column */
__global__ void __launch_bounds__(256) k_colstats(const float *X, long M, int N, double *out) {
  const int n = blockIdx.x;
  double s = 0.0, s2 = 0.0;
  for (long m = threadIdx.x; m < M; m += 256) {
    const double v = X[m * N + n];
    s += v;
    s2 += v * v;
  }
  for (int off = 32; off > 0; off >>= 1) { s += __shfl_xor(s, off); s2 += __shfl_xor(s2, off); }
  __shared__ double part[4][2];
  if ((threadIdx.x & 63) == 0) { part[threadIdx.x >> 6][0] = s; part[threadIdx.x >> 6][1] = s2; }
  __syncthreads();
  if (threadIdx.x == 0) {
    out[2 * n] = part[0][0] + part[1][0] + part[2][0] + part[3][0];
    out[2 * n + 1] = part[0][1] + part[1][1] + part[2][1] + part[3][1];
  }
}

/* x = (x - mu) * isd over the first nu of N columns; the others to 0 */
__global__ void k_normalise(float *X, long M, int N, int nu, const float *mu, const float *isd) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * N) return;
  const int c = (int)(i % N);
  X[i] = c < nu ? (X[i] - mu[c]) * isd[c] : 0.f;
}

/* ---- inference: de-normalisation, realizability, cell stresses ------------------------- */
/* Cell stresses rho*tau (ordered 11, 22, 33, 12, 13, 23, theta1..3) from the network's output
 * of cells [c0, c0+nc); the cell is used where its inputs pass the distribution gate
 * (every |normalised feature| <= gate) and the predicted stress tensor is realizable
 * (positive semi-definite: non-negative diagonal, |tau_ij|^2 <= tau_ii tau_jj, det >= 0,
 * Schumann 1977); its mask is 1 then, else 0. */
__device__ __forceinline__ bool sgs_realizable(float a, float b, float d, float e, float f, float h) {
  bool ok = a >= 0.f && b >= 0.f && d >= 0.f && e * e <= a * b && f * f <= a * d && h * h <= b * d;
  const float det = a * (b * d - h * h) - e * (e * d - h * f) + f * (e * h - b * f);
  ok = ok && det >= 0.f;
  return ok;
}

__global__ void k_sgs_finish(const float *Y, const float *ymu, const float *ysd, const float *gmax, float gate, const float *S,
                             long fs, long ps, int Nx, int Ny, int P, long c0, long nc, float *tauL, long ncell,
                             unsigned char *mask) {
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nc) return;
  const long c = c0 + r;
  int x, y, z;
  cell_xyz(c, Nx, Ny, x, y, z);
  const float rho = S[(long)z * ps + (long)y * P + x];
  float t[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) t[q] = Y[r * SGS_KOUT + q] * ysd[q] + ymu[q];
  mask[c] = gmax[c] <= gate && sgs_realizable(t[0], t[1], t[2], t[3], t[4], t[5]) ? 1 : 0;
#pragma unroll
  for (int q = 0; q < 9; ++q) tauL[q * ncell + c] = rho * t[q];
}

/* ---- fused inference ----------------------------------------------------------------------
 * Features, the four network layers and the finish of 64 cells per work-group iteration,
 * without the intermediate feature and activation arrays in HBM.  Persistent work-groups of
 * four waves: wave w keeps its 16 output columns of W1, W2, W3 and all of W4 in registers (BF16)
 * for the whole launch and loops over tiles of 64 consecutive cells (x-fastest interior index):
 *   features  wave w, lane = cell: features 64 w .. 64 w + 63 from the precomputed gradients of
 *             the eight neighbours that hold them (loaded one tile ahead, while the previous
 *             tile is in layer 1), normalised, their largest magnitude (the
 *             gate), four at a time as BF16 to LDS;
 *   layers    4 cell blocks x 16 (layer 1) or 4 (layers 2, 3) k blocks of
 *             v_mfma_f32_16x16x16_bf16 per wave with the weights as the left operand, so that a
 *             lane holds four consecutive outputs of one cell: bias and GELU in FP32 on the
 *             accumulators, then one 8-byte store of four BF16 activations for the next layer;
 *             layer 4: wave w the cell block w, all 16 outputs;
 *   finish    on the layer-4 accumulators: a lane de-normalises and stores its own outputs, the
 *             first 16 lanes take the two off-diagonal stresses they lack from the next 16 and
 *             decide gate and realizability.
 * LDS holds operands as [k / 4][cell][4], so that both the stores and the operand reads are
 * 8 bytes a lane over consecutive addresses.  Four barriers a tile: the next tile's features are
 * written behind the one that ends layer 1.
 * The rounding points (features and activations to BF16, MFMA accumulation over k blocks in
 * increasing order, FP32 bias and GELU) are those of the unfused kernels, so both paths give
 * the same bits.
 * What bounds it: vector instructions, 970 per wave and tile (600 of them the GELUs), at two waves
 * per SIMD (the prefetched features and the weights are 128 registers; 256 in all, 29 spilled), then
 * its gathers.  128 x 128 x 48: 234 us with four lanes per cell that read each feature's normalisation
 * from LDS, stored it as two bytes and waited for every neighbour's loads, and a serial finish by one
 * wave; 170 us without, 158 us with the gradients by component (k_sgs_grad) instead of in records of
 * 12 floats.  A contiguous run of tiles per XCD made no difference (170 us), nor did scalar
 * normalisation operands; chaining the layers in registers, a wave per 16 cells, was slower (180 us).
 * Three waves per SIMD, the features loaded in two halves (168 registers, 44 spilled): 161 us, and a
 * 64 x 64 x 48 step 145 us against 132 (one tile per work-group, nothing to overlap); the halves at two
 * waves (218, none spilled): 165 us, 131. */
constexpr int FT = 64;

struct FusedArgs {
  const float *G;                        /* gradients from k_sgs_grad */
  int Nx, Ny, Nz;
  const float *mu, *isd;                 /* feature normalisation [256] */
  const float *w;                        /* FP32 master parameters */
  const float *ymu, *ysd;
  float gate;
  const float *S;                        /* stage input (rho) */
  long ps;
  int P;
  float *tauL;
  long ncell;
  unsigned char *mask;
  unsigned long long *count;             /* cells evaluated, cells passing */
  int ntiles;
};

typedef __bf16 bf16v2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned f2bf2(float a, float b) {
  return __builtin_bit_cast(unsigned, bf16v2{(__bf16)a, (__bf16)b});
}
__device__ __forceinline__ bf16x4 ld_frag(const uint2 *p) { return __builtin_bit_cast(bf16x4, *p); }

/* The cell of a lane of the fused kernel: index and coordinates.  A work-group's tiles are a fixed
 * number of cells apart, added with carries instead of two divisions a tile.  Cells past the end
 * repeat the last one; nothing of theirs is stored. */
struct TileCell {
  long c;
  int x, y, z;
  __device__ __forceinline__ TileCell(const FusedArgs &a, long c0) {
    c = min(c0, a.ncell - 1);
    cell_xyz(c, a.Nx, a.Ny, x, y, z);
  }
  __device__ __forceinline__ void advance(const FusedArgs &a, long step, int sx, int sy, int sz) {
    c += step;
    x += sx;
    y += sy;
    z += sz;
    if (x >= a.Nx) { x -= a.Nx; ++y; }
    if (y >= a.Ny) { y -= a.Ny; ++z; }
    if (c >= a.ncell) { c = a.ncell - 1; x = a.Nx - 1; y = a.Ny - 1; z = a.Nz - 1; }
  }
};

/* One wave's share of a tile's features, W the wave: features 64 W .. 64 W + 63, lane = cell.
 * Waves 0 to 2 need components of eight neighbours from their first on, wave 3 the last six
 * neighbours and the seven dtheta/dz. */
template <int W>
struct TileFeatures {
  static constexpr int N0 = SGS_H * W / 9, NN = W < 3 ? 8 : 6, TH = 9 * NN;
  static_assert(SGS_H == FT && SGS_KIN == 4 * FT, "64 features per wave");
  static_assert(W == 3 || 9 * (N0 + NN) >= 64 * (W + 1), "the neighbours hold the wave's features");
  __device__ __forceinline__ static void load(const FusedArgs &a, const TileCell &p, float (&u)[72], float &rho) {
    if (W == 0) rho = a.S[(long)p.z * a.ps + (long)p.y * a.P + p.x];
    /* a neighbour's place is the cell's plus one step per direction, wrapped or clamped by the step
     * (32 bits, modulo 2^32: the sum is a place in the grid) */
    const unsigned c = (unsigned)p.c, row = (unsigned)a.Nx, plane = row * (unsigned)a.Ny;
    const unsigned xo[3] = {p.x == 0 ? row - 1u : -1u, 0u, p.x == a.Nx - 1 ? 1u - row : 1u};
    const unsigned yo[3] = {p.y == 0 ? plane - row : -row, 0u, p.y == a.Ny - 1 ? row - plane : row};
    const unsigned zo[3] = {p.z == 0 ? 0u : -plane, 0u, p.z == a.Nz - 1 ? 0u : plane};
    auto cell = [&](int dx, int dy, int dz) -> unsigned { return c + zo[dz + 1] + yo[dy + 1] + xo[dx + 1]; };
    const float4 *ga = (const float4 *)a.G, *gb = (const float4 *)(a.G + 4 * a.ncell);
    const float *gc = a.G + 8 * a.ncell;
#pragma unroll
    for (int i = 0; i < NN; ++i) {
      const int n = N0 + i;
      const unsigned id = cell(n % 3 - 1, (n / 3) % 3 - 1, n / 9 - 1);
      const float4 u0 = ga[id], u1 = gb[id];
      u[9 * i + 0] = u0.x; u[9 * i + 1] = u0.y; u[9 * i + 2] = u0.z; u[9 * i + 3] = u0.w;
      u[9 * i + 4] = u1.x; u[9 * i + 5] = u1.y; u[9 * i + 6] = u1.z; u[9 * i + 7] = u1.w;
      u[9 * i + 8] = gc[id];
    }
    if constexpr (W == 3) {
      /* dtheta/dz of the cell, x-, x+, y-, y+, z-, z+ (c_sgs_tnb) */
      const float *gt = gc + a.ncell;
      u[TH + 0] = gt[cell(0, 0, 0)];
      u[TH + 1] = gt[cell(-1, 0, 0)];
      u[TH + 2] = gt[cell(1, 0, 0)];
      u[TH + 3] = gt[cell(0, -1, 0)];
      u[TH + 4] = gt[cell(0, 1, 0)];
      u[TH + 5] = gt[cell(0, 0, -1)];
      u[TH + 6] = gt[cell(0, 0, 1)];
      /* the same last element in every wave's branch: the array stays in registers */
#pragma unroll
      for (int i = TH + 7; i < 72; ++i) u[i] = 0.f;
    }
  }
  /* normalised, to As; returns their largest magnitude */
  __device__ __forceinline__ static float put(const float2 *nrm, const float (&u)[72], uint2 (*As)[FT], int lane) {
    float gm = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i > 0 && i % 4 == 0) __builtin_amdgcn_sched_barrier(0);
      float v[4];
      const float4 n01 = *(const float4 *)&nrm[64 * W + 4 * i], n23 = *(const float4 *)&nrm[64 * W + 4 * i + 2];
      const float mu[4] = {n01.x, n01.z, n23.x, n23.z}, isd[4] = {n01.y, n01.w, n23.y, n23.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int q = 64 * W + 4 * i + j;
        if (q < SGS_NIN) {
          const int k = q < 243 ? q - 9 * N0 : TH + q - 243;
          v[j] = (u[k < 72 ? k : 0] - mu[j]) * isd[j];
          gm = fmaxf(gm, fabsf(v[j]));
        } else {
          v[j] = 0.f;
        }
      }
      As[16 * W + i][lane] = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
    }
    return gm;
  }
};

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8))) k_sgs_mlp_fused(FusedArgs a) {
  __shared__ uint2 As[SGS_KIN / 4][FT];        /* features     [k / 4][cell][4] */
  __shared__ uint2 Hs[2][SGS_H / 4][FT];       /* activations, likewise */
  __shared__ float gms[2][4][FT], rhos[2][FT]; /* by tile parity: each wave's largest feature, rho */
  __shared__ __align__(16) float cf[4][SGS_H]; /* biases of layers 1-3; of layer 4, output std, output mean */
  __shared__ __align__(16) float2 nrm[SGS_KIN];  /* feature normalisation: mean, 1 / std */
  __shared__ unsigned cnts[4][2];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  /* weights as the left operand (its row = output column): lane holds W[k = 16 kb + 4 lk + v][n],
   * n = lr of its wave's block (W4: n = lr) */
  bf16x4 w1[16], w2[4], w3[4], w4[4];
  const int ncol = 16 * wave + lr;
#pragma unroll
  for (int kb = 0; kb < 16; ++kb) {
    const int k = 16 * kb + 4 * lk;
    w1[kb] = bf16x4{(short)f2bf(a.w[OW1_ + (long)(k + 0) * SGS_H + ncol]), (short)f2bf(a.w[OW1_ + (long)(k + 1) * SGS_H + ncol]),
                    (short)f2bf(a.w[OW1_ + (long)(k + 2) * SGS_H + ncol]), (short)f2bf(a.w[OW1_ + (long)(k + 3) * SGS_H + ncol])};
  }
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int k = 16 * kb + 4 * lk;
    w2[kb] = bf16x4{(short)f2bf(a.w[OW2_ + (k + 0) * SGS_H + ncol]), (short)f2bf(a.w[OW2_ + (k + 1) * SGS_H + ncol]),
                    (short)f2bf(a.w[OW2_ + (k + 2) * SGS_H + ncol]), (short)f2bf(a.w[OW2_ + (k + 3) * SGS_H + ncol])};
    w3[kb] = bf16x4{(short)f2bf(a.w[OW3_ + (k + 0) * SGS_H + ncol]), (short)f2bf(a.w[OW3_ + (k + 1) * SGS_H + ncol]),
                    (short)f2bf(a.w[OW3_ + (k + 2) * SGS_H + ncol]), (short)f2bf(a.w[OW3_ + (k + 3) * SGS_H + ncol])};
    w4[kb] = bf16x4{(short)f2bf(a.w[OW4_ + (k + 0) * SGS_KOUT + lr]), (short)f2bf(a.w[OW4_ + (k + 1) * SGS_KOUT + lr]),
                    (short)f2bf(a.w[OW4_ + (k + 2) * SGS_KOUT + lr]), (short)f2bf(a.w[OW4_ + (k + 3) * SGS_KOUT + lr])};
  }
  for (int i = tid; i < SGS_KIN; i += 256) nrm[i] = make_float2(a.mu[i], a.isd[i]);
  for (int i = tid; i < SGS_H; i += 256) {
    cf[0][i] = a.w[OB1_ + i];
    cf[1][i] = a.w[OB2_ + i];
    cf[2][i] = a.w[OB3_ + i];
    cf[3][i] = i < SGS_KOUT ? a.w[OB4_ + i] : i < 2 * SGS_KOUT ? a.ysd[i - SGS_KOUT] : i < 3 * SGS_KOUT ? a.ymu[i - 2 * SGS_KOUT] : 0.f;
  }
  float u[72], rho = 0.f;                /* the wave's raw features of a tile (TileFeatures), rho (wave 0) */
#pragma unroll
  for (int i = 0; i < 72; ++i) u[i] = 0.f;
  TileCell p(a, (long)blockIdx.x * FT + lane);
  const long step = (long)gridDim.x * FT;
  int sx, sy, sz;
  cell_xyz(step, a.Nx, a.Ny, sx, sy, sz);
  auto load = [&]() {
    if (wave == 0) TileFeatures<0>::load(a, p, u, rho);
    else if (wave == 1) TileFeatures<1>::load(a, p, u, rho);
    else if (wave == 2) TileFeatures<2>::load(a, p, u, rho);
    else TileFeatures<3>::load(a, p, u, rho);
  };
  auto put = [&](int buf) {
    float gm;
    if (wave == 0) gm = TileFeatures<0>::put(nrm, u, As, lane);
    else if (wave == 1) gm = TileFeatures<1>::put(nrm, u, As, lane);
    else if (wave == 2) gm = TileFeatures<2>::put(nrm, u, As, lane);
    else gm = TileFeatures<3>::put(nrm, u, As, lane);
    gms[buf][wave][lane] = gm;
    if (wave == 0) rhos[buf][lane] = rho;
  };
  f32x4 acc[4];
  auto product = [&](const uint2 (*src)[FT], const bf16x4 *w, int nkb) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < nkb; ++kb) {
      if (kb > 0 && kb % 4 == 0) __builtin_amdgcn_sched_barrier(0);   /* 16 operand reads in flight, no more registers */
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
        acc[rb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w[kb], ld_frag(&src[4 * kb + lk][16 * rb + lr]), acc[rb], 0, 0, 0);
    }
  };
  auto store_act = [&](int buf, int layer) {
    const float4 b4 = *(const float4 *)&cf[layer][16 * wave + 4 * lk];
    const float b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
      Hs[buf][4 * wave + lk][16 * rb + lr] = make_uint2(f2bf2(gelu(acc[rb][0] + b[0]), gelu(acc[rb][1] + b[1])),
                                                        f2bf2(gelu(acc[rb][2] + b[2]), gelu(acc[rb][3] + b[3])));
  };
  unsigned ncnt = 0, npass = 0;          /* cells finished and passing, by lanes 0..15 of each wave */
  int buf = 0;
  if ((int)blockIdx.x < a.ntiles) {
    load();
    __syncthreads();                     /* nrm, cf */
    put(0);
  }
  for (int tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x, buf ^= 1) {
    const int next = tile + gridDim.x;
    __syncthreads();
    if (next < a.ntiles) {
      p.advance(a, step, sx, sy, sz);
      load();
    }
    product(As, w1, 16);
    store_act(0, 0);
    __syncthreads();
    if (next < a.ntiles) put(buf ^ 1);
    product(Hs[0], w2, 4);
    store_act(1, 1);
    __syncthreads();
    product(Hs[1], w3, 4);
    store_act(0, 2);
    __syncthreads();
    /* ---- layer 4 and finish: wave w the cell block w, the lane's outputs 4 lk .. 4 lk + 3 ---- */
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      o = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w4[kb], ld_frag(&Hs[0][4 * kb + lk][16 * wave + lr]), o, 0, 0, 0);
    const int r = 16 * wave + lr;
    const long c = (long)tile * FT + r;
    const float rc = rhos[buf][r];
    float t[4];
    const float *b4 = &cf[3][4 * lk], *ysd = b4 + SGS_KOUT, *ymu = ysd + SGS_KOUT;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float y = o[v] + b4[v];
      t[v] = y * ysd[v] + ymu[v];
    }
    const float t4 = __shfl_down(t[0], 16), t5 = __shfl_down(t[1], 16);
    if (c < a.ncell) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (4 * lk + v < SGS_NOUT) a.tauL[(4 * lk + v) * a.ncell + c] = rc * t[v];
      if (lk == 0) {
        const float gm = fmaxf(fmaxf(gms[buf][0][r], gms[buf][1][r]), fmaxf(gms[buf][2][r], gms[buf][3][r]));
        const bool ok = gm <= a.gate && sgs_realizable(t[0], t[1], t[2], t[3], t4, t5);
        a.mask[c] = ok ? 1 : 0;
        npass += ok ? 1u : 0u;
        ++ncnt;
      }
    }
  }
  /* one pair of atomics per work-group */
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    ncnt += __shfl_xor(ncnt, off);
    npass += __shfl_xor(npass, off);
  }
  if (lane == 0) {
    cnts[wave][0] = ncnt;
    cnts[wave][1] = npass;
  }
  __syncthreads();
  if (tid == 0 && (int)blockIdx.x < a.ntiles) {
    atomicAdd(&a.count[0], (unsigned long long)(cnts[0][0] + cnts[1][0] + cnts[2][0] + cnts[3][0]));
    atomicAdd(&a.count[1], (unsigned long long)(cnts[0][1] + cnts[1][1] + cnts[2][1] + cnts[3][1]));
  }
}

/* The learned stresses replace the TKE closure's in the momentum and theta SGS divergence
 * (cuda_sgsTurbDevice.cu:447-547) on every face or edge whose adjacent cells all pass:
 * the stage output gets coefdt * (-div(tau_L - tau_TKE)) over those faces, tau_L averaged
 * from the adjacent cell centres to the reference's face/edge positions, tau_TKE as the
 * physics stage emitted it (fields 11, 21, 31, 32, 22, 33, theta1..3 at each cell's low-side
 * faces).  The surface faces (the surface layer's fluxes) and the lid keep the TKE
 * closure's values.  One thread per cell. */
__global__ void __launch_bounds__(256) k_sgs_correct(float *Sout, const float *tauT, const float *tauL,
                                                     const unsigned char *mask, long fs, long ps, int Nx, int Ny, int Nz,
                                                     int P, float dXi, float dYi, float dZi, const float *j33,
                                                     float coefdt) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long ncell = (long)Nx * Ny * Nz;
  if (c >= ncell) return;
  int x, y, z;
  cell_xyz(c, Nx, Ny, x, y, z);
  /* Places of the cell and its neighbours as steps from the cell, wrapped laterally and clamped at
   * the ground and the lid (whose faces below are 0): i in the learned arrays, j in the state's.
   * 32 bits, modulo 2^32: the host keeps the learned closure's grids below 2^31 cells and the
   * device state's fields below 4 GiB. */
  const bool lid = z + 1 >= Nz, gnd = z == 0;
  const int nxy = Nx * Ny;
  const int ix[3] = {x == 0 ? Nx - 1 : -1, 0, x == Nx - 1 ? 1 - Nx : 1};
  const int iy[3] = {y == 0 ? nxy - Nx : -Nx, 0, y == Ny - 1 ? Nx - nxy : Nx};
  const int iz[3] = {gnd ? 0 : -nxy, 0, lid ? 0 : nxy};
  const unsigned o = (unsigned)z * (unsigned)ps + (unsigned)y * (unsigned)P + (unsigned)x;
  auto cid = [&](int dx, int dy, int dz) -> unsigned { return (unsigned)((int)c + ix[dx + 1] + iy[dy + 1] + iz[dz + 1]); };
  auto pass = [&](int dx, int dy, int dz) -> bool { return mask[cid(dx, dy, dz)] != 0; };
  /* Every value is loaded whatever the masks say: the loads of a cell are in flight together, where
   * tests between them made a chain.  128 x 128 x 48: 54 -> 28 us. */
  auto T = [&](int e, int dx, int dy, int dz) -> float {
    const int j = (int)o + ix[dx + 1] + (dy < 0 ? (y == 0 ? (Ny - 1) * P : -P) : dy > 0 ? (y == Ny - 1 ? (1 - Ny) * P : P) : 0) +
                  (dz > 0 && !lid ? (int)ps : 0);
    return tauT[(size_t)e * (size_t)fs + (unsigned)j];
  };
  /* Delta tau of emitted field e, learned component q, at the low-side face (edge) of the cell at
   * (+dx, +dy, +dz): the mean over the cell and its low neighbours along the directions, or 0 where
   * one of them does not pass */
  auto L = [&](int q, int dx, int dy, int dz) -> float { return tauL[(size_t)q * (size_t)ncell + cid(dx, dy, dz)]; };
  auto face = [&](int e, int q, int ax, int ay, int az, int dx, int dy, int dz) -> float {
    const float s = L(q, dx, dy, dz) + L(q, dx - ax, dy - ay, dz - az);
    const bool ok = pass(dx, dy, dz) && pass(dx - ax, dy - ay, dz - az);
    const float d = s / 2.f - T(e, dx, dy, dz);
    return ok ? d : 0.f;
  };
  /* edges: k = 1 the first direction's low neighbour, k = 2 the second's */
  auto edge = [&](int e, int q, int ax, int ay, int bx, int by, int bz, int dx, int dy, int dz) -> float {
    float s = L(q, dx, dy, dz) + L(q, dx - ax, dy - ay, dz);
    s += L(q, dx - bx, dy - by, dz - bz);
    s += L(q, dx - ax - bx, dy - ay - by, dz - bz);
    const bool ok = pass(dx, dy, dz) && pass(dx - ax, dy - ay, dz) && pass(dx - bx, dy - by, dz - bz) &&
                    pass(dx - ax - bx, dy - ay - by, dz - bz);
    const float d = s / 4.f - T(e, dx, dy, dz);
    return ok ? d : 0.f;
  };
  const float zdz = j33[z] * dZi;
  const float t11 = face(0, 0, 1, 0, 0, 0, 0, 0), t22 = face(4, 1, 0, 1, 0, 0, 0, 0);
  const float h1 = face(6, 6, 1, 0, 0, 0, 0, 0), h2 = face(7, 7, 0, 1, 0, 0, 0, 0);
  const float t21 = edge(1, 3, 1, 0, 0, 1, 0, 0, 0, 0);
  const float d11 = dXi * (face(0, 0, 1, 0, 0, 1, 0, 0) - t11);
  const float d21x = dXi * (edge(1, 3, 1, 0, 0, 1, 0, 1, 0, 0) - t21);
  const float d21y = dYi * (edge(1, 3, 1, 0, 0, 1, 0, 0, 1, 0) - t21);
  const float d22 = dYi * (face(4, 1, 0, 1, 0, 0, 1, 0) - t22);
  const float dh1 = dXi * (face(6, 6, 1, 0, 0, 1, 0, 0) - h1);
  const float dh2 = dYi * (face(7, 7, 0, 1, 0, 0, 1, 0) - h2);
  /* vertical directions: 0 on the surface's and the lid's faces and edges */
  auto lo = [&](float v) { return gnd ? 0.f : v; };
  auto hi = [&](float v) { return lid ? 0.f : v; };
  const float t31 = lo(edge(2, 4, 1, 0, 0, 0, 1, 0, 0, 0)), t32 = lo(edge(3, 5, 0, 1, 0, 0, 1, 0, 0, 0));
  const float t33 = lo(face(5, 2, 0, 0, 1, 0, 0, 0)), h3 = lo(face(8, 8, 0, 0, 1, 0, 0, 0));
  const float d31x = dXi * (lo(edge(2, 4, 1, 0, 0, 0, 1, 1, 0, 0)) - t31);
  const float d31z = zdz * (hi(edge(2, 4, 1, 0, 0, 0, 1, 0, 0, 1)) - t31);
  const float d32y = dYi * (lo(edge(3, 5, 0, 1, 0, 0, 1, 0, 1, 0)) - t32);
  const float d32z = zdz * (hi(edge(3, 5, 0, 1, 0, 0, 1, 0, 0, 1)) - t32);
  const float d33 = zdz * (hi(face(5, 2, 0, 0, 1, 0, 0, 1)) - t33);
  const float dh3 = zdz * (hi(face(8, 8, 0, 0, 1, 0, 0, 1)) - h3);
  Sout[fs + o] -= coefdt * (d11 + d21y + d31z);
  Sout[2 * fs + o] -= coefdt * (d21x + d22 + d32z);
  Sout[3 * fs + o] -= coefdt * (d31x + d32y + d33);
  Sout[4 * fs + o] -= coefdt * (dh1 + dh2 + dh3);
}

/* count[0] += cells, count[1] += cells whose mask is set (unfused path): grid-stride, one pair
 * of atomics per work-group */
__global__ void __launch_bounds__(256) k_mask_count(const unsigned char *mask, long n, unsigned long long *count) {
  unsigned long long a = 0, p = 0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    ++a;
    p += mask[i] ? 1u : 0u;
  }
  for (int off = 32; off > 0; off >>= 1) { a += __shfl_xor(a, off); p += __shfl_xor(p, off); }
  __shared__ unsigned long long part[4][2];
  if ((threadIdx.x & 63) == 0) { part[threadIdx.x >> 6][0] = a; part[threadIdx.x >> 6][1] = p; }
  __syncthreads();
  if (threadIdx.x == 0) {
    a = part[0][0] + part[1][0] + part[2][0] + part[3][0];
    p = part[0][1] + part[1][1] + part[2][1] + part[3][1];
    if (a) { atomicAdd(&count[0], a); atomicAdd(&count[1], p); }
  }
}

}  // namespace fe
