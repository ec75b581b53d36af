/*
 * fe_sgs.hip -- host side of the learned SGS closure (kernels in fe_sgs_kernels.hip).
 *
 * Training data: fine-grid runs of the plain model itself.  fe_sgs_collect box-filters the
 * current device state of a fine run (and the SGS stresses its physics stage emitted) by
 * an integer factor, and appends the filtered field's 250 features and its Favre-filtered
 * SGS stresses and heat fluxes (the targets) to a device-resident training set.
 * fe_sgs_prepare normalises the set (feature and target means and standard deviations),
 * fe_sgs_train fits the MLP with Adam on mini-batches (BF16 MFMA forward and backward
 * GEMMs, FP32 accumulation, FP32 master weights and moments).
 *
 * Inference: with fe_sgs_enable the physics stage of the plain model evaluates the network
 * on its stage input in chunks of cells, gates each cell (input distribution and
 * realizability), runs the fused physics stage with the TKE closure as usual while it
 * emits that closure's stresses, and then replaces them by the learned ones in the
 * momentum and theta flux divergence wherever the adjacent cells passed
 * (k_sgs_correct).  Elsewhere, and in the TKE equation, the TKE closure stays: it is the
 * fallback.
 */

namespace {

/* parameter vector layout (fe_sgs_kernels.hip) */
constexpr long OW1 = OW1_, OB1 = OB1_, OW2 = OW2_, OB2 = OB2_, OW3 = OW3_, OB3 = OB3_, OW4 = OW4_, OB4 = OB4_,
               NPARAM = NPARAM_;
constexpr long SGS_CHUNK = 262144;   /* cells per inference chunk */
constexpr int GSPLIT = 64, GSPLIT_MIN = 128;   /* parts of a weight gradient, rows of the smallest (gemm_dw) */

struct Sgs {
  float *w = nullptr, *gw = nullptr, *am = nullptr, *av = nullptr;
  int adam_t = 0;
  float *xmu = nullptr, *xisd = nullptr, *ymu = nullptr, *ysd = nullptr;   /* 256, 256, 16, 16 */
  bool have_norm = false, have_w = false;
  float *Xs = nullptr, *Ts = nullptr;                                      /* training set */
  long ns = 0, cap = 0;
  float *Sc = nullptr;                                                     /* last filtered state */
  float *Tf = nullptr, *tlast = nullptr;                                   /* filter-only targets, last targets */
  long ntf_cap = 0;
  long nsc = 0, nsc_cap = 0;
  int sc_dims[3] = {0, 0, 0};
  float *j33c = nullptr;
  int nj33c = 0;
  /* row buffers for a batch or an inference chunk */
  long rows_cap = 0;
  float *Xb = nullptr, *Tb = nullptr, *Z[3] = {nullptr, nullptr, nullptr}, *Aa[3] = {nullptr, nullptr, nullptr};
  float *Y = nullptr, *dY = nullptr, *dA0 = nullptr, *dA1 = nullptr;
  float *part = nullptr;                                                   /* partial weight gradients (gemm_dw) */
  int *idx = nullptr;
  long idx_cap = 0;
  double *dloss = nullptr;
  /* inference on the plain model */
  int on = 0;
  float gate = 6.f;
  float *tauL = nullptr, *gmax = nullptr, *j33 = nullptr, *grad = nullptr;
  unsigned char *mask = nullptr;
  int fused = 1;                          /* fused inference (k_sgs_grad + k_sgs_mlp_fused) */
  int fused_wg = 0;                       /* persistent work-groups of the fused kernel */
  long ncell_cap = 0;
  unsigned long long *dcount = nullptr;   /* cells evaluated, cells passing (device) */
} G;

int sgs_rows(long rows) {
  if (rows <= G.rows_cap) return FE_OK;
  float **b[] = {&G.Xb, &G.Tb, &G.Z[0], &G.Z[1], &G.Z[2], &G.Aa[0], &G.Aa[1], &G.Aa[2], &G.Y, &G.dY, &G.dA0, &G.dA1};
  for (auto p : b) if (*p) { HIPCHK(hipFree(*p)); *p = nullptr; }
  HIPCHK(hipMalloc(&G.Xb, rows * SGS_KIN * sizeof(float)));
  HIPCHK(hipMalloc(&G.Tb, rows * SGS_KOUT * sizeof(float)));
  for (int l = 0; l < 3; ++l) {
    HIPCHK(hipMalloc(&G.Z[l], rows * SGS_H * sizeof(float)));
    HIPCHK(hipMalloc(&G.Aa[l], rows * SGS_H * sizeof(float)));
  }
  HIPCHK(hipMalloc(&G.Y, rows * SGS_KOUT * sizeof(float)));
  HIPCHK(hipMalloc(&G.dY, rows * SGS_KOUT * sizeof(float)));
  HIPCHK(hipMalloc(&G.dA0, rows * SGS_H * sizeof(float)));
  HIPCHK(hipMalloc(&G.dA1, rows * SGS_H * sizeof(float)));
  G.rows_cap = rows;
  return FE_OK;
}

int sgs_params_alloc() {
  if (G.w) return FE_OK;
  float **p[] = {&G.w, &G.gw, &G.am, &G.av};
  for (auto q : p) {
    HIPCHK(hipMalloc(q, NPARAM * sizeof(float)));
    HIPCHK(hipMemset(*q, 0, NPARAM * sizeof(float)));
  }
  float **n[] = {&G.xmu, &G.xisd, &G.ymu, &G.ysd};
  for (auto q : n) {
    HIPCHK(hipMalloc(q, SGS_KIN * sizeof(float)));
    HIPCHK(hipMemset(*q, 0, SGS_KIN * sizeof(float)));
  }
  if (!G.dloss) HIPCHK(hipMalloc(&G.dloss, sizeof(double)));
  if (!G.part) HIPCHK(hipMalloc(&G.part, (size_t)GSPLIT * ((size_t)SGS_KIN * SGS_H + SGS_H) * sizeof(float)));
  return FE_OK;
}

hipStream_t sgs_stream() { return D.stream; }
inline dim3 blocks(long n) { return dim3((unsigned)((n + 255) / 256)); }

/* C = A B with the epilogue of g (its epi, bias, act, Z) */
int gemm(GemmArgs g) {
  if (g.M <= 0) return FE_OK;
  g.kchunk = (g.K + GK - 1) / GK * GK;
  dim3 grid((unsigned)((g.M + GT - 1) / GT), (unsigned)((g.N + GT - 1) / GT));
  hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, sgs_stream(), g);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

/* Gradient of a layer's weights [nin][nout] and, after them, biases [nout] into out:
 * in^T dZ and the column sums of dZ over M rows.  Split over the rows into at most GSPLIT
 * work-groups per output tile of at least 128 rows each (four K steps: below that the partial
 * sums cost more than the steps they replace); 8192 rows: 64 parts, one part 1350 us. */
int gemm_dw(const float *in, int nin, const float *dZ, int nout, long M, float *out) {
  GemmArgs g{in, 1, nin, dZ, nout, 1, out, nout, nin, nout, (int)M};
  const long n = (long)nin * nout + nout;
  const long chunk = std::max<long>(GSPLIT_MIN, (M + GSPLIT - 1) / GSPLIT);
  g.kchunk = (int)((chunk + GK - 1) / GK * GK);
  const int nz = (int)((M + g.kchunk - 1) / g.kchunk);
  if (nz > 1) { g.C = G.part; g.zstride = n; }
  g.csum = g.C + (long)nin * nout;
  dim3 grid((unsigned)((nin + GT - 1) / GT), (unsigned)((nout + GT - 1) / GT), (unsigned)nz);
  hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, sgs_stream(), g);
  if (nz > 1) hipLaunchKernelGGL(k_gemm_reduce, blocks(n), dim3(256), 0, sgs_stream(), (const float *)G.part, nz, n, out);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

/* forward of M rows of X (normalised features) into G.Y; activations kept in G.Z/G.Aa */
int mlp_forward(const float *X, long M) {
  int rc;
  const float *in = X;
  int K = SGS_KIN;
  const long ow[3] = {OW1, OW2, OW3}, ob[3] = {OB1, OB2, OB3};
  for (int l = 0; l < 3; ++l) {
    GemmArgs g{in, K, 1, G.w + ow[l], SGS_H, 1, G.Z[l], SGS_H, (int)M, SGS_H, K};
    g.epi = GEMM_BIAS_GELU; g.bias = G.w + ob[l]; g.act = G.Aa[l];
    if ((rc = gemm(g))) return rc;
    in = G.Aa[l];
    K = SGS_H;
  }
  GemmArgs g{in, SGS_H, 1, G.w + OW4, SGS_KOUT, 1, G.Y, SGS_KOUT, (int)M, SGS_KOUT, SGS_H};
  g.epi = GEMM_BIAS; g.bias = G.w + OB4;
  return gemm(g);
}

/* backward of the loss gradient G.dY (M rows) into G.gw */
int mlp_backward(const float *X, long M) {
  int rc;
  /* output layer */
  if ((rc = gemm_dw(G.Aa[2], SGS_H, G.dY, SGS_KOUT, M, G.gw + OW4))) return rc;
  const long ow[3] = {OW1, OW2, OW3};
  const float *dY = G.dY, *w = G.w + OW4;
  int nout = SGS_KOUT;
  float *dZ = G.dA0, *dZn = G.dA1;
  for (int l = 2; l >= 0; --l) {
    /* dZ of layer l: (dY W^T) GELU'(Z) */
    GemmArgs g{dY, nout, 1, w, 1, nout, dZ, SGS_H, (int)M, SGS_H, nout};
    g.epi = GEMM_GELU_BACK; g.Z = G.Z[l];
    if ((rc = gemm(g))) return rc;
    if ((rc = gemm_dw(l > 0 ? G.Aa[l - 1] : X, l > 0 ? SGS_H : SGS_KIN, dZ, SGS_H, M, G.gw + ow[l]))) return rc;
    dY = dZ;
    w = G.w + ow[l];
    nout = SGS_H;
    std::swap(dZ, dZn);
  }
  return FE_OK;
}

int sgs_loss_grad(const float *T, long M) {
  hipLaunchKernelGGL(k_loss_grad, blocks(M * SGS_KOUT), dim3(256), 0, sgs_stream(), (const float *)G.Y, T, M, SGS_KOUT,
                     SGS_NOUT, G.dY, G.dloss);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

/* Learned stresses of the model's stage input Sin (every cell): G.tauL, G.mask.  Fused: one
 * gradient pass and one persistent network kernel; otherwise in chunks through the feature,
 * GEMM and activation kernels of the training path (the same bits, kept as the reference). */
int sgs_infer(const float *Sin) {
  int rc;
  const long ncell = (long)D.Nx * D.Ny * D.Nz;
  hipStream_t s = sgs_stream();
  if (G.fused) {
    if (!G.fused_wg) {
      int dev = 0, ncu = 256, occ = 1;
      hipDeviceProp_t pr;
      if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&pr, dev) == hipSuccess && pr.multiProcessorCount > 0)
        ncu = pr.multiProcessorCount;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_sgs_mlp_fused, 256, 0) != hipSuccess || occ < 1) occ = 1;
      G.fused_wg = ncu * occ;
    }
    FeatArgs fa{Sin, D.fs, D.ps, D.Nx, D.Ny, D.Nz, D.P, dXi, dYi, dZi, G.j33, nullptr, nullptr, nullptr, nullptr, 0, ncell};
    hipLaunchKernelGGL(k_sgs_grad, blocks(ncell), dim3(256), 0, s, fa, G.grad);
    const int ntiles = (int)((ncell + FT - 1) / FT);
    FusedArgs ua{G.grad, D.Nx, D.Ny, D.Nz, G.xmu, G.xisd, G.w, G.ymu, G.ysd, G.gate, Sin, D.ps, D.P, G.tauL, ncell, G.mask,
                 G.dcount, ntiles};
    hipLaunchKernelGGL(k_sgs_mlp_fused, dim3((unsigned)std::min(ntiles, G.fused_wg)), dim3(256), 0, s, ua);
    HIPCHK(hipGetLastError());
    return FE_OK;
  }
  if ((rc = sgs_rows(std::min(ncell, SGS_CHUNK)))) return rc;
  for (long c0 = 0; c0 < ncell; c0 += SGS_CHUNK) {
    const long nc = std::min(SGS_CHUNK, ncell - c0);
    FeatArgs fa{Sin, D.fs, D.ps, D.Nx, D.Ny, D.Nz, D.P, dXi, dYi, dZi, G.j33, G.xmu, G.xisd, G.Xb, G.gmax, c0, nc};
    hipLaunchKernelGGL(k_sgs_features, blocks(nc), dim3(256), 0, s, fa);
    if ((rc = mlp_forward(G.Xb, nc))) return rc;
    hipLaunchKernelGGL(k_sgs_finish, blocks(nc), dim3(256), 0, s, (const float *)G.Y, (const float *)G.ymu, (const float *)G.ysd,
                       (const float *)G.gmax, G.gate, Sin, D.fs, D.ps, D.Nx, D.Ny, D.P, c0, nc, G.tauL, ncell, G.mask);
    HIPCHK(hipGetLastError());
  }
  hipLaunchKernelGGL(k_mask_count, dim3((unsigned)std::min<long>(1024, (ncell + 255) / 256)), dim3(256), 0, s,
                     (const unsigned char *)G.mask, ncell, G.dcount);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

bool sgs_active() { return G.on != 0; }

int sgs_correct(float *Sout, float coefdt) {
  hipLaunchKernelGGL(k_sgs_correct, blocks((long)D.Nx * D.Ny * D.Nz), dim3(256), 0, sgs_stream(), Sout, (const float *)D.tau,
                     (const float *)G.tauL, (const unsigned char *)G.mask, D.fs, D.ps, D.Nx, D.Ny, D.Nz, D.P, dXi, dYi, dZi,
                     (const float *)G.j33, coefdt);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

int sgs_free_all() {
  float **p[] = {&G.w, &G.gw, &G.am, &G.av, &G.xmu, &G.xisd, &G.ymu, &G.ysd, &G.Xs, &G.Ts, &G.Sc, &G.j33c, &G.Xb, &G.Tb,
                 &G.Z[0], &G.Z[1], &G.Z[2], &G.Aa[0], &G.Aa[1], &G.Aa[2], &G.Y, &G.dY, &G.dA0, &G.dA1, &G.tauL, &G.gmax, &G.j33,
                 &G.grad, &G.Tf, &G.part};
  if (D.stream) HIPCHK(hipStreamSynchronize(D.stream));
  for (auto q : p) if (*q) { HIPCHK(hipFree(*q)); *q = nullptr; }
  if (G.idx) HIPCHK(hipFree(G.idx));
  if (G.mask) HIPCHK(hipFree(G.mask));
  if (G.dcount) HIPCHK(hipFree(G.dcount));
  if (G.dloss) HIPCHK(hipFree(G.dloss));
  G = Sgs();
  return FE_OK;
}


/* Box-filter the current device state of the plain model by fac in every direction (the grid
 * must divide, flat terrain) together with the SGS stresses its last batch emitted
 * (hydroSubGridWrite = 1): the filtered state into G.Sc and the Favre-filtered SGS targets
 * either appended to the training set, with the filtered field's features (append), or into a
 * separate buffer (the filtered profiles of an evaluation run).  Returns the number of samples
 * in the set (append) or of filtered cells, or a negative FE_ERR_* code. */
int sgs_filter(int fac, bool append) {
  int rc;
  if (!D.timeint) return -FE_ERR_STATE;
  if (!D.tau) {
    fprintf(stderr, "fe_sgs_collect: the model emits no SGS stresses (hydroSubGridWrite = 0)\n");
    return -FE_ERR_UNSUPPORTED;
  }
  if (fac < 1 || D.Nx % fac || D.Ny % fac || D.Nz % fac) return -FE_ERR_UNSUPPORTED;
  if (D.terrain) return -FE_ERR_TERRAIN;                              /* the box filter assumes a flat grid */
  if ((long)D.Nx * D.Ny * D.Nz > (long)INT_MAX) return -FE_ERR_UNSUPPORTED;   /* 32-bit cell indexing */
  const float j0 = D.hprof[(size_t)3 * PROW + PR_J33];
  for (int z = 0; z < D.Nz; ++z)
    if (D.hprof[(size_t)(z + 3) * PROW + PR_J33] != j0) {
      fprintf(stderr, "fe_sgs_collect: the filter needs a uniform vertical grid\n");
      return -FE_ERR_UNSUPPORTED;
    }
  if ((rc = sgs_params_alloc())) return -rc;
  const int nxc = D.Nx / fac, nyc = D.Ny / fac, nzc = D.Nz / fac;
  const long nc = (long)nxc * nyc * nzc;
  float *tdst = nullptr;
  if (append) {
    if (G.ns + nc > G.cap) {
      const long cap = std::max(2 * G.cap, G.ns + nc);
      float *X = nullptr, *T = nullptr;
      if (hipMalloc(&X, cap * SGS_KIN * sizeof(float)) != hipSuccess) return -FE_ERR_ALLOC;
      if (hipMalloc(&T, cap * SGS_KOUT * sizeof(float)) != hipSuccess) { (void)hipFree(X); return -FE_ERR_ALLOC; }
      if (G.ns) {
        if (hipMemcpy(X, G.Xs, G.ns * SGS_KIN * sizeof(float), hipMemcpyDeviceToDevice) != hipSuccess ||
            hipMemcpy(T, G.Ts, G.ns * SGS_KOUT * sizeof(float), hipMemcpyDeviceToDevice) != hipSuccess)
          return -FE_ERR_HIP;
      }
      if (G.Xs) (void)hipFree(G.Xs);
      if (G.Ts) (void)hipFree(G.Ts);
      G.Xs = X; G.Ts = T; G.cap = cap;
    }
    tdst = G.Ts + G.ns * SGS_KOUT;
  } else {
    if (nc > G.ntf_cap) {
      if (G.Tf) (void)hipFree(G.Tf);
      G.Tf = nullptr;
      if (hipMalloc(&G.Tf, nc * SGS_KOUT * sizeof(float)) != hipSuccess) return -FE_ERR_ALLOC;
      G.ntf_cap = nc;
    }
    tdst = G.Tf;
  }
  if (5 * nc > G.nsc_cap) {
    if (G.Sc) (void)hipFree(G.Sc);
    if (hipMalloc(&G.Sc, 5 * nc * sizeof(float)) != hipSuccess) return -FE_ERR_ALLOC;
    G.nsc_cap = 5 * nc;
  }
  if (nzc > G.nj33c) {
    if (G.j33c) (void)hipFree(G.j33c);
    if (hipMalloc(&G.j33c, nzc * sizeof(float)) != hipSuccess) return -FE_ERR_ALLOC;
    G.nj33c = nzc;
  }
  {
    std::vector<float> j(nzc, j0);
    if (hipMemcpy(G.j33c, j.data(), nzc * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) return -FE_ERR_HIP;
  }
  hipStream_t s = sgs_stream();
  hipLaunchKernelGGL(k_sgs_filter, blocks(nc), dim3(256), 0, s, (const float *)D.S[0], (const float *)D.tau, D.fs, D.ps, D.P, nxc,
                     nyc, nzc, fac, G.Sc, tdst);
  if (append) {
    const long psc = (long)nxc * nyc;
    FeatArgs fa{G.Sc, psc * nzc, psc, nxc, nyc, nzc, nxc, dXi / fac, dYi / fac, dZi / fac, G.j33c, nullptr, nullptr,
                G.Xs + G.ns * SGS_KIN, nullptr, 0, nc};
    hipLaunchKernelGGL(k_sgs_features, blocks(nc), dim3(256), 0, s, fa);
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return -FE_ERR_HIP;
  if (append) G.ns += nc;
  G.tlast = tdst;
  G.nsc = 5 * nc;
  G.sc_dims[0] = nxc; G.sc_dims[1] = nyc; G.sc_dims[2] = nzc;
  return (int)(append ? G.ns : nc);
}

}  // namespace

extern "C" {

/* Box-filter the current device state (and the SGS stresses its last batch emitted) by fac and
 * append the filtered field's features and SGS targets to the training set.  Returns the number
 * of samples in the set, or a negative FE_ERR_* code. */
int fe_sgs_collect(int fac) { return sgs_filter(fac, true); }

/* The same filter without touching the training set: the filtered state and targets of an
 * evaluation run (read them with fe_sgs_filtered).  Returns the filtered cell count. */
int fe_sgs_filter(int fac) { return sgs_filter(fac, false); }

/* The filtered state of the last filter call ([5][zc][yc][xc]: rho, rho*u, rho*v, rho*w,
 * rho*theta) and its targets ([zc][yc][xc][16]: kinematic until fe_sgs_prepare normalises a
 * collected set). */
int fe_sgs_filtered(float *state, long nstate, float *targets, long ntarget) {
  if (!G.Sc || G.nsc == 0 || !G.tlast) return FE_ERR_STATE;
  const long nc = G.nsc / 5;
  if (state) {
    if (nstate != G.nsc) return FE_ERR_UNSUPPORTED;
    HIPCHK(hipMemcpy(state, G.Sc, nstate * sizeof(float), hipMemcpyDeviceToHost));
  }
  if (targets) {
    if (ntarget != nc * SGS_KOUT) return FE_ERR_UNSUPPORTED;
    HIPCHK(hipMemcpy(targets, G.tlast, ntarget * sizeof(float), hipMemcpyDeviceToHost));
  }
  return FE_OK;
}

/* Normalisation of the collected set: feature and target means and standard deviations
 * (FP64 sums on the device), then the set in place. */
int fe_sgs_prepare(void) {
  if (G.ns < 2 || G.have_norm) return FE_ERR_STATE;
  hipStream_t s = sgs_stream();
  double *st = nullptr;
  HIPCHK(hipMalloc(&st, 2 * SGS_KIN * sizeof(double)));
  std::vector<double> h(2 * SGS_KIN);
  std::vector<float> mu(SGS_KIN, 0.f), isd(SGS_KIN, 0.f), ymu(SGS_KIN, 0.f), ysd(SGS_KIN, 0.f);
  hipLaunchKernelGGL(k_colstats, dim3(SGS_KIN), dim3(256), 0, s, (const float *)G.Xs, G.ns, SGS_KIN, st);
  HIPCHK(hipMemcpyAsync(h.data(), st, 2 * SGS_KIN * sizeof(double), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  for (int q = 0; q < SGS_NIN; ++q) {
    const double m = h[2 * q] / G.ns, var = std::max(0.0, h[2 * q + 1] / G.ns - m * m);
    mu[q] = (float)m;
    isd[q] = var > 0.0 ? (float)(1.0 / sqrt(var)) : 0.f;
  }
  hipLaunchKernelGGL(k_colstats, dim3(SGS_KOUT), dim3(256), 0, s, (const float *)G.Ts, G.ns, SGS_KOUT, st);
  HIPCHK(hipMemcpyAsync(h.data(), st, 2 * SGS_KOUT * sizeof(double), hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  for (int q = 0; q < SGS_NOUT; ++q) {
    const double m = h[2 * q] / G.ns, var = std::max(0.0, h[2 * q + 1] / G.ns - m * m);
    ymu[q] = (float)m;
    ysd[q] = var > 0.0 ? (float)sqrt(var) : 1.f;
  }
  HIPCHK(hipFree(st));
  std::vector<float> yisd(SGS_KOUT, 0.f);
  for (int q = 0; q < SGS_NOUT; ++q) yisd[q] = 1.f / ysd[q];
  HIPCHK(hipMemcpy(G.xmu, mu.data(), SGS_KIN * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(G.xisd, isd.data(), SGS_KIN * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(G.ymu, ymu.data(), SGS_KOUT * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(G.ysd, ysd.data(), SGS_KOUT * sizeof(float), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_normalise, blocks(G.ns * SGS_KIN), dim3(256), 0, s, G.Xs, G.ns, SGS_KIN, SGS_NIN, (const float *)G.xmu,
                     (const float *)G.xisd);
  float *yi = nullptr;
  HIPCHK(hipMalloc(&yi, SGS_KOUT * sizeof(float)));
  HIPCHK(hipMemcpy(yi, yisd.data(), SGS_KOUT * sizeof(float), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_normalise, blocks(G.ns * SGS_KOUT), dim3(256), 0, s, G.Ts, G.ns, SGS_KOUT, SGS_NOUT, (const float *)G.ymu,
                     (const float *)yi);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(s));
  HIPCHK(hipFree(yi));
  G.have_norm = true;
  return FE_OK;
}

/* Glorot-uniform weights and zero biases from a seeded generator (host side). */
int fe_sgs_init_params(unsigned seed) {
  int rc;
  if (!D.fecuda) return FE_ERR_STATE;
  if ((rc = sgs_params_alloc())) return rc;
  std::vector<float> w(NPARAM, 0.f);
  std::mt19937 gen(seed);
  auto fill = [&](long off, int nin, int nout, int nin_used, int nout_used) {
    const float lim = sqrtf(6.f / (float)(nin_used + nout_used));
    std::uniform_real_distribution<float> u(-lim, lim);
    for (int i = 0; i < nin; ++i)
      for (int o = 0; o < nout; ++o) w[off + (long)i * nout + o] = (i < nin_used && o < nout_used) ? u(gen) : 0.f;
  };
  fill(OW1, SGS_KIN, SGS_H, SGS_NIN, SGS_H);
  fill(OW2, SGS_H, SGS_H, SGS_H, SGS_H);
  fill(OW3, SGS_H, SGS_H, SGS_H, SGS_H);
  fill(OW4, SGS_H, SGS_KOUT, SGS_H, SGS_NOUT);
  HIPCHK(hipMemcpy(G.w, w.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(G.am, 0, NPARAM * sizeof(float)));
  HIPCHK(hipMemset(G.av, 0, NPARAM * sizeof(float)));
  G.adam_t = 0;
  G.have_w = true;
  return FE_OK;
}

/* Adam training on the normalised set: epochs passes over a seeded permutation in
 * mini-batches of batch rows; the mean squared error of each epoch (normalised targets,
 * the 9 outputs) goes to loss[epoch] (nloss >= epochs). */
int fe_sgs_train(int epochs, int batch, float lr, unsigned seed, double *loss, int nloss) {
  int rc;
  if (!G.have_norm || !G.have_w || batch < 1 || epochs < 0 || (loss && nloss < epochs)) return FE_ERR_STATE;
  if ((rc = sgs_rows(batch))) return rc;
  if (G.idx_cap < G.ns) {
    if (G.idx) HIPCHK(hipFree(G.idx));
    HIPCHK(hipMalloc(&G.idx, G.ns * sizeof(int)));
    G.idx_cap = G.ns;
  }
  hipStream_t s = sgs_stream();
  std::vector<int> perm(G.ns);
  std::mt19937 gen(seed);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int ep = 0; ep < epochs; ++ep) {
    for (long i = 0; i < G.ns; ++i) perm[i] = (int)i;
    std::shuffle(perm.begin(), perm.end(), gen);
    HIPCHK(hipMemcpyAsync(G.idx, perm.data(), G.ns * sizeof(int), hipMemcpyHostToDevice, s));
    HIPCHK(hipMemsetAsync(G.dloss, 0, sizeof(double), s));
    const long nb = G.ns / batch;
    for (long b = 0; b < nb; ++b) {
      const int *ix = G.idx + b * batch;
      hipLaunchKernelGGL(k_gather_rows, blocks((long)batch * SGS_KIN), dim3(256), 0, s, (const float *)G.Xs, ix, (long)batch,
                         SGS_KIN, G.Xb);
      hipLaunchKernelGGL(k_gather_rows, blocks((long)batch * SGS_KOUT), dim3(256), 0, s, (const float *)G.Ts, ix, (long)batch,
                         SGS_KOUT, G.Tb);
      if ((rc = mlp_forward(G.Xb, batch))) return rc;
      if ((rc = sgs_loss_grad(G.Tb, batch))) return rc;
      if ((rc = mlp_backward(G.Xb, batch))) return rc;
      G.adam_t++;
      const float bc1 = 1.f - powf(b1, (float)G.adam_t), bc2 = 1.f - powf(b2, (float)G.adam_t);
      hipLaunchKernelGGL(k_adam, blocks(NPARAM), dim3(256), 0, s, G.w, (const float *)G.gw, G.am, G.av, NPARAM, lr, b1, b2, eps,
                         bc1, bc2);
    }
    HIPCHK(hipGetLastError());
    double l = 0.0;
    HIPCHK(hipMemcpyAsync(&l, G.dloss, sizeof(double), hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if (loss) loss[ep] = nb > 0 ? l / ((double)nb * batch * SGS_NOUT) : 0.0;
  }
  return FE_OK;
}

/* Parameter vector (NPARAM floats: W1 [256][64], b1, W2 [64][64], b2, W3 [64][64], b3,
 * W4 [64][16], b4 [16]) to out (get = 1) or from it (get = 0). */
int fe_sgs_params(float *buf, long n, int get) {
  int rc;
  if (!buf || n != NPARAM) return FE_ERR_UNSUPPORTED;
  if (!D.fecuda) return FE_ERR_STATE;
  if ((rc = sgs_params_alloc())) return rc;
  HIPCHK(hipStreamSynchronize(sgs_stream()));
  if (get) HIPCHK(hipMemcpy(buf, G.w, n * sizeof(float), hipMemcpyDeviceToHost));
  else {
    HIPCHK(hipMemcpy(G.w, buf, n * sizeof(float), hipMemcpyHostToDevice));
    G.have_w = true;
  }
  return FE_OK;
}
long fe_sgs_nparam(void) { return NPARAM; }

/* Normalisation (4 x 256 floats: feature means, feature 1/std, target means, target std;
 * the target rows use their first 16 entries) to out (get = 1) or from it (get = 0). */
int fe_sgs_norm(float *buf, long n, int get) {
  int rc;
  if (!buf || n != 4 * SGS_KIN) return FE_ERR_UNSUPPORTED;
  if (!D.fecuda) return FE_ERR_STATE;
  if ((rc = sgs_params_alloc())) return rc;
  float *p[4] = {G.xmu, G.xisd, G.ymu, G.ysd};
  for (int k = 0; k < 4; ++k) {
    const size_t nb = (k < 2 ? SGS_KIN : SGS_KOUT) * sizeof(float);
    if (get) {
      std::fill(buf + k * SGS_KIN, buf + (k + 1) * SGS_KIN, 0.f);
      HIPCHK(hipMemcpy(buf + k * SGS_KIN, p[k], nb, hipMemcpyDeviceToHost));
    } else {
      HIPCHK(hipMemcpy(p[k], buf + k * SGS_KIN, nb, hipMemcpyHostToDevice));
    }
  }
  if (!get) G.have_norm = true;
  return FE_OK;
}

/* The network stream, waited for on every way out of a call that has handed it host memory. */
struct SgsDone {
  bool waited = false;
  int wait() {
    waited = true;
    HIPCHK(hipStreamSynchronize(sgs_stream()));
    return FE_OK;
  }
  ~SgsDone() { if (!waited) (void)hipStreamSynchronize(sgs_stream()); }
};

/* n floats of a caller's rows to the device; read when the stream is done (SgsDone) */
static int sgs_rows_up(float *dev, const float *host, long n) {
  const size_t bytes = n * sizeof(float);
  int rc;
  if (bytes < XF_LONE) {
    HIPCHK(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, sgs_stream()));
    return FE_OK;
  }
  if ((rc = xfer_reserve(bytes))) return rc;
  XferScope scope;
  if ((rc = xfer_up(sgs_stream(), dev, host, bytes))) return rc;
  return xfer_finish(sgs_stream());
}

/* Network forward of M normalised feature rows X ([M][256], host) into Y ([M][16], host). */
int fe_mlp_forward(const float *X, long M, float *Y) {
  int rc;
  if (!X || !Y || M < 1) return FE_ERR_UNSUPPORTED;
  if (!G.have_w) return FE_ERR_STATE;
  if ((rc = sgs_rows(M))) return rc;
  SgsDone done;
  if ((rc = sgs_rows_up(G.Xb, X, M * SGS_KIN))) return rc;
  if ((rc = mlp_forward(G.Xb, M))) return rc;
  HIPCHK(hipMemcpyAsync(Y, G.Y, M * SGS_KOUT * sizeof(float), hipMemcpyDeviceToHost, sgs_stream()));
  return done.wait();
}

/* Gradient of the training loss (mean squared error over the first 9 of the 16 output
 * columns of M rows, targets T [M][16]) with respect to the parameter vector, into grad
 * (NPARAM floats); the loss itself to loss[0]. */
int fe_mlp_gradient(const float *X, const float *T, long M, float *grad, double *loss) {
  int rc;
  if (!X || !T || !grad || M < 1) return FE_ERR_UNSUPPORTED;
  if (!G.have_w) return FE_ERR_STATE;
  if ((rc = sgs_rows(M))) return rc;
  hipStream_t s = sgs_stream();
  double l = 0.0;
  SgsDone done;
  if ((rc = sgs_rows_up(G.Xb, X, M * SGS_KIN))) return rc;
  if ((rc = sgs_rows_up(G.Tb, T, M * SGS_KOUT))) return rc;
  HIPCHK(hipMemsetAsync(G.dloss, 0, sizeof(double), s));
  if ((rc = mlp_forward(G.Xb, M))) return rc;
  if ((rc = sgs_loss_grad(G.Tb, M))) return rc;
  if ((rc = mlp_backward(G.Xb, M))) return rc;
  HIPCHK(hipMemcpyAsync(grad, G.gw, NPARAM * sizeof(float), hipMemcpyDeviceToHost, s));
  if (loss) HIPCHK(hipMemcpyAsync(&l, G.dloss, sizeof(double), hipMemcpyDeviceToHost, s));
  if ((rc = done.wait())) return rc;
  if (loss) loss[0] = l / ((double)M * SGS_NOUT);
  return FE_OK;
}

/* Learned closure in the plain model's physics stage on (on = 1) or off; cells pass the
 * input gate where every normalised feature is within [-gate, gate]. */
int fe_sgs_enable(int on, float gate) {
  if (!D.hydro) return FE_ERR_STATE;
  if (on) {
    if (!G.have_w || !G.have_norm) return FE_ERR_STATE;
    if (D.terrain) {
      fprintf(stderr, "fe_sgs_enable: the learned closure was trained on a flat grid\n");
      return FE_ERR_TERRAIN;
    }
    if (D.halo) {
      fprintf(stderr, "fe_sgs_enable: the learned closure runs on periodic grids only (no lateral halo storage)\n");
      return FE_ERR_UNSUPPORTED;
    }
    if (!(turbulenceSelector > 0 && TKESelector > 0) || D.nM > 0) {
      fprintf(stderr, "fe_sgs_enable: the learned closure stands beside the dry prognostic-TKE closure only\n");
      return FE_ERR_UNSUPPORTED;
    }
    const long ncell = (long)D.Nx * D.Ny * D.Nz;
    if (12 * ncell > (long)UINT_MAX) {
      fprintf(stderr, "fe_sgs_enable: %ld cells exceed the learned closure's 32-bit cell indexing\n", ncell);
      return FE_ERR_UNSUPPORTED;
    }
    if (ncell > G.ncell_cap) {
      if (G.tauL) HIPCHK(hipFree(G.tauL));
      if (G.gmax) HIPCHK(hipFree(G.gmax));
      if (G.mask) HIPCHK(hipFree(G.mask));
      if (G.grad) HIPCHK(hipFree(G.grad));
      G.tauL = nullptr; G.gmax = nullptr; G.mask = nullptr; G.grad = nullptr;
      HIPCHK(hipMalloc(&G.tauL, 9 * ncell * sizeof(float)));
      HIPCHK(hipMalloc(&G.gmax, ncell * sizeof(float)));
      HIPCHK(hipMalloc(&G.mask, ncell));
      HIPCHK(hipMalloc(&G.grad, 10 * ncell * sizeof(float)));
      G.ncell_cap = ncell;
    }
    if (G.j33) HIPCHK(hipFree(G.j33));
    G.j33 = nullptr;
    std::vector<float> j(D.Nz);
    for (int z = 0; z < D.Nz; ++z) j[z] = D.hprof[(size_t)(z + 3) * PROW + PR_J33];
    HIPCHK(hipMalloc(&G.j33, D.Nz * sizeof(float)));
    HIPCHK(hipMemcpy(G.j33, j.data(), D.Nz * sizeof(float), hipMemcpyHostToDevice));
    if (!D.tau) {
      HIPCHK(hipMalloc(&D.tau, (size_t)9 * D.fs * sizeof(float)));
      HIPCHK(hipMemset(D.tau, 0, (size_t)9 * D.fs * sizeof(float)));
    }
  }
  if (!G.dcount) HIPCHK(hipMalloc(&G.dcount, 2 * sizeof(unsigned long long)));
  HIPCHK(hipMemset(G.dcount, 0, 2 * sizeof(unsigned long long)));
  G.on = on ? 1 : 0;
  G.gate = gate;
  return FE_OK;
}

/* out[0] cells evaluated by the learned closure since it was enabled, out[1] cells that
 * passed the gate and realizability check (summed over physics stages). */
int fe_sgs_stats(double *out, int n) {
  if (!out || n < 2) return FE_ERR_UNSUPPORTED;
  unsigned long long c[2] = {0, 0};
  if (G.dcount) {
    HIPCHK(hipStreamSynchronize(sgs_stream()));
    HIPCHK(hipMemcpy(c, G.dcount, sizeof c, hipMemcpyDeviceToHost));
  }
  out[0] = (double)c[0];
  out[1] = (double)c[1];
  return FE_OK;
}

/* The learned cell stresses (rho*tau, [9][cells], order 11, 22, 33, 12, 13, 23, theta1..3)
 * and pass masks of the last physics stage; n = cells of the model. */
int fe_sgs_last(float *tau, unsigned char *mask, long n) {
  if (!G.on || n != (long)D.Nx * D.Ny * D.Nz) return FE_ERR_STATE;
  HIPCHK(hipStreamSynchronize(sgs_stream()));
  if (tau) HIPCHK(hipMemcpy(tau, G.tauL, 9 * n * sizeof(float), hipMemcpyDeviceToHost));
  if (mask) HIPCHK(hipMemcpy(mask, G.mask, n, hipMemcpyDeviceToHost));
  return FE_OK;
}

/* The stresses the physics stage emitted ([9][z][y][x], pitch P; order 11, 21, 31, 32, 22,
 * 33, theta1..3), n = 9 Nz Ny P. */
int fe_sgs_emitted(float *tau, long n) {
  if (!D.tau || !tau || n != 9 * D.fs) return FE_ERR_STATE;
  HIPCHK(hipStreamSynchronize(sgs_stream()));
  HIPCHK(hipMemcpy(tau, D.tau, n * sizeof(float), hipMemcpyDeviceToHost));
  return FE_OK;
}

/* Inference through the fused kernels (on = 1, the default) or through the unfused feature,
 * GEMM and activation kernels of the training path (on = 0); both give the same bits. */
int fe_sgs_set_fused(int on) {
  G.fused = on ? 1 : 0;
  return FE_OK;
}

int fe_sgs_clear(void) { return sgs_free_all(); }

}  // extern "C"
