// Host-side launchers of one model's kernels (included in the model
// namespace after engine.h and args.inl).  Grid: ceil(nvox / (256/L)) blocks
// of 256 threads; dynamic LDS holds the staged CFP table and the measurement
// cache.

#define CDM_DISPATCH_L(L, CALL)            \
  switch (L) {                             \
    case 1: { constexpr int LG = 1; CALL; } break;   \
    case 4: { constexpr int LG = 4; CALL; } break;   \
    case 16: { constexpr int LG = 16; CALL; } break; \
    case 64: { constexpr int LG = 64; CALL; } break; \
    default: return hipErrorInvalidValue;  \
  }

#define CDM_DISPATCH_W(W, CALL)            \
  switch (W) {                             \
    case 1: { constexpr int WG = 1; CALL; } break; \
    case 2: { constexpr int WG = 2; CALL; } break; \
    case 4: { constexpr int WG = 4; CALL; } break; \
    default: return hipErrorInvalidValue;  \
  }

template <int L>
static void op_gridsearch_split(const cdm::Geom& g, const cdm_gs_args& a, const cdm_gs_split& sp, hipStream_t s) {
  const dim3 grid = op_grid(g.nvox, L), grid_s(grid.x, (unsigned)sp.S);
  hipLaunchKernelGGL(cdm_gridsearch_split_kernel<L>, grid_s, dim3(cdm_block), op_lds(g), s, a, sp);
  hipLaunchKernelGGL(cdm_gridsearch_merge_kernel<L>, grid, dim3(cdm_block), op_lds(g), s, a, sp);
  if constexpr (sizeof(cdm_tf) != sizeof(double)) {
    hipLaunchKernelGGL(cdm_gridsearch_rescan_kernel<L>, grid_s, dim3(cdm_block), op_lds(g), s, a, sp);
    hipLaunchKernelGGL(cdm_gridsearch_pick_kernel<L>, grid, dim3(cdm_block), 0, s, a, sp);
  }
}

// S > 1: the search split over S slices of the combinations, in the scratch
// `split` (cdm::gs_split_bytes(nvox, S) bytes): the screen
// (cdm_gridsearch_split_kernel), the merge that finishes the voxels that are
// not crowded (cdm_gridsearch_merge_kernel), the crowded voxels' FP64 rescan
// (cdm_gridsearch_rescan_kernel) and their choice (cdm_gridsearch_pick_kernel).
static hipError_t op_gridsearch(int L, const cdm::Geom& g, float* params, int ngp, const int* gparams, int ncombs,
                                const float* grid_f, const double* grid_d, const int* comb_id, const cdm::Consts& c,
                                int* kept, int S, void* split, hipStream_t s) {
  if (g.nvox <= 0) return hipSuccess;
  if (ngp > cdm_np || g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  cdm_gs_args a;
  a.g = op_geom(g);
  a.params = params;
  a.ngp = ngp;
  for (int i = 0; i < cdm_np; ++i) a.gparams[i] = i < ngp ? gparams[i] : -1;
  a.ncombs = ncombs;
  a.grid_f = grid_f;
  a.grid_d = grid_d;
  a.comb_id = comb_id;
  a.c = op_consts(c);
  a.kept_out = kept;
  if (S > 1 && split) {
    const size_t n = (size_t)g.nvox * S;
    cdm_gs_split sp;
    sp.S = S;
    sp.rescan_c = (double*)split;
    sp.list_c = (float*)(sp.rescan_c + n);
    sp.list_i = (int*)(sp.list_c + n * CDM_GS_TOPK);
    sp.rescan_i = sp.list_i + n * CDM_GS_TOPK;
    sp.crowd = sp.rescan_i + n;
    CDM_DISPATCH_L(L, op_gridsearch_split<LG>(g, a, sp, s));
    return hipGetLastError();
  }
  CDM_DISPATCH_L(L, hipLaunchKernelGGL(cdm_gridsearch_kernel<LG>, op_grid(g.nvox, LG), dim3(cdm_block), op_lds(g),
                                       s, a));
  return hipGetLastError();
}

// The search over basis signals: its kernel arguments and dynamic LDS at L
// lanes per voxel (after the CFP table and the measurement cache: the table
// values, the weight parameters' values, the voxels' rows).  A row stride of
// L entries modulo 64 puts the groups of a wave on different banks.
static constexpr size_t cdm_gs_table_max = 16 * 1024;

static cdm_gs_plan op_gs_plan(int L, const cdm::Geom& g, const cdm::GridPlan& p, size_t* lds) {
  cdm_gs_plan k;
  std::memset(&k, 0, sizeof(k));
  k.nshared = p.nshared;
  k.nouter = p.nouter;
  k.ninner = p.ninner;
  unsigned grid = 0;
  for (int i = 0; i < p.ngp; ++i) grid |= 1u << p.gparams[i];
  k.grid = grid;
  k.outer_vals = p.outer_vals;
  k.inner_vals = p.inner_vals;
  k.order = p.order;
  const size_t table = (size_t)p.nshared * cdm_gs_ntab * sizeof(CDM_F64);
  k.table_lds = (cdm_gs_table_dep & ~grid) == 0 && table > 0 && table <= cdm_gs_table_max ? 1 : 0;
  k.table_fixed = (cdm_gs_table_dep & grid) == 0 ? 1 : 0;
  k.frame_fixed = (cdm_gs_frame_dep & grid) == 0 ? 1 : 0;
  size_t at = (op_lds(g) + 15) / 16 * 16;
  k.off_common = (int)at;
  at = (at + (size_t)g.nmeas * cdm_gs_nc * sizeof(cdm_tf) + 15) / 16 * 16;
  k.off_table = (int)at;
  if (k.table_lds) at += table;
  k.off_inner = (int)at;
  at = (at + (size_t)p.ninner * cdm_gs_nw * sizeof(float) + 15) / 16 * 16;
  k.off_rows = (int)at;
  const int n = cdm_gs_row * g.nmeas;
  k.row_stride = n + ((cdm_gs_row * L - n % 64) % 64 + 64) % 64;
  *lds = at + (size_t)(cdm_block / L) * k.row_stride * sizeof(cdm_tf);
  return k;
}

// Whether the scan of every combination is the better search: a grid that moves
// no weight, where an evaluation of the basis serves one combination.  Ratios
// are this search's time to the scan's, at 20k voxels unless said; slots: the
// lanes that fill the GPU.
// - A single combination: 26 and 21 us.
// - Sticks, each combination with its own shared part, several shared signals
//   (directions of the first stick): Ball_3_Sticks 0.8 at 30 measurements, 1.1 at 45,
//   1.8 at 90, 2.6 at 280, 150k voxels 1.8 to 2.9; small volumes gain by the slices
//   of the shared combinations (3,000 voxels 0.5 at 30, 1.0 at 90, 1.7 at 280).
// - The same with the ball alone shared (Ball_1_Stick, diffusivities): 1.0 up to 64
//   measurements, 1.2 to 2.3 from 90 on; 150k voxels 0.6 to 1.0.
// - Sticks, several combinations to a shared part.  The ball alone: directions 1.3
//   to 1.7, with diffusivities 0.8 to 1.6, 150k voxels 0.7 to 1.1, 604 measurements
//   1.2.  Several shared signals: 0.5 to 0.9, but 1.1 to 1.3 at 3,000 voxels with a
//   single shared part, which has no slices.
static bool op_gs_scan_better(const cdm::Geom& g, const cdm::GridPlan& p, long long slots) {
  if (p.ncombs < 2) return true;
  if (p.ninner > 1 || cdm_gs_ntab > 0) return false;
  const bool idle = (long long)g.nvox * 16 < slots, large = (long long)g.nvox * 16 >= 10 * slots;
  if (cdm_gs_ks > 1)
    return p.nouter > 1 ? p.nshared == 1 && idle : (long long)g.nvox * g.nmeas >= (g.nmeas < 40 ? 5 : 2) * slots;
  return p.nouter > 1 ? !large || g.nmeas >= 480 : !large && g.nmeas >= 80;
}

// Lanes the search over basis signals runs at, from L on those whose LDS fits;
// 0: the scan is taken, also where no weight moves and even 64 lanes leave one
// block per CU (NODDI_Watson, 604 measurements, 432 combinations, 20k voxels: 70
// ms against 46).
static int op_grid_basis_lanes(int L, const cdm::Geom& g, const cdm::GridPlan& p, long long slots) {
  if constexpr (!cdm_gs_basis) return 0;
  if ((size_t)p.ninner * cdm_gs_nw * sizeof(float) > cdm_gs_table_max || op_gs_scan_better(g, p, slots)) return 0;
  for (; L <= 64; L *= 4) {
    size_t lds = 0;
    (void)op_gs_plan(L, g, p, &lds);
    if (lds <= cdm_lds_max) return p.ninner == 1 && L == 64 && lds > cdm_lds_max / 2 ? 0 : L;
  }
  return 0;
}

#ifdef CDM_GRID_LINEAR
template <int L>
static void op_gs_screen(const cdm_gs_args& a, const cdm_gs_plan& pl, size_t lds, const cdm_gs_work& wk, hipStream_t s) {
  const dim3 grid = op_grid(a.g.nvox, L);
  hipLaunchKernelGGL(cdm_gs_basis_kernel<L>, dim3(grid.x, (unsigned)wk.S), dim3(cdm_block), lds, s, a, pl, wk);
}
template <int L>
static void op_gs_rescan(const cdm_gs_args& a, const cdm_gs_plan& pl, size_t lds, const cdm_gs_work& wk, int ncu,
                         hipStream_t s) {
  // at most every voxel's slices, else blocks that go through the list
  const unsigned long long most = (unsigned long long)op_grid(a.g.nvox, L).x * (unsigned)wk.SB;
  const unsigned long long cap = 8ull * (unsigned)(ncu > 0 ? ncu : 1);
  hipLaunchKernelGGL(cdm_gs_basis_rescan_kernel<L>, dim3((unsigned)(most < cap ? most : cap)), dim3(cdm_block), lds, s,
                     a, pl, wk);
}
#endif

// L: a group size that op_grid_basis_lanes returned.
static hipError_t op_gridsearch_basis(int L, const cdm::Geom& g, float* params, const cdm::GridPlan& p,
                                      const cdm::Consts& c, int* kept, const cdm::GridWork& w, hipStream_t s) {
#ifdef CDM_GRID_LINEAR
  if (g.nvox <= 0) return hipSuccess;
  if (p.ngp > cdm_np || g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  cdm_gs_args a;
  a.g = op_geom(g);
  a.params = params;
  a.ngp = p.ngp;
  for (int i = 0; i < cdm_np; ++i) a.gparams[i] = i < p.ngp ? p.gparams[i] : -1;
  a.ncombs = p.ncombs;
  a.grid_f = p.grid_f;
  a.grid_d = p.grid_d;
  a.comb_id = p.comb_id;
  a.c = op_consts(c);
  a.kept_out = kept;
  cdm_gs_work wk = {w.S, w.SB, w.part_c1, w.part_c2, w.part_i1, w.sumsq, w.count, w.list, w.thr, w.rescan_c, w.rescan_i};
  size_t lds = 0;
  const cdm_gs_plan pl = op_gs_plan(L, g, p, &lds);
  hipLaunchKernelGGL(cdm_queue_reset_kernel, dim3(1), dim3(cdm_block), 0, s, w.count, 1);
  CDM_DISPATCH_L(L, op_gs_screen<LG>(a, pl, lds, wk, s));
  if (wk.S > 1)
    hipLaunchKernelGGL(cdm_gs_basis_merge_kernel, op_grid(g.nvox, cdm_gs_merge_lanes), dim3(cdm_block), 0, s, a, pl, wk);
  // the FP64 scan runs on few voxels, at 16 lanes or more each
  const int L2 = L < 16 ? 16 : L;
  size_t lds2 = 0;
  const cdm_gs_plan pl2 = op_gs_plan(L2, g, p, &lds2);
  if (L2 == 16) op_gs_rescan<16>(a, pl2, lds2, wk, w.ncu, s);
  else op_gs_rescan<64>(a, pl2, lds2, wk, w.ncu, s);
  const unsigned pick = op_grid(g.nvox, cdm_gs_merge_lanes).x;
  hipLaunchKernelGGL(cdm_gs_basis_pick_kernel, dim3(pick < 1024 ? pick : 1024), dim3(cdm_block), 0, s, a, wk);
  return hipGetLastError();
#else
  return hipErrorInvalidValue;
#endif
}

// Resident blocks per CU of the work-queue LM kernel <L, W> at `lds` bytes,
// queried once per shape (host-side occupancy calculation).
template <int L, int W>
static int op_levmar_queue_residency(size_t lds) {
  static int cached = 0;
  static size_t cached_lds = 0;
  if (cached <= 0 || cached_lds != lds) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (cdm_levmar_queue_kernel<L, W>), cdm_block, lds) !=
            hipSuccess || n <= 0)
      n = W;
    cached = n;
    cached_lds = lds;
  }
  return cached;
}

template <int L, int W>
static void op_levmar_queue_launch(const cdm_lm_args& a, int marquardt, int nvox, size_t lds, int ncu, hipStream_t s) {
  const unsigned need = op_grid(nvox, L).x;
  const unsigned cap = (unsigned)op_levmar_queue_residency<L, W>(lds) * (unsigned)(ncu > 0 ? ncu : 1);
  hipLaunchKernelGGL((cdm_levmar_queue_kernel<L, W>), dim3(need < cap ? need : cap), dim3(cdm_block), lds, s, a,
                     marquardt);
}

// queue: a device int of the model handle; non-null selects the work-queue
// kernel (grid: the resident blocks, at most one per voxel group), null the
// static mapping.  ncu: compute units of the device.
static hipError_t op_levmar(int L, int W, const cdm::Geom& g, float* params, int max_iters, int marquardt,
                            const cdm::Consts& c, int* iters, float* cost, int* queue, int ncu, hipStream_t s) {
  if (g.nvox <= 0) return hipSuccess;
  if (g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  L = op_lm_lanes(g, L);
  if (op_lds_lm(g, L) > cdm_lds_max) return hipErrorInvalidValue;
  cdm_lm_args a = op_lm_args(g, params, max_iters, c, iters, cost);
  if (!queue) {
    CDM_DISPATCH_L(L, CDM_DISPATCH_W(W, hipLaunchKernelGGL((cdm_levmar_kernel<LG, WG>), op_grid(g.nvox, LG),
                                                           dim3(cdm_block), op_lds_lm(g, LG), s, a, marquardt)));
    return hipGetLastError();
  }
  a.queue = queue;
  hipLaunchKernelGGL(cdm_queue_reset_kernel, dim3(1), dim3(cdm_block), 0, s, queue, 1);
  const size_t lds = op_lds_lm(g, L);
  CDM_DISPATCH_L(L, CDM_DISPATCH_W(W, (op_levmar_queue_launch<LG, WG>(a, marquardt, g.nvox, lds, ncu, s))));
  return hipGetLastError();
}

// Slices of an MCMC launch of `tiles` blocks, per_cu of them resident on each of
// ncu compute units (cdm_mcmc_kernel).  Without slices the last round is as long
// as a full one where two blocks per CU wait for their own results, and 0.4 of that
// where more share the CU (they speed up as others leave); n slices take between
// r = tiles / resident and ceil(n r) / n rounds, and each a hand-over (the chain
// state through memory, an L2 write-back, the prologue) worth 250 likelihood terms of
// a lane.  A step has ceil(M / L) terms, eight times the cost for plug-ins with a
// voxel cache, and draws worth three (with 64 lanes and their sums twelve).  At most as many slices as fill sixteen rounds, of
// 16 jumps at least.  Measured with and without: NODDI_Bingham, 35k voxels (r = 1.07), 300
// jumps 28.1 and 43.8 ms, 14k (1.7) 18.7 and 21.4; Ball_1_Stick, 66k (1.01), 300 jumps
// 8.7 and 11.1, but 300k (4.6), 64 jumps 8.6 and 7.3; toymodel, 66k, 300 jumps 3.1 and
// 2.6; DiffusionTensor, 300k, 64 jumps 9.8 and 9.0.
//   With 64 lanes, 70 jumps, 4,153 voxels (r = 2.0), with and without, DiffusionTensor 2.2
// and 2.7, Ball_1_Stick 2.0 and 2.3; 32 jumps, NODDI_Watson 3.3 and 3.7.
//   Rician launches, whose terms are dear and differ in time, take all of them: 4,000
// voxels, 100 jumps, with and without, Ball_2_Sticks 25.5 and 28.8 ms, NODDI_Bingham
// 14.1 and 15.7, DiffusionTensor 7.0 and 7.4; 3,300 and 40 jumps 9.4 and 11.3, 5.2 and
// 5.2, 2.6 and 3.0; 140k and 100 jumps, Ball_1_Stick 103.5 and 108.1.
constexpr int cdm_mcmc_rounds = 16, cdm_mcmc_least_jumps = 16;
static int op_mcmc_slices(int tiles, int per_cu, int ncu, int count, int nmeas, int L, bool rician) {
  const long long R = (long long)per_cu * ncu;
  if (R <= 0 || tiles <= R) return 1;
  const long long want = (cdm_mcmc_rounds * R + tiles - 1) / tiles;
  const int most = (int)std::min<long long>(want, count / cdm_mcmc_least_jumps);
  if (rician) return most > 1 ? most : 1;
  const double r = (double)tiles / R, whole = (double)((tiles + R - 1) / R);
  const double terms = (double)count * cdm_np * ((nmeas + L - 1) / L * (cdm_vc > 1 ? 8 : 1) + (L == 64 ? 12 : 3));
  int n = 1;
  double best = per_cu > 2 ? r + 0.4 * (whole - r) : whole;
  for (int k = 2; k <= most; ++k) {
    const double last = (double)(((long long)k * tiles + R - 1) / R) / k;
    const double t = 0.5 * (r + last) * (1.0 + 250.0 * k / terms);
    if (t < best) {
      best = t;
      n = k;
    }
  }
  return n;
}

template <int L, bool RICIAN, int W>
static hipError_t op_mcmc_launch(cdm_mcmc_args a, size_t lds, int* queue, int ncu, hipStream_t s) {
  dim3 grid((unsigned)a.ntiles);
  if (queue && ncu > 0 && a.ntiles > ncu) {
    int per_cu = 0;
    const hipError_t e =
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (cdm_mcmc_kernel<L, RICIAN, W>), cdm_block, lds);
    if (e != hipSuccess) return e;
    const int n = op_mcmc_slices(a.ntiles, per_cu, ncu, a.count, a.g.nmeas, L, RICIAN);
    if (n > 1) {
      a.queue = queue;
      a.chunk_len = (a.count + n - 1) / n;
      const unsigned slices = (unsigned)((a.count + a.chunk_len - 1) / a.chunk_len);
      const int ints = 16 + a.ntiles;
      hipLaunchKernelGGL(cdm_queue_reset_kernel, dim3((unsigned)((ints + cdm_block - 1) / cdm_block)),
                         dim3(cdm_block), 0, s, queue, ints);
      grid = dim3((unsigned)a.ntiles * slices);
    }
  }
  hipLaunchKernelGGL((cdm_mcmc_kernel<L, RICIAN, W>), grid, dim3(cdm_block), lds, s, a);
  return hipGetLastError();
}

static hipError_t op_mcmc(int L, int W, int rician, const cdm::Geom& g, const cdm::McmcLaunch& m,
                          const cdm::Consts& c, hipStream_t s) {
  if (g.nvox <= 0) return hipSuccess;
  if (g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  // the Rician likelihood is compiled at the default register budget only
  const int We = rician ? 1 : W;
  const cdm_mcmc_args a = op_mcmc_args(g, L, We, m, c);
  const size_t lds = op_lds_mcmc(g, L, We);
  if (rician) {
    CDM_DISPATCH_L(L, return (op_mcmc_launch<LG, true, 1>(a, lds, m.queue, m.ncu, s)));
  } else {
    CDM_DISPATCH_L(L, CDM_DISPATCH_W(W, return (op_mcmc_launch<LG, false, WG>(a, lds, m.queue, m.ncu, s))));
  }
  return hipErrorInvalidValue;
}

// W: the launch's effective register budget (1 for the Rician likelihood).
static int op_mcmc_rows_lds(int L, int W, const cdm::Geom& g) {
  return op_mcmc_rows_lds_bytes(g, L, W) > 0 ? 1 : 0;
}

static hipError_t op_predicted(int L, const cdm::Geom& g, int nsamples, const float* samples, float* out,
                               hipStream_t s) {
  if (g.nvox <= 0) return hipSuccess;
  if (g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  cdm_post_args a;
  a.g = op_geom(g);
  a.nsamples = nsamples;
  a.samples = samples;
  a.tau_samples = nullptr;
  a.out = out;
  a.bic = a.aic = nullptr;
  CDM_DISPATCH_L(L, hipLaunchKernelGGL(cdm_predicted_kernel<LG>, op_grid(g.nvox, LG), dim3(cdm_block),
                                       op_lds_post(g, LG), s, a));
  return hipGetLastError();
}

static hipError_t op_bic_aic(int L, int rician, const cdm::Geom& g, int nsamples, const float* samples,
                             const float* tau_samples, float* bic, float* aic, hipStream_t s) {
  if (g.nvox <= 0) return hipSuccess;
  if (g.cfp_ts > cdm_cfp_max || g.fixp_ts > cdm_fixp_max) return hipErrorInvalidValue;
  cdm_post_args a;
  a.g = op_geom(g);
  a.nsamples = nsamples;
  a.samples = samples;
  a.tau_samples = tau_samples;
  a.out = nullptr;
  a.bic = bic;
  a.aic = aic;
  if (rician) {
    CDM_DISPATCH_L(L, hipLaunchKernelGGL((cdm_bic_aic_kernel<LG, true>), op_grid(g.nvox, LG), dim3(cdm_block),
                                         op_lds_post(g, LG), s, a));
  } else {
    CDM_DISPATCH_L(L, hipLaunchKernelGGL((cdm_bic_aic_kernel<LG, false>), op_grid(g.nvox, LG), dim3(cdm_block),
                                         op_lds_post(g, LG), s, a));
  }
  return hipGetLastError();
}

#undef CDM_DISPATCH_L
#undef CDM_DISPATCH_W
