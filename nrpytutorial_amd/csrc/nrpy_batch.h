// Batched evolutions: many independent grids (uneven sizes, own parameters and
// boundary maps) advanced together, one launch per kernel per RK4 substep.
//
// The array roles (NRPY_BATCH_ROLE_*) and index ranges (NRPY_RANGE_*) are defined in
// nrpy_runtime_pre.h. Included by a generated bundle after it has defined nrpy_batch_instance:
//   typedef struct { paramstruct params; rfm_struct rfm; double *arr[NRPY_BATCH_ROLES];
//                    double dt; long Ntot; } nrpy_batch_instance;
// and the table nrpy_batched_kernels[] of {kernel id, range} pairs.
//
// Every launch covers the tiles of all instances: a block finds its instance by
// binary search in a prefix table of tile counts (NRPY_BATCH_FIND) and its tile
// inside that instance's index box (NRPY_BATCH_TILE). The prefix tables depend
// on the block shape and on the index range (interior or all points); they are
// built on the host for the current shapes by nrpy_batch_prepare, before any
// graph capture.
#pragma once

#define NRPY_BATCH_FIND()                                                                      \
  int nrpy_k;                                                                                  \
  {                                                                                            \
    int lo_ = 0, hi_ = ninst - 1;                                                              \
    const int b_ = (int)blockIdx.x;                                                            \
    while (lo_ < hi_) {                                                                        \
      const int mid_ = (lo_ + hi_ + 1) >> 1;                                                   \
      if (tile_prefix[mid_] <= b_) lo_ = mid_; else hi_ = mid_ - 1;                            \
    }                                                                                          \
    nrpy_k = lo_;                                                                              \
  }

#define NRPY_BATCH_TILE(n0, n1, n2)                                                            \
  int nrpy_bx, nrpy_by, nrpy_bz;                                                               \
  {                                                                                            \
    const int nbx_ = ((n0) + (int)blockDim.x - 1) / (int)blockDim.x;                           \
    const int nby_ = ((n1) + (int)blockDim.y - 1) / (int)blockDim.y;                           \
    const int t_ = (int)blockIdx.x - tile_prefix[nrpy_k];                                      \
    nrpy_bx = t_ % nbx_;                                                                       \
    nrpy_by = (t_ / nbx_) % nby_;                                                              \
    nrpy_bz = t_ / (nbx_ * nby_);                                                              \
  }

// Fill rows of many instances: row r belongs to instance h_inst[r] (a generic row's base
// counts from the start of the concatenated terms).
struct nrpy_batch_fill_list {
  int n = 0;
  std::vector<nrpy_fill_row> h_rows;
  std::vector<nrpy_fill_term> h_terms;
  std::vector<int> h_inst;
  nrpy_fill_row *d_rows = nullptr;
  nrpy_fill_term *d_terms = nullptr;
  int *d_inst = nullptr;
  void append(const nrpy_fill_list &L, const int k) {
    for (nrpy_fill_row R : L.h_rows) {
      if (R.code == NRPY_FILL_GENERIC) R.base += (int)h_terms.size();
      h_rows.push_back(R);
      h_inst.push_back(k);
    }
    h_terms.insert(h_terms.end(), L.h_terms.begin(), L.h_terms.end());
    n = (int)h_rows.size();
  }
  bool upload() {
    return nrpy_upload(&d_rows, h_rows.data(), h_rows.size()) && nrpy_upload(&d_terms, h_terms.data(), h_terms.size()) &&
           nrpy_upload(&d_inst, h_inst.data(), h_inst.size());
  }
  void free_device() {
    (void)hipFree(d_rows);
    (void)hipFree(d_terms);
    (void)hipFree(d_inst);
  }
};

struct nrpy_batch {
  int ninst = 0;
  std::vector<nrpy_batch_instance> h_inst;
  nrpy_batch_instance *d_inst = nullptr;
  // prefix tables: key (bx, by, bz, range) -> device array of ninst + 1 tile offsets
  std::map<std::vector<int>, int *> prefix;
  std::map<std::vector<int>, int> ntiles;
  // the instances' fill lists one after another, every ghost and those a stage's stencils reach
  nrpy_batch_fill_list fill_all, fill_stage;
};

static void nrpy_batch_range(const nrpy_batch_instance &I, int range, int n[3]) {
  if (range == NRPY_RANGE_INTERIOR) {
    n[0] = I.params.Nxx0; n[1] = I.params.Nxx1; n[2] = I.params.Nxx2;
  } else {
    const int s = range == NRPY_RANGE_STAGE ? 2 : 0;
    n[0] = I.params.Nxx_plus_2NGHOSTS0 - s * NRPY_STAGE_LO0;
    n[1] = I.params.Nxx_plus_2NGHOSTS1 - s * NRPY_STAGE_LO1;
    n[2] = I.params.Nxx_plus_2NGHOSTS2 - s * NRPY_STAGE_LO2;
  }
}

static int nrpy_batch_make_prefix(nrpy_batch *b, dim3 block, int range) {
  std::vector<int> key = {(int)block.x, (int)block.y, (int)block.z, range};
  if (b->prefix.count(key)) return NRPY_OK;
  std::vector<int> pre(b->ninst + 1, 0);
  for (int k = 0; k < b->ninst; k++) {
    int n[3];
    nrpy_batch_range(b->h_inst[k], range, n);
    const long t = (long)nrpy_nblocks(block, n[0], n[1], n[2]);
    if ((long)pre[k] + t > 2147483647L) return NRPY_ERR_TOO_LARGE;
    pre[k + 1] = pre[k] + (int)t;
  }
  int *d = nullptr;
  if (!nrpy_upload(&d, pre.data(), pre.size())) return NRPY_ERR_ALLOC;
  b->prefix[key] = d;
  b->ntiles[key] = pre[b->ninst];
  return NRPY_OK;
}

// Device prefix table and total tile count for a launch; NULL if not prepared.
static const int *nrpy_batch_prefix(const nrpy_batch *b, dim3 block, int range, unsigned *nblocks) {
  std::vector<int> key = {(int)block.x, (int)block.y, (int)block.z, range};
  auto it = b->prefix.find(key);
  if (it == b->prefix.end()) return nullptr;
  *nblocks = (unsigned)b->ntiles.at(key);
  return it->second;
}

extern "C" void nrpy_batch_free(nrpy_batch *b) {
  if (!b) return;
  (void)hipFree(b->d_inst);
  for (auto &kv : b->prefix) (void)hipFree(kv.second);
  b->fill_all.free_device();
  b->fill_stage.free_device();
  delete b;
}

// Builds prefix tables for the current block shape of every batched kernel. Call
// after changing shapes with nrpy_set_block_shape and before capturing a graph.
extern "C" int nrpy_batch_prepare(nrpy_batch *b) {
  if (!b) return NRPY_ERR_NULL;
  const int nk = (int)(sizeof(nrpy_batched_kernels) / sizeof(nrpy_batched_kernels[0]));
  for (int i = 0; i < nk; i++) {
    const dim3 block = nrpy_block(nrpy_batched_kernels[i][0], nrpy_batched_kernels[i][2], nrpy_batched_kernels[i][3],
                                  nrpy_batched_kernels[i][4]);
    const int rc = nrpy_batch_make_prefix(b, block, nrpy_batched_kernels[i][1]);
    if (rc) return rc;
  }
  return NRPY_OK;
}

// ninst instances: params[k] (host), rfms[k] and bcs[k] (as returned by rfm_struct_create /
// bcstruct_create for instance k's grid), arrays[6*k + role] device arrays of instance k in
// the roles above (auxevol/aux may be NULL if the system has none), dts[k] its time step.
extern "C" int nrpy_batch_create(const int ninst, const paramstruct *params, const rfm_struct *const *rfms,
                                 const bc_struct *const *bcs, double *const *arrays, const double *dts,
                                 nrpy_batch **out) {
  if (!params || !rfms || !bcs || !arrays || !dts || !out) return NRPY_ERR_NULL;
  *out = nullptr;
  if (ninst < 1) return NRPY_ERR_PARAM;
  nrpy_batch *b = new nrpy_batch();
  b->ninst = ninst;
  b->h_inst.resize(ninst);
  for (int k = 0; k < ninst; k++) {
    if (!rfms[k] || !bcs[k] || nrpy_check_params(&params[k])) {
      nrpy_batch_free(b);
      return rfms[k] && bcs[k] ? NRPY_ERR_SHAPE : NRPY_ERR_NULL;
    }
    const bc_struct *bc = bcs[k];
    if (bc->N[0] != params[k].Nxx_plus_2NGHOSTS0 || bc->N[1] != params[k].Nxx_plus_2NGHOSTS1 ||
        bc->N[2] != params[k].Nxx_plus_2NGHOSTS2) {
      nrpy_batch_free(b);
      return NRPY_ERR_SHAPE;
    }
    nrpy_batch_instance &I = b->h_inst[k];
    memset(&I, 0, sizeof(I));
    I.params = params[k];
    I.rfm = *rfms[k];
    for (int r = 0; r < NRPY_BATCH_ROLES; r++) I.arr[r] = arrays[NRPY_BATCH_ROLES * k + r];
    for (int r = 0; r <= NRPY_BATCH_ROLE_RT; r++)
      if (!I.arr[r]) {
        nrpy_batch_free(b);
        return NRPY_ERR_NULL;
      }
    I.dt = dts[k];
    I.Ntot = (long)bc->N[0] * bc->N[1] * bc->N[2];
    b->fill_all.append(bc->fill_all, k);
    b->fill_stage.append(bc->fill_stage, k);
  }
  const bool ok = nrpy_upload(&b->d_inst, b->h_inst.data(), b->h_inst.size()) && b->fill_all.upload() &&
                  b->fill_stage.upload();
  if (!ok) {
    nrpy_batch_free(b);
    return NRPY_ERR_ALLOC;
  }
  int rc = nrpy_batch_prepare(b);
  if (rc) {
    nrpy_batch_free(b);
    return rc;
  }
  *out = b;
  return NRPY_OK;
}

// Ghost fill of the array in role 'role' of every instance, one launch, from the list of every
// ghost or of those a stage's stencils reach. A thread fills NRPY_BATCH_FILL_K gridfunctions of
// one row, with the code of the single-grid fill, so the values are the same bits.
#define NRPY_BATCH_FILL_K 8
__global__ void __launch_bounds__(256)
nrpy_batch_fill_kernel(const int nrows, const nrpy_batch_instance *__restrict__ inst,
                       const int *__restrict__ row_inst, const nrpy_fill_row *__restrict__ rows,
                       const nrpy_fill_term *__restrict__ terms, const int role, const int num_gfs,
                       const nrpy_gf_parity_args gfp) {
  const int r = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (r >= nrows) return;
  const nrpy_fill_row R = rows[r];
  const nrpy_batch_instance *I = inst + row_inst[r];
  const int N0 = I->params.Nxx_plus_2NGHOSTS0, N01 = N0 * I->params.Nxx_plus_2NGHOSTS1;
  nrpy_fill_point<NRPY_BATCH_FILL_K>(R, terms, N0, N01, (size_t)I->Ntot, NRPY_BATCH_FILL_K * (int)blockIdx.y, num_gfs,
                                     gfp, I->arr[role]);
}

static int nrpy_batch_fill(const nrpy_batch *b, const nrpy_batch_fill_list *L, const int role, const int NUM_GFS,
                           const int8_t *gfs_parity, hipStream_t stream) {
  if (!b || !gfs_parity) return NRPY_ERR_NULL;
  if (role < 0 || role >= NRPY_BATCH_ROLES || NUM_GFS < 1 || NUM_GFS > 64) return NRPY_ERR_PARAM;
  if (L->n == 0) return NRPY_OK;
  nrpy_gf_parity_args gfp;
  memset(&gfp, 0, sizeof(gfp));
  for (int g = 0; g < NUM_GFS; g++) {
    if (gfs_parity[g] < 0 || gfs_parity[g] > 9) return NRPY_ERR_PARAM;
    gfp.p[g] = gfs_parity[g];
  }
  const int B = 256;
  hipLaunchKernelGGL(nrpy_batch_fill_kernel,
                     dim3((unsigned)((L->n + B - 1) / B), (NUM_GFS + NRPY_BATCH_FILL_K - 1) / NRPY_BATCH_FILL_K), dim3(B),
                     0, stream, L->n, b->d_inst, L->d_inst, L->d_rows, L->d_terms, role, NUM_GFS, gfp);
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}

// Every ghost point of the array in role 'role' of every instance, one launch.
extern "C" int nrpy_batch_apply_bcs(const nrpy_batch *b, const int role, const int NUM_GFS, const int8_t *gfs_parity,
                                    hipStream_t stream) {
  if (!b) return NRPY_ERR_NULL;
  return nrpy_batch_fill(b, &b->fill_all, role, NUM_GFS, gfs_parity, stream);
}
