// Generated by nrpytutorial_amd.codegen; do not edit.
#include "../nrpy_runtime_pre.h"
#define NGHOSTS 3
/* Gridfunction indices: alphabetical within each group. */
#define NUM_EVOL_GFS 8
#define GAMMAGF	0
#define AU0GF	1
#define AU1GF	2
#define AU2GF	3
#define EU0GF	4
#define EU1GF	5
#define EU2GF	6
#define PSIGF	7
#define NUM_AUX_GFS 2
#define CGF	0
#define GGF	1
#define NUM_AUXEVOL_GFS 0

typedef struct __paramstruct__ {
  double AMPLRHO;
  double AMPLZ;
  int Nxx0;
  int Nxx1;
  int Nxx2;
  int Nxx_plus_2NGHOSTS0;
  int Nxx_plus_2NGHOSTS1;
  int Nxx_plus_2NGHOSTS2;
  double RHOMAX;
  double SINHWRHO;
  double SINHWZ;
  double ZMAX;
  double ZMIN;
  double amp;
  double dxx0;
  double dxx1;
  double dxx2;
  double invdx0;
  double invdx1;
  double invdx2;
  double lam;
  double time;
  double wavespeed;
  double xmax;
  double xmin;
  double xx0;
  double xx1;
  double xx2;
  double ymax;
  double ymin;
  double zmax;
  double zmin;
} paramstruct;

static const int8_t evol_gf_parity[8] = {0, 1, 2, 3, 1, 2, 3, 0};
// point offsets read by the stencils of the RK4 step's kernels
static const int8_t nrpy_stage_offsets[12][3] = {{-2, 0, 0}, {-1, 0, 0}, {0, -2, 0}, {0, -1, 0}, {0, 0, -2}, {0, 0, -1}, {0, 0, 1}, {0, 0, 2}, {0, 1, 0}, {0, 2, 0}, {1, 0, 0}, {2, 0, 0}};
#define NRPY_STAGE_LO0 0
#define NRPY_STAGE_LO1 0
#define NRPY_STAGE_LO2 0
#define NRPY_SLAB_MIN_PLANE 7812
static int nrpy_check_params(const paramstruct *p) {
  if (p->Nxx0 < 1 || p->Nxx1 < 1 || p->Nxx2 < 1) return 1;
  if (p->Nxx_plus_2NGHOSTS0 != p->Nxx0 + 2*NGHOSTS || p->Nxx_plus_2NGHOSTS1 != p->Nxx1 + 2*NGHOSTS ||
      p->Nxx_plus_2NGHOSTS2 != p->Nxx2 + 2*NGHOSTS) return 1;
  if ((double)p->Nxx_plus_2NGHOSTS0 * p->Nxx_plus_2NGHOSTS1 * p->Nxx_plus_2NGHOSTS2 > 2147483647.0) return 1;
  return 0;
}

extern "C" void xx_to_Cart(const paramstruct *params, double *xx[3], const int i0, const int i1, const int i2, double xCart[3]) {
  const double AMPLRHO = params->AMPLRHO;
  const double AMPLZ = params->AMPLZ;
  const double SINHWRHO = params->SINHWRHO;
  const double SINHWZ = params->SINHWZ;
  const double xx0 = xx[0][i0];
  const double xx1 = xx[1][i1];
  const double xx2 = xx[2][i2];
  const double tmp_0 = (1.0/((SINHWRHO)));
  const double tmp_1 = tmp_0*xx0;
  const double tmp_2 = AMPLRHO*(exp(tmp_1) - exp(-tmp_1))/(exp(tmp_0) - exp(-tmp_0));
  const double tmp_3 = (1.0/((SINHWZ)));
  const double tmp_4 = tmp_3*xx2;
  xCart[0] = tmp_2*cos(xx1);
  xCart[1] = tmp_2*sin(xx1);
  xCart[2] = AMPLZ*(exp(tmp_4) - exp(-tmp_4))/(exp(tmp_3) - exp(-tmp_3));
}
static void EigenCoord_xx_to_Cart(const paramstruct *params, double *xx[3], const int i0, const int i1, const int i2, double xCart[3]) {
  const double xx0 = xx[0][i0];
  const double xx1 = xx[1][i1];
  const double xx2 = xx[2][i2];
  xCart[0] = xx0*cos(xx1);
  xCart[1] = xx0*sin(xx1);
  xCart[2] = xx2;
}
static void EigenCoord_Cart_to_xx(const paramstruct *params, const double xCart[3], double Cart_to_xx[3]) {
  const double Cartx = xCart[0];
  const double Carty = xCart[1];
  const double Cartz = xCart[2];
  Cart_to_xx[0] = sqrt(((Cartx)*(Cartx)) + ((Carty)*(Carty)));
  Cart_to_xx[1] = atan2(Carty, Cartx);
  Cart_to_xx[2] = Cartz;
}
static void eval_parity_dot_products(const paramstruct *params, double parity[10], const double xx0, const double xx1, const double xx2, const double xx0_inbounds, const double xx1_inbounds, const double xx2_inbounds) {
  const double tmp_0 = sin(xx1)*sin(xx1_inbounds) + cos(xx1)*cos(xx1_inbounds);
  const double tmp_1 = ((tmp_0)*(tmp_0));
  parity[0] = 1;
  parity[1] = tmp_0;
  parity[2] = tmp_0;
  parity[3] = 1;
  parity[4] = tmp_1;
  parity[5] = tmp_1;
  parity[6] = tmp_0;
  parity[7] = tmp_1;
  parity[8] = tmp_0;
  parity[9] = 1;
}
extern "C" int set_Nxx_dxx_invdx_params__and__xx(const int EigenCoord, const int Nxx[3], paramstruct *params, double *xx[3]) {
  if (!params || !Nxx || !xx) return NRPY_ERR_NULL;
  if (EigenCoord != 0 && EigenCoord != 1) return NRPY_ERR_PARAM;
  for (int d = 0; d < 3; d++) if (Nxx[d] < 1) return NRPY_ERR_SHAPE;
  params->Nxx0 = Nxx[0]; params->Nxx1 = Nxx[1]; params->Nxx2 = Nxx[2];
  params->Nxx_plus_2NGHOSTS0 = Nxx[0] + 2*NGHOSTS;
  params->Nxx_plus_2NGHOSTS1 = Nxx[1] + 2*NGHOSTS;
  params->Nxx_plus_2NGHOSTS2 = Nxx[2] + 2*NGHOSTS;
  const double RHOMAX = params->RHOMAX;
  const double ZMAX = params->ZMAX;
  const double ZMIN = params->ZMIN;
  double xxmin[3], xxmax[3];
  if (EigenCoord == 0) {
    xxmin[0] = 0;
    xxmax[0] = 1;
    xxmin[1] = -M_PI;
    xxmax[1] = M_PI;
    xxmin[2] = -1;
    xxmax[2] = 1;
  }
  if (EigenCoord == 1) {
    xxmin[0] = 0;
    xxmax[0] = RHOMAX;
    xxmin[1] = -M_PI;
    xxmax[1] = M_PI;
    xxmin[2] = ZMIN;
    xxmax[2] = ZMAX;
  }
  params->dxx0 = (xxmax[0] - xxmin[0]) / ((double)Nxx[0]);
  params->dxx1 = (xxmax[1] - xxmin[1]) / ((double)Nxx[1]);
  params->dxx2 = (xxmax[2] - xxmin[2]) / ((double)Nxx[2]);
  params->invdx0 = 1.0/params->dxx0;
  params->invdx1 = 1.0/params->dxx1;
  params->invdx2 = 1.0/params->dxx2;
  const int NN[3] = {params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2};
  const double dd[3] = {params->dxx0, params->dxx1, params->dxx2};
  for (int d = 0; d < 3; d++) {
    if (!xx[d]) return NRPY_ERR_NULL;
    for (int j = 0; j < NN[d]; j++) xx[d][j] = xxmin[d] + ((double)(j - NGHOSTS) + (1.0/2.0))*dd[d];
  }
  return NRPY_OK;
}
extern "C" double find_timestep(const paramstruct *params, double *xx[3], const double CFL_FACTOR) {
  const double AMPLRHO = params->AMPLRHO;
  const double AMPLZ = params->AMPLZ;
  const double SINHWRHO = params->SINHWRHO;
  const double SINHWZ = params->SINHWZ;
  const double dxx0 = params->dxx0;
  const double dxx1 = params->dxx1;
  const double dxx2 = params->dxx2;
  const int Nxx_plus_2NGHOSTS0 = params->Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params->Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params->Nxx_plus_2NGHOSTS2;
  double dsmin = 1e38;
  for (int i2 = NGHOSTS; i2 < Nxx_plus_2NGHOSTS2 - NGHOSTS; i2++)
  for (int i1 = NGHOSTS; i1 < Nxx_plus_2NGHOSTS1 - NGHOSTS; i1++)
  for (int i0 = NGHOSTS; i0 < Nxx_plus_2NGHOSTS0 - NGHOSTS; i0++) {
    const double xx0 = xx[0][i0]; const double xx1 = xx[1][i1]; const double xx2 = xx[2][i2];
    (void)xx0; (void)xx1; (void)xx2;
    double ds_dirn0, ds_dirn1, ds_dirn2;
    const double tmp_0 = (1.0/((SINHWRHO)));
    const double tmp_1 = tmp_0*xx0;
    const double tmp_2 = exp(tmp_1);
    const double tmp_3 = exp(-tmp_1);
    const double tmp_4 = AMPLRHO/(exp(tmp_0) - exp(-tmp_0));
    const double tmp_5 = (1.0/((SINHWZ)));
    const double tmp_6 = tmp_5*xx2;
    ds_dirn0 = dxx0*tmp_4*(tmp_0*tmp_2 + tmp_0*tmp_3);
    ds_dirn1 = dxx1*tmp_4*(tmp_2 - tmp_3);
    ds_dirn2 = AMPLZ*dxx2*(tmp_5*exp(tmp_6) + tmp_5*exp(-tmp_6))/(exp(tmp_5) - exp(-tmp_5));
    dsmin = fmin(dsmin, fmin(ds_dirn0, fmin(ds_dirn1, ds_dirn2)));
  }
  return dsmin*CFL_FACTOR/params->wavespeed;
}

#include "../nrpy_runtime.h"
typedef struct __rfmstruct__ {
  const double *f0_of_xx0;
  const double *f0_of_xx0__D0;
  const double *f0_of_xx0__DD00;
  const double *f0_of_xx0__DDD000;
  const double *f4_of_xx2;
  const double *f4_of_xx2__D2;
  const double *f4_of_xx2__DD22;
} rfm_struct;
extern "C" int rfm_struct_create(const paramstruct *params, double *xx[3], rfm_struct **out) {
  if (!params || !xx || !out) return NRPY_ERR_NULL;
  *out = nullptr;
  const int NN[3] = {params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2};
  (void)NN;
  double *tab[7] = {0};
  int rc = NRPY_OK;
  { std::vector<double> h(NN[0]);
    for (int i0 = 0; i0 < NN[0]; i0++) {
      const double xx0 = xx[0][i0];
      double v;
      const double AMPLRHO = params->AMPLRHO;
      const double SINHWRHO = params->SINHWRHO;
      const double tmp_0 = (1.0/((SINHWRHO)));
      const double tmp_1 = tmp_0*xx0;
      v = AMPLRHO*(exp(tmp_1) - exp(-tmp_1))/(exp(tmp_0) - exp(-tmp_0));
      h[i0] = v;
    }
    if (!nrpy_upload(&tab[0], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[0]);
    for (int i0 = 0; i0 < NN[0]; i0++) {
      const double xx0 = xx[0][i0];
      double v;
      const double AMPLRHO = params->AMPLRHO;
      const double SINHWRHO = params->SINHWRHO;
      const double tmp_0 = (1.0/((SINHWRHO)));
      const double tmp_1 = tmp_0*xx0;
      v = AMPLRHO*(tmp_0*exp(tmp_1) + tmp_0*exp(-tmp_1))/(exp(tmp_0) - exp(-tmp_0));
      h[i0] = v;
    }
    if (!nrpy_upload(&tab[1], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[0]);
    for (int i0 = 0; i0 < NN[0]; i0++) {
      const double xx0 = xx[0][i0];
      double v;
      const double AMPLRHO = params->AMPLRHO;
      const double SINHWRHO = params->SINHWRHO;
      const double tmp_0 = (1.0/((SINHWRHO)));
      const double tmp_1 = (1.0/((SINHWRHO)*(SINHWRHO)));
      const double tmp_2 = tmp_0*xx0;
      v = AMPLRHO*(tmp_1*exp(tmp_2) - tmp_1*exp(-tmp_2))/(exp(tmp_0) - exp(-tmp_0));
      h[i0] = v;
    }
    if (!nrpy_upload(&tab[2], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[0]);
    for (int i0 = 0; i0 < NN[0]; i0++) {
      const double xx0 = xx[0][i0];
      double v;
      const double AMPLRHO = params->AMPLRHO;
      const double SINHWRHO = params->SINHWRHO;
      const double tmp_0 = (1.0/((SINHWRHO)));
      const double tmp_1 = (1.0/((SINHWRHO)*(SINHWRHO)*(SINHWRHO)));
      const double tmp_2 = tmp_0*xx0;
      v = AMPLRHO*(tmp_1*exp(tmp_2) + tmp_1*exp(-tmp_2))/(exp(tmp_0) - exp(-tmp_0));
      h[i0] = v;
    }
    if (!nrpy_upload(&tab[3], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[2]);
    for (int i2 = 0; i2 < NN[2]; i2++) {
      const double xx2 = xx[2][i2];
      double v;
      const double AMPLZ = params->AMPLZ;
      const double SINHWZ = params->SINHWZ;
      const double tmp_0 = (1.0/((SINHWZ)));
      const double tmp_1 = tmp_0*xx2;
      v = AMPLZ*(tmp_0*exp(tmp_1) + tmp_0*exp(-tmp_1))/(exp(tmp_0) - exp(-tmp_0));
      h[i2] = v;
    }
    if (!nrpy_upload(&tab[4], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[2]);
    for (int i2 = 0; i2 < NN[2]; i2++) {
      const double xx2 = xx[2][i2];
      double v;
      const double AMPLZ = params->AMPLZ;
      const double SINHWZ = params->SINHWZ;
      const double tmp_0 = (1.0/((SINHWZ)));
      const double tmp_1 = (1.0/((SINHWZ)*(SINHWZ)));
      const double tmp_2 = tmp_0*xx2;
      v = AMPLZ*(tmp_1*exp(tmp_2) - tmp_1*exp(-tmp_2))/(exp(tmp_0) - exp(-tmp_0));
      h[i2] = v;
    }
    if (!nrpy_upload(&tab[5], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  { std::vector<double> h(NN[2]);
    for (int i2 = 0; i2 < NN[2]; i2++) {
      const double xx2 = xx[2][i2];
      double v;
      const double AMPLZ = params->AMPLZ;
      const double SINHWZ = params->SINHWZ;
      const double tmp_0 = (1.0/((SINHWZ)));
      const double tmp_1 = (1.0/((SINHWZ)*(SINHWZ)*(SINHWZ)));
      const double tmp_2 = tmp_0*xx2;
      v = AMPLZ*(tmp_1*exp(tmp_2) + tmp_1*exp(-tmp_2))/(exp(tmp_0) - exp(-tmp_0));
      h[i2] = v;
    }
    if (!nrpy_upload(&tab[6], h.data(), h.size())) rc = NRPY_ERR_ALLOC; }
  rfm_struct *r = new rfm_struct();
  memset(r, 0, sizeof(*r));
  r->f0_of_xx0 = tab[0];
  r->f0_of_xx0__D0 = tab[1];
  r->f0_of_xx0__DD00 = tab[2];
  r->f0_of_xx0__DDD000 = tab[3];
  r->f4_of_xx2 = tab[4];
  r->f4_of_xx2__D2 = tab[5];
  r->f4_of_xx2__DD22 = tab[6];
  *out = r;
  return rc;
}
extern "C" void rfm_struct_free(rfm_struct *rfmstruct) {
  if (!rfmstruct) return;
  (void)hipFree((void *)rfmstruct->f0_of_xx0);
  (void)hipFree((void *)rfmstruct->f0_of_xx0__D0);
  (void)hipFree((void *)rfmstruct->f0_of_xx0__DD00);
  (void)hipFree((void *)rfmstruct->f0_of_xx0__DDD000);
  (void)hipFree((void *)rfmstruct->f4_of_xx2);
  (void)hipFree((void *)rfmstruct->f4_of_xx2__D2);
  (void)hipFree((void *)rfmstruct->f4_of_xx2__DD22);
  delete rfmstruct;
}


/* Evaluate the vacuum Maxwell System II RHSs, rescaled curvilinear form */
__global__ void __launch_bounds__(256) rhs_eval__gpu(const rfm_struct rfmstruct, const paramstruct params, const double *__restrict__ in_gfs, double *__restrict__ rhs_gfs) {
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  
  NRPY_BLOCK_COORDS(Nxx0, Nxx1, Nxx2);
  const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
  const double f0_of_xx0 = rfmstruct.f0_of_xx0[i0];
  const double f0_of_xx0__D0 = rfmstruct.f0_of_xx0__D0[i0];
  const double f0_of_xx0__DD00 = rfmstruct.f0_of_xx0__DD00[i0];
  const double f0_of_xx0__DDD000 = rfmstruct.f0_of_xx0__DDD000[i0];
  const double f4_of_xx2 = rfmstruct.f4_of_xx2[i2];
  const double f4_of_xx2__D2 = rfmstruct.f4_of_xx2__D2[i2];
  const double f4_of_xx2__DD22 = rfmstruct.f4_of_xx2__DD22[i2];
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double eU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double eU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double eU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double aU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double aU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double aU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double aU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double aU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double aU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double aU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double aU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double aU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double aU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double aU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double aU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double aU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double aU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double aU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double aU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double aU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double aU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double aU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double aU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double aU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double aU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double aU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double aU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double aU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double aU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double aU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double aU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double aU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double aU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double aU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double aU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double aU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double aU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double aU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double aU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double aU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double aU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double aU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    const double psi_i0_i1_i2m2 = in_gfs[IDX4(PSIGF, i0,i1,i2-2)];
    const double psi_i0_i1_i2m1 = in_gfs[IDX4(PSIGF, i0,i1,i2-1)];
    const double psi_i0_i1m2_i2 = in_gfs[IDX4(PSIGF, i0,i1-2,i2)];
    const double psi_i0_i1m1_i2 = in_gfs[IDX4(PSIGF, i0,i1-1,i2)];
    const double psi_i0m2_i1_i2 = in_gfs[IDX4(PSIGF, i0-2,i1,i2)];
    const double psi_i0m1_i1_i2 = in_gfs[IDX4(PSIGF, i0-1,i1,i2)];
    const double psi = in_gfs[IDX4(PSIGF, i0,i1,i2)];
    const double psi_i0p1_i1_i2 = in_gfs[IDX4(PSIGF, i0+1,i1,i2)];
    const double psi_i0p2_i1_i2 = in_gfs[IDX4(PSIGF, i0+2,i1,i2)];
    const double psi_i0_i1p1_i2 = in_gfs[IDX4(PSIGF, i0,i1+1,i2)];
    const double psi_i0_i1p2_i2 = in_gfs[IDX4(PSIGF, i0,i1+2,i2)];
    const double psi_i0_i1_i2p1 = in_gfs[IDX4(PSIGF, i0,i1,i2+1)];
    const double psi_i0_i1_i2p2 = in_gfs[IDX4(PSIGF, i0,i1,i2+2)];
    const double Gamma_i0_i1_i2m2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-2)];
    const double Gamma_i0_i1_i2m1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-1)];
    const double Gamma_i0_i1m2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-2,i2)];
    const double Gamma_i0_i1m1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-1,i2)];
    const double Gamma_i0m2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-2,i1,i2)];
    const double Gamma_i0m1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-1,i1,i2)];
    const double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    const double Gamma_i0p1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+1,i1,i2)];
    const double Gamma_i0p2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+2,i1,i2)];
    const double Gamma_i0_i1p1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+1,i2)];
    const double Gamma_i0_i1p2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+2,i2)];
    const double Gamma_i0_i1_i2p1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+1)];
    const double Gamma_i0_i1_i2p2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+2)];
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_4_3 = 4.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double FDPart1_Rational_m5_2 = -5.0/2.0;
    const double FDPart1_0 = FDPart1_Rational_m1_12*aU0_i0p2_i1_i2;
    const double FDPart1_1 = FDPart1_Rational_m1_12*aU0_i0_i1p2_i2;
    const double FDPart1_2 = FDPart1_Rational_m1_12*aU0_i0_i1_i2p2;
    const double FDPart1_3 = FDPart1_Rational_m1_12*aU1_i0p2_i1_i2;
    const double FDPart1_4 = FDPart1_Rational_m1_12*aU1_i0_i1p2_i2;
    const double FDPart1_5 = FDPart1_Rational_m1_12*aU1_i0_i1_i2p2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*aU2_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*aU2_i0_i1_i2p2;
    const double FDPart1_8 = ((invdx0)*(invdx0));
    const double FDPart1_9 = FDPart1_Rational_m5_2*aU0;
    const double FDPart1_10 = ((invdx1)*(invdx1));
    const double FDPart1_11 = ((invdx2)*(invdx2));
    const double FDPart1_12 = FDPart1_Rational_m5_2*aU1;
    const double FDPart1_13 = FDPart1_Rational_m5_2*aU2;
    const double FDPart1_14 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_15 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_16 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_17 = FDPart1_Rational_m5_2*psi;
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double aU_dD00 = invdx0*(FDPart1_0 + FDPart1_Rational_1_12*aU0_i0m2_i1_i2 + FDPart1_Rational_2_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU0_i0m1_i1_i2);
    const double aU_dD01 = invdx1*(FDPart1_1 + FDPart1_Rational_1_12*aU0_i0_i1m2_i2 + FDPart1_Rational_2_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU0_i0_i1m1_i2);
    const double aU_dD02 = invdx2*(FDPart1_2 + FDPart1_Rational_1_12*aU0_i0_i1_i2m2 + FDPart1_Rational_2_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU0_i0_i1_i2m1);
    const double aU_dD10 = invdx0*(FDPart1_3 + FDPart1_Rational_1_12*aU1_i0m2_i1_i2 + FDPart1_Rational_2_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU1_i0m1_i1_i2);
    const double aU_dD11 = invdx1*(FDPart1_4 + FDPart1_Rational_1_12*aU1_i0_i1m2_i2 + FDPart1_Rational_2_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU1_i0_i1m1_i2);
    const double aU_dD12 = invdx2*(FDPart1_5 + FDPart1_Rational_1_12*aU1_i0_i1_i2m2 + FDPart1_Rational_2_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU1_i0_i1_i2m1);
    const double aU_dD20 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*aU2_i0m2_i1_i2 + FDPart1_Rational_2_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU2_i0m1_i1_i2);
    const double aU_dD22 = invdx2*(FDPart1_7 + FDPart1_Rational_1_12*aU2_i0_i1_i2m2 + FDPart1_Rational_2_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU2_i0_i1_i2m1);
    const double aU_dDD000 = FDPart1_8*(FDPart1_0 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0m1_i1_i2 + FDPart1_Rational_4_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU0_i0m2_i1_i2);
    const double aU_dDD011 = FDPart1_10*(FDPart1_1 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1m1_i2 + FDPart1_Rational_4_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU0_i0_i1m2_i2);
    const double aU_dDD022 = FDPart1_11*(FDPart1_2 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1_i2m1 + FDPart1_Rational_4_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU0_i0_i1_i2m2);
    const double aU_dDD100 = FDPart1_8*(FDPart1_12 + FDPart1_3 + FDPart1_Rational_4_3*aU1_i0m1_i1_i2 + FDPart1_Rational_4_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU1_i0m2_i1_i2);
    const double aU_dDD111 = FDPart1_10*(FDPart1_12 + FDPart1_4 + FDPart1_Rational_4_3*aU1_i0_i1m1_i2 + FDPart1_Rational_4_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU1_i0_i1m2_i2);
    const double aU_dDD122 = FDPart1_11*(FDPart1_12 + FDPart1_5 + FDPart1_Rational_4_3*aU1_i0_i1_i2m1 + FDPart1_Rational_4_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU1_i0_i1_i2m2);
    const double aU_dDD200 = FDPart1_8*(FDPart1_13 + FDPart1_6 + FDPart1_Rational_4_3*aU2_i0m1_i1_i2 + FDPart1_Rational_4_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU2_i0m2_i1_i2);
    const double aU_dDD211 = FDPart1_10*(FDPart1_13 + FDPart1_Rational_4_3*aU2_i0_i1m1_i2 + FDPart1_Rational_4_3*aU2_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU2_i0_i1m2_i2 + FDPart1_Rational_m1_12*aU2_i0_i1p2_i2);
    const double aU_dDD222 = FDPart1_11*(FDPart1_13 + FDPart1_7 + FDPart1_Rational_4_3*aU2_i0_i1_i2m1 + FDPart1_Rational_4_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU2_i0_i1_i2m2);
    const double psi_dD0 = invdx0*(FDPart1_14 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_15 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_16 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_8*(FDPart1_14 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_10*(FDPart1_15 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_11*(FDPart1_16 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    const double FDPart3_0 = (1.0/((f0_of_xx0__D0)));
    const double FDPart3_1 = FDPart3_0*psi_dD0;
    const double FDPart3_2 = (1.0/((f0_of_xx0)));
    const double FDPart3_3 = (1.0/((f4_of_xx2)));
    const double FDPart3_4 = ((f0_of_xx0__D0)*(f0_of_xx0__D0));
    const double FDPart3_5 = (1.0/((FDPart3_4)));
    const double FDPart3_6 = (1.0/((f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_7 = FDPart3_3*f4_of_xx2__D2;
    const double FDPart3_8 = (1.0/((f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_9 = FDPart3_0*aU0;
    const double FDPart3_10 = (1.0/((f0_of_xx0__D0)*(f0_of_xx0__D0)*(f0_of_xx0__D0)));
    const double FDPart3_11 = aU0*f0_of_xx0__DD00;
    const double FDPart3_12 = FDPart3_0*(FDPart3_0*aU_dD00 - FDPart3_11*FDPart3_5);
    const double FDPart3_13 = ((f0_of_xx0__DD00)*(f0_of_xx0__DD00));
    const double FDPart3_14 = 2*FDPart3_2;
    const double FDPart3_15 = FDPart3_8*f0_of_xx0__D0;
    const double FDPart3_16 = -FDPart3_15*aU1 + FDPart3_2*aU_dD10;
    const double FDPart3_17 = FDPart3_0*FDPart3_16;
    const double FDPart3_18 = FDPart3_8*f0_of_xx0__DD00;
    const double FDPart3_19 = (1.0/((f0_of_xx0)*(f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_20 = FDPart3_0*FDPart3_3*aU_dD20;
    const double FDPart3_21 = FDPart3_6*f4_of_xx2__D2;
    const double FDPart3_22 = (1.0/((f4_of_xx2)*(f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_23 = ((f4_of_xx2__D2)*(f4_of_xx2__D2));
    rhs_gfs[IDX4(AU0GF, i0, i1, i2)] = -FDPart3_1 - eU0;
    rhs_gfs[IDX4(AU1GF, i0, i1, i2)] = -FDPart3_2*psi_dD1 - eU1;
    rhs_gfs[IDX4(AU2GF, i0, i1, i2)] = -FDPart3_3*psi_dD2 - eU2;
    rhs_gfs[IDX4(EU0GF, i0, i1, i2)] = f0_of_xx0__D0*(FDPart3_5*Gamma_dD0 - FDPart3_5*(FDPart3_0*aU_dDD000 + FDPart3_12*f0_of_xx0__DD00 - 2*FDPart3_5*aU_dD00*f0_of_xx0__DD00 + FDPart3_9*(FDPart3_0*f0_of_xx0__DDD000 - FDPart3_13*FDPart3_5) + aU0*(2*FDPart3_10*FDPart3_13 - FDPart3_5*f0_of_xx0__DDD000)) - FDPart3_6*(-FDPart3_0*FDPart3_7*aU_dD02 + FDPart3_0*aU_dDD022) - FDPart3_8*(-2*FDPart3_0*aU_dD11 + FDPart3_0*aU_dDD011 + FDPart3_10*FDPart3_11*f0_of_xx0 + FDPart3_12*f0_of_xx0 - FDPart3_9));
    rhs_gfs[IDX4(EU1GF, i0, i1, i2)] = f0_of_xx0*(-FDPart3_5*(FDPart3_14*FDPart3_16*f0_of_xx0__D0 - 2*FDPart3_15*aU_dD10 - FDPart3_17*f0_of_xx0__DD00 - FDPart3_18*aU1 + FDPart3_19*FDPart3_4*aU1 + FDPart3_2*aU1*(FDPart3_2*f0_of_xx0__DD00 - FDPart3_4*FDPart3_8) + FDPart3_2*aU_dDD100 + aU1*(-FDPart3_18 + 2*FDPart3_19*FDPart3_4)) - FDPart3_6*(-FDPart3_2*FDPart3_7*aU_dD12 + FDPart3_2*aU_dDD122) + FDPart3_8*Gamma_dD1 - FDPart3_8*(FDPart3_14*aU_dD01 + FDPart3_17*f0_of_xx0 + FDPart3_2*aU_dDD111));
    rhs_gfs[IDX4(EU2GF, i0, i1, i2)] = f4_of_xx2*(-FDPart3_5*(-FDPart3_20*f0_of_xx0__DD00 + FDPart3_3*aU_dDD200) + FDPart3_6*Gamma_dD2 - FDPart3_6*(-2*FDPart3_21*aU_dD22 + FDPart3_3*aU2*(-FDPart3_23*FDPart3_6 + FDPart3_3*f4_of_xx2__DD22) + FDPart3_3*aU_dDD222 + FDPart3_7*(-FDPart3_21*aU2 + FDPart3_3*aU_dD22) + aU2*(2*FDPart3_22*FDPart3_23 - FDPart3_6*f4_of_xx2__DD22)) - FDPart3_8*(FDPart3_20*f0_of_xx0 + FDPart3_3*aU_dDD211));
    rhs_gfs[IDX4(PSIGF, i0, i1, i2)] = -Gamma;
    rhs_gfs[IDX4(GAMMAGF, i0, i1, i2)] = -FDPart3_1*FDPart3_2 + FDPart3_10*f0_of_xx0__DD00*psi_dD0 + FDPart3_22*f4_of_xx2__D2*psi_dD2 - FDPart3_5*psi_dDD00 - FDPart3_6*psi_dDD22 - FDPart3_8*psi_dDD11;
  }
  
}

extern "C" int rhs_eval(const rfm_struct *rfmstruct, const paramstruct *params, const double *in_gfs, double *rhs_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs || !rhs_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(0, 64, 1, 4);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  hipLaunchKernelGGL(rhs_eval__gpu, grid, block, 0, stream, *rfmstruct, *params, in_gfs, rhs_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}


/* Evaluate the constraints C = Dhat_i E^i and G */
__global__ void __launch_bounds__(256) Maxwell_constraints__gpu(const rfm_struct rfmstruct, const paramstruct params, const double *__restrict__ in_gfs, double *__restrict__ aux_gfs) {
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  
  NRPY_BLOCK_COORDS(Nxx0, Nxx1, Nxx2);
  const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
  const double f0_of_xx0 = rfmstruct.f0_of_xx0[i0];
  const double f0_of_xx0__D0 = rfmstruct.f0_of_xx0__D0[i0];
  const double f0_of_xx0__DD00 = rfmstruct.f0_of_xx0__DD00[i0];
  const double f4_of_xx2 = rfmstruct.f4_of_xx2[i2];
  const double f4_of_xx2__D2 = rfmstruct.f4_of_xx2__D2[i2];
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double eU0_i0m2_i1_i2 = in_gfs[IDX4(EU0GF, i0-2,i1,i2)];
    const double eU0_i0m1_i1_i2 = in_gfs[IDX4(EU0GF, i0-1,i1,i2)];
    const double eU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double eU0_i0p1_i1_i2 = in_gfs[IDX4(EU0GF, i0+1,i1,i2)];
    const double eU0_i0p2_i1_i2 = in_gfs[IDX4(EU0GF, i0+2,i1,i2)];
    const double eU1_i0_i1m2_i2 = in_gfs[IDX4(EU1GF, i0,i1-2,i2)];
    const double eU1_i0_i1m1_i2 = in_gfs[IDX4(EU1GF, i0,i1-1,i2)];
    const double eU1_i0_i1p1_i2 = in_gfs[IDX4(EU1GF, i0,i1+1,i2)];
    const double eU1_i0_i1p2_i2 = in_gfs[IDX4(EU1GF, i0,i1+2,i2)];
    const double eU2_i0_i1_i2m2 = in_gfs[IDX4(EU2GF, i0,i1,i2-2)];
    const double eU2_i0_i1_i2m1 = in_gfs[IDX4(EU2GF, i0,i1,i2-1)];
    const double eU2_i0_i1_i2p1 = in_gfs[IDX4(EU2GF, i0,i1,i2+1)];
    const double eU2_i0_i1_i2p2 = in_gfs[IDX4(EU2GF, i0,i1,i2+2)];
    const double aU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double aU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double aU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double aU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double aU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double aU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double aU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double aU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double aU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double aU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double aU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double aU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double aU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double aU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    const double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double aU_dD00 = invdx0*(FDPart1_Rational_1_12*aU0_i0m2_i1_i2 + FDPart1_Rational_2_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU0_i0p2_i1_i2 + FDPart1_Rational_m2_3*aU0_i0m1_i1_i2);
    const double aU_dD11 = invdx1*(FDPart1_Rational_1_12*aU1_i0_i1m2_i2 + FDPart1_Rational_2_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU1_i0_i1p2_i2 + FDPart1_Rational_m2_3*aU1_i0_i1m1_i2);
    const double aU_dD22 = invdx2*(FDPart1_Rational_1_12*aU2_i0_i1_i2m2 + FDPart1_Rational_2_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU2_i0_i1_i2p2 + FDPart1_Rational_m2_3*aU2_i0_i1_i2m1);
    const double eU_dD00 = invdx0*(FDPart1_Rational_1_12*eU0_i0m2_i1_i2 + FDPart1_Rational_2_3*eU0_i0p1_i1_i2 + FDPart1_Rational_m1_12*eU0_i0p2_i1_i2 + FDPart1_Rational_m2_3*eU0_i0m1_i1_i2);
    const double eU_dD11 = invdx1*(FDPart1_Rational_1_12*eU1_i0_i1m2_i2 + FDPart1_Rational_2_3*eU1_i0_i1p1_i2 + FDPart1_Rational_m1_12*eU1_i0_i1p2_i2 + FDPart1_Rational_m2_3*eU1_i0_i1m1_i2);
    const double eU_dD22 = invdx2*(FDPart1_Rational_1_12*eU2_i0_i1_i2m2 + FDPart1_Rational_2_3*eU2_i0_i1_i2p1 + FDPart1_Rational_m1_12*eU2_i0_i1_i2p2 + FDPart1_Rational_m2_3*eU2_i0_i1_i2m1);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    const double FDPart3_0 = (1.0/((f0_of_xx0)));
    const double FDPart3_1 = (1.0/((f0_of_xx0__D0)));
    const double FDPart3_2 = (1.0/((f4_of_xx2)));
    aux_gfs[IDX4(CGF, i0, i1, i2)] = FDPart3_0*eU0 + FDPart3_0*eU_dD11 + FDPart3_1*eU_dD00 + FDPart3_2*eU_dD22;
    aux_gfs[IDX4(GGF, i0, i1, i2)] = FDPart3_0*aU0 - FDPart3_0*aU_dD11 - FDPart3_1*aU_dD00 - FDPart3_2*aU_dD22 + Gamma + 2*aU0*f0_of_xx0__DD00/((f0_of_xx0__D0)*(f0_of_xx0__D0)) + 2*aU2*f4_of_xx2__D2/((f4_of_xx2)*(f4_of_xx2));
  }
  
}

extern "C" int Maxwell_constraints(const rfm_struct *rfmstruct, const paramstruct *params, const double *in_gfs, double *aux_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs || !aux_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(1, 64, 1, 4);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  hipLaunchKernelGGL(Maxwell_constraints__gpu, grid, block, 0, stream, *rfmstruct, *params, in_gfs, aux_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}

template <int S>
__global__ void __launch_bounds__(256) rhs_eval_rk4_substep__gpu(const paramstruct params, const rfm_struct rfmstruct, const double *__restrict__ auxevol_gfs, const double *__restrict__ in_gfs, double *rk_yn, double *rk_rt, double *rk_out, const double dt) {
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  NRPY_BLOCK_COORDS(Nxx0, Nxx1, Nxx2);
  const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
  const double f0_of_xx0 = rfmstruct.f0_of_xx0[i0];
  const double f0_of_xx0__D0 = rfmstruct.f0_of_xx0__D0[i0];
  const double f0_of_xx0__DD00 = rfmstruct.f0_of_xx0__DD00[i0];
  const double f0_of_xx0__DDD000 = rfmstruct.f0_of_xx0__DDD000[i0];
  const double f4_of_xx2 = rfmstruct.f4_of_xx2[i2];
  const double f4_of_xx2__D2 = rfmstruct.f4_of_xx2__D2[i2];
  const double f4_of_xx2__DD22 = rfmstruct.f4_of_xx2__DD22[i2];
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double eU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double eU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double eU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double aU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double aU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double aU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double aU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double aU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double aU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double aU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double aU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double aU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double aU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double aU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double aU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double aU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double aU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double aU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double aU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double aU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double aU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double aU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double aU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double aU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double aU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double aU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double aU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double aU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double aU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double aU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double aU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double aU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double aU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double aU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double aU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double aU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double aU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double aU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double aU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double aU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double aU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double aU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    const double psi_i0_i1_i2m2 = in_gfs[IDX4(PSIGF, i0,i1,i2-2)];
    const double psi_i0_i1_i2m1 = in_gfs[IDX4(PSIGF, i0,i1,i2-1)];
    const double psi_i0_i1m2_i2 = in_gfs[IDX4(PSIGF, i0,i1-2,i2)];
    const double psi_i0_i1m1_i2 = in_gfs[IDX4(PSIGF, i0,i1-1,i2)];
    const double psi_i0m2_i1_i2 = in_gfs[IDX4(PSIGF, i0-2,i1,i2)];
    const double psi_i0m1_i1_i2 = in_gfs[IDX4(PSIGF, i0-1,i1,i2)];
    const double psi = in_gfs[IDX4(PSIGF, i0,i1,i2)];
    const double psi_i0p1_i1_i2 = in_gfs[IDX4(PSIGF, i0+1,i1,i2)];
    const double psi_i0p2_i1_i2 = in_gfs[IDX4(PSIGF, i0+2,i1,i2)];
    const double psi_i0_i1p1_i2 = in_gfs[IDX4(PSIGF, i0,i1+1,i2)];
    const double psi_i0_i1p2_i2 = in_gfs[IDX4(PSIGF, i0,i1+2,i2)];
    const double psi_i0_i1_i2p1 = in_gfs[IDX4(PSIGF, i0,i1,i2+1)];
    const double psi_i0_i1_i2p2 = in_gfs[IDX4(PSIGF, i0,i1,i2+2)];
    const double Gamma_i0_i1_i2m2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-2)];
    const double Gamma_i0_i1_i2m1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-1)];
    const double Gamma_i0_i1m2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-2,i2)];
    const double Gamma_i0_i1m1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-1,i2)];
    const double Gamma_i0m2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-2,i1,i2)];
    const double Gamma_i0m1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-1,i1,i2)];
    const double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    const double Gamma_i0p1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+1,i1,i2)];
    const double Gamma_i0p2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+2,i1,i2)];
    const double Gamma_i0_i1p1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+1,i2)];
    const double Gamma_i0_i1p2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+2,i2)];
    const double Gamma_i0_i1_i2p1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+1)];
    const double Gamma_i0_i1_i2p2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+2)];
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_4_3 = 4.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double FDPart1_Rational_m5_2 = -5.0/2.0;
    const double FDPart1_0 = FDPart1_Rational_m1_12*aU0_i0p2_i1_i2;
    const double FDPart1_1 = FDPart1_Rational_m1_12*aU0_i0_i1p2_i2;
    const double FDPart1_2 = FDPart1_Rational_m1_12*aU0_i0_i1_i2p2;
    const double FDPart1_3 = FDPart1_Rational_m1_12*aU1_i0p2_i1_i2;
    const double FDPart1_4 = FDPart1_Rational_m1_12*aU1_i0_i1p2_i2;
    const double FDPart1_5 = FDPart1_Rational_m1_12*aU1_i0_i1_i2p2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*aU2_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*aU2_i0_i1_i2p2;
    const double FDPart1_8 = ((invdx0)*(invdx0));
    const double FDPart1_9 = FDPart1_Rational_m5_2*aU0;
    const double FDPart1_10 = ((invdx1)*(invdx1));
    const double FDPart1_11 = ((invdx2)*(invdx2));
    const double FDPart1_12 = FDPart1_Rational_m5_2*aU1;
    const double FDPart1_13 = FDPart1_Rational_m5_2*aU2;
    const double FDPart1_14 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_15 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_16 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_17 = FDPart1_Rational_m5_2*psi;
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double aU_dD00 = invdx0*(FDPart1_0 + FDPart1_Rational_1_12*aU0_i0m2_i1_i2 + FDPart1_Rational_2_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU0_i0m1_i1_i2);
    const double aU_dD01 = invdx1*(FDPart1_1 + FDPart1_Rational_1_12*aU0_i0_i1m2_i2 + FDPart1_Rational_2_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU0_i0_i1m1_i2);
    const double aU_dD02 = invdx2*(FDPart1_2 + FDPart1_Rational_1_12*aU0_i0_i1_i2m2 + FDPart1_Rational_2_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU0_i0_i1_i2m1);
    const double aU_dD10 = invdx0*(FDPart1_3 + FDPart1_Rational_1_12*aU1_i0m2_i1_i2 + FDPart1_Rational_2_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU1_i0m1_i1_i2);
    const double aU_dD11 = invdx1*(FDPart1_4 + FDPart1_Rational_1_12*aU1_i0_i1m2_i2 + FDPart1_Rational_2_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU1_i0_i1m1_i2);
    const double aU_dD12 = invdx2*(FDPart1_5 + FDPart1_Rational_1_12*aU1_i0_i1_i2m2 + FDPart1_Rational_2_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU1_i0_i1_i2m1);
    const double aU_dD20 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*aU2_i0m2_i1_i2 + FDPart1_Rational_2_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU2_i0m1_i1_i2);
    const double aU_dD22 = invdx2*(FDPart1_7 + FDPart1_Rational_1_12*aU2_i0_i1_i2m2 + FDPart1_Rational_2_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU2_i0_i1_i2m1);
    const double aU_dDD000 = FDPart1_8*(FDPart1_0 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0m1_i1_i2 + FDPart1_Rational_4_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU0_i0m2_i1_i2);
    const double aU_dDD011 = FDPart1_10*(FDPart1_1 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1m1_i2 + FDPart1_Rational_4_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU0_i0_i1m2_i2);
    const double aU_dDD022 = FDPart1_11*(FDPart1_2 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1_i2m1 + FDPart1_Rational_4_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU0_i0_i1_i2m2);
    const double aU_dDD100 = FDPart1_8*(FDPart1_12 + FDPart1_3 + FDPart1_Rational_4_3*aU1_i0m1_i1_i2 + FDPart1_Rational_4_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU1_i0m2_i1_i2);
    const double aU_dDD111 = FDPart1_10*(FDPart1_12 + FDPart1_4 + FDPart1_Rational_4_3*aU1_i0_i1m1_i2 + FDPart1_Rational_4_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU1_i0_i1m2_i2);
    const double aU_dDD122 = FDPart1_11*(FDPart1_12 + FDPart1_5 + FDPart1_Rational_4_3*aU1_i0_i1_i2m1 + FDPart1_Rational_4_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU1_i0_i1_i2m2);
    const double aU_dDD200 = FDPart1_8*(FDPart1_13 + FDPart1_6 + FDPart1_Rational_4_3*aU2_i0m1_i1_i2 + FDPart1_Rational_4_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU2_i0m2_i1_i2);
    const double aU_dDD211 = FDPart1_10*(FDPart1_13 + FDPart1_Rational_4_3*aU2_i0_i1m1_i2 + FDPart1_Rational_4_3*aU2_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU2_i0_i1m2_i2 + FDPart1_Rational_m1_12*aU2_i0_i1p2_i2);
    const double aU_dDD222 = FDPart1_11*(FDPart1_13 + FDPart1_7 + FDPart1_Rational_4_3*aU2_i0_i1_i2m1 + FDPart1_Rational_4_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU2_i0_i1_i2m2);
    const double psi_dD0 = invdx0*(FDPart1_14 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_15 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_16 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_8*(FDPart1_14 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_10*(FDPart1_15 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_11*(FDPart1_16 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    const double FDPart3_0 = (1.0/((f0_of_xx0__D0)));
    const double FDPart3_1 = FDPart3_0*psi_dD0;
    const double FDPart3_2 = (1.0/((f0_of_xx0)));
    const double FDPart3_3 = (1.0/((f4_of_xx2)));
    const double FDPart3_4 = ((f0_of_xx0__D0)*(f0_of_xx0__D0));
    const double FDPart3_5 = (1.0/((FDPart3_4)));
    const double FDPart3_6 = (1.0/((f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_7 = FDPart3_3*f4_of_xx2__D2;
    const double FDPart3_8 = (1.0/((f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_9 = FDPart3_0*aU0;
    const double FDPart3_10 = (1.0/((f0_of_xx0__D0)*(f0_of_xx0__D0)*(f0_of_xx0__D0)));
    const double FDPart3_11 = aU0*f0_of_xx0__DD00;
    const double FDPart3_12 = FDPart3_0*(FDPart3_0*aU_dD00 - FDPart3_11*FDPart3_5);
    const double FDPart3_13 = ((f0_of_xx0__DD00)*(f0_of_xx0__DD00));
    const double FDPart3_14 = 2*FDPart3_2;
    const double FDPart3_15 = FDPart3_8*f0_of_xx0__D0;
    const double FDPart3_16 = -FDPart3_15*aU1 + FDPart3_2*aU_dD10;
    const double FDPart3_17 = FDPart3_0*FDPart3_16;
    const double FDPart3_18 = FDPart3_8*f0_of_xx0__DD00;
    const double FDPart3_19 = (1.0/((f0_of_xx0)*(f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_20 = FDPart3_0*FDPart3_3*aU_dD20;
    const double FDPart3_21 = FDPart3_6*f4_of_xx2__D2;
    const double FDPart3_22 = (1.0/((f4_of_xx2)*(f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_23 = ((f4_of_xx2__D2)*(f4_of_xx2__D2));
  const double __rhs_AU0 = -FDPart3_1 - eU0;
  const double __rhs_AU1 = -FDPart3_2*psi_dD1 - eU1;
  const double __rhs_AU2 = -FDPart3_3*psi_dD2 - eU2;
  const double __rhs_EU0 = f0_of_xx0__D0*(FDPart3_5*Gamma_dD0 - FDPart3_5*(FDPart3_0*aU_dDD000 + FDPart3_12*f0_of_xx0__DD00 - 2*FDPart3_5*aU_dD00*f0_of_xx0__DD00 + FDPart3_9*(FDPart3_0*f0_of_xx0__DDD000 - FDPart3_13*FDPart3_5) + aU0*(2*FDPart3_10*FDPart3_13 - FDPart3_5*f0_of_xx0__DDD000)) - FDPart3_6*(-FDPart3_0*FDPart3_7*aU_dD02 + FDPart3_0*aU_dDD022) - FDPart3_8*(-2*FDPart3_0*aU_dD11 + FDPart3_0*aU_dDD011 + FDPart3_10*FDPart3_11*f0_of_xx0 + FDPart3_12*f0_of_xx0 - FDPart3_9));
  const double __rhs_EU1 = f0_of_xx0*(-FDPart3_5*(FDPart3_14*FDPart3_16*f0_of_xx0__D0 - 2*FDPart3_15*aU_dD10 - FDPart3_17*f0_of_xx0__DD00 - FDPart3_18*aU1 + FDPart3_19*FDPart3_4*aU1 + FDPart3_2*aU1*(FDPart3_2*f0_of_xx0__DD00 - FDPart3_4*FDPart3_8) + FDPart3_2*aU_dDD100 + aU1*(-FDPart3_18 + 2*FDPart3_19*FDPart3_4)) - FDPart3_6*(-FDPart3_2*FDPart3_7*aU_dD12 + FDPart3_2*aU_dDD122) + FDPart3_8*Gamma_dD1 - FDPart3_8*(FDPart3_14*aU_dD01 + FDPart3_17*f0_of_xx0 + FDPart3_2*aU_dDD111));
  const double __rhs_EU2 = f4_of_xx2*(-FDPart3_5*(-FDPart3_20*f0_of_xx0__DD00 + FDPart3_3*aU_dDD200) + FDPart3_6*Gamma_dD2 - FDPart3_6*(-2*FDPart3_21*aU_dD22 + FDPart3_3*aU2*(-FDPart3_23*FDPart3_6 + FDPart3_3*f4_of_xx2__DD22) + FDPart3_3*aU_dDD222 + FDPart3_7*(-FDPart3_21*aU2 + FDPart3_3*aU_dD22) + aU2*(2*FDPart3_22*FDPart3_23 - FDPart3_6*f4_of_xx2__DD22)) - FDPart3_8*(FDPart3_20*f0_of_xx0 + FDPart3_3*aU_dDD211));
  const double __rhs_PSI = -Gamma;
  const double __rhs_GAMMA = -FDPart3_1*FDPart3_2 + FDPart3_10*f0_of_xx0__DD00*psi_dD0 + FDPart3_22*f4_of_xx2__D2*psi_dD2 - FDPart3_5*psi_dDD00 - FDPart3_6*psi_dDD22 - FDPart3_8*psi_dDD11;
  __builtin_amdgcn_sched_barrier(0);
  NRPY_RK4_PRELOAD(S, AU0GF, 0)
  NRPY_RK4_PRELOAD(S, AU1GF, 1)
  NRPY_RK4_PRELOAD(S, AU2GF, 2)
  NRPY_RK4_PRELOAD(S, EU0GF, 3)
  NRPY_RK4_PRELOAD(S, EU1GF, 4)
  NRPY_RK4_PRELOAD(S, EU2GF, 5)
  NRPY_RK4_PRELOAD(S, PSIGF, 6)
  NRPY_RK4_PRELOAD(S, GAMMAGF, 7)
  NRPY_RK4_STORE(S, 0, __rhs_AU0);
  NRPY_RK4_STORE(S, 1, __rhs_AU1);
  NRPY_RK4_STORE(S, 2, __rhs_AU2);
  NRPY_RK4_STORE(S, 3, __rhs_EU0);
  NRPY_RK4_STORE(S, 4, __rhs_EU1);
  NRPY_RK4_STORE(S, 5, __rhs_EU2);
  NRPY_RK4_STORE(S, 6, __rhs_PSI);
  NRPY_RK4_STORE(S, 7, __rhs_GAMMA);
  }
}
extern "C" int rhs_eval_rk4_substep(const int S, const rfm_struct *rfmstruct, const paramstruct *params, const double *auxevol_gfs, const double *in_gfs, double *y_n, double *rt, double *out, const double dt, hipStream_t stream) {
  if (!params || !y_n || !rt || !out) return NRPY_ERR_NULL;
  if (S < 0 || S > 3) return NRPY_ERR_PARAM;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(2, 64, 1, 4);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<0>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt); break;
    case 1: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<1>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt); break;
    case 2: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<2>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt); break;
    case 3: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<3>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}


/* Set up the initial data at all points on the numerical grid. */
__global__ void __launch_bounds__(256) initial_data__gpu(const paramstruct params, const double *__restrict__ xx0_arr, const double *__restrict__ xx1_arr, const double *__restrict__ xx2_arr, double *__restrict__ in_gfs) {
  const double AMPLRHO = params.AMPLRHO;
  const double AMPLZ = params.AMPLZ;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  const double SINHWRHO = params.SINHWRHO;
  const double SINHWZ = params.SINHWZ;
  const double amp = params.amp;
  const double lam = params.lam;
  const double time = params.time;
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  
  NRPY_BLOCK_COORDS_POINTWISE(Nxx_plus_2NGHOSTS0, Nxx_plus_2NGHOSTS1, Nxx_plus_2NGHOSTS2);
  const int i0 = 0 + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = 0 + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = 0 + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx_plus_2NGHOSTS0 || i1 >= Nxx_plus_2NGHOSTS1 || i2 >= Nxx_plus_2NGHOSTS2) return;
  const double xx0 = xx0_arr[i0];
  const double xx1 = xx1_arr[i1];
  const double xx2 = xx2_arr[i2];
  const double tmp_0 = (1.0/((SINHWZ)));
  const double tmp_1 = exp(tmp_0);
  const double tmp_2 = (1.0/((SINHWRHO)));
  const double tmp_3 = exp(tmp_2);
  const double tmp_4 = tmp_2*xx0;
  const double tmp_5 = exp(tmp_4);
  const double tmp_6 = tmp_0*xx2;
  const double tmp_7 = exp(tmp_6);
  const double tmp_8 = SINHWZ*tmp_5*tmp_7;
  const double tmp_9 = tmp_3*tmp_8;
  const double tmp_10 = tmp_1*tmp_9;
  const double tmp_11 = exp(-tmp_2);
  const double tmp_12 = tmp_11*tmp_8;
  const double tmp_13 = tmp_1*tmp_12;
  const double tmp_14 = exp(-tmp_0);
  const double tmp_15 = tmp_14*tmp_9;
  const double tmp_16 = tmp_12*tmp_14;
  const double tmp_17 = (1.0/((tmp_10 - tmp_13 - tmp_15 + tmp_16)));
  const double tmp_18 = tmp_1 - tmp_14;
  const double tmp_19 = exp(-tmp_6);
  const double tmp_20 = sin(xx1);
  const double tmp_21 = ((tmp_20)*(tmp_20));
  const double tmp_22 = exp(-tmp_4);
  const double tmp_23 = -tmp_22 + tmp_5;
  const double tmp_24 = -tmp_11 + tmp_3;
  const double tmp_25 = ((AMPLRHO)*(AMPLRHO))/((tmp_24)*(tmp_24));
  const double tmp_26 = ((tmp_23)*(tmp_23))*tmp_25;
  const double tmp_27 = cos(xx1);
  const double tmp_28 = ((tmp_27)*(tmp_27));
  const double tmp_29 = ((AMPLZ)*(AMPLZ))*((-tmp_19 + tmp_7)*(-tmp_19 + tmp_7))/((tmp_18)*(tmp_18)) + tmp_21*tmp_26 + tmp_26*tmp_28;
  const double tmp_30 = sqrt(tmp_29);
  const double tmp_31 = time - tmp_30;
  const double tmp_32 = ((tmp_31)*(tmp_31));
  const double tmp_33 = exp(lam*tmp_32);
  const double tmp_34 = time + tmp_30;
  const double tmp_35 = ((tmp_34)*(tmp_34));
  const double tmp_36 = exp(lam*tmp_35);
  const double tmp_37 = tmp_31*tmp_36;
  const double tmp_38 = tmp_33*tmp_34;
  const double tmp_39 = 2*lam*tmp_29;
  const double tmp_40 = tmp_2*tmp_22 + tmp_2*tmp_5;
  const double tmp_41 = AMPLZ*tmp_23*tmp_25*tmp_40*(tmp_0*tmp_19 + tmp_0*tmp_7)/tmp_18;
  const double tmp_42 = (1.0/((tmp_21*tmp_41 + tmp_28*tmp_41)));
  const double tmp_43 = (1.0/((tmp_29)*(tmp_29)));
  const double tmp_44 = exp(-lam*(tmp_32 + tmp_35));
  const double tmp_45 = (1.0/((tmp_24)));
  const double tmp_46 = AMPLRHO*tmp_45;
  const double tmp_47 = tmp_23*tmp_46;
  const double tmp_48 = amp*tmp_42*tmp_43*tmp_44*tmp_47;
  const double tmp_49 = tmp_48*(tmp_30*(tmp_33 - tmp_36) + tmp_39*(tmp_37 + tmp_38));
  const double tmp_50 = tmp_17*tmp_49;
  const double tmp_51 = exp(2*tmp_6);
  const double tmp_52 = exp(2*tmp_4);
  const double tmp_53 = AMPLRHO*AMPLZ;
  const double tmp_54 = tmp_20*tmp_53;
  const double tmp_55 = tmp_51*tmp_54;
  const double tmp_56 = tmp_52*tmp_54 + tmp_52*tmp_55;
  const double tmp_57 = tmp_27*(AMPLRHO*AMPLZ*tmp_20*tmp_51 + AMPLRHO*AMPLZ*tmp_20 - tmp_56);
  const double tmp_58 = tmp_50*tmp_57;
  const double tmp_59 = tmp_27*tmp_53;
  const double tmp_60 = tmp_51*tmp_59;
  const double tmp_61 = tmp_52*tmp_59;
  const double tmp_62 = tmp_51*tmp_61 + tmp_61;
  const double tmp_63 = tmp_20*(-tmp_59 - tmp_60 + tmp_62);
  const double tmp_64 = tmp_50*tmp_63;
  const double tmp_65 = tmp_40*tmp_46;
  const double tmp_66 = (1.0/((SINHWRHO*tmp_10 - SINHWRHO*tmp_13 - SINHWRHO*tmp_15 + SINHWRHO*tmp_16)));
  const double tmp_67 = tmp_49*tmp_66;
  const double tmp_68 = tmp_54 + tmp_55 + tmp_56;
  const double tmp_69 = tmp_20*tmp_67*tmp_68;
  const double tmp_70 = tmp_59 + tmp_60 + tmp_62;
  const double tmp_71 = tmp_27*tmp_67*tmp_70;
  const double tmp_72 = 4*lam*time;
  const double tmp_73 = 2*time;
  const double tmp_74 = 2*tmp_30;
  const double tmp_75 = lam*(tmp_73 + tmp_74);
  const double tmp_76 = lam*(tmp_73 - tmp_74);
  const double tmp_77 = tmp_30*(tmp_33*tmp_76 - tmp_36*tmp_75) + tmp_39*(tmp_33 + tmp_36 + tmp_37*tmp_75 + tmp_38*tmp_76);
  const double tmp_78 = tmp_17*tmp_48*tmp_77;
  in_gfs[IDX4(AU0GF, i0, i1, i2)] = tmp_65*(tmp_58 + tmp_64);
  in_gfs[IDX4(AU1GF, i0, i1, i2)] = tmp_47*(-tmp_69 - tmp_71);
  in_gfs[IDX4(AU2GF, i0, i1, i2)] = 0;
  in_gfs[IDX4(EU0GF, i0, i1, i2)] = tmp_65*(-tmp_57*tmp_78 + tmp_58*tmp_72 - tmp_63*tmp_78 + tmp_64*tmp_72);
  in_gfs[IDX4(EU1GF, i0, i1, i2)] = tmp_47*(AMPLRHO*amp*tmp_20*tmp_23*tmp_42*tmp_43*tmp_44*tmp_45*tmp_66*tmp_68*tmp_77 + AMPLRHO*amp*tmp_23*tmp_27*tmp_42*tmp_43*tmp_44*tmp_45*tmp_66*tmp_70*tmp_77 - tmp_69*tmp_72 - tmp_71*tmp_72);
  in_gfs[IDX4(EU2GF, i0, i1, i2)] = 0;
  in_gfs[IDX4(GAMMAGF, i0, i1, i2)] = 0;
  in_gfs[IDX4(PSIGF, i0, i1, i2)] = 0;
  
}

extern "C" int initial_data(const paramstruct *params, double *xx[3], double *in_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(3, 64, 1, 4);
  const dim3 grid(nrpy_nblocks(block, params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2));
  hipLaunchKernelGGL(initial_data__gpu, grid, block, 0, stream, *params, xx[0], xx[1], xx[2], in_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}

// One RK4 step (MoLtimestepping/C_Code_Generation.py:266-329 for RK4): four substeps, each
// [Ricci] -> RHS + update at interior points -> ghost fill -> [det(gammabar) enforcement].
extern "C" int MoL_step_forward_in_time(const rfm_struct *rfmstruct, const paramstruct *params, const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, double *auxevol_gfs, const double dt, hipStream_t stream) {
  if (!rfmstruct || !params || !bcstruct || !y_n_gfs || !k_odd_gfs || !k_even_gfs ||
      !y_nplus1_running_total_gfs) return NRPY_ERR_NULL;
  int rc;
  /* substep 0: y_n_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep(0, rfmstruct, params, auxevol_gfs, y_n_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  if ((rc = nrpy_stage_fill(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, stream))) return rc;
  /* substep 1: k_odd_gfs -> k_even_gfs */
  if ((rc = rhs_eval_rk4_substep(1, rfmstruct, params, auxevol_gfs, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, dt, stream))) return rc;
  if ((rc = nrpy_stage_fill(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_even_gfs, stream))) return rc;
  /* substep 2: k_even_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep(2, rfmstruct, params, auxevol_gfs, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  if ((rc = nrpy_stage_fill(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, stream))) return rc;
  /* substep 3: k_odd_gfs -> y_n_gfs */
  if ((rc = rhs_eval_rk4_substep(3, rfmstruct, params, auxevol_gfs, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, dt, stream))) return rc;
  if ((rc = apply_bcs_curvilinear_composed(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, y_n_gfs, stream))) return rc;
  return NRPY_OK;
}

struct MoL_graph {
  hipGraph_t graph;
  hipGraphExec_t exec;
  double *scratch = nullptr;  // device memory of the captured Sommerfeld step, owned by the graph
  paramstruct params;         // what its geometry table is computed from at each launch
  const double *xx[3];
};
static int nrpy_sommerfeld_geometry_fill(const paramstruct *params, const double *const xx[3], double *scratch, hipStream_t stream);
// Capture one RK4 step into a hipGraph; replay with MoL_graph_launch. Pointers and dt are fixed
// at capture time.
extern "C" int MoL_graph_create(const rfm_struct *rfmstruct, const paramstruct *params, const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, double *auxevol_gfs, const double dt, MoL_graph **out) {
  if (!out) return NRPY_ERR_NULL;
  *out = nullptr;
  hipStream_t s;
  if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return NRPY_ERR_LAUNCH;
  MoL_graph *g = new MoL_graph();
  int rc = NRPY_OK;
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) rc = NRPY_ERR_LAUNCH;
  if (!rc) {
    rc = MoL_step_forward_in_time(rfmstruct, params, bcstruct, y_n_gfs, k_odd_gfs, k_even_gfs,
                                  y_nplus1_running_total_gfs, auxevol_gfs, dt, s);
    hipGraph_t gr;
    const hipError_t e = hipStreamEndCapture(s, &gr);
    if (!rc && e != hipSuccess) rc = NRPY_ERR_LAUNCH;
    if (!rc) {
      g->graph = gr;
      if (hipGraphInstantiate(&g->exec, gr, nullptr, nullptr, 0) != hipSuccess) rc = NRPY_ERR_LAUNCH;
    }
  }
  (void)hipStreamDestroy(s);
  if (rc) { delete g; return rc; }
  *out = g;
  return NRPY_OK;
}
extern "C" int MoL_graph_launch(MoL_graph *g, const int nsteps, hipStream_t stream) {
  if (!g) return NRPY_ERR_NULL;
  if (nsteps < 0) return NRPY_ERR_PARAM;
  // in the stream's order, as the replays themselves: the coordinates are those of this launch
  if (g->scratch && nsteps > 0) {
    const int rc = nrpy_sommerfeld_geometry_fill(&g->params, g->xx, g->scratch, stream);
    if (rc) return rc;
  }
  for (int n = 0; n < nsteps; n++)
    if (hipGraphLaunch(g->exec, stream) != hipSuccess) return NRPY_ERR_LAUNCH;
  return NRPY_OK;
}
extern "C" void MoL_graph_free(MoL_graph *g) {
  if (!g) return;
  (void)hipGraphExecDestroy(g->exec);
  (void)hipGraphDestroy(g->graph);
  (void)hipFree(g->scratch);
  delete g;
}

// One RK4 step with the Sommerfeld radiation condition on the RHS.
// Sommerfeld EVOL grid function parameters
static __constant__ double evolgf_at_inf[NUM_EVOL_GFS] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
static __constant__ double evolgf_radial_falloff_power[NUM_EVOL_GFS] = {3.0, 3.0, 3.0, 3.0, 3.0, 3.0, 3.0, 3.0};
static __constant__ double evolgf_speed[NUM_EVOL_GFS] = {1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
#define NRPY_SOMMERFELD_MIN_N (NGHOSTS + 4 + 1)
#define NRPY_SOMMERFELD_FD 4
// r and d f/d r at (i0,i1,i2) of one gridfunction f, read as fa(i0,i1,i2); F = the point's
// FACE (CurviBoundaryConditions.py:329-516).
template <typename FA>
static __device__ void nrpy_sommerfeld_r_dfdr(const paramstruct &params, const double *__restrict__ xx0_arr, const double *__restrict__ xx1_arr, const double *__restrict__ xx2_arr, FA fa, const int F0, const int F1, const int F2, const int i0, const int i1, const int i2, double *r_out, double *dfdr_out) {
  const double AMPLRHO = params.AMPLRHO;
  const double AMPLZ = params.AMPLZ;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  const double SINHWRHO = params.SINHWRHO;
  const double SINHWZ = params.SINHWZ;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const double xx0 = xx0_arr[i0], xx1 = xx1_arr[i1], xx2 = xx2_arr[i2];
  (void)xx0; (void)xx1; (void)xx2; (void)F0; (void)F1; (void)F2;
  double fdD0 = 1e100, fdD1 = 1e100, fdD2 = 1e100;
  (void)fdD0; (void)fdD1; (void)fdD2;
  const double u0 = -25./12., u1 = 4., u2 = -3., u3 = 4./3., u4 = -1./4.;
  const double c1 = 2./3., c2 = 1./12.;
  {
    const bool one_sided = abs(F0) == 1 || i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0 || i0 - NGHOSTS <= 0;
    int S = F0;
    if (i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0) S = -1;
    if (i0 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic0 = min(max(i0, 2), Nxx_plus_2NGHOSTS0 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0+1*S,i1,i2) + u2*fa(i0+2*S,i1,i2) + u3*fa(i0+3*S,i1,i2) + u4*fa(i0+4*S,i1,i2))*invdx0;
    const double cen = (-c2*fa(nrpy_ic0+2,i1,i2) + c1*fa(nrpy_ic0+1,i1,i2) - c1*fa(nrpy_ic0+-1,i1,i2) + c2*fa(nrpy_ic0+-2,i1,i2))*invdx0;
    fdD0 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F1) == 1 || i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1 || i1 - NGHOSTS <= 0;
    int S = F1;
    if (i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1) S = -1;
    if (i1 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic1 = min(max(i1, 2), Nxx_plus_2NGHOSTS1 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0,i1+1*S,i2) + u2*fa(i0,i1+2*S,i2) + u3*fa(i0,i1+3*S,i2) + u4*fa(i0,i1+4*S,i2))*invdx1;
    const double cen = (-c2*fa(i0,nrpy_ic1+2,i2) + c1*fa(i0,nrpy_ic1+1,i2) - c1*fa(i0,nrpy_ic1+-1,i2) + c2*fa(i0,nrpy_ic1+-2,i2))*invdx1;
    fdD1 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F2) == 1 || i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2 || i2 - NGHOSTS <= 0;
    int S = F2;
    if (i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2) S = -1;
    if (i2 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic2 = min(max(i2, 2), Nxx_plus_2NGHOSTS2 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0,i1,i2+1*S) + u2*fa(i0,i1,i2+2*S) + u3*fa(i0,i1,i2+3*S) + u4*fa(i0,i1,i2+4*S))*invdx2;
    const double cen = (-c2*fa(i0,i1,nrpy_ic2+2) + c1*fa(i0,i1,nrpy_ic2+1) - c1*fa(i0,i1,nrpy_ic2+-1) + c2*fa(i0,i1,nrpy_ic2+-2))*invdx2;
    fdD2 = one_sided ? one : cen;
  }
  double J00, J01, J02, J10, J11, J12, J20, J21, J22;
  const double tmp_0 = (1.0/((SINHWRHO)));
  const double tmp_1 = tmp_0*xx0;
  const double tmp_2 = exp(tmp_1);
  const double tmp_3 = exp(-tmp_1);
  const double tmp_4 = tmp_2 - tmp_3;
  const double tmp_5 = ((AMPLRHO)*(AMPLRHO))/((exp(tmp_0) - exp(-tmp_0))*(exp(tmp_0) - exp(-tmp_0)));
  const double tmp_6 = (1.0/((SINHWZ)));
  const double tmp_7 = tmp_6*xx2;
  const double tmp_8 = exp(tmp_7);
  const double tmp_9 = exp(-tmp_7);
  const double tmp_10 = tmp_8 - tmp_9;
  const double tmp_11 = ((tmp_10)*(tmp_10));
  const double tmp_12 = exp(tmp_6) - exp(-tmp_6);
  const double tmp_13 = ((AMPLZ)*(AMPLZ))/((tmp_12)*(tmp_12));
  const double tmp_14 = tmp_11*tmp_13;
  const double tmp_15 = tmp_14 + ((tmp_4)*(tmp_4))*tmp_5;
  const double tmp_16 = sqrt(tmp_15);
  const double tmp_17 = (1.0/((tmp_16)));
  const double tmp_18 = ((1.0/2.0))*tmp_17;
  const double tmp_19 = 2*tmp_0;
  const double tmp_20 = tmp_4*tmp_5*(tmp_19*tmp_2 + tmp_19*tmp_3);
  const double tmp_21 = tmp_6*tmp_8;
  const double tmp_22 = tmp_6*tmp_9;
  const double tmp_23 = 2*tmp_21 + 2*tmp_22;
  const double tmp_24 = (1.0/sqrt(-tmp_14/tmp_15 + 1));
  const double tmp_25 = (1.0/((tmp_12)));
  const double tmp_26 = ((1.0/2.0))/pow(tmp_15, (3.0/2.0));
  *r_out = tmp_16;
  J00 = tmp_18*tmp_20;
  J01 = 0;
  J02 = tmp_10*tmp_13*tmp_18*tmp_23;
  J10 = AMPLZ*tmp_10*tmp_20*tmp_24*tmp_25*tmp_26;
  J11 = 0;
  J12 = -tmp_24*(-((AMPLZ)*(AMPLZ)*(AMPLZ))*tmp_11*tmp_23*tmp_26/((tmp_12)*(tmp_12)*(tmp_12)) + AMPLZ*tmp_17*tmp_25*(tmp_21 + tmp_22));
  J20 = 0;
  J21 = 1;
  J22 = 0;
  const double cof0 = J11*J22 - J12*J21, cof1 = -(J10*J22 - J12*J20), cof2 = J10*J21 - J11*J20;
  *dfdr_out = (fdD0*cof0 + fdD1*cof1 + fdD2*cof2)/(J00*cof0 + J01*cof1 + J02*cof2);
}

// The radiation condition's right-hand side at outer point (i0,i1,i2) of gridfunction gf
// (apply_bcs_sommerfeld in CurviBoundaryConditions.py:538-620). fa(i,j,k): that gridfunction
// of the state the RHS is evaluated from; rn(o): the same gridfunction's RHS at the point's
// inward neighbour (i0,i1,i2) + FACE, flat index o.
// (r_offset / r)^n: the falloff powers in use are small integers (2 or 3), for which products
// replace the general FP64 pow, the largest part of a lane's arithmetic in the face kernels
// (within 2 ulp of the rounded power); any other power takes pow.
__device__ __forceinline__ double nrpy_som_falloff(const double q, const double n) {
  return n == 3.0 ? q * q * q : n == 2.0 ? q * q : n == 1.0 ? q : pow(q, n);
}
template <typename FA, typename RN>
__device__ __forceinline__ double nrpy_sommerfeld_rhs(const paramstruct &params, const double *__restrict__ xx0,
                                                      const double *__restrict__ xx1, const double *__restrict__ xx2,
                                                      const int gf, const int i0, const int i1, const int i2,
                                                      const int F0, const int F1, const int F2, FA fa, RN rn) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const double char_speed = evolgf_speed[gf];
  const double var_at_infinity = evolgf_at_inf[gf];
  const double radial_falloff_power = evolgf_radial_falloff_power[gf];
  double r = 1e100, partial_i_f = 1e100;
  nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, F1, F2, i0, i1, i2, &r, &partial_i_f);
  const double invr = 1. / r;
  const double source_rhs = -char_speed * (partial_i_f + invr * (fa(i0, i1, i2) - var_at_infinity));
  double out = source_rhs;
  if (radial_falloff_power > 0) {
    const int j0 = i0 + F0, j1 = i1 + F1, j2 = i2 + F2;
    double r_offset = 1e100, partial_i_f_offset = 1e100;
    nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, F1, F2, j0, j1, j2, &r_offset, &partial_i_f_offset);
    const double invr_offset = 1. / r_offset;
    const size_t o = (size_t)j0 + (size_t)N0 * ((size_t)j1 + (size_t)N1 * (size_t)j2);
    const double extrap_rhs = char_speed * (partial_i_f_offset + invr_offset * (fa(j0, j1, j2) - var_at_infinity));
    const double diff_between_advection_and_f_rhs = rn(o) + extrap_rhs;
    out = source_rhs + diff_between_advection_and_f_rhs * nrpy_som_falloff(r_offset * invr, radial_falloff_power);
  }
  return out;
}
// The same along an i0-face row, layer after layer (FACE (F0, 0, 0)): the inward neighbour of
// layer gz + 1's point is layer gz's point, with the same FACE, so its r and
// X = d f/d r + (f - f_inf)/r are the ones that point computed. have_in: r_in and X_in hold
// them (from the call for the layer before); else they are evaluated at (i0 + F0, i1, i2).
// On return r_in and X_in hold this point's. rn: the neighbour's RHS.
template <typename FA>
__device__ __forceinline__ double nrpy_sommerfeld_rhs_row(const paramstruct &params, const double *__restrict__ xx0,
                                                          const double *__restrict__ xx1,
                                                          const double *__restrict__ xx2, const int gf, const int i0,
                                                          const int i1, const int i2, const int F0, FA fa,
                                                          const double rn, const bool have_in, double &r_in,
                                                          double &X_in) {
  const double char_speed = evolgf_speed[gf];
  const double var_at_infinity = evolgf_at_inf[gf];
  const double radial_falloff_power = evolgf_radial_falloff_power[gf];
  double r = 1e100, partial_i_f = 1e100;
  nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, 0, 0, i0, i1, i2, &r, &partial_i_f);
  const double invr = 1. / r;
  const double X = partial_i_f + invr * (fa(i0, i1, i2) - var_at_infinity);
  const double source_rhs = -char_speed * X;
  double out = source_rhs;
  if (radial_falloff_power > 0) {
    double r_offset = r_in, X_offset = X_in;
    if (!have_in) {
      const int j0 = i0 + F0;
      double partial_i_f_offset = 1e100;
      r_offset = 1e100;
      nrpy_sommerfeld_r_dfdr(params, xx0, xx1, xx2, fa, F0, 0, 0, j0, i1, i2, &r_offset, &partial_i_f_offset);
      const double invr_offset = 1. / r_offset;
      X_offset = partial_i_f_offset + invr_offset * (fa(j0, i1, i2) - var_at_infinity);
    }
    const double extrap_rhs = char_speed * X_offset;
    const double diff_between_advection_and_f_rhs = rn + extrap_rhs;
    out = source_rhs + diff_between_advection_and_f_rhs * nrpy_som_falloff(r_offset * invr, radial_falloff_power);
  }
  r_in = r;
  X_in = X;
  return out;
}
// The same at outer point d, f read from global memory.
__device__ __forceinline__ double nrpy_sommerfeld_point(const paramstruct &params, const double *__restrict__ xx0,
                                                        const double *__restrict__ xx1,
                                                        const double *__restrict__ xx2, const int gf, const int d,
                                                        const int F0, const int F1, const int F2,
                                                        const double *__restrict__ f, const double *rhs) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const int i0 = d % N0, i1 = (d / N0) % N1, i2 = d / (N0 * N1);
  return nrpy_sommerfeld_rhs(params, xx0, xx1, xx2, gf, i0, i1, i2, F0, F1, F2,
                             [f, N0, N1](const int a, const int b, const int c) { return f[a + N0 * (b + N1 * c)]; },
                             [rhs](const size_t o) { return rhs[o]; });
}

// The i0-faces on grids whose ghost points are all outer points: there the group of layer
// gz is every (i0, i1, i2) with i0 = NGHOSTS - 1 - gz (FACE +1) or N0 - NGHOSTS + gz (FACE -1)
// and (i1, i2) in the box the earlier layers grew, [NGHOSTS - gz, N - NGHOSTS + gz). In a row
// whose (i1, i2) is interior, each of these points needs only the RHS of its inward
// neighbour in the same row (the interior point, or the layer before), and no other face
// group feeds it, while those that read it come later in the reference's order: so one
// launch before the layers takes every layer of the interior rows, each lane its row's
// points layer after layer (the edge rows stay in their layers' i0 slots).
// On an i0-face consecutive points lie in different rows, so a load of one value per lane
// touches as many cache lines as lanes. A block of 256 lanes takes a 32 x 8 tile of interior
// rows (i1, i2) and first copies what the stencils reach into LDS, rows of NRPY_SOM_XW
// points, x fastest: along i0 the one-sided and centred stencils of the points and of their
// inward neighbours stay in [0, NGHOSTS + FD] (mirrored on the high side); along i1 and i2
// a row's centred stencil stays within FD / 2 of it, and the one-sided one (the row next
// to the ghost zone, i = NGHOSTS) reaches FD points inward, inside the tile's own rows or
// its upper halo (the box ends at the grid's edge).
#define NRPY_SOM_TY 32
#define NRPY_SOM_TZ 8
#define NRPY_SOM_HALO (NRPY_SOMMERFELD_FD / 2)
#define NRPY_SOM_XW (NGHOSTS + NRPY_SOMMERFELD_FD + 1)
#define NRPY_SOM_BOXN (NRPY_SOM_XW * (NRPY_SOM_TY + 2 * NRPY_SOM_HALO) * (NRPY_SOM_TZ + 2 * NRPY_SOM_HALO))
static_assert(NRPY_SOM_HALO <= NGHOSTS, "the x-face box starts inside the grid");
struct nrpy_som_xtile {
  int F0, y0, z0, hi1, hi2, bx0, by0, by1, bz0, bz1;
};
__host__ __device__ static inline int nrpy_som_xface_ntiles(const int N1, const int N2) {
  const int n1 = N1 - 2 * NGHOSTS, n2 = N2 - 2 * NGHOSTS;
  return 2 * ((n1 + NRPY_SOM_TY - 1) / NRPY_SOM_TY) * ((n2 + NRPY_SOM_TZ - 1) / NRPY_SOM_TZ);
}
// tile t of nrpy_som_xface_ntiles(N1, N2): its rows [y0, min(y0 + TY, hi1)) x [z0, min(z0 +
// TZ, hi2)), its side (F0 +1: the low i0-faces) and the box [bx0, bx0 + XW) x [by0, by1) x
// [bz0, bz1) copied to LDS
__host__ __device__ static inline nrpy_som_xtile nrpy_som_xface_tile(const int N0, const int N1, const int N2,
                                                                     int t) {
  nrpy_som_xtile T;
  T.hi1 = N1 - NGHOSTS;
  T.hi2 = N2 - NGHOSTS;
  const int nty = (T.hi1 - NGHOSTS + NRPY_SOM_TY - 1) / NRPY_SOM_TY;
  const int side = t % 2;
  t /= 2;
  T.y0 = NGHOSTS + (t % nty) * NRPY_SOM_TY;
  T.z0 = NGHOSTS + (t / nty) * NRPY_SOM_TZ;
  T.F0 = side == 0 ? 1 : -1;
  T.bx0 = side == 0 ? 0 : N0 - NRPY_SOM_XW;
  T.by0 = T.y0 - NRPY_SOM_HALO;
  T.by1 = T.y0 + NRPY_SOM_TY + NRPY_SOM_HALO < N1 ? T.y0 + NRPY_SOM_TY + NRPY_SOM_HALO : N1;
  T.bz0 = T.z0 - NRPY_SOM_HALO;
  T.bz1 = T.z0 + NRPY_SOM_TZ + NRPY_SOM_HALO < N2 ? T.z0 + NRPY_SOM_TZ + NRPY_SOM_HALO : N2;
  return T;
}
// Block (tile blockIdx.x of the interior rows, i.e. of layer 0's group; gridfunction
// blockIdx.y) of 256 lanes: copies the box, then lane l takes row (y0 + l % 32, z0 + l / 32)
// if it is interior and computes its i0-face points from the innermost layer out, the
// inward neighbour's RHS the interior point's (read from rhs), then the one this lane
// computed last. FUSED: the RK4 update of substep S as nrpy_sommerfeld_outer_rk4_kernel does,
// with R as the RHS array; else the RHS goes to rhs. Every global load is issued before the
// box copy, so a lane waits for memory once.
template <int FUSED, int S>
__global__ void __launch_bounds__(NRPY_SOM_TY * NRPY_SOM_TZ) nrpy_sommerfeld_xface_kernel(const paramstruct params,
                                                                   const double *__restrict__ xx0,
                                                                   const double *__restrict__ xx1,
                                                                   const double *__restrict__ xx2,
                                                                   const double *__restrict__ gfs, double *rhs_gfs,
                                                                   double *y_n, double *rt, double *out,
                                                                   const double dt) {
  __shared__ double box[NRPY_SOM_BOXN];
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2;
  const nrpy_som_xtile T = nrpy_som_xface_tile(N0, N1, N2, (int)blockIdx.x);
  const int gf = (int)blockIdx.y;
  const double *f = gfs + (size_t)gf * Ntot;
  const int BY = T.by1 - T.by0, BZ = T.bz1 - T.bz0, nbox = NRPY_SOM_XW * BY * BZ;
  const int i1 = T.y0 + (int)threadIdx.x % NRPY_SOM_TY, i2 = T.z0 + (int)threadIdx.x / NRPY_SOM_TY;
  const bool live = i1 < T.hi1 && i2 < T.hi2;
  // a lane past the grid's edge loads at the tile's first row (inside the grid) and stores nothing
  const size_t row = (size_t)N0 * ((size_t)(live ? i1 : T.y0) + (size_t)N1 * (size_t)(live ? i2 : T.z0));
  double *rhs = rhs_gfs + (size_t)gf * Ntot;
  size_t dl[NGHOSTS];
  double yv[NGHOSTS], rv[NGHOSTS];
#pragma unroll
  for (int gz = 0; gz < NGHOSTS; gz++) {
    dl[gz] = row + (size_t)(T.F0 > 0 ? NGHOSTS - 1 - gz : N0 - NGHOSTS + gz);
    yv[gz] = FUSED && S < 3 ? y_n[(size_t)gf * Ntot + dl[gz]] : 0.0;
    rv[gz] = FUSED && S > 0 ? (S < 3 ? rt[(size_t)gf * Ntot + dl[gz]]
                                     : y_n[(size_t)gf * Ntot + dl[gz]] + rt[(size_t)gf * Ntot + dl[gz]])
                            : 0.0;
  }
  // the interior RHS next to the face: FUSED, from the compact array the shell kernel fills after
  // the NUM_EVOL_GFS grids of R ([gf][i2][i1][side]); else from the RHS grid
  const size_t xrow = (size_t)(live ? i1 : T.y0) + (size_t)N1 * (size_t)(live ? i2 : T.z0);
  double prev = FUSED ? rhs_gfs[(size_t)NUM_EVOL_GFS * Ntot + 2 * ((size_t)gf * N1 * N2 + xrow) + (T.F0 > 0 ? 0 : 1)]
                      : rhs[row + (size_t)(T.F0 > 0 ? NGHOSTS : N0 - 1 - NGHOSTS)];
  for (int e = (int)threadIdx.x; e < nbox; e += (int)blockDim.x) {
    const int x = e % NRPY_SOM_XW, y = (e / NRPY_SOM_XW) % BY, z = e / (NRPY_SOM_XW * BY);
    box[e] = f[(T.bx0 + x) + N0 * ((T.by0 + y) + N1 * (T.bz0 + z))];
  }
  __syncthreads();
  if (!live) return;
  const auto fa = [&](const int a, const int b, const int c) {
    return box[(a - T.bx0) + NRPY_SOM_XW * ((b - T.by0) + BY * (c - T.bz0))];
  };
  // r and d f/d r + (f - f_inf)/r of the point this lane computed last (its next inward neighbour)
  double r_in = 0.0, X_in = 0.0;
#pragma unroll
  for (int gz = 0; gz < NGHOSTS; gz++) {
    const int i0 = T.F0 > 0 ? NGHOSTS - 1 - gz : N0 - NGHOSTS + gz;
    const double ki = nrpy_sommerfeld_rhs_row(params, xx0, xx1, xx2, gf, i0, i1, i2, T.F0, fa, prev, gz > 0, r_in, X_in);
    prev = ki;
    rhs[dl[gz]] = ki;
    if (FUSED) {
      const size_t i = (size_t)gf * Ntot + dl[gz];
      if (S == 0) {
        rt[i] = ki * dt * (1.0 / 6.0);
        out[i] = yv[gz] + ki * dt * (1.0 / 2.0);
      } else if (S == 1) {
        rt[i] = rv[gz] + ki * dt * (1.0 / 3.0);
        out[i] = yv[gz] + ki * dt * (1.0 / 2.0);
      } else if (S == 2) {
        rt[i] = rv[gz] + ki * dt * (1.0 / 3.0);
        out[i] = yv[gz] + ki * dt;
      } else {
        out[i] = rv[gz] + ki * dt * (1.0 / 6.0);
      }
    }
  }
}
static void nrpy_sommerfeld_xface_launch(const int fused, const int S, const paramstruct *params, double *xx[3],
                                         const int num_gfs, double *gfs, double *rhs, double *y_n, double *rt,
                                         double *out, const double dt, hipStream_t stream) {
  const dim3 grid((unsigned)nrpy_som_xface_ntiles(params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2),
                  (unsigned)num_gfs);
  const dim3 block(NRPY_SOM_TY * NRPY_SOM_TZ);
  if (!fused)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<0, 0>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 0)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 0>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 1)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 1>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else if (S == 2)
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 2>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
  else
    hipLaunchKernelGGL((nrpy_sommerfeld_xface_kernel<1, 3>), grid, block, 0, stream, *params, xx[0], xx[1], xx[2],
                       gfs, rhs, y_n, rt, out, dt);
}

// One face group of one ghost layer: lane p of block row blockIdx.y handles outer point p of
// gridfunction blockIdx.y (no integer division per lane).
__global__ void nrpy_sommerfeld_outer_kernel(const paramstruct params, const double *__restrict__ xx0,
                                             const double *__restrict__ xx1, const double *__restrict__ xx2, int n,
                                             const int *__restrict__ dest, const int8_t *__restrict__ face, int num_gfs,
                                             const double *__restrict__ gfs, double *__restrict__ rhs_gfs) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= n || gf >= num_gfs) return;
  const size_t Ntot = (size_t)params.Nxx_plus_2NGHOSTS0 * params.Nxx_plus_2NGHOSTS1 * params.Nxx_plus_2NGHOSTS2;
  const int d = dest[p];
  double *rhs = rhs_gfs + (size_t)gf * Ntot;
  rhs[d] = nrpy_sommerfeld_point(params, xx0, xx1, xx2, gf, d, face[3 * p], face[3 * p + 1], face[3 * p + 2],
                                 gfs + (size_t)gf * Ntot, rhs);
}

// The same, fused with the RK4 update at the outer point (the arithmetic of
// nrpy_rk4_update_all): the RHS at outer points goes to the scratch array R (where the
// interior kernel left it at the points next to the boundary), and the stage value of
// substep S to out (and the running total to rt).
template <int S>
__global__ void nrpy_sommerfeld_outer_rk4_kernel(const paramstruct params, const double *__restrict__ xx0,
                                                 const double *__restrict__ xx1, const double *__restrict__ xx2,
                                                 int n, const int *__restrict__ dest, const int8_t *__restrict__ face,
                                                 int num_gfs, const double *__restrict__ gfs, double *__restrict__ R,
                                                 double *y_n, double *rt, double *out, const double dt) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= n || gf >= num_gfs) return;
  const size_t Ntot = (size_t)params.Nxx_plus_2NGHOSTS0 * params.Nxx_plus_2NGHOSTS1 * params.Nxx_plus_2NGHOSTS2;
  const int d = dest[p];
  double *rhs = R + (size_t)gf * Ntot;
  const size_t i = (size_t)gf * Ntot + d;
  // the update's operands are loaded before the condition's arithmetic, not after its store
  const double yv = S < 3 ? y_n[i] : 0.0;
  const double rv = S == 0 ? 0.0 : S < 3 ? rt[i] : y_n[i] + rt[i];
  const double ki = nrpy_sommerfeld_point(params, xx0, xx1, xx2, gf, d, face[3 * p], face[3 * p + 1],
                                          face[3 * p + 2], gfs + (size_t)gf * Ntot, rhs);
  rhs[d] = ki;
  if (S == 0) {
    rt[i] = ki * dt * (1.0 / 6.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 1) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 2) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt;
  } else {
    out[i] = rv + ki * dt * (1.0 / 6.0);
  }
}

// Substep S of the fused Sommerfeld RK4 step at the outer points, layer by layer and face
// group by face group in the reference's order. gfs: the substep's input state; R: the
// RHS scratch, holding the interior RHS at the points next to the boundary. For grids
// without inner boundary points only (NRPY_ERR_PARAM otherwise).
extern "C" int apply_bcs_sommerfeld_rk4(const int S, const paramstruct *params, double *xx[3], const bc_struct *bc,
                                        const int NUM_GFS, double *gfs, double *R, double *y_n, double *rt,
                                        double *out, const double dt, hipStream_t stream) {
  if (!params || !bc || !xx || !xx[0] || !xx[1] || !xx[2] || !gfs || !R || !y_n || !rt || !out)
    return NRPY_ERR_NULL;
  if (S < 0 || S > 3 || NUM_GFS < 1 || NUM_GFS > NUM_EVOL_GFS) return NRPY_ERR_PARAM;
  if (bc->N[0] != params->Nxx_plus_2NGHOSTS0 || bc->N[1] != params->Nxx_plus_2NGHOSTS1 ||
      bc->N[2] != params->Nxx_plus_2NGHOSTS2)
    return NRPY_ERR_SHAPE;
  if (bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N || bc->N[2] < NRPY_SOMMERFELD_MIN_N)
    return NRPY_ERR_SHAPE;
  for (int gz = 0; gz < NGHOSTS; gz++)
    if (bc->num_ib_gz_pts[gz] > 0) return NRPY_ERR_PARAM;
  const int B = 256;
  nrpy_sommerfeld_xface_launch(1, S, params, xx, NUM_GFS, gfs, R, y_n, rt, out, dt, stream);
  for (int gz = 0; gz < NGHOSTS; gz++) {
    int start = 0;
    for (int dir = 0; dir < 3; dir++) {
      const int end = bc->ob_dir_end[gz][dir];
      // the i0-face group: its edge rows only (the interior rows were launched above)
      const int n = dir == 0 ? bc->ob_xedge_off[gz + 1] - bc->ob_xedge_off[gz] : end - start;
      if (n > 0) {
        const dim3 grid((unsigned)((n + B - 1) / B), (unsigned)NUM_GFS);
        const int *dst = dir == 0 ? bc->d_ob_xedge_dest + bc->ob_xedge_off[gz] : bc->d_ob_dest + bc->ob_off[gz] + start;
        const int8_t *fc = dir == 0 ? bc->d_ob_xedge_face + 3 * (size_t)bc->ob_xedge_off[gz]
                                    : bc->d_ob_face + 3 * (size_t)(bc->ob_off[gz] + start);
        switch (S) {
          case 0: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<0>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          case 1: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<1>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          case 2: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<2>, grid, dim3(B), 0, stream, *params, xx[0],
                                     xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
          default: hipLaunchKernelGGL(nrpy_sommerfeld_outer_rk4_kernel<3>, grid, dim3(B), 0, stream, *params, xx[0],
                                      xx[1], xx[2], n, dst, fc, NUM_GFS, gfs, R, y_n, rt, out, dt); break;
        }
      }
      start = end;
    }
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}

// Sommerfeld radiation condition on the RHS at every ghost point: outer points
// from the radiation condition, inner points by parity from their sources.
// xx: the three device coordinate arrays; gfs_parity: host array of NUM_GFS
// parity types; gfs: the state the RHS was evaluated from; rhs_gfs: its RHS,
// valid at interior points. NUM_GFS <= NUM_EVOL_GFS (per-gridfunction
// parameters are those of the EVOL gridfunctions).
extern "C" int apply_bcs_sommerfeld(const paramstruct *params, double *xx[3], const bc_struct *bc, const int NUM_GFS,
                                    const int8_t *gfs_parity, double *gfs, double *rhs_gfs, hipStream_t stream) {
  if (!xx || !xx[0] || !xx[1] || !xx[2] || !rhs_gfs) return NRPY_ERR_NULL;
  if (NUM_GFS > NUM_EVOL_GFS) return NRPY_ERR_PARAM;
  nrpy_gf_parity_args gfp;
  memset(&gfp, 0, sizeof(gfp));
  int rc = nrpy_bc_check(params, bc, NUM_GFS, gfs_parity, gfs, &gfp);
  if (rc) return rc;
  if (bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N || bc->N[2] < NRPY_SOMMERFELD_MIN_N)
    return NRPY_ERR_SHAPE;
  const size_t Ntot = (size_t)bc->N[0] * bc->N[1] * bc->N[2];
  const int B = 256;
  bool all_outer = true;   // every ghost point an outer point: the interior rows' i0-faces take the tiled kernel
  for (int gz = 0; gz < NGHOSTS; gz++) all_outer = all_outer && bc->num_ib_gz_pts[gz] == 0;
  if (all_outer)
    nrpy_sommerfeld_xface_launch(0, 0, params, xx, NUM_GFS, gfs, rhs_gfs, nullptr, nullptr, nullptr, 0.0, stream);
  for (int gz = 0; gz < NGHOSTS; gz++) {
    int start = 0;
    for (int dir = 0; dir < 3; dir++) {
      const int end = bc->ob_dir_end[gz][dir];
      const bool edge = dir == 0 && all_outer;   // the i0-face group's edge rows only
      const int n = edge ? bc->ob_xedge_off[gz + 1] - bc->ob_xedge_off[gz] : end - start;
      if (n > 0) {
        hipLaunchKernelGGL(nrpy_sommerfeld_outer_kernel, dim3((unsigned)((n + B - 1) / B), (unsigned)NUM_GFS), dim3(B),
                           0, stream,
                           *params, xx[0], xx[1], xx[2], n,
                           edge ? bc->d_ob_xedge_dest + bc->ob_xedge_off[gz] : bc->d_ob_dest + bc->ob_off[gz] + start,
                           edge ? bc->d_ob_xedge_face + 3 * (size_t)bc->ob_xedge_off[gz]
                                : bc->d_ob_face + 3 * (size_t)(bc->ob_off[gz] + start),
                           NUM_GFS, gfs, rhs_gfs);
      }
      start = end;
    }
    const int ni = bc->num_ib_gz_pts[gz];
    if (ni > 0) {
      const size_t work = (size_t)ni * NUM_GFS;
      hipLaunchKernelGGL(nrpy_bc_inner_kernel, dim3((unsigned)((work + B - 1) / B)), dim3(B), 0, stream, ni,
                         bc->d_ib_dest + bc->ib_off[gz], bc->d_ib_src + bc->ib_off[gz],
                         bc->d_ib_parity + 10 * (size_t)bc->ib_off[gz], NUM_GFS, gfp, Ntot, rhs_gfs);
    }
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
// r and the radial derivative's geometry at a point: geo = r, then a_i and b of
// d f/d r = sum_i fdD_i a_i / b.
static __device__ void nrpy_sommerfeld_geometry(const paramstruct &params, const double xx0, const double xx1, const double xx2, double *geo) {
  const double AMPLRHO = params.AMPLRHO;
  const double AMPLZ = params.AMPLZ;
  const double SINHWRHO = params.SINHWRHO;
  const double SINHWZ = params.SINHWZ;
  (void)xx0; (void)xx1; (void)xx2;
  double J00, J01, J02, J10, J11, J12, J20, J21, J22;
  const double tmp_0 = (1.0/((SINHWRHO)));
  const double tmp_1 = tmp_0*xx0;
  const double tmp_2 = exp(tmp_1);
  const double tmp_3 = exp(-tmp_1);
  const double tmp_4 = tmp_2 - tmp_3;
  const double tmp_5 = ((AMPLRHO)*(AMPLRHO))/((exp(tmp_0) - exp(-tmp_0))*(exp(tmp_0) - exp(-tmp_0)));
  const double tmp_6 = (1.0/((SINHWZ)));
  const double tmp_7 = tmp_6*xx2;
  const double tmp_8 = exp(tmp_7);
  const double tmp_9 = exp(-tmp_7);
  const double tmp_10 = tmp_8 - tmp_9;
  const double tmp_11 = ((tmp_10)*(tmp_10));
  const double tmp_12 = exp(tmp_6) - exp(-tmp_6);
  const double tmp_13 = ((AMPLZ)*(AMPLZ))/((tmp_12)*(tmp_12));
  const double tmp_14 = tmp_11*tmp_13;
  const double tmp_15 = tmp_14 + ((tmp_4)*(tmp_4))*tmp_5;
  const double tmp_16 = sqrt(tmp_15);
  const double tmp_17 = (1.0/((tmp_16)));
  const double tmp_18 = ((1.0/2.0))*tmp_17;
  const double tmp_19 = 2*tmp_0;
  const double tmp_20 = tmp_4*tmp_5*(tmp_19*tmp_2 + tmp_19*tmp_3);
  const double tmp_21 = tmp_6*tmp_8;
  const double tmp_22 = tmp_6*tmp_9;
  const double tmp_23 = 2*tmp_21 + 2*tmp_22;
  const double tmp_24 = (1.0/sqrt(-tmp_14/tmp_15 + 1));
  const double tmp_25 = (1.0/((tmp_12)));
  const double tmp_26 = ((1.0/2.0))/pow(tmp_15, (3.0/2.0));
  geo[0] = tmp_16;
  J00 = tmp_18*tmp_20;
  J01 = 0;
  J02 = tmp_10*tmp_13*tmp_18*tmp_23;
  J10 = AMPLZ*tmp_10*tmp_20*tmp_24*tmp_25*tmp_26;
  J11 = 0;
  J12 = -tmp_24*(-((AMPLZ)*(AMPLZ)*(AMPLZ))*tmp_11*tmp_23*tmp_26/((tmp_12)*(tmp_12)*(tmp_12)) + AMPLZ*tmp_17*tmp_25*(tmp_21 + tmp_22));
  J20 = 0;
  J21 = 1;
  J22 = 0;
  const double cof0 = J11*J22 - J12*J21, cof1 = -(J10*J22 - J12*J20), cof2 = J10*J21 - J11*J20;
  geo[1] = cof0; geo[2] = cof1; geo[3] = cof2;
  geo[4] = J00*cof0 + J01*cof1 + J02*cof2;
}
template <typename FA>
static __device__ double nrpy_sommerfeld_dfdr_from(const paramstruct &params, const double *geo, FA fa, const int F0, const int F1, const int F2, const int i0, const int i1, const int i2) {
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  double fdD0 = 1e100, fdD1 = 1e100, fdD2 = 1e100;
  const double u0 = -25./12., u1 = 4., u2 = -3., u3 = 4./3., u4 = -1./4.;
  const double c1 = 2./3., c2 = 1./12.;
  {
    const bool one_sided = abs(F0) == 1 || i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0 || i0 - NGHOSTS <= 0;
    int S = F0;
    if (i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0) S = -1;
    if (i0 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic0 = min(max(i0, 2), Nxx_plus_2NGHOSTS0 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0+1*S,i1,i2) + u2*fa(i0+2*S,i1,i2) + u3*fa(i0+3*S,i1,i2) + u4*fa(i0+4*S,i1,i2))*invdx0;
    const double cen = (-c2*fa(nrpy_ic0+2,i1,i2) + c1*fa(nrpy_ic0+1,i1,i2) - c1*fa(nrpy_ic0+-1,i1,i2) + c2*fa(nrpy_ic0+-2,i1,i2))*invdx0;
    fdD0 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F1) == 1 || i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1 || i1 - NGHOSTS <= 0;
    int S = F1;
    if (i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1) S = -1;
    if (i1 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic1 = min(max(i1, 2), Nxx_plus_2NGHOSTS1 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0,i1+1*S,i2) + u2*fa(i0,i1+2*S,i2) + u3*fa(i0,i1+3*S,i2) + u4*fa(i0,i1+4*S,i2))*invdx1;
    const double cen = (-c2*fa(i0,nrpy_ic1+2,i2) + c1*fa(i0,nrpy_ic1+1,i2) - c1*fa(i0,nrpy_ic1+-1,i2) + c2*fa(i0,nrpy_ic1+-2,i2))*invdx1;
    fdD1 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F2) == 1 || i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2 || i2 - NGHOSTS <= 0;
    int S = F2;
    if (i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2) S = -1;
    if (i2 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic2 = min(max(i2, 2), Nxx_plus_2NGHOSTS2 - 1 - 2);
    const double one = S*(u0*fa(i0,i1,i2) + u1*fa(i0,i1,i2+1*S) + u2*fa(i0,i1,i2+2*S) + u3*fa(i0,i1,i2+3*S) + u4*fa(i0,i1,i2+4*S))*invdx2;
    const double cen = (-c2*fa(i0,i1,nrpy_ic2+2) + c1*fa(i0,i1,nrpy_ic2+1) - c1*fa(i0,i1,nrpy_ic2+-1) + c2*fa(i0,i1,nrpy_ic2+-2))*invdx2;
    fdD2 = one_sided ? one : cen;
  }
  const double cof0 = geo[1], cof1 = geo[2], cof2 = geo[3];
  return (fdD0*cof0 + fdD1*cof1 + fdD2*cof2)/geo[4];
}

// The whole condition in two launches per substep, for grids with inner boundary points. The
// reference's order (layer by layer, face group by face group, then the parity copies) makes a
// chain of each outer point: its RHS is
//   rhs_p = A_p + (rhs_q + B_p) (r_q / r_p)^n,   q its inward neighbour (an interior point, or an
// outer point one step further in), A_p = -v X_p, B_p = v X_q, X = d f/d r + (f - f_inf)/r with
// the stencils of p's FACE. A and B need only the state the substep starts from, so they are
// evaluated for every outer point at once, in extra blocks of the interior RHS launch
// (nrpy_sommerfeld_eval); the second launch (nrpy_sommerfeld_chain_kernel) walks each ghost
// point's chain from the interior out, at most 3 NGHOSTS multiply-adds, an inner point that of
// the point it copies, and does the RK4 update there. Every point's FACE follows from its
// indices: the axis with the largest distance outside the interior, the last of equals
// (nrpy_sommerfeld_chainable: known from building the lists). The operations are those of
// nrpy_sommerfeld_rhs; the results agree to rounding.
// Both launches are bound by latency. On the Maxwell 50x4x100 grid (MI355X) the condition's 9
// launches of 4-7 us with gaps of 2.4 us took 70 us a substep; one launch that evaluated the
// chains point after point 48 us, 25 us with r, the cofactors and the determinant from a table
// (geo, 5 values per point) instead of the Jacobian. MoL_graph_launch fills the table before its
// replays, on their stream, so that the coordinates are read when and where the step reads its
// other arrays (one launch of about 5 us per call, not per step).
// Scratch of a captured step: R, NUM_EVOL_GFS gridfunctions: the RHS at the interior points a
// chain or copy ends at (rhs_eval_rk4_substep_rim), A at the outer points; then B, as many; then geo.
#define NRPY_SOM_NSCRATCH (2 * NUM_EVOL_GFS + 5)

// Step k of n (k = 0 the innermost) of the chain with layers l: its axis.
__device__ __forceinline__ int nrpy_som_chain_axis(const int l0, const int l1, const int l2, const int k) {
  int m0 = l0, m1 = l1, m2 = l2, a = 0;
  for (int j = l0 + l1 + l2 - 1; j >= k; j--) {
    const int far = max(m0, max(m1, m2));
    a = m2 == far ? 2 : m1 == far ? 1 : 0;
    m0 -= a == 0;
    m1 -= a == 1;
    m2 -= a == 2;
  }
  return a;
}

// A and B at outer point number t % n of the lists (all layers) of gridfunction t / n.
__device__ __forceinline__ void nrpy_sommerfeld_eval(const paramstruct &params, const size_t t, const int n,
                                                     const int *__restrict__ dest, const int8_t *__restrict__ face,
                                                     const double *__restrict__ gfs, double *__restrict__ R) {
  if (t >= (size_t)n * NUM_EVOL_GFS) return;
  const int gf = (int)(t / n), p = (int)(t % n);
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1;
  const size_t Ntot = (size_t)N0 * N1 * params.Nxx_plus_2NGHOSTS2;
  const double *__restrict__ geo = R + (size_t)(2 * NUM_EVOL_GFS) * Ntot;
  const double *__restrict__ f = gfs + (size_t)gf * Ntot;
  const int d = dest[p], F0 = face[3 * p], F1 = face[3 * p + 1], F2 = face[3 * p + 2];
  const int i0 = d % N0, i1 = (d / N0) % N1, i2 = d / (N0 * N1);
  const auto fa = [f, N0, N1](const int a, const int b, const int c) { return f[a + N0 * (b + N1 * c)]; };
  const double char_speed = evolgf_speed[gf], var_at_infinity = evolgf_at_inf[gf];
  double X[2];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int j0 = i0 + q * F0, j1 = i1 + q * F1, j2 = i2 + q * F2;
    const size_t at = (size_t)j0 + N0 * ((size_t)j1 + N1 * (size_t)j2);
    const double g[5] = {geo[at], geo[Ntot + at], geo[2 * Ntot + at], geo[3 * Ntot + at], geo[4 * Ntot + at]};
    const double invr = 1. / g[0];
    X[q] = nrpy_sommerfeld_dfdr_from(params, g, fa, F0, F1, F2, j0, j1, j2) + invr * (fa(j0, j1, j2) - var_at_infinity);
  }
  R[(size_t)gf * Ntot + d] = -char_speed * X[0];
  R[(size_t)(NUM_EVOL_GFS + gf) * Ntot + d] = char_speed * X[1];
}

// The chain of at most MAX steps: every operand is loaded before the first multiply-add.
template <int MAX>
__device__ __forceinline__ double nrpy_som_walk(const nrpy_fill_row row, const int *l, const int *F, const int n,
                                                const int N0, const int N1, const size_t Ntot, const int gf,
                                                const double *__restrict__ R) {
  const double *__restrict__ A = R + (size_t)gf * Ntot;
  const double *__restrict__ B = A + (size_t)NUM_EVOL_GFS * Ntot;
  const double *__restrict__ r = R + (size_t)(2 * NUM_EVOL_GFS) * Ntot;
  const double power = evolgf_radial_falloff_power[gf];
  double a[MAX], b[MAX], rp[MAX + 1];
  double ki = A[row.base];
  rp[0] = r[row.base];
  int at = row.base;
#pragma unroll
  for (int k = 0; k < MAX; k++) {
    if (k < n) {
      const int ax = nrpy_som_chain_axis(l[0], l[1], l[2], k);
      at -= ax == 0 ? F[0] : ax == 1 ? F[1] * N0 : F[2] * N0 * N1;
    }
    a[k] = A[at];
    b[k] = B[at];
    rp[k + 1] = r[at];
  }
#pragma unroll
  for (int k = 0; k < MAX; k++) {
    const double invr = 1. / rp[k + 1];
    const double next = power > 0 ? a[k] + (ki + b[k]) * nrpy_som_falloff(rp[k] * invr, power) : a[k];
    ki = k < n ? next : ki;
  }
  return ki;
}

template <int S>
__global__ void __launch_bounds__(256)
nrpy_sommerfeld_chain_kernel(const paramstruct params, const int nrows, const nrpy_fill_row *__restrict__ rows,
                             const nrpy_gf_parity_args gfp, const double *__restrict__ R, double *y_n, double *rt,
                             double *out, const double dt) {
  const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x), gf = (int)blockIdx.y;
  if (p >= nrows) return;
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2;
  const nrpy_fill_row row = rows[p];
  const size_t i = (size_t)gf * Ntot + row.dest;
  const double yv = S < 3 ? y_n[i] : 0.0;
  const double rv = S == 0 ? 0.0 : S < 3 ? rt[i] : y_n[i] + rt[i];
  int l[3], F[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int c = (row.code >> (3 * d)) & 7;
    l[d] = c > 3 ? c - 3 : c;
    F[d] = c > 3 ? -1 : 1;
  }
  const int n = l[0] + l[1] + l[2];
  double ki;
  if (n == 0)
    ki = R[(size_t)gf * Ntot + row.base];
  else if (n <= NGHOSTS)
    ki = nrpy_som_walk<NGHOSTS>(row, l, F, n, N0, N1, Ntot, gf, R);
  else
    ki = nrpy_som_walk<3 * NGHOSTS>(row, l, F, n, N0, N1, Ntot, gf, R);
  if (row.negmask & (1 << gfp.p[gf])) ki = -ki;
  if (S == 0) {
    rt[i] = ki * dt * (1.0 / 6.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 1) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt * (1.0 / 2.0);
  } else if (S == 2) {
    rt[i] = rv + ki * dt * (1.0 / 3.0);
    out[i] = yv + ki * dt;
  } else {
    out[i] = rv + ki * dt * (1.0 / 6.0);
  }
}

// The geometry table, at the ghost points and the interior points next to them.
__global__ void __launch_bounds__(256)
nrpy_sommerfeld_geometry_kernel(const paramstruct params, const double *__restrict__ xx0,
                                const double *__restrict__ xx1, const double *__restrict__ xx2,
                                double *__restrict__ geo) {
  const int N0 = params.Nxx_plus_2NGHOSTS0, N1 = params.Nxx_plus_2NGHOSTS1, N2 = params.Nxx_plus_2NGHOSTS2;
  const size_t Ntot = (size_t)N0 * N1 * N2, at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= Ntot) return;
  const int i0 = (int)(at % N0), i1 = (int)((at / N0) % N1), i2 = (int)(at / ((size_t)N0 * N1));
  if (i0 > NGHOSTS && i0 < N0 - 1 - NGHOSTS && i1 > NGHOSTS && i1 < N1 - 1 - NGHOSTS && i2 > NGHOSTS &&
      i2 < N2 - 1 - NGHOSTS)
    return;
  double g[5];
  nrpy_sommerfeld_geometry(params, xx0[i0], xx1[i1], xx2[i2], g);
#pragma unroll
  for (int k = 0; k < 5; k++) geo[k * Ntot + at] = g[k];
}

// Whether the two launches cover the grid's ghost points: each is an outer point or a copy of
// an outer or interior point (no generic row), each outer point's FACE is the one its indices
// give, and every interior point a chain or copy ends at lies within NGHOSTS of an edge. All of it
// is known from building the maps: going over the rows here took 2 ms of each graph creation
// at 200x16x400.
static bool nrpy_sommerfeld_chainable(const bc_struct *bc) {
  return bc->fill_all.n > 0 && bc->fill_all.near_edges && bc->face_by_distance;
}

// The geometry table in the scratch of a captured step.
static int nrpy_sommerfeld_geometry_fill(const paramstruct *params, const double *const xx[3], double *scratch,
                                         hipStream_t stream) {
  const size_t Ntot =
      (size_t)params->Nxx_plus_2NGHOSTS0 * params->Nxx_plus_2NGHOSTS1 * params->Nxx_plus_2NGHOSTS2;
  hipLaunchKernelGGL(nrpy_sommerfeld_geometry_kernel, dim3((unsigned)((Ntot + 255) / 256)), dim3(256), 0, stream, *params,
                     xx[0], xx[1], xx[2], scratch + 2 * NUM_EVOL_GFS * Ntot);
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}

// Device memory of a captured step on the grid, nothing in it yet. nullptr where the two launches do
// not cover the grid, or without memory: the caller takes the unfused step.
static double *nrpy_sommerfeld_chain_scratch(const paramstruct *params, double *xx[3], const bc_struct *bc) {
  if (!params || !bc || !xx || !xx[0] || !xx[1] || !xx[2] || nrpy_check_params(params)) return nullptr;
  if (bc->N[0] != params->Nxx_plus_2NGHOSTS0 || bc->N[1] != params->Nxx_plus_2NGHOSTS1 ||
      bc->N[2] != params->Nxx_plus_2NGHOSTS2 || bc->N[0] < NRPY_SOMMERFELD_MIN_N || bc->N[1] < NRPY_SOMMERFELD_MIN_N ||
      bc->N[2] < NRPY_SOMMERFELD_MIN_N || !nrpy_sommerfeld_chainable(bc))
    return nullptr;
  const size_t Ntot = (size_t)bc->N[0] * bc->N[1] * bc->N[2];
  double *p = nullptr;
  if (hipMalloc((void **)&p, sizeof(double) * NRPY_SOM_NSCRATCH * Ntot) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

static int nrpy_sommerfeld_chain(const int S, const paramstruct *params, const bc_struct *bc, const int8_t *gfs_parity,
                                 double *R, double *y_n, double *rt, double *out, const double dt, hipStream_t stream) {
  nrpy_gf_parity_args gfp;
  memset(&gfp, 0, sizeof(gfp));
  const int rc = nrpy_bc_check(params, bc, NUM_EVOL_GFS, gfs_parity, R, &gfp);
  if (rc) return rc;
  const nrpy_fill_list &L = bc->fill_all;
  const int B = 64;
  const dim3 grid((unsigned)((L.n + B - 1) / B), NUM_EVOL_GFS);
  switch (S) {
    case 0: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<0>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    case 1: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<1>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    case 2: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<2>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp, R,
                               y_n, rt, out, dt); break;
    default: hipLaunchKernelGGL(nrpy_sommerfeld_chain_kernel<3>, grid, dim3(B), 0, stream, *params, L.n, L.d_rows, gfp,
                                R, y_n, rt, out, dt); break;
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
template <int S>
__global__ void __launch_bounds__(256) rhs_eval_rk4_substep_rim__gpu(const paramstruct params, const rfm_struct rfmstruct, const double *__restrict__ auxevol_gfs, const double *__restrict__ in_gfs, double *rk_yn, double *rk_rt, double *rk_out, const double dt, double *rim_rhs, const int rim_blocks, const int rim_n, const int *__restrict__ rim_dest, const int8_t *__restrict__ rim_face) {
  if ((int)blockIdx.x >= rim_blocks) {
    const int nrpy_t = (int)threadIdx.x + (int)blockDim.x * ((int)threadIdx.y + (int)blockDim.y * (int)threadIdx.z);
    nrpy_sommerfeld_eval(params, (size_t)((int)blockIdx.x - rim_blocks) * (blockDim.x * blockDim.y * blockDim.z) + nrpy_t, rim_n, rim_dest, rim_face, in_gfs, rim_rhs);
    return;
  }
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  NRPY_BLOCK_COORDS_OF(rim_blocks, Nxx0, Nxx1, Nxx2);
  const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
  const double f0_of_xx0 = rfmstruct.f0_of_xx0[i0];
  const double f0_of_xx0__D0 = rfmstruct.f0_of_xx0__D0[i0];
  const double f0_of_xx0__DD00 = rfmstruct.f0_of_xx0__DD00[i0];
  const double f0_of_xx0__DDD000 = rfmstruct.f0_of_xx0__DDD000[i0];
  const double f4_of_xx2 = rfmstruct.f4_of_xx2[i2];
  const double f4_of_xx2__D2 = rfmstruct.f4_of_xx2__D2[i2];
  const double f4_of_xx2__DD22 = rfmstruct.f4_of_xx2__DD22[i2];
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double eU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double eU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double eU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double aU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double aU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double aU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double aU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double aU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double aU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double aU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double aU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double aU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double aU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double aU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double aU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double aU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double aU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double aU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double aU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double aU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double aU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double aU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double aU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double aU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double aU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double aU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double aU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double aU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double aU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double aU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double aU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double aU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double aU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double aU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double aU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double aU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double aU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double aU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double aU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double aU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double aU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double aU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    const double psi_i0_i1_i2m2 = in_gfs[IDX4(PSIGF, i0,i1,i2-2)];
    const double psi_i0_i1_i2m1 = in_gfs[IDX4(PSIGF, i0,i1,i2-1)];
    const double psi_i0_i1m2_i2 = in_gfs[IDX4(PSIGF, i0,i1-2,i2)];
    const double psi_i0_i1m1_i2 = in_gfs[IDX4(PSIGF, i0,i1-1,i2)];
    const double psi_i0m2_i1_i2 = in_gfs[IDX4(PSIGF, i0-2,i1,i2)];
    const double psi_i0m1_i1_i2 = in_gfs[IDX4(PSIGF, i0-1,i1,i2)];
    const double psi = in_gfs[IDX4(PSIGF, i0,i1,i2)];
    const double psi_i0p1_i1_i2 = in_gfs[IDX4(PSIGF, i0+1,i1,i2)];
    const double psi_i0p2_i1_i2 = in_gfs[IDX4(PSIGF, i0+2,i1,i2)];
    const double psi_i0_i1p1_i2 = in_gfs[IDX4(PSIGF, i0,i1+1,i2)];
    const double psi_i0_i1p2_i2 = in_gfs[IDX4(PSIGF, i0,i1+2,i2)];
    const double psi_i0_i1_i2p1 = in_gfs[IDX4(PSIGF, i0,i1,i2+1)];
    const double psi_i0_i1_i2p2 = in_gfs[IDX4(PSIGF, i0,i1,i2+2)];
    const double Gamma_i0_i1_i2m2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-2)];
    const double Gamma_i0_i1_i2m1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-1)];
    const double Gamma_i0_i1m2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-2,i2)];
    const double Gamma_i0_i1m1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-1,i2)];
    const double Gamma_i0m2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-2,i1,i2)];
    const double Gamma_i0m1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-1,i1,i2)];
    const double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    const double Gamma_i0p1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+1,i1,i2)];
    const double Gamma_i0p2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+2,i1,i2)];
    const double Gamma_i0_i1p1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+1,i2)];
    const double Gamma_i0_i1p2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+2,i2)];
    const double Gamma_i0_i1_i2p1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+1)];
    const double Gamma_i0_i1_i2p2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+2)];
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_4_3 = 4.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double FDPart1_Rational_m5_2 = -5.0/2.0;
    const double FDPart1_0 = FDPart1_Rational_m1_12*aU0_i0p2_i1_i2;
    const double FDPart1_1 = FDPart1_Rational_m1_12*aU0_i0_i1p2_i2;
    const double FDPart1_2 = FDPart1_Rational_m1_12*aU0_i0_i1_i2p2;
    const double FDPart1_3 = FDPart1_Rational_m1_12*aU1_i0p2_i1_i2;
    const double FDPart1_4 = FDPart1_Rational_m1_12*aU1_i0_i1p2_i2;
    const double FDPart1_5 = FDPart1_Rational_m1_12*aU1_i0_i1_i2p2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*aU2_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*aU2_i0_i1_i2p2;
    const double FDPart1_8 = ((invdx0)*(invdx0));
    const double FDPart1_9 = FDPart1_Rational_m5_2*aU0;
    const double FDPart1_10 = ((invdx1)*(invdx1));
    const double FDPart1_11 = ((invdx2)*(invdx2));
    const double FDPart1_12 = FDPart1_Rational_m5_2*aU1;
    const double FDPart1_13 = FDPart1_Rational_m5_2*aU2;
    const double FDPart1_14 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_15 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_16 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_17 = FDPart1_Rational_m5_2*psi;
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double aU_dD00 = invdx0*(FDPart1_0 + FDPart1_Rational_1_12*aU0_i0m2_i1_i2 + FDPart1_Rational_2_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU0_i0m1_i1_i2);
    const double aU_dD01 = invdx1*(FDPart1_1 + FDPart1_Rational_1_12*aU0_i0_i1m2_i2 + FDPart1_Rational_2_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU0_i0_i1m1_i2);
    const double aU_dD02 = invdx2*(FDPart1_2 + FDPart1_Rational_1_12*aU0_i0_i1_i2m2 + FDPart1_Rational_2_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU0_i0_i1_i2m1);
    const double aU_dD10 = invdx0*(FDPart1_3 + FDPart1_Rational_1_12*aU1_i0m2_i1_i2 + FDPart1_Rational_2_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU1_i0m1_i1_i2);
    const double aU_dD11 = invdx1*(FDPart1_4 + FDPart1_Rational_1_12*aU1_i0_i1m2_i2 + FDPart1_Rational_2_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m2_3*aU1_i0_i1m1_i2);
    const double aU_dD12 = invdx2*(FDPart1_5 + FDPart1_Rational_1_12*aU1_i0_i1_i2m2 + FDPart1_Rational_2_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU1_i0_i1_i2m1);
    const double aU_dD20 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*aU2_i0m2_i1_i2 + FDPart1_Rational_2_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m2_3*aU2_i0m1_i1_i2);
    const double aU_dD22 = invdx2*(FDPart1_7 + FDPart1_Rational_1_12*aU2_i0_i1_i2m2 + FDPart1_Rational_2_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m2_3*aU2_i0_i1_i2m1);
    const double aU_dDD000 = FDPart1_8*(FDPart1_0 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0m1_i1_i2 + FDPart1_Rational_4_3*aU0_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU0_i0m2_i1_i2);
    const double aU_dDD011 = FDPart1_10*(FDPart1_1 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1m1_i2 + FDPart1_Rational_4_3*aU0_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU0_i0_i1m2_i2);
    const double aU_dDD022 = FDPart1_11*(FDPart1_2 + FDPart1_9 + FDPart1_Rational_4_3*aU0_i0_i1_i2m1 + FDPart1_Rational_4_3*aU0_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU0_i0_i1_i2m2);
    const double aU_dDD100 = FDPart1_8*(FDPart1_12 + FDPart1_3 + FDPart1_Rational_4_3*aU1_i0m1_i1_i2 + FDPart1_Rational_4_3*aU1_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU1_i0m2_i1_i2);
    const double aU_dDD111 = FDPart1_10*(FDPart1_12 + FDPart1_4 + FDPart1_Rational_4_3*aU1_i0_i1m1_i2 + FDPart1_Rational_4_3*aU1_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU1_i0_i1m2_i2);
    const double aU_dDD122 = FDPart1_11*(FDPart1_12 + FDPart1_5 + FDPart1_Rational_4_3*aU1_i0_i1_i2m1 + FDPart1_Rational_4_3*aU1_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU1_i0_i1_i2m2);
    const double aU_dDD200 = FDPart1_8*(FDPart1_13 + FDPart1_6 + FDPart1_Rational_4_3*aU2_i0m1_i1_i2 + FDPart1_Rational_4_3*aU2_i0p1_i1_i2 + FDPart1_Rational_m1_12*aU2_i0m2_i1_i2);
    const double aU_dDD211 = FDPart1_10*(FDPart1_13 + FDPart1_Rational_4_3*aU2_i0_i1m1_i2 + FDPart1_Rational_4_3*aU2_i0_i1p1_i2 + FDPart1_Rational_m1_12*aU2_i0_i1m2_i2 + FDPart1_Rational_m1_12*aU2_i0_i1p2_i2);
    const double aU_dDD222 = FDPart1_11*(FDPart1_13 + FDPart1_7 + FDPart1_Rational_4_3*aU2_i0_i1_i2m1 + FDPart1_Rational_4_3*aU2_i0_i1_i2p1 + FDPart1_Rational_m1_12*aU2_i0_i1_i2m2);
    const double psi_dD0 = invdx0*(FDPart1_14 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_15 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_16 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_8*(FDPart1_14 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_10*(FDPart1_15 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_11*(FDPart1_16 + FDPart1_17 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    const double FDPart3_0 = (1.0/((f0_of_xx0__D0)));
    const double FDPart3_1 = FDPart3_0*psi_dD0;
    const double FDPart3_2 = (1.0/((f0_of_xx0)));
    const double FDPart3_3 = (1.0/((f4_of_xx2)));
    const double FDPart3_4 = ((f0_of_xx0__D0)*(f0_of_xx0__D0));
    const double FDPart3_5 = (1.0/((FDPart3_4)));
    const double FDPart3_6 = (1.0/((f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_7 = FDPart3_3*f4_of_xx2__D2;
    const double FDPart3_8 = (1.0/((f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_9 = FDPart3_0*aU0;
    const double FDPart3_10 = (1.0/((f0_of_xx0__D0)*(f0_of_xx0__D0)*(f0_of_xx0__D0)));
    const double FDPart3_11 = aU0*f0_of_xx0__DD00;
    const double FDPart3_12 = FDPart3_0*(FDPart3_0*aU_dD00 - FDPart3_11*FDPart3_5);
    const double FDPart3_13 = ((f0_of_xx0__DD00)*(f0_of_xx0__DD00));
    const double FDPart3_14 = 2*FDPart3_2;
    const double FDPart3_15 = FDPart3_8*f0_of_xx0__D0;
    const double FDPart3_16 = -FDPart3_15*aU1 + FDPart3_2*aU_dD10;
    const double FDPart3_17 = FDPart3_0*FDPart3_16;
    const double FDPart3_18 = FDPart3_8*f0_of_xx0__DD00;
    const double FDPart3_19 = (1.0/((f0_of_xx0)*(f0_of_xx0)*(f0_of_xx0)));
    const double FDPart3_20 = FDPart3_0*FDPart3_3*aU_dD20;
    const double FDPart3_21 = FDPart3_6*f4_of_xx2__D2;
    const double FDPart3_22 = (1.0/((f4_of_xx2)*(f4_of_xx2)*(f4_of_xx2)));
    const double FDPart3_23 = ((f4_of_xx2__D2)*(f4_of_xx2__D2));
  const double __rhs_AU0 = -FDPart3_1 - eU0;
  const double __rhs_AU1 = -FDPart3_2*psi_dD1 - eU1;
  const double __rhs_AU2 = -FDPart3_3*psi_dD2 - eU2;
  const double __rhs_EU0 = f0_of_xx0__D0*(FDPart3_5*Gamma_dD0 - FDPart3_5*(FDPart3_0*aU_dDD000 + FDPart3_12*f0_of_xx0__DD00 - 2*FDPart3_5*aU_dD00*f0_of_xx0__DD00 + FDPart3_9*(FDPart3_0*f0_of_xx0__DDD000 - FDPart3_13*FDPart3_5) + aU0*(2*FDPart3_10*FDPart3_13 - FDPart3_5*f0_of_xx0__DDD000)) - FDPart3_6*(-FDPart3_0*FDPart3_7*aU_dD02 + FDPart3_0*aU_dDD022) - FDPart3_8*(-2*FDPart3_0*aU_dD11 + FDPart3_0*aU_dDD011 + FDPart3_10*FDPart3_11*f0_of_xx0 + FDPart3_12*f0_of_xx0 - FDPart3_9));
  const double __rhs_EU1 = f0_of_xx0*(-FDPart3_5*(FDPart3_14*FDPart3_16*f0_of_xx0__D0 - 2*FDPart3_15*aU_dD10 - FDPart3_17*f0_of_xx0__DD00 - FDPart3_18*aU1 + FDPart3_19*FDPart3_4*aU1 + FDPart3_2*aU1*(FDPart3_2*f0_of_xx0__DD00 - FDPart3_4*FDPart3_8) + FDPart3_2*aU_dDD100 + aU1*(-FDPart3_18 + 2*FDPart3_19*FDPart3_4)) - FDPart3_6*(-FDPart3_2*FDPart3_7*aU_dD12 + FDPart3_2*aU_dDD122) + FDPart3_8*Gamma_dD1 - FDPart3_8*(FDPart3_14*aU_dD01 + FDPart3_17*f0_of_xx0 + FDPart3_2*aU_dDD111));
  const double __rhs_EU2 = f4_of_xx2*(-FDPart3_5*(-FDPart3_20*f0_of_xx0__DD00 + FDPart3_3*aU_dDD200) + FDPart3_6*Gamma_dD2 - FDPart3_6*(-2*FDPart3_21*aU_dD22 + FDPart3_3*aU2*(-FDPart3_23*FDPart3_6 + FDPart3_3*f4_of_xx2__DD22) + FDPart3_3*aU_dDD222 + FDPart3_7*(-FDPart3_21*aU2 + FDPart3_3*aU_dD22) + aU2*(2*FDPart3_22*FDPart3_23 - FDPart3_6*f4_of_xx2__DD22)) - FDPart3_8*(FDPart3_20*f0_of_xx0 + FDPart3_3*aU_dDD211));
  const double __rhs_PSI = -Gamma;
  const double __rhs_GAMMA = -FDPart3_1*FDPart3_2 + FDPart3_10*f0_of_xx0__DD00*psi_dD0 + FDPart3_22*f4_of_xx2__D2*psi_dD2 - FDPart3_5*psi_dDD00 - FDPart3_6*psi_dDD22 - FDPart3_8*psi_dDD11;
  __builtin_amdgcn_sched_barrier(0);
  NRPY_RK4_PRELOAD(S, AU0GF, 0)
  NRPY_RK4_PRELOAD(S, AU1GF, 1)
  NRPY_RK4_PRELOAD(S, AU2GF, 2)
  NRPY_RK4_PRELOAD(S, EU0GF, 3)
  NRPY_RK4_PRELOAD(S, EU1GF, 4)
  NRPY_RK4_PRELOAD(S, EU2GF, 5)
  NRPY_RK4_PRELOAD(S, PSIGF, 6)
  NRPY_RK4_PRELOAD(S, GAMMAGF, 7)
  NRPY_RK4_STORE(S, 0, __rhs_AU0);
  NRPY_RK4_STORE(S, 1, __rhs_AU1);
  NRPY_RK4_STORE(S, 2, __rhs_AU2);
  NRPY_RK4_STORE(S, 3, __rhs_EU0);
  NRPY_RK4_STORE(S, 4, __rhs_EU1);
  NRPY_RK4_STORE(S, 5, __rhs_EU2);
  NRPY_RK4_STORE(S, 6, __rhs_PSI);
  NRPY_RK4_STORE(S, 7, __rhs_GAMMA);
  if (i0 < 2*NGHOSTS || i0 >= Nxx0 || i1 < 2*NGHOSTS || i1 >= Nxx1 || i2 < 2*NGHOSTS || i2 >= Nxx2) {
    rim_rhs[IDX4(AU0GF, i0, i1, i2)] = __rhs_AU0;
    rim_rhs[IDX4(AU1GF, i0, i1, i2)] = __rhs_AU1;
    rim_rhs[IDX4(AU2GF, i0, i1, i2)] = __rhs_AU2;
    rim_rhs[IDX4(EU0GF, i0, i1, i2)] = __rhs_EU0;
    rim_rhs[IDX4(EU1GF, i0, i1, i2)] = __rhs_EU1;
    rim_rhs[IDX4(EU2GF, i0, i1, i2)] = __rhs_EU2;
    rim_rhs[IDX4(PSIGF, i0, i1, i2)] = __rhs_PSI;
    rim_rhs[IDX4(GAMMAGF, i0, i1, i2)] = __rhs_GAMMA;
  }
  }
}
static int rhs_eval_rk4_substep_rim(const int S, const rfm_struct *rfmstruct, const paramstruct *params, const bc_struct *bc, const double *auxevol_gfs, const double *in_gfs, double *y_n, double *rt, double *out, double *rim_rhs, const double dt, hipStream_t stream) {
  if (!params || !bc || !y_n || !rt || !out || !rim_rhs) return NRPY_ERR_NULL;
  if (S < 0 || S > 3) return NRPY_ERR_PARAM;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(2, 64, 1, 4);
  const unsigned nb = nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2);
  const int n = bc->ob_off[NGHOSTS];
  const size_t threads = (size_t)block.x * block.y * block.z;
  const dim3 grid(nb + (unsigned)(((size_t)n * NUM_EVOL_GFS + threads - 1) / threads));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_rk4_substep_rim__gpu<0>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt, rim_rhs, (int)nb, n, bc->d_ob_dest, bc->d_ob_face); break;
    case 1: hipLaunchKernelGGL(rhs_eval_rk4_substep_rim__gpu<1>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt, rim_rhs, (int)nb, n, bc->d_ob_dest, bc->d_ob_face); break;
    case 2: hipLaunchKernelGGL(rhs_eval_rk4_substep_rim__gpu<2>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt, rim_rhs, (int)nb, n, bc->d_ob_dest, bc->d_ob_face); break;
    case 3: hipLaunchKernelGGL(rhs_eval_rk4_substep_rim__gpu<3>, grid, block, 0, stream, *params, *rfmstruct, auxevol_gfs, in_gfs, y_n, rt, out, dt, rim_rhs, (int)nb, n, bc->d_ob_dest, bc->d_ob_face); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}
extern "C" int MoL_step_forward_in_time_sommerfeld_unfused(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, hipStream_t stream) {
  if (!params || !y_n_gfs || !k_odd_gfs || !k_even_gfs || !y_nplus1_running_total_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const size_t Ntot = (size_t)params->Nxx_plus_2NGHOSTS0 * params->Nxx_plus_2NGHOSTS1 * params->Nxx_plus_2NGHOSTS2;
  int rc;
  /* substep 0: RHS(y_n_gfs) -> k_odd_gfs */
  if ((rc = rhs_eval(rfmstruct, params, y_n_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, y_n_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(0, (size_t)NUM_EVOL_GFS * Ntot, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 1: RHS(k_odd_gfs) -> k_even_gfs */
  if ((rc = rhs_eval(rfmstruct, params, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(1, (size_t)NUM_EVOL_GFS * Ntot, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 2: RHS(k_even_gfs) -> k_odd_gfs */
  if ((rc = rhs_eval(rfmstruct, params, k_even_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_even_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(2, (size_t)NUM_EVOL_GFS * Ntot, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 3: RHS(k_odd_gfs) -> k_even_gfs */
  if ((rc = rhs_eval(rfmstruct, params, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(3, (size_t)NUM_EVOL_GFS * Ntot, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  return NRPY_OK;
}
// One RK4 step of the Sommerfeld branch (see MoL_step_forward_in_time_sommerfeld_unfused for
// the reference's order of operations; the fused form gives the same values).
extern "C" int MoL_step_forward_in_time_sommerfeld(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, hipStream_t stream) {
  return MoL_step_forward_in_time_sommerfeld_unfused(params, rfmstruct, xx, bcstruct, y_n_gfs, k_odd_gfs, k_even_gfs, y_nplus1_running_total_gfs, dt, stream);
}
// The same step as two launches per substep (equal to the unfused step to rounding); R:
// the scratch of nrpy_sommerfeld_chain_scratch, not shared with a step on another stream.
static int nrpy_sommerfeld_chain_step(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, double *R, const double dt, hipStream_t stream) {
  int rc;
  if ((rc = rhs_eval_rk4_substep_rim(0, rfmstruct, params, bcstruct, nullptr, y_n_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, R, dt, stream))) return rc;
  if ((rc = nrpy_sommerfeld_chain(0, params, bcstruct, evol_gf_parity, R, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  if ((rc = rhs_eval_rk4_substep_rim(1, rfmstruct, params, bcstruct, nullptr, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, R, dt, stream))) return rc;
  if ((rc = nrpy_sommerfeld_chain(1, params, bcstruct, evol_gf_parity, R, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, dt, stream))) return rc;
  if ((rc = rhs_eval_rk4_substep_rim(2, rfmstruct, params, bcstruct, nullptr, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, R, dt, stream))) return rc;
  if ((rc = nrpy_sommerfeld_chain(2, params, bcstruct, evol_gf_parity, R, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  if ((rc = rhs_eval_rk4_substep_rim(3, rfmstruct, params, bcstruct, nullptr, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, R, dt, stream))) return rc;
  if ((rc = nrpy_sommerfeld_chain(3, params, bcstruct, evol_gf_parity, R, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, dt, stream))) return rc;
  return NRPY_OK;
}
// The Sommerfeld RK4 step captured into a hipGraph (every launch is a kernel; the pointers, those of
// xx among them, and dt are fixed at capture); replay with MoL_graph_launch, free with MoL_graph_free.
extern "C" int MoL_sommerfeld_graph_create(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, MoL_graph **out) {
  if (!out) return NRPY_ERR_NULL;
  *out = nullptr;
  hipStream_t s;
  if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return NRPY_ERR_LAUNCH;
  MoL_graph *g = new MoL_graph();
  int rc = NRPY_OK;
  // without scratch memory, or on a grid the chain kernel does not cover: the unfused step
  if (rfmstruct && y_n_gfs && k_odd_gfs && k_even_gfs && y_nplus1_running_total_gfs)
    g->scratch = nrpy_sommerfeld_chain_scratch(params, xx, bcstruct);
  if (g->scratch) {
    g->params = *params;
    for (int d = 0; d < 3; d++) g->xx[d] = xx[d];
  }
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) rc = NRPY_ERR_LAUNCH;
  if (!rc) {
    rc = g->scratch ? nrpy_sommerfeld_chain_step(params, rfmstruct, xx, bcstruct, y_n_gfs, k_odd_gfs,
                                                 k_even_gfs, y_nplus1_running_total_gfs, g->scratch, dt, s)
                    : MoL_step_forward_in_time_sommerfeld(params, rfmstruct, xx, bcstruct, y_n_gfs, k_odd_gfs,
                                                          k_even_gfs, y_nplus1_running_total_gfs, dt, s);
    hipGraph_t gr;
    const hipError_t e = hipStreamEndCapture(s, &gr);
    if (!rc && e != hipSuccess) rc = NRPY_ERR_LAUNCH;
    if (!rc) {
      g->graph = gr;
      if (hipGraphInstantiate(&g->exec, gr, nullptr, nullptr, 0) != hipSuccess) rc = NRPY_ERR_LAUNCH;
    }
  }
  (void)hipStreamDestroy(s);
  if (rc) { (void)hipFree(g->scratch); delete g; return rc; }
  *out = g;
  return NRPY_OK;
}
