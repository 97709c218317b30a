// Generated by nrpytutorial_amd.codegen; do not edit.
#include "../nrpy_runtime_pre.h"
#define NGHOSTS 3
/* Gridfunction indices: alphabetical within each group. */
#define NUM_EVOL_GFS 8
#define AU0GF	0
#define AU1GF	1
#define AU2GF	2
#define EU0GF	3
#define EU1GF	4
#define EU2GF	5
#define GAMMAGF	6
#define PSIGF	7
#define NUM_AUX_GFS 2
#define DIVEGF	0
#define GGF	1
#define NUM_AUXEVOL_GFS 0

typedef struct __paramstruct__ {
  int Nxx0;
  int Nxx1;
  int Nxx2;
  int Nxx_plus_2NGHOSTS0;
  int Nxx_plus_2NGHOSTS1;
  int Nxx_plus_2NGHOSTS2;
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

static const int8_t evol_gf_parity[8] = {1, 2, 3, 1, 2, 3, 0, 0};
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
  const double xx0 = xx[0][i0];
  const double xx1 = xx[1][i1];
  const double xx2 = xx[2][i2];
  xCart[0] = xx0;
  xCart[1] = xx1;
  xCart[2] = xx2;
}
static void EigenCoord_xx_to_Cart(const paramstruct *params, double *xx[3], const int i0, const int i1, const int i2, double xCart[3]) {
  const double xx0 = xx[0][i0];
  const double xx1 = xx[1][i1];
  const double xx2 = xx[2][i2];
  xCart[0] = xx0;
  xCart[1] = xx1;
  xCart[2] = xx2;
}
static void EigenCoord_Cart_to_xx(const paramstruct *params, const double xCart[3], double Cart_to_xx[3]) {
  const double Cartx = xCart[0];
  const double Carty = xCart[1];
  const double Cartz = xCart[2];
  Cart_to_xx[0] = Cartx;
  Cart_to_xx[1] = Carty;
  Cart_to_xx[2] = Cartz;
}
static void eval_parity_dot_products(const paramstruct *params, double parity[10], const double xx0, const double xx1, const double xx2, const double xx0_inbounds, const double xx1_inbounds, const double xx2_inbounds) {
  parity[0] = 1;
  parity[1] = 1;
  parity[2] = 1;
  parity[3] = 1;
  parity[4] = 1;
  parity[5] = 1;
  parity[6] = 1;
  parity[7] = 1;
  parity[8] = 1;
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
  const double xmax = params->xmax;
  const double xmin = params->xmin;
  const double ymax = params->ymax;
  const double ymin = params->ymin;
  const double zmax = params->zmax;
  const double zmin = params->zmin;
  double xxmin[3], xxmax[3];
  if (EigenCoord == 0) {
    xxmin[0] = xmin;
    xxmax[0] = xmax;
    xxmin[1] = ymin;
    xxmax[1] = ymax;
    xxmin[2] = zmin;
    xxmax[2] = zmax;
  }
  if (EigenCoord == 1) {
    xxmin[0] = xmin;
    xxmax[0] = xmax;
    xxmin[1] = ymin;
    xxmax[1] = ymax;
    xxmin[2] = zmin;
    xxmax[2] = zmax;
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
    ds_dirn0 = dxx0;
    ds_dirn1 = dxx1;
    ds_dirn2 = dxx2;
    dsmin = fmin(dsmin, fmin(ds_dirn0, fmin(ds_dirn1, ds_dirn2)));
  }
  return dsmin*CFL_FACTOR/params->wavespeed;
}

#include "../nrpy_runtime.h"
typedef struct __rfmstruct__ {
  const double *unused;
} rfm_struct;
extern "C" int rfm_struct_create(const paramstruct *params, double *xx[3], rfm_struct **out) {
  if (!params || !xx || !out) return NRPY_ERR_NULL;
  *out = nullptr;
  const int NN[3] = {params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2};
  (void)NN;
  double *tab[1] = {0};
  int rc = NRPY_OK;
  rfm_struct *r = new rfm_struct();
  memset(r, 0, sizeof(*r));
  *out = r;
  return rc;
}
extern "C" void rfm_struct_free(rfm_struct *rfmstruct) {
  if (!rfmstruct) return;
  delete rfmstruct;
}


/* Evaluate the vacuum Maxwell System II RHSs */
__global__ void __launch_bounds__(256) rhs_eval__gpu(const paramstruct params, const double *__restrict__ in_gfs, double *__restrict__ rhs_gfs) {
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
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double EU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double EU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double EU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double AU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double AU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double AU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double AU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double AU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double AU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double AU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double AU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double AU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double AU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double AU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double AU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double AU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double AU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double AU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double AU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double AU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double AU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double AU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double AU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double AU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double AU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double AU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double AU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double AU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double AU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double AU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
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
    const double FDPart1_0 = ((invdx0)*(invdx0));
    const double FDPart1_1 = AU0*FDPart1_Rational_m5_2;
    const double FDPart1_2 = ((invdx1)*(invdx1));
    const double FDPart1_3 = ((invdx2)*(invdx2));
    const double FDPart1_4 = AU1*FDPart1_Rational_m5_2;
    const double FDPart1_5 = AU2*FDPart1_Rational_m5_2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_8 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_9 = FDPart1_Rational_m5_2*psi;
    const double AU_dDD000 = FDPart1_0*(AU0_i0m1_i1_i2*FDPart1_Rational_4_3 + AU0_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_4_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD011 = FDPart1_2*(AU0_i0_i1m1_i2*FDPart1_Rational_4_3 + AU0_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU0_i0_i1p1_i2*FDPart1_Rational_4_3 + AU0_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD022 = FDPart1_3*(AU0_i0_i1_i2m1*FDPart1_Rational_4_3 + AU0_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU0_i0_i1_i2p1*FDPart1_Rational_4_3 + AU0_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD100 = FDPart1_0*(AU1_i0m1_i1_i2*FDPart1_Rational_4_3 + AU1_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU1_i0p1_i1_i2*FDPart1_Rational_4_3 + AU1_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD111 = FDPart1_2*(AU1_i0_i1m1_i2*FDPart1_Rational_4_3 + AU1_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_4_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD122 = FDPart1_3*(AU1_i0_i1_i2m1*FDPart1_Rational_4_3 + AU1_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU1_i0_i1_i2p1*FDPart1_Rational_4_3 + AU1_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD200 = FDPart1_0*(AU2_i0m1_i1_i2*FDPart1_Rational_4_3 + AU2_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU2_i0p1_i1_i2*FDPart1_Rational_4_3 + AU2_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD211 = FDPart1_2*(AU2_i0_i1m1_i2*FDPart1_Rational_4_3 + AU2_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU2_i0_i1p1_i2*FDPart1_Rational_4_3 + AU2_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD222 = FDPart1_3*(AU2_i0_i1_i2m1*FDPart1_Rational_4_3 + AU2_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_4_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double psi_dD0 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_7 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_8 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_0*(FDPart1_6 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_2*(FDPart1_7 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_3*(FDPart1_8 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    rhs_gfs[IDX4(AU0GF, i0, i1, i2)] = -EU0 - psi_dD0;
    rhs_gfs[IDX4(AU1GF, i0, i1, i2)] = -EU1 - psi_dD1;
    rhs_gfs[IDX4(AU2GF, i0, i1, i2)] = -EU2 - psi_dD2;
    rhs_gfs[IDX4(EU0GF, i0, i1, i2)] = -AU_dDD000 - AU_dDD011 - AU_dDD022 + Gamma_dD0;
    rhs_gfs[IDX4(EU1GF, i0, i1, i2)] = -AU_dDD100 - AU_dDD111 - AU_dDD122 + Gamma_dD1;
    rhs_gfs[IDX4(EU2GF, i0, i1, i2)] = -AU_dDD200 - AU_dDD211 - AU_dDD222 + Gamma_dD2;
    rhs_gfs[IDX4(GAMMAGF, i0, i1, i2)] = -psi_dDD00 - psi_dDD11 - psi_dDD22;
    rhs_gfs[IDX4(PSIGF, i0, i1, i2)] = -Gamma;
  }
  
}

extern "C" int rhs_eval(const paramstruct *params, const double *in_gfs, double *rhs_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs || !rhs_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(0, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  hipLaunchKernelGGL(rhs_eval__gpu, grid, block, 0, stream, *params, in_gfs, rhs_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}


/* Evaluate the constraints div E and G = Gamma - div A */
__global__ void __launch_bounds__(256) Maxwell_constraints__gpu(const paramstruct params, const double *__restrict__ in_gfs, double *__restrict__ aux_gfs) {
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
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double EU0_i0m2_i1_i2 = in_gfs[IDX4(EU0GF, i0-2,i1,i2)];
    const double EU0_i0m1_i1_i2 = in_gfs[IDX4(EU0GF, i0-1,i1,i2)];
    const double EU0_i0p1_i1_i2 = in_gfs[IDX4(EU0GF, i0+1,i1,i2)];
    const double EU0_i0p2_i1_i2 = in_gfs[IDX4(EU0GF, i0+2,i1,i2)];
    const double EU1_i0_i1m2_i2 = in_gfs[IDX4(EU1GF, i0,i1-2,i2)];
    const double EU1_i0_i1m1_i2 = in_gfs[IDX4(EU1GF, i0,i1-1,i2)];
    const double EU1_i0_i1p1_i2 = in_gfs[IDX4(EU1GF, i0,i1+1,i2)];
    const double EU1_i0_i1p2_i2 = in_gfs[IDX4(EU1GF, i0,i1+2,i2)];
    const double EU2_i0_i1_i2m2 = in_gfs[IDX4(EU2GF, i0,i1,i2-2)];
    const double EU2_i0_i1_i2m1 = in_gfs[IDX4(EU2GF, i0,i1,i2-1)];
    const double EU2_i0_i1_i2p1 = in_gfs[IDX4(EU2GF, i0,i1,i2+1)];
    const double EU2_i0_i1_i2p2 = in_gfs[IDX4(EU2GF, i0,i1,i2+2)];
    const double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    const double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double AU_dD00 = invdx0*(AU0_i0m1_i1_i2*FDPart1_Rational_m2_3 + AU0_i0m2_i1_i2*FDPart1_Rational_1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_2_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12);
    const double AU_dD11 = invdx1*(AU1_i0_i1m1_i2*FDPart1_Rational_m2_3 + AU1_i0_i1m2_i2*FDPart1_Rational_1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_2_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12);
    const double AU_dD22 = invdx2*(AU2_i0_i1_i2m1*FDPart1_Rational_m2_3 + AU2_i0_i1_i2m2*FDPart1_Rational_1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_2_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12);
    const double EU_dD00 = invdx0*(EU0_i0m1_i1_i2*FDPart1_Rational_m2_3 + EU0_i0m2_i1_i2*FDPart1_Rational_1_12 + EU0_i0p1_i1_i2*FDPart1_Rational_2_3 + EU0_i0p2_i1_i2*FDPart1_Rational_m1_12);
    const double EU_dD11 = invdx1*(EU1_i0_i1m1_i2*FDPart1_Rational_m2_3 + EU1_i0_i1m2_i2*FDPart1_Rational_1_12 + EU1_i0_i1p1_i2*FDPart1_Rational_2_3 + EU1_i0_i1p2_i2*FDPart1_Rational_m1_12);
    const double EU_dD22 = invdx2*(EU2_i0_i1_i2m1*FDPart1_Rational_m2_3 + EU2_i0_i1_i2m2*FDPart1_Rational_1_12 + EU2_i0_i1_i2p1*FDPart1_Rational_2_3 + EU2_i0_i1_i2p2*FDPart1_Rational_m1_12);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
    aux_gfs[IDX4(DIVEGF, i0, i1, i2)] = EU_dD00 + EU_dD11 + EU_dD22;
    aux_gfs[IDX4(GGF, i0, i1, i2)] = -AU_dD00 - AU_dD11 - AU_dD22 + Gamma;
  }
  
}

extern "C" int Maxwell_constraints(const paramstruct *params, const double *in_gfs, double *aux_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs || !aux_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(1, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  hipLaunchKernelGGL(Maxwell_constraints__gpu, grid, block, 0, stream, *params, in_gfs, aux_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}

template <int S>
__global__ void __launch_bounds__(256) rhs_eval_rk4_substep__gpu(const paramstruct params, const double *__restrict__ in_gfs, double *rk_yn, double *rk_rt, double *rk_out, const double dt) {
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
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double EU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double EU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double EU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double AU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double AU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double AU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double AU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double AU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double AU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double AU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double AU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double AU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double AU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double AU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double AU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double AU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double AU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double AU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double AU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double AU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double AU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double AU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double AU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double AU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double AU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double AU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double AU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double AU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double AU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double AU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
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
    const double FDPart1_0 = ((invdx0)*(invdx0));
    const double FDPart1_1 = AU0*FDPart1_Rational_m5_2;
    const double FDPart1_2 = ((invdx1)*(invdx1));
    const double FDPart1_3 = ((invdx2)*(invdx2));
    const double FDPart1_4 = AU1*FDPart1_Rational_m5_2;
    const double FDPart1_5 = AU2*FDPart1_Rational_m5_2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_8 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_9 = FDPart1_Rational_m5_2*psi;
    const double AU_dDD000 = FDPart1_0*(AU0_i0m1_i1_i2*FDPart1_Rational_4_3 + AU0_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_4_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD011 = FDPart1_2*(AU0_i0_i1m1_i2*FDPart1_Rational_4_3 + AU0_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU0_i0_i1p1_i2*FDPart1_Rational_4_3 + AU0_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD022 = FDPart1_3*(AU0_i0_i1_i2m1*FDPart1_Rational_4_3 + AU0_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU0_i0_i1_i2p1*FDPart1_Rational_4_3 + AU0_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD100 = FDPart1_0*(AU1_i0m1_i1_i2*FDPart1_Rational_4_3 + AU1_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU1_i0p1_i1_i2*FDPart1_Rational_4_3 + AU1_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD111 = FDPart1_2*(AU1_i0_i1m1_i2*FDPart1_Rational_4_3 + AU1_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_4_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD122 = FDPart1_3*(AU1_i0_i1_i2m1*FDPart1_Rational_4_3 + AU1_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU1_i0_i1_i2p1*FDPart1_Rational_4_3 + AU1_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD200 = FDPart1_0*(AU2_i0m1_i1_i2*FDPart1_Rational_4_3 + AU2_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU2_i0p1_i1_i2*FDPart1_Rational_4_3 + AU2_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD211 = FDPart1_2*(AU2_i0_i1m1_i2*FDPart1_Rational_4_3 + AU2_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU2_i0_i1p1_i2*FDPart1_Rational_4_3 + AU2_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD222 = FDPart1_3*(AU2_i0_i1_i2m1*FDPart1_Rational_4_3 + AU2_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_4_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double psi_dD0 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_7 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_8 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_0*(FDPart1_6 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_2*(FDPart1_7 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_3*(FDPart1_8 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
  const double __rhs_AU0 = -EU0 - psi_dD0;
  const double __rhs_AU1 = -EU1 - psi_dD1;
  const double __rhs_AU2 = -EU2 - psi_dD2;
  const double __rhs_EU0 = -AU_dDD000 - AU_dDD011 - AU_dDD022 + Gamma_dD0;
  const double __rhs_EU1 = -AU_dDD100 - AU_dDD111 - AU_dDD122 + Gamma_dD1;
  const double __rhs_EU2 = -AU_dDD200 - AU_dDD211 - AU_dDD222 + Gamma_dD2;
  const double __rhs_GAMMA = -psi_dDD00 - psi_dDD11 - psi_dDD22;
  const double __rhs_PSI = -Gamma;
  __builtin_amdgcn_sched_barrier(0);
  NRPY_RK4_PRELOAD(S, AU0GF, 0)
  NRPY_RK4_PRELOAD(S, AU1GF, 1)
  NRPY_RK4_PRELOAD(S, AU2GF, 2)
  NRPY_RK4_PRELOAD(S, EU0GF, 3)
  NRPY_RK4_PRELOAD(S, EU1GF, 4)
  NRPY_RK4_PRELOAD(S, EU2GF, 5)
  NRPY_RK4_PRELOAD(S, GAMMAGF, 6)
  NRPY_RK4_PRELOAD(S, PSIGF, 7)
  NRPY_RK4_STORE(S, 0, __rhs_AU0);
  NRPY_RK4_STORE(S, 1, __rhs_AU1);
  NRPY_RK4_STORE(S, 2, __rhs_AU2);
  NRPY_RK4_STORE(S, 3, __rhs_EU0);
  NRPY_RK4_STORE(S, 4, __rhs_EU1);
  NRPY_RK4_STORE(S, 5, __rhs_EU2);
  NRPY_RK4_STORE(S, 6, __rhs_GAMMA);
  NRPY_RK4_STORE(S, 7, __rhs_PSI);
  }
}
extern "C" int rhs_eval_rk4_substep(const int S, const rfm_struct *rfmstruct, const paramstruct *params, const double *auxevol_gfs, const double *in_gfs, double *y_n, double *rt, double *out, const double dt, hipStream_t stream) {
  if (!params || !y_n || !rt || !out) return NRPY_ERR_NULL;
  if (S < 0 || S > 3) return NRPY_ERR_PARAM;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(2, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<0>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 1: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<1>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 2: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<2>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 3: hipLaunchKernelGGL(rhs_eval_rk4_substep__gpu<3>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}
template <int S>
__global__ void __launch_bounds__(256) rhs_eval_rk4_substep_edge__gpu(const paramstruct params, const double *__restrict__ in_gfs, double *rk_yn, double *rk_rt, double *rk_out, const double dt) {
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
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    double EU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    double EU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    double EU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    double AU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    double AU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    double AU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    double AU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    double AU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    double AU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    double AU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    double AU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    double AU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    double AU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    double AU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    double AU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    double AU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    double AU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    double AU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    double AU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    double AU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    double AU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    double AU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    double AU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    double AU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    double AU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    double AU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    double AU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    double AU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    double AU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    double AU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
    double psi_i0_i1_i2m2 = in_gfs[IDX4(PSIGF, i0,i1,i2-2)];
    double psi_i0_i1_i2m1 = in_gfs[IDX4(PSIGF, i0,i1,i2-1)];
    double psi_i0_i1m2_i2 = in_gfs[IDX4(PSIGF, i0,i1-2,i2)];
    double psi_i0_i1m1_i2 = in_gfs[IDX4(PSIGF, i0,i1-1,i2)];
    double psi_i0m2_i1_i2 = in_gfs[IDX4(PSIGF, i0-2,i1,i2)];
    double psi_i0m1_i1_i2 = in_gfs[IDX4(PSIGF, i0-1,i1,i2)];
    double psi = in_gfs[IDX4(PSIGF, i0,i1,i2)];
    double psi_i0p1_i1_i2 = in_gfs[IDX4(PSIGF, i0+1,i1,i2)];
    double psi_i0p2_i1_i2 = in_gfs[IDX4(PSIGF, i0+2,i1,i2)];
    double psi_i0_i1p1_i2 = in_gfs[IDX4(PSIGF, i0,i1+1,i2)];
    double psi_i0_i1p2_i2 = in_gfs[IDX4(PSIGF, i0,i1+2,i2)];
    double psi_i0_i1_i2p1 = in_gfs[IDX4(PSIGF, i0,i1,i2+1)];
    double psi_i0_i1_i2p2 = in_gfs[IDX4(PSIGF, i0,i1,i2+2)];
    double Gamma_i0_i1_i2m2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-2)];
    double Gamma_i0_i1_i2m1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2-1)];
    double Gamma_i0_i1m2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-2,i2)];
    double Gamma_i0_i1m1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1-1,i2)];
    double Gamma_i0m2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-2,i1,i2)];
    double Gamma_i0m1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0-1,i1,i2)];
    double Gamma = in_gfs[IDX4(GAMMAGF, i0,i1,i2)];
    double Gamma_i0p1_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+1,i1,i2)];
    double Gamma_i0p2_i1_i2 = in_gfs[IDX4(GAMMAGF, i0+2,i1,i2)];
    double Gamma_i0_i1p1_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+1,i2)];
    double Gamma_i0_i1p2_i2 = in_gfs[IDX4(GAMMAGF, i0,i1+2,i2)];
    double Gamma_i0_i1_i2p1 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+1)];
    double Gamma_i0_i1_i2p2 = in_gfs[IDX4(GAMMAGF, i0,i1,i2+2)];
    if (i0 == NGHOSTS) {
      AU0_i0m1_i1_i2 = fma(1.0, AU0_i0p2_i1_i2, fma(-3.0, AU0_i0p1_i1_i2, 3.0 * AU0));
      AU0_i0m2_i1_i2 = fma(3.0, AU0_i0p2_i1_i2, fma(-8.0, AU0_i0p1_i1_i2, 6.0 * AU0));
    } else if (i0 == NGHOSTS + 1) {
      AU0_i0m2_i1_i2 = fma(1.0, AU0_i0p1_i1_i2, fma(-3.0, AU0, 3.0 * AU0_i0m1_i1_i2));
    }
    if (i0 == Nxx0 + NGHOSTS - 1) {
      AU0_i0p1_i1_i2 = fma(1.0, AU0_i0m2_i1_i2, fma(-3.0, AU0_i0m1_i1_i2, 3.0 * AU0));
      AU0_i0p2_i1_i2 = fma(3.0, AU0_i0m2_i1_i2, fma(-8.0, AU0_i0m1_i1_i2, 6.0 * AU0));
    } else if (i0 == Nxx0 + NGHOSTS - 2) {
      AU0_i0p2_i1_i2 = fma(1.0, AU0_i0m1_i1_i2, fma(-3.0, AU0, 3.0 * AU0_i0p1_i1_i2));
    }
    if (i1 == NGHOSTS) {
      AU0_i0_i1m1_i2 = fma(1.0, AU0_i0_i1p2_i2, fma(-3.0, AU0_i0_i1p1_i2, 3.0 * AU0));
      AU0_i0_i1m2_i2 = fma(3.0, AU0_i0_i1p2_i2, fma(-8.0, AU0_i0_i1p1_i2, 6.0 * AU0));
    } else if (i1 == NGHOSTS + 1) {
      AU0_i0_i1m2_i2 = fma(1.0, AU0_i0_i1p1_i2, fma(-3.0, AU0, 3.0 * AU0_i0_i1m1_i2));
    }
    if (i1 == Nxx1 + NGHOSTS - 1) {
      AU0_i0_i1p1_i2 = fma(1.0, AU0_i0_i1m2_i2, fma(-3.0, AU0_i0_i1m1_i2, 3.0 * AU0));
      AU0_i0_i1p2_i2 = fma(3.0, AU0_i0_i1m2_i2, fma(-8.0, AU0_i0_i1m1_i2, 6.0 * AU0));
    } else if (i1 == Nxx1 + NGHOSTS - 2) {
      AU0_i0_i1p2_i2 = fma(1.0, AU0_i0_i1m1_i2, fma(-3.0, AU0, 3.0 * AU0_i0_i1p1_i2));
    }
    if (i2 == NGHOSTS) {
      AU0_i0_i1_i2m1 = fma(1.0, AU0_i0_i1_i2p2, fma(-3.0, AU0_i0_i1_i2p1, 3.0 * AU0));
      AU0_i0_i1_i2m2 = fma(3.0, AU0_i0_i1_i2p2, fma(-8.0, AU0_i0_i1_i2p1, 6.0 * AU0));
    } else if (i2 == NGHOSTS + 1) {
      AU0_i0_i1_i2m2 = fma(1.0, AU0_i0_i1_i2p1, fma(-3.0, AU0, 3.0 * AU0_i0_i1_i2m1));
    }
    if (i2 == Nxx2 + NGHOSTS - 1) {
      AU0_i0_i1_i2p1 = fma(1.0, AU0_i0_i1_i2m2, fma(-3.0, AU0_i0_i1_i2m1, 3.0 * AU0));
      AU0_i0_i1_i2p2 = fma(3.0, AU0_i0_i1_i2m2, fma(-8.0, AU0_i0_i1_i2m1, 6.0 * AU0));
    } else if (i2 == Nxx2 + NGHOSTS - 2) {
      AU0_i0_i1_i2p2 = fma(1.0, AU0_i0_i1_i2m1, fma(-3.0, AU0, 3.0 * AU0_i0_i1_i2p1));
    }
    if (i0 == NGHOSTS) {
      AU1_i0m1_i1_i2 = fma(1.0, AU1_i0p2_i1_i2, fma(-3.0, AU1_i0p1_i1_i2, 3.0 * AU1));
      AU1_i0m2_i1_i2 = fma(3.0, AU1_i0p2_i1_i2, fma(-8.0, AU1_i0p1_i1_i2, 6.0 * AU1));
    } else if (i0 == NGHOSTS + 1) {
      AU1_i0m2_i1_i2 = fma(1.0, AU1_i0p1_i1_i2, fma(-3.0, AU1, 3.0 * AU1_i0m1_i1_i2));
    }
    if (i0 == Nxx0 + NGHOSTS - 1) {
      AU1_i0p1_i1_i2 = fma(1.0, AU1_i0m2_i1_i2, fma(-3.0, AU1_i0m1_i1_i2, 3.0 * AU1));
      AU1_i0p2_i1_i2 = fma(3.0, AU1_i0m2_i1_i2, fma(-8.0, AU1_i0m1_i1_i2, 6.0 * AU1));
    } else if (i0 == Nxx0 + NGHOSTS - 2) {
      AU1_i0p2_i1_i2 = fma(1.0, AU1_i0m1_i1_i2, fma(-3.0, AU1, 3.0 * AU1_i0p1_i1_i2));
    }
    if (i1 == NGHOSTS) {
      AU1_i0_i1m1_i2 = fma(1.0, AU1_i0_i1p2_i2, fma(-3.0, AU1_i0_i1p1_i2, 3.0 * AU1));
      AU1_i0_i1m2_i2 = fma(3.0, AU1_i0_i1p2_i2, fma(-8.0, AU1_i0_i1p1_i2, 6.0 * AU1));
    } else if (i1 == NGHOSTS + 1) {
      AU1_i0_i1m2_i2 = fma(1.0, AU1_i0_i1p1_i2, fma(-3.0, AU1, 3.0 * AU1_i0_i1m1_i2));
    }
    if (i1 == Nxx1 + NGHOSTS - 1) {
      AU1_i0_i1p1_i2 = fma(1.0, AU1_i0_i1m2_i2, fma(-3.0, AU1_i0_i1m1_i2, 3.0 * AU1));
      AU1_i0_i1p2_i2 = fma(3.0, AU1_i0_i1m2_i2, fma(-8.0, AU1_i0_i1m1_i2, 6.0 * AU1));
    } else if (i1 == Nxx1 + NGHOSTS - 2) {
      AU1_i0_i1p2_i2 = fma(1.0, AU1_i0_i1m1_i2, fma(-3.0, AU1, 3.0 * AU1_i0_i1p1_i2));
    }
    if (i2 == NGHOSTS) {
      AU1_i0_i1_i2m1 = fma(1.0, AU1_i0_i1_i2p2, fma(-3.0, AU1_i0_i1_i2p1, 3.0 * AU1));
      AU1_i0_i1_i2m2 = fma(3.0, AU1_i0_i1_i2p2, fma(-8.0, AU1_i0_i1_i2p1, 6.0 * AU1));
    } else if (i2 == NGHOSTS + 1) {
      AU1_i0_i1_i2m2 = fma(1.0, AU1_i0_i1_i2p1, fma(-3.0, AU1, 3.0 * AU1_i0_i1_i2m1));
    }
    if (i2 == Nxx2 + NGHOSTS - 1) {
      AU1_i0_i1_i2p1 = fma(1.0, AU1_i0_i1_i2m2, fma(-3.0, AU1_i0_i1_i2m1, 3.0 * AU1));
      AU1_i0_i1_i2p2 = fma(3.0, AU1_i0_i1_i2m2, fma(-8.0, AU1_i0_i1_i2m1, 6.0 * AU1));
    } else if (i2 == Nxx2 + NGHOSTS - 2) {
      AU1_i0_i1_i2p2 = fma(1.0, AU1_i0_i1_i2m1, fma(-3.0, AU1, 3.0 * AU1_i0_i1_i2p1));
    }
    if (i0 == NGHOSTS) {
      AU2_i0m1_i1_i2 = fma(1.0, AU2_i0p2_i1_i2, fma(-3.0, AU2_i0p1_i1_i2, 3.0 * AU2));
      AU2_i0m2_i1_i2 = fma(3.0, AU2_i0p2_i1_i2, fma(-8.0, AU2_i0p1_i1_i2, 6.0 * AU2));
    } else if (i0 == NGHOSTS + 1) {
      AU2_i0m2_i1_i2 = fma(1.0, AU2_i0p1_i1_i2, fma(-3.0, AU2, 3.0 * AU2_i0m1_i1_i2));
    }
    if (i0 == Nxx0 + NGHOSTS - 1) {
      AU2_i0p1_i1_i2 = fma(1.0, AU2_i0m2_i1_i2, fma(-3.0, AU2_i0m1_i1_i2, 3.0 * AU2));
      AU2_i0p2_i1_i2 = fma(3.0, AU2_i0m2_i1_i2, fma(-8.0, AU2_i0m1_i1_i2, 6.0 * AU2));
    } else if (i0 == Nxx0 + NGHOSTS - 2) {
      AU2_i0p2_i1_i2 = fma(1.0, AU2_i0m1_i1_i2, fma(-3.0, AU2, 3.0 * AU2_i0p1_i1_i2));
    }
    if (i1 == NGHOSTS) {
      AU2_i0_i1m1_i2 = fma(1.0, AU2_i0_i1p2_i2, fma(-3.0, AU2_i0_i1p1_i2, 3.0 * AU2));
      AU2_i0_i1m2_i2 = fma(3.0, AU2_i0_i1p2_i2, fma(-8.0, AU2_i0_i1p1_i2, 6.0 * AU2));
    } else if (i1 == NGHOSTS + 1) {
      AU2_i0_i1m2_i2 = fma(1.0, AU2_i0_i1p1_i2, fma(-3.0, AU2, 3.0 * AU2_i0_i1m1_i2));
    }
    if (i1 == Nxx1 + NGHOSTS - 1) {
      AU2_i0_i1p1_i2 = fma(1.0, AU2_i0_i1m2_i2, fma(-3.0, AU2_i0_i1m1_i2, 3.0 * AU2));
      AU2_i0_i1p2_i2 = fma(3.0, AU2_i0_i1m2_i2, fma(-8.0, AU2_i0_i1m1_i2, 6.0 * AU2));
    } else if (i1 == Nxx1 + NGHOSTS - 2) {
      AU2_i0_i1p2_i2 = fma(1.0, AU2_i0_i1m1_i2, fma(-3.0, AU2, 3.0 * AU2_i0_i1p1_i2));
    }
    if (i2 == NGHOSTS) {
      AU2_i0_i1_i2m1 = fma(1.0, AU2_i0_i1_i2p2, fma(-3.0, AU2_i0_i1_i2p1, 3.0 * AU2));
      AU2_i0_i1_i2m2 = fma(3.0, AU2_i0_i1_i2p2, fma(-8.0, AU2_i0_i1_i2p1, 6.0 * AU2));
    } else if (i2 == NGHOSTS + 1) {
      AU2_i0_i1_i2m2 = fma(1.0, AU2_i0_i1_i2p1, fma(-3.0, AU2, 3.0 * AU2_i0_i1_i2m1));
    }
    if (i2 == Nxx2 + NGHOSTS - 1) {
      AU2_i0_i1_i2p1 = fma(1.0, AU2_i0_i1_i2m2, fma(-3.0, AU2_i0_i1_i2m1, 3.0 * AU2));
      AU2_i0_i1_i2p2 = fma(3.0, AU2_i0_i1_i2m2, fma(-8.0, AU2_i0_i1_i2m1, 6.0 * AU2));
    } else if (i2 == Nxx2 + NGHOSTS - 2) {
      AU2_i0_i1_i2p2 = fma(1.0, AU2_i0_i1_i2m1, fma(-3.0, AU2, 3.0 * AU2_i0_i1_i2p1));
    }
    if (i0 == NGHOSTS) {
      Gamma_i0m1_i1_i2 = fma(1.0, Gamma_i0p2_i1_i2, fma(-3.0, Gamma_i0p1_i1_i2, 3.0 * Gamma));
      Gamma_i0m2_i1_i2 = fma(3.0, Gamma_i0p2_i1_i2, fma(-8.0, Gamma_i0p1_i1_i2, 6.0 * Gamma));
    } else if (i0 == NGHOSTS + 1) {
      Gamma_i0m2_i1_i2 = fma(1.0, Gamma_i0p1_i1_i2, fma(-3.0, Gamma, 3.0 * Gamma_i0m1_i1_i2));
    }
    if (i0 == Nxx0 + NGHOSTS - 1) {
      Gamma_i0p1_i1_i2 = fma(1.0, Gamma_i0m2_i1_i2, fma(-3.0, Gamma_i0m1_i1_i2, 3.0 * Gamma));
      Gamma_i0p2_i1_i2 = fma(3.0, Gamma_i0m2_i1_i2, fma(-8.0, Gamma_i0m1_i1_i2, 6.0 * Gamma));
    } else if (i0 == Nxx0 + NGHOSTS - 2) {
      Gamma_i0p2_i1_i2 = fma(1.0, Gamma_i0m1_i1_i2, fma(-3.0, Gamma, 3.0 * Gamma_i0p1_i1_i2));
    }
    if (i1 == NGHOSTS) {
      Gamma_i0_i1m1_i2 = fma(1.0, Gamma_i0_i1p2_i2, fma(-3.0, Gamma_i0_i1p1_i2, 3.0 * Gamma));
      Gamma_i0_i1m2_i2 = fma(3.0, Gamma_i0_i1p2_i2, fma(-8.0, Gamma_i0_i1p1_i2, 6.0 * Gamma));
    } else if (i1 == NGHOSTS + 1) {
      Gamma_i0_i1m2_i2 = fma(1.0, Gamma_i0_i1p1_i2, fma(-3.0, Gamma, 3.0 * Gamma_i0_i1m1_i2));
    }
    if (i1 == Nxx1 + NGHOSTS - 1) {
      Gamma_i0_i1p1_i2 = fma(1.0, Gamma_i0_i1m2_i2, fma(-3.0, Gamma_i0_i1m1_i2, 3.0 * Gamma));
      Gamma_i0_i1p2_i2 = fma(3.0, Gamma_i0_i1m2_i2, fma(-8.0, Gamma_i0_i1m1_i2, 6.0 * Gamma));
    } else if (i1 == Nxx1 + NGHOSTS - 2) {
      Gamma_i0_i1p2_i2 = fma(1.0, Gamma_i0_i1m1_i2, fma(-3.0, Gamma, 3.0 * Gamma_i0_i1p1_i2));
    }
    if (i2 == NGHOSTS) {
      Gamma_i0_i1_i2m1 = fma(1.0, Gamma_i0_i1_i2p2, fma(-3.0, Gamma_i0_i1_i2p1, 3.0 * Gamma));
      Gamma_i0_i1_i2m2 = fma(3.0, Gamma_i0_i1_i2p2, fma(-8.0, Gamma_i0_i1_i2p1, 6.0 * Gamma));
    } else if (i2 == NGHOSTS + 1) {
      Gamma_i0_i1_i2m2 = fma(1.0, Gamma_i0_i1_i2p1, fma(-3.0, Gamma, 3.0 * Gamma_i0_i1_i2m1));
    }
    if (i2 == Nxx2 + NGHOSTS - 1) {
      Gamma_i0_i1_i2p1 = fma(1.0, Gamma_i0_i1_i2m2, fma(-3.0, Gamma_i0_i1_i2m1, 3.0 * Gamma));
      Gamma_i0_i1_i2p2 = fma(3.0, Gamma_i0_i1_i2m2, fma(-8.0, Gamma_i0_i1_i2m1, 6.0 * Gamma));
    } else if (i2 == Nxx2 + NGHOSTS - 2) {
      Gamma_i0_i1_i2p2 = fma(1.0, Gamma_i0_i1_i2m1, fma(-3.0, Gamma, 3.0 * Gamma_i0_i1_i2p1));
    }
    if (i0 == NGHOSTS) {
      psi_i0m1_i1_i2 = fma(1.0, psi_i0p2_i1_i2, fma(-3.0, psi_i0p1_i1_i2, 3.0 * psi));
      psi_i0m2_i1_i2 = fma(3.0, psi_i0p2_i1_i2, fma(-8.0, psi_i0p1_i1_i2, 6.0 * psi));
    } else if (i0 == NGHOSTS + 1) {
      psi_i0m2_i1_i2 = fma(1.0, psi_i0p1_i1_i2, fma(-3.0, psi, 3.0 * psi_i0m1_i1_i2));
    }
    if (i0 == Nxx0 + NGHOSTS - 1) {
      psi_i0p1_i1_i2 = fma(1.0, psi_i0m2_i1_i2, fma(-3.0, psi_i0m1_i1_i2, 3.0 * psi));
      psi_i0p2_i1_i2 = fma(3.0, psi_i0m2_i1_i2, fma(-8.0, psi_i0m1_i1_i2, 6.0 * psi));
    } else if (i0 == Nxx0 + NGHOSTS - 2) {
      psi_i0p2_i1_i2 = fma(1.0, psi_i0m1_i1_i2, fma(-3.0, psi, 3.0 * psi_i0p1_i1_i2));
    }
    if (i1 == NGHOSTS) {
      psi_i0_i1m1_i2 = fma(1.0, psi_i0_i1p2_i2, fma(-3.0, psi_i0_i1p1_i2, 3.0 * psi));
      psi_i0_i1m2_i2 = fma(3.0, psi_i0_i1p2_i2, fma(-8.0, psi_i0_i1p1_i2, 6.0 * psi));
    } else if (i1 == NGHOSTS + 1) {
      psi_i0_i1m2_i2 = fma(1.0, psi_i0_i1p1_i2, fma(-3.0, psi, 3.0 * psi_i0_i1m1_i2));
    }
    if (i1 == Nxx1 + NGHOSTS - 1) {
      psi_i0_i1p1_i2 = fma(1.0, psi_i0_i1m2_i2, fma(-3.0, psi_i0_i1m1_i2, 3.0 * psi));
      psi_i0_i1p2_i2 = fma(3.0, psi_i0_i1m2_i2, fma(-8.0, psi_i0_i1m1_i2, 6.0 * psi));
    } else if (i1 == Nxx1 + NGHOSTS - 2) {
      psi_i0_i1p2_i2 = fma(1.0, psi_i0_i1m1_i2, fma(-3.0, psi, 3.0 * psi_i0_i1p1_i2));
    }
    if (i2 == NGHOSTS) {
      psi_i0_i1_i2m1 = fma(1.0, psi_i0_i1_i2p2, fma(-3.0, psi_i0_i1_i2p1, 3.0 * psi));
      psi_i0_i1_i2m2 = fma(3.0, psi_i0_i1_i2p2, fma(-8.0, psi_i0_i1_i2p1, 6.0 * psi));
    } else if (i2 == NGHOSTS + 1) {
      psi_i0_i1_i2m2 = fma(1.0, psi_i0_i1_i2p1, fma(-3.0, psi, 3.0 * psi_i0_i1_i2m1));
    }
    if (i2 == Nxx2 + NGHOSTS - 1) {
      psi_i0_i1_i2p1 = fma(1.0, psi_i0_i1_i2m2, fma(-3.0, psi_i0_i1_i2m1, 3.0 * psi));
      psi_i0_i1_i2p2 = fma(3.0, psi_i0_i1_i2m2, fma(-8.0, psi_i0_i1_i2m1, 6.0 * psi));
    } else if (i2 == Nxx2 + NGHOSTS - 2) {
      psi_i0_i1_i2p2 = fma(1.0, psi_i0_i1_i2m1, fma(-3.0, psi, 3.0 * psi_i0_i1_i2p1));
    }
    const double FDPart1_Rational_1_12 = 1.0/12.0;
    const double FDPart1_Rational_2_3 = 2.0/3.0;
    const double FDPart1_Rational_4_3 = 4.0/3.0;
    const double FDPart1_Rational_m1_12 = -1.0/12.0;
    const double FDPart1_Rational_m2_3 = -2.0/3.0;
    const double FDPart1_Rational_m5_2 = -5.0/2.0;
    const double FDPart1_0 = ((invdx0)*(invdx0));
    const double FDPart1_1 = AU0*FDPart1_Rational_m5_2;
    const double FDPart1_2 = ((invdx1)*(invdx1));
    const double FDPart1_3 = ((invdx2)*(invdx2));
    const double FDPart1_4 = AU1*FDPart1_Rational_m5_2;
    const double FDPart1_5 = AU2*FDPart1_Rational_m5_2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_8 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_9 = FDPart1_Rational_m5_2*psi;
    const double AU_dDD000 = FDPart1_0*(AU0_i0m1_i1_i2*FDPart1_Rational_4_3 + AU0_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_4_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD011 = FDPart1_2*(AU0_i0_i1m1_i2*FDPart1_Rational_4_3 + AU0_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU0_i0_i1p1_i2*FDPart1_Rational_4_3 + AU0_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD022 = FDPart1_3*(AU0_i0_i1_i2m1*FDPart1_Rational_4_3 + AU0_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU0_i0_i1_i2p1*FDPart1_Rational_4_3 + AU0_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD100 = FDPart1_0*(AU1_i0m1_i1_i2*FDPart1_Rational_4_3 + AU1_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU1_i0p1_i1_i2*FDPart1_Rational_4_3 + AU1_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD111 = FDPart1_2*(AU1_i0_i1m1_i2*FDPart1_Rational_4_3 + AU1_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_4_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD122 = FDPart1_3*(AU1_i0_i1_i2m1*FDPart1_Rational_4_3 + AU1_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU1_i0_i1_i2p1*FDPart1_Rational_4_3 + AU1_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD200 = FDPart1_0*(AU2_i0m1_i1_i2*FDPart1_Rational_4_3 + AU2_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU2_i0p1_i1_i2*FDPart1_Rational_4_3 + AU2_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD211 = FDPart1_2*(AU2_i0_i1m1_i2*FDPart1_Rational_4_3 + AU2_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU2_i0_i1p1_i2*FDPart1_Rational_4_3 + AU2_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD222 = FDPart1_3*(AU2_i0_i1_i2m1*FDPart1_Rational_4_3 + AU2_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_4_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double psi_dD0 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_7 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_8 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_0*(FDPart1_6 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_2*(FDPart1_7 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_3*(FDPart1_8 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
  const double __rhs_AU0 = -EU0 - psi_dD0;
  const double __rhs_AU1 = -EU1 - psi_dD1;
  const double __rhs_AU2 = -EU2 - psi_dD2;
  const double __rhs_EU0 = -AU_dDD000 - AU_dDD011 - AU_dDD022 + Gamma_dD0;
  const double __rhs_EU1 = -AU_dDD100 - AU_dDD111 - AU_dDD122 + Gamma_dD1;
  const double __rhs_EU2 = -AU_dDD200 - AU_dDD211 - AU_dDD222 + Gamma_dD2;
  const double __rhs_GAMMA = -psi_dDD00 - psi_dDD11 - psi_dDD22;
  const double __rhs_PSI = -Gamma;
  __builtin_amdgcn_sched_barrier(0);
  NRPY_RK4_PRELOAD(S, AU0GF, 0)
  NRPY_RK4_PRELOAD(S, AU1GF, 1)
  NRPY_RK4_PRELOAD(S, AU2GF, 2)
  NRPY_RK4_PRELOAD(S, EU0GF, 3)
  NRPY_RK4_PRELOAD(S, EU1GF, 4)
  NRPY_RK4_PRELOAD(S, EU2GF, 5)
  NRPY_RK4_PRELOAD(S, GAMMAGF, 6)
  NRPY_RK4_PRELOAD(S, PSIGF, 7)
  NRPY_RK4_STORE(S, 0, __rhs_AU0);
  NRPY_RK4_STORE(S, 1, __rhs_AU1);
  NRPY_RK4_STORE(S, 2, __rhs_AU2);
  NRPY_RK4_STORE(S, 3, __rhs_EU0);
  NRPY_RK4_STORE(S, 4, __rhs_EU1);
  NRPY_RK4_STORE(S, 5, __rhs_EU2);
  NRPY_RK4_STORE(S, 6, __rhs_GAMMA);
  NRPY_RK4_STORE(S, 7, __rhs_PSI);
  }
}
extern "C" int rhs_eval_rk4_substep_edge(const int S, const rfm_struct *rfmstruct, const paramstruct *params, const double *auxevol_gfs, const double *in_gfs, double *y_n, double *rt, double *out, const double dt, hipStream_t stream) {
  if (!params || !y_n || !rt || !out) return NRPY_ERR_NULL;
  if (S < 0 || S > 3) return NRPY_ERR_PARAM;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(3, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_rk4_substep_edge__gpu<0>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 1: hipLaunchKernelGGL(rhs_eval_rk4_substep_edge__gpu<1>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 2: hipLaunchKernelGGL(rhs_eval_rk4_substep_edge__gpu<2>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
    case 3: hipLaunchKernelGGL(rhs_eval_rk4_substep_edge__gpu<3>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}
template <int S>
__global__ void __launch_bounds__(256) rhs_eval_rk4_substep_shell__gpu(const paramstruct params, const double *__restrict__ in_gfs, double *rk_yn, double *rk_rt, double *rk_out, const double dt, double *__restrict__ shell_rhs) {
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
  {
    /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
    const double EU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
    const double EU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
    const double EU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
    const double AU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
    const double AU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
    const double AU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
    const double AU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
    const double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
    const double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
    const double AU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
    const double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
    const double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
    const double AU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
    const double AU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
    const double AU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
    const double AU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
    const double AU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
    const double AU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
    const double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
    const double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
    const double AU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
    const double AU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
    const double AU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
    const double AU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
    const double AU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
    const double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
    const double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
    const double AU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
    const double AU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
    const double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
    const double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
    const double AU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
    const double AU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
    const double AU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
    const double AU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
    const double AU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
    const double AU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
    const double AU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
    const double AU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
    const double AU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
    const double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
    const double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
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
    const double FDPart1_0 = ((invdx0)*(invdx0));
    const double FDPart1_1 = AU0*FDPart1_Rational_m5_2;
    const double FDPart1_2 = ((invdx1)*(invdx1));
    const double FDPart1_3 = ((invdx2)*(invdx2));
    const double FDPart1_4 = AU1*FDPart1_Rational_m5_2;
    const double FDPart1_5 = AU2*FDPart1_Rational_m5_2;
    const double FDPart1_6 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
    const double FDPart1_7 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
    const double FDPart1_8 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
    const double FDPart1_9 = FDPart1_Rational_m5_2*psi;
    const double AU_dDD000 = FDPart1_0*(AU0_i0m1_i1_i2*FDPart1_Rational_4_3 + AU0_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_4_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD011 = FDPart1_2*(AU0_i0_i1m1_i2*FDPart1_Rational_4_3 + AU0_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU0_i0_i1p1_i2*FDPart1_Rational_4_3 + AU0_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD022 = FDPart1_3*(AU0_i0_i1_i2m1*FDPart1_Rational_4_3 + AU0_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU0_i0_i1_i2p1*FDPart1_Rational_4_3 + AU0_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_1);
    const double AU_dDD100 = FDPart1_0*(AU1_i0m1_i1_i2*FDPart1_Rational_4_3 + AU1_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU1_i0p1_i1_i2*FDPart1_Rational_4_3 + AU1_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD111 = FDPart1_2*(AU1_i0_i1m1_i2*FDPart1_Rational_4_3 + AU1_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_4_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD122 = FDPart1_3*(AU1_i0_i1_i2m1*FDPart1_Rational_4_3 + AU1_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU1_i0_i1_i2p1*FDPart1_Rational_4_3 + AU1_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_4);
    const double AU_dDD200 = FDPart1_0*(AU2_i0m1_i1_i2*FDPart1_Rational_4_3 + AU2_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU2_i0p1_i1_i2*FDPart1_Rational_4_3 + AU2_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD211 = FDPart1_2*(AU2_i0_i1m1_i2*FDPart1_Rational_4_3 + AU2_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU2_i0_i1p1_i2*FDPart1_Rational_4_3 + AU2_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double AU_dDD222 = FDPart1_3*(AU2_i0_i1_i2m1*FDPart1_Rational_4_3 + AU2_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_4_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_5);
    const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
    const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
    const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
    const double psi_dD0 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
    const double psi_dD1 = invdx1*(FDPart1_7 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
    const double psi_dD2 = invdx2*(FDPart1_8 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
    const double psi_dDD00 = FDPart1_0*(FDPart1_6 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
    const double psi_dDD11 = FDPart1_2*(FDPart1_7 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
    const double psi_dDD22 = FDPart1_3*(FDPart1_8 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
    /* Step 2 of 2: evaluate right-hand sides and write to memory */
  const double __rhs_AU0 = -EU0 - psi_dD0;
  const double __rhs_AU1 = -EU1 - psi_dD1;
  const double __rhs_AU2 = -EU2 - psi_dD2;
  const double __rhs_EU0 = -AU_dDD000 - AU_dDD011 - AU_dDD022 + Gamma_dD0;
  const double __rhs_EU1 = -AU_dDD100 - AU_dDD111 - AU_dDD122 + Gamma_dD1;
  const double __rhs_EU2 = -AU_dDD200 - AU_dDD211 - AU_dDD222 + Gamma_dD2;
  const double __rhs_GAMMA = -psi_dDD00 - psi_dDD11 - psi_dDD22;
  const double __rhs_PSI = -Gamma;
  __builtin_amdgcn_sched_barrier(0);
  NRPY_RK4_PRELOAD(S, AU0GF, 0)
  NRPY_RK4_PRELOAD(S, AU1GF, 1)
  NRPY_RK4_PRELOAD(S, AU2GF, 2)
  NRPY_RK4_PRELOAD(S, EU0GF, 3)
  NRPY_RK4_PRELOAD(S, EU1GF, 4)
  NRPY_RK4_PRELOAD(S, EU2GF, 5)
  NRPY_RK4_PRELOAD(S, GAMMAGF, 6)
  NRPY_RK4_PRELOAD(S, PSIGF, 7)
  NRPY_RK4_STORE(S, 0, __rhs_AU0);
  NRPY_RK4_STORE(S, 1, __rhs_AU1);
  NRPY_RK4_STORE(S, 2, __rhs_AU2);
  NRPY_RK4_STORE(S, 3, __rhs_EU0);
  NRPY_RK4_STORE(S, 4, __rhs_EU1);
  NRPY_RK4_STORE(S, 5, __rhs_EU2);
  NRPY_RK4_STORE(S, 6, __rhs_GAMMA);
  NRPY_RK4_STORE(S, 7, __rhs_PSI);
  if (i1 == NGHOSTS || i1 == Nxx1 + NGHOSTS - 1 || i2 == NGHOSTS || i2 == Nxx2 + NGHOSTS - 1) {
    shell_rhs[IDX4(AU0GF, i0, i1, i2)] = __rhs_AU0;
    shell_rhs[IDX4(AU1GF, i0, i1, i2)] = __rhs_AU1;
    shell_rhs[IDX4(AU2GF, i0, i1, i2)] = __rhs_AU2;
    shell_rhs[IDX4(EU0GF, i0, i1, i2)] = __rhs_EU0;
    shell_rhs[IDX4(EU1GF, i0, i1, i2)] = __rhs_EU1;
    shell_rhs[IDX4(EU2GF, i0, i1, i2)] = __rhs_EU2;
    shell_rhs[IDX4(GAMMAGF, i0, i1, i2)] = __rhs_GAMMA;
    shell_rhs[IDX4(PSIGF, i0, i1, i2)] = __rhs_PSI;
  }
  if (i0 == NGHOSTS || i0 == Nxx0 + NGHOSTS - 1) {
    double *__restrict__ xb = shell_rhs + (size_t)NUM_EVOL_GFS * Nxx_plus_2NGHOSTS0 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2 + 2 * ((size_t)i1 + (size_t)Nxx_plus_2NGHOSTS1 * i2) + (i0 == NGHOSTS ? 0 : 1);
    xb[(size_t)AU0GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_AU0;
    xb[(size_t)AU1GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_AU1;
    xb[(size_t)AU2GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_AU2;
    xb[(size_t)EU0GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_EU0;
    xb[(size_t)EU1GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_EU1;
    xb[(size_t)EU2GF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_EU2;
    xb[(size_t)GAMMAGF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_GAMMA;
    xb[(size_t)PSIGF * 2 * Nxx_plus_2NGHOSTS1 * Nxx_plus_2NGHOSTS2] = __rhs_PSI;
  }
  }
}
extern "C" int rhs_eval_rk4_substep_shell(const int S, const paramstruct *params, const double *in_gfs, double *y_n, double *rt, double *out, double *shell_rhs, const double dt, hipStream_t stream) {
  if (!params || !y_n || !rt || !out || !shell_rhs) return NRPY_ERR_NULL;
  if (S < 0 || S > 3) return NRPY_ERR_PARAM;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(2, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_rk4_substep_shell__gpu<0>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt, shell_rhs); break;
    case 1: hipLaunchKernelGGL(rhs_eval_rk4_substep_shell__gpu<1>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt, shell_rhs); break;
    case 2: hipLaunchKernelGGL(rhs_eval_rk4_substep_shell__gpu<2>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt, shell_rhs); break;
    case 3: hipLaunchKernelGGL(rhs_eval_rk4_substep_shell__gpu<3>, grid, block, 0, stream, *params, in_gfs, y_n, rt, out, dt, shell_rhs); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}


/* Set up the initial data at all points on the numerical grid. */
__global__ void __launch_bounds__(256) initial_data__gpu(const paramstruct params, const double *__restrict__ xx0_arr, const double *__restrict__ xx1_arr, const double *__restrict__ xx2_arr, double *__restrict__ in_gfs) {
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
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
  const double tmp_0 = ((xx0)*(xx0)) + ((xx1)*(xx1)) + ((xx2)*(xx2));
  const double tmp_1 = sqrt(tmp_0);
  const double tmp_2 = time - tmp_1;
  const double tmp_3 = ((tmp_2)*(tmp_2));
  const double tmp_4 = exp(lam*tmp_3);
  const double tmp_5 = time + tmp_1;
  const double tmp_6 = ((tmp_5)*(tmp_5));
  const double tmp_7 = exp(lam*tmp_6);
  const double tmp_8 = tmp_2*tmp_7;
  const double tmp_9 = tmp_4*tmp_5;
  const double tmp_10 = 2*lam*tmp_0;
  const double tmp_11 = (1.0/((tmp_0)*(tmp_0)));
  const double tmp_12 = exp(-lam*(tmp_3 + tmp_6));
  const double tmp_13 = amp*tmp_11*tmp_12;
  const double tmp_14 = tmp_13*(tmp_1*(tmp_4 - tmp_7) + tmp_10*(tmp_8 + tmp_9));
  const double tmp_15 = tmp_14*xx1;
  const double tmp_16 = tmp_14*xx0;
  const double tmp_17 = 4*lam*time;
  const double tmp_18 = 2*time;
  const double tmp_19 = 2*tmp_1;
  const double tmp_20 = lam*(tmp_18 + tmp_19);
  const double tmp_21 = lam*(tmp_18 - tmp_19);
  const double tmp_22 = tmp_1*(-tmp_20*tmp_7 + tmp_21*tmp_4) + tmp_10*(tmp_20*tmp_8 + tmp_21*tmp_9 + tmp_4 + tmp_7);
  in_gfs[IDX4(AU0GF, i0, i1, i2)] = tmp_15;
  in_gfs[IDX4(AU1GF, i0, i1, i2)] = -tmp_16;
  in_gfs[IDX4(AU2GF, i0, i1, i2)] = 0;
  in_gfs[IDX4(EU0GF, i0, i1, i2)] = -tmp_13*tmp_22*xx1 + tmp_15*tmp_17;
  in_gfs[IDX4(EU1GF, i0, i1, i2)] = amp*tmp_11*tmp_12*tmp_22*xx0 - tmp_16*tmp_17;
  in_gfs[IDX4(EU2GF, i0, i1, i2)] = 0;
  in_gfs[IDX4(GAMMAGF, i0, i1, i2)] = 0;
  in_gfs[IDX4(PSIGF, i0, i1, i2)] = 0;
  
}

extern "C" int initial_data(const paramstruct *params, double *xx[3], double *in_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(4, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2));
  hipLaunchKernelGGL(initial_data__gpu, grid, block, 0, stream, *params, xx[0], xx[1], xx[2], in_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}


/* VJP pass 1: pointwise adjoint of rhs_eval */
__global__ void __launch_bounds__(256) rhs_eval_vjp_pointwise__gpu(const paramstruct params, const double *__restrict__ in_gfs, const double *__restrict__ cot_rhs_gfs, double *__restrict__ vjp_G) {
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
  /* Step 1 of 2: read gridfunctions and compute finite-difference stencils */
  const double EU0 = in_gfs[IDX4(EU0GF, i0,i1,i2)];
  const double EU1 = in_gfs[IDX4(EU1GF, i0,i1,i2)];
  const double EU2 = in_gfs[IDX4(EU2GF, i0,i1,i2)];
  const double AU0_i0_i1_i2m2 = in_gfs[IDX4(AU0GF, i0,i1,i2-2)];
  const double AU0_i0_i1_i2m1 = in_gfs[IDX4(AU0GF, i0,i1,i2-1)];
  const double AU0_i0_i1m2_i2 = in_gfs[IDX4(AU0GF, i0,i1-2,i2)];
  const double AU0_i0_i1m1_i2 = in_gfs[IDX4(AU0GF, i0,i1-1,i2)];
  const double AU0_i0m2_i1_i2 = in_gfs[IDX4(AU0GF, i0-2,i1,i2)];
  const double AU0_i0m1_i1_i2 = in_gfs[IDX4(AU0GF, i0-1,i1,i2)];
  const double AU0 = in_gfs[IDX4(AU0GF, i0,i1,i2)];
  const double AU0_i0p1_i1_i2 = in_gfs[IDX4(AU0GF, i0+1,i1,i2)];
  const double AU0_i0p2_i1_i2 = in_gfs[IDX4(AU0GF, i0+2,i1,i2)];
  const double AU0_i0_i1p1_i2 = in_gfs[IDX4(AU0GF, i0,i1+1,i2)];
  const double AU0_i0_i1p2_i2 = in_gfs[IDX4(AU0GF, i0,i1+2,i2)];
  const double AU0_i0_i1_i2p1 = in_gfs[IDX4(AU0GF, i0,i1,i2+1)];
  const double AU0_i0_i1_i2p2 = in_gfs[IDX4(AU0GF, i0,i1,i2+2)];
  const double AU1_i0_i1_i2m2 = in_gfs[IDX4(AU1GF, i0,i1,i2-2)];
  const double AU1_i0_i1_i2m1 = in_gfs[IDX4(AU1GF, i0,i1,i2-1)];
  const double AU1_i0_i1m2_i2 = in_gfs[IDX4(AU1GF, i0,i1-2,i2)];
  const double AU1_i0_i1m1_i2 = in_gfs[IDX4(AU1GF, i0,i1-1,i2)];
  const double AU1_i0m2_i1_i2 = in_gfs[IDX4(AU1GF, i0-2,i1,i2)];
  const double AU1_i0m1_i1_i2 = in_gfs[IDX4(AU1GF, i0-1,i1,i2)];
  const double AU1 = in_gfs[IDX4(AU1GF, i0,i1,i2)];
  const double AU1_i0p1_i1_i2 = in_gfs[IDX4(AU1GF, i0+1,i1,i2)];
  const double AU1_i0p2_i1_i2 = in_gfs[IDX4(AU1GF, i0+2,i1,i2)];
  const double AU1_i0_i1p1_i2 = in_gfs[IDX4(AU1GF, i0,i1+1,i2)];
  const double AU1_i0_i1p2_i2 = in_gfs[IDX4(AU1GF, i0,i1+2,i2)];
  const double AU1_i0_i1_i2p1 = in_gfs[IDX4(AU1GF, i0,i1,i2+1)];
  const double AU1_i0_i1_i2p2 = in_gfs[IDX4(AU1GF, i0,i1,i2+2)];
  const double AU2_i0_i1_i2m2 = in_gfs[IDX4(AU2GF, i0,i1,i2-2)];
  const double AU2_i0_i1_i2m1 = in_gfs[IDX4(AU2GF, i0,i1,i2-1)];
  const double AU2_i0_i1m2_i2 = in_gfs[IDX4(AU2GF, i0,i1-2,i2)];
  const double AU2_i0_i1m1_i2 = in_gfs[IDX4(AU2GF, i0,i1-1,i2)];
  const double AU2_i0m2_i1_i2 = in_gfs[IDX4(AU2GF, i0-2,i1,i2)];
  const double AU2_i0m1_i1_i2 = in_gfs[IDX4(AU2GF, i0-1,i1,i2)];
  const double AU2 = in_gfs[IDX4(AU2GF, i0,i1,i2)];
  const double AU2_i0p1_i1_i2 = in_gfs[IDX4(AU2GF, i0+1,i1,i2)];
  const double AU2_i0p2_i1_i2 = in_gfs[IDX4(AU2GF, i0+2,i1,i2)];
  const double AU2_i0_i1p1_i2 = in_gfs[IDX4(AU2GF, i0,i1+1,i2)];
  const double AU2_i0_i1p2_i2 = in_gfs[IDX4(AU2GF, i0,i1+2,i2)];
  const double AU2_i0_i1_i2p1 = in_gfs[IDX4(AU2GF, i0,i1,i2+1)];
  const double AU2_i0_i1_i2p2 = in_gfs[IDX4(AU2GF, i0,i1,i2+2)];
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
  const double FDPart1_0 = ((invdx0)*(invdx0));
  const double FDPart1_1 = AU0*FDPart1_Rational_m5_2;
  const double FDPart1_2 = ((invdx1)*(invdx1));
  const double FDPart1_3 = ((invdx2)*(invdx2));
  const double FDPart1_4 = AU1*FDPart1_Rational_m5_2;
  const double FDPart1_5 = AU2*FDPart1_Rational_m5_2;
  const double FDPart1_6 = FDPart1_Rational_m1_12*psi_i0p2_i1_i2;
  const double FDPart1_7 = FDPart1_Rational_m1_12*psi_i0_i1p2_i2;
  const double FDPart1_8 = FDPart1_Rational_m1_12*psi_i0_i1_i2p2;
  const double FDPart1_9 = FDPart1_Rational_m5_2*psi;
  const double AU_dDD000 = FDPart1_0*(AU0_i0m1_i1_i2*FDPart1_Rational_4_3 + AU0_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU0_i0p1_i1_i2*FDPart1_Rational_4_3 + AU0_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_1);
  const double AU_dDD011 = FDPart1_2*(AU0_i0_i1m1_i2*FDPart1_Rational_4_3 + AU0_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU0_i0_i1p1_i2*FDPart1_Rational_4_3 + AU0_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_1);
  const double AU_dDD022 = FDPart1_3*(AU0_i0_i1_i2m1*FDPart1_Rational_4_3 + AU0_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU0_i0_i1_i2p1*FDPart1_Rational_4_3 + AU0_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_1);
  const double AU_dDD100 = FDPart1_0*(AU1_i0m1_i1_i2*FDPart1_Rational_4_3 + AU1_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU1_i0p1_i1_i2*FDPart1_Rational_4_3 + AU1_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_4);
  const double AU_dDD111 = FDPart1_2*(AU1_i0_i1m1_i2*FDPart1_Rational_4_3 + AU1_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU1_i0_i1p1_i2*FDPart1_Rational_4_3 + AU1_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_4);
  const double AU_dDD122 = FDPart1_3*(AU1_i0_i1_i2m1*FDPart1_Rational_4_3 + AU1_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU1_i0_i1_i2p1*FDPart1_Rational_4_3 + AU1_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_4);
  const double AU_dDD200 = FDPart1_0*(AU2_i0m1_i1_i2*FDPart1_Rational_4_3 + AU2_i0m2_i1_i2*FDPart1_Rational_m1_12 + AU2_i0p1_i1_i2*FDPart1_Rational_4_3 + AU2_i0p2_i1_i2*FDPart1_Rational_m1_12 + FDPart1_5);
  const double AU_dDD211 = FDPart1_2*(AU2_i0_i1m1_i2*FDPart1_Rational_4_3 + AU2_i0_i1m2_i2*FDPart1_Rational_m1_12 + AU2_i0_i1p1_i2*FDPart1_Rational_4_3 + AU2_i0_i1p2_i2*FDPart1_Rational_m1_12 + FDPart1_5);
  const double AU_dDD222 = FDPart1_3*(AU2_i0_i1_i2m1*FDPart1_Rational_4_3 + AU2_i0_i1_i2m2*FDPart1_Rational_m1_12 + AU2_i0_i1_i2p1*FDPart1_Rational_4_3 + AU2_i0_i1_i2p2*FDPart1_Rational_m1_12 + FDPart1_5);
  const double Gamma_dD0 = invdx0*(FDPart1_Rational_1_12*Gamma_i0m2_i1_i2 + FDPart1_Rational_2_3*Gamma_i0p1_i1_i2 + FDPart1_Rational_m1_12*Gamma_i0p2_i1_i2 + FDPart1_Rational_m2_3*Gamma_i0m1_i1_i2);
  const double Gamma_dD1 = invdx1*(FDPart1_Rational_1_12*Gamma_i0_i1m2_i2 + FDPart1_Rational_2_3*Gamma_i0_i1p1_i2 + FDPart1_Rational_m1_12*Gamma_i0_i1p2_i2 + FDPart1_Rational_m2_3*Gamma_i0_i1m1_i2);
  const double Gamma_dD2 = invdx2*(FDPart1_Rational_1_12*Gamma_i0_i1_i2m2 + FDPart1_Rational_2_3*Gamma_i0_i1_i2p1 + FDPart1_Rational_m1_12*Gamma_i0_i1_i2p2 + FDPart1_Rational_m2_3*Gamma_i0_i1_i2m1);
  const double psi_dD0 = invdx0*(FDPart1_6 + FDPart1_Rational_1_12*psi_i0m2_i1_i2 + FDPart1_Rational_2_3*psi_i0p1_i1_i2 + FDPart1_Rational_m2_3*psi_i0m1_i1_i2);
  const double psi_dD1 = invdx1*(FDPart1_7 + FDPart1_Rational_1_12*psi_i0_i1m2_i2 + FDPart1_Rational_2_3*psi_i0_i1p1_i2 + FDPart1_Rational_m2_3*psi_i0_i1m1_i2);
  const double psi_dD2 = invdx2*(FDPart1_8 + FDPart1_Rational_1_12*psi_i0_i1_i2m2 + FDPart1_Rational_2_3*psi_i0_i1_i2p1 + FDPart1_Rational_m2_3*psi_i0_i1_i2m1);
  const double psi_dDD00 = FDPart1_0*(FDPart1_6 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0m1_i1_i2 + FDPart1_Rational_4_3*psi_i0p1_i1_i2 + FDPart1_Rational_m1_12*psi_i0m2_i1_i2);
  const double psi_dDD11 = FDPart1_2*(FDPart1_7 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1m1_i2 + FDPart1_Rational_4_3*psi_i0_i1p1_i2 + FDPart1_Rational_m1_12*psi_i0_i1m2_i2);
  const double psi_dDD22 = FDPart1_3*(FDPart1_8 + FDPart1_9 + FDPart1_Rational_4_3*psi_i0_i1_i2m1 + FDPart1_Rational_4_3*psi_i0_i1_i2p1 + FDPart1_Rational_m1_12*psi_i0_i1_i2m2);
  /* Reverse sweep: forward temporaries, then their adjoints in reverse order */
  const double cot_AU0 = cot_rhs_gfs[IDX4(AU0GF, i0, i1, i2)];
  const double cot_AU1 = cot_rhs_gfs[IDX4(AU1GF, i0, i1, i2)];
  const double cot_AU2 = cot_rhs_gfs[IDX4(AU2GF, i0, i1, i2)];
  const double cot_EU0 = cot_rhs_gfs[IDX4(EU0GF, i0, i1, i2)];
  const double cot_EU1 = cot_rhs_gfs[IDX4(EU1GF, i0, i1, i2)];
  const double cot_EU2 = cot_rhs_gfs[IDX4(EU2GF, i0, i1, i2)];
  const double cot_Gamma = cot_rhs_gfs[IDX4(GAMMAGF, i0, i1, i2)];
  const double cot_psi = cot_rhs_gfs[IDX4(PSIGF, i0, i1, i2)];
  vjp_G[IDX4(0, i0, i1, i2)] = -cot_EU0;
  vjp_G[IDX4(1, i0, i1, i2)] = -cot_EU0;
  vjp_G[IDX4(2, i0, i1, i2)] = -cot_EU0;
  vjp_G[IDX4(3, i0, i1, i2)] = -cot_EU1;
  vjp_G[IDX4(4, i0, i1, i2)] = -cot_EU1;
  vjp_G[IDX4(5, i0, i1, i2)] = -cot_EU1;
  vjp_G[IDX4(6, i0, i1, i2)] = -cot_EU2;
  vjp_G[IDX4(7, i0, i1, i2)] = -cot_EU2;
  vjp_G[IDX4(8, i0, i1, i2)] = -cot_EU2;
  vjp_G[IDX4(9, i0, i1, i2)] = -cot_AU0;
  vjp_G[IDX4(10, i0, i1, i2)] = -cot_AU1;
  vjp_G[IDX4(11, i0, i1, i2)] = -cot_AU2;
  vjp_G[IDX4(12, i0, i1, i2)] = -cot_psi;
  vjp_G[IDX4(13, i0, i1, i2)] = cot_EU0;
  vjp_G[IDX4(14, i0, i1, i2)] = cot_EU1;
  vjp_G[IDX4(15, i0, i1, i2)] = cot_EU2;
  vjp_G[IDX4(16, i0, i1, i2)] = -cot_AU0;
  vjp_G[IDX4(17, i0, i1, i2)] = -cot_AU1;
  vjp_G[IDX4(18, i0, i1, i2)] = -cot_AU2;
  vjp_G[IDX4(19, i0, i1, i2)] = -cot_Gamma;
  vjp_G[IDX4(20, i0, i1, i2)] = -cot_Gamma;
  vjp_G[IDX4(21, i0, i1, i2)] = -cot_Gamma;
  
}

extern "C" int rhs_eval_vjp_pointwise(const paramstruct *params, const double *in_gfs, const double *cot_rhs_gfs, double *vjp_G, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!in_gfs || !cot_rhs_gfs || !vjp_G) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(5, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  hipLaunchKernelGGL(rhs_eval_vjp_pointwise__gpu, grid, block, 0, stream, *params, in_gfs, cot_rhs_gfs, vjp_G);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}

/* VJP pass 2: transposed stencils of rhs_eval */
__global__ void __launch_bounds__(256) rhs_eval_vjp_transpose__gpu(const paramstruct params, const double *__restrict__ vjp_G, double *__restrict__ cot_in_gfs) {
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  
  NRPY_BLOCK_COORDS(Nxx_plus_2NGHOSTS0, Nxx_plus_2NGHOSTS1, Nxx_plus_2NGHOSTS2);
  const int i0 = 0 + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = 0 + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = 0 + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx_plus_2NGHOSTS0 || i1 >= Nxx_plus_2NGHOSTS1 || i2 >= Nxx_plus_2NGHOSTS2) return;
  cot_in_gfs[IDX4(AU0GF, i0, i1, i2)] = ((invdx0)*(invdx0))*((-1.0/12.0)*VJP_G_AT(0, 2, 0, 0) + (4.0/3.0)*VJP_G_AT(0, 1, 0, 0) + (-5.0/2.0)*VJP_G_AT(0, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(0, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(0, -2, 0, 0)) +
      ((invdx1)*(invdx1))*((-1.0/12.0)*VJP_G_AT(1, 0, 2, 0) + (4.0/3.0)*VJP_G_AT(1, 0, 1, 0) + (-5.0/2.0)*VJP_G_AT(1, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(1, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(1, 0, -2, 0)) +
      ((invdx2)*(invdx2))*((-1.0/12.0)*VJP_G_AT(2, 0, 0, 2) + (4.0/3.0)*VJP_G_AT(2, 0, 0, 1) + (-5.0/2.0)*VJP_G_AT(2, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(2, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(2, 0, 0, -2));
  cot_in_gfs[IDX4(AU1GF, i0, i1, i2)] = ((invdx0)*(invdx0))*((-1.0/12.0)*VJP_G_AT(3, 2, 0, 0) + (4.0/3.0)*VJP_G_AT(3, 1, 0, 0) + (-5.0/2.0)*VJP_G_AT(3, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(3, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(3, -2, 0, 0)) +
      ((invdx1)*(invdx1))*((-1.0/12.0)*VJP_G_AT(4, 0, 2, 0) + (4.0/3.0)*VJP_G_AT(4, 0, 1, 0) + (-5.0/2.0)*VJP_G_AT(4, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(4, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(4, 0, -2, 0)) +
      ((invdx2)*(invdx2))*((-1.0/12.0)*VJP_G_AT(5, 0, 0, 2) + (4.0/3.0)*VJP_G_AT(5, 0, 0, 1) + (-5.0/2.0)*VJP_G_AT(5, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(5, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(5, 0, 0, -2));
  cot_in_gfs[IDX4(AU2GF, i0, i1, i2)] = ((invdx0)*(invdx0))*((-1.0/12.0)*VJP_G_AT(6, 2, 0, 0) + (4.0/3.0)*VJP_G_AT(6, 1, 0, 0) + (-5.0/2.0)*VJP_G_AT(6, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(6, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(6, -2, 0, 0)) +
      ((invdx1)*(invdx1))*((-1.0/12.0)*VJP_G_AT(7, 0, 2, 0) + (4.0/3.0)*VJP_G_AT(7, 0, 1, 0) + (-5.0/2.0)*VJP_G_AT(7, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(7, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(7, 0, -2, 0)) +
      ((invdx2)*(invdx2))*((-1.0/12.0)*VJP_G_AT(8, 0, 0, 2) + (4.0/3.0)*VJP_G_AT(8, 0, 0, 1) + (-5.0/2.0)*VJP_G_AT(8, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(8, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(8, 0, 0, -2));
  cot_in_gfs[IDX4(EU0GF, i0, i1, i2)] = VJP_G_AT(9, 0, 0, 0);
  cot_in_gfs[IDX4(EU1GF, i0, i1, i2)] = VJP_G_AT(10, 0, 0, 0);
  cot_in_gfs[IDX4(EU2GF, i0, i1, i2)] = VJP_G_AT(11, 0, 0, 0);
  cot_in_gfs[IDX4(GAMMAGF, i0, i1, i2)] = VJP_G_AT(12, 0, 0, 0) +
      invdx0*((1.0/12.0)*VJP_G_AT(13, 2, 0, 0) + (-2.0/3.0)*VJP_G_AT(13, 1, 0, 0) + (2.0/3.0)*VJP_G_AT(13, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(13, -2, 0, 0)) +
      invdx1*((1.0/12.0)*VJP_G_AT(14, 0, 2, 0) + (-2.0/3.0)*VJP_G_AT(14, 0, 1, 0) + (2.0/3.0)*VJP_G_AT(14, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(14, 0, -2, 0)) +
      invdx2*((1.0/12.0)*VJP_G_AT(15, 0, 0, 2) + (-2.0/3.0)*VJP_G_AT(15, 0, 0, 1) + (2.0/3.0)*VJP_G_AT(15, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(15, 0, 0, -2));
  cot_in_gfs[IDX4(PSIGF, i0, i1, i2)] = invdx0*((1.0/12.0)*VJP_G_AT(16, 2, 0, 0) + (-2.0/3.0)*VJP_G_AT(16, 1, 0, 0) + (2.0/3.0)*VJP_G_AT(16, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(16, -2, 0, 0)) +
      invdx1*((1.0/12.0)*VJP_G_AT(17, 0, 2, 0) + (-2.0/3.0)*VJP_G_AT(17, 0, 1, 0) + (2.0/3.0)*VJP_G_AT(17, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(17, 0, -2, 0)) +
      invdx2*((1.0/12.0)*VJP_G_AT(18, 0, 0, 2) + (-2.0/3.0)*VJP_G_AT(18, 0, 0, 1) + (2.0/3.0)*VJP_G_AT(18, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(18, 0, 0, -2)) +
      ((invdx0)*(invdx0))*((-1.0/12.0)*VJP_G_AT(19, 2, 0, 0) + (4.0/3.0)*VJP_G_AT(19, 1, 0, 0) + (-5.0/2.0)*VJP_G_AT(19, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(19, -1, 0, 0) + (-1.0/12.0)*VJP_G_AT(19, -2, 0, 0)) +
      ((invdx1)*(invdx1))*((-1.0/12.0)*VJP_G_AT(20, 0, 2, 0) + (4.0/3.0)*VJP_G_AT(20, 0, 1, 0) + (-5.0/2.0)*VJP_G_AT(20, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(20, 0, -1, 0) + (-1.0/12.0)*VJP_G_AT(20, 0, -2, 0)) +
      ((invdx2)*(invdx2))*((-1.0/12.0)*VJP_G_AT(21, 0, 0, 2) + (4.0/3.0)*VJP_G_AT(21, 0, 0, 1) + (-5.0/2.0)*VJP_G_AT(21, 0, 0, 0) + (4.0/3.0)*VJP_G_AT(21, 0, 0, -1) + (-1.0/12.0)*VJP_G_AT(21, 0, 0, -2));
  
}

extern "C" int rhs_eval_vjp_transpose(const paramstruct *params, const double *vjp_G, double *cot_in_gfs, hipStream_t stream) {
  if (!params) return NRPY_ERR_NULL;
  if (!vjp_G || !cot_in_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const dim3 block = nrpy_block(6, 64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx_plus_2NGHOSTS0, params->Nxx_plus_2NGHOSTS1, params->Nxx_plus_2NGHOSTS2));
  hipLaunchKernelGGL(rhs_eval_vjp_transpose__gpu, grid, block, 0, stream, *params, vjp_G, cot_in_gfs);
  return hipGetLastError() == hipSuccess ? 0 : NRPY_ERR_LAUNCH;
}
/* Vector-Jacobian product of rhs_eval: given cot_rhs_gfs (cotangent of the RHS at interior
 * points), writes the cotangent of every input gridfunction at every point into
 * cot_in_gfs (evolved) and cot_auxevol_gfs (auxiliary evolved; may be NULL when the
 * system has none). vjp_G is caller-allocated scratch of 22 gridfunctions. Gridfunctions
 * of in_gfs that the RHS does not read get no write: clear cot_in_gfs first. */
extern "C" int rhs_eval_vjp(const paramstruct *params, const double *auxevol_gfs, const double *in_gfs,
    const double *cot_rhs_gfs, double *vjp_G, double *cot_in_gfs, double *cot_auxevol_gfs,
    hipStream_t stream) {
  int rc;
  (void)auxevol_gfs;
  (void)cot_auxevol_gfs;
  if ((rc = rhs_eval_vjp_pointwise(params, in_gfs, cot_rhs_gfs, vjp_G, stream))) return rc;
  if ((rc = rhs_eval_vjp_transpose(params, vjp_G, cot_in_gfs, stream))) return rc;
  return NRPY_OK;
}

// One RK4 step (MoLtimestepping/C_Code_Generation.py:266-329 for RK4): four substeps, each
// [Ricci] -> RHS + update at interior points -> ghost fill -> [det(gammabar) enforcement].
extern "C" int MoL_step_forward_in_time(const rfm_struct *rfmstruct, const paramstruct *params, const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, double *auxevol_gfs, const double dt, hipStream_t stream) {
  if (!rfmstruct || !params || !bcstruct || !y_n_gfs || !k_odd_gfs || !k_even_gfs ||
      !y_nplus1_running_total_gfs) return NRPY_ERR_NULL;
  int rc;
  nrpy_gf_parity_args gfp;  // the boundary struct is the grid's: checked before the first substep
  memset(&gfp, 0, sizeof(gfp));
  if ((rc = nrpy_bc_check(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, y_n_gfs, &gfp))) return rc;
  /* substep 0: y_n_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep(0, rfmstruct, params, auxevol_gfs, y_n_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  /* substep 1: k_odd_gfs -> k_even_gfs */
  if ((rc = rhs_eval_rk4_substep_edge(1, rfmstruct, params, auxevol_gfs, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, dt, stream))) return rc;
  /* substep 2: k_even_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep_edge(2, rfmstruct, params, auxevol_gfs, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  /* substep 3: k_odd_gfs -> y_n_gfs */
  if ((rc = rhs_eval_rk4_substep_edge(3, rfmstruct, params, auxevol_gfs, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, dt, stream))) return rc;
  if ((rc = apply_bcs_curvilinear_composed(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, y_n_gfs, stream))) return rc;
  return NRPY_OK;
}

struct MoL_graph {
  hipGraph_t graph;
  hipGraphExec_t exec;
};
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
  for (int n = 0; n < nsteps; n++)
    if (hipGraphLaunch(g->exec, stream) != hipSuccess) return NRPY_ERR_LAUNCH;
  return NRPY_OK;
}
extern "C" void MoL_graph_free(MoL_graph *g) {
  if (!g) return;
  (void)hipGraphExecDestroy(g->exec);
  (void)hipGraphDestroy(g->graph);
  delete g;
}


// A cotangent array, 0 outside the interior; the load stays in range as VJP_G_AT's does.
#define VJP_COT_AT(gf, o0, o1, o2)                                                                  \
  nrpy_vjp_select((i0) + (o0) >= NGHOSTS && (i0) + (o0) < Nxx0 + NGHOSTS && (i1) + (o1) >= NGHOSTS && \
                      (i1) + (o1) < Nxx1 + NGHOSTS && (i2) + (o2) >= NGHOSTS &&                     \
                      (i2) + (o2) < Nxx2 + NGHOSTS,                                                 \
                  cot[IDX4(gf, (i0) + (o0), (i1) + (o1), (i2) + (o2))])
// One stage of the RK4 step adjoint: w = (transposed ghost fill and stencils of rhs_eval) cot, times
// scale in stage 3 (whose kbar is scale L). Bound by its arrays: five read or written per gridfunction
// (three in stages 3 and 0) besides the stencil's neighbours, which the caches hold. Scalar wave at
// 128^3: 30 us a stage; slots, transposed stencils, ghost transpose, clearing and the update as
// launches of their own took 18 + 35 + 12 + 6 + 26 us. One point a lane and 64 x 4 tiles, as the
// forward substep: neighbours along x in the same cache lines.
template <int S>
__global__ void __launch_bounds__(256) rhs_eval_vjp_rk4_stage__gpu(const paramstruct params, const double *cot, const double *L, const double *acc_in, double *acc_out, double *__restrict__ kbar_out, const double scale, const double a, const double b) {
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const int Nxx0 = params.Nxx0;
  const int Nxx1 = params.Nxx1;
  const int Nxx2 = params.Nxx2;
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  NRPY_BLOCK_COORDS(Nxx0, Nxx1, Nxx2);
  const int i0 = NGHOSTS + nrpy_bx*(int)blockDim.x + (int)threadIdx.x;
  const int i1 = NGHOSTS + nrpy_by*(int)blockDim.y + (int)threadIdx.y;
  const int i2 = NGHOSTS + nrpy_bz*(int)blockDim.z + (int)threadIdx.z;
  if (i0 >= Nxx0 + NGHOSTS || i1 >= Nxx1 + NGHOSTS || i2 >= Nxx2 + NGHOSTS) return;
  const double cot_EU0_i0p2 = VJP_COT_AT(EU0GF, 2, 0, 0);
  const double cot_EU0_i0p1 = VJP_COT_AT(EU0GF, 1, 0, 0);
  const double cot_EU0 = VJP_COT_AT(EU0GF, 0, 0, 0);
  const double cot_EU0_i0m1 = VJP_COT_AT(EU0GF, -1, 0, 0);
  const double cot_EU0_i0m2 = VJP_COT_AT(EU0GF, -2, 0, 0);
  const double cot_EU0_i1p2 = VJP_COT_AT(EU0GF, 0, 2, 0);
  const double cot_EU0_i1p1 = VJP_COT_AT(EU0GF, 0, 1, 0);
  const double cot_EU0_i1m1 = VJP_COT_AT(EU0GF, 0, -1, 0);
  const double cot_EU0_i1m2 = VJP_COT_AT(EU0GF, 0, -2, 0);
  const double cot_EU0_i2p2 = VJP_COT_AT(EU0GF, 0, 0, 2);
  const double cot_EU0_i2p1 = VJP_COT_AT(EU0GF, 0, 0, 1);
  const double cot_EU0_i2m1 = VJP_COT_AT(EU0GF, 0, 0, -1);
  const double cot_EU0_i2m2 = VJP_COT_AT(EU0GF, 0, 0, -2);
  const double cot_EU1_i0p2 = VJP_COT_AT(EU1GF, 2, 0, 0);
  const double cot_EU1_i0p1 = VJP_COT_AT(EU1GF, 1, 0, 0);
  const double cot_EU1 = VJP_COT_AT(EU1GF, 0, 0, 0);
  const double cot_EU1_i0m1 = VJP_COT_AT(EU1GF, -1, 0, 0);
  const double cot_EU1_i0m2 = VJP_COT_AT(EU1GF, -2, 0, 0);
  const double cot_EU1_i1p2 = VJP_COT_AT(EU1GF, 0, 2, 0);
  const double cot_EU1_i1p1 = VJP_COT_AT(EU1GF, 0, 1, 0);
  const double cot_EU1_i1m1 = VJP_COT_AT(EU1GF, 0, -1, 0);
  const double cot_EU1_i1m2 = VJP_COT_AT(EU1GF, 0, -2, 0);
  const double cot_EU1_i2p2 = VJP_COT_AT(EU1GF, 0, 0, 2);
  const double cot_EU1_i2p1 = VJP_COT_AT(EU1GF, 0, 0, 1);
  const double cot_EU1_i2m1 = VJP_COT_AT(EU1GF, 0, 0, -1);
  const double cot_EU1_i2m2 = VJP_COT_AT(EU1GF, 0, 0, -2);
  const double cot_EU2_i0p2 = VJP_COT_AT(EU2GF, 2, 0, 0);
  const double cot_EU2_i0p1 = VJP_COT_AT(EU2GF, 1, 0, 0);
  const double cot_EU2 = VJP_COT_AT(EU2GF, 0, 0, 0);
  const double cot_EU2_i0m1 = VJP_COT_AT(EU2GF, -1, 0, 0);
  const double cot_EU2_i0m2 = VJP_COT_AT(EU2GF, -2, 0, 0);
  const double cot_EU2_i1p2 = VJP_COT_AT(EU2GF, 0, 2, 0);
  const double cot_EU2_i1p1 = VJP_COT_AT(EU2GF, 0, 1, 0);
  const double cot_EU2_i1m1 = VJP_COT_AT(EU2GF, 0, -1, 0);
  const double cot_EU2_i1m2 = VJP_COT_AT(EU2GF, 0, -2, 0);
  const double cot_EU2_i2p2 = VJP_COT_AT(EU2GF, 0, 0, 2);
  const double cot_EU2_i2p1 = VJP_COT_AT(EU2GF, 0, 0, 1);
  const double cot_EU2_i2m1 = VJP_COT_AT(EU2GF, 0, 0, -1);
  const double cot_EU2_i2m2 = VJP_COT_AT(EU2GF, 0, 0, -2);
  const double cot_AU0 = VJP_COT_AT(AU0GF, 0, 0, 0);
  const double cot_AU1 = VJP_COT_AT(AU1GF, 0, 0, 0);
  const double cot_AU2 = VJP_COT_AT(AU2GF, 0, 0, 0);
  const double cot_psi = VJP_COT_AT(PSIGF, 0, 0, 0);
  const double cot_AU0_i0p2 = VJP_COT_AT(AU0GF, 2, 0, 0);
  const double cot_AU0_i0p1 = VJP_COT_AT(AU0GF, 1, 0, 0);
  const double cot_AU0_i0m1 = VJP_COT_AT(AU0GF, -1, 0, 0);
  const double cot_AU0_i0m2 = VJP_COT_AT(AU0GF, -2, 0, 0);
  const double cot_AU1_i1p2 = VJP_COT_AT(AU1GF, 0, 2, 0);
  const double cot_AU1_i1p1 = VJP_COT_AT(AU1GF, 0, 1, 0);
  const double cot_AU1_i1m1 = VJP_COT_AT(AU1GF, 0, -1, 0);
  const double cot_AU1_i1m2 = VJP_COT_AT(AU1GF, 0, -2, 0);
  const double cot_AU2_i2p2 = VJP_COT_AT(AU2GF, 0, 0, 2);
  const double cot_AU2_i2p1 = VJP_COT_AT(AU2GF, 0, 0, 1);
  const double cot_AU2_i2m1 = VJP_COT_AT(AU2GF, 0, 0, -1);
  const double cot_AU2_i2m2 = VJP_COT_AT(AU2GF, 0, 0, -2);
  const double cot_Gamma_i0p2 = VJP_COT_AT(GAMMAGF, 2, 0, 0);
  const double cot_Gamma_i0p1 = VJP_COT_AT(GAMMAGF, 1, 0, 0);
  const double cot_Gamma = VJP_COT_AT(GAMMAGF, 0, 0, 0);
  const double cot_Gamma_i0m1 = VJP_COT_AT(GAMMAGF, -1, 0, 0);
  const double cot_Gamma_i0m2 = VJP_COT_AT(GAMMAGF, -2, 0, 0);
  const double cot_Gamma_i1p2 = VJP_COT_AT(GAMMAGF, 0, 2, 0);
  const double cot_Gamma_i1p1 = VJP_COT_AT(GAMMAGF, 0, 1, 0);
  const double cot_Gamma_i1m1 = VJP_COT_AT(GAMMAGF, 0, -1, 0);
  const double cot_Gamma_i1m2 = VJP_COT_AT(GAMMAGF, 0, -2, 0);
  const double cot_Gamma_i2p2 = VJP_COT_AT(GAMMAGF, 0, 0, 2);
  const double cot_Gamma_i2p1 = VJP_COT_AT(GAMMAGF, 0, 0, 1);
  const double cot_Gamma_i2m1 = VJP_COT_AT(GAMMAGF, 0, 0, -1);
  const double cot_Gamma_i2m2 = VJP_COT_AT(GAMMAGF, 0, 0, -2);
  double t_EU0_dDD00 = (-1.0/12.0)*cot_EU0_i0p2 + (4.0/3.0)*cot_EU0_i0p1 + (-5.0/2.0)*cot_EU0 + (4.0/3.0)*cot_EU0_i0m1 + (-1.0/12.0)*cot_EU0_i0m2;
  if (i0 == NGHOSTS + 0) t_EU0_dDD00 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i0p1;
  if (i0 == NGHOSTS + 1) t_EU0_dDD00 += (-10.0/3.0)*cot_EU0_i0m1 + (1.0/4.0)*cot_EU0;
  if (i0 == NGHOSTS + 2) t_EU0_dDD00 += (13.0/12.0)*cot_EU0_i0m2 + (-1.0/12.0)*cot_EU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_EU0_dDD00 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_EU0_dDD00 += (-10.0/3.0)*cot_EU0_i0p1 + (1.0/4.0)*cot_EU0;
  if (i0 == Nxx0 + NGHOSTS - 3) t_EU0_dDD00 += (13.0/12.0)*cot_EU0_i0p2 + (-1.0/12.0)*cot_EU0_i0p1;
  double t_EU0_dDD11 = (-1.0/12.0)*cot_EU0_i1p2 + (4.0/3.0)*cot_EU0_i1p1 + (-5.0/2.0)*cot_EU0 + (4.0/3.0)*cot_EU0_i1m1 + (-1.0/12.0)*cot_EU0_i1m2;
  if (i1 == NGHOSTS + 0) t_EU0_dDD11 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i1p1;
  if (i1 == NGHOSTS + 1) t_EU0_dDD11 += (-10.0/3.0)*cot_EU0_i1m1 + (1.0/4.0)*cot_EU0;
  if (i1 == NGHOSTS + 2) t_EU0_dDD11 += (13.0/12.0)*cot_EU0_i1m2 + (-1.0/12.0)*cot_EU0_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_EU0_dDD11 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_EU0_dDD11 += (-10.0/3.0)*cot_EU0_i1p1 + (1.0/4.0)*cot_EU0;
  if (i1 == Nxx1 + NGHOSTS - 3) t_EU0_dDD11 += (13.0/12.0)*cot_EU0_i1p2 + (-1.0/12.0)*cot_EU0_i1p1;
  double t_EU0_dDD22 = (-1.0/12.0)*cot_EU0_i2p2 + (4.0/3.0)*cot_EU0_i2p1 + (-5.0/2.0)*cot_EU0 + (4.0/3.0)*cot_EU0_i2m1 + (-1.0/12.0)*cot_EU0_i2m2;
  if (i2 == NGHOSTS + 0) t_EU0_dDD22 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i2p1;
  if (i2 == NGHOSTS + 1) t_EU0_dDD22 += (-10.0/3.0)*cot_EU0_i2m1 + (1.0/4.0)*cot_EU0;
  if (i2 == NGHOSTS + 2) t_EU0_dDD22 += (13.0/12.0)*cot_EU0_i2m2 + (-1.0/12.0)*cot_EU0_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_EU0_dDD22 += (7.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_EU0_dDD22 += (-10.0/3.0)*cot_EU0_i2p1 + (1.0/4.0)*cot_EU0;
  if (i2 == Nxx2 + NGHOSTS - 3) t_EU0_dDD22 += (13.0/12.0)*cot_EU0_i2p2 + (-1.0/12.0)*cot_EU0_i2p1;
  double t_EU1_dDD00 = (-1.0/12.0)*cot_EU1_i0p2 + (4.0/3.0)*cot_EU1_i0p1 + (-5.0/2.0)*cot_EU1 + (4.0/3.0)*cot_EU1_i0m1 + (-1.0/12.0)*cot_EU1_i0m2;
  if (i0 == NGHOSTS + 0) t_EU1_dDD00 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i0p1;
  if (i0 == NGHOSTS + 1) t_EU1_dDD00 += (-10.0/3.0)*cot_EU1_i0m1 + (1.0/4.0)*cot_EU1;
  if (i0 == NGHOSTS + 2) t_EU1_dDD00 += (13.0/12.0)*cot_EU1_i0m2 + (-1.0/12.0)*cot_EU1_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_EU1_dDD00 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_EU1_dDD00 += (-10.0/3.0)*cot_EU1_i0p1 + (1.0/4.0)*cot_EU1;
  if (i0 == Nxx0 + NGHOSTS - 3) t_EU1_dDD00 += (13.0/12.0)*cot_EU1_i0p2 + (-1.0/12.0)*cot_EU1_i0p1;
  double t_EU1_dDD11 = (-1.0/12.0)*cot_EU1_i1p2 + (4.0/3.0)*cot_EU1_i1p1 + (-5.0/2.0)*cot_EU1 + (4.0/3.0)*cot_EU1_i1m1 + (-1.0/12.0)*cot_EU1_i1m2;
  if (i1 == NGHOSTS + 0) t_EU1_dDD11 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i1p1;
  if (i1 == NGHOSTS + 1) t_EU1_dDD11 += (-10.0/3.0)*cot_EU1_i1m1 + (1.0/4.0)*cot_EU1;
  if (i1 == NGHOSTS + 2) t_EU1_dDD11 += (13.0/12.0)*cot_EU1_i1m2 + (-1.0/12.0)*cot_EU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_EU1_dDD11 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_EU1_dDD11 += (-10.0/3.0)*cot_EU1_i1p1 + (1.0/4.0)*cot_EU1;
  if (i1 == Nxx1 + NGHOSTS - 3) t_EU1_dDD11 += (13.0/12.0)*cot_EU1_i1p2 + (-1.0/12.0)*cot_EU1_i1p1;
  double t_EU1_dDD22 = (-1.0/12.0)*cot_EU1_i2p2 + (4.0/3.0)*cot_EU1_i2p1 + (-5.0/2.0)*cot_EU1 + (4.0/3.0)*cot_EU1_i2m1 + (-1.0/12.0)*cot_EU1_i2m2;
  if (i2 == NGHOSTS + 0) t_EU1_dDD22 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i2p1;
  if (i2 == NGHOSTS + 1) t_EU1_dDD22 += (-10.0/3.0)*cot_EU1_i2m1 + (1.0/4.0)*cot_EU1;
  if (i2 == NGHOSTS + 2) t_EU1_dDD22 += (13.0/12.0)*cot_EU1_i2m2 + (-1.0/12.0)*cot_EU1_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_EU1_dDD22 += (7.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_EU1_dDD22 += (-10.0/3.0)*cot_EU1_i2p1 + (1.0/4.0)*cot_EU1;
  if (i2 == Nxx2 + NGHOSTS - 3) t_EU1_dDD22 += (13.0/12.0)*cot_EU1_i2p2 + (-1.0/12.0)*cot_EU1_i2p1;
  double t_EU2_dDD00 = (-1.0/12.0)*cot_EU2_i0p2 + (4.0/3.0)*cot_EU2_i0p1 + (-5.0/2.0)*cot_EU2 + (4.0/3.0)*cot_EU2_i0m1 + (-1.0/12.0)*cot_EU2_i0m2;
  if (i0 == NGHOSTS + 0) t_EU2_dDD00 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i0p1;
  if (i0 == NGHOSTS + 1) t_EU2_dDD00 += (-10.0/3.0)*cot_EU2_i0m1 + (1.0/4.0)*cot_EU2;
  if (i0 == NGHOSTS + 2) t_EU2_dDD00 += (13.0/12.0)*cot_EU2_i0m2 + (-1.0/12.0)*cot_EU2_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_EU2_dDD00 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_EU2_dDD00 += (-10.0/3.0)*cot_EU2_i0p1 + (1.0/4.0)*cot_EU2;
  if (i0 == Nxx0 + NGHOSTS - 3) t_EU2_dDD00 += (13.0/12.0)*cot_EU2_i0p2 + (-1.0/12.0)*cot_EU2_i0p1;
  double t_EU2_dDD11 = (-1.0/12.0)*cot_EU2_i1p2 + (4.0/3.0)*cot_EU2_i1p1 + (-5.0/2.0)*cot_EU2 + (4.0/3.0)*cot_EU2_i1m1 + (-1.0/12.0)*cot_EU2_i1m2;
  if (i1 == NGHOSTS + 0) t_EU2_dDD11 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i1p1;
  if (i1 == NGHOSTS + 1) t_EU2_dDD11 += (-10.0/3.0)*cot_EU2_i1m1 + (1.0/4.0)*cot_EU2;
  if (i1 == NGHOSTS + 2) t_EU2_dDD11 += (13.0/12.0)*cot_EU2_i1m2 + (-1.0/12.0)*cot_EU2_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_EU2_dDD11 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_EU2_dDD11 += (-10.0/3.0)*cot_EU2_i1p1 + (1.0/4.0)*cot_EU2;
  if (i1 == Nxx1 + NGHOSTS - 3) t_EU2_dDD11 += (13.0/12.0)*cot_EU2_i1p2 + (-1.0/12.0)*cot_EU2_i1p1;
  double t_EU2_dDD22 = (-1.0/12.0)*cot_EU2_i2p2 + (4.0/3.0)*cot_EU2_i2p1 + (-5.0/2.0)*cot_EU2 + (4.0/3.0)*cot_EU2_i2m1 + (-1.0/12.0)*cot_EU2_i2m2;
  if (i2 == NGHOSTS + 0) t_EU2_dDD22 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i2p1;
  if (i2 == NGHOSTS + 1) t_EU2_dDD22 += (-10.0/3.0)*cot_EU2_i2m1 + (1.0/4.0)*cot_EU2;
  if (i2 == NGHOSTS + 2) t_EU2_dDD22 += (13.0/12.0)*cot_EU2_i2m2 + (-1.0/12.0)*cot_EU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_EU2_dDD22 += (7.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_EU2_dDD22 += (-10.0/3.0)*cot_EU2_i2p1 + (1.0/4.0)*cot_EU2;
  if (i2 == Nxx2 + NGHOSTS - 3) t_EU2_dDD22 += (13.0/12.0)*cot_EU2_i2p2 + (-1.0/12.0)*cot_EU2_i2p1;
  double t_EU0_dD0 = (1.0/12.0)*cot_EU0_i0p2 + (-2.0/3.0)*cot_EU0_i0p1 + (2.0/3.0)*cot_EU0_i0m1 + (-1.0/12.0)*cot_EU0_i0m2;
  if (i0 == NGHOSTS + 0) t_EU0_dD0 += (-3.0/2.0)*cot_EU0 + (1.0/4.0)*cot_EU0_i0p1;
  if (i0 == NGHOSTS + 1) t_EU0_dD0 += (4.0/3.0)*cot_EU0_i0m1 + (-1.0/4.0)*cot_EU0;
  if (i0 == NGHOSTS + 2) t_EU0_dD0 += (-5.0/12.0)*cot_EU0_i0m2 + (1.0/12.0)*cot_EU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_EU0_dD0 += (3.0/2.0)*cot_EU0 + (-1.0/4.0)*cot_EU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_EU0_dD0 += (-4.0/3.0)*cot_EU0_i0p1 + (1.0/4.0)*cot_EU0;
  if (i0 == Nxx0 + NGHOSTS - 3) t_EU0_dD0 += (5.0/12.0)*cot_EU0_i0p2 + (-1.0/12.0)*cot_EU0_i0p1;
  double t_EU1_dD1 = (1.0/12.0)*cot_EU1_i1p2 + (-2.0/3.0)*cot_EU1_i1p1 + (2.0/3.0)*cot_EU1_i1m1 + (-1.0/12.0)*cot_EU1_i1m2;
  if (i1 == NGHOSTS + 0) t_EU1_dD1 += (-3.0/2.0)*cot_EU1 + (1.0/4.0)*cot_EU1_i1p1;
  if (i1 == NGHOSTS + 1) t_EU1_dD1 += (4.0/3.0)*cot_EU1_i1m1 + (-1.0/4.0)*cot_EU1;
  if (i1 == NGHOSTS + 2) t_EU1_dD1 += (-5.0/12.0)*cot_EU1_i1m2 + (1.0/12.0)*cot_EU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_EU1_dD1 += (3.0/2.0)*cot_EU1 + (-1.0/4.0)*cot_EU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_EU1_dD1 += (-4.0/3.0)*cot_EU1_i1p1 + (1.0/4.0)*cot_EU1;
  if (i1 == Nxx1 + NGHOSTS - 3) t_EU1_dD1 += (5.0/12.0)*cot_EU1_i1p2 + (-1.0/12.0)*cot_EU1_i1p1;
  double t_EU2_dD2 = (1.0/12.0)*cot_EU2_i2p2 + (-2.0/3.0)*cot_EU2_i2p1 + (2.0/3.0)*cot_EU2_i2m1 + (-1.0/12.0)*cot_EU2_i2m2;
  if (i2 == NGHOSTS + 0) t_EU2_dD2 += (-3.0/2.0)*cot_EU2 + (1.0/4.0)*cot_EU2_i2p1;
  if (i2 == NGHOSTS + 1) t_EU2_dD2 += (4.0/3.0)*cot_EU2_i2m1 + (-1.0/4.0)*cot_EU2;
  if (i2 == NGHOSTS + 2) t_EU2_dD2 += (-5.0/12.0)*cot_EU2_i2m2 + (1.0/12.0)*cot_EU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_EU2_dD2 += (3.0/2.0)*cot_EU2 + (-1.0/4.0)*cot_EU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_EU2_dD2 += (-4.0/3.0)*cot_EU2_i2p1 + (1.0/4.0)*cot_EU2;
  if (i2 == Nxx2 + NGHOSTS - 3) t_EU2_dD2 += (5.0/12.0)*cot_EU2_i2p2 + (-1.0/12.0)*cot_EU2_i2p1;
  double t_AU0_dD0 = (1.0/12.0)*cot_AU0_i0p2 + (-2.0/3.0)*cot_AU0_i0p1 + (2.0/3.0)*cot_AU0_i0m1 + (-1.0/12.0)*cot_AU0_i0m2;
  if (i0 == NGHOSTS + 0) t_AU0_dD0 += (-3.0/2.0)*cot_AU0 + (1.0/4.0)*cot_AU0_i0p1;
  if (i0 == NGHOSTS + 1) t_AU0_dD0 += (4.0/3.0)*cot_AU0_i0m1 + (-1.0/4.0)*cot_AU0;
  if (i0 == NGHOSTS + 2) t_AU0_dD0 += (-5.0/12.0)*cot_AU0_i0m2 + (1.0/12.0)*cot_AU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_AU0_dD0 += (3.0/2.0)*cot_AU0 + (-1.0/4.0)*cot_AU0_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_AU0_dD0 += (-4.0/3.0)*cot_AU0_i0p1 + (1.0/4.0)*cot_AU0;
  if (i0 == Nxx0 + NGHOSTS - 3) t_AU0_dD0 += (5.0/12.0)*cot_AU0_i0p2 + (-1.0/12.0)*cot_AU0_i0p1;
  double t_AU1_dD1 = (1.0/12.0)*cot_AU1_i1p2 + (-2.0/3.0)*cot_AU1_i1p1 + (2.0/3.0)*cot_AU1_i1m1 + (-1.0/12.0)*cot_AU1_i1m2;
  if (i1 == NGHOSTS + 0) t_AU1_dD1 += (-3.0/2.0)*cot_AU1 + (1.0/4.0)*cot_AU1_i1p1;
  if (i1 == NGHOSTS + 1) t_AU1_dD1 += (4.0/3.0)*cot_AU1_i1m1 + (-1.0/4.0)*cot_AU1;
  if (i1 == NGHOSTS + 2) t_AU1_dD1 += (-5.0/12.0)*cot_AU1_i1m2 + (1.0/12.0)*cot_AU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_AU1_dD1 += (3.0/2.0)*cot_AU1 + (-1.0/4.0)*cot_AU1_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_AU1_dD1 += (-4.0/3.0)*cot_AU1_i1p1 + (1.0/4.0)*cot_AU1;
  if (i1 == Nxx1 + NGHOSTS - 3) t_AU1_dD1 += (5.0/12.0)*cot_AU1_i1p2 + (-1.0/12.0)*cot_AU1_i1p1;
  double t_AU2_dD2 = (1.0/12.0)*cot_AU2_i2p2 + (-2.0/3.0)*cot_AU2_i2p1 + (2.0/3.0)*cot_AU2_i2m1 + (-1.0/12.0)*cot_AU2_i2m2;
  if (i2 == NGHOSTS + 0) t_AU2_dD2 += (-3.0/2.0)*cot_AU2 + (1.0/4.0)*cot_AU2_i2p1;
  if (i2 == NGHOSTS + 1) t_AU2_dD2 += (4.0/3.0)*cot_AU2_i2m1 + (-1.0/4.0)*cot_AU2;
  if (i2 == NGHOSTS + 2) t_AU2_dD2 += (-5.0/12.0)*cot_AU2_i2m2 + (1.0/12.0)*cot_AU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_AU2_dD2 += (3.0/2.0)*cot_AU2 + (-1.0/4.0)*cot_AU2_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_AU2_dD2 += (-4.0/3.0)*cot_AU2_i2p1 + (1.0/4.0)*cot_AU2;
  if (i2 == Nxx2 + NGHOSTS - 3) t_AU2_dD2 += (5.0/12.0)*cot_AU2_i2p2 + (-1.0/12.0)*cot_AU2_i2p1;
  double t_Gamma_dDD00 = (-1.0/12.0)*cot_Gamma_i0p2 + (4.0/3.0)*cot_Gamma_i0p1 + (-5.0/2.0)*cot_Gamma + (4.0/3.0)*cot_Gamma_i0m1 + (-1.0/12.0)*cot_Gamma_i0m2;
  if (i0 == NGHOSTS + 0) t_Gamma_dDD00 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i0p1;
  if (i0 == NGHOSTS + 1) t_Gamma_dDD00 += (-10.0/3.0)*cot_Gamma_i0m1 + (1.0/4.0)*cot_Gamma;
  if (i0 == NGHOSTS + 2) t_Gamma_dDD00 += (13.0/12.0)*cot_Gamma_i0m2 + (-1.0/12.0)*cot_Gamma_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 1) t_Gamma_dDD00 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i0m1;
  if (i0 == Nxx0 + NGHOSTS - 2) t_Gamma_dDD00 += (-10.0/3.0)*cot_Gamma_i0p1 + (1.0/4.0)*cot_Gamma;
  if (i0 == Nxx0 + NGHOSTS - 3) t_Gamma_dDD00 += (13.0/12.0)*cot_Gamma_i0p2 + (-1.0/12.0)*cot_Gamma_i0p1;
  double t_Gamma_dDD11 = (-1.0/12.0)*cot_Gamma_i1p2 + (4.0/3.0)*cot_Gamma_i1p1 + (-5.0/2.0)*cot_Gamma + (4.0/3.0)*cot_Gamma_i1m1 + (-1.0/12.0)*cot_Gamma_i1m2;
  if (i1 == NGHOSTS + 0) t_Gamma_dDD11 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i1p1;
  if (i1 == NGHOSTS + 1) t_Gamma_dDD11 += (-10.0/3.0)*cot_Gamma_i1m1 + (1.0/4.0)*cot_Gamma;
  if (i1 == NGHOSTS + 2) t_Gamma_dDD11 += (13.0/12.0)*cot_Gamma_i1m2 + (-1.0/12.0)*cot_Gamma_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 1) t_Gamma_dDD11 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i1m1;
  if (i1 == Nxx1 + NGHOSTS - 2) t_Gamma_dDD11 += (-10.0/3.0)*cot_Gamma_i1p1 + (1.0/4.0)*cot_Gamma;
  if (i1 == Nxx1 + NGHOSTS - 3) t_Gamma_dDD11 += (13.0/12.0)*cot_Gamma_i1p2 + (-1.0/12.0)*cot_Gamma_i1p1;
  double t_Gamma_dDD22 = (-1.0/12.0)*cot_Gamma_i2p2 + (4.0/3.0)*cot_Gamma_i2p1 + (-5.0/2.0)*cot_Gamma + (4.0/3.0)*cot_Gamma_i2m1 + (-1.0/12.0)*cot_Gamma_i2m2;
  if (i2 == NGHOSTS + 0) t_Gamma_dDD22 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i2p1;
  if (i2 == NGHOSTS + 1) t_Gamma_dDD22 += (-10.0/3.0)*cot_Gamma_i2m1 + (1.0/4.0)*cot_Gamma;
  if (i2 == NGHOSTS + 2) t_Gamma_dDD22 += (13.0/12.0)*cot_Gamma_i2m2 + (-1.0/12.0)*cot_Gamma_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 1) t_Gamma_dDD22 += (7.0/2.0)*cot_Gamma + (-1.0/4.0)*cot_Gamma_i2m1;
  if (i2 == Nxx2 + NGHOSTS - 2) t_Gamma_dDD22 += (-10.0/3.0)*cot_Gamma_i2p1 + (1.0/4.0)*cot_Gamma;
  if (i2 == Nxx2 + NGHOSTS - 3) t_Gamma_dDD22 += (13.0/12.0)*cot_Gamma_i2p2 + (-1.0/12.0)*cot_Gamma_i2p1;
  const double w_AU0 = -((invdx0)*(invdx0))*t_EU0_dDD00 + -((invdx1)*(invdx1))*t_EU0_dDD11 + -((invdx2)*(invdx2))*t_EU0_dDD22;
  const double w_AU1 = -((invdx0)*(invdx0))*t_EU1_dDD00 + -((invdx1)*(invdx1))*t_EU1_dDD11 + -((invdx2)*(invdx2))*t_EU1_dDD22;
  const double w_AU2 = -((invdx0)*(invdx0))*t_EU2_dDD00 + -((invdx1)*(invdx1))*t_EU2_dDD11 + -((invdx2)*(invdx2))*t_EU2_dDD22;
  const double w_EU0 = -1*cot_AU0;
  const double w_EU1 = -1*cot_AU1;
  const double w_EU2 = -1*cot_AU2;
  const double w_Gamma = -1*cot_psi + invdx0*t_EU0_dD0 + invdx1*t_EU1_dD1 + invdx2*t_EU2_dD2;
  const double w_psi = -invdx0*t_AU0_dD0 + -invdx1*t_AU1_dD1 + -invdx2*t_AU2_dD2 + -((invdx0)*(invdx0))*t_Gamma_dDD00 + -((invdx1)*(invdx1))*t_Gamma_dDD11 + -((invdx2)*(invdx2))*t_Gamma_dDD22;
  const double acc_AU0 = acc_in[IDX4(AU0GF, i0, i1, i2)], L_AU0 = S > 0 ? L[IDX4(AU0GF, i0, i1, i2)] : 0.0;
  const double acc_AU1 = acc_in[IDX4(AU1GF, i0, i1, i2)], L_AU1 = S > 0 ? L[IDX4(AU1GF, i0, i1, i2)] : 0.0;
  const double acc_AU2 = acc_in[IDX4(AU2GF, i0, i1, i2)], L_AU2 = S > 0 ? L[IDX4(AU2GF, i0, i1, i2)] : 0.0;
  const double acc_EU0 = acc_in[IDX4(EU0GF, i0, i1, i2)], L_EU0 = S > 0 ? L[IDX4(EU0GF, i0, i1, i2)] : 0.0;
  const double acc_EU1 = acc_in[IDX4(EU1GF, i0, i1, i2)], L_EU1 = S > 0 ? L[IDX4(EU1GF, i0, i1, i2)] : 0.0;
  const double acc_EU2 = acc_in[IDX4(EU2GF, i0, i1, i2)], L_EU2 = S > 0 ? L[IDX4(EU2GF, i0, i1, i2)] : 0.0;
  const double acc_Gamma = acc_in[IDX4(GAMMAGF, i0, i1, i2)], L_Gamma = S > 0 ? L[IDX4(GAMMAGF, i0, i1, i2)] : 0.0;
  const double acc_psi = acc_in[IDX4(PSIGF, i0, i1, i2)], L_psi = S > 0 ? L[IDX4(PSIGF, i0, i1, i2)] : 0.0;
  {
    const double w = S == 3 ? scale * w_AU0 : w_AU0;
    acc_out[IDX4(AU0GF, i0, i1, i2)] = acc_AU0 + w;
    if (S > 0) kbar_out[IDX4(AU0GF, i0, i1, i2)] = a * L_AU0 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_AU1 : w_AU1;
    acc_out[IDX4(AU1GF, i0, i1, i2)] = acc_AU1 + w;
    if (S > 0) kbar_out[IDX4(AU1GF, i0, i1, i2)] = a * L_AU1 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_AU2 : w_AU2;
    acc_out[IDX4(AU2GF, i0, i1, i2)] = acc_AU2 + w;
    if (S > 0) kbar_out[IDX4(AU2GF, i0, i1, i2)] = a * L_AU2 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_EU0 : w_EU0;
    acc_out[IDX4(EU0GF, i0, i1, i2)] = acc_EU0 + w;
    if (S > 0) kbar_out[IDX4(EU0GF, i0, i1, i2)] = a * L_EU0 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_EU1 : w_EU1;
    acc_out[IDX4(EU1GF, i0, i1, i2)] = acc_EU1 + w;
    if (S > 0) kbar_out[IDX4(EU1GF, i0, i1, i2)] = a * L_EU1 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_EU2 : w_EU2;
    acc_out[IDX4(EU2GF, i0, i1, i2)] = acc_EU2 + w;
    if (S > 0) kbar_out[IDX4(EU2GF, i0, i1, i2)] = a * L_EU2 + b * w;
  }
  {
    const double w = S == 3 ? scale * w_Gamma : w_Gamma;
    acc_out[IDX4(GAMMAGF, i0, i1, i2)] = acc_Gamma + w;
    if (S > 0) kbar_out[IDX4(GAMMAGF, i0, i1, i2)] = a * L_Gamma + b * w;
  }
  {
    const double w = S == 3 ? scale * w_psi : w_psi;
    acc_out[IDX4(PSIGF, i0, i1, i2)] = acc_psi + w;
    if (S > 0) kbar_out[IDX4(PSIGF, i0, i1, i2)] = a * L_psi + b * w;
  }
}
static int rhs_eval_vjp_rk4_stage(const int S, const paramstruct *params, const double *cot, const double *L, const double *acc_in, double *acc_out, double *kbar_out, const double scale, const double a, const double b, hipStream_t stream) {
  const dim3 block(64, 4, 1);
  const dim3 grid(nrpy_nblocks(block, params->Nxx0, params->Nxx1, params->Nxx2));
  switch (S) {
    case 0: hipLaunchKernelGGL(rhs_eval_vjp_rk4_stage__gpu<0>, grid, block, 0, stream, *params, cot, L, acc_in, acc_out, kbar_out, scale, a, b); break;
    case 1: hipLaunchKernelGGL(rhs_eval_vjp_rk4_stage__gpu<1>, grid, block, 0, stream, *params, cot, L, acc_in, acc_out, kbar_out, scale, a, b); break;
    case 2: hipLaunchKernelGGL(rhs_eval_vjp_rk4_stage__gpu<2>, grid, block, 0, stream, *params, cot, L, acc_in, acc_out, kbar_out, scale, a, b); break;
    case 3: hipLaunchKernelGGL(rhs_eval_vjp_rk4_stage__gpu<3>, grid, block, 0, stream, *params, cot, L, acc_in, acc_out, kbar_out, scale, a, b); break;
  }
  return hipGetLastError() == hipSuccess ? NRPY_OK : NRPY_ERR_LAUNCH;
}
// Adjoint of one RK4 step. On entry lambda_gfs holds the cotangent of y_{n+1} (interior points;
// ghost cotangents zero), y_n_gfs the state at the start of the step with its ghosts filled. On
// exit lambda_gfs holds the cotangent of y_n. U1, U2, U3, rt, acc, kbar, w are caller-allocated
// scratch arrays of NUM_EVOL_GFS gridfunctions; vjp_G has the rhs_eval_vjp slot count. (The
// right-hand side is linear: of them only acc, kbar and w are used, and y_n_gfs is not read.)
extern "C" int MoL_step_adjoint(const rfm_struct *rfmstruct, const paramstruct *params,
    const bc_struct *bcstruct, const double *y_n_gfs, double *lambda_gfs, double *U1, double *U2,
    double *U3, double *rt, double *acc, double *kbar, double *w, double *vjp_G, double *auxevol_gfs,
    const double dt, hipStream_t stream) {
  if (!rfmstruct || !params || !bcstruct || !y_n_gfs || !lambda_gfs || !U1 || !U2 || !U3 || !rt ||
      !acc || !kbar || !w || !vjp_G) return NRPY_ERR_NULL;
  (void)auxevol_gfs;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  nrpy_gf_parity_args gfp;
  int rc = nrpy_bc_check(params, bcstruct, NUM_EVOL_GFS, evol_gf_parity, lambda_gfs, &gfp);
  if (rc) return rc;
  if ((rc = rhs_eval_vjp_rk4_stage(3, params, lambda_gfs, lambda_gfs, lambda_gfs, acc, kbar, dt / 6.0, dt / 3.0, dt, stream))) return rc;
  if ((rc = rhs_eval_vjp_rk4_stage(2, params, kbar, lambda_gfs, acc, acc, w, 1.0, dt / 3.0, dt / 2.0, stream))) return rc;
  if ((rc = rhs_eval_vjp_rk4_stage(1, params, w, lambda_gfs, acc, acc, kbar, 1.0, dt / 6.0, dt / 2.0, stream))) return rc;
  if ((rc = rhs_eval_vjp_rk4_stage(0, params, kbar, lambda_gfs, acc, lambda_gfs, nullptr, 1.0, 0.0, 0.0, stream))) return rc;
  return NRPY_OK;
}

// One RK4 step with the Sommerfeld radiation condition on the RHS.
// Sommerfeld EVOL grid function parameters
static __constant__ double evolgf_at_inf[NUM_EVOL_GFS] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
static __constant__ double evolgf_radial_falloff_power[NUM_EVOL_GFS] = {3.0, 3.0, 3.0, 3.0, 3.0, 3.0, 3.0, 3.0};
static __constant__ double evolgf_speed[NUM_EVOL_GFS] = {1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
#define NRPY_SOMMERFELD_MIN_N (NGHOSTS + 2 + 1)
#define NRPY_SOMMERFELD_FD 2
// r and d f/d r at (i0,i1,i2) of one gridfunction f, read as fa(i0,i1,i2); F = the point's
// FACE (CurviBoundaryConditions.py:329-516).
template <typename FA>
static __device__ void nrpy_sommerfeld_r_dfdr(const paramstruct &params, const double *__restrict__ xx0_arr, const double *__restrict__ xx1_arr, const double *__restrict__ xx2_arr, FA fa, const int F0, const int F1, const int F2, const int i0, const int i1, const int i2, double *r_out, double *dfdr_out) {
  const int Nxx_plus_2NGHOSTS0 = params.Nxx_plus_2NGHOSTS0;
  const int Nxx_plus_2NGHOSTS1 = params.Nxx_plus_2NGHOSTS1;
  const int Nxx_plus_2NGHOSTS2 = params.Nxx_plus_2NGHOSTS2;
  const double invdx0 = params.invdx0;
  const double invdx1 = params.invdx1;
  const double invdx2 = params.invdx2;
  const double xx0 = xx0_arr[i0], xx1 = xx1_arr[i1], xx2 = xx2_arr[i2];
  (void)xx0; (void)xx1; (void)xx2; (void)F0; (void)F1; (void)F2;
  double fdD0 = 1e100, fdD1 = 1e100, fdD2 = 1e100;
  (void)fdD0; (void)fdD1; (void)fdD2;
  {
    const bool one_sided = abs(F0) == 1 || i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0 || i0 - NGHOSTS <= 0;
    int S = F0;
    if (i0 + NGHOSTS >= Nxx_plus_2NGHOSTS0) S = -1;
    if (i0 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic0 = min(max(i0, 1), Nxx_plus_2NGHOSTS0 - 1 - 1);
    const double one = S*(-1.5*fa(i0,i1,i2) + 2.*fa(i0+1*S,i1,i2) + -0.5*fa(i0+2*S,i1,i2))*invdx0;
    const double cen = (fa(nrpy_ic0+1,i1,i2) - fa(nrpy_ic0+-1,i1,i2))*0.5*invdx0;
    fdD0 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F1) == 1 || i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1 || i1 - NGHOSTS <= 0;
    int S = F1;
    if (i1 + NGHOSTS >= Nxx_plus_2NGHOSTS1) S = -1;
    if (i1 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic1 = min(max(i1, 1), Nxx_plus_2NGHOSTS1 - 1 - 1);
    const double one = S*(-1.5*fa(i0,i1,i2) + 2.*fa(i0,i1+1*S,i2) + -0.5*fa(i0,i1+2*S,i2))*invdx1;
    const double cen = (fa(i0,nrpy_ic1+1,i2) - fa(i0,nrpy_ic1+-1,i2))*0.5*invdx1;
    fdD1 = one_sided ? one : cen;
  }
  {
    const bool one_sided = abs(F2) == 1 || i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2 || i2 - NGHOSTS <= 0;
    int S = F2;
    if (i2 + NGHOSTS >= Nxx_plus_2NGHOSTS2) S = -1;
    if (i2 - NGHOSTS <= 0) S = +1;
    const int nrpy_ic2 = min(max(i2, 1), Nxx_plus_2NGHOSTS2 - 1 - 1);
    const double one = S*(-1.5*fa(i0,i1,i2) + 2.*fa(i0,i1,i2+1*S) + -0.5*fa(i0,i1,i2+2*S))*invdx2;
    const double cen = (fa(i0,i1,nrpy_ic2+1) - fa(i0,i1,nrpy_ic2+-1))*0.5*invdx2;
    fdD2 = one_sided ? one : cen;
  }
  const double tmp_0 = sqrt(((xx0)*(xx0)) + ((xx1)*(xx1)) + ((xx2)*(xx2)));
  *r_out = tmp_0;
  *dfdr_out = (fdD0*xx0 + fdD1*xx1 + fdD2*xx2)/tmp_0;
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
extern "C" int MoL_step_forward_in_time_sommerfeld_unfused(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, hipStream_t stream) {
  if (!params || !y_n_gfs || !k_odd_gfs || !k_even_gfs || !y_nplus1_running_total_gfs) return NRPY_ERR_NULL;
  if (nrpy_check_params(params)) return NRPY_ERR_SHAPE;
  const size_t Ntot = (size_t)params->Nxx_plus_2NGHOSTS0 * params->Nxx_plus_2NGHOSTS1 * params->Nxx_plus_2NGHOSTS2;
  int rc;
  /* substep 0: RHS(y_n_gfs) -> k_odd_gfs */
  if ((rc = rhs_eval(params, y_n_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, y_n_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(0, (size_t)NUM_EVOL_GFS * Ntot, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 1: RHS(k_odd_gfs) -> k_even_gfs */
  if ((rc = rhs_eval(params, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(1, (size_t)NUM_EVOL_GFS * Ntot, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 2: RHS(k_even_gfs) -> k_odd_gfs */
  if ((rc = rhs_eval(params, k_even_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_even_gfs, k_odd_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(2, (size_t)NUM_EVOL_GFS * Ntot, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  /* substep 3: RHS(k_odd_gfs) -> k_even_gfs */
  if ((rc = rhs_eval(params, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld(params, xx, bcstruct, NUM_EVOL_GFS, evol_gf_parity, k_odd_gfs, k_even_gfs, stream))) return rc;
  if ((rc = nrpy_rk4_update_all(3, (size_t)NUM_EVOL_GFS * Ntot, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, dt, stream))) return rc;
  return NRPY_OK;
}
// One RK4 step of the Sommerfeld branch (see MoL_step_forward_in_time_sommerfeld_unfused for
// the reference's order of operations; the fused form gives the same values).
extern "C" int MoL_step_forward_in_time_sommerfeld(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, hipStream_t stream) {
  if (!params || !bcstruct || !xx || !y_n_gfs || !k_odd_gfs || !k_even_gfs ||
      !y_nplus1_running_total_gfs) return NRPY_ERR_NULL;
  bool inner = false;
  for (int gz = 0; gz < NGHOSTS; gz++) inner = inner || bcstruct->num_ib_gz_pts[gz] > 0;
  double *R = inner ? nullptr : nrpy_sommerfeld_scratch(bcstruct, NUM_EVOL_GFS, stream);
  if (!R) return MoL_step_forward_in_time_sommerfeld_unfused(params, rfmstruct, xx, bcstruct, y_n_gfs, k_odd_gfs, k_even_gfs, y_nplus1_running_total_gfs, dt, stream);
  int rc;
  /* substep 0: y_n_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep_shell(0, params, y_n_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, R, dt, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld_rk4(0, params, xx, bcstruct, NUM_EVOL_GFS, y_n_gfs, R, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  /* substep 1: k_odd_gfs -> k_even_gfs */
  if ((rc = rhs_eval_rk4_substep_shell(1, params, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, R, dt, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld_rk4(1, params, xx, bcstruct, NUM_EVOL_GFS, k_odd_gfs, R, y_n_gfs, y_nplus1_running_total_gfs, k_even_gfs, dt, stream))) return rc;
  /* substep 2: k_even_gfs -> k_odd_gfs */
  if ((rc = rhs_eval_rk4_substep_shell(2, params, k_even_gfs, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, R, dt, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld_rk4(2, params, xx, bcstruct, NUM_EVOL_GFS, k_even_gfs, R, y_n_gfs, y_nplus1_running_total_gfs, k_odd_gfs, dt, stream))) return rc;
  /* substep 3: k_odd_gfs -> y_n_gfs */
  if ((rc = rhs_eval_rk4_substep_shell(3, params, k_odd_gfs, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, R, dt, stream))) return rc;
  if ((rc = apply_bcs_sommerfeld_rk4(3, params, xx, bcstruct, NUM_EVOL_GFS, k_odd_gfs, R, y_n_gfs, y_nplus1_running_total_gfs, y_n_gfs, dt, stream))) return rc;
  return NRPY_OK;
}
// The Sommerfeld RK4 step captured into a hipGraph (every launch is a kernel; the pointers, those of
// xx among them, and dt are fixed at capture); replay with MoL_graph_launch, free with MoL_graph_free.
extern "C" int MoL_sommerfeld_graph_create(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3], const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt, MoL_graph **out) {
  if (!out) return NRPY_ERR_NULL;
  *out = nullptr;
  hipStream_t s;
  if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return NRPY_ERR_LAUNCH;
  if (bcstruct) {  /* the fused step's scratch, allocated before capture */
    bool inner = false;
    for (int gz = 0; gz < NGHOSTS; gz++) inner = inner || bcstruct->num_ib_gz_pts[gz] > 0;
    if (!inner) (void)nrpy_sommerfeld_scratch(bcstruct, NUM_EVOL_GFS, s);
  }
  MoL_graph *g = new MoL_graph();
  int rc = NRPY_OK;
  if (hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal) != hipSuccess) rc = NRPY_ERR_LAUNCH;
  if (!rc) {
    rc = MoL_step_forward_in_time_sommerfeld(params, rfmstruct, xx, bcstruct, y_n_gfs, k_odd_gfs, k_even_gfs,
                                             y_nplus1_running_total_gfs, dt, s);
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
