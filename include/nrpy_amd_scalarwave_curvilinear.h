/* Scalar wave equation in a curvilinear reference metric (bundles
 * scalarwave_sinhspherical, scalarwave_sinhsphericalv2, scalarwave_sinhcylindrical,
 * scalarwave_sinhcylindricalv2, scalarwave_symtp, scalarwave_sinhsymtp).
 * Entry points of Tutorial-Start_to_Finish-ScalarWaveCurvilinear.ipynb's C
 * driver with rfm precompute; common declarations in nrpy_amd.h. */
#ifndef NRPY_AMD_SCALARWAVE_CURVILINEAR_H
#define NRPY_AMD_SCALARWAVE_CURVILINEAR_H
#include "nrpy_amd.h"
#ifdef __cplusplus
extern "C" {
#endif

/* Replaces rhs_eval(rfm_struct *, const paramstruct *, const REAL *in_gfs, REAL *rhs_gfs)
 * of the curvilinear scalar-wave driver (ScalarWaveCurvilinear_RHSs.py:43-98):
 * vv_rhs = c^2 (ghat^ij uu_{,ij} - ghat^ij Gammahat^k_ij uu_{,k}). */
int rhs_eval(const rfm_struct *rfmstruct, const paramstruct *params, const double *in_gfs, double *rhs_gfs,
             hipStream_t stream);

/* Plane-wave data in the curvilinear coordinates (ScalarWave/InitialData.py:59-88). */
int initial_data(const paramstruct *params, double *xx[3], double *in_gfs, hipStream_t stream);

/* Sommerfeld radiation condition on the RHS (apply_bcs_sommerfeld,
 * CurviBoundaryConditions.py:538-620; no stream in the reference): at every outer ghost
 * point, innermost layer first, rhs = -v [d f/dr + (f - f_inf)/r] plus the falloff term
 * extrapolated from one point inward; then the parity copies at inner ghost points.
 * xx: the three device coordinate arrays; gfs: the state rhs_gfs was evaluated from;
 * gfs_parity: host array of NUM_GFS parity types; NUM_GFS <= NUM_EVOL_GFS. The
 * per-gridfunction v, f_inf and falloff power are the bundle's (<bundle>.json "sommerfeld"). */
int apply_bcs_sommerfeld(const paramstruct *params, double *xx[3], const bc_struct *bc, const int NUM_GFS,
                         const int8_t *gfs_parity, double *gfs, double *rhs_gfs, hipStream_t stream);

/* One RK4 step of the Start-to-Finish drivers' BoundaryCondition = "Sommerfeld" branch
 * (per substep rhs_eval + apply_bcs_sommerfeld, then the RK4 update at every point; no ghost
 * fill of the state). This bundle's grids have inner boundary points, so the step is
 * MoL_step_forward_in_time_sommerfeld_unfused. xx: device coordinate arrays. */
int MoL_step_forward_in_time_sommerfeld(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3],
                                        const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs,
                                        double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt,
                                        hipStream_t stream);

/* The same step in the reference's order of operations: per substep rhs_eval +
 * apply_bcs_sommerfeld, then the RK4 update at every point. */
int MoL_step_forward_in_time_sommerfeld_unfused(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3],
                                                const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs,
                                                double *k_even_gfs, double *y_nplus1_running_total_gfs, const double dt,
                                                hipStream_t stream);


/* The Sommerfeld step above captured into a hipGraph (no counterpart in the reference; the pointers,
 * those in xx among them, and dt are fixed at capture), replayed nsteps times per MoL_graph_launch,
 * freed with MoL_graph_free. Creating it reads no device memory; a launch reads all of it, the
 * coordinates too, in its stream's order.
 * The captured step takes two launches per substep instead of one per layer and face group, and
 * equals it to rounding (1e-13 of the largest value). It allocates device memory that the graph owns until MoL_graph_free
 * (2 NUM_EVOL_GFS + 5 gridfunctions); without that memory it captures the step above. */
int MoL_sommerfeld_graph_create(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3],
                                const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs,
                                double *y_nplus1_running_total_gfs, const double dt, MoL_graph **out);

#ifdef __cplusplus
}
#endif
#endif
