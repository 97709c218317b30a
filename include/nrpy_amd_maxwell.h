/* Vacuum Maxwell System II, Cartesian coordinates (bundle maxwell_cartesian).
 * Entry points of Tutorial-Start_to_Finish-Solving_Maxwells_Equations_in_Vacuum-Cartesian.ipynb's
 * C driver; common declarations in nrpy_amd.h. Evolved gridfunctions in
 * alphabetical order: AU0..2, EU0..2, Gamma, psi; aux DivE, G. */
#ifndef NRPY_AMD_MAXWELL_H
#define NRPY_AMD_MAXWELL_H
#include "nrpy_amd.h"
#ifdef __cplusplus
extern "C" {
#endif

/* Replaces rhs_eval(const paramstruct *, const REAL *in_gfs, REAL *rhs_gfs) of the
 * Maxwell Cartesian driver (VacuumMaxwell_Flat_Evol_Cartesian.py:84-112, System II). */
int rhs_eval(const paramstruct *params, const double *in_gfs, double *rhs_gfs, hipStream_t stream);

/* The constraints C = div E (DivE) and G = Gamma - div A at interior points
 * (VacuumMaxwell_Flat_Evol_Cartesian.py:56-58, 93-96). */
int Maxwell_constraints(const paramstruct *params, const double *in_gfs, double *aux_gfs, hipStream_t stream);

/* Toroidal dipole data (Maxwell/InitialData.py:25-113) at all points. */
int initial_data(const paramstruct *params, double *xx[3], double *in_gfs, hipStream_t stream);

/* Vector-Jacobian product of rhs_eval (no counterpart in the reference): for the
 * cotangent cot_rhs_gfs of the RHS at interior points, the cotangent of every input
 * gridfunction at every point, ghost points included (fold those with bc_apply_T).
 * vjp_G: scratch of <bundle>.json "vjp_slots" gridfunctions (one per pointwise slot:
 * gridfunction value or stencil). auxevol_gfs and cot_auxevol_gfs may be NULL. */
int rhs_eval_vjp(const paramstruct *params, const double *auxevol_gfs, const double *in_gfs,
                 const double *cot_rhs_gfs, double *vjp_G, double *cot_in_gfs, double *cot_auxevol_gfs,
                 hipStream_t stream);

/* Adjoint of one RK4 step (MoL_step_forward_in_time): lambda_gfs holds the cotangent of
 * y_{n+1} on entry and that of y_n on exit; y_n_gfs is the state at the start of the step.
 * acc, kbar, w: three scratch states. The right-hand side is linear, so the state is not read, and
 * U1..U3, rt and vjp_G are neither read nor written (not NULL). */
int MoL_step_adjoint(const rfm_struct *rfmstruct, const paramstruct *params, const bc_struct *bcstruct,
                     const double *y_n_gfs, double *lambda_gfs, double *U1, double *U2, double *U3, double *rt,
                     double *acc, double *kbar, double *w, double *vjp_G, double *auxevol_gfs, const double dt,
                     hipStream_t stream);

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
 * (Tutorial-Start_to_Finish-Solving_Maxwells_Equations_in_Vacuum-Cartesian.ipynb:240-246).
 * Fused where the grid has no inner boundary points (this Cartesian bundle): per substep the
 * interior RHS with its RK4 update (rhs_eval_rk4_substep_shell), then the radiation condition
 * at the outer points with theirs (apply_bcs_sommerfeld_rk4). The values are those of the
 * reference's order, MoL_step_forward_in_time_sommerfeld_unfused below. The first call
 * allocates a right-hand-side scratch array (all gridfunctions, whole grid) kept in bcstruct;
 * a step recorded into a graph before that array exists takes the unfused form.
 * xx: device coordinate arrays. */
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

/* Substep S (0-3) of the fused Sommerfeld step at the interior: the RHS and its RK4 update
 * (as rhs_eval_rk4_substep), and at the interior points next to the boundary the RHS also
 * into shell_rhs: NUM_EVOL_GFS whole-grid gridfunctions (points next to an i1 or i2 boundary),
 * followed by NUM_EVOL_GFS x N2 x N1 x 2 doubles [gf][i2][i1][side] (points next to an i0
 * boundary; side 0 at i0 = NGHOSTS, 1 at i0 = N0 - 1 - NGHOSTS), N = Nxx_plus_2NGHOSTS.
 * apply_bcs_sommerfeld_rk4 reads R in this layout. No counterpart in the reference. */
int rhs_eval_rk4_substep_shell(const int S, const paramstruct *params, const double *in_gfs, double *y_n,
                               double *rt, double *out, double *shell_rhs, const double dt,
                               hipStream_t stream);

/* Substep S of the fused Sommerfeld step at the outer points: the radiation condition
 * (apply_bcs_sommerfeld's arithmetic) with the RHS at each point's inward neighbour read from
 * R and its own written there, and the RK4 update of that point (nrpy_rk4_update_all's
 * arithmetic), layer by layer. gfs: the substep's input state. NRPY_ERR_PARAM for grids with
 * inner boundary points. No counterpart in the reference. */
int apply_bcs_sommerfeld_rk4(const int S, const paramstruct *params, double *xx[3], const bc_struct *bc,
                             const int NUM_GFS, double *gfs, double *R, double *y_n, double *rt,
                             double *out, const double dt, hipStream_t stream);


/* The Sommerfeld step above captured into a hipGraph (no counterpart in the reference; the pointers,
 * those in xx among them, and dt are fixed at capture), replayed nsteps times per MoL_graph_launch,
 * freed with MoL_graph_free. Creating it reads no device memory; a launch reads all of it, the
 * coordinates too, in its stream's order. */
int MoL_sommerfeld_graph_create(const paramstruct *params, const rfm_struct *rfmstruct, double *xx[3],
                                const bc_struct *bcstruct, double *y_n_gfs, double *k_odd_gfs, double *k_even_gfs,
                                double *y_nplus1_running_total_gfs, const double dt, MoL_graph **out);

#ifdef __cplusplus
}
#endif
#endif
