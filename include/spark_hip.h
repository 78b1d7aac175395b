/*
 * spark_hip.h -- C ABI of the MI355X-native Spark unsplit-hydro RK stage.
 *
 * This is the drop-in boundary that a new Spark variant's Fortran Hydro(),
 * Hydro_computeDt() and Hydro_init() call through ISO_C_BINDING
 * (flash-x_amd/fortran/spark_hip_mod.F90 holds the bind(C) interfaces).
 * All entry points are extern "C", take plain pointers and sizes, return
 * an int status (SPARK_OK = 0) and never abort: a Fortran caller maps a
 * non-zero status to Driver_abort(spark_last_error text), which is how the
 * reference reports failures (Driver/Driver_abort.F90).
 *
 * Paths below are relative to Flash-X/source/.
 *
 * Data model.  The host hands over LEAF blocks as the reference tile
 * iterator exposes them: one pointer per block to unk(NUNK_VARS, i, j, k)
 * over the guard-celled box, variable index fastest
 * (Grid/GridMain/AMR/Paramesh4/Grid_tile.F90:157-267, getDataPtr).  The
 * library keeps its own device copy in structure-of-arrays form for the
 * whole batch, from spark_pack() to spark_unpack().
 */
#ifndef SPARK_HIP_H
#define SPARK_HIP_H
#ifdef __cplusplus
extern "C" {
#endif

#define SPARK_OK 0
#define SPARK_ERR_ARG 1         /* invalid argument or unsupported option */
#define SPARK_ERR_HIP 2         /* HIP runtime error */
#define SPARK_ERR_STATE 3       /* call out of sequence */
#define SPARK_ERR_NUMERIC 4     /* negative a^2 faces were met (Riemann ierr) */

#define SPARK_MAX_SCALARS 8
#define SPARK_NPROP 11          /* dens eint ener gamc game pres shok temp velx vely velz */

enum spark_recon { SPARK_RECON_WENO5 = 0, SPARK_RECON_MP5 = 1, SPARK_RECON_PLM = 2, SPARK_RECON_FOG = 3 };
enum spark_riemann { SPARK_RIEMANN_HLLC = 0, SPARK_RIEMANN_HLL = 1 };
/* plain FP64 form (directional sweeps, one launch per sweep, stage and block
 * shape); FP32-flux form (one fused persistent launch per stage over blocks
 * of any size, FP32 reconstruction/Riemann arithmetic and FP64
 * accumulation); batched FP64 form (the plain form's sweeps; its stage entry
 * points read same-level halos as the FP32-flux form's do) */
enum spark_form { SPARK_FORM_PLAIN_FP64 = 0, SPARK_FORM_FP32_FLUX = 1, SPARK_FORM_BATCHED_FP64 = 2 };
/* guard policy: telescoping stages over guard cells filled once per step
 * (the reference's own scheme, Spark/Hydro.ini:19,37), or refilling the
 * guards of a uniform block grid on the device between stages */
enum spark_guard_mode { SPARK_GUARD_TELESCOPE = 0, SPARK_GUARD_REFILL = 1 };
/* equation of state: the gamma law (Eos/EosMain/Gamma) or a mixture of
 * gamma-law species (Eos/EosMain/Multigamma/Eos.F90) */
enum spark_eos { SPARK_EOS_GAMMA = 0, SPARK_EOS_MULTIGAMMA = 1 };

/* Runtime parameters (Hydro_init.F90 / Eos_init.F90 subset).
 * Replaces the RuntimeParameters_get calls of Spark/Hydro_init.F90:60-104
 * and Eos/EosMain/Gamma/Eos_init.F90:55-86. */
typedef struct spark_params {
  double gamma;        /* Eos/EosMain/Config:43                             */
  double cfl;          /* Hydro/HydroMain/Config:26                         */
  double cvisc;        /* Spark/Config:17                                   */
  double smlrho;       /* smallest density                                  */
  double smallp;       /* smallest pressure                                 */
  double smalle;       /* smallest specific energy                          */
  double smallx;       /* smallest mass fraction                            */
  double eintSwitch;   /* Eos/EosMain/Config:39                             */
  double tiny;         /* hy_tiny, Spark/Hydro_data.F90:85                  */
  double gasConst;     /* ideal gas constant, PhysicalConstants_init.F90:186 */
  double abar;         /* eos_singleSpeciesA                                */
  double grav[3];      /* constant gravitational acceleration (source term) */
  int ndim;            /* 1, 2 or 3                                         */
  int nguard;          /* NGUARD                                            */
  int nstencil;        /* NSTENCIL (3 for WENO5/MP5, 2 for PLM/FOG)         */
  int rk_order;        /* 2 or 3 (Spark/Hydro.ini:2-48)                     */
  int recon;           /* enum spark_recon                                  */
  int riemann;         /* enum spark_riemann                                */
  int use_flattening;  /* Spark/Config:42                                   */
  int use_hybrid_riemann; /* Spark/Config:43                                */
  int nscalars;        /* NMASS_SCALARS, 0..SPARK_MAX_SCALARS               */
  int use_gravity;     /* apply grav[] as a source in the update            */
  int flux_correct;    /* accumulate flux registers (Spark/Hydro.F90-mc:160) */
  int form;            /* enum spark_form                                   */
  int guard_mode;      /* enum spark_guard_mode                             */
  int nunk_vars;       /* NUNK_VARS of the host unk array                   */
  /* 0-based unk slot of dens eint ener gamc game pres shok temp velx vely
   * velz, then the mass scalars (the *_VAR map of Simulation.h minus 1) */
  int var_index[SPARK_NPROP + SPARK_MAX_SCALARS];
  /* Species: the first nspecies of the nscalars mass scalars are species
   * mass fractions (SPECIES_BEGIN precedes MASS_SCALARS_BEGIN in unk).  Their
   * face states are clamped to [smallx, 1] and renormalised
   * (Spark/Hydro.ini:227-235).  eos = SPARK_EOS_MULTIGAMMA mixes them with
   * per-species gamma and mass number A (Multigamma/Eos.F90, ORIGINAL_GAMC_
   * AVERAGE; eos_initMgamma.F90:12-18); needs nspecies >= 1.  The batched
   * forms take at most 4 species, and the FP32-flux form the gamma law only
   * (Multigamma runs in the plain and batched FP64 forms). */
  int nspecies;
  int eos;             /* enum spark_eos                                    */
  int reserved;        /* 0; keeps the arrays below 8-byte aligned with no implicit padding */
  double species_a[SPARK_MAX_SCALARS];      /* A of each species           */
  double species_gamma[SPARK_MAX_SCALARS];  /* gamma of each species       */
} spark_params;

/* One LEAF block (tileDesc%limits, %deltas, %level). */
typedef struct spark_block_desc {
  int nx, ny, nz;      /* interior cells (1 for unused dimensions) */
  int level;           /* refinement level (1 = coarsest)          */
  double dx, dy, dz;   /* cell widths                              */
} spark_block_desc;

typedef struct spark_batch spark_batch;

/* Reference defaults (Spark/Config, Eos/EosMain/Config, Grid Configs). */
int spark_params_default(spark_params* p);

/* Select the device and create the library's stream.
 * Replaces: the device set-up implicit in Spark/Hydro_init.F90:24-179. */
int spark_init(int device);
int spark_finalize(void);

/* Device storage for a set of LEAF blocks, alive until destroy.
 * Replaces: allocate_scr/deallocate_scr, Spark/Hydro_funcs.F90-mc:337-422
 * (the reference allocates scratch per block; here once per batch).  Three
 * states of 11 + N_s doubles per guard-celled cell and one field; rows are
 * padded to memory lines (a third more at most) where the padded states take
 * no more than 3/8 of the device memory that is free, and the FP64 forms hold
 * 5 + N_s fields more where those take no more than a quarter of what is left. */
int spark_batch_create(const spark_params* p, int nblocks, const spark_block_desc* blocks, spark_batch** out);
int spark_batch_destroy(spark_batch* b);

/* Host unk blocks (guard-celled box, nunk_vars fastest) -> device.
 * Replaces: tileDesc%getDataPtr + saveState's read of Uin,
 * Grid_tile.F90:157-267 and Spark/Hydro_funcs.F90-mc:512-541.
 * pack and unpack stage through 4 x 8 MiB of pinned host and of device
 * memory that the library keeps from its first transfer to spark_finalize
 * (transfers of several threads take turns); from 4 MiB on, three helper
 * threads share the host copies for the length of the call. */
int spark_pack(spark_batch* b, const double* const* unk_blocks);
/* spark_pack without device allocation.  No counterpart in the reference:
 * it is for callers that cannot allocate device memory (tight stepping
 * loops, harnesses that forbid hipMalloc).  The host blocks are staged in a
 * fixed 64 MiB device area per GPU, held from spark_init until the process
 * ends, in rounds of at most 1024 blocks; a block larger than the area
 * (nunk_vars * NX * NY * NZ doubles beyond 64 MiB less 8.25 KiB) is refused
 * with SPARK_ERR_ARG.  The result equals spark_pack's.  All calls on one
 * GPU share the area: calls that overlap in time on one GPU (from several
 * threads) race. */
int spark_pack_noalloc(spark_batch* b, const double* const* unk_blocks);
/* Device -> host unk blocks; interior_only mirrors updateState
 * (Spark/Hydro_funcs.F90-mc:573-574) and writes only the interior cells;
 * unk slots outside the variable map keep their host values.  which = 0:
 * solution, 1: the stage state (hy_starState) written by the last stage run
 * before a step's final stage.  Guard cells (interior_only = 0): spark_hydro_step
 * and spark_advance write no guard cell of the new solution (updateState copies
 * the interior), so after them the guards of the solution hold the guard fill
 * at the start of the last step, as the reference's unk does, and those of the
 * stage state what the last stage before the final one computed there, or the
 * refill after it:
 *   plain form                   solution: the layers the first stage reaches
 *                                (refill: nstencil layers); stage state: the
 *                                layers that stage covers (refill: nstencil)
 *   batched forms, 3D refill     solution: one layer, two with the hybrid
 *                                solver; stage state: none
 *   batched forms, hierarchy     solution: the guard sectors (face, edge or
 *                                corner regions of the guard band) with no
 *                                leaf of the block's own level across them,
 *                                and of blocks with such sectors the first
 *                                layer of the others (every layer with the
 *                                hybrid solver); stage state: those sectors
 *   batched forms, otherwise     as the plain form
 * Other guard cells keep what they held.  spark_fill_guardcells fills all of
 * the solution's from its present interior. */
int spark_unpack(spark_batch* b, double* const* unk_blocks, int interior_only, int which);

/* Declare the batch a uniform nbx x nby x nbz block grid (blocks numbered
 * x fastest) with OUTFLOW domain faces, enabling device guard fills.
 * Replaces: Grid_fillGuardCells for one refinement level,
 * Grid/GridMain/AMR/Paramesh4/Grid_fillGuardCells.F90:436-546 and
 * Grid/GridBoundaryConditions/Grid_bcApplyToRegion.F90:526-532. */
int spark_set_uniform_grid(spark_batch* b, int nbx, int nby, int nbz);

/* Declare the batch a Paramesh-like hierarchy of leaf blocks (3D,
 * telescope guard mode, all blocks n^3 with n even): level-1 grid of
 * nbx0 x nby0 x nbz0 blocks; block i (its spark_block_desc level is 1-based)
 * has its first interior cell at origins[3*i .. 3*i+2], the global cell
 * index at its own level; bc[3] (NULL: all OUTFLOW) gives each dimension's
 * domain boundary, SPARK_BC_OUTFLOW, SPARK_BC_PERIODIC or SPARK_BC_REFLECT.  The leaves must tile the domain, and
 * every leaf under a block's guard cells must be within one level of it.
 * Enables the device guard fill over levels (same-level copy, the mean of 8
 * cells of a finer leaf, limited linear prolongation from a coarser leaf)
 * and, with flux_correct, the device flux-register exchange after every
 * step.  In spark_hydro_step and spark_advance, and in the batched forms'
 * stage entry points, a leaf reads a guard sector with a leaf of its own level
 * across it from that leaf, and an edge or corner sector beside a leaf of its
 * level that computes it from that leaf's guard cells, and computes only its
 * interior and the other sectors (the values telescoping would give;
 * spark_unpack says which guard cells are left in its own box).  The plain
 * form's stage entry points telescope over the block's own guard cells:
 * spark_fill_guardcells goes before them.  With flux_correct the
 * FP32-flux form corrects only the cells on faces toward a finer leaf (the
 * correction is zero elsewhere; the FP64 forms still pass those cells
 * through the reference's conserved/primitive round trip).  A declaration
 * that returns SPARK_ERR_HIP (no memory for its tables) leaves the batch
 * without a hierarchy; it may be declared again.
 * Replaces: Grid_fillGuardCells over PARAMESH leaves,
 * Grid/GridMain/AMR/Paramesh4/Grid_fillGuardCells.F90:436-546, and the
 * flux hand-off of Spark/Hydro.F90-mc:197-236. */
#define SPARK_BC_OUTFLOW 0   /* guard = first interior layer (Grid_bcApplyToRegion.F90:526-532) */
#define SPARK_BC_PERIODIC 1
#define SPARK_BC_REFLECT 2   /* mirror image, normal velocity negated */
int spark_set_amr_grid(spark_batch* b, int nbx0, int nby0, int nbz0, const int* origins, const int* bc);
int spark_fill_guardcells(spark_batch* b);

/* CFL time step over all blocks.  minloc = (i, j, k, level, block): the
 * cell indices 1-based in the guard-celled box as Fortran sees them, as
 * dtMinLoc(1:4) of the reference (Spark/Hydro_computeDt.F90:126-134); the
 * fifth entry, the MPI rank there, is the 0-based batch index of the block.
 * Replaces: Hydro_computeDt, Hydro_interface.F90:24-42 /
 * Spark/Hydro_computeDt.F90:27-150 (per tile) plus the MIN over tiles of
 * Driver/DriverMain/Driver_computeDt.F90:306. */
int spark_compute_dt(spark_batch* b, double* dt, int minloc[5]);

/* One full RK step of every block: the guard fill when a uniform grid or a
 * hierarchy was declared (Spark/Hydro.F90-mc:106), shockDetect, saveState, the stages,
 * updateState; flux registers when flux_correct.
 * Replaces: Hydro(timeEndAdv, dt, dtOld, sweepOrder),
 * Hydro_interface.F90:61-66 / Spark/Hydro.F90-mc:24-202. */
int spark_hydro_step(spark_batch* b, double dt, double dtOld);

/* Stage-level entry points (parity testing, custom drivers).
 * step_begin = shockDetect + saveState (Spark/Hydro.F90-mc:129-137);
 * stage = one pass of the stage loop body (Spark/Hydro.F90-mc:144-192)
 * with ngoff extra guard layers; step_end = updateState. */
int spark_step_begin(spark_batch* b);
int spark_stage(spark_batch* b, int stage, double dt, int ngoff);
int spark_step_end(spark_batch* b);

/* nsteps device-resident steps: dt (CFL, on the device) -> guard fill (if a
 * grid was declared; only the cells a step reads before the last one) -> step.  dts (optional, nsteps) receives the
 * dt used at each step.  No host synchronisation between steps.
 * Replaces: the Hydro / Driver_computeDt pair of the step loop,
 * Driver/DriverMain/Unsplit/Driver_evolveAll.F90:136-275. */
int spark_advance(spark_batch* b, int nsteps, double* dts);
/* The driver's limits on the dt of the spark_advance steps, kept on the
 * device: the next step takes dt_init as its dt (Flash-X's dtinit, the
 * first step of Driver_evolveAll) when dt_init > 0; every later step takes
 * the CFL dt limited to the previous dt x change_factor (when > 0) and
 * clamped to [dt_min, dt_max] (each when > 0), in that order.  All zero:
 * the CFL dt (the default).  spark_compute_dt is not affected.
 * Replaces: Driver/DriverMain/Driver_computeDt.F90:450-460 (dr_tstepChangeFactor,
 * dr_dtMin, dr_dtMax) and dr_dtInit. */
int spark_set_dt_control(spark_batch* b, double dt_init, double change_factor, double dt_min, double dt_max);

/* Geometry of the plain form (the batched forms are Cartesian only).
 * SPARK_GEOM_CYLINDRICAL: 2D (r, z), x the radius, the z velocity the
 * azimuthal one.  SPARK_GEOM_SPHERICAL: 1D (r) or 2D (r, theta), the y and
 * z velocities the polar and azimuthal ones.  Per block, over its
 * guard-celled box of NX x NY cells (NY = 1 in 1D): the cell-centre radius,
 * the area of each cell's low x face (NX * NY, x fastest), each cell's
 * volume (NX * NY), the left and right edge radius (NX each) -- the Grid's
 * hy_xCenter, hy_farea, hy_cvol, hy_xLeft and hy_xRight, which the update
 * and the flux correction turn into facM/facP = farea dx / cvol and the
 * geometric sources ((rho vphi^2 + alpha p) / r, -rho vphi vr / r, and in
 * spherical geometry (rho vtheta)^2 / rho / r, scaled by dx / dx_sph); the
 * CFL step takes r dtheta as the theta width.
 * Replaces: Spark/Hydro.ini:40-56 (geom_1d_alloc), geoFacs in
 * Spark/hy_rk_updateSoln.F90-mc:98-175 and hy_rk_correctFluxes.F90:341-358,
 * Spark/Hydro_computeDt.F90:103-111.
 * SPARK_GEOM_CARTESIAN (the default) takes no arrays.  A block hierarchy
 * (spark_set_amr_grid) is Cartesian only. */
enum spark_geometry { SPARK_GEOM_CARTESIAN = 0, SPARK_GEOM_CYLINDRICAL = 1, SPARK_GEOM_SPHERICAL = 2 };
int spark_set_geometry(spark_batch* b, int geometry, const double* const* r_center, const double* const* x_face_area,
                       const double* const* cell_volume, const double* const* r_left, const double* const* r_right);

/* Flux registers (weighted sum over stages) in the shape of hy_fluxBuf[XYZ]:
 * every face of the block's interior, (NFLUXES, nx+1, ny, nz) for x etc.
 * Only the block's boundary faces (index 0 and n along the direction) are
 * accumulated, the faces Grid_putFluxData_block hands to PARAMESH
 * (Paramesh4/Grid_putFluxData_block.F90:200-202, 278-279); the others read 0.
 * get: device -> host fluxBufX/Y/Z(NFLUXES, ...) per block, Fortran order;
 *      replaces the hy_fluxBuf[XYZ] hand-off of Grid_putFluxData_block,
 *      Spark/Hydro.F90-mc:197-198.
 * set: host -> device correction data (restricted fine - coarse on the
 *      coarse side of fine/coarse faces, zero elsewhere), as
 *      Grid_getFluxCorrData_block returns it (Paramesh4/Grid_getFluxCorrData_block.F90:182-216).
 * correct: hy_rk_correctFluxes on every block (Spark/hy_rk_correctFluxes.F90:46-338). */
int spark_get_flux_registers(spark_batch* b, double* const* fbx, double* const* fby, double* const* fbz);
int spark_set_flux_corrections(spark_batch* b, const double* const* fbx, const double* const* fby,
                               const double* const* fbz);
int spark_flux_correct(spark_batch* b, double dt);

/* The flux-register exchange on the device over the declared hierarchy:
 * corrections = mean of the 4 fine faces (red_f = 0.25, flux densities)
 * minus the coarse block's own face flux on fine/coarse faces, 0 on every
 * other boundary face; they replace what spark_set_flux_corrections set.
 * Replaces: Grid_putFluxData_block + Grid_communicateFluxes +
 * Grid_getFluxCorrData_block (Paramesh4/Grid_putFluxData_block.F90:83-392,
 * Grid_communicateFluxes.F90:81-106, Grid_getFluxCorrData_block.F90:88-360,
 * PM4_package/source/amr_restrict_red.F90). */
int spark_flux_exchange(spark_batch* b);

/* Per-kernel timing of the library's own launches: HIP events recorded on
 * the library stream around every launch while enabled (enabling clears
 * earlier records).  read() returns one entry per kernel name with the
 * launch count, summed event time and summed algorithmic bytes and flops
 * of those launches.  No counterpart in the reference (its Timers_start /
 * Timers_stop labels, Spark/Hydro.F90-mc:76-191, time host regions). */
typedef struct spark_kernel_stat {
  char name[32];
  long long launches;
  double total_ms;
  double bytes;
  double flops;
} spark_kernel_stat;
int spark_profile(spark_batch* b, int enable);
int spark_profile_read(spark_batch* b, spark_kernel_stat* stats, int max, int* n);

/* Options.  SPARK_OPT_GRAPH (default 1): spark_advance captures one step
 * into a hipGraph and replays it.  SPARK_OPT_AUTOTUNE (default 1): the
 * batched FP32-flux form times candidate tile shapes per block shape and
 * stage region on the first step and keeps the fastest.
 * SPARK_OPT_SAME_LEVEL_HALOS (default 1): on a block hierarchy a leaf reads
 * guard sectors from leaves of its own level (spark_set_amr_grid) and
 * telescopes only over the others; 0 makes every leaf telescope over all its
 * guard cells (the same values, more work).  No counterpart in the
 * reference. */
#define SPARK_OPT_GRAPH 1
#define SPARK_OPT_AUTOTUNE 2
#define SPARK_OPT_SAME_LEVEL_HALOS 3
int spark_set_option(spark_batch* b, int option, int value);
/* Tiles chosen by the batched forms: rows of (nx, ny, nz, ngoff, tx, ty); the
 * batched FP64 form runs whole regions, (tx, ty) their cross-sections. */
int spark_batched_tiles(spark_batch* b, int* rows, int max_rows, int* nrows);

int spark_synchronize(spark_batch* b);
/* counters[0] = faces whose Riemann solve met a negative a^2 */
int spark_get_counters(spark_batch* b, long long* counters, int n);
/* Copy the last error message of this thread into buf (NUL-terminated). */
int spark_last_error(char* buf, int len);

#ifdef __cplusplus
}
#endif
#endif
