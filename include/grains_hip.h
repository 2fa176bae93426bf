/*
 * grains_hip.h -- C-ABI of the MI355X DEM time-step library (libgrains_hip.so).
 *
 * One explicit DEM time step = linked-cell broad phase (cell hash, LDS radix
 * sort, cell ranges) -> candidate pairs -> narrow phase (sphere analytic,
 * rectangle plane, bounding sphere + OBB prefilter, GJK on support maps) ->
 * Hooke spring-dashpot / Coulomb contact force -> gravity -> first-order
 * explicit integration with quaternion rotation update.
 *
 * Every symbol here replaces a piece of the reference's C++ component manager
 * (Grains/Component/include/ComponentManager.hh:24-184) and the objects it is
 * handed (RigidBody, LinkedCell, ContactForceModel, TimeIntegrator).  The
 * reference passes `T const* const*` arrays of polymorphic objects; this ABI
 * passes plain arrays and sizes.  All functions are synchronous at the
 * boundary (they return after the device work they enqueue has finished),
 * return 0 on success and a negative GRAINS_E* code on failure, and never
 * call exit() (the reference exits on configuration errors, e.g.
 * Grains/Base/src/Grains.cpp:103,131).  The context owns all device memory;
 * caller buffers are host memory unless the name says `_device`.
 *
 * Conventions
 *  - lengths in the caller's units (the reference uses SI), FP64 at the ABI;
 *  - quaternions are (x, y, z, w): w last, as Quaternion<T>::operator[]
 *    (Grains/Geometry/src/Quaternion.cpp:316-319);
 *  - a "transform" is the 12-double Transform3 buffer of the reference
 *    (Grains/Geometry/src/Transform3.cpp:26-29,133-137): row-major 3x3 basis
 *    (body -> world) followed by the origin;
 *  - pairs (i, j) use particle indices as given to grains_set_particles.
 */
#ifndef GRAINS_HIP_H
#define GRAINS_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- error codes ------------------------------------------------------- */
#define GRAINS_OK 0
#define GRAINS_EINVAL (-1)     /* bad argument or configuration            */
#define GRAINS_ENOMEM (-2)     /* device or host allocation failed         */
#define GRAINS_EDEVICE (-3)    /* HIP runtime error                        */
#define GRAINS_ESTATE (-4)     /* call out of order (e.g. step before set) */
#define GRAINS_EOVERFLOW (-5)  /* a fixed capacity was exceeded            */
#define GRAINS_EUNSUPPORTED (-6)

/* ---- convex kinds: numbering of ConvexType, Grains/Geometry/include/Convex.hh:7-16 */
#define GRAINS_SPHERE 0
#define GRAINS_BOX 1
#define GRAINS_CYLINDER 2      /* axis y, y in [-h/2, h/2] (Cylinder.cpp)    */
#define GRAINS_CONE 3          /* axis y, origin at the centroid: apex +3h/4,
                                  base -h/4 (Cone.cpp)                         */
#define GRAINS_SUPERQUADRIC 4
#define GRAINS_POLYHEDRON 5    /* enum value exists in the reference, class does not */
#define GRAINS_RECTANGLE 6

/* ---- arithmetic of the narrow phase and force ---------------------------- */
#define GRAINS_FP64 0          /* plain: everything in FP64                  */
#define GRAINS_FP32_MIXED 1    /* GJK, support maps, forces in FP32; FP64
                                  state, accumulators, cell keys, obstacle
                                  contacts, and an FP64 re-run of GJK near
                                  degenerate simplices and of every contact
                                  decision within FP32's rounding band      */

/* ---- semantics flags (grains_config_t.flags) ---------------------------- */
/* Reproduce the reference narrow phase exactly: GJK_JH with its early exit
 * on mu < 1e-4*LOWEPS (GJK_JH.cpp:370-372), no crust core
 * (CollisionDetection.cpp:231-236 commented out), and the relative velocity
 * taken with the world contact point as lever arm
 * (ComponentManagerCPU.cpp:404-407, Kinematics.cpp:86-91).  Without it the
 * "physics" semantics apply: GJK on the crust cores with the standard
 * van den Bergen termination and the lever arm cp - x_i. */
#define GRAINS_REF_QUIRKS 0x1u
/* Nesterov-accelerated support directions in GJK (physics semantics only). */
#define GRAINS_NESTEROV 0x2u
/* FP32-mixed, physics semantics: every GJK search of a particle pair starts
 * from that pair's search direction of the previous step (kept on the device
 * per (particle, candidate slot): 32 B x max_neighbors per particle).  A
 * resting or slowly moving pair then ends after one support pair.  Results
 * meet the same gap test as cold searches but depend on the previous step:
 * grains_set_state, grains_set_transforms and grains_restore start cold,
 * so a restored run differs from an uninterrupted one in the last bits.
 * Ignored under GRAINS_FP64 and GRAINS_REF_QUIRKS; the adjoint rejects it. */
#define GRAINS_WARM_START 0x4u
/* FP32-mixed: every entry the FP32 pass finds in contact is re-run in FP64
 * (GJK to gjk_rel_tol_fp64, contact geometry and Hooke force), as the
 * entries near the contact threshold are.  The FP32 pair frame resolves a
 * support point to ~2^-24 of the pair's size (~1e-10 m for mm grains), and
 * an overlap of ~1e-6 m then carries ~1e-4 relative error in its force;
 * with this flag contact forces carry FP64 geometry, while separation
 * decisions, the broad phase and the screening stay in FP32.  Costs one
 * FP64 search per contact per step.  Ignored under GRAINS_FP64. */
#define GRAINS_FP64_CONTACTS 0x8u

/* ---- time integration (grains_config_t.integrator) ------------------------ */
/* FirstOrderExplicit::Move (FirstOrderExplicit.cpp:46-60): x += dt v,
 * v += dt a, rotation by w over dt, w += dt alpha. */
#define GRAINS_FIRST_ORDER_EXPLICIT 0
/* The three further names TimeIntegratorBuilderFactory.cpp:45-49 lists (the
 * reference implements none of them).  Same Move interface; a = F/m and
 * alpha from computeMomentum at the step's start:
 *  SECOND_ORDER_EXPLICIT  x += dt v + dt^2/2 a, rotation by w + dt/2 alpha,
 *                         v += dt a, w += dt alpha: exact under constant
 *                         accelerations, first order in general;
 *  SECOND_ORDER_LEAPFROG  velocities live at half steps: v += dt a (dt/2 on
 *                         the first step after grains_set_state), then
 *                         x += dt v (the new v), rotation by the new w;
 *                         second order for forces of the positions only;
 *  SECOND_ORDER_ADAMS_BASHFORTH  two-step: x += dt (3/2 v - 1/2 v_prev),
 *                         v += dt (3/2 a - 1/2 a_prev), rotation by
 *                         3/2 w - 1/2 w_prev; the first step after
 *                         grains_set_state (no history) is first order;
 *                         second order. */
#define GRAINS_SECOND_ORDER_EXPLICIT 1
#define GRAINS_SECOND_ORDER_LEAPFROG 2
#define GRAINS_SECOND_ORDER_ADAMS_BASHFORTH 3

/* ---- pair lists ----------------------------------------------------------- */
#define GRAINS_PAIRS_CANDIDATE 0 /* passed the bounding-sphere prefilter     */
#define GRAINS_PAIRS_CONTACT 1   /* overlap distance < 0                     */

/* One particle or obstacle shape, the data of RigidBody<T,T>
 * (Grains/Geometry/src/RigidBody.cpp:19-59) plus its Convex. */
typedef struct grains_shape_t {
  int32_t kind;          /* GRAINS_SPHERE ... GRAINS_RECTANGLE                */
  int32_t material;      /* material id; contact table index via computeHash  */
  double dims[5];        /* SPHERE r | BOX ex,ey,ez (half) | SUPERQUADRIC
                            a,b,c,n1,n2 | RECTANGLE LX,LY (half) | CYLINDER
                            r,h | CONE r,h (full height, as Cylinder(r, h),
                            Cone(r, h))                                      */
  double crust;          /* CrustThickness                                    */
  double density;        /* 0 gives mass 0 (obstacles)                        */
  int32_t n_vertices;    /* POLYHEDRON: vertex count (convex hull points)     */
  int32_t vertex_offset; /* POLYHEDRON: first (x,y,z) triplet in the array
                            passed to grains_set_shapes                      */
} grains_shape_t;

/* Hooke parameters of one material pair, HookeContactForceModel ctor
 * (Grains/Component/src/HookeContactForceModel.cpp:48-57). */
typedef struct grains_hooke_t {
  double kn, en, etat, muc, kr;
} grains_hooke_t;

/* One independent simulation (a LinkedCell domain plus its forces).
 * Several of them run batched in one context. */
typedef struct grains_sim_t {
  double domain_min[3];     /* Origin OX,OY,OZ (Grains.cpp:114-120)         */
  double domain_max[3];     /* LinkedCell MX,MY,MZ (Grains.cpp:108-112)      */
  double cell_size;         /* > 0: explicit cell extent; 0: derived as
                               max(1,CellSizeFactor) * 2 * max R_c
                               (Grains.cpp:226-245)                          */
  double cell_size_factor;  /* CellSizeFactor                                */
  double gravity[3];        /* Forces/Gravity (Grains.cpp:305-336)           */
  int32_t periodic;         /* bitmask 1 x, 2 y, 4 z: periodic directions
                               (not in the reference: Grains.cpp:129-133
                               aborts); each needs >= 3 cells               */
  int32_t contact_table;    /* which table block of grains_set_contact_tables */
} grains_sim_t;

typedef struct grains_config_t {
  double dt;                /* TimeInterval dt                               */
  int32_t precision;        /* GRAINS_FP64 | GRAINS_FP32_MIXED               */
  uint32_t flags;           /* GRAINS_REF_QUIRKS | GRAINS_NESTEROV           */
  double gjk_rel_tol;       /* 0: LOWEPS of the precision (Basic.hh:126-128) */
  int32_t max_neighbors;    /* candidate capacity per particle, 0: 48        */
  int32_t block_size;       /* threads per block of the per-particle and
                               per-entry kernels: 64, 128 or 256 (0: 256)    */
  int32_t narrow_blocks_per_cu; /* resident blocks per CU of the persistent
                               narrow-phase launch, in [1, 64] (0: 8;
                               above 64: GRAINS_EINVAL)                     */
  int32_t narrow_passes;    /* 2 = a screening pass over every entry (bounding
                               sphere, OBB and, physics semantics, GJK's first
                               support pair) and a complete pass over the
                               undecided entries, compacted; 1 = one complete
                               pass over the entries that pass the prefilter
                               (0: 2; REF_QUIRKS in FP32 and FP64 beds of
                               spheres take one).  Results do not depend on
                               it.                                          */
  int32_t candidate_staging; /* broad phase: 1 = each unordered pair tested
                               once (the residents after it in its cell and
                               13 of the 26 neighbour cells), by cell, dense
                               cells shared among several lane groups, when
                               every periodic axis has at least 3 cells,
                               else as 3; 3 = every lane reads its
                               neighbours' records from global memory and
                               tests from both particles of every pair, as
                               the reference's loop visits them; 2 = a block
                               first stages its neighbour windows in LDS;
                               0 = 1 where it applies, else 2 when particles
                               outnumber cells 8 to 1, else 3.  Results do
                               not depend on it.                            */
  int32_t integrator;       /* GRAINS_FIRST_ORDER_EXPLICIT (0, the reference's
                               only scheme) or a second-order scheme below  */
  double gjk_rel_tol_fp64;  /* GRAINS_FP32_MIXED: GJK tolerance of the FP64
                               re-runs (0: 1e-10).  Every pair whose FP32
                               contact decision lies within FP32's rounding
                               of the threshold is re-run in FP64; with the
                               FP64 path's tolerance here its contact
                               decisions equal that path's. */
} grains_config_t;

/* Counters of the last grains_step call (summed over its steps). */
typedef struct grains_stats_t {
  uint64_t steps;
  uint64_t candidate_pairs;   /* ordered pairs passing the prefilter          */
  uint64_t gjk_calls;         /* ordered pairs that ran GJK                   */
  uint64_t gjk_iterations;    /* summed GJK iterations (the support pair that
                                 proves a separation is not counted)          */
  uint64_t contacts;          /* ordered particle-particle contacts           */
  uint64_t wall_contacts;     /* particle-obstacle contacts                   */
  uint64_t out_of_domain;     /* particle-steps whose centre left the grid    */
  uint64_t deep_contacts;     /* physics semantics: crust cores overlapped    */
  uint64_t fp64_refines;      /* FP32-mixed: GJK re-run in FP64               */
  uint64_t neighbor_overflow; /* candidates dropped: capacity exceeded         */
  uint32_t max_candidates;    /* largest per-particle candidate count seen    */
  uint32_t sort_passes;       /* radix passes a sort of the reference's cells takes */
  double   elapsed_ms;        /* device time of the last grains_step call      */
  uint64_t narrow_deferred;   /* entries the screening pass queued for the
                                 complete narrow pass                          */
  uint64_t gjk_max_iterations; /* the longest GJK search                       */
  uint64_t fp64_near_refines; /* FP32-mixed: entries re-run in FP64 because
                                 their contact decision lay within FP32's
                                 rounding of the threshold (included in
                                 fp64_refines)                                */
  uint64_t nonfinite_states;  /* particle-steps that ended with a NaN or
                                 infinity in the position, orientation or
                                 velocities (the reference carries them on
                                 silently)                                    */
  uint64_t fp64_refine_iterations;     /* FP32-mixed: GJK iterations of the
                                          FP64 re-runs                       */
  uint64_t fp64_refine_max_iterations; /* the longest FP64 re-run            */
} grains_stats_t;

typedef struct grains_ctx grains_ctx_t;

/* Context ---------------------------------------------------------------- */
/* Replaces GrainsGPU::initialize/setupGPUDevice (Grains/Base/src/GrainsGPU.cpp:27-85).
 * The environment variable GRAINS_SMALL_SORT_MAX (read when a layout is
 * built) sets the largest bed whose cell sort runs in one block instead of
 * the radix passes and the merge (default 1024, at most 8192; 0: never).
 * Results do not depend on it. */
int grains_create(const grains_config_t* cfg, grains_ctx_t** out);
void grains_destroy(grains_ctx_t* ctx);
const char* grains_last_error(const grains_ctx_t* ctx);
/* Library version string, e.g. "grains_hip 0.1 gfx950". */
const char* grains_version(void);

/* Scene ------------------------------------------------------------------ */
/* Shapes: RigidBody table (Grains.cpp:164-218, RigidBodyGPUWrapper.cpp:20-181).
 * `vertices` holds (x,y,z) triplets for POLYHEDRON shapes, may be NULL. */
int grains_set_shapes(grains_ctx_t* ctx, const grains_shape_t* shapes,
                      uint32_t n_shapes, const double* vertices,
                      uint32_t n_vertices);
/* Contact table blocks, each n_materials*(n_materials+1)/2 entries indexed by
 * ContactForceModelBuilderFactory::computeHash(matA, matB) = l(l+1)/2 + s
 * (Grains/Component/src/ContactForceModelBuilderFactory.cpp:77-83). */
int grains_set_contact_tables(grains_ctx_t* ctx, const grains_hooke_t* tables,
                              uint32_t n_materials, uint32_t n_tables);
/* Simulations (LinkedCell<T> ctor, Grains/Component/src/LinkedCell.cpp:16-73). */
int grains_set_sims(grains_ctx_t* ctx, const grains_sim_t* sims, uint32_t n_sims);
/* Obstacles: ComponentManager::initializeObstacles (ComponentManagerCPU.cpp:215-231).
 * `transforms` is n x 12 (Transform3 buffer). `sim` may be NULL (all sim 0). */
int grains_set_obstacles(grains_ctx_t* ctx, const uint32_t* shape,
                         const uint32_t* sim, const double* transforms,
                         uint32_t n_obstacles);
/* Particles: ComponentManager::initializeParticles (ComponentManagerCPU.cpp:236-252).
 * Particles of one sim must be contiguous and sims in ascending order.
 * `sim` may be NULL (all sim 0).  Resets the state to rest at the origin. */
int grains_set_particles(grains_ctx_t* ctx, const uint32_t* shape,
                         const uint32_t* sim, uint64_t n);

/* State ------------------------------------------------------------------ */
/* pos n x 3, quat n x 4 (x,y,z,w), vel n x 3, omega n x 3; NULL = unchanged. */
int grains_set_state(grains_ctx_t* ctx, const double* pos, const double* quat,
                     const double* vel, const double* omega, uint64_t n);
int grains_get_state(grains_ctx_t* ctx, double* pos, double* quat, double* vel,
                     double* omega, uint64_t n);
/* ComponentManager::setTransform/getTransform (ComponentManager.hh:46,85):
 * n x 12 Transform3 buffers. */
int grains_set_transforms(grains_ctx_t* ctx, const double* transforms, uint64_t n);
int grains_get_transforms(grains_ctx_t* ctx, double* transforms, uint64_t n);

/* Launch shape of the per-particle / per-entry kernels (block_size 64, 128
 * or 256; narrow_blocks_per_cu in [1, 64]), changeable between steps; used by the
 * autotuner.  No counterpart in the reference (its kernels hard-code 256,
 * ComponentManagerGPU.cpp:265-352). */
int grains_set_launch(grains_ctx_t* ctx, int block_size, int narrow_blocks_per_cu);
/* Passes of the narrow phase (1 or 2, see grains_config_t.narrow_passes),
 * changeable between steps; used by the autotuner.  No counterpart in the
 * reference (one pass, one lane per pair, ComponentManagerGPU_Kernels.cpp:141-226). */
int grains_set_narrow_passes(grains_ctx_t* ctx, int passes);
/* Candidate search mode (0 to 3, see grains_config_t.candidate_staging),
 * changeable between steps; used by the autotuner.  No counterpart in the
 * reference (its particle loop reads every neighbour through the cell lists,
 * ComponentManagerCPU.cpp:364-421). */
int grains_set_candidate_staging(grains_ctx_t* ctx, int mode);

/* Time stepping ------------------------------------------------------------ */
/* n_steps iterations of the GrainsCPU::simulate loop body
 * (Grains/Base/src/GrainsCPU.cpp:55-66): detectCollisionAndComputeContactForces,
 * addExternalForces, moveParticles. */
int grains_step(grains_ctx_t* ctx, uint32_t n_steps);
/* Same, replayed from captured HIP graphs: one of grains_set_graph_steps
 * steps (default 1), launched n_steps / that many times, and one of one step
 * for the rest (and for every step while the adjoint records).  Results equal
 * grains_step's bit for bit. */
int grains_step_graph(grains_ctx_t* ctx, uint32_t n_steps);
/* Steps captured in one graph by grains_step_graph, in [1, 1000] (capturing
 * k steps takes k times one step's graph nodes, ~20 each); a change drops the
 * captured graph.  No counterpart in the reference (GrainsGPU.cpp:118-140
 * launches every kernel of every step from the host). */
int grains_set_graph_steps(grains_ctx_t* ctx, uint32_t steps);

/* Results of the most recent step's broad and narrow phase ------------------ */
/* keys[i]: linear cell hash of particle i (LinkedCell::computeLinearCellHash,
 * LinkedCell.cpp:117-149; offset by the sim's first cell when batched).
 * sorted[k]: stable (key, index) order.  Either pointer may be NULL. */
int grains_get_cell_keys(grains_ctx_t* ctx, uint32_t* keys, uint32_t* sorted, uint64_t n);
/* Pairs (i, j) as 2*m uint32, ordered by i then by the reference visiting
 * order (27 cells k,j,i outer->inner, residents ascending; ComponentManagerCPU.cpp:364-421).
 * *m receives the total count; at most `cap` pairs are written. */
int grains_get_pairs(grains_ctx_t* ctx, int which, uint32_t* ij, uint64_t cap, uint64_t* m);
/* Cumulative per-particle contact counts, the `result` array of
 * detectCollisionAndComputeContactForcesParticles (ComponentManagerCPU.cpp:419). */
int grains_get_contact_count(grains_ctx_t* ctx, int32_t* counts, uint64_t n);
int grains_reset_contact_count(grains_ctx_t* ctx);
/* Torce (force, torque) accumulated by the last step before the integrator
 * reset it (ComponentManagerCPU.cpp:428-460, 483). n x 3 each. */
int grains_get_torce(grains_ctx_t* ctx, double* force, double* torque, uint64_t n);
int grains_get_stats(grains_ctx_t* ctx, grains_stats_t* stats);

/* Per-phase device time of the steps run while profiling is on: HIP events
 * on the context's stream around each kernel group, summed over the steps
 * of the last grains_step call.  Phases, in order: cell hash, radix sort,
 * cell ranges + sorted records, candidates, scan + expand (these five: the
 * neighbour lists' builds, each serving the steps until a particle has moved
 * half the lists' skin), narrow phase + force (first pass), narrow phase of
 * the deferred entries (second pass), FP64 re-run, reduction + walls +
 * integration. */
#define GRAINS_NUM_PHASES 9
int grains_set_profiling(grains_ctx_t* ctx, int on);
int grains_get_phase_times(grains_ctx_t* ctx, double* ms, int n_phases);

/* Differentiation ------------------------------------------------------------
 * No counterpart in the reference.  Reverse-mode gradients of a trajectory
 * with respect to the contact-table parameters, for the physics semantics,
 * spheres and ellipsoids (superquadrics n1 = n2 = 2), Rectangle walls and
 * kr = 0.  The contact set of every step is the one the forward step finds
 * (held fixed within the step); contact geometry, Hooke force and
 * integration are differentiated exactly (separated crust cores by implicit
 * differentiation of the closest-point conditions).
 * grains_adjoint_record starts a trajectory at the current state and keeps a
 * checkpoint every `checkpoint_every` steps of the following grains_step /
 * grains_step_graph calls, and the states of the steps between while they
 * take no more than 4 GiB (104 B per particle and step) and the device has
 * them (they are freed when a checkpoint or the sweep finds no memory).
 * grains_adjoint then sweeps back over every recorded step, first
 * re-running from its checkpoint a block whose states were not kept:
 * dL_dstate (13 n: pos n x 3, quat n x 4, vel n x 3, omega n x 3, the
 * gradient of the loss at the current state) -> dL_dparams (n_table_entries
 * x 4: kn, en, etat, muc, in the order of grains_set_contact_tables) and,
 * when not NULL, dL_dstate0 (13 n, the gradient with respect to the recorded
 * initial state).  The current state is left as it was. */
int grains_adjoint_record(grains_ctx_t* ctx, uint32_t checkpoint_every);
int grains_adjoint(grains_ctx_t* ctx, const double* dL_dstate, double* dL_dparams, double* dL_dstate0);

/* Narrow phase alone ------------------------------------------------------- */
/* GJK distance between shape_a[k] at transform ta[k] and shape_b[k] at tb[k]
 * (12-double Transform3 buffers), the GrainsTestDev microbenchmark
 * (Grains/Base/src/GrainsTestDev.cpp:35-55, 168-185) calling
 * computeClosestPoints_GJK_JH (GJK_JH.cpp:310-391).  Returns distance, the
 * witness points in world coordinates (may be NULL) and iteration counts
 * (may be NULL).  Honours precision, REF_QUIRKS and NESTEROV of the context;
 * shapes are the full shapes (no crust core).  The kernel's device time is
 * left in grains_stats_t.elapsed_ms. */
int grains_gjk_batch(grains_ctx_t* ctx, const uint32_t* shape_a,
                     const uint32_t* shape_b, const double* ta,
                     const double* tb, uint64_t n, double* dist, double* pa,
                     double* pb, int32_t* iters);
/* Device-resident variant for timing: all pointers are device pointers; the
 * call comes after what is on the device's default stream. */
int grains_gjk_batch_device(grains_ctx_t* ctx, const uint32_t* shape_a_device,
                            const uint32_t* shape_b_device, const double* ta_device,
                            const double* tb_device, uint64_t n,
                            double* dist_device, int32_t* iters_device,
                            float* elapsed_ms);
/* grains_gjk_batch_device that allocates nothing: no counterpart in the
 * reference; for callers that cannot allocate device memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc).  Up
 * to eight shapes without polyhedra go as kernel arguments; larger sets' tables
 * are copied into a fixed 1 MiB device array that
 * the library holds on each GPU until the process ends (at most ~6,500
 * shapes in FP64, ~10,900 in FP32, fewer with polyhedron vertices; larger
 * sets return GRAINS_EINVAL).  Results equal grains_gjk_batch_device's.
 * Every call on one GPU shares that array: calls that overlap on one GPU
 * (several threads or contexts) race.  Shape indices must be < the number
 * of shapes (device memory: not checked).  n = 0 returns at once. */
int grains_gjk_batch_device_noalloc(grains_ctx_t* ctx, const uint32_t* shape_a_device,
                                    const uint32_t* shape_b_device, const double* ta_device,
                                    const double* tb_device, uint64_t n,
                                    double* dist_device, int32_t* iters_device,
                                    float* elapsed_ms);

/* Checkpoint / restore of the particle state (pos, quat, vel, omega, contact
 * counts).  `bytes` = NULL with *size queries the size. */
int grains_snapshot(grains_ctx_t* ctx, void* bytes, size_t* size);
int grains_restore(grains_ctx_t* ctx, const void* bytes, size_t size);

#ifdef __cplusplus
}
#endif

#endif /* GRAINS_HIP_H */
