/*
 * ggx.h -- C-ABI of libggx, the MI355X-native per-grain level-set timestep of GraGLeS2D.
 *
 * The reference has no plugin API: its timestep is the body of grainhdl::run_sim
 * (src/grainhdl.cpp:1049-1141), a sequence of OpenMP phase loops that call one LSbox method
 * per grain (src/box.h:124-191).  libggx replaces that loop body.  The retained driver
 * (settings, microstructure input, output writers) stays on the host; one ggx_step() call
 * performs what the phase loops switchDistancebuffer / convolution / updateSecondOrderNeighbors /
 * comparison_box / level_set / redistancing do for every grain, on the GPU.
 *
 * Conventions: plain C types only; every function returns a status code (GGX_OK == 0 or a
 * negative GGX_E_*); no exceptions cross the ABI; host buffers passed in are caller-owned and
 * copied; ggx_last_error() describes the last failure of a context.
 */
#ifndef GGX_H
#define GGX_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define GGX_OK        0
#define GGX_E_CONFIG (-1)   /* invalid settings (reference: exit(2), Settings.cpp:88-108) */
#define GGX_E_HIP    (-2)   /* a HIP runtime call failed */
#define GGX_E_OOM    (-3)   /* device arena or host allocation exhausted */
#define GGX_E_BOUNDS (-4)   /* an index left its buffer (reference: std::out_of_range) */
#define GGX_E_STATE  (-5)   /* call out of order (e.g. step before load) */
#define GGX_E_ARG    (-6)   /* bad argument */
#define GGX_E_IO     (-7)   /* file could not be read or written */

/* ---------------------------------------------------------------------------------------
 * Settings: the parameters.xml keys the timestep reads (Settings.h:69-121,
 * Settings::initializeParameters, src/Settings.cpp:84-289).
 * ------------------------------------------------------------------------------------- */
typedef struct ggx_settings {
    int32_t start_time;                /* StartTime */
    int32_t number_of_particles;       /* NumberOfParticles */
    int32_t number_of_points_per_grain;/* NumberOfPointsPerGrain */
    int32_t number_of_timesteps;       /* NumberOfTimesteps */
    int32_t breakup_number;            /* BreakupNumber */
    int32_t analysis_timestep;         /* AnalysisTimestep */
    int32_t plot_interval;             /* PlotInterval */
    int32_t discrete_sampling_rate;    /* DiscreteSamplingRate */
    int32_t domain_border_size;        /* DomainBorderSize (grid_blowup) */
    int32_t microstructure_gen_mode;   /* MicrostructureGenMode (0 = read from file) */
    int32_t lattice_type;              /* LatticeType (0 cubic) */
    int32_t use_mobility_model;        /* UseMobilityModel */
    int32_t identify_twins;            /* IdentifyTwins */
    int32_t use_magnetic_field;        /* UseMagneticField */
    int32_t is_isotropic_network;      /* IsIsotropicNetwork */
    int32_t use_texture;               /* UseTexture */
    int32_t execute_in_parallel;       /* ExecuteInParallel */
    int32_t maximum_number_of_threads; /* MaximumNumberOfThreads */
    int32_t grid_coarsement;           /* GridCoarsement */
    int32_t convolution_mode;          /* ConvolutionMode: 0 Laplace, 1 Richardson, 2 Gaussian */
    int32_t research_mode;             /* ResearchMode */
    int32_t research_project;          /* ResearchProject */
    int32_t neighbour_tracking;        /* NeighbourTracking */
    int32_t use_stored_elastic_energy; /* UseStoredElasticEnergy */
    int32_t grain_scheduler;           /* GrainScheduler */
    int32_t decouple_grains;           /* DecoupleGrains */
    int32_t user_def_number_of_points_per_grain; /* UserDefNumberOfPointsPerGrain */
    double  hagb_mobility;             /* HAGB_Mobility */
    double  hagb_energy;               /* HAGB_Energy */
    double  physical_domain_size;      /* Physical_Domain_Size */
    double  triple_point_drag;         /* TriplePointDrag */
    double  disloc_en_per_m;           /* DislocEnPerM */
    double  max_misorientation;        /* MaxMisOrientation */
    double  grid_coarsement_gradient;  /* GridCoarsementGradient */
    double  constant_sector_radius;    /* ConstantSectorRadius (grid points, as read) */
    double  interpolating_sector_radius; /* InterpolatingSectorRadius (grid points, as read) */
    double  gaussian_kernel_time_slope;/* GaussianKernelUserDefTimeSlope */
    double  box_default_stored_elastic_energy; /* BoxDefaultStoredElasticEnergy */
    char    read_from_filename[512];   /* ReadFromFilename */
    char    additional_filename[512];  /* AdditionalFilename */
} ggx_settings;

/* Reference defaults of the static Settings fields (src/Settings.cpp:29-80). */
int ggx_settings_default(ggx_settings* s);
/* Settings::initializeParameters (src/Settings.cpp:84-289): same keys, same parsing. */
int ggx_settings_read_xml(const char* path, ggx_settings* s);
/* Settings::generateXMLParametersNode + grainhdl::createParamsForSim
 * (src/Settings.cpp:363-400, src/grainhdl.cpp:1205-1223). */
int ggx_settings_write_xml(const char* path, const ggx_settings* s, const char* network_file,
                           int32_t loop, int32_t grains);

/* Derived simulation constants, grainhdl::setSimulationParameter (src/grainhdl.cpp:56-136)
 * and find_correctTimestepSize (250-274) for MicrostructureGenMode 0. */
typedef struct ggx_derived {
    int32_t real_domain_size;  /* R */
    int32_t ngridpoints;       /* R + 2 grid_blowup */
    int32_t grid_blowup;
    double  h, dt, delta, time_slope, ds;
} ggx_derived;
int ggx_settings_derive(const ggx_settings* s, ggx_derived* d);

/* ---------------------------------------------------------------------------------------
 * Microstructure: the mode-0 network file (grainhdl::readMicrostructure,
 * src/grainhdl.cpp:605-661; writer LSbox::plot_full_grain, src/box.cpp:1552-1596).
 * ------------------------------------------------------------------------------------- */
typedef struct ggx_network ggx_network;

/* Seeded microstructure: Voronoi (lognormal_sigma == 0) or power diagram with lognormal
 * weights, uniform seed points in [0,1)^2 and Shoemake-uniform orientations.  Stands in for
 * grainhdl::VOROMicrostructure (src/grainhdl.cpp:513-603), whose rand()/voro++ path is not
 * reproducible.  Polygons are closed (first vertex repeated last). */
int  ggx_network_generate(int32_t n, uint64_t seed, double lognormal_sigma, ggx_network** out);
int  ggx_network_read(const char* path, int32_t ngrains, ggx_network** out);
int  ggx_network_write(const char* path, const ggx_network* net);
int  ggx_network_count(const ggx_network* net);
/* View of grain `idx` (0-based): its ID, vertex count and pointers valid until the network is
 * freed. */
int  ggx_network_grain(const ggx_network* net, int32_t idx, int32_t* id, int32_t* nverts,
                       const double** xy, const double** quat);
int  ggx_network_add(ggx_network* net, int32_t id, int32_t nverts, const double* xy,
                     const double* quat);
int  ggx_network_new(ggx_network** out);
/* grainhdl::find_neighbors (src/grainhdl.cpp:1258-1283) with LSbox::computeDirectNeighbours
 * (src/box.cpp:2220-2237) on the host, without a device: the initial comparison list of every
 * grain in the reference's R-tree order.  counts[id] (count_cap >= max id + 1 entries) and
 * ids[id * list_cap + k].  Returns max id + 1 or a negative status. */
int  ggx_network_neighbours(const ggx_network* net, const ggx_settings* s, int32_t* counts, int32_t* ids,
                            int32_t count_cap, int32_t list_cap);
void ggx_network_free(ggx_network* net);

/* ---------------------------------------------------------------------------------------
 * Device context.
 * ------------------------------------------------------------------------------------- */
typedef struct ggx_ctx ggx_ctx;

#define GGX_PREC_FP64 0
#define GGX_PREC_FP32 1

#define GGX_BATCH_FUSED    0  /* all grains per launch (the batched step) */
#define GGX_BATCH_PERGRAIN 1  /* one launch per grain per kernel (the per-grain baseline) */

#define GGX_CONV_AUTO      0  /* the engine chosen per box size (GGX_CONV_FFT for ConvolutionMode 0 and 1) */
#define GGX_CONV_CIRCULANT 1  /* exact dense circulant, K_n phi K_n (real space; the separable Gaussian only) */
#define GGX_CONV_FFT       2  /* by transforms, any n, every ConvolutionMode: products with the real transform
                                 matrix (FP64), mixed-radix FFT (FP32, or a small lds_budget) */

typedef struct ggx_options {
    int32_t precision;        /* GGX_PREC_* */
    int32_t batching;         /* GGX_BATCH_* */
    int32_t conv_engine;      /* GGX_CONV_* */
    int32_t device;           /* HIP device ordinal */
    int32_t lds_budget;       /* bytes of LDS a workgroup may use; 0 = device maximum */
    int32_t use_graph;        /* 1: each step is captured once per buffer parity as a hipGraph and
                                 replayed (needs persistent = 1 and batched launches) */
    int32_t persistent;       /* 1: fixed grids pull grains from device work lists (no host sync);
                                 0: one workgroup per grain, counts read back after scheduling */
    double  arena_headroom;   /* arena capacity = headroom * initial sum of box areas (> 0).  Below
                                 1.0 the network loads but a step's output cannot fit: grains that
                                 find no room leave the step, GGX_E_BOUNDS is reported (for tests) */
    int32_t bucket_edges[16]; /* box-size buckets: ascending upper edges, the last one 512, the rest
                                 0; all 0 = the built-in table (24 32 40 48 56 64 96 128 192 256 512).
                                 Written by the autotuner (gragles2d_amd/autotune.py) */
    int32_t fft_buckets;      /* GGX_CONV_AUTO with ConvolutionMode 2: bit b set = bucket b
                                 convolves by FFT instead of the circulant (autotuner) */
} ggx_options;
int ggx_options_default(ggx_options* o);

/* Replaces grainhdl::setSimulationParameter's context set-up (grainhdl.cpp:56-136). */
int ggx_create(const ggx_settings* s, const ggx_options* o, ggx_ctx** out);
void ggx_destroy(ggx_ctx* ctx);
const char* ggx_last_error(const ggx_ctx* ctx);  /* NULL: the calling thread's last context-free failure */

/* Builds every grain (LSbox file constructor, box.cpp:108-158), its initial signed distance
 * (LSbox::calculateDistanceFunction, box.cpp:318-402) and the initial neighbour lists
 * (grainhdl::find_neighbors, grainhdl.cpp:1258-1283), then uploads them to the device arena. */
int ggx_load_network(ggx_ctx* ctx, const ggx_network* net);

/* Runs `nsteps` passes of the run_sim loop body (grainhdl.cpp:1049-1141): per grain
 * LSbox::executeConvolution (box.cpp:408-536), computeSecondOrderNeighbours (1027-1068),
 * executeComparison (890-943), executeSetComparison (838-879), extractContour (1089-1153),
 * computeVolumeAndEnergy (1201-1228), executeRedistancing (1259-1399), with the buffer
 * switches of switchInNOut (826-832).  The loop index advances by one per step. */
int ggx_step(ggx_ctx* ctx, int32_t nsteps);
/* Blocks until queued device work is done; returns the first deferred device error. */
int ggx_sync(ggx_ctx* ctx);
/* Current loop index (the next step runs with this `loop`). */
int ggx_loop(const ggx_ctx* ctx);
/* Grid constants in force (they change when the grid coarsens: grainhdl::gridCoarsement,
 * grainhdl.cpp:1396-1477, run before a step whose grain count has fallen below
 * GridCoarsementGradient of the count at the last coarsening).  Returns the number of
 * coarsenings so far. */
int ggx_get_grid(const ggx_ctx* ctx, ggx_derived* out);
/* grainhdl::get_biggestGrainVol currentNrGrains (grainhdl.cpp:1744-1754). */
int ggx_current_grains(ggx_ctx* ctx);
int ggx_max_id(const ggx_ctx* ctx);

/* Per-grain state after the last step (LSbox fields, box.h:71-96). */
typedef struct ggx_grain_info {
    int32_t present;              /* grains[id] != NULL */
    int32_t exists;               /* LSbox::grainExists() */
    int32_t motion_regular;       /* LSbox::isMotionRegular() */
    int32_t intersects_boundary;  /* LSbox::intersectsBoundaryGrain() */
    int32_t xmin, xmax, ymin, ymax;             /* getMinX()..getMaxY() (output buffer) */
    int32_t id_xmin, id_xmax, id_ymin, id_ymax; /* bounds of m_IDLocal */
    int32_t contour_len;          /* m_grainBoundary.getBoundarySegmentCount() */
    int32_t n_neighbours;         /* getDirectNeighbourCount() */
    int32_t n_compare;            /* comparison-list length */
    int32_t error;                /* non-zero: the reference would have aborted */
    double  volume, perimeter, energy, mean_da;  /* getVolume(), getPerimeter(), ... */
} ggx_grain_info;

int ggx_get_info(ggx_ctx* ctx, int32_t id, ggx_grain_info* out);
/* Bulk copy of every grain's info, out[id] for id in [0, max_id] (out[0] is the boundary). */
int ggx_get_info_all(ggx_ctx* ctx, ggx_grain_info* out, int32_t count);
/* Signed distance of grain `id` on its box, row-major (row = y), widened to double for the
 * FP32 path.  Returns the element count or a negative status. */
int ggx_get_phi(ggx_ctx* ctx, int32_t id, double* out, int32_t cap);
/* m_IDLocal of grain `id` (its full flat vector). */
int ggx_get_idlocal(ggx_ctx* ctx, int32_t id, uint32_t* out, int32_t cap);
/* Ordered contour (x, y pairs, grid-index units) -- m_grainBoundary.getRawBoundary(). */
int ggx_get_contour(ggx_ctx* ctx, int32_t id, double* xy, int32_t cap_points);
/* getDirectNeighbourIDs() / getGBLengths() (box.cpp:2212-2218), first-encounter order. */
int ggx_get_neighbours(ggx_ctx* ctx, int32_t id, int32_t* ids, double* lengths, int32_t cap);
/* Comparison list in list order (LSbox::m_comparisonList). */
int ggx_get_compare_list(ggx_ctx* ctx, int32_t id, int32_t* ids, int32_t cap);

/* Anisotropic networks (IsIsotropicNetwork = 0).
 * Per direct neighbour, in the order of ggx_get_neighbours: energy density and mobility of the
 * boundary (characteristics::energyDensity / mobility set by buildDirectNeighbours,
 * grainBoundary.cpp:169-192; the initial lists carry 0, grainBoundary.h:68). */
int ggx_get_neighbour_props(ggx_ctx* ctx, int32_t id, double* energy, double* mobility, int32_t cap);
/* Junctions of the grain's last contour (m_grainJunctions: generateJunction,
 * marchingSquares.cpp:266-301, projected by extractBoundaryAndJunctions,
 * grainBoundary.cpp:50-61), in walk order: 6 ints each (order, contour segment, grains[4], unused
 * entries 0xFFFFFF) and 3 doubles (x, y on the contour, lambda).  Returns the count. */
int ggx_get_junctions(ggx_ctx* ctx, int32_t id, int32_t* ints, double* dbls, int32_t cap);
/* UseMobilityModel 4 (no counterpart in the reference; the nearest hook is LSbox::GBmobilityModel,
 * box.cpp:1825-1865): the mobility of each of 16 misorientation bins of 62.8/16 degrees.  All
 * bins 1.0 (the default) reproduce UseMobilityModel 0 when TriplePointDrag is 0.  On a loaded
 * network the recorded boundary mobilities (those with an energy) take their bin's new value. */
int ggx_set_mobility_bins(ggx_ctx* ctx, const double* bins16);

/* The adjoint of one step with respect to the 16 mobility bins (no counterpart in the reference;
 * it differentiates the corrector of LSbox::executeConvolution, box.cpp:452-510, the comparison
 * and set comparison, box.cpp:838-943, and the area and perimeter of the contour,
 * grainBoundary.cpp:201-231).  ggx_record_next_step arms the next ggx_step to keep what the
 * adjoint reads; ggx_step_adjoint then takes dJ/d(area) and dJ/d(perimeter) of every grain after
 * that step (arrays indexed by grain id, ggx_max_id + 1 entries) and returns dJ/d(bin) in
 * grad16.  The state entering the step is held (redistancing is a stop-gradient), recorded
 * boundary mobilities count as functions of their bins, and the step's discrete decisions stay
 * as recorded.  FP64 batched steps of anisotropic networks with UseMobilityModel 4, ResearchMode
 * 0 and no grid coarsening (GGX_E_CONFIG otherwise); the record holds until the next step. */
int ggx_record_next_step(ggx_ctx* ctx);
int ggx_step_adjoint(ggx_ctx* ctx, const double* d_area, const double* d_perimeter, double* grad16);

/* Bulk readback of the whole state after the queued steps, for the output writers
 * (grainhdl::save_Texture, save_NetworkPlot, save_NrGrainsStats, save_Full_Microstructure_for_Restart,
 * src/grainhdl.cpp:871-1026, 1179-1308) and for analysis.  ggx_frame_begin waits for the last
 * queued step, stages what the next step overwrites and starts the device->host copies on a copy
 * stream, then returns: the next ggx_step runs while the copies are in flight (the step after it
 * waits for them).  ggx_frame_get waits for the copies and fills the view; its pointers stay
 * valid until the next ggx_frame_begin or ggx_destroy. */
typedef struct ggx_frame {
    int32_t nslots;                /* max id + 1; arrays below are indexed by grain id */
    int32_t loop;                  /* loop index of the next step when the frame was taken */
    int32_t precision;             /* GGX_PREC_* of the context (phi is always double here) */
    int32_t nb_stride;             /* entries per grain of nb_id / nb_len */
    int32_t list_stride;           /* entries per grain of cmp */
    int32_t real_domain_size;      /* R of the grid the frame's coordinates are on (grid coarsening) */
    int64_t field_elems, idl_elems, contour_points;  /* sizes of phi, idl, contour (points) */
    const ggx_grain_info* info;    /* [nslots], as ggx_get_info_all */
    const int64_t* phi_off;        /* [nslots] offset of grain id's field (n*n, row-major) in phi */
    const double* phi;
    const int64_t* idl_off;        /* [nslots] offset of grain id's IDLocal (the id box of info) */
    const uint32_t* idl;
    const int64_t* contour_off;    /* [nslots] point offset of grain id's contour (info.contour_len) */
    const double* contour;         /* x, y pairs */
    const int32_t* nb_id;          /* [nslots * nb_stride], count info.n_neighbours */
    const double* nb_len;
    const int32_t* cmp;            /* [nslots * list_stride], count info.n_compare */
    const double* quat;            /* [nslots * 4] orientation quaternion q0..q3 of each grain */
} ggx_frame;
int ggx_frame_begin(ggx_ctx* ctx);
int ggx_frame_get(ggx_ctx* ctx, ggx_frame* out);

/* The retained driver's output files from a frame, in the reference's formats and std::ostream
 * default number formatting.  dir: output directory ("" = current).  The network plot of an
 * anisotropic network needs per-point boundary weights a frame does not hold: GGX_E_CONFIG. */
/* Quaternion::quaternion2EulerConst (src/Quaternion.cpp:242-289): Bunge (phi1, PHI, phi2). */
int ggx_quat_to_euler(const double* q, double* euler);
/* grainhdl::save_Texture (src/grainhdl.cpp:871-1026): Texture_<loop>.ori (or the empty .bin files
 * with NeighbourTracking) and MODF_<loop>.txt (the misorientation distribution of anisotropic
 * networks, empty for isotropic ones); returns 0.5 * total energy and the total GB length. */
int ggx_write_texture(const ggx_frame* f, const ggx_settings* s, const char* dir, int32_t loop,
                      double* total_energy, double* total_length);
/* grainhdl::save_NetworkPlot (src/grainhdl.cpp:1291-1308) + LSbox::plot_box_contour
 * (src/box.cpp:1497-1549): Network_Timestep_<loop>.gnu, grains in IterativeGrainScheduler order. */
int ggx_write_network_plot(const ggx_frame* f, const ggx_settings* s, const char* dir, int32_t loop);
/* grainhdl::save_NrGrainsStats (src/grainhdl.cpp:1225-1241): one line, file truncated at loop 0. */
int ggx_write_nrgrains_stats(const char* dir, int32_t loop, double realtime, int32_t ngrains,
                             double total_energy, int32_t real_domain_size);
/* grainhdl::save_Full_Microstructure_for_Restart (src/grainhdl.cpp:1179-1223) + LSbox::plot_full_grain
 * (src/box.cpp:1552-1596): the parameters XML and the mode-0 network file of the current state. */
int ggx_write_restart(const ggx_frame* f, const ggx_settings* s, const char* dir, int32_t loop, int32_t ngrains);

/* Per-phase timers in the reference's stdout categories (grainhdl.cpp:1144-1154), in ms, and
 * work / traffic counters, all accumulated over every step of the context. */
typedef struct ggx_stats {
    double  convolution_ms, comparison_ms, levelset_ms, redistancing_ms, rest_ms, total_ms;
    int64_t steps;
    int64_t grid_point_updates;   /* sum over steps and live grains of n_g^2 */
    int64_t algorithmic_bytes;    /* compulsory HBM bytes of all steps: convolution (2 S n^2),
                                     comparison (S n^2 + S * neighbour overlap), IDLocal (4 n^2),
                                     redistanced field (S n'^2) */
    int64_t conv_bytes;           /* the convolution's part of algorithmic_bytes */
    int32_t live_grains;          /* live grains of the last step */
    int32_t max_box;              /* largest box side of the last step */
} ggx_stats;
int ggx_get_stats(ggx_ctx* ctx, ggx_stats* out);

/* ---------------------------------------------------------------------------------------
 * Batched convolution without a context, on caller-owned device buffers.
 * ------------------------------------------------------------------------------------- */

/* Replaces LSbox::convolutionGeneratorFFTW (src/box.cpp:622-695) -- the FFTW r2c plan, the
 * symbol multiply and the c2r plan of executeConvolution (box.cpp:408-536, plans made by
 * makeFFTPlans 580-608) -- for `count` square boxes in one call.  Box b has side n[b]
 * (1 <= n[b] <= max_n <= 512) and is read from in + off[b] and written to out + off[b], row-major
 * n x n doubles (out[b] = IDFT2(G . DFT2(in[b])), G of ConvolutionMode `mode`: 0 Laplace,
 * 1 Laplace-Richardson, 2 Gaussian, with the time step dt and nsq = R^2 of the global grid,
 * box.cpp:636-691).  n, off, in and out are device pointers; in and out must not overlap,
 * and no two boxes of a batch may share elements of out (a box listed twice is not computed twice but
 * spoiled: the passes work in place on out).
 * `stream` is a hipStream_t (NULL: the null stream).  The call allocates an error flag, runs on
 * `stream` (out holds intermediate values meanwhile), waits for it and frees the flag.  Returns
 * GGX_OK, GGX_E_ARG, GGX_E_BOUNDS (max_n above 512, or a side outside [1, max_n]: that box is left
 * unwritten), GGX_E_OOM or GGX_E_HIP. */
int ggx_convolve_boxes(int32_t count, const int32_t* n, const int64_t* off, const double* in, double* out,
                       int32_t max_n, int32_t mode, double dt, int32_t R, void* stream);

/* ggx_convolve_boxes without any allocation.  No counterpart in the reference: it is for callers
 * that cannot allocate device memory (code under hipGraph capture, tight serving loops, harnesses
 * that forbid hipMalloc).  Its error flag is a static device word; max_n is limited to 256
 * (GGX_E_BOUNDS above, with the reason in ggx_last_error(NULL)).  Same arguments and results as
 * ggx_convolve_boxes.  Calls that overlap on one GPU share that word and race: serialise them. */
int ggx_convolve_boxes_noalloc(int32_t count, const int32_t* n, const int64_t* off, const double* in, double* out,
                               int32_t max_n, int32_t mode, double dt, int32_t R, void* stream);

#ifdef __cplusplus
}
#endif
#endif
