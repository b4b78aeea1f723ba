// mfg_internal.h -- device data layout of the MI355X tracer, shared by the
// host runtime (mfg_host.cpp) and the HIP kernels (mfg_trace.hip).
//
// HBM layout (all variants concatenated; a plain model is one variant):
//   LeafFacet[]           the ray/facet test data in leaf order (128 B): a
//                         leaf is a contiguous run, no index indirection
//   BvhNode[]             up to 8-wide nodes, 128 B each, 8-bit quantised boxes
//   DHit[nF_total]        128 B, what a wall event always needs of its facet
//   DFacet[nF_total]      frame and polygon: sources, teleport destinations and
//                         the (u,v) of hits that are recorded by place
//   DPhys[nF_total]       physics and recording parameters beyond DHit, read
//                         for what the facet's flags name
//   Root[]                where the rays of each (variant, structure) start
//   double2 poly[]        normalised (u,v) polygon vertices
//   LeafUV[]              quadrilateral (u,v) corners (64 B), leaf order
//   DVariant[nV]          per-variant bases and settings
//   tallies               [variant][slot][facet] 64 B counters, textures,
//                         profiles, ... (layout of include/molflow_gpu.h)
#pragma once
#include <stdint.h>

#include "../../include/molflow_gpu.h"

#define MFG_ADJ_SEG 32            // target scores kept per lane for the adjoint's cutoff term
#define MFG_BVH_WIDTH 8          // children per node (a 4-wide build uses 4 of the 8 slots)
#define MFG_MAX_STACK 64         // (width - 1) * depth + width of the deepest tree the host accepts
#define MFG_WALK_NODES 512       // (ray, node) tasks of one wave's walk
#define MFG_WALK_RESERVE 72      // of these for the depth-first tail: width - 1 entries a level, + width
#define MFG_WALK_LEAVES 256      // (ray, facet record) tasks waiting: below 64 plus one node's 8 leaves of 16
static_assert(MFG_WALK_LEAVES >= 63 + 64 * 3, "a step of 8 nodes with leaves of 3 facets fits the list");
static_assert(MFG_WALK_LEAVES >= 63 + 8 * 16, "a node's 8 leaves of 16 facets fit the list whenever a node step runs");
static_assert(MFG_WALK_RESERVE >= MFG_MAX_STACK, "the reserve holds a depth-first walk of the deepest tree");
static_assert(MFG_WALK_NODES - MFG_WALK_RESERVE >= 64 && MFG_WALK_NODES >= 16 * 8,
              "64 roots, or the children of 16 nodes, fit below the reserve");
// Rays of a wave whose walk tasks give `bits` bits to the index of a node or
// record (26 up to 2^26 of them, else as many as they need).
constexpr uint32_t mfg_task_rays(uint32_t bits) { return bits <= 26u ? 64u : 1u << (32u - bits); }
constexpr bool mfg_task_fits(uint32_t bits) {
    return mfg_task_rays(bits) <= 64u && ((uint64_t)(mfg_task_rays(bits) - 1u) << bits | ((1ull << bits) - 1ull)) <= 0xffffffffull;
}
static_assert(mfg_task_fits(26) && mfg_task_fits(27) && mfg_task_fits(28), "ray and index fit a task's word");
#define MFG_LANE_STACK ((MFG_WALK_NODES + MFG_WALK_LEAVES) / 64)   // entries of a lane's own stack in the same LDS
#define MFG_REFILL 6             // TraceParams::refill_at of a long queue (1e6-particle tube 4.0 -> 3.5 ms; 12 and
                                 // more leave a steady beam-pipe launch slower)
#define MFG_MAX_GROUPS 64
#define MFG_MAXWELL_POINTS 100
#define MFG_MAXWELL_GUIDE 128
#define MFG_MAXWELL_LDS (16 * MFG_MAXWELL_POINTS + MFG_MAXWELL_GUIDE)
#define MFG_MAX_HOT 32           // facets whose counters are privatised per block
#define MFG_MAX_PROF_HOT 4       // profiles privatised per block

// feature bits of a trace-kernel instantiation / of a loaded model
enum : uint32_t {
    FEAT_TRANSPARENT = 1u << 0,   // opacity < 1 somewhere (coin + pass traversal)
    FEAT_MOMENTS = 1u << 1,       // time moments
    FEAT_TDPARAM = 1u << 2,       // time-dependent sticking/opacity/temperature/outgassing
    FEAT_VOLUME = 1u << 3,        // overtime, decay or scattering
    FEAT_TELEPORT = 1u << 4,      // teleport or link facets
    FEAT_MOVING = 1u << 5,
    FEAT_SOJOURN = 1u << 6,
    FEAT_LOWFLUX = 1u << 7,
    FEAT_FORCE = 1u << 8,
    FEAT_HIST = 1u << 9,
    FEAT_LOG = 1u << 10,
    FEAT_OGMAP = 1u << 11,
    FEAT_TRACE = 1u << 12,
    FEAT_AMSRC = 1u << 13,        // DES_ANGLEMAP sources
    FEAT_ADJOINT = 1u << 14,
    FEAT_ALL = (1u << 14) - 1,
};

// facet flags (DFacet::flags, DPhys::flags)
enum : uint32_t {
    FF_2SIDED = 1u << 0,
    FF_OPAQUE = 1u << 1,        // constant opacity 1
    FF_TRANSP = 1u << 2,        // constant opacity 0
    FF_TD_OPACITY = 1u << 3,
    FF_TEXTURE = 1u << 4,
    FF_COUNT_DES = 1u << 5,
    FF_COUNT_ABS = 1u << 6,
    FF_COUNT_REFL = 1u << 7,
    FF_COUNT_TRANS = 1u << 8,
    FF_COUNT_DIR = 1u << 9,
    FF_PROFILE = 1u << 10,
    FF_ANGLEMAP = 1u << 11,
    FF_MOVING = 1u << 12,
    FF_SOJOURN = 1u << 13,
    FF_FHIST = 1u << 14,
    FF_TELEPORT = 1u << 15,
    FF_LINK = 1u << 16,
    FF_DIFFUSE = 1u << 17,      // diffuse_part > 0.999999
    FF_FULL_ACC = 1u << 18,     // accomodation > 0.9999
    FF_OGMAP = 1u << 19,
    FF_TD_STICKING = 1u << 20,  // DHit::flags only: sticking / temperature from a
    FF_TD_TEMP = 1u << 21,      // time-dependent parameter (DPhys names it)
};

struct alignas(16) DFacet {
    double O[3];
    double N[3];
    double U[3];
    double V[3];
    double invU2, invV2;
    uint32_t poly_off;
    uint32_t poly_n;
    uint32_t flags;
    float opacity;
};
static_assert(sizeof(DFacet) == 128, "DFacet must be one 128-byte line");

struct alignas(16) DPhys {
    double nU[3], nV[3];
    double sticking, opacity, temperature, sqrt_temp, accomodation;
    double diffuse, specular, cos_exp, des_exp;
    double sojourn_freq, sojourn_e;
    double tex_wp, tex_hp;          // precise texture size
    double max_speed;
    double am_theta_limit;
    double fh_dist_bin, fh_time_bin;
    double og_wp, og_hp;            // outgassing map precise size
    double centre[3];
    int64_t tex_off, dir_off;       // cell offsets within the variant, -1 none
    int32_t prof_off, am_off;       // -1 none
    int32_t fh_off;                 // facet histogram offset, -1 none
    int32_t tex_w, tex_h;
    uint32_t flags;
    int32_t profile_type;
    int32_t super_idx, super_dest, teleport_dest;
    int32_t sticking_param, opacity_param, temperature_param, outgassing_param;
    int32_t id_index;               // integrated-desorption table (variant-local), -1
    int32_t local_id;               // facet index within its variant
    uint32_t am_phi, am_lo, am_hi;
    uint32_t fh_bounce_bin, fh_nb_bounce, fh_nb_dist, fh_nb_time;
    int32_t adj_group;              // sticking group, -1
    int32_t adj_target;             // adjoint target index, -1
    uint32_t og_w, og_h;
    int64_t og_off;                 // into og cdf array (global), -1
    int32_t desorb_type;
    int32_t pad_;
    int64_t am_src_off;             // DES_ANGLEMAP source table in the pool (global), -1
    int32_t hot_idx;                // slot in the per-block hot-facet counter table, -1
    int32_t prof_hot;               // index among the profiles summed in LDS, -1
};

// What a wall event always needs of its facet, in one line: loaded as six
// 16 B loads issued together (the last three words only by facets that are
// not purely diffuse or thermalising). DFacet and DPhys are read beyond it
// only for what the flags name (recordings, teleports, parameters).
struct alignas(128) DHit {
    double N[3], nU[3], nV[3];
    double sticking, sqrt_temp;
    uint32_t flags;                 // DPhys::flags + FF_TD_*
    int32_t hot_idx;                // as in DPhys
    int32_t adj_group, adj_target;
    double accomodation, diffuse, specular;
};
static_assert(sizeof(DHit) == 128, "DHit must be one 128-byte line");

// One BVH node of up to 8 children in one 128 B line. Child boxes are
// quantised to 8-bit steps per plane relative to the node's origin with a
// power-of-two step per axis: lo = o + qlo * 2^e, hi = o + qhi * 2^e in FP32
// (the builder checks that these FP32 values enclose the padded FP64 box).
// The steps are stored as the FP16 values of those integers (exact), which
// the kernel converts and scales in one v_fma_mix_f32. Children are found
// without per-child words: a node's inner children are consecutive nodes
// from node_base in slot order, and the leaf records of its leaf children
// are consecutive from leaf_base in slot order, each leaf holding 1 + its
// 4-bit count facets.
struct alignas(128) BvhNode {
    float ox, oy, oz;           // quantisation origin
    int8_t ex, ey, ez;          // per-axis step exponents
    uint8_t leaf_mask;          // bit c set when child slot c is a leaf
    int32_t node_base;          // first inner child (0 without inner children)
    int32_t leaf_base;          // first leaf record of the first leaf child (0 without leaves)
    uint32_t counts;            // bits 4c..4c+3: facets - 1 of a leaf child in slot c
    uint8_t inner_mask;         // bit c set when child slot c is an inner node
    uint8_t pad[3];
    uint16_t qlo[3][8];         // [axis][child], FP16 bit patterns of 0..255
    uint16_t qhi[3][8];
};
static_assert(sizeof(BvhNode) == 128, "BvhNode must be 128 bytes");

// Exact (FP64) ray/facet test data of one leaf entry, stored in leaf order
// so that a leaf's facets are contiguous (no index indirection). One record
// is one 128 B line, loaded as eight 16 B loads issued together.
//
// A triangle's record is complete: of the three u values of its corners one
// is 0, one is 1 (the facet's frame is their bounding rectangle) and the same
// holds for v, so two numbers and which corner has which give all six, in
// the place of 1/|V|^2 (recomputed, one division) and of the polygon. That
// spares a second line a test, read after the first.
struct alignas(128) LeafFacet {
    int32_t id;            // global facet index
    uint32_t flags;        // FF_* of the facet (low 24 bits), corner code << 24
    double O[3], N[3], U[3], V[3];
    double invU2;
    // triangle (corner code not 0): the u and the v that are not 0 or 1.
    // Others: first (u,v) pair in poly | vertices << 32 (bits), and 1/|V|^2
    double a, b;
};
static_assert(sizeof(LeafFacet) == 128, "LeafFacet must be one 128 B line");
// Corner code of a triangle: bits 0-1 the corner with u = 0, 2-3 with u = 1,
// 4-5 with v = 0, 6-7 with v = 1 (never 0, the two of an axis differ)
#define MFG_LEAF_FLAGS 0xffffffu

// (u,v) of the corners of a quadrilateral, parallel to LeafFacet in models
// that have one (read when the ray meets the facet's (u,v) rectangle); larger
// polygons are read from poly
struct alignas(64) LeafUV {
    double uv[8];
};
static_assert(sizeof(LeafUV) == 64, "LeafUV layout");

#ifdef __HIPCC__
// LDS of one wave's walk: slot r holds ray r (the ray of lane r). The FP32
// copy serves the box tests, the FP64 one the facet tests.
struct alignas(16) WaveLds {
    // (after the walk the same memory holds the event's tally updates)
    union {
        struct {
            float4 ra[64];             // origin, nearest t so far (widened)
            float4 rb[64];             // 1 / direction, facet to skip (bits)
        };
        double cell[3 * 64];           // texture cell updates, t names the cells
    };
    union {
        struct {
            double2 p01[64], p2d0[64], d12[64];   // position x y | z, direction x | y z
        };
        struct {
            double sums[5 * 64];       // facet counter updates (words 3.. of a record)
            unsigned long long record[64];
        };
    };
    unsigned long long t[64];          // nearest t so far (bits of a positive double)
    int32_t facet[64];                 // its facet, -1 none
    uint32_t nodes[MFG_WALK_NODES];    // ray << task_bits | node
    uint32_t leaves[MFG_WALK_LEAVES];  // ray << task_bits | facet record
};
#endif
// Transparent facets each ray of a wave met on its walk (more than
// MFG_PASSES: only counted), beside WaveLds in the kernels that need it.
#define MFG_PASSES 4
struct alignas(16) PassLds {
    uint32_t n[64];
    uint32_t rec[64][MFG_PASSES];      // facet records
};

// Where the rays of a structure start: its root node (-1: no facets), and
// the nodes a wave with few rays starts from, first << 4 | how many: the
// root's children if none of them is a leaf, else the root (a model has fewer
// than 2^27 leaf records, and no more nodes than those).
struct Root {
    int32_t node;
    uint32_t first;
};

// global counters of one variant (mfg_global_counters)
struct DGlobal {
    unsigned long long nb_mc_hit;
    double nb_hit_equiv;
    unsigned long long nb_desorbed;
    double nb_abs_equiv;
    unsigned long long nb_leak;
    double dist_total;
    double dist_full;
    unsigned long long nb_decayed;
};

struct DVariant {
    // geometry
    uint32_t facet_base, n_facets;
    uint32_t root_base, n_struct;      // into root table (one BVH root per structure)
    // source table
    uint32_t src_base, src_n;          // cumulative weights / facet ids
    double total_des;
    // settings
    double latest, gas_mass, half_life, low_flux_cutoff, c_factor;
    double scatter_mr, scatter_mfp, scatter_cut, scatter_rho;
    double motion1[3], motion2[3], torque[3];
    double gh_dist_bin, gh_time_bin;
    uint32_t flags;                    // FEAT_* actually used by this variant
    int32_t use_maxwell, calc_const_flow, enable_decay, scatter_enabled, scatter_cutoff, low_flux, motion_type;
    int32_t enable_force;
    uint32_t gh_bounce_bin, gh_nb_bounce, gh_nb_dist, gh_nb_time;
    int32_t log_facet;                 // global facet id or -1
    uint32_t log_limit;
    // tables (global offsets)
    uint32_t maxwell_base;             // 100 (v,p) pairs
    uint32_t maxwell_guide;            // MFG_MAXWELL_GUIDE entries into `guides`
    uint32_t param_base, n_params;     // into param table headers
    uint32_t id_base, n_ids;           // into ID table headers
    uint32_t mom_base, n_moments;      // into interval arrays
    // tally bases
    uint64_t fc_base;                  // facet counters, [slot][facet]
    uint64_t force_base;               // doubles
    uint64_t tex_base, n_tex;          // texture cells per slot
    uint64_t dir_base, n_dir;
    uint64_t prof_base, n_prof;
    uint64_t am_base;
    uint64_t gh_base, n_gh;
    uint64_t fh_base, n_fh;
    uint32_t n_slots, glob_index;
    // run
    uint64_t seed;
    uint64_t pid_base;                 // particle index offset of this run
};

struct DTable {                        // a (x,y) table in the global table pool
    uint32_t off, n;
    int32_t log_x, log_y;
};

// Everything a trace launch needs; passed by value (kernarg segment).
// One particle still in flight at the end of a launch, kept on the device
// and resumed first by the next launch (the particle state that persists
// between the reference's SimulationMCStep calls, Particle.h:95-122).
struct CarryRec {
    double pos[3], dir[3];
    double time, vel, ori, gen_time, dist, decay_t, scatter_path, hu, hv;
    uint64_t pid, events_left;
    uint32_t k0, k1, blk, b0, b1, b2, b3, avail;   // random stream position
    int32_t structure, last_hit, tele_from;
    uint32_t nb_bounces, nb_events, variant, tr_n;
};
static_assert(sizeof(CarryRec) == 200, "CarryRec layout");

struct TraceParams {
    // a launch of one variant (the kernels built for it): its constants,
    // read as scalars; seed and pid_base change between replays of a captured
    // launch and are read from `variants`
    DVariant one;
    Root one_root;                    // root of its only structure; node -2: look it up
    const DHit* hits;
    const DFacet* facets;
    const DPhys* phys;
    const double* poly;               // (u,v) pairs
    const BvhNode* nodes;
    const LeafFacet* leaves;
    const LeafUV* leaf_uv;
    const Root* roots;                // per (variant, structure)
    const DVariant* variants;
    const uint64_t* var_prefix;       // n_variants+1 prefix of this run's desorptions
    uint32_t n_variants;
    uint32_t task_bits;               // bits of a walk task's node or record index (the rest: its ray)
    uint32_t child_lanes;             // facets a leaf may hold if so few (at most 3) that 8 nodes' facets fit the list, else 0
    uint32_t lane_quota;              // lanes of a wave that take particles
    uint32_t refill_at;               // lanes without a particle that make a wave refill them
    uint64_t dealt;                   // items dealt out by wave index (waves * lane_quota) before the queue's
    uint32_t stack_total;             // entries a lane's own walk may need; the ones past MFG_LANE_STACK
    int32_t* stack_spill;             // live in this per-lane global area (lane-major)
    const double* src_cum;            // cumulative source weights
    const int32_t* src_facet;
    const double* og_cdf;
    const uint32_t* guides;           // guide tables of the Maxwell CDFs
    double maxwell_scale;             // > 0: all variants share one gas, whose CDF the blocks copy
                                      // to LDS (guide entries per unit of probability)
    const double* tab_x;              // table pool (maxwell CDFs, params, IDs)
    const double* tab_y;
    const DTable* params;
    const DTable* ids;
    const double* mom_start;
    const double* mom_end;
    // DES_ANGLEMAP source tables, one block per facet:
    // [W, L, H, theta limit, lower ratio, total count, line sums (T),
    //  theta CDF (T), phi CDFs (T*W), phi pdfs (T*W)], T = L + H
    const double* am_src;
    // hot facets: their counter updates of the first hot_slots slots (0 =
    // steady state, then the moments) are summed in LDS per block
    // and added to the global records once, when the block ends
    const uint64_t* hot_fc;           // index into fc of each hot facet's slot-0 record
    uint32_t n_hot;
    uint32_t hot_slots;               // slots of each kept there (1 with several variants)
    // profiles of a model with few of them: the slices of the first
    // prof_slots slots are summed in LDS per block, like the hot facets
    const uint64_t* hot_prof;         // first slice of each in slot 0
    uint32_t n_prof_hot, prof_slots;
    // tallies
    mfg_facet_counters* fc;
    double* force;
    mfg_texture_cell* tex;
    const double* tex_inc;            // per texture cell (same layout as slot 0)
    mfg_direction_cell* dir;
    mfg_profile_slice* prof;
    unsigned long long* am;
    double* gh;
    double* fh;
    DGlobal* glob;
    mfg_log_entry* log;
    unsigned long long* log_count;
    double* leaks;
    unsigned long long* leak_count;
    uint32_t leak_cap;
    // run control
    unsigned long long* next_particle; // work queue head
    uint64_t total;                    // desorptions in this run
    uint64_t max_events;
    volatile int32_t* stop_flag;       // host-mapped
    // a wave that has run for time_limit ticks of the device wall clock
    // starts nothing more, parks (carry) or ends its particles, sets
    // *expired and leaves: every launch ends even if no particle can
    uint64_t time_limit;
    unsigned long long* expired;
    // particles kept between launches: two halves of carry_cap records;
    // carry_ctl[0..1] count the records of each half, carry_ctl[2] names the
    // half this launch resumes from (the other half receives its leftovers)
    CarryRec* carry;
    unsigned long long* carry_ctl;
    uint64_t carry_cap;
    uint32_t carry_keep;               // 1: leave particles in flight when the queue runs dry
    // nodes [0, lds_nodes) (the top of the breadth-first node array) are
    // read from a copy each block keeps in LDS
    uint32_t lds_nodes;
    // trace
    int32_t* trace_facet;
    int32_t* trace_kind;
    uint32_t trace_n, trace_k;
    // adjoint
    double* adj_j0;
    double* adj_jac;
    const double* adj_sticking;
    uint32_t* adj_counts;             // per lane: sticky collisions per group
    // per lane: the target scores recorded since the particle last survived
    // a sticky collision (MFG_ADJ_SEG entries), for the cutoff term; a lane
    // with more sets *adj_seg_overflow
    int32_t* adj_seg_t;
    double* adj_seg_x;
    unsigned long long* adj_seg_overflow;
    uint32_t adj_groups, adj_targets;
};

struct IsectParams {
    const DFacet* facets;
    const double* poly;
    const BvhNode* nodes;
    const LeafFacet* leaves;
    const LeafUV* leaf_uv;
    Root root;
    uint32_t task_bits, child_lanes;
    uint32_t rays_per_wave;
    uint64_t n;
    const double* origins;
    const double* dirs;
    const int32_t* last_hit;
    int32_t* out_facet;
    double* out_t;
    double* out_u;
    double* out_v;
    uint32_t facet_base;
};

// Staging layout of the allocation-free intersect entry: the library's
// static device array `scratch` (mfg_trace.hip) holds one of these
#define MFG_MAX_DEVICES 64
struct StaticRays {
    double origins[3 * MFG_STATIC_MAX_RAYS];
    double dirs[3 * MFG_STATIC_MAX_RAYS];
    double t[MFG_STATIC_MAX_RAYS], u[MFG_STATIC_MAX_RAYS], v[MFG_STATIC_MAX_RAYS];
    int32_t last_hit[MFG_STATIC_MAX_RAYS];
    int32_t facet[MFG_STATIC_MAX_RAYS];
};
// device address of `scratch` on `device`, which must be the current
// device; looked up once per device (hipGetSymbolAddress), 0 on success
int mfg_scratch_address(int device, StaticRays** out);

// kernel launchers (mfg_trace.hip)
// (single: the launch has one variant, whose constants are in p.one)
int mfg_launch_trace(const TraceParams& p, uint32_t features, bool single, int waves, int grid, int block, void* stream);
int mfg_launch_intersect(const IsectParams& p, void* stream);
// after a carry launch: append the parked particles the launch did not
// claim (time limit) to the output half, then swap the halves
int mfg_launch_carry_flip(unsigned long long* carry_ctl, const unsigned long long* claimed, uint64_t dealt, CarryRec* carry,
                          uint64_t cap, unsigned long long* overflow, void* stream);
// arrays of 8-byte words to clear in one launch
struct ZeroList {
    uint64_t* p[16];
    uint64_t words[16];
    uint32_t n = 0;
    void add(void* ptr, uint64_t bytes) {
        if (bytes < 8) return;
        p[n] = (uint64_t*)ptr;
        words[n++] = bytes / 8;
    }
};
int mfg_launch_zero(const ZeroList& z, void* stream);
int mfg_launch_backward(const double* jac, const double* up, double* grad, uint32_t n_targets, uint32_t n_groups,
                        double scale, void* stream);
uint32_t mfg_trace_kernel_features(uint32_t model_features);
// LDS of one wave of the kernel that runs these features (its walk areas)
size_t mfg_wave_lds(uint32_t model_features);
int mfg_trace_occupancy(uint32_t features, bool single, int waves, int block, size_t lds_bytes);
int mfg_trace_variants(uint32_t features, int* waves_out, int cap);
// 1 when the feature set has a one-block-per-CU kernel of `block` lanes
// (768: 3 waves per SIMD, 1024: 4); only for launches of one variant
int mfg_trace_has_cu_block(uint32_t features, bool single, int block);
