/* annarchy_hip_model.h -- plug-in ABI between the simulation runtime
 * (libannarchy_hip.so) and a generated neuron-model library.
 *
 * A model library is produced from a neuron description: the equation
 * snippets that the sympy front end emits are spliced into a HIP kernel
 * template (one thread per neuron, fused ODE + bounds + threshold + reset +
 * refractory + spike flags).  This mirrors the reference's per-population
 * generated code: PopStruct::update()/spike_gather()
 * (generator/Population/OpenMPGenerator.py:765-1237,
 *  generator/Population/CUDATemplates.py:543-720), which the reference emits
 * as text per network; here it is one shared object per model that the
 * runtime loads with dlopen() and launches from inside its captured step.
 *
 * Plain pointers and sizes only; the stream is passed as an opaque pointer.
 */
#ifndef ANNARCHY_HIP_MODEL_H
#define ANNARCHY_HIP_MODEL_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define AHIP_MODEL_ABI 16
#define AHIP_MAX_SLOTS 48
#define AHIP_MAX_RAND 8
#define AHIP_UPDATE_BLOCK 256 /* threads per block of every update kernel */

/* Ordered spike delivery folded into the update of the post population.
 * head[i] = (base << AHIP_HEAD_SHIFT) | count: neuron i's events of this
 * step are bucket records base .. base + count (head[i + 1] >> SHIFT bounds
 * the range).  A record is a key (the projection's key offset + the
 * synapse's column-order index, so keys sort projection by projection and in
 * ascending pre-synaptic rank: the reference's summation order) and the
 * event's weight: uint32 key, uint32 padding, double weight in FP64 (16
 * bytes); uint32 key, float weight in FP32 (8 bytes).  The weights are added
 * to g[i] in ascending key before the equations read g; the count is
 * cleared. */
typedef struct ahip_deliver_desc {
    void* g;
    uint64_t* head;                     /* size + 1 words */
    const void* bucket;                 /* records */
    const void* reserved;
} ahip_deliver_desc;
#define AHIP_HEAD_SHIFT 24
#define AHIP_HEAD_COUNT ((1ull << AHIP_HEAD_SHIFT) - 1ull)
#define AHIP_MAX_DELIVER 4 /* ordered conductances one update delivers */
#define AHIP_MAX_PSUM 2    /* psp sums one update completes from panel partials */

/* Spike events counted per post neuron: the scatter adds 1 (or, `sums`, the
 * synapse's weight) at ring slot (arrival step) mod depth, the update adds
 * them to the conductance in slot `slot` before its statements, projection by
 * projection, one addition of the weight per event, and clears them.  All
 * addends of a projection are equal, so the result does not depend on the
 * order in which the events were counted. */
typedef struct ahip_counted_desc {
    void* ring;                         /* depth x size int32 counts, or sums in the network precision */
    double w;
    int32_t slot, depth, sums, reserved;
} ahip_counted_desc;
#define AHIP_MAX_COUNTED 4 /* counted projections one update delivers */

/* Recording of a monitor, in device memory (the host rewrites it when the
 * monitor is emptied; a captured step reads it): step t_start + k * period goes
 * to row base + k, below capacity. */
typedef struct ahip_record_state {
    int64_t t_start, base, period, capacity;
} ahip_record_state;
#define AHIP_MAX_REC 4     /* value monitors one update records */
#define AHIP_MASK_BLOCKS 512 /* blocks of 256 neurons whose spikes kernels read from the mask, at most */
#define AHIP_FILL_RING 32  /* > steps of one compaction launch + 1, a power of two */

/* Arguments of one population update launch.  Device pointers unless noted. */
typedef struct ahip_pop_args {
    int32_t size;                       /* number of neurons */
    int32_t step;                       /* step index inside the launched batch */
    const int64_t* t_base;              /* simulation step at the start of the batch */
    double dt;                          /* host value */
    void* slot[AHIP_MAX_SLOTS];         /* local: size elements, global: 1 element */
    const void* rand_inject[AHIP_MAX_RAND]; /* injected draws [steps][size] or NULL */
    int64_t rand_inject_steps;          /* rows available in the injected buffers */
    int64_t rand_t0;                    /* simulation step of row 0 of the injected buffers */
    uint64_t seed;                      /* counter-based generator key */
    uint32_t stream_id;                 /* population id, second key word */
    int32_t* refractory;                /* steps, per neuron */
    int32_t* refractory_remaining;
    int64_t* last_spike;
    uint64_t* spike_mask;               /* ceil(size/64) words, bit i = neuron spiked (of this step) */
    int32_t* block_counts;              /* ceil(size/256) spike counts per update block */
    const ahip_deliver_desc* deliver;   /* ordered conductances delivered by this update, or NULL */
    int32_t n_deliver;
    /* psp sums the update completes: slot psum_slot[k] (a _sum_<target>) is
     * the sum over the panels q < psum_panels[k] of psum_part[k][q *
     * psum_stride[k] + i], added in ascending q (compensated in FP32), plus
     * the slot's own value when psum_acc[k]; the update stores it to the
     * slot before its statements read it */
    int32_t n_psum;
    int32_t psum_slot[AHIP_MAX_PSUM];
    int32_t psum_panels[AHIP_MAX_PSUM];
    int32_t psum_acc[AHIP_MAX_PSUM];
    int32_t psum_stride[AHIP_MAX_PSUM];
    const void* psum_part[AHIP_MAX_PSUM];
    /* rate-coded: rings the update copies the new r to (depth 0: none), value
     * of neuron i at push_buf[k][(t mod push_depth[k]) * size + i]: the delay
     * queue and the two-step buffer that fused updates read */
    void* push_buf[2];
    int32_t push_depth[2];
    /* value monitors the update records: local slot rec_slot[k] of every
     * neuron, before its statements (after compute_psp) or after them, into
     * rows of `size` values */
    int32_t n_rec;
    int32_t rec_slot[AHIP_MAX_REC];
    int32_t rec_before[AHIP_MAX_REC];
    const ahip_record_state* rec_state[AHIP_MAX_REC];
    void* rec_data[AHIP_MAX_REC];
    int32_t n_counted;
    ahip_counted_desc counted[AHIP_MAX_COUNTED];
} ahip_pop_args;

typedef int (*ahip_launch_fn)(const ahip_pop_args* args, void* stream);

/* ---- several steps of an input population in one launch --------------------
 * A population that no projection reaches and whose values are functions of the
 * step alone (draws, constants, the clock; no value of the step before) does not
 * have to wait for the network: one launch computes `steps` steps from the
 * args' step on, a workgroup per 256 neurons and step.  Rates go to the rings
 * (push_buf), recorded values to their rows, spikes to the mask and the counts of
 * each step (ceil(size / 64) words and ceil(size / 256) counts a step), the
 * population's values are those of the last step.  last_spike is left to the
 * compaction of each step. */
#define AHIP_AHEAD 16      /* steps of a launch at most */
typedef int (*ahip_ahead_fn)(const ahip_pop_args* args, int32_t steps, void* stream);

/* ---- psp and update of a rate-coded population in one launch --------------
 * The rows (post neurons) of every projection into the population are summed
 * by the update kernel itself, 2^lane_shift lanes per row, while the first
 * update_waves waves of the workgroup load the neurons' values and draw their
 * random numbers; they run the statements after a barrier.  Pre-synaptic rates come from rings indexed
 * by the step (push_buf of the pre population's update), so no launch reads a
 * rate that another workgroup of the same launch writes. */
#define AHIP_MAX_FUSE 4
#define AHIP_FUSE_CSR 0       /* ptr: row pointer; col, w: entries */
#define AHIP_FUSE_SELL 1      /* ptr: slice offsets (SELL-C-sigma, 2^lane_shift threads per row) */
#define AHIP_FUSE_DENSE 2     /* w: row-major, ld values per row; 64 lanes per row */
#define AHIP_FUSE_CSR_DELAY 3 /* CSR with a delay (steps) per entry */
#define AHIP_FUSE_MIX 4       /* launch: projections of several forms */
#define AHIP_FUSE_THREADS 512
#define AHIP_FUSE_STAGE_THREADS 1024
#define AHIP_FUSE_ROWS 256    /* rows of a workgroup at most */
#define AHIP_FUSE_DENSE_ROWS 8 /* of a dense projection alone */
typedef struct ahip_fuse_proj {
    int32_t kind;
    int32_t sum;                        /* which psp sum of the model (slots of kind 2, in slot order) */
    int32_t n_cols;                     /* pre-synaptic neurons */
    int32_t depth;                      /* ring depth of x */
    int32_t delay;                      /* x of step t: ring slot (t - delay) mod depth */
    int32_t ld;                         /* dense: values per row, a multiple of 4 */
    const int64_t* ptr;
    const int32_t* col;
    const void* w;
    const int16_t* delays;
    const void* x;                      /* ring of n_cols values per slot */
} ahip_fuse_proj;
typedef struct ahip_fuse_args {
    int32_t n;                          /* projections, in creation order */
    int32_t lane_shift;                 /* log2 of the lanes per row (0 .. 6) */
    int32_t units;                      /* rows, or SELL slices of 64 >> lane_shift rows */
    int32_t kind;                       /* the form of every projection, AHIP_FUSE_MIX: not one form */
    int32_t blocks;                     /* workgroups */
    int32_t share;                      /* units per workgroup */
    int32_t update_waves;               /* waves that run the statements, 64 rows each */
    int32_t stage;                      /* 1: x staged in LDS (lds_values values), 1024 threads */
    int32_t lds_values;
    uint32_t mask;                      /* psp sums that have a projection (bit = sum index) */
    const int32_t* perm;                /* SELL: row of every slice position (-1: none), else NULL */
    ahip_fuse_proj p[AHIP_MAX_FUSE];
} ahip_fuse_args;
typedef int (*ahip_fused_fn)(const ahip_pop_args* args, const ahip_fuse_args* fa, void* stream);

/* ---- persistent steps of a small network --------------------------------
 * A network of one spiking population whose projections all start and end
 * in it (constant weight each, no delays, no synapse model) can run a whole
 * batch of steps in ONE launch of one workgroup: per step the scatter of the
 * previous step's spikes into the conductances, the update of every neuron
 * and the ascending spike list with its recording.  The state the
 * statements touch (the model's persist_slots) and the refractory counters
 * live in LDS for the whole launch.  The steps are the ordinary ones (the
 * same statements, the same order), so spike trains and state equal those of
 * the per-kernel step. */
#define AHIP_PERSIST_MAX_PROJ 8
#define AHIP_PERSIST_THREADS 1024
#define AHIP_PERSIST_ITEMS 512      /* (projection, spike) items per scatter pass */
typedef struct ahip_persist_proj {
    const int64_t* col_ptr;             /* CSRC backward view (pre rank -> synapse range) */
    const int32_t* row_idx;             /* post rank of every synapse, column order */
    double w;                           /* the projection's one weight */
    int32_t n_cols;                     /* pre ranks covered by col_ptr */
    int32_t target;                     /* index of the conductance in the model's persist_slots */
    int32_t round;                      /* scatter round: same-target projections in creation order */
    int32_t lds_cols;                   /* offset of its column ranges in the LDS table (-1: col_ptr) */
} ahip_persist_proj;
typedef struct ahip_persist_args {
    int32_t steps;                      /* steps of this launch */
    int32_t n_proj, n_rounds;
    int32_t n_lds_cols;                 /* entries of the LDS column-range table (0: none) */
    ahip_persist_proj proj[AHIP_PERSIST_MAX_PROJ];
    int32_t* spiked;                    /* the population's spike list and count (kept up to date) */
    int32_t* spike_count;
    /* the population's spike monitor (rec_counts == NULL: none), as filled
     * by the compaction of the per-kernel step */
    int32_t* rec_counts;
    int32_t* rec_idx;
    int64_t* rec_fill;                  /* [s mod AHIP_FILL_RING]: indices before the list of row s */
    int64_t rec_idx_capacity;
    const ahip_record_state* rec_state;
} ahip_persist_args;
typedef int (*ahip_persist_fn)(const ahip_pop_args* args, const ahip_persist_args* pa, size_t lds_bytes,
                               void* stream);
/* Host-side evaluation of the hoisted step sizes (exponential Euler
 * "pre_loop" values, parser/Equation.py:559-604) from the global slots; writes
 * one value per pre-loop slot.  Host libm is used on purpose so the values
 * equal those of a CPU build. */
typedef void (*ahip_preloop_fn)(const double* globals_host, double dt, double* out);

typedef struct ahip_model_desc {
    int32_t abi;                        /* AHIP_MODEL_ABI */
    const char* name;
    int32_t spiking;                    /* 1: spiking (threshold/reset), 0: rate-coded */
    int32_t n_slots;
    const char* const* slot_names;      /* attributes, _sum_<target>, pre-loop step sizes */
    const int32_t* slot_local;          /* 1: one value per neuron, 0: population-wide */
    const double* slot_init;            /* initial value of each slot */
    const int32_t* slot_kind;           /* 0 parameter, 1 variable, 2 psp sum, 3 pre-loop,
                                           4 network constant (population-wide, written by
                                           ahip_net_set_constant) */
    int32_t n_rand;                     /* random variables drawn per step */
    const int32_t* rand_dist;           /* 0 Uniform(a,b), 1 Normal(mu,sigma) */
    const double* rand_args;            /* two per random variable */
    int32_t has_refractory;
    int32_t has_global_update;          /* a one-thread kernel runs before the local one */
    ahip_launch_fn launch_f64;
    ahip_launch_fn launch_f32;
    ahip_preloop_fn preloop;            /* NULL when there is no pre-loop value */
    const char* source_hash;
    ahip_persist_fn persist_f64;        /* NULL for rate-coded models or with a global update */
    ahip_persist_fn persist_f32;
    int32_t persist_n_slots;            /* local slots the persistent steps hold in LDS, in LDS order: */
    const int32_t* persist_slots;       /* those the statements touch and the conductances */
    ahip_fused_fn fused_f64;            /* NULL for spiking models and models without a psp sum */
    ahip_fused_fn fused_f32;
    ahip_ahead_fn ahead_f64;            /* NULL: the statements read a value of the step before */
    ahip_ahead_fn ahead_f32;
} ahip_model_desc;

/* Every model library exports this symbol. */
typedef const ahip_model_desc* (*ahip_model_describe_fn)(void);

#ifdef __cplusplus
}
#endif

#endif
