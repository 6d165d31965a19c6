// Device-side data structures and kernel launchers shared by the engine.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gss.h"

namespace gss {

// Hit records are claimed by each wave in chunks of this many records.
constexpr int kHitChunk = 1024;

// One non-empty length bucket, as seen by the sweep kernel.
struct BucketDesc {
    const uint32_t *lits;  // row-major: literal i of row r at lits[r * len + i], stored as
                           // row offsets (literal << 7)
    uint32_t len;
    uint32_t count;        // rows
    uint32_t pass_begin;   // first wave pass of this bucket: plain sweeps (64 / words clauses
    uint32_t screen_begin; // a pass) and screened ones (64)
};

struct SweepArgs {
    const BucketDesc *buckets;
    int nbuckets;
    int npasses;             // wave passes over all buckets (sweep_clauses_per_pass clauses each)
    int task_passes;         // passes a wave takes at a time (0: see kTaskRounds in kernels.hip)
    const uint64_t *table;   // [2 * vars + 2][words]: row l = slots where literal l is not
                             // false; rows 2*vars (zeros), 2*vars+1 (ones) are sentinels
    const uint64_t *valid;   // [words]
    gss_hit *hits;           // chunk_cap * kHitChunk records
    uint32_t *fills;         // [chunk_cap] records used in each chunk
    uint32_t *alloc;         // zero before the sweep: [0] chunks claimed past the waves' own
                             // (wave g starts in chunk g), [1] chunks past chunk_cap with records
    uint32_t chunk_cap;
    uint32_t sentinel;       // stored row offset of the sentinel literal
    const int32_t *dyn;      // if set, {nbuckets, npasses} and the passes of the
                             // screened kernel are read here (steps)
    int rec_words;           // 8-byte words per record: 3 (gss_hit), 1 (gss_hit_id) or 2
                             // (gss_hit_clause: one record per clause, its words as a mask)
    // Serving and screened batched steps (null otherwise): for each literal l
    // a 16-bit entry (two per variable in one 32-bit word, literal 2v low);
    // bit b is set only if l is non-false in every valid slot of group b, bit
    // 8 + b only if it is true there -- serving: the step's admitted requests r
    // with r % 8 = b; screened steps: word group b, over all its slots
    // (launch_table_agg).  agg_words[b] = the table words of group b (serving:
    // of its requests; screened: with a valid slot).  Where a literal of a
    // clause is true, or two occurrences are non-false, no slot of the group
    // can report, so the exact check reads table rows only for the clause's
    // other words.
    const uint32_t *agg;
    const uint64_t *agg_words;  // [8]
    // launch_sweep_choose's: the screened kernel runs where screen_chosen, the plain
    // one elsewhere (null: whichever is launched)
    const uint32_t *choose;
};

// What launch_sweep_choose found.  choose[0], of the variables: 0 too few known, 1
// enough, 2 so many that the clauses need no look; choose[1 ..]: what the sample's
// 128 clauses cost by its blocks, in 48ths of a row per literal (open_cost in
// kernels.hip).  Screened where that is at most kOpenCost in 100.
constexpr unsigned kOpenBlocks = 16;
constexpr uint32_t kOpenCost = 21, kOpenLimit = 128 * 48 * kOpenCost / 100;
constexpr int kChooseWords = 1 + (int)kOpenBlocks;
__host__ __device__ inline bool screen_chosen(const uint32_t *choose) {
    uint32_t cost = 0;
    for (unsigned b = 0; b < kOpenBlocks; b++) cost += choose[1 + b];
    return choose[0] == 2 || (choose[0] == 1 && cost <= kOpenLimit);
}

// 64 clauses spread over the buckets: a row, its length and, from bit 24 on, how many
// rows there are from it on (1 or 2, if more).
struct ClauseSample {
    const uint32_t *row[4 * kOpenBlocks];
    uint32_t len[4 * kOpenBlocks];
};

// Staged regions of a batched step, read by k_step_in.
enum StepRegion {
    kRegHeader = 0,
    kRegDesc,
    kRegClauses,
    kRegLits,
    kRegUps,
    kRegPatches,
    kRegBaseUps,
    kRegLoads,
    kStageRegions
};

// Per-step inputs of a batched step (gss_step_*), written by the host into a
// pinned staging slot and copied to the device by k_step_in.
struct StepHeader {
    int32_t nbuckets;
    int32_t npasses;
    int32_t screen_passes;  // npasses of a screened sweep (of 64 clauses)
    int32_t nclauses;
    // 1 in the device copy when the step found the engine halted: every
    // count is then 0 and the step does nothing (it is replayed later)
    int32_t halted;
    int64_t nups, npatches, nbups, nloads;
    int64_t region_words[kStageRegions];  // uint32 words of each region to copy
    uint64_t valid[GSS_MAX_WORDS];
    int8_t last_pos[GSS_MAX_WORDS];
    uint64_t *host_rec;  // pinned memory that takes the step's records if they fit there
};

struct StepEndArgs {
    const StepHeader *dh;
    const gss_var_update *ups;
    uint64_t *table;
    int words;
    uint32_t *agg;        // as in StepInArgs
    uint32_t *halt;       // set if records were dropped
    uint32_t *out;        // counts for the host: see write_counts in kernels.hip
    uint64_t *dense;
    uint64_t dense_cap;   // records
    uint64_t host_words;  // 8-byte words at StepHeader::host_rec
};

// The hit chunks a sweep of `waves` waves left (SweepArgs).
struct ChunkArgs {
    const uint64_t *hits;
    const uint32_t *fills;
    const uint32_t *alloc;
    uint32_t cap;        // chunks in the buffer
    uint32_t waves;
    uint32_t rec_words;  // 8-byte words per record
};

struct ScatterSeg {
    uint32_t *dst;
    uint64_t src;    // offset in the staging buffer (uint32 units)
    uint64_t count;  // uint32 elements
};

// One clause staged by a batched step: its literals at src (uint32 units) of
// the staged literals, copied to its bucket row at dst.
struct ClauseSeg {
    uint32_t *dst;
    uint32_t src;
    uint32_t len;
};

// ---- serving: requests admitted on the device -------------------------------

// One request of the serving ring (fine-grained pinned host memory, written
// by the host before it publishes the request).
struct ServeReq {
    uint32_t solver;     // base the request's words are loaded from
    uint32_t k;          // assignments: slots [0, k) of words [0, ceil(k / 64))
    uint64_t patch_off;  // first patch (running index; ring position = modulo capacity)
    uint32_t n_patches;
    uint32_t pad;
    uint64_t seq;        // request sequence number
};

// A request admitted by a step: where it landed and where its patches are.
struct ServeAdmitted {
    uint64_t patch_off;
    uint64_t patch_pfx;  // patches of the step's earlier admitted requests
    uint32_t n_patches;
    uint32_t w0;         // first table word
};

// What a step admitted (pinned host memory, read after the step).
struct ServeReport {
    uint64_t first;  // sequence number of the first admitted request
    uint32_t count;  // requests admitted (in sequence order)
    uint32_t words;  // table words they took
};

// The serving kernels' view of the rings and the device-side cursor.
struct ServeRing {
    const ServeReq *reqs;          // pinned ring, req_cap entries
    const gss_var_patch *patches;  // pinned ring, patch_cap entries (words relative to the request)
    const uint64_t *head;          // pinned: requests published
    uint64_t *tail;                // device: next request to admit
    ServeAdmitted *adm;            // device: [kServeMaxRequests]
    uint32_t *adm_count;           // device
    gss_var_patch *dpatches;       // device: the step's admitted patches, in admission order
                                   // (patch_cap entries)
    uint32_t req_cap;
    uint32_t pad;
    uint64_t patch_cap;
};
constexpr int kServeMaxRequests = 64;  // one admission wave: at most 64 requests per step

struct StepInArgs {
    StepHeader header;                 // read over PCIe it cost k_step_in ~2 us more
    const uint32_t *h[kStageRegions];  // pinned host (the header's unused)
    uint32_t *d[kStageRegions];        // device
    // device word, nonzero while the engine is halted: an earlier step's
    // records overflowed its hit buffer and its sweep is to be re-run before
    // the table moves on
    const uint32_t *halt;
    uint32_t *alloc;      // the sweep's counters, cleared
    uint32_t *counts;     // serving: 2 * 64 counters of the grouping, cleared (else null)
    uint64_t *table;
    uint32_t *agg;        // apply with at most 8 words: screening entries to keep current
                          // (null: none, or a later kernel does it)
    uint64_t *agg_words;  // screened steps: [8], written from the header (else null)
    int words;
    int apply;            // apply the updates (else they are copied for a later kernel)
    int clauses;          // copy the clauses to their rows (else to the staged regions)
    int shift;            // of a literal on its way to its row
    uint64_t *bases;      // solver base planes (see launch_words_load_dyn)
    int64_t bases_vw;
    // Serving steps (report null otherwise): the published requests whose words
    // fit the table are admitted in sequence order (FIFO: the first that does
    // not fit waits for the next step).  The step's word loads, valid masks,
    // load and patch counts go to the device header and loads (and no passes
    // when nothing was admitted), the admitted list to serve.adm.
    ServeRing serve;
    ServeReport *report;  // pinned
};

// Plain sweeps, words >= 8: decides from a sample of the table and of the clauses
// whether sweep a (the screened kernel's) is screened (choose, kChooseWords), and if
// so builds the entries and agg_words.  valid is host memory, read before the launch.
hipError_t launch_sweep_choose(const SweepArgs &a, const ClauseSample &sample,
                               const uint64_t *valid, int64_t vars, int words, uint32_t *agg,
                               uint64_t *agg_words, uint32_t *choose, hipStream_t s);
// Screening entries of a batched step from the table itself (SweepArgs::agg):
// group b = words [b * words / 8, (b + 1) * words / 8) (one word per group
// below 8 words), over every slot of its words (valid or not: what holds in
// all of them holds in the valid ones).  Reads the table once.
hipError_t launch_table_agg(const uint64_t *table, const StepHeader *dh, int64_t vars, int words,
                            uint32_t *agg, hipStream_t s);
// Keeps such entries current without reading the table: for each of the
// step's updates (and patches, if with_patches) the bits of the update's word
// group, from the table as it is when the kernel runs.  Run after the updates are applied and again after the roll
// forward.
hipError_t launch_table_agg_update(const uint64_t *table, const StepHeader *dh,
                                   const gss_var_update *ups, const gss_var_patch *patches,
                                   bool with_patches, int words, uint32_t *agg, hipStream_t s);
// After the admission (launch_step_in): copies the admitted requests' patches
// from the pinned ring to r.dpatches, sets the words they took from their
// solvers' bases (and the rest of the rows' lines to all ones), and builds the
// step's screening entries and agg_words (none if agg is null).
hipError_t launch_serve_load(const ServeRing &r, const StepHeader *dh, const gss_word_load *loads,
                             const uint64_t *bases, int64_t vw, uint64_t *table, int words,
                             int64_t vars, uint32_t *agg, uint64_t *agg_words, hipStream_t s);
// Applies the admitted requests' patches (staged in r.dpatches) with their
// words shifted to where each request landed; with agg, clears the group's
// bits that a patch undoes in a valid slot.
hipError_t launch_serve_patch(const ServeRing &r, const StepHeader *dh, uint64_t *table,
                              int words, uint32_t *agg, hipStream_t s);

// One non-empty bucket of a tagged DB during compaction.
struct CompactRef {
    const uint32_t *lits;  // source rows (stored offsets)
    const uint32_t *tags;
    uint32_t *dst_lits;    // kept rows, in order
    uint32_t *dst_tags;
    int64_t start;         // first row of this bucket in the concatenation
    uint32_t len;
    uint32_t pad;
};

// words is the table row width (power of two, 1..64); a.agg and a.rec_words
// choose the kernel.
hipError_t launch_sweep(const SweepArgs &a, int words, int blocks, hipStream_t s);
int sweep_clauses_per_pass(int words, bool screened);
// Resident 256-thread blocks per CU of a sweep kernel (mode 0: plain, 1:
// screened, 2: clause records, 3: screened with clause records).
int sweep_occupancy(int words, int mode);

hipError_t launch_reset_u32(uint32_t *p, int n, hipStream_t s);
hipError_t launch_scatter(const ScatterSeg *segs, int nseg, const uint32_t *src, int shift,
                          hipStream_t s);
hipError_t launch_assig_apply(const gss_var_update *ups, int64_t n, uint64_t *table, int words,
                              hipStream_t s);
hipError_t launch_assig_roll(const gss_var_update *ups, int64_t n, uint64_t *table, int words,
                             const int8_t *last_pos, hipStream_t s);
hipError_t launch_fill_u64(uint64_t *p, int64_t n, uint64_t v, hipStream_t s);

// Fixed-shape launches of a batched step (counts read from the device header,
// which a serving step's admission sets there).  While the engine is
// halted k_step_in writes a header with no work and `halted` set instead of
// staging: every later kernel of the step then has nothing to do (the
// serving kernels and k_table_agg, whose work is not counted by the header,
// test `halted` themselves).
hipError_t launch_step_in(const StepInArgs &a, hipStream_t s);
hipError_t launch_step_end(const ChunkArgs &c, const StepEndArgs &a, hipStream_t s);
// Copies each staged clause (n read on the device) to its bucket row,
// shifting literals left by `shift`.
hipError_t launch_scatter_clauses(const ClauseSeg *cls, const int32_t *n, const uint32_t *src,
                                  int shift, hipStream_t s);
hipError_t launch_assig_apply_dyn(const gss_var_update *ups, const int64_t *n, uint64_t *table,
                                  int words, hipStream_t s);
// Rolls the step's updated entries forward (k_step_end does, after a sweep
// that kept its records).
hipError_t launch_assig_roll_dyn(const gss_var_update *ups, const int64_t *n, uint64_t *table,
                                 int words, const int8_t *last_pos, hipStream_t s);
// Counts of a plain sweep to pinned host memory (write_counts in
// kernels.hip); next = the counters of the sweep after it, cleared.
hipError_t launch_count_records(const ChunkArgs &c, uint32_t *out, uint32_t *next, uint32_t seq,
                                hipStream_t s);
// Dense copy of a sweep's records (chunk order, the records of a chunk in
// place) when they all fit in dense_cap records; counts are read on the
// device (records = how many the host knows of, for the grid).  Chunk c starts
// at word c * kHitChunk * rec_words.
hipError_t launch_gather(const ChunkArgs &c, uint64_t records, void *dense, uint64_t dense_cap,
                         hipStream_t s);
// Dense copy of a sweep's records grouped by assignment word, ascending:
// counts = 2 * 64 uint32 of device scratch (zero), group = 66 uint64:
// group[w] = first record of word w, group[64] = all, group[65] = 1 if they
// fitted in dense_cap records (else nothing moved); out = the counts for the
// host, *halt set if records were dropped.
hipError_t launch_group_by_word(const ChunkArgs &c, uint32_t *counts, void *dense,
                                uint64_t dense_cap, uint64_t *group, uint32_t *out,
                                uint32_t *halt, hipStream_t s);
// Sets word w of every variable's two rows from base b, for each load.  Solver
// base planes: bases[(2 b) * vw + i] / bases[(2 b + 1) * vw + i] hold bit (v
// mod 64) of word i = v / 64 of base b's is_def / is_true.
hipError_t launch_words_load_dyn(const gss_word_load *loads, const int64_t *n,
                                 const uint64_t *bases, int64_t vw, uint64_t *table, int words,
                                 int64_t vars, hipStream_t s);
hipError_t launch_assig_patch_dyn(const gss_var_patch *p, const int64_t *n, uint64_t *table,
                                  int words, hipStream_t s);

// Compaction of a tagged DB (rows of every bucket concatenated, N rows):
// flags[g] = keep[tag of row g] (tags >= ntags are kept), an exclusive scan
// of the flags, the kept count of each bucket, then the moves.
hipError_t launch_compact_flags(const CompactRef *refs, int nb, int64_t n, const uint8_t *keep,
                                int64_t ntags, uint32_t *flags, hipStream_t s);
hipError_t scan_exclusive_u32(const uint32_t *in, uint32_t *out, int64_t n, void *temp,
                              size_t &temp_bytes, hipStream_t s);
hipError_t launch_compact_bounds(const CompactRef *refs, int nb, int64_t n, const uint32_t *flags,
                                 const uint32_t *pos, uint32_t *kept, hipStream_t s);
hipError_t launch_compact_move(const CompactRef *refs, int nb, int64_t n, const uint32_t *flags,
                               const uint32_t *pos, hipStream_t s);

}  // namespace gss
