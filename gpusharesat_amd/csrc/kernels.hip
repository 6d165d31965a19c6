// CDNA4 (gfx950, wave64) kernels of the clause-vs-assignment check.
//
// The usefulness rule of the reference (gpuShareLib/GpuRunner.cu:34-57,
// ReportComputer) reports slot s of a clause when every literal is false
// ("falsified") or when exactly one literal occurrence is undefined and every
// other one is false ("unit").  The sweep evaluates it in an equivalent form
// over table rows, where row l holds nf_l = the slots in which literal l is
// NOT false (true or undefined); literal l is true exactly where its negation
// l^1 is false, i.e. outside nf_{l^1}:
//
//   count   c1/c2 = "at least one / at least two non-false occurrences",
//           saturating:  c2 |= c1 & nf_l;  c1 |= nf_l
//   true    nt = AND over the clause of nf_{l^1} (no literal is true)
//   report  falsified = ~c1;  unit = c1 & ~c2 & nt
//
// A slot with c2 set can never report, so a clause stops once every valid
// slot is dead.  The check reads the rows nf_l first (1 bit per slot per
// literal) until then; a slot that ends with exactly one non-false occurrence
// needs nt, and there only the row nf_{l^1} of that one literal can hold a
// zero, so only those negated rows are read.  Duplicate literals are separate
// occurrences, as in the reference (GpuRunner.cu:68-89 walks the literal
// list), so "x, x" with x undefined is not unit.  tests/test_oracle.py and the
// GPU parity tests check the forms agree.
//
// Clause literals are stored on the device as row offsets: literal l as
// l << 7, the byte offset of its row in a table of 16 words (scaled by the
// actual width at compile time); negation is "xor 128".  Padding lanes past
// the end of a clause hold the offset of a sentinel row pair (nf = 0, and
// all ones for its negation) that contributes nothing, so they need no mask.
//
// Work mapping.  k_sweep: W lanes check one clause, one table word each, 64 / W
// clauses per wave pass, literals handed out with DPP (no LDS); k_sweep_screened:
// one clause per lane against the screening entries, then two words of a surviving
// clause per lane, or W lanes per clause where most words are left.  Waves are
// persistent and walk the clauses in tasks of passes.  Steps are screened on
// request; other sweeps where a look at the table and the clauses says that it
// pays (k_sweep_choose).
//
// What bounds it is the row reads: 128-byte lines of a table that the L2s do
// not hold, ~6.9 TB/s of them at any size past 32 MB.  Measured on one MI355X,
// kernel alone, before (16 lanes per clause at every width, 4 rows per step,
// all negated rows of a clause left with a candidate, both rows of every
// literal up to 4 literals) and now:
//   16 words, 4M clauses, 1M variables, random values   711 -> 618 us
//   16 words, 2M clauses, 500k variables, planted       204 -> 119 us (screened: 73)
//   64 words, 400k clauses, 200k variables, planted     140 ->  87 us (screened: 72)
//    8 words, 1M clauses, 100k variables, planted       109 ->  45 us (screened: 32)
//    1 word,  100k clauses, 10k variables, random        32 ->   8 us
// Rows read per clause, counted on the CPU: 7.97 -> 6.95 (random), 4.54 -> 2.77
// (planted).
//
// Hits.  A clause/word with a report becomes one 24-byte record (gss_hit:
// clause, word and both masks), or, for delivery to the solvers, which never
// read the masks, one 8-byte record (gss_hit_id: the first word of the
// gss_hit), or one gss_hit_clause per clause.  Each wave compacts its records
// with a ballot + mbcnt prefix into chunks of kHitChunk records of its own
// (HitWriter).  Capacity is sized on the host so that nothing is dropped (the
// reference drops on overflow, gpuShareLib/Reporter.cuh:46-48); if it ever is
// exceeded the counters tell, and the host re-runs the sweep.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <hipcub/hipcub.hpp>
#include <utility>

#include "chunks.h"
#include "kernels.h"

namespace gss {

// k_sweep writes a record as three 8-byte words: {row, len, word}, false_mask,
// unit_mask.
static_assert(sizeof(gss_hit) == 24 && offsetof(gss_hit, len) == 4 &&
                  offsetof(gss_hit, word) == 6 && offsetof(gss_hit, false_mask) == 8 &&
                  offsetof(gss_hit, unit_mask) == 16,
              "gss_hit layout");
static_assert(sizeof(gss_hit_id) == 8 && offsetof(gss_hit_id, len) == 4 &&
                  offsetof(gss_hit_id, word) == 6,
              "gss_hit_id is the first word of a gss_hit");
static_assert(sizeof(gss_hit_clause) == 16 && offsetof(gss_hit_clause, len) == 4 &&
                  offsetof(gss_hit_clause, words) == 8,
              "gss_hit_clause: {row, len, 0} then the word mask");

namespace {

__device__ __forceinline__ uint32_t prefix_count(unsigned long long bal) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
    return (uint64_t)(uint32_t)uniform((int)(uint32_t)x) |
           ((uint64_t)(uint32_t)uniform((int)(uint32_t)(x >> 32)) << 32);
}

// Byte offset inside the table of row word w, from a stored row offset
// (literal << 7, i.e. the offset for a 16-word table).
template <int W>
__device__ __forceinline__ uint32_t scale_offset(uint32_t stored) {
    if constexpr (W == 16) return stored;
    else if constexpr (W > 16) return stored << (W == 32 ? 1 : 2);
    else return stored >> (W == 8 ? 1 : W == 4 ? 2 : W == 2 ? 3 : 4);
}

// Offset of the negated literal's row: stored offsets are literal << 7, so the
// negation flips bit 7, scaled like the offset.
template <int W>
__device__ __forceinline__ uint32_t neg_bit() {
    return scale_offset<W>(128u);
}

__device__ __forceinline__ uint64_t load_word(const uint64_t *__restrict__ table, uint32_t off) {
    return *(const uint64_t *)((const char *)table + off);
}

// Clause literals: a global-memory pointer (made from the bucket descriptor's
// address, which the compiler would otherwise read with FLAT loads).
typedef const __attribute__((address_space(1))) uint32_t *LitPtr;

// A clause is checked by W lanes (lane w: table word w), which share its
// literals: each lane of a group of G = min(W, 16) holds kRegs consecutive ones,
// the group the first kHeld.  Wider clauses repeat the group (every 16-lane DPP
// row holds the same 16 literals), so a literal is always handed out inside
// one DPP row.
template <int W>
struct Lits {
    static constexpr int G = W < 16 ? W : 16;
    static constexpr int kRegs = W >= 4 ? 1 : 4 / W;
    static constexpr int kHeld = G * kRegs;  // 16, 8 (W = 8) or 4
    uint32_t r[kRegs];
};

// The literal at position J of the held ones, in every lane of the group: a
// DPP broadcast (row_newbcast for 16 lanes, two of them under bank masks for
// 8, quad_perm for 4 and 2), so no LDS.  All 64 lanes must call it.
template <int W, int J>
__device__ __forceinline__ uint32_t lit_at(const Lits<W> &l) {
    constexpr int G = Lits<W>::G, R = J % Lits<W>::kRegs, Q = J / Lits<W>::kRegs;
    const int x = (int)l.r[R];
    if constexpr (G == 16) {
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, 0x150 + Q, 0xF, 0xF, false);
    } else if constexpr (G == 8) {
        const int lo = __builtin_amdgcn_mov_dpp(x, 0x150 + Q, 0xF, 0xF, false);
        return (uint32_t)__builtin_amdgcn_update_dpp(lo, x, 0x150 + 8 + Q, 0xF, 0xC, false);
    } else if constexpr (G == 4) {
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, Q * 0x55, 0xF, 0xF, false);
    } else if constexpr (G == 2) {
        return (uint32_t)__builtin_amdgcn_mov_dpp(x, Q * 0x55 + 0xA0, 0xF, 0xF, false);
    } else {
        return (uint32_t)x;
    }
}

// Literals [base, base + kHeld) of the clause whose row starts at cl (lane q of
// its group holds kRegs of them from base + q * kRegs on), the sentinel past its
// end and for lanes without a clause (on = false).  One load a lane where they
// are all there (rows are 4-byte aligned, as these loads may be): the lanes of a
// narrow table read lines of their own, one each per load (1 word, 150k clauses of
// 20 to 60 literals: 65 us with a load per literal, 55 so).
template <int W>
__device__ __forceinline__ Lits<W> load_lits(LitPtr cl, int base, int len,
                                             int q, bool on, uint32_t sentinel) {
    constexpr int R = Lits<W>::kRegs;
    const int j = base + q * R;
    Lits<W> l;
#pragma unroll
    for (int r = 0; r < R; r++) l.r[r] = sentinel;
    if constexpr (R == 1) {
        if (on && j < len) l.r[0] = cl[j];
    } else {
        typedef uint32_t Vec __attribute__((ext_vector_type(R), aligned(4)));
        if (on && j + R <= len) {
            const Vec v = *(const __attribute__((address_space(1))) Vec *)(cl + j);
#pragma unroll
            for (int r = 0; r < R; r++) l.r[r] = v[r];
        } else {
#pragma unroll
            for (int r = 0; r < R; r++)
                if (on && j + r < len) l.r[r] = cl[j + r];
        }
    }
    return l;
}

// Bucket of pass p: the last one whose first pass is <= p.  One lane per
// bucket (a binary search is a chain of 6-9 dependent scalar loads).
template <bool SCREENED>
__device__ __forceinline__ uint32_t pass_begin(const BucketDesc &b) {
    return SCREENED ? b.screen_begin : b.pass_begin;
}

template <bool SCREENED>
__device__ __forceinline__ int find_bucket(const BucketDesc *__restrict__ b, int nb, int p,
                                           int lane) {
    int n = 0;
    for (int i = 0; i < nb; i += 64) {
        const bool le = i + lane < nb && (int)pass_begin<SCREENED>(b[i + lane]) <= p;
        n += __popcll(__ballot(le));
    }
    return uniform(n - 1);
}

// 7 blocks of 4 waves per CU need at most 96 scalar registers: the device
// counts them in sixteens, with sixteen more per wave than the kernel's own
// (measured: kernels of 97-106 ran 6 blocks per CU, of 81-96 seven).
#define GSS_SWEEP_BOUNDS __attribute__((amdgpu_num_sgpr(96))) __launch_bounds__(256)
constexpr int kSweepBlocksPerCu = 7;

// Tables of less than 8 words: kRows rows read per step past a clause's held
// literals, and kept of these for the negated-row reads.
// A row there is part of a line and comes from the L2s, so long clauses are bound
// by the chain of reads, not by their number; with the literals one step ahead.
// 200k variables x 1 word, 150k clauses of 20 to 60 literals, nine in ten false:
// 65 us with two rows per step, 49 with eight; 40k of 150 to 400, 97 in 100 false:
// 148 and 94 (four rows: 55 and 128).
constexpr int kRows = 8;

// How a wave walks the clauses: the passes of all buckets (CPW clauses of one
// length each) form one sequence, cut into tasks of `tp` passes that the
// persistent waves take round-robin.  tp gives every wave kTaskRounds tasks
// of the same number of passes, so the waves finish together whatever the
// number of clauses (tasks of a fixed 64 clauses left 4.4 tasks per wave on 2M
// clauses: some waves had 5), and a wave reads its literals in long runs.
//
// A pass of a screened sweep is 64 clauses, checked one after the other as far as
// they survive: where there are fewer passes than waves it is split into up to
// max_split parts (a power of two, at most the table's words).  A pass of 32 words
// and more is so much work that three parts per wave are better than one (600k
// clauses x 64 words, 9,375 passes, nothing known: 1,097 us whole, 956 in halves);
// four were not (400k: 255 us per sweep whole, 254 in halves, 281 in quarters).
constexpr int kTaskRounds = 4;

struct Passes {
    int nbuckets, total, tp, gw, nw;
    int split = 0;  // log2 of the parts

    __device__ __forceinline__ Passes(const SweepArgs &a, bool screened, int max_split) {
        nbuckets = a.nbuckets;
        total = a.npasses;
        if (a.dyn) {
            nbuckets = uniform(a.dyn[0]);
            total = uniform(a.dyn[screened ? 2 : 1]);
        }
        gw = uniform((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));  // 256-thread blocks
        nw = (int)gridDim.x * 4;
        const int64_t room = max_split > 16 ? 3ll * nw : nw;
        while ((2 << split) <= max_split && ((int64_t)total << (split + 1)) <= room) split++;
        total <<= split;
        tp = a.task_passes << split;
        if (tp <= 0) tp = (total - 1) / (nw * kTaskRounds) + 1;
    }
};

// Appends a wave's records to its hit chunks.  A wave's first chunk is the
// one of its own number, so a sweep with few records claims nothing (one
// device-scope atomic costs ~10 ns and they all meet on one address: claims
// of the first chunk by ~8,000 waves took 80 us); a full chunk is replaced by
// one claimed past those.  Chunks past the buffer take no records: alloc[1]
// counts them, and the host re-runs the sweep with room.
struct HitWriter {
    gss_hit *hits;
    uint32_t *fills;
    uint32_t *alloc;  // [0] chunks claimed past the waves' own, [1] chunks past the buffer
    uint32_t cap;     // chunks in the buffer
    int waves;        // first claimable chunk
    int chunk;
    int fill = 0;

    __device__ __forceinline__ HitWriter(const SweepArgs &a, const Passes &ps)
        : hits(a.hits), fills(a.fills), alloc(a.alloc), cap(a.chunk_cap), waves(ps.nw),
          chunk(ps.gw) {}

    // Room for n more records (n <= 64): true if they may be written.
    __device__ __forceinline__ bool room(int n, int lane) {
        if (fill + n > kHitChunk) {
            if (lane == 0 && (uint32_t)chunk < cap) fills[chunk] = (uint32_t)fill;
            uint32_t c = 0;
            if (lane == 0) c = atomicAdd(alloc, 1u);
            chunk = waves + uniform((int)__shfl(c, 0));
            fill = 0;
        }
        if ((uint32_t)chunk < cap) return true;
        if (fill == 0 && lane == 0) atomicAdd(alloc + 1, 1u);
        return false;
    }

    __device__ __forceinline__ void end(int lane) {
        if (lane == 0 && (uint32_t)chunk < cap) fills[chunk] = (uint32_t)fill;
    }

    // One record per lane with a report: a gss_hit (rec_words 3) or its first
    // word.  Records are streamed out and never read by the sweep:
    // non-temporal stores keep them from displacing table rows in L2 and the
    // memory-side cache.
    __device__ __forceinline__ void words(bool hit, uint32_t row, int len, int word, uint64_t fm,
                                          uint64_t um, int rec_words, int lane) {
        const unsigned long long bal = __ballot(hit);
        if (!bal) return;
        const int n = __popcll(bal);
        if (room(n, lane) && hit) {
            const size_t r = (size_t)chunk * kHitChunk + fill + prefix_count(bal);
            uint64_t *dst = (uint64_t *)hits + r * (size_t)rec_words;
            __builtin_nontemporal_store(
                (uint64_t)row | ((uint64_t)len << 32) | ((uint64_t)word << 48), dst);
            if (rec_words == 3) {
                __builtin_nontemporal_store(fm, dst + 1);
                __builtin_nontemporal_store(um, dst + 2);
            }
        }
        fill += n;
    }

    // One gss_hit_clause per lane with hit set: its clause and the words with
    // a report.
    __device__ __forceinline__ void clause(bool hit, uint32_t row, int len, uint64_t wm,
                                           int lane) {
        const unsigned long long bal = __ballot(hit);
        if (!bal) return;
        const int n = __popcll(bal);
        if (room(n, lane) && hit) {
            const size_t r = (size_t)chunk * kHitChunk + fill + prefix_count(bal);
            uint64_t *dst = (uint64_t *)hits + r * 2;
            __builtin_nontemporal_store((uint64_t)row | ((uint64_t)len << 32), dst);
            __builtin_nontemporal_store(wm, dst + 1);
        }
        fill += n;
    }
};

// Passes (parts of them, if split) [first, first + n) of one bucket.
struct Run {
    LitPtr lits;  // of the bucket
    int len, count, first, n;
};

// Calls run(Run) for every run of passes that belongs to this wave.
template <int CPW, bool SCREENED, typename F>
__device__ __forceinline__ void walk(const SweepArgs &a, const Passes &ps, int lane, F &&run) {
    for (int64_t t = ps.gw;; t += ps.nw) {
        const int64_t first = t * ps.tp;
        if (first >= ps.total) break;
        int p = (int)first;
        const int end = ps.total - p < ps.tp ? ps.total : p + ps.tp;
        int bi = find_bucket<SCREENED>(a.buckets, ps.nbuckets, p >> ps.split, lane);
        while (p < end) {
            const BucketDesc d = a.buckets[bi];
            Run r;
            r.lits = (LitPtr)uniform64((uint64_t)d.lits);
            r.len = uniform((int)d.len);
            r.count = uniform((int)d.count);
            r.first = p - (uniform((int)pass_begin<SCREENED>(d)) << ps.split);
            const int have = (((r.count - 1) / CPW + 1) << ps.split) - r.first;
            r.n = end - p < have ? end - p : have;
            const int n = r.n;
            run(r);
            p += n;
            bi++;
        }
    }
}

// The exact check of one clause per W lanes, one table word per lane: the
// clause's literals at cl (len, the same in all lanes, of them; cur: those held)
// and its first two rows of the lane's word.  Slots in dead are not looked at;
// on = false: no clause.  All 64 lanes call it; a lane stops reading rows once
// its 64 slots are dead, and the check ends when every lane is.
//
// The rows are the traffic (a line per row and 16 words), so the schedule
// reads few of them: two per step up to the sixth, then one (random 1024-slot
// clauses of 8 literals and more die after the sixth to eighth: 642 us with pairs
// throughout, 618 so); and, only for lanes left with a slot of exactly one
// non-false literal, the negated row of that literal alone (the first ROWS
// literals' rows are kept in registers for it; past those every negated row is
// read).  A per-step choice by the number of live lanes read as few rows but
// spilled: 845 us.
//
// Below 8 words ROWS rows are read per step past the held literals (4 beside the
// screening code, where 8 would spill).
template <int W, int ROWS = kRows>
__device__ __forceinline__ void check_clause(const uint64_t *__restrict__ table, LitPtr cl,
                                             int len, int q, bool on, uint32_t w8,
                                             uint32_t sentinel, uint64_t dead, const Lits<W> &cur,
                                             uint64_t x0, uint64_t x1, uint64_t &fm,
                                             uint64_t &um) {
    constexpr int H = Lits<W>::kHeld;
    constexpr int kKeep = H < ROWS ? H : ROWS;
    uint64_t c2 = dead, c1 = dead;
    uint64_t f[kKeep];
    f[0] = x0;
    f[1] = x1;
    auto fold = [&](uint64_t x) {
        c2 |= c1 & x;
        c1 |= x;
    };
    fold(x0);
    fold(x1);
    // two rows from position J of the literals l; rows kept when J is
    // among the first kKeep of the clause
    auto step = [&]<int J, bool KEEP>(const Lits<W> &l) {
        const uint32_t o0 = scale_offset<W>(lit_at<W, J>(l)) | w8;
        const uint32_t o1 = scale_offset<W>(lit_at<W, J + 1>(l)) | w8;
        if (c2 != ~0ull) {
            const uint64_t y0 = load_word(table, o0), y1 = load_word(table, o1);
            if constexpr (KEEP) {
                f[J % kKeep] = y0;
                f[(J + 1) % kKeep] = y1;
            }
            fold(y0);
            fold(y1);
        }
        return __ballot(c2 != ~0ull) != 0;
    };
    auto step1 = [&]<int J, bool KEEP>(const Lits<W> &l) {
        const uint32_t o0 = scale_offset<W>(lit_at<W, J>(l)) | w8;
        if (c2 != ~0ull) {
            const uint64_t y0 = load_word(table, o0);
            if constexpr (KEEP) f[J % kKeep] = y0;
            fold(y0);
        }
        return __ballot(c2 != ~0ull) != 0;
    };
    bool go = len > 2 && __ballot(c2 != ~0ull) != 0;
    constexpr int P2 = H / 2 - 1 < 2 ? H / 2 - 1 : 2;
    [&]<int... I>(std::integer_sequence<int, I...>) {
        ((go = go && 2 * I + 2 < len &&
               step.template operator()<2 * I + 2, (2 * I + 2 < kKeep)>(cur)),
         ...);
    }(std::make_integer_sequence<int, P2>{});
    [&]<int... I>(std::integer_sequence<int, I...>) {
        ((go = go && 2 + 2 * P2 + I < len &&
               step1.template operator()<2 + 2 * P2 + I, (2 + 2 * P2 + I < kKeep)>(cur)),
         ...);
    }(std::make_integer_sequence<int, H - 2 - 2 * P2>{});
    if constexpr (W < 8) {
        if (go && len > H) {
            constexpr int R = ROWS / H;
            Lits<W> l[R];
#pragma unroll
            for (int s = 0; s < R; s++)
                l[s] = load_lits<W>(cl, H + s * H, len, q, on, sentinel);
            for (int base = H; base < len && go; base += R * H) {
                Lits<W> next[R];
                uint32_t o[R * H];
#pragma unroll
                for (int s = 0; s < R; s++)
                    next[s] = load_lits<W>(cl, base + (R + s) * H, len, q, on,
                                           sentinel);
                [&]<int... I>(std::integer_sequence<int, I...>) {
                    ((o[I] = scale_offset<W>(lit_at<W, I % H>(l[I / H])) | w8), ...);
                }(std::make_integer_sequence<int, R * H>{});
                if (c2 != ~0ull) {
                    uint64_t y[R * H];
#pragma unroll
                    for (int i = 0; i < R * H; i++) y[i] = load_word(table, o[i]);
#pragma unroll
                    for (int i = 0; i < R * H; i++) fold(y[i]);
                }
                go = __ballot(c2 != ~0ull) != 0;
#pragma unroll
                for (int s = 0; s < R; s++) l[s] = next[s];
            }
        }
    } else if (go && len > H) {
        for (int base = H; base < len && go; base += H) {
            const Lits<W> l = load_lits<W>(cl, base, len, q, on, sentinel);
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ((go = go && base + 2 * I < len &&
                       step.template operator()<2 * I, false>(l)),
                 ...);
            }(std::make_integer_sequence<int, H / 2>{});
        }
    }
    fm = ~c1;
    um = c1 & ~c2;  // exactly one non-false literal
    if (__ballot(um != 0)) {
        // a slot's one non-false literal must not be true there
        auto neg_row = [&]<int J>(const Lits<W> &l, bool need) {
            const uint32_t o = (scale_offset<W>(lit_at<W, J>(l)) ^ neg_bit<W>()) | w8;
            return need ? load_word(table, o) : ~0ull;
        };
        [&]<int... I>(std::integer_sequence<int, I...>) {
            uint64_t rest = um, t[kKeep];
            ((t[I] = I < len ? neg_row.template operator()<I>(cur, (f[I] & um) != 0)
                             : ~0ull),
             ...);
            ((rest &= I < len ? ~f[I] : ~0ull), ...);
            ((um &= t[I]), ...);
            // positions past the kept rows, for the slots left over
            constexpr int R = W < 8 ? ROWS / H : 1;
            for (int base = kKeep; base < len && __ballot((rest & um) != 0);
                 base += R * kKeep) {
                Lits<W> l[R];
                uint64_t u[R][kKeep];
#pragma unroll
                for (int s = 0; s < R; s++)
                    l[s] = load_lits<W>(cl, base + s * kKeep, len, q, on,
                                        sentinel);
                const bool need = (rest & um) != 0;
#pragma unroll
                for (int s = 0; s < R; s++)
                    ((u[s][I] = base + s * kKeep + I < len
                                    ? neg_row.template operator()<I>(l[s], need)
                                    : ~0ull),
                     ...);
#pragma unroll
                for (int s = 0; s < R; s++) ((um &= ~rest | u[s][I]), ...);
            }
        }(std::make_integer_sequence<int, kKeep>{});
    }
}

// Every clause checked: W lanes check one clause, one table word per lane, 64 / W
// clauses per wave pass, the first two rows of each prefetched during the pass
// before.
template <int W, bool CLAUSES>
__global__ GSS_SWEEP_BOUNDS void k_sweep(SweepArgs a) {
    if (a.choose && screen_chosen(a.choose)) return;  // the screened kernel's
    constexpr int CPW = 64 / W;  // clauses per wave pass
    const int lane = (int)__lane_id();
    const int c = lane / W;           // clause of the pass
    const int w = lane % W;           // table word
    const int q = lane % Lits<W>::G;  // literal of the group's registers
    const uint32_t w8 = (uint32_t)w * 8u;
    const uint64_t valid = a.valid[w];
    const uint64_t *__restrict__ table = a.table;
    const Passes ps(a, false, 1);
    HitWriter out(a, ps);

    walk<CPW, false>(a, ps, lane, [&](const Run &run) {
        const int len = run.len, n = run.n;
        const int row0 = run.first * CPW;   // of the run's first pass
        const int left = run.count - row0;  // rows from there on
        const LitPtr cl = run.lits + (size_t)row0 * len;
        auto clause = [&](int pass) {
            return cl + (size_t)(uint32_t)(pass * CPW + c) * (uint32_t)len;
        };
        auto lits_of = [&](int pass) {
            return load_lits<W>(clause(pass), 0, len, q, pass < n && pass * CPW + c < left,
                                a.sentinel);
        };
        auto row = [&]<int J>(const Lits<W> &l) {
            return load_word(table, scale_offset<W>(lit_at<W, J>(l)) | w8);
        };
        // Clause records wait, one per lane, for W passes' clauses: written pass by
        // pass they took 13 % of a sweep of 64 words where most clauses have one
        // (a batched step of random clauses: 1.545 ms, 1.339 now).
        uint64_t found = 0;
        // One pass: its held literals and first two rows.
        auto check = [&](int pass, const Lits<W> &cur, uint64_t x0, uint64_t x1) {
            const int r = pass * CPW + c;
            const bool on = r < left;
            uint64_t fm, um;
            // invalid slots (and lanes without a clause) start dead
            check_clause<W>(table, clause(pass), len, q, on, w8, a.sentinel, on ? ~valid : ~0ull,
                            cur, x0, x1, fm, um);
            const bool hit = (fm | um) != 0;
            if constexpr (CLAUSES) {
                const unsigned long long bw = __ballot(hit);
                if (bw && pass % W == lane / CPW) {
                    const int k = lane % CPW;  // its clause of the pass
                    found = W == 64 ? bw : (bw >> (k * W)) & ((1ull << (W & 63)) - 1ull);
                }
            } else {
                out.words(hit, (uint32_t)(row0 + r), len, w, fm, um, a.rec_words, lane);
            }
        };
        auto flush = [&](int pass) {
            if (__ballot(found != 0))
                out.clause(found != 0, (uint32_t)(row0 + pass / W * 64 + lane), len, found, lane);
            found = 0;
        };
        // Two passes per turn: the rows of one are in flight while the other
        // is checked, and the literals of the next two (separate registers: a
        // rotation would wait for what it copies).
        Lits<W> la = lits_of(0), lb = lits_of(1);
        uint64_t a0 = row.template operator()<0>(la), a1 = row.template operator()<1>(la);
        for (int pass = 0; pass < n; pass += 2) {
            const uint64_t b0 = row.template operator()<0>(lb), b1 = row.template operator()<1>(lb);
            const Lits<W> na = lits_of(pass + 2), nb = lits_of(pass + 3);
            check(pass, la, a0, a1);
            a0 = row.template operator()<0>(na);
            a1 = row.template operator()<1>(na);
            if constexpr (CLAUSES && W == 1) flush(pass);
            if (pass + 1 < n) check(pass + 1, lb, b0, b1);
            if constexpr (CLAUSES) {
                if (W == 1 ? pass + 1 < n : (pass + 2) % W == 0 || pass + 2 >= n)
                    flush(W == 1 ? pass + 1 : pass);
            }
            la = na;
            lb = nb;
        }
    });
    out.end(lane);
}

// ---- screened sweeps -----------------------------------------------------------

// One clause per lane: the groups in which it can report, i.e. where none of
// its literals (its row of len stored offsets) is true in every valid slot and
// fewer than two occurrences are non-false in every valid slot (SweepArgs::agg);
// 0 once none is left.  unknown (where some are): its (literal, group) pairs,
// groups in gdead aside, whose entry is neither non-false nor false.  Literals
// are read four at a time, the entries two per vote.
__device__ __forceinline__ uint32_t lane_agg(LitPtr row, int len,
                                             const uint32_t *__restrict__ agg, uint32_t gdead,
                                             int &unknown) {
    typedef uint32_t Vec __attribute__((ext_vector_type(4), aligned(4)));
    uint32_t a1 = 0, a2 = gdead;  // groups with a non-false occurrence / that cannot report
    unknown = 0;
    for (int j = 0; j < len; j += 4) {
        uint32_t l[4] = {};
        if (j + 4 <= len) {
            const Vec v = *(const __attribute__((address_space(1))) Vec *)(row + j);
#pragma unroll
            for (int u = 0; u < 4; u++) l[u] = v[u];
        } else {
#pragma unroll
            for (int u = 0; u < 3; u++)
                if (j + u < len) l[u] = row[j + u];
        }
#pragma unroll
        for (int u = 0; u < 4; u += 2) {
            if (j + u >= len) break;
            const uint32_t e0 = agg[l[u] >> 8], e1 = agg[l[u + 1] >> 8];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (j + u + k >= len) break;
                const uint32_t at = (l[u + k] >> 3) & 16u, e = k ? e1 : e0;
                const uint32_t x = e >> at, no = e >> (at ^ 16u);
                a2 |= (a1 & x) | (x >> 8);
                a1 |= x;
                unknown += __popc(~(x | (no >> 8) | gdead) & 0xFFu);
            }
            if ((a2 & 0xFFu) == 0xFFu) return 0;
        }
    }
    return ~a2 & 0xFFu;
}

// Position of set bit number r (r < popcount(m)) of m.
__device__ __forceinline__ int nth_bit(uint64_t m, int r) {
    int pos = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const int k = __popcll(m & ((1ull << s) - 1ull));
        if (r >= k) {
            r -= k;
            m >>= s;
            pos += s;
        }
    }
    return pos;
}

// P neighbouring words of a row, from byte offset off of the table.
template <int P>
struct RowWords {
    uint64_t w[P];
};

template <int P>
__device__ __forceinline__ RowWords<P> load_words(const uint64_t *__restrict__ table,
                                                  uint32_t off) {
    RowWords<P> r;
    if constexpr (P == 2) {
        const ulonglong2 x = *(const ulonglong2 *)((const char *)table + off);
        r.w[0] = x.x;
        r.w[1] = x.y;
    } else {
        r.w[0] = load_word(table, off);
    }
    return r;
}

// One clause and P words of the table per lane: the clause's len stored offsets
// at cl, the words from byte offset w8 of a row (word p of screening group
// g[p]), the slots not in dead.  All 64 lanes call it (len is uniform).
//
// A literal that its entry has non-false, or its negation true, in every slot
// of a word's group needs no row: it is all ones or all zeros there.  A row is a
// line from memory; the entries (4 MB for 1M variables) mostly stay in L2.  On 3M
// clauses x 2176 slots 6.6M lines were read, 5.4M so: 152 us, 143 now.
template <int W, int P>
__device__ __forceinline__ void check_words(LitPtr cl, int len,
                                            const uint64_t *__restrict__ table,
                                            const uint32_t *__restrict__ agg, uint32_t w8,
                                            const uint32_t (&g)[P], const uint64_t (&dead)[P],
                                            uint64_t (&fm)[P], uint64_t (&um)[P]) {
    uint64_t c1[P], c2[P];
    bool alive = false;
#pragma unroll
    for (int p = 0; p < P; p++) {
        c1[p] = c2[p] = dead[p];
        alive |= dead[p] != ~0ull;
    }
    // positions (the last one: all from 31 on) where the literal may be true in
    // a slot that has it as its one non-false literal
    uint32_t open = 0;
    const auto take = [&](int j, uint32_t l, uint32_t e) {
        const uint32_t own = e >> ((l >> 3) & 16u), neg = e >> (~(l >> 3) & 16u);
        uint64_t x[P];
        bool read = false, tru = false;
#pragma unroll
        for (int p = 0; p < P; p++) {
            const bool nf = (own >> g[p]) & 1u;
            x[p] = nf ? ~0ull : 0ull;
            read |= !nf && !((neg >> (8 + g[p])) & 1u) && c2[p] != ~0ull;
        }
        if (read) {
            const RowWords<P> r = load_words<P>(table, scale_offset<W>(l) | w8);
#pragma unroll
            for (int p = 0; p < P; p++) x[p] = r.w[p];
        }
#pragma unroll
        for (int p = 0; p < P; p++) {
            tru |= (x[p] & ~c2[p]) != 0 && !((neg >> g[p]) & 1u);
            c2[p] |= c1[p] & x[p];
            c1[p] |= x[p];
        }
        if (tru) open |= 1u << (j < 31 ? j : 31);
    };
    uint32_t l0 = 0, l1 = 0, e0 = 0, e1 = 0;
    if (alive) {
        l0 = cl[0];
        if (len > 1) l1 = cl[1];
        e0 = agg[l0 >> 8];
        e1 = agg[l1 >> 8];
    }
    for (int j = 0; j < len && __ballot(alive); j += 2) {
        if (!alive) continue;
        const uint32_t a0 = l0, a1 = l1, x0 = e0, x1 = e1;
        if (j + 2 < len) {
            l0 = cl[j + 2];
            l1 = j + 3 < len ? cl[j + 3] : 0u;
            e0 = agg[l0 >> 8];
            e1 = agg[l1 >> 8];
        }
        take(j, a0, x0);
        if (j + 1 < len) take(j + 1, a1, x1);
        alive = false;
#pragma unroll
        for (int p = 0; p < P; p++) alive |= c2[p] != ~0ull;
    }
    bool unit = false;
#pragma unroll
    for (int p = 0; p < P; p++) {
        fm[p] = ~c1[p];
        um[p] = c1[p] & ~c2[p];
        unit |= um[p] != 0;
    }
    // a negated row has ones where the literal is not true
    if (!unit) open = 0;
    while (__ballot(open != 0)) {
        if (open) {
            int j = __ffs(open) - 1;
            open &= open - 1;
            const int last = j == 31 ? len : j + 1;
            for (; j < last; j++) {
                const RowWords<P> x =
                    load_words<P>(table, (scale_offset<W>(cl[j]) ^ neg_bit<W>()) | w8);
#pragma unroll
                for (int p = 0; p < P; p++) um[p] &= x.w[p];
            }
        }
    }
}

// Clauses screened against a.agg first (serving and screened steps, sweeps where
// that pays).  A wave screens 64 clauses, one per lane, and checks what is left
// of them exactly, in one of two ways:
//
// Few words left, or rows mostly known from the entries: the words are spread
// over the wave, two neighbouring ones (16 bytes of a row) per lane, whatever
// clause they belong to (a word per lane: 167 us where two take 152; a clause per
// 16 lanes kept most lanes idle, as a clause survives in one or two of its eight
// word groups).  A lane follows one literal after the other, with the entries.
//
// Else, clause after clause as in k_sweep, W lanes each: every row is read, but
// several at a time and whole lines of it.
//
// The first way costs a wave about len * (2 + 8 u) per 64 items, u the share of
// unknown (literal, group) pairs of the clauses left, the second len * kDense / 10
// per clause (the two were equal at u = 0.4 with 1 word, 0.25 with 4, 0.15 with 8
// and 16, 0.4 with 64, clauses of 12 literals nine in ten false).  From 24 literals
// on the chain of reads decides, and with an eighth of the words left the second
// way is the faster.  Measured with the first way alone, now, and as a group of
// 16 lanes per clause did: 2M clauses x 16 words, slots of two in five words
// differing 1602, 1046, 1137 us; 600k x 64 words 2274, 910, 1006; 40k clauses of
// 150 to 400 literals x 16 words, which 625 waves checked before passes were split
// 18061, 1560, 1858; 3M x 1 word 791, 644, 918.
constexpr int kDenseLen = 24;
template <int W, bool CLAUSES>
__global__ __attribute__((amdgpu_num_sgpr(96))) __launch_bounds__(256, 7) void k_sweep_screened(SweepArgs a) {
    if (a.choose && !screen_chosen(a.choose)) return;  // the plain kernel's
    constexpr int P = W == 1 ? 1 : 2;  // words of an item
    constexpr int kDense = W <= 16 ? 50 + 5 * W : 17 * W;
    __shared__ uint64_t s_valid[W], s_words[4][64], s_hit[4][64];
    __shared__ uint32_t s_start[4][64], s_group[W];
    const int lane = (int)__lane_id(), wv = (int)(threadIdx.x >> 6);
    if (threadIdx.x < W) {
        s_valid[threadIdx.x] = a.valid[threadIdx.x];
        uint32_t g = 0;
        for (int b = 1; b < 8; b++)
            if ((a.agg_words[b] >> threadIdx.x) & 1ull) g = (uint32_t)b;
        s_group[threadIdx.x] = g;
    }
    __syncthreads();
    uint32_t gdead = 0;  // groups without a word
    for (int b = 0; b < 8; b++)
        if (!a.agg_words[b]) gdead |= 1u << b;
    const int live = 8 - __popc(gdead);
    const Passes ps(a, true, W);
    HitWriter out(a, ps);

    const int part = 64 >> ps.split;  // clauses at a time
    walk<64, true>(a, ps, lane, [&](const Run &run) {
        const int len = run.len, count = run.count;
        const float sixteenth = 16.0f / (float)(live * len);
        for (int pass = 0; pass < run.n; pass++) {
            const int row0 = (run.first + pass) * part;
            const LitPtr cl = run.lits + (size_t)row0 * len;
            int unknown = 0;
            const uint32_t grp =
                lane < part && row0 + lane < count
                    ? lane_agg(cl + (size_t)lane * len, len, a.agg, gdead, unknown)
                    : 0u;
            uint64_t left = __ballot(grp != 0);  // clauses to check
            if (!left) continue;
            uint64_t m = 0;  // table words to check
#pragma unroll
            for (int b = 0; b < 8; b++)
                if ((grp >> b) & 1u) m |= a.agg_words[b];
            // bit w: words w .. w + P - 1 are an item
            const uint64_t items = P == 1 ? m : (m | (m >> 1)) & 0x5555555555555555ull;
            const int cnt = __popcll(items);
            // items in the low half, 16ths of unknown pairs in the upper
            const int add = cnt | (grp ? (int)((float)unknown * sixteenth) << 16 : 0);
            int incl = add;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int y = __shfl_up(incl, d);
                if (lane >= d) incl += y;
            }
            const int sums = uniform(__shfl(incl, 63));
            const int total = sums & 0xFFFF, surv = __popcll(left);
            incl = (incl - add) & 0xFFFF;
            s_start[wv][lane] = (uint32_t)incl;
            s_words[wv][lane] = m;
            if constexpr (CLAUSES) s_hit[wv][lane] = 0;
            __builtin_amdgcn_wave_barrier();
            const bool dense =
                len >= kDenseLen ? 8 * total >= surv * W
                                 : 5 * total * (4 * surv + (sums >> 16)) >= surv * surv * kDense;
            if (dense) {
                constexpr int CPW = 64 / W;
                const int c = lane / W, w = lane % W, q = lane % Lits<W>::G;
                const uint32_t w8 = (uint32_t)w * 8u;
                // the lane's clause among those left, its literals
                int i;
                bool on;
                Lits<W> held;
                const auto next = [&] {
                    on = c < __popcll(left);
                    i = on ? nth_bit(left, c) : 0;
                    held = load_lits<W>(cl + (size_t)i * len, 0, len, q, on, a.sentinel);
                    left = __popcll(left) > CPW ? left & (~0ull << nth_bit(left, CPW)) : 0ull;
                };
                next();
                for (bool more = true; more;) {
                    const int at = i;
                    const bool in = on;
                    const Lits<W> cur = held;
                    more = left != 0;
                    if (more) next();
                    const uint64_t dead =
                        in && ((s_words[wv][at] >> w) & 1ull) ? ~s_valid[w] : ~0ull;
                    const uint32_t o0 = scale_offset<W>(lit_at<W, 0>(cur)) | w8;
                    const uint32_t o1 = scale_offset<W>(lit_at<W, 1>(cur)) | w8;
                    uint64_t x0 = 0, x1 = 0, fm, um;
                    if (dead != ~0ull) {
                        x0 = load_word(a.table, o0);
                        x1 = load_word(a.table, o1);
                    }
                    check_clause<W, 4>(a.table, cl + (size_t)at * len, len, q, in, w8, a.sentinel,
                                       dead, cur, x0, x1, fm, um);
                    const bool hit = (fm | um) != 0;
                    if constexpr (CLAUSES) {
                        const uint64_t bw = __ballot(hit);
                        if (in && w == 0)
                            s_hit[wv][at] =
                                W == 64 ? bw : (bw >> lane) & ((1ull << (W & 63)) - 1ull);
                    } else {
                        out.words(hit, (uint32_t)(row0 + at), len, w, fm, um, a.rec_words, lane);
                    }
                }
            }
            for (int base = 0; !dense && base < total; base += 64) {
                const int item = base + lane;
                const bool on = item < total;
                // the clause it belongs to: the last one that starts at or before it
                int i = 0;
#pragma unroll
                for (int s = 32; s > 0; s >>= 1)
                    if (i + s < 64 && (int)s_start[wv][i + s] <= item) i += s;
                const uint64_t mi = s_words[wv][i];
                const int w = on ? nth_bit(P == 1 ? mi : (mi | (mi >> 1)) & 0x5555555555555555ull,
                                           item - (int)s_start[wv][i])
                                 : 0;
                uint64_t dead[P], fm[P], um[P];
                uint32_t g[P];
#pragma unroll
                for (int p = 0; p < P; p++) {
                    dead[p] = on && ((mi >> (w + p)) & 1ull) ? ~s_valid[w + p] : ~0ull;
                    g[p] = s_group[w + p];
                }
                check_words<W, P>(cl + (size_t)i * len, len, a.table, a.agg, (uint32_t)w * 8u, g,
                                  dead, fm, um);
                if constexpr (CLAUSES) {
                    uint64_t hit = 0;
#pragma unroll
                    for (int p = 0; p < P; p++)
                        if (fm[p] | um[p]) hit |= 1ull << (w + p);
                    if (hit) atomicOr((unsigned long long *)&s_hit[wv][i], hit);
                } else {
#pragma unroll
                    for (int p = 0; p < P; p++)
                        out.words((fm[p] | um[p]) != 0, (uint32_t)(row0 + i), len, w + p, fm[p],
                                  um[p], a.rec_words, lane);
                }
            }
            __builtin_amdgcn_wave_barrier();
            if constexpr (CLAUSES) {
                const uint64_t wm = s_hit[wv][lane];
                out.clause(wm != 0, (uint32_t)(row0 + lane), len, wm, lane);
            }
            __builtin_amdgcn_wave_barrier();
        }
    });
    out.end(lane);
}

// Bit b of a variable's screening entries (SweepArgs::agg; one 32-bit word per
// variable): literal v non-false / true, literal ~v non-false / true in every
// slot of group b.
__device__ __forceinline__ void agg_set(uint32_t *entry, uint32_t b, bool nf, bool tr, bool nfn,
                                        bool trn) {
    const uint32_t m = 0x01010101u << b;
    const uint32_t x =
        ((nf ? 1u : 0u) | (tr ? 0x100u : 0u) | (nfn ? 0x10000u : 0u) | (trn ? 0x1000000u : 0u))
        << b;
    if (x) atomicOr(entry, x);
    if (x != m) atomicAnd(entry, ~(m & ~x));
}

__global__ void k_reset_u32(uint32_t *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_fill_u64(uint64_t *p, int64_t n, uint64_t v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Copies segments of uint32; with shift > 0 each element is shifted left
// (literal -> stored row offset on clause upload).
__global__ void k_scatter(const ScatterSeg *__restrict__ segs, int nseg,
                          const uint32_t *__restrict__ src, int shift) {
    for (int s = blockIdx.x; s < nseg; s += gridDim.x) {
        const ScatterSeg sg = segs[s];
        for (uint64_t i = threadIdx.x; i < sg.count; i += blockDim.x)
            sg.dst[i] = src[sg.src + i] << shift;
    }
}

// Row 2v holds the slots where literal 2v (v) is not false, i.e. v is not
// false; row 2v+1 the slots where v is not true.
__global__ void k_assig_apply(const gss_var_update *__restrict__ ups, int64_t n,
                              uint64_t *__restrict__ table, int words) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const gss_var_update u = ups[i];
    const size_t base = (size_t)u.var * 2 * words + u.word;
    table[base] = ~(u.is_def & ~u.is_true);
    table[base + words] = ~(u.is_def & u.is_true);
}

__global__ void k_assig_roll(const gss_var_update *__restrict__ ups, int64_t n,
                             uint64_t *__restrict__ table, int words,
                             const int8_t *__restrict__ last_pos) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const gss_var_update u = ups[i];
    const int p = last_pos[u.word];
    if (p < 0) return;
    const size_t base = (size_t)u.var * 2 * words + u.word;
    const uint64_t f = table[base], t = table[base + words];
    table[base] = ((f >> p) & 1ull) ? ~0ull : 0ull;
    table[base + words] = ((t >> p) & 1ull) ? ~0ull : 0ull;
}

// Screening entries of a variable where a word is its own group (at most 8
// words): the word's bits, from the variable's rows f and t there.
__device__ __forceinline__ void agg_word_bits(uint32_t *agg, uint32_t var, uint32_t word,
                                              uint64_t f, uint64_t t) {
    agg_set(agg + var, word, f == ~0ull, t == 0, t == ~0ull, f == 0);
}

// ---- batched steps: fixed launch shapes, counts from device memory --------

__device__ __forceinline__ void base_update(const gss_base_update &x, uint64_t *bases,
                                            int64_t vw) {
    const uint64_t bit = 1ull << (x.var & 63);
    unsigned long long *def = (unsigned long long *)bases + (size_t)(2 * x.base) * vw + x.var / 64;
    unsigned long long *tru = def + vw;
    if (x.is_def) atomicOr(def, bit);
    else atomicAnd(def, ~bit);
    if (x.is_def && x.is_true) atomicOr(tru, bit);
    else atomicAnd(tru, ~bit);
}

// Admission of a serving step: in sequence order, the published requests whose
// words fit the table.  One wave reads the ring (two reads over PCIe, one
// after the other) while the header is on its way, and fills the header in
// once it is there.
struct ServePending {
    uint64_t tail, patch_off;
    uint32_t solver, k, n_patches;
    int avail;
};

__device__ __forceinline__ ServePending serve_pending(const ServeRing &r, int lane) {
    ServePending p{};
    p.tail = *r.tail;
    // published by the host with a release store after the entries
    uint64_t head = 0;
    if (lane == 0) head = __hip_atomic_load(r.head, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
    head = uniform64(head);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");  // later reads see the published entries
    const uint64_t pend = head > p.tail ? head - p.tail : 0;
    p.avail = (int)(pend < (uint64_t)kServeMaxRequests ? pend : kServeMaxRequests);
    if (lane < p.avail) {
        const volatile ServeReq *q = r.reqs + (p.tail + lane) % r.req_cap;
        p.solver = q->solver;
        p.k = q->k;
        p.n_patches = q->n_patches;
        p.patch_off = q->patch_off;
    }
    return p;
}

__device__ __forceinline__ void serve_admit(const ServePending &p, const ServeRing &r,
                                            StepHeader *dh, gss_word_load *loads,
                                            ServeReport *report, int words, int lane) {
    const int avail = p.avail;
    const uint32_t k = p.k, np = p.n_patches;
    const uint64_t nw = lane < avail ? (k + 63u) / 64u : 0;
    const uint64_t end = wave_incl_scan(nw, lane);
    // end grows with the lane (every request takes at least one word), so
    // the requests that fit are a prefix
    const bool fits = lane < avail && end <= (uint64_t)words;
    const unsigned long long bal = __ballot(fits);
    const int count = __popcll(bal);
    const uint64_t pend_p = wave_incl_scan(fits ? (uint64_t)np : 0, lane);
    const uint64_t used = __shfl(end, count > 0 ? count - 1 : 0);
    const uint64_t total_words = count > 0 ? used : 0;
    const uint64_t total_patches = __shfl(pend_p, count > 0 ? count - 1 : 0);
    if (fits) {
        const uint32_t w0 = (uint32_t)(end - nw);
        ServeAdmitted a;
        a.patch_off = p.patch_off;
        a.patch_pfx = pend_p - np;
        a.n_patches = np;
        a.w0 = w0;
        r.adm[lane] = a;
        for (uint32_t j = 0; j < (uint32_t)nw; j++) {
            gss_word_load ld;
            ld.word = (uint16_t)(w0 + j);
            ld.base = (uint16_t)p.solver;
            loads[w0 + j] = ld;
            const uint32_t last = k - 64u * j;  // slots of this word
            dh->valid[w0 + j] = last >= 64u ? ~0ull : ((1ull << last) - 1ull);
        }
    }
    // words no request took are not checked
    if ((uint64_t)lane < (uint64_t)GSS_MAX_WORDS && (uint64_t)lane >= total_words)
        dh->valid[lane] = 0ull;
    if (lane == 0) {
        *r.adm_count = (uint32_t)count;
        dh->nloads = (int64_t)total_words;
        dh->npatches = count > 0 ? (int64_t)total_patches : 0;
        if (count == 0) dh->npasses = dh->screen_passes = 0;  // nothing to check
        *r.tail = p.tail + (uint64_t)count;
        report->first = p.tail;
        report->count = (uint32_t)count;
        report->words = (uint32_t)total_words;
    }
}

// A step's inputs from pinned host memory: the header (which comes with the
// launch) and the regions a later kernel reads are copied, the counters of its
// sweep cleared, and -- straight from the staging, each byte crossing PCIe once
// -- its clauses copied to their rows (a.clauses), its base updates and its
// updates applied (a.apply).  Staging first and applying in kernels after it
// took 3 launches more, 3-5 us each on a step of few updates.  A serving step's
// requests are admitted by the first block.
//
// Updates go through LDS, 256 at a time, so that the 24-byte records are read
// in whole lines.
__global__ __launch_bounds__(256) void k_step_in(StepInArgs a) {
    const StepHeader &h = a.header;
    static_assert(sizeof(StepHeader) / 4 <= 192, "three waves copy the header");
    if (blockIdx.x == 0 && threadIdx.x < 2) a.alloc[threadIdx.x] = 0;
    if (a.counts && blockIdx.x == 1 && threadIdx.x < 2 * GSS_MAX_WORDS) a.counts[threadIdx.x] = 0;
    if (*a.halt) {
        // halted: a header with no work (and `halted` set) instead of the step
        constexpr int kFlag = (int)(offsetof(StepHeader, halted) / 4);
        if (blockIdx.x == 0 && threadIdx.x < sizeof(StepHeader) / 4)
            a.d[kRegHeader][threadIdx.x] = threadIdx.x == kFlag ? 1u : 0u;
        return;
    }
    __shared__ uint64_t s_up[3 * 256];
    if (blockIdx.x == 0) {
        ServePending p{};
        if (threadIdx.x < sizeof(StepHeader) / 4)
            a.d[kRegHeader][threadIdx.x] = ((const uint32_t *)&h)[threadIdx.x];
        else if (threadIdx.x >= 192 && a.report)
            p = serve_pending(a.serve, (int)threadIdx.x & 63);
        __syncthreads();
        if (threadIdx.x >= 192 && a.report)
            serve_admit(p, a.serve, (StepHeader *)a.d[kRegHeader], (gss_word_load *)a.d[kRegLoads],
                        a.report, a.words, (int)threadIdx.x & 63);
    }
    // words of each screening group with a valid slot
    if (a.agg_words && blockIdx.x == 1 && threadIdx.x >= 128 && threadIdx.x < 136) {
        const int b = (int)threadIdx.x - 128, gw = a.words < 8 ? 1 : a.words / 8;
        uint64_t m = 0;
        for (int w = b * gw; w < (b + 1) * gw && w < a.words; w++)
            if (h.valid[w]) m |= 1ull << w;
        a.agg_words[b] = m;
    }
    const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
#pragma unroll
    for (int r = kRegHeader + 1; r < kStageRegions; r++) {
        if (r == kRegBaseUps) continue;  // applied below
        if (r == kRegUps && a.apply) continue;
        if ((r == kRegClauses || r == kRegLits) && a.clauses) continue;
        const uint32_t *src = a.h[r];
        uint32_t *dst = a.d[r];
        // short regions by different blocks, beside the updates' and the
        // clauses': a trip over PCIe takes ~1.5 us, and a block's follow each other
        int64_t i = tid + r * (stride / kStageRegions);
        if (i >= stride) i -= stride;
        for (; i < h.region_words[r]; i += stride) dst[i] = src[i];
    }
    const gss_base_update *bups = (const gss_base_update *)a.h[kRegBaseUps];
    for (int64_t i = tid; i < h.nbups; i += stride) base_update(bups[i], a.bases, a.bases_vw);
    if (a.clauses) {  // eight lanes per clause
        const ClauseSeg *cls = (const ClauseSeg *)a.h[kRegClauses];
        const uint32_t *lits = a.h[kRegLits];
        for (int64_t i = tid >> 3; i < h.nclauses; i += stride >> 3) {
            const ClauseSeg c = cls[i];
            for (uint32_t j = threadIdx.x & 7; j < c.len; j += 8)
                c.dst[j] = lits[(uint64_t)c.src + j] << a.shift;
        }
    }
    if (a.apply) {
        const uint64_t *src = (const uint64_t *)a.h[kRegUps];
        uint64_t *dst = (uint64_t *)a.d[kRegUps];
        for (int64_t t = (int64_t)blockIdx.x * 256; t < h.nups; t += (int64_t)gridDim.x * 256) {
            const int n = h.nups - t < 256 ? (int)(h.nups - t) : 256;
            for (int i = (int)threadIdx.x; i < 3 * n; i += 256) {
                const uint64_t x = src[3 * t + i];
                s_up[i] = x;
                dst[3 * t + i] = x;
            }
            __syncthreads();
            if ((int)threadIdx.x < n) {
                const uint64_t vw = s_up[3 * threadIdx.x];  // {var, word}
                const uint64_t def = s_up[3 * threadIdx.x + 1], tru = s_up[3 * threadIdx.x + 2];
                const uint32_t var = (uint32_t)vw, word = (uint32_t)(vw >> 32);
                const size_t base = (size_t)var * 2 * a.words + word;
                const uint64_t f = ~(def & ~tru), t1 = ~(def & tru);
                a.table[base] = f;
                a.table[base + a.words] = t1;
                if (a.agg) agg_word_bits(a.agg, var, word, f, t1);
            }
            __syncthreads();
        }
    }
}

// Element i covers variable i / nloads and load i % nloads, so the lanes of
// a wave write neighbouring words of the same rows.
__global__ void k_words_load_dyn(const gss_word_load *__restrict__ loads, const int64_t *n_p,
                                 const uint64_t *__restrict__ bases, int64_t vw,
                                 uint64_t *__restrict__ table, int words, int64_t vars) {
    const int64_t nl = *n_p;
    const int64_t total = nl * vars;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = i / nl;
        const gss_word_load ld = loads[i - v * nl];
        const uint64_t *def = bases + (size_t)(2 * ld.base) * vw;
        const uint64_t bit = 1ull << (v & 63);
        const bool d = (def[v >> 6] & bit) != 0;
        const bool t = (def[vw + (v >> 6)] & bit) != 0;
        const size_t row = (size_t)v * 2 * words + ld.word;
        table[row] = (d && !t) ? 0ull : ~0ull;     // literal v is false where v is false
        table[row + words] = (d && t) ? 0ull : ~0ull;  // literal ~v is false where v is true
    }
}

// Slots in mask take the patch's value; the others keep theirs.
__global__ void k_assig_patch_dyn(const gss_var_patch *__restrict__ p, const int64_t *n_p,
                                  uint64_t *__restrict__ table, int words) {
    const int64_t n = *n_p;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const gss_var_patch x = p[i];
        const size_t base = (size_t)x.var * 2 * words + x.word;
        const uint64_t m = x.mask;
        table[base] = (table[base] & ~m) | (~(x.is_def & ~x.is_true) & m);
        table[base + words] = (table[base + words] & ~m) | (~(x.is_def & x.is_true) & m);
    }
}

// Eight lanes per staged clause: lane j copies literals j, j + 8, ...
__global__ void k_scatter_clauses(const ClauseSeg *__restrict__ cls, const int32_t *n_p,
                                  const uint32_t *__restrict__ src, int shift) {
    const int64_t n = *n_p;
    const int lane = threadIdx.x & 7;
    const int64_t ng = ((int64_t)gridDim.x * blockDim.x) >> 3;
    for (int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 3; i < n; i += ng) {
        const ClauseSeg c = cls[i];
        for (uint32_t j = lane; j < c.len; j += 8) c.dst[j] = src[(uint64_t)c.src + j] << shift;
    }
}

__global__ void k_assig_apply_dyn(const gss_var_update *__restrict__ ups, const int64_t *n_p,
                                  uint64_t *__restrict__ table, int words) {
    const int64_t n = *n_p;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const gss_var_update u = ups[i];
        const size_t base = (size_t)u.var * 2 * words + u.word;
        table[base] = ~(u.is_def & ~u.is_true);
        table[base + words] = ~(u.is_def & u.is_true);
    }
}

// One update rolled forward: every slot of its word takes the value of slot
// last_pos[word] (none if negative).
__device__ __forceinline__ void roll_update(const gss_var_update *__restrict__ ups, int64_t i,
                                            uint64_t *__restrict__ table, int words,
                                            const int8_t *__restrict__ last_pos,
                                            uint32_t *agg) {
    const uint32_t var = ups[i].var, word = ups[i].word;
    const int p = last_pos[word];
    if (p < 0) return;
    const size_t base = (size_t)var * 2 * words + word;
    const uint64_t f = ((table[base] >> p) & 1ull) ? ~0ull : 0ull;
    const uint64_t t = ((table[base + words] >> p) & 1ull) ? ~0ull : 0ull;
    table[base] = f;
    table[base + words] = t;
    if (agg) agg_word_bits(agg, var, word, f, t);
}

__global__ void k_assig_roll_dyn(const gss_var_update *__restrict__ ups, const int64_t *n_p,
                                 uint64_t *__restrict__ table, int words,
                                 const int8_t *__restrict__ last_pos) {
    const int64_t n = *n_p;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        roll_update(ups, i, table, words, last_pos, nullptr);
}

// ---- records made dense ---------------------------------------------------------

// Chunks of a sweep of `waves` waves that hold records (at most its buffer's).
__device__ __forceinline__ uint32_t chunks_held(const ChunkArgs &c) {
    const uint32_t used = c.waves + c.alloc[0];
    return used < c.cap ? used : c.cap;
}

// What the host reads: out[0] = the chunks, more than the buffer's if records
// were dropped; out[1], out[2] = low and high word of the records kept.
__device__ __forceinline__ void write_counts(const ChunkArgs &c, uint64_t total, uint32_t *out) {
    out[0] = c.alloc[1] ? c.waves + c.alloc[0] : chunks_held(c);
    out[1] = (uint32_t)total;
    out[2] = (uint32_t)(total >> 32);
}

// Sums of fills[0, at) and fills[0, n) over a block of 256 threads.
__device__ __forceinline__ void sum_fills(const uint32_t *__restrict__ fills, uint32_t at,
                                          uint32_t n, uint64_t &before, uint64_t &total) {
    __shared__ uint64_t s_sum[2][4];
    uint64_t x = 0, y = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 256u * 4) {
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = i + 256u * u < n ? fills[i + 256u * u] : 0u;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            y += v[u];
            if (i + 256u * u < at) x += v[u];
        }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        x += __shfl_xor(x, d);
        y += __shfl_xor(y, d);
    }
    if ((threadIdx.x & 63) == 0) {
        s_sum[0][threadIdx.x >> 6] = x;
        s_sum[1][threadIdx.x >> 6] = y;
    }
    __syncthreads();
    before = s_sum[0][0] + s_sum[0][1] + s_sum[0][2] + s_sum[0][3];
    total = s_sum[1][0] + s_sum[1][1] + s_sum[1][2] + s_sum[1][3];
}

// Words [0, m) of 64 chunks' records (ends: fill_ends) to dst, a thread per
// word and four of them in flight.
template <uint32_t RW>
__device__ __forceinline__ void copy_words(const uint64_t *__restrict__ hits, const uint32_t *ends,
                                           uint32_t m, uint64_t *__restrict__ dst) {
    for (uint32_t i = threadIdx.x; i < m; i += 256 * 4) {
        uint64_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t x = i + 256 * u;
            if (x < m) {
                const uint32_t k = chunk_of(ends, x / RW);
                v[u] = hits[(uint64_t)k * kHitChunk * RW + x - (k ? ends[k - 1] : 0u) * RW];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (i + 256 * u < m) dst[i + 256 * u] = v[u];
    }
}

// Block `blk` of `blocks` (256 threads) of the dense copy: its share of the
// chunks to their place in the dense array.  Every block sums the fills itself
// (32 KB from L2 for a sweep of ~8,000 waves): an offsets kernel before this
// one took longer, on one CU, than the sums do.  Where chunks hold few records
// (at most 128 on average: 40 in a screened step of 280,000) a thread copies a
// word, whatever chunk it is in; with a wave per chunk the block's chunks were
// a chain of reads (k_step_end of a step of 1,930 records: 10.5 us, now 7.6; of
// 285,000: 25.9, now 21.6).  Full chunks take a wave each, without the search.  Records go straight to `host` when
// they take at most host_words there (the wait then has no copy to start),
// else to `dense` if they fit.
__device__ __forceinline__ void gather_block(const ChunkArgs &c, uint32_t blk, uint32_t blocks,
                                             uint64_t *dense, uint64_t dense_cap, uint64_t *host,
                                             uint64_t host_words, uint32_t *out) {
    __shared__ uint32_t s_end[64];
    const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const uint32_t n = chunks_held(c);
    const uint32_t per = (n + blocks - 1) / blocks;
    const uint32_t c0 = blk * per < n ? blk * per : n, c1 = c0 + per < n ? c0 + per : n;
    if (blk != 0 && c0 == c1) return;
    uint32_t fill = c0 + lane < c1 ? c.fills[c0 + lane] : 0u;
    uint64_t at, total;
    sum_fills(c.fills, c0, n, at, total);
    if (out && blk == 0 && threadIdx.x == 0) write_counts(c, total, out);
    if (c.alloc[1]) return;  // records were dropped: the sweep runs again
    const uint32_t rw = c.rec_words;
    uint64_t *to = host && total * rw <= host_words ? host : total <= dense_cap ? dense : nullptr;
    if (!to) return;
    for (uint32_t k0 = c0; k0 < c1; k0 += 64) {
        const uint32_t held = c1 - k0 < 64 ? c1 - k0 : 64;
        fill_ends(fill, s_end);
        __syncthreads();
        const uint32_t records = s_end[63];
        const uint64_t *__restrict__ src = c.hits + (uint64_t)k0 * kHitChunk * rw;
        uint64_t *__restrict__ dst = to + at * rw;
        if (records <= 128 * held) {
            if (rw == 1) copy_words<1>(src, s_end, records, dst);
            else if (rw == 2) copy_words<2>(src, s_end, records * 2, dst);
            else copy_words<3>(src, s_end, records * 3, dst);
        } else {
            for (uint32_t k = wv; k < held; k += 4) {
                const uint32_t first = k ? s_end[k - 1] : 0u, m = (s_end[k] - first) * rw;
                const uint64_t *__restrict__ x = src + (uint64_t)k * kHitChunk * rw;
                uint64_t *__restrict__ y = dst + (uint64_t)first * rw;
                uint32_t i = lane;
                for (; i + 64 * 3 < m; i += 64 * 4) {
                    uint64_t v[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) v[u] = x[i + 64 * u];
#pragma unroll
                    for (int u = 0; u < 4; u++) y[i + 64 * u] = v[u];
                }
                for (; i < m; i += 64) y[i] = x[i];
            }
        }
        at += records;
        if (k0 + 64 < c1) {  // more than 64 chunks in the block's share
            fill = k0 + 64 + lane < c1 ? c.fills[k0 + 64 + lane] : 0u;
            __syncthreads();  // everyone is done with the ends
        }
    }
}

__global__ __launch_bounds__(256) void k_gather(ChunkArgs c, uint64_t *dense, uint64_t dense_cap) {
    gather_block(c, blockIdx.x, gridDim.x, dense, dense_cap, nullptr, 0, nullptr);
}

// Counts of a plain sweep to pinned memory.  The counters are read by the
// gather after it; the next sweep starts from `next`, cleared here.
// `seq` goes to out[3] last: the host waits for it there (ending with the
// stream's own wait instead took 7 us more).
__global__ __launch_bounds__(1024) void k_count_records(ChunkArgs c, uint32_t *out, uint32_t *next,
                                                        uint32_t seq) {
    __shared__ uint64_t part[16];
    const uint32_t n = chunks_held(c);
    uint64_t sum = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 4096u) {
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = i + 1024u * u < n ? c.fills[i + 1024u * u] : 0u;
        sum += (uint64_t)v[0] + v[1] + v[2] + v[3];
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        for (int i = 0; i < 16; i++) t += part[i];
        write_counts(c, t, out);
        next[0] = next[1] = 0;
        __hip_atomic_store(out + 3, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// What follows a step's sweep, in one launch: the first kGatherBlocks blocks
// make its records dense (and write its counts for the host), the others roll
// its updates forward -- unless records were dropped: then the table stays as
// the sweep read it and the engine halts.
constexpr unsigned kGatherBlocks = 512, kRollBlocks = 512;
__global__ __launch_bounds__(256) void k_step_end(ChunkArgs c, StepEndArgs a) {
    if (blockIdx.x < kGatherBlocks) {
        gather_block(c, blockIdx.x, kGatherBlocks, a.dense, a.dense_cap, a.dh->host_rec,
                     a.host_words, a.out);
        return;
    }
    if (c.alloc[1]) {
        if (blockIdx.x == kGatherBlocks && threadIdx.x == 0) *a.halt = 1u;
        return;
    }
    const int64_t n = a.dh->nups;
    for (int64_t i = (blockIdx.x - kGatherBlocks) * (int64_t)256 + threadIdx.x; i < n;
         i += (int64_t)kRollBlocks * 256)
        roll_update(a.ups, i, a.table, a.words, a.dh->last_pos, a.agg);
}

// ---- records grouped by assignment word (serving steps) ----------------------

// f(record) for every record of the block's share of the chunks, a thread per
// record (as in gather_block).
template <typename F>
__device__ __forceinline__ void for_records(const ChunkArgs &ch, F &&f) {
    __shared__ uint32_t s_end[64];
    const uint32_t n = chunks_held(ch), rw = ch.rec_words;
    const uint32_t per = (n + gridDim.x - 1) / gridDim.x;
    const uint32_t c0 = blockIdx.x * per, c1 = c0 + per < n ? c0 + per : n;
    for (uint32_t c = c0; c < c1; c += 64) {
        fill_ends(threadIdx.x < 64 && c + threadIdx.x < c1 ? ch.fills[c + threadIdx.x] : 0u, s_end);
        __syncthreads();
        const uint32_t total = s_end[63];
        for (uint32_t i = threadIdx.x; i < total; i += 256) {
            const uint32_t k = chunk_of(s_end, i), at = i - (k ? s_end[k - 1] : 0u);
            f(ch.hits + ((uint64_t)(c + k) * kHitChunk + at) * rw);
        }
        __syncthreads();
    }
}

// The word a record is of: the top 16 bits of its first word.
__device__ __forceinline__ uint32_t record_word(const uint64_t *r) {
    return (uint32_t)(r[0] >> 48) & (GSS_MAX_WORDS - 1);
}

// Records per word; counts[64] must start at zero.  The two grouping kernels
// run kGroupBlocks blocks, and a block adds to a word's counter once:
// device-scope atomics on one address take ~10 ns each.  With one per chunk and
// word, over the 1,024 blocks' chunks, the kernels took 12 and 14 us.
constexpr unsigned kGroupBlocks = 128;
__global__ __launch_bounds__(256) void k_word_count(ChunkArgs ch, uint32_t *counts) {
    __shared__ uint32_t h[GSS_MAX_WORDS];
    if (threadIdx.x < GSS_MAX_WORDS) h[threadIdx.x] = 0;
    __syncthreads();
    for_records(ch, [&](const uint64_t *r) { atomicAdd(&h[record_word(r)], 1u); });
    __syncthreads();
    if (threadIdx.x < GSS_MAX_WORDS && h[threadIdx.x]) atomicAdd(&counts[threadIdx.x], h[threadIdx.x]);
}

// Moves the records into `dense` grouped by word, ascending (within a word in
// no set order): a block counts its records per word in LDS, reserves each
// word's share with one atomic on that word's cursor, then places them.
// group[w] = first record of word w, group[64] = all records, group[65] = 1
// when they fitted in dense_cap (else nothing is moved and the host groups the
// records itself).  cursor[64] starts at zero.
__global__ __launch_bounds__(256) void k_word_scatter(ChunkArgs ch,
                                                      const uint32_t *__restrict__ counts,
                                                      uint32_t *cursor, uint64_t *__restrict__ dense,
                                                      uint64_t dense_cap, uint64_t *group,
                                                      uint32_t *out, uint32_t *halt) {
    __shared__ uint64_t base[GSS_MAX_WORDS + 1];
    __shared__ uint32_t lc[GSS_MAX_WORDS];
    const int tid = (int)threadIdx.x;
    if (tid < GSS_MAX_WORDS) {
        static_assert(GSS_MAX_WORDS == 64, "one wave");
        const uint64_t k = counts[tid], end = wave_incl_scan(k, tid);
        base[tid] = end - k;
        if (tid == GSS_MAX_WORDS - 1) base[GSS_MAX_WORDS] = end;
        lc[tid] = 0;
    }
    __syncthreads();
    const uint64_t total = base[GSS_MAX_WORDS];
    const bool fits = total <= dense_cap;
    if (blockIdx.x == 0 && tid == 0) {
        write_counts(ch, total, out);
        if (ch.alloc[1]) *halt = 1u;  // records were dropped: the step is re-run
    }
    if (blockIdx.x == 0 && tid <= GSS_MAX_WORDS + 1)
        group[tid] = tid <= GSS_MAX_WORDS ? base[tid] : (fits ? 1ull : 0ull);
    if (!fits) return;  // the same for every thread of every block
    for_records(ch, [&](const uint64_t *r) { atomicAdd(&lc[record_word(r)], 1u); });
    __syncthreads();
    if (tid < GSS_MAX_WORDS) {
        const uint32_t k = lc[tid];
        if (k) base[tid] += atomicAdd(&cursor[tid], k);
        lc[tid] = 0;
    }
    __syncthreads();
    const uint32_t rw = ch.rec_words;
    for_records(ch, [&](const uint64_t *r) {
        const uint32_t w = record_word(r);
        const uint64_t pos = base[w] + atomicAdd(&lc[w], 1u);
        for (uint32_t q = 0; q < rw; q++) dense[pos * rw + q] = r[q];
    });
}

// ---- serving: requests admitted on the device ---------------------------------

// The admitted request (index into r.adm) of the step's i-th patch.
__device__ __forceinline__ int admitted_of(const ServeRing &r, int cnt, int64_t i) {
    int lo = 0, hi = cnt;  // last admitted request whose patches start at or before i
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if ((int64_t)r.adm[mid].patch_pfx <= i) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Screening entries of a batched step (SweepArgs::agg), over every slot of a
// group's words, valid or not, so that they follow the table alone and a
// step's updates refresh them: all of them implies the valid ones.
template <int W>
struct TableGroups {
    static constexpr int NG = W < 8 ? W : 8;  // word groups
    static constexpr int GW = W / NG;         // words per group
};

// AND and OR of group b of a row.
template <int W>
__device__ __forceinline__ void group_fold(const uint64_t *__restrict__ row, int b, uint64_t &all,
                                           uint64_t &any) {
    constexpr int GW = TableGroups<W>::GW;
    all = ~0ull;
    any = 0;
#pragma unroll
    for (int w = 0; w < GW; w++) {
        const uint64_t x = row[b * GW + w];
        all &= x;
        any |= x;
    }
}

// One read of the table: from 16 words on a wave reads 64 words at a time, a
// word per lane, and votes.  A thread per variable, its two rows each (as still
// for the narrow tables, whose rows are neighbours), took 490 us for 1 GB; now
// 185, 5.5 TB/s.
template <int W>
struct TableEntries {
    static constexpr int VARS = W <= 8 ? 64 : W == 16 ? 8 : 4;  // per turn of a wave

    // Entry of variable v0 + lane, in the first VARS lanes.
    static __device__ __forceinline__ uint32_t turn(const uint64_t *__restrict__ table, int64_t v0,
                                                    int64_t vars, int lane) {
        if constexpr (W <= 8) {
            if (v0 + lane >= vars) return 0;
            const uint64_t *f = table + (size_t)(v0 + lane) * 2 * W, *t = f + W;
            uint32_t x = 0;
#pragma unroll
            for (int b = 0; b < W; b++)
                x |= ((f[b] == ~0ull ? 1u : 0u) | (t[b] == 0 ? 0x100u : 0u) |
                      (t[b] == ~0ull ? 0x10000u : 0u) | (f[b] == 0 ? 0x1000000u : 0u))
                     << b;
            return x;
        } else {
            constexpr int LINES = VARS * 2 * W / 64;  // of 64 words
            // lane 8 k + b: group b of the entry's field k (literal v non-false /
            // true, ~v non-false / true)
            const int k = (lane >> 3) & 3, first = (lane & 7) * (W / 8);
            const uint64_t words = ((1ull << (W / 8)) - 1ull) << first;
            uint64_t x[LINES];
            uint32_t out = 0;
#pragma unroll
            for (int l = 0; l < LINES; l++) {
                const int64_t at = v0 * 2 * W + l * 64 + lane;
                x[l] = at < vars * 2 * W ? table[at] : 0ull;
            }
#pragma unroll
            for (int j = 0; j < VARS; j++) {
                const int fl = j * 2 * W / 64, fs = j * 2 * W % 64;  // line and lane of row f
                const int tl = (j * 2 + 1) * W / 64, ts = (j * 2 + 1) * W % 64;
                const uint64_t f1 = __ballot(x[fl] == ~0ull) >> fs, f0 = __ballot(x[fl] == 0) >> fs;
                const uint64_t t1 = __ballot(x[tl] == ~0ull) >> ts, t0 = __ballot(x[tl] == 0) >> ts;
                const uint64_t m = k == 0 ? f1 : k == 1 ? t0 : k == 2 ? t1 : f0;
                const uint32_t e = (uint32_t)__ballot((~m & words) == 0);
                if (lane == j) out = e;
            }
            return out;
        }
    }
};

template <int W>
__global__ __launch_bounds__(256) void k_table_agg(const uint64_t *__restrict__ table,
                                                   const StepHeader *__restrict__ dh,
                                                   int64_t vars, uint32_t *__restrict__ agg) {
    if (dh->halted) return;  // the aggregate stays the halted step's
    constexpr int VARS = TableEntries<W>::VARS;
    const int lane = (int)__lane_id();
    for (int64_t v0 = (blockIdx.x * 4ll + (threadIdx.x >> 6)) * VARS; v0 < vars;
         v0 += gridDim.x * 4ll * VARS) {
        const uint32_t e = TableEntries<W>::turn(table, v0, vars, lane);
        if (lane < VARS && v0 + lane < vars) agg[v0 + lane] = e;
    }
}

// What the screened kernel would be left with: the wave's clause of the sample and
// the row after it, each looked at in one word group's valid slots, straight from the
// table (the entries are not there yet), a lane per word of a literal's two rows, its
// first 16 literals at once.  A clause that stays open costs the screened kernel its
// known literals (a third each) and its unknown ones (a row each), here per literal
// and in 48ths; kOpenCost in 100 is where it takes as long as the plain one.
// Plain and screened, 2M clauses, mean length 12, by the share of literals that are
// false and of groups that are known: half and 60 % x 8 words 260 and 183 us, three
// quarters and 60 % 390 and 373, nine in ten and 90 % 575 and 453, 80 % 606 and 661,
// 60 % 632 and 696; x 16 words, nine in ten and 96 % 582 and 412, 64 % 692 and 845.
//
// A clause per lane of one block, a literal after the other, took longer than the
// other blocks need for a table of 128 MB (29 us), so the clauses are spread over
// kOpenBlocks of them.
template <int W>
__device__ __forceinline__ uint32_t open_cost(const SweepArgs &a, const ClauseSample &sample,
                                              uint32_t groups, int gw, int lane) {
    constexpr int GW = W / 8, PER = 32 / GW, READS = PER < 16 ? 16 / PER : 1;  // literals a read
    constexpr uint64_t kOwn = ~0ull / ((1ull << (GW < 8 ? 2 * GW : 16)) - 1ull);
    const uint32_t len = sample.len[gw] & 0xFFFFFFu, rows = sample.len[gw] >> 24;
    const int n = len < 16u ? (int)len : 16;
    const int u = lane / (2 * GW);
    uint64_t x[2][READS], in[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const uint32_t *lits = sample.row[gw] + (c && rows > 1 ? len : 0u);
        const int w = nth_bit(groups, (2 * gw + c) % __popc(groups)) * GW + lane % GW;
        in[c] = a.valid[w];
#pragma unroll
        for (int r = 0; r < READS; r++) {
            const int j = r * PER + u;
            const uint32_t l = lits[j < n ? j : 0] ^ ((lane / GW) & 1 ? 128u : 0u);
            x[c][r] = load_word(a.table, scale_offset<W>(l) + (uint32_t)w * 8u);
        }
    }
    uint32_t cost = 0;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        int nonfalse = 0, unknown = n;
        bool tru = false;
#pragma unroll
        for (int r = 0; r < READS; r++) {
            uint64_t f = __ballot((x[c][r] | ~in[c]) == ~0ull), z = __ballot((x[c][r] & in[c]) == 0);
#pragma unroll
            for (int d = 1; d < GW; d <<= 1) {
                f &= f >> d;
                z &= z >> d;
            }
            const uint64_t own = kOwn & __ballot(r * PER + u < n);
            nonfalse += __popcll(f & own);
            unknown -= __popcll((f | z) & own);
            tru |= ((z >> GW) & own) != 0;
        }
        if (!tru && nonfalse < 2) cost += 16u + 48u * (uint32_t)unknown / (uint32_t)n;
    }
    return cost;
}

// Whether a plain sweep is screened, and the entries if it is.  The screened
// kernel pays where entries know what a variable is (true or false in all
// slots of a group) and the clauses are mostly closed by that.  Each block but the
// first kOpenBlocks looks at the same kSample variables spread over the table, each in one
// group; where kScreenKnown in 100 are known the entries are built, else nothing
// is.  Meanwhile the first blocks look at the clauses (open_cost), the next one writes
// what became of the variables: see screen_chosen.  A variable's groups mostly
// agree, so one group each of 128 variables tells more (the share to within 4
// points, one standard deviation) than all groups of 16 (12 points, 7 in 100 tables
// of 60 % known judged wrong) for as many bytes.
//
// Only groups with a valid slot count: words of no request hold one value (rolled
// forward) or none, whatever the others do.  Counted too, 14 such words beside 2
// mixed ones took 2M clauses to the screened kernel: 330 us, 213 plain.
//
// Plain against screened, entries included, by the share that is known, clauses
// mostly true: 400K clauses x 4096 slots 89 and 75 us at 58 %, 92 and 83 at 48, 95
// and 94 at 38; 1M x 333 slots 55 and 42 at 44 %; 2M x 1024 slots 149 and 94 at 55
// %, 119 and 73 at 88.
constexpr int kScreenKnown = 40, kScreenSure = 90, kSample = 128;
template <int W>
__global__ __launch_bounds__(256) void k_sweep_choose(SweepArgs a,
                                                      const uint64_t *__restrict__ table,
                                                      ClauseSample sample, uint64_t words,
                                                      int64_t vars,
                                                      uint32_t *__restrict__ agg,
                                                      uint64_t *__restrict__ agg_words,
                                                      uint32_t *choose) {
    static_assert(W >= 8, "eight groups");
    constexpr int VARS = TableEntries<W>::VARS, GW = W / 8;
    __shared__ int s_known[4];
    const int lane = (int)__lane_id(), wv = (int)(threadIdx.x >> 6);
    uint32_t groups = 0;  // with a valid slot
#pragma unroll
    for (int b = 0; b < 8; b++)
        if ((words >> (b * GW)) & ((1ull << GW) - 1ull)) groups |= 1u << b;
    if (blockIdx.x < kOpenBlocks) {
        __shared__ uint32_t s_cost[4];
        // (a halted step's clauses are not all there)
        const bool on = groups && (a.dyn ? a.dyn[2] : a.npasses) > 0;
        if (on) s_cost[wv] = open_cost<W>(a, sample, groups, (int)blockIdx.x * 4 + wv, lane);
        __syncthreads();
        if (threadIdx.x == 0)
            choose[1 + blockIdx.x] =
                on ? s_cost[0] + s_cost[1] + s_cost[2] + s_cost[3] : kOpenLimit + 1u;
        return;
    }
    const int ng = __popc(groups);
    if (ng) {
        // a lane per word: GW lanes of a variable's row f, then GW of its row t
        uint64_t x[GW];
#pragma unroll
        for (int l = 0; l < GW; l++) {
            const int i = wv * (kSample / 4) + l * (32 / GW) + lane / (2 * GW);
            const int64_t v = vars >= kSample ? vars * i / kSample : i % (int)vars;
            const int g = nth_bit(groups, (vars >= kSample ? i : i + i / (int)vars) % ng);
            x[l] = table[(size_t)(2 * v + ((lane / GW) & 1)) * W + g * GW + lane % GW];
        }
        int known = 0;
#pragma unroll
        for (int l = 0; l < GW; l++) {
            uint64_t z = __ballot(x[l] == 0);  // false, or true, in all slots: one of the rows
#pragma unroll
            for (int d = 1; d < GW; d <<= 1) z &= z >> d;
            known += __popcll(z & (~0ull / ((1ull << GW) - 1ull)));
        }
        if (lane == 0) s_known[wv] = known;
    }
    __syncthreads();
    const int in100 =
        ng ? (s_known[0] + s_known[1] + s_known[2] + s_known[3]) * 100 / kSample : 0;
    const bool screen = in100 >= kScreenKnown;
    if (blockIdx.x == kOpenBlocks) {
        if (threadIdx.x == 0) choose[0] = in100 >= kScreenSure ? 2u : screen ? 1u : 0u;
        if (threadIdx.x < 8)
            agg_words[threadIdx.x] = words & (((1ull << GW) - 1ull) << (threadIdx.x * GW));
    }
    if (!screen) return;
    for (int64_t v0 = ((blockIdx.x - kOpenBlocks) * 4ll + wv) * VARS; v0 < vars;
         v0 += (gridDim.x - kOpenBlocks) * 4ll * VARS) {
        const uint32_t e = TableEntries<W>::turn(table, v0, vars, lane);
        if (lane < VARS && v0 + lane < vars) agg[v0 + lane] = e;
    }
}

// Refreshes the entries that the step's updates (and patches) may have
// changed: for each (var, word), the bits of the word's group, from the table
// as it is now.  Two updates of one (var, group) write the same bits.
template <int W>
__global__ void k_table_agg_update(const uint64_t *__restrict__ table,
                                   const StepHeader *__restrict__ dh,
                                   const gss_var_update *__restrict__ ups,
                                   const gss_var_patch *__restrict__ patches, int with_patches,
                                   uint32_t *__restrict__ agg) {
    constexpr int GW = TableGroups<W>::GW;
    if (dh->halted) return;
    const int64_t nu = dh->nups, n = nu + (with_patches ? dh->npatches : 0);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t var, word;
        if (i < nu) {
            var = ups[i].var;
            word = ups[i].word;
        } else {
            var = patches[i - nu].var;
            word = patches[i - nu].word;
        }
        const int b = (int)(word / GW);
        const uint64_t *f = table + (size_t)var * 2 * W;
        uint64_t fa, fo, ta, to;
        group_fold<W>(f, b, fa, fo);
        group_fold<W>(f + W, b, ta, to);
        agg_set(agg + var, (uint32_t)b, fa == ~0ull, to == 0, ta == ~0ull, fo == 0);
    }
}

// A serving step's table words, screening entries and patches, in one launch.
//
// Load k (0 <= k < n) sets word k from loads[k].base (the admission hands out
// words 0..n-1 in order), and the words a serving step does not load are not
// valid in it.  So each row is written in whole 128-byte lines: words [0, L), L
// = n rounded up to 16 (at most `words`), words n..L-1 all ones.  Written word
// by word, 1 to 12 words of a 64-word table cost 0.19-0.29 ms at 2M variables:
// each row line was written in part.
//
// Screening entries (SweepArgs::agg): group b = the admitted requests r with
// r % 8 = b, from their solvers' bases (a request's words are loaded whole from
// its base, so until its patches the base value holds in all its slots;
// k_serve_patch clears what a patch undoes).  Bits of empty groups are not read.
//
// What bounds it: the row writes (256 MB at 1M variables and up to 16 words: 53
// us) or, over few variables, the patches.  Three kernels in a row took 60 us
// where it takes 45.
//
// The first kPatchBlocks blocks copy the admitted requests' patches from the
// pinned ring (consecutive lanes read consecutive 4-byte words: one pass over
// PCIe); each other block covers 64 variables: the bases' 64-variable words go
// through LDS, then each lane writes 16 bytes (2 words) of a variable's F row
// and of its T row, neighbouring lanes neighbouring words.
constexpr unsigned kPatchBlocks = 128;
__global__ __launch_bounds__(256) void k_serve_load(ServeRing r, const StepHeader *__restrict__ dh,
                                                    const gss_word_load *__restrict__ loads,
                                                    const uint64_t *__restrict__ bases,
                                                    int64_t vw, uint64_t *__restrict__ table,
                                                    int words, int64_t vars,
                                                    uint32_t *__restrict__ agg,
                                                    uint64_t *__restrict__ agg_words) {
    if (dh->halted) return;  // the words and the entries stay the halted step's
    const int nl = (int)dh->nloads, cnt = (int)*r.adm_count;
    const int tid = (int)threadIdx.x;
    if (blockIdx.x < kPatchBlocks) {
        if (agg && blockIdx.x == 0 && tid < 8) {
            uint64_t m = 0;
            for (int q = tid; q < cnt; q += 8) {
                const uint32_t w0 = r.adm[q].w0;
                const uint32_t w1 = q + 1 < cnt ? r.adm[q + 1].w0 : (uint32_t)nl;
                for (uint32_t w = w0; w < w1 && w < 64u; w++) m |= 1ull << w;
            }
            agg_words[tid] = m;
        }
        constexpr int kWords = (int)(sizeof(gss_var_patch) / 4);
        const int64_t n = dh->npatches * kWords;
        for (int64_t k = blockIdx.x * (int64_t)256 + tid; k < n; k += kPatchBlocks * 256) {
            const int64_t i = k / kWords;
            const int f = (int)(k - i * kWords);
            const ServeAdmitted a = r.adm[admitted_of(r, cnt, i)];
            const uint64_t j = (uint64_t)(i - (int64_t)a.patch_pfx);
            const uint32_t *src = (const uint32_t *)(r.patches + (a.patch_off + j) % r.patch_cap);
            ((uint32_t *)(r.dpatches + i))[f] = src[f];
        }
        return;
    }
    if (nl <= 0) return;
    __shared__ uint64_t s_bits[2 * GSS_MAX_WORDS];  // [2k] def, [2k + 1] true of load k
    __shared__ uint32_t s_w0[kServeMaxRequests];
    const int64_t blk = blockIdx.x - kPatchBlocks;  // variables [64 blk, 64 blk + 64)
    if (tid < 2 * nl) s_bits[tid] = bases[(size_t)(2 * loads[tid >> 1].base + (tid & 1)) * vw + blk];
    if (tid >= 192 && tid - 192 < cnt) s_w0[tid - 192] = r.adm[tid - 192].w0;
    __syncthreads();
    if (agg && tid < 64 && blk * 64 + tid < vars) {
        uint32_t x = ~0u;
        for (int q = 0; q < cnt; q++) {
            const bool d = (s_bits[2 * s_w0[q]] >> tid) & 1ull;
            const bool t = (s_bits[2 * s_w0[q] + 1] >> tid) & 1ull;
            // true: v non-false and true; false: ~v; undefined: both non-false
            const uint32_t keep = !d ? 0x00010001u : t ? 0x00000101u : 0x01010000u;
            x &= ~((0x01010101u & ~keep) << (q & 7));
        }
        agg[blk * 64 + tid] = x;
    }
    // literal v is false where v is false, ~v where v is true
    const auto word = [&](int w, int vi, uint64_t &f, uint64_t &t) {
        f = t = ~0ull;
        if (w < nl && ((s_bits[2 * w] >> vi) & 1ull))
            (((s_bits[2 * w + 1] >> vi) & 1ull) ? t : f) = 0ull;
    };
    if (words == 1) {
        const int64_t v = blk * 64 + tid;
        if (tid < 64 && v < vars) word(0, tid, table[2 * v], table[2 * v + 1]);
        return;
    }
    int L = (nl + 15) & ~15;
    if (L > words) L = words;
    const int pairs = L >> 1;  // 16-byte stores per row; words is a power of two
    for (int it = tid; it < 64 * pairs; it += 256) {
        const int vi = it / pairs, p = it - vi * pairs;
        const int64_t v = blk * 64 + vi;
        if (v >= vars) break;  // it grows with vi
        uint64_t f[2], t[2];
        word(2 * p, vi, f[0], t[0]);
        word(2 * p + 1, vi, f[1], t[1]);
        uint64_t *row = table + (size_t)v * 2 * words + 2 * p;
        *(ulonglong2 *)row = make_ulonglong2(f[0], f[1]);
        *(ulonglong2 *)(row + words) = make_ulonglong2(t[0], t[1]);
    }
}

__global__ void k_serve_patch(ServeRing r, const StepHeader *__restrict__ dh,
                              uint64_t *__restrict__ table, int words,
                              uint32_t *__restrict__ agg) {
    const int64_t n = dh->npatches;
    const int cnt = (int)*r.adm_count;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int q = admitted_of(r, cnt, i);
        const uint32_t w0 = r.adm[q].w0;
        const gss_var_patch pp = r.dpatches[i];
        const uint32_t var = pp.var;
        const uint32_t word = pp.word + w0;
        const uint64_t m = pp.mask, d = pp.is_def, t = pp.is_true;
        const size_t base = (size_t)var * 2 * words + word;
        table[base] = (table[base] & ~m) | (~(d & ~t) & m);
        table[base + words] = (table[base + words] & ~m) | (~(d & t) & m);
        if (agg && word < 64u) {
            // the request's group keeps what holds in the patched slots too
            const uint64_t vm = m & dh->valid[word];
            const uint64_t fal = d & ~t & vm, tru = d & t & vm;
            uint32_t clr = 0;
            if (fal) clr |= 0x1u;               // v non-false
            if (vm & ~tru) clr |= 0x100u;       // v true
            if (tru) clr |= 0x10000u;           // ~v non-false
            if (vm & ~fal) clr |= 0x1000000u;   // ~v true
            if (clr) atomicAnd(agg + var, ~(clr << (q & 7)));
        }
    }
}

// ---- tagged DB compaction --------------------------------------------------

__device__ __forceinline__ int find_ref(const CompactRef *__restrict__ r, int nb, int64_t g) {
    int lo = 0, hi = nb;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (r[mid].start <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

__global__ void k_compact_flags(const CompactRef *__restrict__ refs, int nb, int64_t n,
                                const uint8_t *__restrict__ keep, int64_t ntags,
                                uint32_t *__restrict__ flags) {
    for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n;
         g += (int64_t)gridDim.x * blockDim.x) {
        const int b = find_ref(refs, nb, g);
        const uint32_t tag = refs[b].tags[g - refs[b].start];
        flags[g] = tag < (uint64_t)ntags ? (keep[tag] ? 1u : 0u) : 1u;
    }
}

__global__ void k_compact_bounds(const CompactRef *__restrict__ refs, int nb, int64_t n,
                                 const uint32_t *__restrict__ flags,
                                 const uint32_t *__restrict__ pos, uint32_t *__restrict__ kept) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const int64_t st = refs[b].start;
    const int64_t en = b + 1 < nb ? refs[b + 1].start : n;
    const uint32_t pe = en < n ? pos[en] : pos[n - 1] + flags[n - 1];
    kept[b] = pe - pos[st];
}

// One thread per source row: kept rows move to their rank within the bucket.
__global__ void k_compact_move(const CompactRef *__restrict__ refs, int nb, int64_t n,
                               const uint32_t *__restrict__ flags,
                               const uint32_t *__restrict__ pos) {
    for (int64_t g = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; g < n;
         g += (int64_t)gridDim.x * blockDim.x) {
        if (!flags[g]) continue;
        const int b = find_ref(refs, nb, g);
        const CompactRef r = refs[b];
        const int64_t row = g - r.start;
        const int64_t dst = (int64_t)(pos[g] - pos[r.start]);
        const uint32_t *src = r.lits + row * r.len;
        uint32_t *d = r.dst_lits + dst * r.len;
        for (uint32_t i = 0; i < r.len; i++) d[i] = src[i];
        r.dst_tags[dst] = r.tags[row];
    }
}

template <int W>
hipError_t launch_sweep_w(const SweepArgs &a, int blocks, hipStream_t s) {
    const dim3 g(blocks), b(256);
    const bool clauses = a.rec_words == 2;
    if (a.agg) {
        if (clauses) hipLaunchKernelGGL((k_sweep_screened<W, true>), g, b, 0, s, a);
        else hipLaunchKernelGGL((k_sweep_screened<W, false>), g, b, 0, s, a);
    } else {
        if (clauses) hipLaunchKernelGGL((k_sweep<W, true>), g, b, 0, s, a);
        else hipLaunchKernelGGL((k_sweep<W, false>), g, b, 0, s, a);
    }
    return hipGetLastError();
}

// Resident blocks per CU: as the runtime counts them, which leaves the scalar
// registers out, at most kSweepBlocksPerCu.  A persistent grid of one block
// per CU more than is resident runs that block's share alone at the end
// (k_sweep at 16 words, 4M clauses: 640 -> 773 us).
template <int W>
int occupancy_w(int mode) {
    int nb = 0;
    hipError_t e = hipErrorInvalidValue;
    if (mode == 0)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sweep<W, false>, 256, 0);
    else if (mode == 1)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sweep_screened<W, false>, 256, 0);
    else if (mode == 2)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sweep<W, true>, 256, 0);
    else if (mode == 3)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_sweep_screened<W, true>, 256, 0);
    if (e != hipSuccess || nb < 1) return 1;
    return nb < kSweepBlocksPerCu ? nb : kSweepBlocksPerCu;
}

#define GSS_WORDS(X) X(1) X(2) X(4) X(8) X(16) X(32) X(64)

}  // namespace

int sweep_clauses_per_pass(int words, bool screened) { return screened ? 64 : 64 / words; }

hipError_t launch_sweep(const SweepArgs &a, int words, int blocks, hipStream_t s) {
#define X(W_) \
    if (words == W_) return launch_sweep_w<W_>(a, blocks, s);
    GSS_WORDS(X)
#undef X
    return hipErrorInvalidValue;
}

int sweep_occupancy(int words, int mode) {
#define X(W_) \
    if (words == W_) return occupancy_w<W_>(mode);
    GSS_WORDS(X)
#undef X
    return 1;
}

hipError_t launch_reset_u32(uint32_t *p, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reset_u32, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

hipError_t launch_fill_u64(uint64_t *p, int64_t n, uint64_t v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

hipError_t launch_scatter(const ScatterSeg *segs, int nseg, const uint32_t *src, int shift,
                          hipStream_t s) {
    if (nseg <= 0) return hipSuccess;
    const int blocks = nseg < 4096 ? nseg : 4096;
    hipLaunchKernelGGL(k_scatter, dim3(blocks), dim3(256), 0, s, segs, nseg, src, shift);
    return hipGetLastError();
}

hipError_t launch_assig_apply(const gss_var_update *ups, int64_t n, uint64_t *table, int words,
                              hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_assig_apply, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ups, n,
                       table, words);
    return hipGetLastError();
}

hipError_t launch_step_in(const StepInArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_step_in, dim3(512), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_step_end(const ChunkArgs &c, const StepEndArgs &a, hipStream_t s) {
    hipLaunchKernelGGL(k_step_end, dim3(kGatherBlocks + kRollBlocks), dim3(256), 0, s, c, a);
    return hipGetLastError();
}

hipError_t launch_words_load_dyn(const gss_word_load *loads, const int64_t *n,
                                 const uint64_t *bases, int64_t vw, uint64_t *table, int words,
                                 int64_t vars, hipStream_t s) {
    hipLaunchKernelGGL(k_words_load_dyn, dim3(4096), dim3(256), 0, s, loads, n, bases, vw, table,
                       words, vars);
    return hipGetLastError();
}

hipError_t launch_assig_patch_dyn(const gss_var_patch *p, const int64_t *n, uint64_t *table,
                                  int words, hipStream_t s) {
    hipLaunchKernelGGL(k_assig_patch_dyn, dim3(1024), dim3(256), 0, s, p, n, table, words);
    return hipGetLastError();
}

hipError_t launch_scatter_clauses(const ClauseSeg *cls, const int32_t *n, const uint32_t *src,
                                  int shift, hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_clauses, dim3(1024), dim3(256), 0, s, cls, n, src, shift);
    return hipGetLastError();
}

hipError_t launch_assig_apply_dyn(const gss_var_update *ups, const int64_t *n, uint64_t *table,
                                  int words, hipStream_t s) {
    hipLaunchKernelGGL(k_assig_apply_dyn, dim3(1024), dim3(256), 0, s, ups, n, table, words);
    return hipGetLastError();
}

hipError_t launch_assig_roll_dyn(const gss_var_update *ups, const int64_t *n, uint64_t *table,
                                 int words, const int8_t *last_pos, hipStream_t s) {
    hipLaunchKernelGGL(k_assig_roll_dyn, dim3(1024), dim3(256), 0, s, ups, n, table, words,
                       last_pos);
    return hipGetLastError();
}

hipError_t launch_count_records(const ChunkArgs &c, uint32_t *out, uint32_t *next, uint32_t seq,
                                hipStream_t s) {
    hipLaunchKernelGGL(k_count_records, dim3(1), dim3(1024), 0, s, c, out, next, seq);
    return hipGetLastError();
}

hipError_t launch_gather(const ChunkArgs &c, uint64_t records, void *dense, uint64_t dense_cap,
                         hipStream_t s) {
    if (c.rec_words < 1 || c.rec_words > 3) return hipErrorInvalidValue;
    // a block per 16 KB of records (each block sums the fills: 28 KB for 7,168
    // waves), at least one per CU and at most eight
    const uint64_t want = records * c.rec_words / 2048;
    const unsigned blocks = (unsigned)(want < 256 ? 256 : want < 2048 ? want : 2048);
    hipLaunchKernelGGL(k_gather, dim3(blocks), dim3(256), 0, s, c, (uint64_t *)dense, dense_cap);
    return hipGetLastError();
}

hipError_t launch_group_by_word(const ChunkArgs &c, uint32_t *counts, void *dense,
                                uint64_t dense_cap, uint64_t *group, uint32_t *out,
                                uint32_t *halt, hipStream_t s) {
    if (c.rec_words != 1 && c.rec_words != 3) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_word_count, dim3(kGroupBlocks), dim3(256), 0, s, c, counts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_word_scatter, dim3(kGroupBlocks), dim3(256), 0, s, c, counts,
                       counts + GSS_MAX_WORDS, (uint64_t *)dense, dense_cap, group, out, halt);
    return hipGetLastError();
}

hipError_t launch_table_agg(const uint64_t *table, const StepHeader *dh, int64_t vars, int words,
                            uint32_t *agg, hipStream_t s) {
    if (vars <= 0) return hipSuccess;
    const int64_t per = words <= 8 ? 256 : words == 16 ? 32 : 16;  // variables a block takes
    const unsigned blocks = (unsigned)std::min<int64_t>((vars + per - 1) / per, 4096);
#define X(W_)                                                                               \
    if (words == W_) {                                                                      \
        hipLaunchKernelGGL(k_table_agg<W_>, dim3(blocks), dim3(256), 0, s, table, dh, vars, \
                           agg);                                                            \
        return hipGetLastError();                                                           \
    }
    GSS_WORDS(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_sweep_choose(const SweepArgs &a, const ClauseSample &sample,
                               const uint64_t *valid, int64_t vars, int words, uint32_t *agg,
                               uint64_t *agg_words, uint32_t *choose, hipStream_t s) {
    uint64_t used = 0;
    for (int w = 0; w < words; w++)
        if (valid[w]) used |= 1ull << w;
    if (vars <= 0 || words < 8) return hipErrorInvalidValue;
    const int64_t per = words == 8 ? 256 : words == 16 ? 32 : 16;  // variables a block takes
    const unsigned blocks =
        kOpenBlocks + (unsigned)std::min<int64_t>((vars + per - 1) / per, 2048 - kOpenBlocks);
#define X(W_)                                                                                \
    if (words == W_) {                                                                       \
        hipLaunchKernelGGL(k_sweep_choose<W_>, dim3(blocks), dim3(256), 0, s, a, a.table, sample, \
                           used, vars, agg, agg_words, choose);                              \
        return hipGetLastError();                                                            \
    }
    X(8) X(16) X(32) X(64)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_table_agg_update(const uint64_t *table, const StepHeader *dh,
                                   const gss_var_update *ups, const gss_var_patch *patches,
                                   bool with_patches, int words, uint32_t *agg, hipStream_t s) {
    const int wp = with_patches ? 1 : 0;
#define X(W_)                                                                              \
    if (words == W_) {                                                                     \
        hipLaunchKernelGGL(k_table_agg_update<W_>, dim3(1024), dim3(256), 0, s, table, dh, \
                           ups, patches, wp, agg);                                         \
        return hipGetLastError();                                                          \
    }
    GSS_WORDS(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_serve_load(const ServeRing &r, const StepHeader *dh, const gss_word_load *loads,
                             const uint64_t *bases, int64_t vw, uint64_t *table, int words,
                             int64_t vars, uint32_t *agg, uint64_t *agg_words, hipStream_t s) {
    const unsigned blocks = kPatchBlocks + (unsigned)((vars + 63) / 64);
    hipLaunchKernelGGL(k_serve_load, dim3(blocks), dim3(256), 0, s, r, dh, loads, bases, vw, table,
                       words, vars, agg, agg_words);
    return hipGetLastError();
}

hipError_t launch_serve_patch(const ServeRing &r, const StepHeader *dh, uint64_t *table,
                              int words, uint32_t *agg, hipStream_t s) {
    hipLaunchKernelGGL(k_serve_patch, dim3(1024), dim3(256), 0, s, r, dh, table, words,
                       agg);
    return hipGetLastError();
}

static unsigned grid_for(int64_t n, unsigned cap = 65536) {
    const int64_t b = (n + 255) / 256;
    return (unsigned)(b < 1 ? 1 : b > cap ? cap : b);
}

hipError_t launch_compact_flags(const CompactRef *refs, int nb, int64_t n, const uint8_t *keep,
                                int64_t ntags, uint32_t *flags, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_compact_flags, dim3(grid_for(n)), dim3(256), 0, s, refs, nb, n, keep,
                       ntags, flags);
    return hipGetLastError();
}

hipError_t scan_exclusive_u32(const uint32_t *in, uint32_t *out, int64_t n, void *temp,
                              size_t &temp_bytes, hipStream_t s) {
    return hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, in, out, (int)n, s);
}

hipError_t launch_compact_bounds(const CompactRef *refs, int nb, int64_t n, const uint32_t *flags,
                                 const uint32_t *pos, uint32_t *kept, hipStream_t s) {
    if (nb <= 0 || n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_compact_bounds, dim3((nb + 255) / 256), dim3(256), 0, s, refs, nb, n,
                       flags, pos, kept);
    return hipGetLastError();
}

hipError_t launch_compact_move(const CompactRef *refs, int nb, int64_t n, const uint32_t *flags,
                               const uint32_t *pos, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_compact_move, dim3(grid_for(n)), dim3(256), 0, s, refs, nb, n, flags,
                       pos);
    return hipGetLastError();
}

hipError_t launch_assig_roll(const gss_var_update *ups, int64_t n, uint64_t *table, int words,
                             const int8_t *last_pos, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_assig_roll, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ups, n,
                       table, words, last_pos);
    return hipGetLastError();
}

}  // namespace gss
