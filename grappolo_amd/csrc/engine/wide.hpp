// wide.hpp -- whole-GPU persistent colored iteration for graphs above
// kDenseMaxNV vertices and smaller ones with large color classes.
//
// One launch per colored iteration (all color steps of the iteration, the
// per-color loop of Coloring/parallelLouvainWithColoring.cpp:169-218 with the
// community updates of :213-217) on a grid of 1024-thread workgroups, at most
// one per CU (wide_grid), with one grid barrier per color step.  The work of a
// color step is a list of items fixed when the phase starts:
//   workgroup items: a heavy vertex (kWMidMaxDeg + 1..kWHeavyMaxDeg entries, LDS
//     table of the whole workgroup), a chunk of kWChunk entries of a giant vertex
//     (summed per community in LDS, then written out as (community, weight)
//     pairs grouped by a hash partition of the community ids) and a
//     partition of a giant's communities (its pairs from every chunk summed in
//     LDS and scored; the last partition scored decides the move).  Once at
//     most kWMergeLive communities are left there are no partitions: the
//     workgroup of the last chunk sums and scores the giant's pairs;
//   wavefront items: one mid vertex (65..kWMidMaxDeg entries, a wavefront's
//     LDS table) or 64/G light vertices of degree bin b (G lanes each, the
//     in-order sums of buildLocalMapCounter,
//     Utility/utilityClusteringFunctions.cpp:172-194).
// What an item reads that its step does not change (its record, the vertex's
// own label and degree, a light vertex's weights) is loaded one item ahead,
// across the grid barrier too.
//
// Labels are held per adjacency entry: lab[j] is the label of entry j's
// neighbour, so a vertex reads its row in order instead of gathering one
// random line per entry, and a vertex that moves writes its new label into the
// entries that hold it (tpos, the entry positions grouped by neighbour, sorted
// out once per phase).  After the first iterations few vertices move, so the
// scattered writes are few: on the second phase of a 4.2-million-vertex RMAT
// graph (125 million entries, 285 classes, 138 iterations) an iteration takes
// 8.1 ms against 10.7 ms with the gathers, whose steps waited on a CU's misses.
// Entries of a class's rows hold labels of other classes, so a move may be
// written in its own step; with a coloring whose classes hold edges it is
// written after the step, behind a second barrier (WideArgs::defer).  Entry
// positions are 32-bit words, with a byte more each from 2^32 entries on: the
// sweep serves graphs below 2^40 entries and 2^31 vertices.
//
// Workgroup items are dealt out when the phase starts (longest first, each to
// the least loaded workgroup), wavefront items in turn to the wavefronts of
// the least loaded workgroups, so a run is reproducible.  Community degrees and
// sizes are double-buffered as in the small-graph persistent sweep: step k
// reads the state after step k-1 and writes into the other buffer the moves of
// steps k-1 and k.
#pragma once

#include <vector>

#include "kernels.hpp"

namespace glv {

constexpr int kWBlock = 1024;            // threads per workgroup
constexpr i64 kWideMaxEntries = i64(1) << (kTposBits + 8);  // entry positions of a word and a byte
constexpr int kWHeavySlots = 12288;      // LDS table of a workgroup: u32 keys + f64 values
constexpr i64 kWHeavyMaxDeg = 8192;      // larger vertices are giants (several workgroups)
constexpr i64 kWChunk = 4096;            // entries of a giant per accumulation item
constexpr i64 kWPartKeys = 4096;         // communities per partition of a giant (expected)
constexpr int kWMaxParts = 1024;         // partitions of a giant at most
constexpr int kWMaxChunks = 1024;        // chunks of a giant at most (4,194,304 entries; a phase
                                         // with a larger vertex takes the per-color launches)
constexpr int kWMergeLive = 8192;        // communities up to which a giant is decided by the workgroup
                                         // that finishes its last chunk (they fit its table)
constexpr int kWMoves = 128;             // moves of a step that a workgroup lists in LDS
constexpr int kWWavesPerGroup = kWBlock / kWave;
constexpr int kWMidSlots = kWHeavySlots / kWWavesPerGroup;  // LDS table of a wavefront
constexpr i64 kWMidMaxDeg = 512;         // largest vertex of a wavefront (load <= 2/3 of kWMidSlots)
// Phases whose color classes hold more vertices than this on average take the
// per-color launches instead (a class that large fills the GPU by itself).
constexpr i64 kWideMaxPerColor = 100000;
// Phases of at most kDenseMaxNV vertices take the sweep from this many
// vertices per color class on (the mean).
constexpr i64 kWideDensePerColor = 64;

// Phases without a vertex above 256 entries keep the per-color launches up to
// kWideLightNV vertices (64-bit labels within an XCD's 4 MB L2) when a class
// holds more than `vertices` on average and takes at most `launches` of them or
// holds `entries` entries (measured where the choice is made,
// Engine::colored_phase).
struct WideLight {
    double launches;
    i64 entries, vertices;
};
constexpr WideLight kWideLight{2.2, 250000, kPersistMaxPerColor};  // a caller's colors, classes that hold edges
constexpr WideLight kWideLightRun{1.5, 400000, 1024};              // a coloring known to be proper
constexpr i64 kWideLightNV = 524288;

// Relative costs of workgroup items (about microseconds): a heavy vertex
// kWCostHeavy plus three per 1024 entries.  Runs hardly depend on them (RMAT of
// 4.2M vertices, RMAT of 250,007, LFR of 1M, ms: 1420, 110.4, 48.8; workgroup
// items at half 1441, 110.5, 48.9; one per 1024 entries 1420, 110.7, 48.9;
// wavefront items at half 1428, 110.8, 48.9, at 1.7 times 1425, 110.3, 48.7).
constexpr double kWCostHeavy = 10.0, kWCostChunk = 10.0, kWCostPart = 10.0;
// wavefront items: a mid vertex, a batch of light vertices (a workgroup runs
// kWWavesPerGroup of them at a time)
constexpr double kWCostMid = 8.0, kWCostLight = 6.0;

// A workgroup item: the entries [beg, beg + len) of vertex v, whole (heavy, g
// < 0) or chunk j of giant g.  Each workgroup has one stream of them over the
// phase's classes, so the entries of its next item are read ahead whatever
// class it belongs to.
struct WideItem {
    i64 beg;
    int32_t v;
    int32_t len;
    int32_t g;
    int32_t j;
};
// A vertex in the order of PhaseSetup::perm: what its sweep needs that the
// phase does not change, in one record.
struct WideRow {
    i64 beg;
    double k;
    double sl;  // self-loop weight
    int32_t v;
    int32_t deg;
};
// The entries of a row as a WideRow holds them: a row of a multigraph can have
// 2^31 and more, which is more than the chunks of a giant hold either way.
constexpr int32_t wide_row_deg(i64 d) { return d < INT32_MAX ? (int32_t)d : INT32_MAX; }
static_assert(wide_row_deg(i64(1) << 31) > kWMaxChunks * kWChunk && wide_row_deg((i64(1) << 32) - 1) > kWMaxChunks * kWChunk,
              "a row that no item serves must look like one");
// A color class: its vertices cperm[lo, hi) and its wavefront items in order
// -- the vertices of bin 7 with at most kWMidMaxDeg entries (`nextra` rows from
// `extra0` on, behind the others), the vertices of bins 6, 5, .. 1 (rows
// bin_lo[b] .. + bin_n[b], b = 0 for bin 6) -- dealt to the `groups` workgroups
// with the least other work.
struct WideClass {
    int32_t lo, hi;
    int32_t nextra, extra0;
    int32_t bin_lo[6], bin_n[6];
    int32_t groups;
};
constexpr int kWClassWords = sizeof(WideClass) / 4;  // read as 32-bit words, one per lane
static_assert(kWClassWords <= 64, "a wavefront reads a WideClass at once");
// A giant vertex of the phase: chunk j writes its pairs at pairs + j *
// kWChunk (partition p's from cnt[j * (nparts + 1) + p] on, relative) and the
// partition bounds at cnt + j * (nparts + 1) (offsets into the pair arrays and
// the count array of its color class).
struct WideGiant {
    i64 v;
    i64 pairs;
    i64 cnt;
    int32_t nchunks;
    int32_t nparts;
};

// Degree and size of a community side by side (one 16-byte load serves both,
// as the reference's Comm record, DefineStructure/defs.h:66-70, holds them).
struct CommInfo {
    double a;
    i64 n;
};

struct WideArgs {
    const double *w;             // the adjacency's weights
    const double *k;             // vertex degrees
    double constant;             // 1 / (2m)
    i64 nv;
    int32_t *C;                  // labels, 32-bit
    int32_t *tgt;                // moves beyond a workgroup's list (kWMoves): the new label, else -1
    int32_t *over;               // per class: such a move was made
    int32_t *lab;                // per adjacency entry, the label of its neighbour
    const uint32_t *tpos;        // the entries whose neighbour is v: tpos[toff[v]] .. tpos[toff[v + 1]]
    const uint8_t *tpos_hi;      // their bits from kTposBits on; null when there are none
    const i64 *toff;
    const double *selfw;         // self-loop weight of every vertex
    bool defer;                  // a class may hold an edge: labels enter `lab` after the step
    double *a;                   // community degrees and sizes of the phase, read at the
    i64 *n;                      //   start of the iteration and written at its end
    CommInfo *m0, *m1;           // community degrees and sizes, two buffers
    const WideRow *rows;         // vertices grouped by (degree bin, color), the classes' extra rows
    const i64 *cperm;            // vertices grouped by color
    const WideClass *classes;    // the non-empty classes
    int ncls;
    const int32_t *rank;         // class k, workgroup w: its turn among the class's wavefront workgroups at
                                 //   k * nb + w, -1 for a workgroup that takes no wavefront items
    const WideItem *witems;      // workgroup w's stream; class k ends at wend[w * ncls + k], starts where k - 1 ended
    const i64 *wbeg, *wend;      // wbeg[w]: start of the stream
    const int2 *pitems;          // (giant, partition), streams as above
    const i64 *pbeg, *pend;
    int live;                    // communities with vertices at most (none appears during a phase); up
                                 //   to kWMergeLive the giants are decided with their last chunk
    const WideGiant *giants;
    i64 ngiants;
    uint32_t *gpk;               // giant pairs: community ids (one class at a time)
    double *gpv;                 //   and summed weights
    int32_t *gcnt;               // partition bounds of every chunk
    int32_t *gstate;             // per giant: chunks written, pairs ready, partitions scored
    double *gsc;                 // per giant: weight to its own community
    double *gcand;               // per giant and partition: gain, weight to the candidate, its size
    i64 *gcid;                   // per giant and partition: candidate (-1: none)
    i64 gparts;                  // partitions per giant in gcand/gcid (the largest nparts)
    double *gout;                // per giant: 2(e_t - e_s) of its move this iteration, 0 if none
    unsigned *bar;               // 16 + 16 * grid words, zero at launch; word 0: abort, word 1 receives
                                 //   the communities with vertices at the end
    double *part;                // per workgroup: [0, nb) movers' 2 (e_t - e_s), [nb, 2nb) sum of a^2
    i64 *moves;                  // vertices moved (added once per workgroup)
};

struct PhaseSetup;

// The items and giant tables of one phase.
struct WidePlan {
    DBuf<WideItem> witems;
    DBuf<int2> pitems;
    DBuf<i64> wbeg, wend, pbeg, pend;
    DBuf<WideClass> classes;
    DBuf<WideRow> rows;
    DBuf<int32_t> rank, over;
    DBuf<WideGiant> giants;
    DBuf<uint32_t> gpk;
    DBuf<double> gpv, gsc, gcand, gout;
    DBuf<int32_t> gcnt, gstate;
    DBuf<i64> gcid;
    int ncls = 0;
    i64 ngiants = 0, gparts = 1, gpairs = 0, gcounts = 0;
    i64 nwitems = 0, nvitems = 0;
};
// Builds the items of every color class of P (vertices of g grouped by
// degree bin and color) for a grid of nb workgroups; false (nothing built)
// when a vertex has more entries than kWMaxChunks chunks hold.
bool build_wide_plan(const DevGraph &g, const PhaseSetup &P, const double *selfw, int nb, WidePlan &L,
                     hipStream_t s);

// false when the environment sets GLV_WIDE=0 (large graphs then take the
// per-color launches; for comparisons)
bool wide_enabled();
// Resident workgroups of the wide sweep on the current device (0: unavailable).
int wide_blocks();
// The grid for color classes of `entries` adjacency entries on average: the
// smallest power of two with a thread per entry, from kWMinGrid up to every
// CU.  A larger grid lengthens each step's barrier, a smaller one its work;
// measured (RMAT 100,001 vertices, 34k entries per class: first phase 25.9 ms
// at 64 workgroups, 27.1 at 128, 28.5 at 32; RMAT 500,001, 103k: 112.6 ms at
// 128, 118.8 at 256, 123.7 at 64; LFR 200,001, 290k: 6.5 ms at 256, 7.3 at 128).
constexpr int kWMinGrid = 32;
int wide_grid(i64 entries);
// One colored iteration; false when the launch is not possible.
bool launch_wide_iteration(const WideArgs &W, int nblocks, hipStream_t s);
// the rows of perm[lo .. hi)
void launch_wide_rows(const i64 *perm, const i64 *off, const double *k, const double *selfw, i64 lo, i64 hi,
                      WideRow *rows, hipStream_t s);
// 64-bit ids to 32-bit (all below 2^31) and back
void launch_narrow_ids(const i64 *src, i64 n, int32_t *dst, hipStream_t s);
void launch_widen_ids(const int32_t *src, i64 n, i64 *dst, hipStream_t s);

}  // namespace glv
