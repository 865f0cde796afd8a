// plan_dev.h -- plain-old-data query plan read by the kernels.  Shared by the
// host planner and the HIP code; no host or device library types inside.
#pragma once

#include <stdint.h>

#define GFSM_MAXQ 32
#define GFSM_MAXCHK 31

// Work at depth d >= 1 (the query vertex placed d-th):
//   candidates = segment (f(anc at depth d - gen_dist), gen_rel);
//   a candidate w survives when it differs from every placed vertex and, for
//   each check j, w lies in segment (f(anc at depth d - chk_dist[j]), chk_rel[j])
//   (chk_dist 0 = w's own segment: a query self loop);
//   nxt_* is the generator of depth d+1 (its segment length is the number of
//   children a survivor will have; survivors with none are dropped).
struct DepthPlanDev {
    uint32_t gen_dist;
    uint32_t gen_rel;
    uint32_t nchk;
    uint32_t nxt_dist;
    uint32_t nxt_rel;
    // Placed columns a candidate of this depth has to be compared with for
    // injectivity (bit k: the vertex placed at depth k); the others differ from
    // every candidate by construction (see set_injectivity).
    uint32_t inj;
    uint32_t chk_dist[GFSM_MAXCHK];
    uint32_t chk_rel[GFSM_MAXCHK];
    // Dense segment tables ({begin, end} per data vertex, see DevGraph) of
    // nxt_rel and of the first four chk_rel, filled in per run where one
    // exists; null: the segment hash table.
    const void *nxt_seg;
    const void *chk_seg[4];
};

// The last depths of a query as leaves: each generated from, and checked
// against, vertices placed at depths <= d only, so that a node of depth d has a
// number of completions that is counted from the leaves' candidate sets (the
// entries of the generator's segment that pass the checks and are no placed
// vertex) without placing them.
#define GFSM_MAXTAIL 3
#define GFSM_TAILCHK 2
struct TailLeafDev {
    uint32_t col, rel;  // generator: depth of its ancestor (<= d), relation
    uint32_t inj;       // placed columns (bits 0..d) its candidates can equal
    uint32_t twins;     // earlier leaves of the tail with this very set
    uint32_t pair;      // 1: may also meet the leaf before it, whose set is another
    uint32_t nchk;
    uint32_t chk_col[GFSM_TAILCHK], chk_rel[GFSM_TAILCHK];
    const void *tab;    // dense segment tables, as in DepthPlanDev
    const void *chk_tab[GFSM_TAILCHK];
};
struct TailPlanDev {
    uint32_t m;         // leaves: depths d + 1 .. q - 1 (0: not countable this way)
    uint32_t wide;      // some leaf has checks or a pair
    TailLeafDev leaf[GFSM_MAXTAIL];
};

struct QueryPlanDev {
    uint32_t q;
    uint32_t root_rel;                   // generator relation of depth 1
    uint32_t nroot_chk;                  // self-loop relations of the root
    uint32_t root_chk_rel[GFSM_MAXCHK];
    uint32_t col[GFSM_MAXQ];             // original query id placed at depth d
    uint32_t dcol[GFSM_MAXQ];            // depth whose vertex is column c
    DepthPlanDev depth[GFSM_MAXQ];
    TailPlanDev tail[GFSM_MAXTAIL];      // tail[m - 1]: the last m depths as leaves of depth q - 1 - m
};
