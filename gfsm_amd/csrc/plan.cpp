// plan.cpp -- query compilation: matching order and per-depth requirements.
//
// Keeps the reference's order (HnGPU.cu:749-773 preProcessQuery,
// ccsr.cpp:98-204 genereateCCSRRequirements) so per-depth work is comparable:
//   * query vertices ranked by out-degree descending, then id ascending
//     (the CCSR row order, HnHelper.cuh:21-31, 413);
//   * depth 0 places rank 0; each later depth places the lowest-ranked vertex
//     that is an out-neighbour of a placed vertex and is not yet placed;
//   * when n is placed at depth d, each entry n->u to a placed u (u == n for a
//     self loop) becomes a requirement (distance d - depth(u), relation of
//     u->n when the query has it, else of n->u), sorted by distance;
//   * firstQ = smallest non-zero distance; its ancestor generates candidates.
// The reference generates from every entry of that ancestor's row and then
// checks all requirements; here the generator's requirement selects the
// segment that is streamed, and the remaining requirements become checks.
//
// With a data graph given (GFSM_ORDER_COST, no reference counterpart) the
// order is chosen from the data graph's relation statistics instead: the
// root is the vertex whose cheapest out-relation has the fewest source
// vertices, and each later depth places the reachable vertex with the
// smallest expected number of children per node (mean generator segment
// length times the pass rate of its checks).  Requirements are derived the
// same way for either order; the set of embeddings does not depend on it.
#include "host.h"

#include <algorithm>
#include <cstring>
#include <numeric>

namespace gfsm {

// Mean segment length of `rel` over every vertex that could own one (those
// without a segment count as length 0) and the number of vertices its
// segments can reach (the reverse relation's sources in labelled mode).
void rel_model(const HostGraph &data, uint32_t rel, double &mean, double &reach)
{
    mean = 0;
    reach = 1;
    uint64_t src, ent;
    if (!relation_sources(data, rel, src, ent) || src == 0) return;
    mean = (double)ent / (double)std::max<uint64_t>(src, relation_pool(data, rel));
    uint32_t rev = rel;
    if (data.mode == GFSM_MODE_VLABEL) rev = ((rel >> 10) & 0x7FF) << 21 | (rel >> 21) << 10 | (rel & 0x3FF);
    uint64_t rsrc = src, rent;
    if (!relation_sources(data, rev, rsrc, rent)) rsrc = src;
    reach = std::max<double>(1.0, (double)rsrc);
}

// Expected level sizes: a candidate from a segment of relation r passes a
// check of relation c with probability min(1, mean length of c / vertices c
// reaches); each survivor has (mean length of the next generator) children.
void project_levels(const HostGraph &data, const Plan &plan, uint64_t nroots, uint64_t g1, double *nodes,
                    double *cand)
{
    const uint32_t q = plan.q;
    double S = (double)nroots, G = (double)g1;
    for (uint32_t k = 0; k < q; k++) nodes[k] = cand[k] = 0;
    if (!q) return;
    nodes[0] = S;
    cand[0] = S;
    for (uint32_t d = 1; d < q; d++) {
        const DepthPlanDev &dp = plan.dev.depth[d];
        cand[d] = G;
        double p = 1;
        for (uint32_t r = 0; r < dp.nchk; r++) {
            double m, reach;
            rel_model(data, dp.chk_rel[r], m, reach);
            p *= std::min(1.0, m / reach);
        }
        S = std::min(G * p, 1e30);
        nodes[d] = S;
        double m, reach;
        rel_model(data, dp.nxt_rel, m, reach);
        G = std::min(S * m, 1e30);
    }
}

// Which placed vertices a candidate can coincide with:
//   * labelled mode: a vertex placed at depth k >= 1 came from a segment of
//     that depth's generator relation, whose target label it carries (the
//     root: the source label of the depth-1 generator relation), so a
//     candidate with another label differs from it;
//   * a data graph without self loops: a candidate is an entry of the segment
//     of its generator's ancestor and of every checked ancestor, so equal to
//     none of them (a candidate that is, fails that check anyway).
// The candidate test reads one LDS word per candidate and compared column, and
// at 4 to 16 labels most columns drop out (measured, start against now: labelled
// random graph of 200,000 vertices, 7-vertex count, 7.93 -> 7.55 ms; nine capped
// 8-vertex queries on a power-law graph, 5.69 -> 5.37 ms; unlabelled grids, where
// only the loop rule helps, -0.3% to -2.5%).
void set_injectivity(const HostGraph &data, Plan &plan)
{
    const bool by_label = data.mode == GFSM_MODE_VLABEL;
    uint32_t label[GFSM_MAXQ] = {};
    for (uint32_t k = 0; by_label && k < plan.q; k++)
        label[k] = k ? (plan.dev.depth[k].gen_rel >> 10) & 0x7FFu : plan.dev.root_rel >> 21;
    for (uint32_t d = 1; d < plan.q; d++) {
        DepthPlanDev &dp = plan.dev.depth[d];
        uint32_t m = 0;
        for (uint32_t k = 0; k < d; k++)
            if (!by_label || label[k] == label[d]) m |= 1u << k;
        if (!data.has_loops) {
            m &= ~(1u << (d - dp.gen_dist));
            for (uint32_t r = 0; r < dp.nchk; r++)
                if (dp.chk_dist[r]) m &= ~(1u << (d - dp.chk_dist[r]));
        }
        dp.inj = m;
    }
}

// Graphs whose largest degree is at most this have no hubs: a candidate's sets
// are compared entry by entry on one thread (checks, pairs), 64 x 64 at worst.
// Past it such a leaf is placed, its candidates spread over the threads.
static constexpr uint32_t kWideDegree = 64;
// The relations compared have segments of at most this mean length (over entries),
// and the step itself checks nothing: behind a check few lanes of a wave hold a
// survivor, and one's comparing holds up all.  Measured, all depths expanded /
// compared: checked step: 3 x 3 patch of the 1400 x 1400 grid 10.0 / 11.9 ms, cliques
// of four at mean degree 30 1.34 / 2.46 ms.  Unchecked, 4-cycles / triangles with a
// tail-free step: degree 12, 20,000 vertices 0.36 / 0.24 and 0.088 / 0.089 ms; degree 20
// 1.20 / 0.86 and 0.117 / 0.198 ms; degree 36 6.98 / 5.34 and 0.24 / 0.38 ms.
static constexpr double kWideMean = 16;

void set_tails(const HostGraph &data, Plan &plan, bool wide)
{
    const uint32_t q = plan.q;
    const bool by_label = data.mode == GFSM_MODE_VLABEL;
    wide = wide && data.max_degree <= kWideDegree && data.V < 0xFFFFFFFEu;
    auto label = [&](uint32_t k) { return by_label ? (plan.dev.depth[k].gen_rel >> 10) & 0x7FFu : 0u; };
    auto brief = [&](uint32_t rel) { return relation_biased_mean(data, rel) <= kWideMean; };
    uint32_t bits = 1;  // of a segment's length
    while (bits < 32 && (data.max_degree >> bits)) bits++;
    for (uint32_t m = 1; m <= GFSM_MAXTAIL; m++) {
        TailPlanDev &tp = plan.dev.tail[m - 1];
        tp = TailPlanDev{};
        // A tile keeps at most 2^11 nodes; its number of completions fits 62 bits.
        if (q < m + 2 || m * bits + 11 > 62) continue;
        const uint32_t d = q - 1 - m;
        bool ok = true, any_wide = false;
        const bool compare = wide && plan.dev.depth[d].nchk == 0;
        for (uint32_t i = 0; i < m && ok; i++) {
            const uint32_t k = d + 1 + i;
            const DepthPlanDev &dp = plan.dev.depth[k];
            TailLeafDev &l = tp.leaf[i];
            l.col = k - dp.gen_dist;
            l.rel = dp.gen_rel;
            l.inj = dp.inj & (uint32_t)((1ull << (d + 1)) - 1);
            l.nchk = dp.nchk;
            ok = l.col <= d && (dp.nchk == 0 || (compare && dp.nchk <= GFSM_TAILCHK && brief(dp.gen_rel)));
            for (uint32_t r = 0; r < dp.nchk && ok; r++) {
                ok = dp.chk_dist[r] && k - dp.chk_dist[r] <= d && brief(dp.chk_rel[r]);
                l.chk_col[r] = k - dp.chk_dist[r];
                l.chk_rel[r] = dp.chk_rel[r];
            }
            // Earlier leaves with the same label: all this very set, or one
            // other set, the leaf before it, that meets nothing else.
            uint32_t same = 0, twin = 0;
            for (uint32_t j = 0; j < i && ok; j++) {
                if (label(d + 1 + j) != label(k)) continue;
                same++;
                const TailLeafDev &o = tp.leaf[j];
                if (o.col == l.col && o.rel == l.rel && !o.nchk && !l.nchk && !o.pair && !data.has_dups) twin++;
            }
            if (same == twin)
                l.twins = twin;
            else if (compare && same == 1 && label(k - 1) == label(k) && !tp.leaf[i - 1].pair && brief(l.rel) &&
                     brief(tp.leaf[i - 1].rel))
                l.pair = 1;
            else
                ok = false;
            any_wide = any_wide || l.nchk || l.pair;
        }
        if (!ok) continue;
        tp.m = m;
        tp.wide = any_wide ? 1u : 0u;
    }
}

// A cap that ends inside a tile has that tile expanded after all: where a tile's
// leaf candidates pass the cap by themselves the counting step is wasted.  Measured
// on 20 queries of an R-MAT 18 graph, without the rule / 1 / 4 / 16 tiles: 64 hub roots
// under a cap of 2^25 7.3 / 7.2 / 6.5 / 6.8 ms (every depth expanded: 8.8), under 2^22
// 8.6 / 6.9 / 6.5 / 6.4 ms (6.4); 64 middle roots under 2^25 8.9 / 8.8 / 8.3 / 9.5 ms
// (12.2), under 2^22 8.8 / 6.4 / 6.0 / 5.8 ms (8.0).
static constexpr double kCapTiles = 4;

uint32_t usable_leaves(const HostGraph &data, const Plan &plan, uint64_t max_depth_cand, uint64_t tc)
{
    uint32_t best = 0;
    for (uint32_t m = 1; m <= GFSM_MAXTAIL; m++) {
        if (!plan.dev.tail[m - 1].m) continue;
        if (max_depth_cand) {
            double per = kCapTiles * (double)tc;
            for (uint32_t i = 0; i < m; i++) per *= std::max(1.0, relation_biased_mean(data, plan.dev.tail[m - 1].leaf[i].rel));
            if (per > (double)max_depth_cand) break;
        }
        best = m;
    }
    return best;
}

Status plan_query(const HostGraph &qg, Plan &out, const HostGraph *by_cost)
{
    out = Plan{};
    uint32_t q = qg.V;
    if (q == 0) return Status::err(GFSM_ERR_QUERY, "empty query");
    if (q > GFSM_MAXQ) return Status::err(GFSM_ERR_QUERY, "query larger than 32 vertices");
    std::vector<uint32_t> deg(q);
    uint32_t maxval = 0;
    for (uint32_t v = 0; v < q; v++) {
        deg[v] = qg.degree(v);
        maxval = std::max(maxval, deg[v]);
    }
    // Every query vertex needs a CCSR row in the reference (its offset walk,
    // ccsr.cpp:103-108, assumes one); a lone vertex has none.
    if (q >= 2)
        for (uint32_t v = 0; v < q; v++)
            if (!deg[v]) return Status::err(GFSM_ERR_QUERY, "query vertex " + std::to_string(v) + " has no out-entries");
    std::vector<uint32_t> rank(q);
    std::iota(rank.begin(), rank.end(), 0u);
    std::sort(rank.begin(), rank.end(), [&](uint32_t a, uint32_t b) {
        if (deg[a] != deg[b]) return deg[a] > deg[b];
        return a < b;
    });

    out.q = q;
    out.maxval = maxval;
    out.col.assign(q, 0);
    out.header.assign(3 * q, 0);
    out.requirements.assign((size_t)2 * std::max(maxval, 1u) * q, 0);
    std::memset(&out.dev, 0, sizeof(out.dev));
    out.dev.q = q;

    std::vector<int32_t> placed(q, -1);
    std::vector<char> seen(q, 0);
    struct Req { uint32_t dist, rel; };
    // Requirements of vertex n if it is placed at depth d: each entry n->u to
    // a placed u (the relation of u->n when the query has it, else of n->u),
    // by distance.  Placing n itself makes its self loops distance 0.
    auto reqs_of = [&](uint32_t n, uint32_t d) {
        std::vector<Req> reqs;
        for (uint32_t j = qg.dir_ptr[n]; j < qg.dir_ptr[n + 1]; j++) {
            uint32_t r = qg.dir[j].rel;
            for (uint32_t p = qg.dir[j].beg; p < qg.dir[j + 1].beg; p++) {
                uint32_t u = qg.nbr[p];
                if (placed[u] < 0 && u != n) continue;
                const uint32_t du = (u == n) ? d : (uint32_t)placed[u];
                uint32_t rel = r;
                for (uint32_t k = qg.dir_ptr[u]; k < qg.dir_ptr[u + 1]; k++) {
                    const uint32_t *b = qg.nbr.data() + qg.dir[k].beg, *e = qg.nbr.data() + qg.dir[k + 1].beg;
                    if (std::binary_search(b, e, (uint32_t)n)) { rel = qg.dir[k].rel; break; }
                }
                reqs.push_back({d - du, rel});
            }
        }
        std::sort(reqs.begin(), reqs.end(), [](const Req &a, const Req &b) {
            return a.dist != b.dist ? a.dist < b.dist : a.rel < b.rel;
        });
        return reqs;
    };
    // Next vertex in the reference order: the lowest-ranked reachable one.
    auto next_reference = [&](uint32_t d) -> int64_t {
        if (d == 0) return rank[0];
        for (uint32_t i = 0; i < q; i++)
            if (seen[rank[i]] && placed[rank[i]] < 0) return rank[i];
        return -1;
    };
    // Next vertex by expected cost on the data graph (ties: rank order).
    auto next_by_cost = [&](uint32_t d) -> int64_t {
        int64_t best = -1;
        double best_cost = 0;
        size_t best_reqs = 0;
        for (uint32_t i = 0; i < q; i++) {
            const uint32_t n = rank[i];
            if (placed[n] >= 0 || (d && !seen[n])) continue;
            double cost;
            size_t nreq = 0;
            if (d == 0) {
                cost = 1e300;  // fewest roots: the cheapest out-relation's sources
                for (uint32_t j = qg.dir_ptr[n]; j < qg.dir_ptr[n + 1]; j++) {
                    uint64_t src = 0, ent;
                    if (!relation_sources(*by_cost, qg.dir[j].rel, src, ent)) src = 0;
                    cost = std::min(cost, (double)src);
                }
            } else {
                const std::vector<Req> reqs = reqs_of(n, d);
                bool gen = false;
                cost = 1;
                for (auto &r : reqs) {
                    double mean, reach;
                    rel_model(*by_cost, r.rel, mean, reach);
                    if (!gen && r.dist) {
                        cost *= mean;  // children per node: the generator segment
                        gen = true;
                    } else {
                        cost *= std::min(1.0, mean / reach);  // pass rate of a check
                    }
                }
                if (!gen) continue;  // no placed out-neighbour to generate from
                nreq = reqs.size();
            }
            if (best < 0 || cost < best_cost || (cost == best_cost && nreq > best_reqs)) {
                best = n;
                best_cost = cost;
                best_reqs = nreq;
            }
        }
        return best;
    };
    for (uint32_t d = 0; d < q; d++) {
        const int64_t n = by_cost ? next_by_cost(d) : next_reference(d);
        if (n < 0) return Status::err(GFSM_ERR_QUERY, "query is not connected through out-entries");
        const std::vector<Req> reqs = reqs_of((uint32_t)n, d);
        placed[n] = (int32_t)d;
        out.col[d] = (uint32_t)n;
        for (uint32_t p = qg.dir[qg.dir_ptr[n]].beg; p < qg.dir[qg.dir_ptr[n + 1]].beg; p++) seen[qg.nbr[p]] = 1;
        uint32_t firstQ = 0;
        for (auto &r : reqs)
            if (r.dist) { firstQ = r.dist; break; }
        if (d && (!firstQ || firstQ > d))
            return Status::err(GFSM_ERR_QUERY, "query compile failure at depth " + std::to_string(d));
        uint32_t off = d * std::max(maxval, 1u) * 2;
        out.header[3 * d + 0] = (uint32_t)reqs.size();
        out.header[3 * d + 1] = off;
        out.header[3 * d + 2] = firstQ;
        for (size_t i = 0; i < reqs.size(); i++) {
            out.requirements[off + 2 * i] = i ? reqs[i].dist - reqs[i - 1].dist : reqs[i].dist;
            out.requirements[off + 2 * i + 1] = reqs[i].rel;
        }
        // Device plan.
        if (d == 0) {
            for (auto &r : reqs) {
                if (out.dev.nroot_chk >= GFSM_MAXCHK) return Status::err(GFSM_ERR_QUERY, "too many requirements");
                out.dev.root_chk_rel[out.dev.nroot_chk++] = r.rel;
            }
        } else {
            DepthPlanDev &dp = out.dev.depth[d];
            bool gen_taken = false;
            for (auto &r : reqs) {
                if (!gen_taken && r.dist == firstQ) {
                    dp.gen_dist = r.dist;
                    dp.gen_rel = r.rel;
                    gen_taken = true;
                    continue;
                }
                if (dp.nchk >= GFSM_MAXCHK) return Status::err(GFSM_ERR_QUERY, "too many requirements");
                dp.chk_dist[dp.nchk] = r.dist;
                dp.chk_rel[dp.nchk] = r.rel;
                dp.nchk++;
            }
        }
    }
    for (uint32_t d = 0; d < q; d++) {
        out.dev.col[d] = out.col[d];
        out.dev.dcol[out.col[d]] = d;
        if (d + 1 < q) {
            out.dev.depth[d].nxt_dist = out.dev.depth[d + 1].gen_dist;
            out.dev.depth[d].nxt_rel = out.dev.depth[d + 1].gen_rel;
        }
    }
    if (q >= 2) out.dev.root_rel = out.dev.depth[1].gen_rel;
    return Status::ok();
}

}  // namespace gfsm
