// single.hip -- host side of the single-root search (single.h): pg_perft for
// the slider variants whose tables leave the LDS to the fused leaf.
#include <chrono>
#include <cstring>
#include <memory>
#include "engine.h"
#include "single.h"

using namespace pg;

namespace pg {

struct Single {
    SPlan *plan = nullptr;
    SResult *res = nullptr;  // pinned; the last kernel of a search writes it
    u64 seq = 0;
    bool clear = false;      // the counters are zero: the last search ended with its last kernel
};

void single_delete(Single *s) {
    if (!s) return;
    if (s->plan) (void)hipFree(s->plan);
    if (s->res) (void)hipHostFree(s->res);
    delete s;
}

// (nothing half made is kept)
static int single_init(Engine &e) {
    std::unique_ptr<Single, void (*)(Single *)> s(new Single(), single_delete);
    HIP_TRY(hipMalloc(&s->plan, sizeof(SPlan)));
    HIP_TRY(hipHostMalloc(&s->res, sizeof(SResult)));
    memset(s->res, 0, sizeof(SResult));
    e.single = s.release();
    return PG_OK;
}

// Waits for the result: the last work-group writes it to pinned memory, which
// the host sees sooner than the stream's end (a search of a few plies takes
// tens of microseconds); a long search is waited for by the stream.
static int wait_result(Engine &e, const Single &s) {
    const auto t0 = std::chrono::steady_clock::now();
    for (u32 spin = 0;; spin++) {
        if (__atomic_load_n(&s.res->seq, __ATOMIC_ACQUIRE) == s.seq) return PG_OK;
        if (spin % 64 == 63 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(500)) break;
    }
    HIP_TRY(hipStreamSynchronize(e.stream));
    if (__atomic_load_n(&s.res->seq, __ATOMIC_ACQUIRE) == s.seq) return PG_OK;
    set_error("perft: the search ended without a result");
    return PG_EHIP;
}

template <int V>
static void launch(Engine &e, const Single &s, const SRoot &r, const SRegion &rg, int depth, u64 bias) {
    hipStream_t st = e.stream;
    if (depth <= 2) {
        ks_one<V><<<1, LEAF_WG, 0, st>>>(r, s.plan, depth, bias, s.res, s.seq, e.dt);
    } else if (depth == 3 || r.n == 0) {
        const int g = r.n ? (r.n + S_WAVES - 1) / S_WAVES : 1;
        ks_three<V><<<g, LEAF_WG, 0, st>>>(r, s.plan, bias, s.res, s.seq, e.dt);
    } else if (depth == 4) {
        ks_four<V><<<r.n * S_FOUR_PARTS, LEAF_WG, 0, st>>>(r, s.plan, bias, s.res, s.seq, e.dt);
    } else {
        ks_top<V><<<r.n * S_TOP_PARTS, LEAF_WG, 0, st>>>(r, s.plan, rg, e.dt);
        for (int l = 3; l <= depth - 2; l++) {
            const bool set = (rg.collapse >> l) & 1;
            if (set) {
                ks_clear<<<l <= 3 ? 64 : e.cus * 8, 256, 0, st>>>(s.plan, rg, l);
                ks_collapse<<<l <= 3 ? 256 : e.cus * 8, S_COLLAPSE_WG, 0, st>>>(s.plan, rg, l, e.dt);
            }
            if (l == depth - 2) {
                const int g = e.cus * 3;  // as many as are resident
                if (set) ks_leaf<V, false><<<g, LEAF_WG, 0, st>>>(s.plan, rg, depth, bias, s.res, s.seq, e.dt);
                else ks_leaf<V, true><<<g, LEAF_WG, 0, st>>>(s.plan, rg, depth, bias, s.res, s.seq, e.dt);
            } else {
                const int g = l <= 3 ? S_RESIDENT : e.cus * 16;
                if (set) ks_level<V, false><<<g, LEAF_WG, 0, st>>>(s.plan, rg, l, e.dt);
                else ks_level<V, true><<<g, LEAF_WG, 0, st>>>(s.plan, rg, l, e.dt);
            }
        }
    }
}

// perft of one root.  *fits is false (and nothing is returned) when a level
// does not fit the arena, or a board's moves a list.  collapse: merge the equal boards of each ply from
// the third on (two plies have no transpositions) of searches deep enough.
int perft_single(Engine &e, const Pos &root, u32 depth, int v, bool collapse, u64 *out, bool *fits) {
    *fits = false;
    if (!e.single) {
        const int rc = single_init(e);
        if (rc) return rc;
    }
    Single &s = *e.single;
    const HostTables *ht = host_tables(nullptr);
    if (!ht) return PG_ETABLE;
    SRoot r{};
    r.b = root;
    u32 word[256];
    r.n = generate_words<SL_KOGGE>(root, ht->view(), word, 256, 0);
    if (r.n > S_MOVES) return PG_OK;  // more queens than a game has: the root's list does not hold them
    for (u32 i = 0; i < r.n; i++) {
        r.mv[i] = (u16)word[i];
        r.piece[i] = (u8)piece_code(word[i] >> 24);
    }
    SRegion rg{};
    rg.bytes = (e.arenaBytes / 2) & ~(size_t)255;
    rg.half[0] = e.arena;
    rg.half[1] = e.arena + rg.bytes;
    rg.node2 = (u64)r.n * S_MOVES;
    if (collapse && depth >= 6)
        for (u32 l = 3; l + 2 <= depth; l++) rg.collapse |= 1ULL << l;
    if (depth >= 5 && rg.node2 * sizeof(SNode) > rg.bytes / 2) return PG_OK;
    // before the first search, and after one that broke off
    if (!s.clear) HIP_TRY(hipMemsetAsync(s.plan, 0, sizeof(SPlan), e.stream));
    s.clear = false;
    s.seq++;
    PG_VARIANT_CALL_LDS(v, launch, e, s, r, rg, (int)depth, e.bias);
    HIP_TRY(hipGetLastError());
    const int rc = wait_result(e, s);
    if (rc) return rc;
    s.clear = true;
    const SResult &h = *s.res;
    if (h.overflow) return PG_OK;
    if (h.ovf) {
        set_error("perft: a perft total does not fit 64 bits");
        return PG_EOVERFLOW;
    }
    if (h.err) {
        set_error("perft: device consistency check failed (flag %u)", h.err);
        return PG_EINVAL;
    }
    *fits = true;
    *out = h.acc;
    e.stats.leaf_items = h.items;
    e.stats.leaf_parents = depth == 2 ? 1 : depth <= 4 ? h.paths[depth >= 2 ? depth - 2 : 0] : h.boards;
    e.stats.leaf_launches = depth >= 2 ? 1 : 0;
    for (u32 l = 1; l < depth && l < 16; l++) e.stats.nodes[l] = h.paths[l];
    return PG_OK;
}

}  // namespace pg
