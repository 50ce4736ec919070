// Host-side construction of the per-network device programs: the production/loss sums of the RHS,
// the Newton-matrix entries, the elimination of the sparse pivots, the Schur update of the dense
// tail and the triangular solves, from the network's tables and the filled pattern of its sparse
// plan (newton_plan.py).
//
// Every program is a list of items (one result each, a list of operands) laid out for 64-lane
// waves.  A slice is 64 lanes working on 64/G items, G lanes an item: entry e of an item belongs
// to lane e % G of its group, position e / G; slices hold items of one G and similar length, so
// that little is padded, and are dealt to the waves longest first.  Operand records are stored by
// position, then lane: a wave's loads are contiguous and depend on nothing, so they can be issued
// ahead of the barrier before the phase that uses them.
#pragma once
#include <algorithm>
#include <array>
#include <cstdint>
#include <cstdlib>
#include <functional>
#include <map>
#include <set>
#include <vector>

namespace ucg {

// Slices of one phase in wave order: {first record row, positions, lanes per item, first header}.
struct SliceSet {
    std::vector<int> item;         // [slice][64] item of each lane's group, -1 none
    std::vector<int> len, lanes;   // per slice: positions, G
    std::vector<int> wave_ptr;     // [nwave + 1] slices of each wave
    int n() const { return (int)len.size(); }
};

// Packs items of the given lengths for nwave waves, at most `most` positions a lane where 64 lanes
// an item allow; `cost0` is a slice's fixed cost in positions.
inline SliceSet pack_slices_at(const std::vector<int> &length, int nwave, int most, double cost0, double &cost)
{
    struct It { int i, G, per; };
    std::vector<It> its;
    for (int i = 0; i < (int)length.size(); i++) {
        int G = 1;
        while (G < 64 && (length[i] + G - 1) / G > most) G *= 2;
        its.push_back({i, G, (length[i] + G - 1) / G});
    }
    std::stable_sort(its.begin(), its.end(), [](const It &a, const It &b) {
        return a.G != b.G ? a.G > b.G : a.per > b.per;
    });
    struct Sl { std::vector<int> item; int len, G; };
    std::vector<Sl> sl;
    for (size_t q = 0; q < its.size();) {
        Sl s;
        s.G = its[q].G;
        s.len = 0;
        s.item.assign(64, -1);
        for (int lane = 0; lane < 64 && q < its.size() && its[q].G == s.G; lane += s.G, q++) {
            for (int k = 0; k < s.G; k++) s.item[lane + k] = its[q].i;
            s.len = std::max(s.len, its[q].per);
        }
        sl.push_back(s);
    }
    std::vector<int> ord(sl.size());
    for (size_t k = 0; k < ord.size(); k++) ord[k] = (int)k;
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return sl[a].len > sl[b].len; });
    std::vector<double> load(nwave, 0.0);
    std::vector<std::vector<int>> mine(nwave);
    for (int k : ord) {
        const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        mine[w].push_back(k);
        int red = 0;
        for (int g = sl[k].G; g > 1; g /= 2) red++;
        load[w] += sl[k].len + cost0 + red;
    }
    cost = load.empty() ? 0.0 : *std::max_element(load.begin(), load.end());
    SliceSet S;
    S.wave_ptr.push_back(0);
    for (int w = 0; w < nwave; w++) {
        for (int k : mine[w]) {
            S.item.insert(S.item.end(), sl[k].item.begin(), sl[k].item.end());
            S.len.push_back(sl[k].len);
            S.lanes.push_back(sl[k].G);
        }
        S.wave_ptr.push_back(S.n());
    }
    return S;
}

// The packing whose busiest wave has least to do.
inline SliceSet pack_slices(const std::vector<int> &length, int nwave, double cost0 = 4.0)
{
    SliceSet best;
    double best_cost = -1.0;
    for (int most : {1, 2, 3, 4, 6, 8, 10, 12, 16, 20, 24, 28, 32, 40, 48, 64, 96, 128, 256}) {
        double cost;
        SliceSet S = pack_slices_at(length, nwave, most, cost0, cost);
        if (best_cost < 0.0 || cost < best_cost) {
            best = S;
            best_cost = cost;
        }
    }
    return best;
}

// Device form of one or more phases: slice descriptors, headers (one per lane) and operand records
// (RW 32-bit words per lane and row; `per_row` positions a row).  finish() gives every wave its
// slices of all phases as one list with the barriers that follow each, so that a wave can hold its
// descriptors in its lanes and fetch ahead across phases; `joined` puts no barriers between phases.
struct Program {
    std::vector<int> slices;       // [n][4] {first record row, rows, lanes per item, first header}
    std::vector<int> wave_ptr;     // [phases][nwave + 1]
    std::vector<uint32_t> hdr;     // [slice][64][hw]
    std::vector<uint32_t> rec;     // [row][64][rw]
    std::vector<int> list;         // [n][4] {first record row, rows, lanes per item + 256 x barriers after, first header}
    std::vector<int> list_ptr;     // [nwave + 1]
    int phases = 0;

    void finish(int nwave, bool joined = false)
    {
        const int none = (int)hdr.size();             // a header row of lanes without an item
        hdr.resize(hdr.size() + 64, 0u);
        list.clear();
        list_ptr.assign(1, 0);
        for (int w = 0; w < nwave; w++) {
            const size_t at = list.size();
            for (int p = 0; p < phases; p++) {
                const int *wp = &wave_ptr[p * (nwave + 1) + w];
                for (int s = wp[0]; s < wp[1]; s++) list.insert(list.end(), &slices[4 * s], &slices[4 * s] + 4);
                if (joined) continue;
                if (list.size() == at) list.insert(list.end(), {0, 0, 1, none});   // nothing yet in any phase
                list[list.size() - 2] += 256;
            }
            list_ptr.push_back((int)list.size() / 4);
        }
        list.resize(list.size() + 4 * 64, 0);         // lanes read a full wave of descriptors
    }

    // head(item or -1, words): fills the lane's header; entry(item, e, slot in row, words): fills
    // operand e of the item (or padding when e < 0) at its place in the row's words.
    void add(const SliceSet &S, int nwave, int hw, int rw, int per_row,
             const std::function<void(int, uint32_t *)> &head,
             const std::function<void(int, int, int, uint32_t *)> &entry, const std::vector<int> &length)
    {
        const int first = (int)slices.size() / 4;
        for (int w = 0; w <= nwave; w++) wave_ptr.push_back(first + S.wave_ptr[w]);
        for (int s = 0; s < S.n(); s++) {
            const int rows = (S.len[s] + per_row - 1) / per_row, G = S.lanes[s];
            slices.push_back((int)(rec.size() / (64 * rw)));
            slices.push_back(rows);
            slices.push_back(G);
            slices.push_back((int)(hdr.size() / hw));
            for (int l = 0; l < 64; l++) {
                uint32_t h[4] = {0, 0, 0, 0};
                const int it = S.item[64 * s + l];
                head(l % G == 0 ? it : -1, h);
                for (int k = 0; k < hw; k++) hdr.push_back(h[k]);
            }
            const size_t at = rec.size();
            rec.resize(at + (size_t)rows * 64 * rw, 0u);
            for (int r = 0; r < rows; r++)
                for (int l = 0; l < 64; l++)
                    for (int k = 0; k < per_row; k++) {
                        const int it = S.item[64 * s + l], e = (r * per_row + k) * G + l % G;
                        entry(it, it >= 0 && e < length[it] ? e : -1, k, &rec[at + ((size_t)r * 64 + l) * rw]);
                    }
        }
        phases++;
    }
};

inline void put16(uint32_t *w, int k, unsigned v) { w[k / 2] |= (v & 0xffffu) << (16 * (k & 1)); }

// ---------------------------------------------------------------- operand layout

// Extended state: y[0..neq) (density last), then these factors of the reaction terms.
enum { YX_ONE, YX_BLR, YX_ISM, YX_TSM, YX_N };

// Operands of the Newton-matrix entries: the partials of every reaction term (fac_off order), then
// one group of slots per structured coupling, then a zero for padding.
struct PartialSlots {
    int swap_u, swap_g, swap_nb, photo, transfer_t, transfer_d, densdot, zero, n;
};

inline PartialSlots partial_slots(int npart, int nsx, int nswap, int nsurfl)
{
    PartialSlots p;
    p.swap_u = npart;                       // d term / d totalSwap of each SURFSWAP term
    p.swap_g = p.swap_u + nsx;              // d totalSwap / d y of each BULKSWAP reactant
    p.swap_nb = p.swap_g + nswap;           // d totalSwap / d BULK
    p.photo = p.swap_nb + 1;                // H2: by y(H2), density; CO: by y(H2), y(CO), density
    p.transfer_t = p.photo + 5;             // transfer factor t of each surface species
    p.transfer_d = p.transfer_t + nsurfl;   // its derivatives by surface, bulk, SURFACE, BULK
    p.densdot = p.transfer_d + 4 * nsurfl;
    p.zero = p.densdot + 1;
    p.n = p.zero + 1;
    return p;
}

// Entry headers: target in bits 0..22 (a working slot, or a place in the tail or its panel), flags
// (ENTRY_TAIL: the value waits in the workspace).
enum : uint32_t { ENTRY_TARGET = 0x7fffffu, ENTRY_TAIL = 1u << 23, ENTRY_UNSCALED = 1u << 24, ENTRY_ONE = 1u << 25,
                  ENTRY_MINUS = 1u << 26, ENTRY_CHARGE = 1u << 27, ENTRY_CHARGE_ONE = 1u << 28,
                  ENTRY_CHARGE_MINUS = 1u << 29, ENTRY_VALID = 1u << 31 };
// Elimination headers: working slot, reciprocal flag; solve and sum headers: row.
enum : uint32_t { HDR_INDEX = 0xffffffu, HDR_RECIP = 1u << 30, HDR_VALID = 1u << 31 };
constexpr unsigned NO_SLOT = 0xffffu;

// Working slots of the sparse pivots in LDS, in order: the constants 1 and -1 and the scratch
// entries of L11 and U11; T = -inv(L11) below the diagonal; X = inv(U11); from slot at_L on L21,
// U12 and a zero.  The tail (t x t) overlays everything before at_L once the factors are stored.
// They are stored as four streams in the order the solves' slices read them, padded: stream
// element q takes slot[q] & 0xffff, times slot[q] >> 16 unless that is NO_SLOT; stream k starts at
// at[k].
struct SparsePrograms {
    int ns = 0, t = 0, nlev = 0;
    int at_L = 0, zero = 0, n_slots = 0, tail_hdr = 0, end_hdr = 0;
    int at[4] = {0, 0, 0, 0};
    std::vector<uint32_t> stream;
    std::vector<int> part_wave;       // [entry parts][nwave + 1] first header of each wave
    bool presum = false;              // the sum rows are not all tail rows: subtract sums up front
    std::vector<int> sum_rows;        // presum: {row, first, end} of the permuted members
    std::vector<int> sum_members;
    Program elim, entries, solve[4];   // solve: T, X, L21, U12
    // the tail's Schur update: one program, or with a wide tail one for each panel of 128 rows (x) 64
    // columns that is formed in LDS at a time
    std::vector<Program> schur;
    bool wide = false, ok = false;
};

struct EntryItem {
    uint32_t flags = 0;
    std::vector<std::pair<int, int>> c;   // (partial, coefficient)
};

// A wide tail (more rows than the waves hold as block columns) is inverted as 2 x 2 blocks, the
// first of WIDE_ROWS rows, and formed panel by panel: (row half, 64 columns), in columns of
// WIDE_LD doubles in LDS.
constexpr int WIDE_ROWS = 128, WIDE_COLS = 64, WIDE_LD = 130, WIDE_PANELS = 8;

// One network's tables as the planner reads them (the fields of ucg_network_desc it needs).
// `whole_blocks`: the tail may take more rows than the plan gives it.
template <class Desc>
SparsePrograms build_sparse_programs(const Desc *d, int nwave, int max_tail, const std::vector<int> &fac_off, int npart,
                                     bool whole_blocks = true)
{
    SparsePrograms S;
    const int neq = d->neq, NN = d->nw_sizes[0], ns0 = d->nw_sizes[1], T0 = d->nw_sizes[2], nsp0 = d->nw_sizes[3];
    if (T0 > 2 * max_tail) return S;
    S.wide = T0 > max_tail;
    if (S.wide) max_tail *= 2;
    // the tail fills whole 16-row blocks: the rows up to the next block cost its inversion nothing
    // and leave the sparse pivots with fewer levels.  They cost LDS, though: up to 15 rows and columns
    // of up to 128 doubles, 13.8 KB with the default network's tail, so that a plan which fits
    // without them is built without them if it does not fit with them.
    const int T = whole_blocks || S.wide ? std::min(std::min((T0 + 15) / 16 * 16, max_tail), NN) : T0, ns = NN - T;
    S.ns = ns;
    S.t = T;
    if (S.wide && T % 16 != 0) return S;
    // tail element -> panel and place in it
    const int halves = S.wide ? 2 : 1, cols = S.wide ? (T + WIDE_COLS - 1) / WIDE_COLS : 1, panels = halves * cols;
    auto panel_of = [&](int r, int c) { return S.wide ? ((c - ns) / WIDE_COLS) * halves + (r - ns) / WIDE_ROWS : 0; };
    auto place_of = [&](int r, int c) {
        return S.wide ? ((c - ns) % WIDE_COLS) * WIDE_LD + (r - ns) % WIDE_ROWS : (c - ns) * T + (r - ns);
    };
    // filled pattern
    std::vector<std::vector<int>> Lrow(NN), Urow(ns), Ucol(NN);   // L(r, c < r), U(r, c >= r), sparse pivots only
    auto pivot_row = [&](int r, int c) {
        if (c < r) Lrow[r].push_back(c);
        else {
            Urow[r].push_back(c);
            if (c > r) Ucol[c].push_back(r);
        }
    };
    for (int r = 0; r < NN; r++) {
        const std::set<int> cols(d->nw_sp_col + d->nw_sp_ptr[r], d->nw_sp_col + d->nw_sp_ptr[r + 1]);
        for (int c : cols)
            if (std::min(r, c) < ns) pivot_row(r, c);
    }
    // the pattern must hold its own fill (and every pivot), or the caller's schedule is used as it is
    {
        std::set<std::pair<int, int>> has;
        std::vector<std::vector<int>> Lcol(ns);
        for (int r = 0; r < NN; r++)
            for (int c : Lrow[r]) {
                has.insert({r, c});
                Lcol[c].push_back(r);
            }
        for (int r = 0; r < ns; r++) {
            for (int c : Urow[r]) has.insert({r, c});
            if (!has.count({r, r})) return S;
        }
        for (int p = 0; p < ns; p++)
            for (int r : Lcol[p])
                for (int c : Urow[p])
                    if (c > p && std::min(r, c) < ns && !has.count({r, c})) return S;
    }
    std::vector<int> level(ns, 0);
    for (int k = 0; k < ns; k++) {
        for (int p : Lrow[k]) level[k] = std::max(level[k], level[p] + 1);
        for (int p : Ucol[k]) level[k] = std::max(level[k], level[p] + 1);
        S.nlev = std::max(S.nlev, level[k] + 1);
    }
    // patterns of T = -inv(L11) (strict) and X = inv(U11)
    std::vector<std::set<int>> Tp(ns), Xc(ns);
    for (int r = 0; r < ns; r++)
        for (int p : Lrow[r]) {
            Tp[r].insert(p);
            Tp[r].insert(Tp[p].begin(), Tp[p].end());
        }
    for (int c = 0; c < ns; c++) {
        Xc[c].insert(c);
        for (int p : Ucol[c]) Xc[c].insert(Xc[p].begin(), Xc[p].end());
    }
    std::vector<std::vector<int>> Xr(ns);
    for (int c = 0; c < ns; c++)
        for (int r : Xc[c]) Xr[r].push_back(c);
    // right-hand-side sums of the replaced rows: entries of their L21 rows on the permuted
    // right-hand side itself when all those rows lie in the tail
    const int NB = d->special_species[24], NS = d->special_species[23], NE = d->special_species[21];
    const bool charge = NE < d->nspec;   // as the device decides: with no positive ion the sum is empty
    std::vector<std::pair<int, std::vector<int>>> sums(3);
    sums[0].first = d->nw_inv[NB];
    for (int q = 0; q < d->nbulkl; q++) sums[0].second.push_back(d->nw_inv[d->bulk_list[q]]);
    sums[1].first = d->nw_inv[NS];
    for (int q = 0; q < d->nsurfl; q++) sums[1].second.push_back(d->nw_inv[d->surface_list[q]]);
    sums[2].first = charge ? d->nw_inv[NE] : -1;
    if (charge)
        for (int q = 0; q < d->nion; q++) sums[2].second.push_back(d->nw_inv[d->ion_list[q]]);
    S.presum = sums[0].first < ns || sums[1].first < ns || (charge && sums[2].first < ns);
    for (auto &x : sums) {
        S.sum_rows.push_back(x.first);
        S.sum_rows.push_back((int)S.sum_members.size());
        S.sum_members.insert(S.sum_members.end(), x.second.begin(), x.second.end());
        S.sum_rows.push_back((int)S.sum_members.size());
    }
    // solve phases: rows and their operands
    const int npad = (NN + 7) & ~7;   // w at 0, v at npad, x at 2 npad of the solve's vectors
    struct Op { int col; int kind; };   // kind 0: pivot entry, 1: constant 1, 2: 1 under charge enforcement
    std::vector<std::vector<Op>> rows[4];
    for (int r = 0; r < ns; r++) {
        std::vector<Op> t, x, u;
        for (int c : Tp[r]) t.push_back({c, 0});
        for (int c : Xr[r]) x.push_back({c, 0});
        for (int c : Urow[r])
            if (c >= ns) u.push_back({2 * npad + c, 0});
        rows[0].push_back(t);
        rows[1].push_back(x);
        rows[3].push_back(u);
    }
    for (int r = ns; r < NN; r++) {
        std::vector<Op> l;
        for (int c : Lrow[r]) l.push_back({npad + c, 0});
        if (!S.presum)
            for (int k = 0; k < 3; k++)
                if (sums[k].first == r)
                    for (int c : sums[k].second) l.push_back({c, k == 2 ? 2 : 1});
        rows[2].push_back(l);
    }
    // slots
    std::map<std::pair<int, int>, int> slotL, slotU, slotT, slotX;   // by (row, column)
    std::vector<int> one_slots, charge_slots;
    int n = 0;
    const int ONE = n++, MONE = n++;
    for (int r = 0; r < ns; r++) {
        for (int c : Lrow[r]) slotL[{r, c}] = n++;
        for (int c : Urow[r])
            if (c > r && c < ns) slotU[{r, c}] = n++;
    }
    const int first_row[4] = {0, 0, ns, 0};
    std::vector<int> stream_slot;     // -1: padding
    for (int ph = 0; ph < 4; ph++) {
        std::vector<int> len;
        for (auto &r : rows[ph]) len.push_back((int)r.size());
        const SliceSet P = pack_slices(len, nwave);
        if (ph == 2) S.at_L = n;
        S.at[ph] = (int)stream_slot.size();
        S.solve[ph].add(
            P, nwave, 1, 1, 1,
            [&](int it, uint32_t *h) { h[0] = it >= 0 ? (HDR_VALID | (uint32_t)(first_row[ph] + it)) : 0u; },
            [&](int it, int e, int, uint32_t *w) { w[0] = e >= 0 ? (uint32_t)rows[ph][it][e].col : 0u; }, len);
        for (int s = 0; s < P.n(); s++)
            for (int pos = 0; pos < P.len[s]; pos++)
                for (int l = 0; l < 64; l++) {
                    const int it = P.item[64 * s + l], e = pos * P.lanes[s] + l % P.lanes[s];
                    if (it < 0 || e >= len[it]) {
                        stream_slot.push_back(-1);
                        continue;
                    }
                    const Op &o = rows[ph][it][e];
                    const int sl = n++, r = first_row[ph] + it;
                    stream_slot.push_back(sl);
                    if (o.kind == 1) one_slots.push_back(sl);
                    else if (o.kind == 2) charge_slots.push_back(sl);
                    else if (ph == 0) slotT[{r, o.col}] = sl;
                    else if (ph == 1) slotX[{r, o.col}] = sl;
                    else if (ph == 2) slotL[{r, o.col - npad}] = sl;
                    else slotU[{r, o.col - 2 * npad}] = sl;
                }
    }
    S.zero = n++;
    S.n_slots = n;
    if (n >= (int)NO_SLOT) return S;
    const int ZERO = S.zero;
    auto X = [&](int r, int c) { return slotX.at({r, c}); };
    // the pivot U(k, k) is eliminated in the slot of X(k, k), its reciprocal
    auto Us = [&](int r, int c) { return r == c ? X(r, r) : slotU.at({r, c}); };
    // elimination: one phase a level.  L and X hold their unscaled values (L D and X without the
    // column's reciprocal), so that a level needs nothing of itself; products carry the pivot's
    // reciprocal as a third factor
    struct Target { int slot; bool recip; std::vector<std::array<int, 3>> p; };
    std::vector<std::vector<Target>> ph(S.nlev);
    std::vector<std::vector<int>> Lcol(ns);
    for (int r = 0; r < NN; r++)
        for (int c : Lrow[r]) Lcol[c].push_back(r);
    auto pairs = [&](int r, int c, int stop) {   // sum over p < stop of L(r, p) U(p, c)
        std::vector<std::array<int, 3>> v;
        for (int p : Lrow[r])
            if (p < stop && slotU.count({p, c})) v.push_back({slotL.at({r, p}), X(p, p), slotU.at({p, c})});
        return v;
    };
    for (int k = 0; k < ns; k++) {
        auto &t = ph[level[k]];
        for (int c : Urow[k]) {
            auto v = pairs(k, c, k);
            if (c == k) t.push_back({Us(k, k), true, v});
            else if (!v.empty()) t.push_back({slotU.at({k, c}), false, v});
        }
        for (int r : Lcol[k]) {
            auto v = pairs(r, k, k);
            if (!v.empty()) t.push_back({slotL.at({r, k}), false, v});
        }
        for (int c : Tp[k]) {   // T(k, c) = L(k, c) - sum L(k, p) T(p, c)
            std::vector<std::array<int, 3>> v;
            if (slotL.count({k, c})) v.push_back({slotL.at({k, c}), X(c, c), MONE});
            for (int p : Lrow[k])
                if (p > c && slotT.count({p, c})) v.push_back({slotL.at({k, p}), X(p, p), slotT.at({p, c})});
            t.push_back({slotT.at({k, c}), false, v});
        }
        for (int r : Xc[k]) {   // X(r, k) X(k, k)^-1 = -sum X(r, p) U(p, k)
            if (r == k) continue;
            std::vector<std::array<int, 3>> v;
            for (int p : Ucol[k])
                if (p == r) v.push_back({ONE, X(r, r), slotU.at({r, k})});
                else if (p > r && slotX.count({r, p})) v.push_back({X(r, p), X(p, p), slotU.at({p, k})});
            t.push_back({X(r, k), false, v});
        }
    }
    for (auto &t : ph) {
        std::vector<int> len;
        for (auto &x : t) len.push_back((int)x.p.size());
        const SliceSet P = pack_slices(len, nwave);
        S.elim.add(
            P, nwave, 1, 2, 1,
            [&](int it, uint32_t *h) {
                h[0] = it >= 0 ? (HDR_VALID | (t[it].recip ? HDR_RECIP : 0u) | (uint32_t)t[it].slot) : 0u;
            },
            [&](int it, int e, int, uint32_t *w) {
                for (int q = 0; q < 3; q++) put16(w, q, e >= 0 ? t[it].p[e][q] : ZERO);
            },
            len);
    }
    // X off the diagonal and L21 take their column's pivot when they are stored
    std::vector<unsigned> scale(S.n_slots, NO_SLOT);
    for (auto &kv : slotX)
        if (kv.first.first != kv.first.second) scale[kv.second] = (unsigned)X(kv.first.second, kv.first.second);
    for (auto &kv : slotL)
        if (kv.first.first >= ns) scale[kv.second] = (unsigned)X(kv.first.second, kv.first.second);
    for (int sl : stream_slot)
        S.stream.push_back(sl < 0 ? ((unsigned)ZERO | NO_SLOT << 16) : ((unsigned)sl | scale[sl] << 16));
    // Schur complement of the tail
    {
        std::vector<std::vector<int>> ucols(ns);
        for (int r = 0; r < ns; r++)
            for (int c : Urow[r])
                if (c >= ns) ucols[r].push_back(c);
        std::vector<std::map<std::pair<int, int>, std::vector<std::array<int, 2>>>> by(panels);
        for (int r = ns; r < NN; r++)
            for (int p : Lrow[r])
                for (int c : ucols[p]) by[panel_of(r, c)][{r, c}].push_back({slotL.at({r, p}), slotU.at({p, c})});
        for (auto &m : by) {
            std::vector<const std::vector<std::array<int, 2>> *> it;
            std::vector<int> where, len;
            for (auto &kv : m) {
                it.push_back(&kv.second);
                where.push_back(place_of(kv.first.first, kv.first.second));
                len.push_back((int)kv.second.size());
            }
            const SliceSet P = pack_slices(len, nwave);
            S.schur.emplace_back();
            S.schur.back().add(
                P, nwave, 1, 2, 2, [&](int i, uint32_t *h) { h[0] = i >= 0 ? (HDR_VALID | (uint32_t)where[i]) : 0u; },
                [&](int i, int e, int k, uint32_t *w) {
                    put16(w, 2 * k, e >= 0 ? (*it[i])[e][0] : ZERO);
                    put16(w, 2 * k + 1, e >= 0 ? (*it[i])[e][1] : ZERO);
                },
                len);
            S.schur.back().finish(nwave, true);
        }
    }
    // ---------------- entries of M = I - gamma J (augmented), by place
    std::vector<std::pair<int, int>> place(nsp0 + T0 * T0);   // plan slot -> (row, column)
    for (int r = 0; r < NN; r++)
        for (int q = d->nw_sp_ptr[r]; q < d->nw_sp_ptr[r + 1]; q++) place[q] = {r, d->nw_sp_col[q]};
    for (int c = 0; c < T0; c++)
        for (int r = 0; r < T0; r++) place[nsp0 + c * T0 + r] = {ns0 + r, ns0 + c};
    std::map<std::pair<int, int>, EntryItem> ent;
    auto E = [&](int plan_slot) -> EntryItem & { return ent[place[plan_slot]]; };
    const PartialSlots ps = [&] {
        int nsx = 0;
        for (int k = 0; k < d->nreac; k++) {
            bool sw = false;
            for (int m = 0; m < d->nfac[k]; m++) sw |= d->fac[10 * k + m] == -3;
            nsx += sw;
        }
        return partial_slots(npart, nsx, d->nswap, d->nsurfl);
    }();
    std::vector<int> sx(d->nreac, -1);
    for (int k = 0, q = 0; k < d->nreac; k++)
        for (int m = 0; m < d->nfac[k]; m++)
            if (d->fac[10 * k + m] == -3) {
                sx[k] = q++;
                break;
            }
    // generated terms
    for (int e = 0; e < d->nnz; e++)
        for (int q = d->jnz_ptr[e]; q < d->jnz_ptr[e + 1]; q++)
            E(d->nw_jnz_slot[e]).c.push_back({fac_off[d->jc_k[q]] + d->jc_m[q], d->jc_c[q]});
    for (int i = 0; i < neq; i++)
        if (d->nw_diag_slot[i] >= 0) E(d->nw_diag_slot[i]).flags |= ENTRY_ONE;
    // totalSwap column u1 and row g1, the coupling c1 of the two borders
    EntryItem &c1 = E(d->nw_misc[2]);
    c1.flags |= ENTRY_UNSCALED;
    std::vector<char> is_surf(neq, 0);
    for (int q = 0; q < d->nsurfl; q++) is_surf[d->surface_list[q]] = 1;
    for (int i = 0; i < neq; i++) {
        if (d->nw_s1c[i] >= 0) {
            EntryItem &u = E(d->nw_s1c[i]);
            u.flags |= ENTRY_UNSCALED;
            for (int q = d->sw_ptr[i]; q < d->sw_ptr[i + 1]; q++) {
                if (sx[d->sw_k[q]] < 0) return S;
                u.c.push_back({ps.swap_u + sx[d->sw_k[q]], d->sw_c[q]});
            }
        }
        if (is_surf[i])
            for (int q = d->sw_ptr[i]; q < d->sw_ptr[i + 1]; q++) {
                if (sx[d->sw_k[q]] < 0) return S;
                c1.c.push_back({ps.swap_u + sx[d->sw_k[q]], d->sw_c[q]});
            }
    }
    for (int q = 0; q < d->nswap; q++) {
        const int b = d->ops[6 * d->swap_list[q]];
        if (d->nw_s1r[b] >= 0) E(d->nw_s1r[b]).c.push_back({ps.swap_g + q, 1});
    }
    if (d->nw_s1r[NB] >= 0) E(d->nw_s1r[NB]).c.push_back({ps.swap_nb, 1});
    // gsum0: the generated terms of the surface rows, summed by column (what moves between surface
    // species cancels here)
    {
        std::vector<int> entry_of(nsp0 + T0 * T0, -1);
        for (int e = 0; e < d->nnz; e++) entry_of[d->nw_jnz_slot[e]] = e;
        for (int j = 0; j < neq; j++) {
            if (d->nw_s2r[j] < 0) continue;
            EntryItem &g = E(d->nw_s2r[j]);
            for (int q = d->nw_gs_ptr[j]; q < d->nw_gs_ptr[j + 1]; q++) {
                const int e = entry_of[d->nw_gs_slot[q]];
                if (e < 0) return S;
                for (int k = d->jnz_ptr[e]; k < d->jnz_ptr[e + 1]; k++)
                    g.c.push_back({fac_off[d->jc_k[k]] + d->jc_m[k], d->jc_c[k]});
            }
        }
    }
    // transfer column w2, its S-terms, photo columns, the density row
    for (int q = 0; q < d->nsurfl; q++) {
        const int s = d->surface_list[q], b = d->bulk_partner_of_surface[s];
        if (b < 0 || d->nw_s2c[s] < 0 || d->nw_s2c[b] < 0) return S;
        E(d->nw_s2c[s]).flags |= ENTRY_UNSCALED;
        E(d->nw_s2c[b]).flags |= ENTRY_UNSCALED;
        E(d->nw_s2c[s]).c.push_back({ps.transfer_t + q, -1});
        E(d->nw_s2c[b]).c.push_back({ps.transfer_t + q, 1});
        for (int m = 0; m < 4; m++) {
            E(d->nw_tr_slot[8 * q + m]).c.push_back({ps.transfer_d + 4 * q + m, -1});
            E(d->nw_tr_slot[8 * q + 4 + m]).c.push_back({ps.transfer_d + 4 * q + m, 1});
        }
    }
    {
        int m3 = 0;
        for (int which = 0; which < 2; which++) {
            const int k = d->special_reactions[which ? 7 : 6];
            for (int q = d->aff_ptr[k]; q < d->aff_ptr[k + 1]; q++, m3 += 3) {
                const int *p = d->nw_ph_slot + m3, f = d->aff_cf[q];
                E(p[0]).c.push_back({ps.photo + (which ? 2 : 0), f});
                if (which) E(p[1]).c.push_back({ps.photo + 3, f});
                E(p[2]).c.push_back({ps.photo + (which ? 4 : 1), f});
            }
        }
    }
    if (d->nw_diag_slot[neq - 1] >= 0) E(d->nw_diag_slot[neq - 1]).c.push_back({ps.densdot, 1});
    // constants: the replaced rows, the borders' diagonals, the charge row
    auto constant = [&](int slot, uint32_t f) {
        EntryItem &e = E(slot);
        e.c.clear();
        e.flags = (e.flags & ~(ENTRY_ONE | ENTRY_MINUS)) | f;
    };
    for (int q = 0; q < d->nbulkl; q++) constant(d->nw_nbrow[q], ENTRY_MINUS);
    for (int q = 0; q < d->nsurfl; q++) constant(d->nw_nsrow[q], ENTRY_MINUS);
    constant(d->nw_misc[0], ENTRY_MINUS);
    constant(d->nw_misc[1], ENTRY_MINUS);
    constant(d->nw_misc[3], ENTRY_ONE);
    constant(d->nw_misc[4], ENTRY_ONE);
    if (charge) {
        for (int q = 0; q < d->nw_nerow; q++) E(d->nw_erow[q]).flags |= ENTRY_CHARGE;
        for (int q = 0; q < d->nion; q++) E(d->nw_eion[q]).flags |= ENTRY_CHARGE | ENTRY_CHARGE_MINUS;
        if (d->nw_diag_slot[NE] >= 0) E(d->nw_diag_slot[NE]).flags |= ENTRY_CHARGE | ENTRY_CHARGE_ONE;
    }
    // items: working slots (with the constant slots of the streams), then the panels of the tail.
    // Values whose place the operands still occupy wait in the workspace (ENTRY_TAIL).
    std::vector<uint32_t> head;
    std::vector<std::vector<unsigned>> op;
    std::vector<int> len;
    for (int part = 0; part < 1 + panels; part++) {
        head.clear();
        op.clear();
        len.clear();
        const uint32_t waits = part > 0 || S.wide ? ENTRY_TAIL : 0u;
        auto item = [&](uint32_t h, const std::vector<std::pair<int, int>> &c) {
            std::map<int, int> merged;
            for (auto &x : c) merged[x.first] += x.second;
            std::vector<unsigned> v;
            for (auto &x : merged)
                for (int k = 0; k < std::abs(x.second); k++) v.push_back((unsigned)x.first | (x.second < 0 ? 0x8000u : 0u));
            head.push_back(h);
            len.push_back((int)v.size());
            op.push_back(v);
        };
        for (auto &kv : ent) {
            const int r = kv.first.first, c = kv.first.second;
            const bool tail = r >= ns && c >= ns;
            if ((tail ? 1 + panel_of(r, c) : 0) != part) continue;
            const int target = tail ? place_of(r, c) : c < r ? slotL.at({r, c}) : Us(r, c);
            item(ENTRY_VALID | kv.second.flags | waits | (uint32_t)target, kv.second.c);
        }
        if (part == 0) {
            const std::vector<std::pair<int, int>> none;
            item(ENTRY_VALID | waits | ENTRY_ONE | (uint32_t)ONE, none);
            item(ENTRY_VALID | waits | ENTRY_MINUS | (uint32_t)MONE, none);
            for (int sl : one_slots) item(ENTRY_VALID | waits | ENTRY_ONE | (uint32_t)sl, none);
            for (int sl : charge_slots) item(ENTRY_VALID | waits | ENTRY_CHARGE | ENTRY_CHARGE_ONE | (uint32_t)sl, none);
        }
        const SliceSet P = pack_slices(len, nwave);
        if (part == (S.wide ? 0 : 1)) S.tail_hdr = (int)S.entries.hdr.size();   // the first that waits
        for (int w = 0; w <= nwave; w++) S.part_wave.push_back((int)S.entries.hdr.size() + 64 * P.wave_ptr[w]);
        S.entries.add(
            P, nwave, 1, 2, 4, [&](int i, uint32_t *h) { h[0] = i >= 0 ? head[i] : 0u; },
            [&](int i, int e, int k, uint32_t *w) { put16(w, k, e >= 0 ? op[i][e] : (unsigned)ps.zero); }, len);
    }
    S.end_hdr = (int)S.entries.hdr.size();
    S.elim.finish(nwave);
    S.entries.finish(nwave, true);
    for (Program &P : S.solve) P.finish(nwave, true);
    S.ok = ps.n < 0x8000;
    return S;
}

}  // namespace ucg
