// compact.cpp — builds the 16-bit LDS plan image (compact.h) from a Plan.
//
// Same F pattern and the same entry-level LU tasks as the global plan, with
//   * the forward substitution merged into the LU levels: y_k is one more
//     task whose level is one past the latest of its L entries and y inputs;
//   * MOSFET stamps reduced to (id, dI/dVd, dI/dVg) in structure-of-arrays
//     order (dI/dVs is their negated sum);
//   * the linear stamps kept only where an entry has a G or C contribution;
//   * every operand as a byte offset into the instance's region.
#include "compact.h"

#include <algorithm>

#include "plan.h"

namespace cedar {

namespace {

struct Blob {
    std::vector<uint16_t> w;
    bool ok = true;
    void align(int a) {
        while (w.size() % a) w.push_back(0);
    }
    int32_t add(const std::vector<int32_t>& v, int a = 1) {
        align(a);
        int32_t off = (int32_t)w.size();
        for (int32_t x : v) {
            if (x < 0 || x > 0xFFFF) ok = false;
            w.push_back((uint16_t)(x & 0xFFFF));
        }
        return off;
    }
};

}  // namespace

bool build_compact(const Plan& P, std::vector<uint16_t>& blob, CPlan& cp,
                   std::vector<int32_t>& lpos, std::vector<int32_t>& colnat, std::vector<int32_t>& diffrow,
                   std::vector<int32_t>& probe, std::vector<int32_t>& dev,
                   std::vector<int32_t>& devrow, const char** why) {
    const int32_t n = P.n, nnz = P.nnz, nm = P.n_mos, ns = P.n_src;
    cp = CPlan{};
    *why = "";
    if (n >= 0x7FFF || nnz >= 0xFFFF || 3 * nm + ns >= 0x7FFF) {
        *why = "circuit too large for 16-bit indices";
        return false;
    }
    if (P.n_va > 0) {
        *why = "Verilog-A devices run on the global-plan kernel";
        return false;
    }
    // linear entries by row
    lpos.clear();
    std::vector<int32_t> lptr(n + 1, 0), lcolk, elin(nnz, -1);
    for (int32_t k = 0; k < n; k++) {
        for (int32_t e = P.rowptr[k]; e < P.rowptr[k + 1]; e++)
            if (P.g_ptr[e + 1] > P.g_ptr[e] || P.c_ptr[e + 1] > P.c_ptr[e]) {
                elin[e] = (int32_t)lpos.size();
                lpos.push_back(e);
                lcolk.push_back(P.colperm[e]);
            }
        lptr[k + 1] = (int32_t)lpos.size();
    }
    const int32_t nlin = (int32_t)lpos.size();
    // sources: data and dc value copied to wd
    int32_t nwd = 0;
    for (int32_t s = 0; s < ns; s++) nwd += P.src[s].len + 1;

    // the region
    int32_t q8 = 2 * (nlin + 1);
    auto take = [&](int32_t k) { const int32_t o = 8 * q8; q8 += k; return o; };
    cp.b_F = take(nnz);
    cp.b_x = take(n);
    cp.b_inv = take(n);
    cp.b_u = take(n);
    cp.b_zero = take(1);
    cp.b_one = take(1);
    cp.b_trash = take(1);
    cp.b_st = take(3 * nm + ns);
    cp.b_wd = take(nwd);
    cp.dbl = q8;
    // A region past 16-bit byte offsets is larger than a workgroup's LDS
    // limit: the caller refuses it by its size and the image is never read.
    const bool fits = 8 * (int64_t)q8 < 0x10000;
    auto bF = [&](int32_t e) { return cp.b_F + 8 * e; };
    auto bX = [&](int32_t k) { return cp.b_x + 8 * k; };
    auto bI = [&](int32_t k) { return cp.b_inv + 8 * k; };
    auto bU = [&](int32_t k) { return cp.b_u + 8 * k; };

    // stamp references: old 4-per-device layout -> SoA 3-per-device byte offsets
    auto conv = [&](int32_t ref, std::vector<int32_t>& out) {
        const int32_t s = ref >> 1;
        const bool neg = ref & 1;
        auto put = [&](int32_t idx, bool ng) { out.push_back((cp.b_st + 8 * idx) | (ng ? 1 : 0)); };
        if (s < 4 * nm) {
            const int32_t m = s / 4, j = s % 4;
            if (j == 0) put(m, neg);
            else if (j == 1) put(nm + m, neg);
            else if (j == 2) put(2 * nm + m, neg);
            else {
                put(nm + m, !neg);
                put(2 * nm + m, !neg);
            }
        } else {
            put(3 * nm + (s - 4 * nm), neg);
        }
    };

    // LU tasks with their levels (recomputed from the task list: level of a
    // task = 1 + max level of the entries it reads; a diagonal's level gates
    // the L entries scaled by it).  Level 0 diagonals are formed and inverted
    // by the assembly.
    struct Task {
        int32_t d, s;          // destination; scale, or the inverse's slot
        bool dia;
        std::vector<int32_t> up;   // a b pairs
    };
    const int32_t n_lulev = (int32_t)P.lu_lptr.size() - 1;
    std::vector<int32_t> lev(nnz, -1);
    std::vector<char> dia0(nnz, 0);
    for (int32_t l = 0; l < n_lulev; l++)
        for (int32_t q = P.lu_lptr[l]; q < P.lu_lptr[l + 1]; q++) {
            const LuTask& t = P.lu_task[q];
            lev[t.e] = l;
            if (t.piv <= -2 && t.ub == t.ue) dia0[t.e] = 1;
        }
    // assembly records
    std::vector<int32_t> ea, eb, ec, ed, ez, items, refs;
    const int32_t Z = cp.b_zero, ZL = 16 * nlin;   // zero stamp, zero (G, C) pair
    std::vector<int32_t> diaInv(nnz, -1);
    for (int32_t k = 0; k < n; k++) diaInv[P.diag[k]] = k;
    std::vector<char> inv_step(n, 0);   // a level-0 diagonal left to a step of its own
    for (int32_t e = 0; e < nnz; e++) {
        std::vector<int32_t> r;
        for (int32_t q = P.jnl_ptr[e]; q < P.jnl_ptr[e + 1]; q++) conv(P.jnl_ref[q], r);
        const int32_t l = elin[e] >= 0 ? 16 * elin[e] : ZL;
        const size_t nrf = r.size();
        const bool d0 = dia0[e] != 0;
        if (d0 && nrf <= 4) {
            if (nrf > 2) cp.wide_ed = 1;
            r.resize(4, Z);
            ed.insert(ed.end(), {bF(e), l, r[0], r[1], bI(diaInv[e]), r[2], r[3], 0});
            continue;
        }
        if (d0) inv_step[diaInv[e]] = 1;
        if (nrf > (size_t)kEntRefs) {
            items.insert(items.end(), {bF(e), (int32_t)refs.size(), (int32_t)(refs.size() + nrf),
                                       elin[e] >= 0 ? elin[e] : 0, elin[e] >= 0 ? elin[e] + 1 : 0, 0, 0, 0});
            refs.insert(refs.end(), r.begin(), r.end());
        } else if (nrf > 2) {
            r.resize(kEntRefs, Z);
            ec.insert(ec.end(), {bF(e), l, r[0], r[1], r[2], r[3], r[4], r[5]});
        } else if (elin[e] >= 0) {
            r.resize(2, Z);
            eb.insert(eb.end(), {bF(e), l, r[0], r[1]});
        } else if (nrf > 0) {
            r.resize(2, Z);
            ea.insert(ea.end(), {bF(e), r[0], r[1], 0});
        } else {
            ez.push_back(bF(e));
        }
    }
    // residual records
    std::vector<int32_t> rr;
    cp.wide_rows = 0;
    for (int32_t k = 0; k < n; k++) {
        std::vector<int32_t> r;
        for (int32_t q = P.rnl_ptr[k]; q < P.rnl_ptr[k + 1]; q++) conv(P.rnl_ref[q], r);
        const int32_t nl = lptr[k + 1] - lptr[k];
        const bool lng = r.size() > (size_t)kRowRefs || nl > kLongRow;
        if (lng) {
            items.insert(items.end(), {bX(k), (int32_t)refs.size(), (int32_t)(refs.size() + r.size()),
                                       lptr[k], lptr[k + 1], k, 1, 0});
            refs.insert(refs.end(), r.begin(), r.end());
            r.assign(1, nl);   // in a long row's record, its linear entries' count
        } else if (r.size() > 2 || nl > 1) {
            cp.wide_rows = 1;
        }
        r.resize(kRowRefs, Z);
        // a row without linear entries reads the zero pair
        rr.insert(rr.end(), {nl > 0 ? lptr[k] : nlin, lng ? 0xFFFF : nl, nl > 0 ? bU(lcolk[lptr[k]]) : Z,
                             r[0], r[1], r[2], r[3], r[4]});
    }

    // one record at least in every class, and items in pairs
    if (ea.empty()) ea = {cp.b_trash, Z, Z, 0};
    if (eb.empty()) eb = {cp.b_trash, ZL, Z, Z};
    if (ed.empty()) ed = {cp.b_trash, ZL, Z, Z, cp.b_trash, Z, Z, 0};
    if (items.size() % 16) items.insert(items.end(), {cp.b_trash, 0, 0, 0, 0, 0, 0, 0});

    // the solve program, level by level
    std::vector<int32_t> steps, rec, upd;
    auto emit = [&](uint32_t kind, std::vector<int32_t>& words) {
        const int32_t cnt = (int32_t)words.size() / 8;
        for (int32_t q = 0; q < cnt; q += 64) {
            steps.push_back((int32_t)rec.size() / 8 + q);
            steps.push_back((std::min(64, cnt - q) - 1) | (int32_t)(kind << 6));
        }
        rec.insert(rec.end(), words.begin(), words.end());
        words.clear();
    };
    // One level: its tasks are independent.  Passes of three products each;
    // within a pass one kind for the products, the narrow one when the whole
    // pass fits it, and scalings alone four to a record.
    auto level = [&](std::vector<Task>& ts) {
        std::vector<int32_t> sc, mul, dia, lm, ld;
        size_t maxp = 0;
        for (Task& t : ts) {
            const size_t np = t.up.size() / 2;
            if (np > (size_t)kLongTask) {
                auto& v = t.dia ? ld : lm;
                v.insert(v.end(), {t.d, t.s, (int32_t)upd.size() / 2, (int32_t)(upd.size() / 2 + np), 0, 0, 0, 0});
                upd.insert(upd.end(), t.up.begin(), t.up.end());
                t.d = -1;
            } else {
                maxp = std::max(maxp, np);
            }
        }
        emit(SP_LMUL, lm);
        emit(SP_LDIA, ld);
        for (size_t p0 = 0; p0 == 0 || p0 < maxp; p0 += 3) {
            size_t most = 0, n_mul = 0;
            for (int pass = 0; pass < 2; pass++)
                for (const Task& t : ts) {
                    const size_t np = t.up.size() / 2;
                    if (t.d < 0 || (p0 > 0 && np <= p0)) continue;
                    const size_t left = np - p0;
                    const bool d = t.dia && left <= 3;
                    if (pass == 0) {
                        if (!d && left > 0) {
                            most = std::max(most, left);
                            n_mul++;
                        }
                        continue;
                    }
                    std::vector<int32_t> w{t.d, left > 3 ? cp.b_one : t.s};
                    for (size_t q = 0; q < 3; q++) {
                        w.push_back(q < left ? t.up[2 * (p0 + q)] : Z);
                        w.push_back(q < left ? t.up[2 * (p0 + q) + 1] : Z);
                    }
                    if (d) {
                        dia.insert(dia.end(), w.begin(), w.end());
                    } else if (left > 0) {
                        mul.insert(mul.end(), w.begin(), w.end());
                    } else if (t.s != cp.b_one) {
                        // few scalings ride along with the products
                        auto& v = n_mul > 0 && n_mul + ts.size() <= 64 ? mul : sc;
                        v.insert(v.end(), w.begin(), w.begin() + (&v == &mul ? 8 : 2));
                    }
                }
            while (sc.size() % 8) sc.insert(sc.end(), {cp.b_trash, cp.b_one});
            emit(SP_DIA3, dia);
            emit(most > 1 ? SP_MUL3 : SP_MUL1, mul);
            emit(SP_SCALE, sc);
        }
        ts.clear();
    };
    // forward substitution levels: y_k for rows with L entries
    int32_t nA = n_lulev;
    std::vector<int32_t> yl(n, -1);
    for (int32_t k = 0; k < n; k++) {
        int32_t mx = -1;
        bool any = false;
        for (int32_t e = P.rowptr[k]; e < P.diag[k]; e++) {
            any = true;
            mx = std::max(mx, std::max(lev[e], yl[P.colperm[e]]));
        }
        if (any) {
            yl[k] = mx + 1;
            nA = std::max(nA, yl[k] + 1);
        }
    }
    // A task of level lf with more products than a record holds: three at a
    // time, in the order their operands are ready, go to earlier levels (one
    // record a level), so that its own level is left with the latest ones.
    // ready[q]: level that forms product q's operands.
    typedef std::vector<std::vector<Task>> Schedule;
    auto place = [&](Schedule& by_level, Task t, const std::vector<int32_t>& ready, int32_t lf) {
        const size_t np = ready.size();
        if (np > 3 && np <= (size_t)kLongTask) {
            std::vector<int32_t> o(np);
            for (size_t q = 0; q < np; q++) o[q] = (int32_t)q;
            std::stable_sort(o.begin(), o.end(), [&](int32_t x, int32_t y) { return ready[x] < ready[y]; });
            size_t q = 0;
            for (int32_t prev = -1; np - q > 3; q += 3) {
                const int32_t l = std::max(prev, ready[o[q + 2]]) + 1;
                if (l >= lf) break;
                Task p{t.d, cp.b_one, false, {}};
                for (size_t z = q; z < q + 3; z++) p.up.insert(p.up.end(), {t.up[2 * o[z]], t.up[2 * o[z] + 1]});
                by_level[l].push_back(std::move(p));
                prev = l;
            }
            std::vector<int32_t> rest;
            for (; q < np; q++) rest.insert(rest.end(), {t.up[2 * o[q]], t.up[2 * o[q] + 1]});
            t.up = rest;
        }
        by_level[lf].push_back(std::move(t));
    };
    std::vector<int32_t> ready;
    Schedule lu(nA);
    for (int32_t l = 0; l < nA; l++) {
        if (l < n_lulev)
            for (int32_t q = P.lu_lptr[l]; q < P.lu_lptr[l + 1]; q++) {
                const LuTask& t = P.lu_task[q];
                // a U entry with no updates keeps its assembled value; a
                // level-0 diagonal was inverted by the assembly
                if (t.piv == -1 && t.ub == t.ue) continue;
                if (t.piv <= -2 && t.ub == t.ue && !inv_step[-2 - t.piv]) continue;
                Task k{bF(t.e), t.piv >= 0 ? bI(t.piv) : t.piv == -1 ? cp.b_one : bI(-2 - t.piv), t.piv <= -2, {}};
                ready.clear();
                for (int32_t u = t.ub; u < t.ue; u++) {
                    const int32_t fa = P.lu_upd[2 * u], fb = P.lu_upd[2 * u + 1];
                    k.up.insert(k.up.end(), {bF(fa), bF(fb)});
                    ready.push_back(std::max(lev[fa], lev[fb]));
                }
                place(lu, std::move(k), ready, l);
            }
        for (int32_t k = 0; k < n; k++) {
            if (yl[k] != l) continue;
            Task t{bX(k), cp.b_one, false, {}};
            ready.clear();
            for (int32_t e = P.rowptr[k]; e < P.diag[k]; e++) {
                t.up.insert(t.up.end(), {bF(e), bX(P.colperm[e])});
                ready.push_back(std::max(lev[e], yl[P.colperm[e]]));
            }
            place(lu, std::move(t), ready, l);
        }
    }
    for (auto& ts : lu) level(ts);
    cp.n_lu = (int32_t)steps.size() / 2;
    // a triangular solve as tasks by level: rows(k) lists (F entry, x index),
    // ascending or descending dependency order
    auto solve = [&](bool ascending, bool scaled, const std::vector<std::vector<std::pair<int32_t, int32_t>>>& rows) {
        std::vector<int32_t> sl(n, -1);
        int32_t nl = 0;
        for (int32_t q = 0; q < n; q++) {
            const int32_t k = ascending ? q : n - 1 - q;
            int32_t mx = -1;
            for (auto& ex : rows[k]) mx = std::max(mx, sl[ex.second]);
            sl[k] = mx + 1;
            nl = std::max(nl, sl[k] + 1);
        }
        Schedule tri(nl);
        for (int32_t k = 0; k < n; k++) {
            if (!scaled && rows[k].empty()) continue;
            Task t{bX(k), scaled ? bI(k) : cp.b_one, false, {}};
            ready.clear();
            for (auto& ex : rows[k]) {
                t.up.insert(t.up.end(), {bF(ex.first), bX(ex.second)});
                ready.push_back(sl[ex.second]);
            }
            place(tri, std::move(t), ready, sl[k]);
        }
        for (auto& ts : tri) level(ts);
    };
    std::vector<std::vector<std::pair<int32_t, int32_t>>> urow(n), ucol(n), lcolv(n);   // (F entry, x index)
    for (int32_t i = 0; i < n; i++)
        for (int32_t e = P.rowptr[i]; e < P.rowptr[i + 1]; e++) {
            const int32_t j = P.colperm[e];
            if (j > i) {
                urow[i].push_back({e, j});
                ucol[j].push_back({e, i});
            } else if (j < i) {
                lcolv[j].push_back({e, i});
            }
        }
    solve(false, true, urow);
    cp.n_steps = (int32_t)steps.size() / 2;
    steps.insert(steps.end(), {0, 0});   // read ahead, never run
    if (rec.empty()) rec.assign(8, Z);
    const std::vector<int32_t> steps_tran = steps, rec_tran = rec, upd_tran = upd;
    // transposed solves (adjoint): U^T z = b over U's columns, ascending
    // (scaled by 1/U_kk), then L^T w = z over L's columns, descending
    steps.clear();
    solve(true, true, ucol);
    solve(false, false, lcolv);
    const int32_t n_tsteps = (int32_t)steps.size() / 2;
    steps.insert(steps.end(), {0, 0});
    const std::vector<int32_t> tsteps = steps;
    // linear entries by column
    std::vector<int32_t> cdesc(2 * (size_t)n), lcl, lrow;
    {
        std::vector<std::vector<std::pair<int32_t, int32_t>>> bycol(n);   // (lin index, row)
        for (int32_t k = 0; k < n; k++)
            for (int32_t l = lptr[k]; l < lptr[k + 1]; l++) bycol[lcolk[l]].push_back({l, k});
        for (int32_t j = 0; j < n; j++) {
            cdesc[2 * j] = (int32_t)lcl.size();
            for (auto& lr : bycol[j]) {
                lcl.push_back(lr.first);
                lrow.push_back(lr.second);
            }
            cdesc[2 * j + 1] = (int32_t)lcl.size();
        }
    }

    std::vector<int32_t> src, lcol;
    int32_t wo = 0;
    for (int32_t s = 0; s < ns; s++) {
        src.insert(src.end(), {P.src[s].kind, cp.b_wd + 8 * wo, P.src[s].len, cp.b_st + 8 * (3 * nm + s)});
        wo += P.src[s].len + 1;
    }
    for (int32_t l = 0; l < nlin; l++) lcol.push_back(bU(lcolk[l]));
    lcol.push_back(Z);
    // record and update offsets of a step are relative to o_rec and o_upd, and
    // the adjoint's records continue the transient's: its part of the image
    // repeats nothing, so rec and upd come last and grow into it
    Blob b;
    cp.o_ea = b.add(ea, 8);
    cp.o_eb = b.add(eb, 4);
    cp.o_ec = b.add(ec, 8);
    cp.o_ed = b.add(ed, 8);
    cp.o_rr = b.add(rr, 8);
    cp.o_items = b.add(items, 8);
    cp.o_src = b.add(src, 4);
    cp.o_steps = b.add(steps_tran, 2);
    cp.o_ez = b.add(ez);
    cp.o_lcol = b.add(lcol);
    cp.o_refs = b.add(refs);
    cp.o_upd = b.add(upd_tran, 2);
    cp.o_rec = b.add(rec_tran, 8);
    b.align(8);
    cp.words = (int32_t)b.w.size();
    // adjoint part; its long tasks' pairs are numbered from o_upd, its records from o_rec
    {
        const std::vector<int32_t> rest(rec.begin() + rec_tran.size(), rec.end());
        const std::vector<int32_t> urest(upd.begin() + upd_tran.size(), upd.end());
        const int32_t o2 = b.add(rest, 8), u2 = b.add(urest, 2);
        const int32_t drec = (o2 - cp.o_rec - (int32_t)rec_tran.size()) / 8;
        const int32_t dupd = (u2 - cp.o_upd - (int32_t)upd_tran.size()) / 2;
        std::vector<int32_t> t2 = tsteps;
        for (size_t q = 0; q + 2 < t2.size(); q += 2) {   // all but the read-ahead one
            const uint32_t kind = (uint32_t)t2[q + 1] >> 6;
            t2[q] += drec;
            if (kind == SP_LMUL || kind == SP_LDIA)
                for (int32_t m = 0; m <= (t2[q + 1] & 63); m++) {
                    const size_t at = (size_t)cp.o_rec + 8 * ((size_t)t2[q] + m);
                    for (int z = 2; z < 4; z++) {
                        const int32_t v = b.w[at + z] + dupd;
                        if (v > 0xFFFF) b.ok = false;
                        b.w[at + z] = (uint16_t)v;
                    }
                }
        }
        cp.o_tsteps = b.add(t2, 2);
    }
    cp.o_cdesc = b.add(cdesc, 2);
    cp.o_lcl = b.add(lcl);
    cp.o_lrow = b.add(lrow);
    b.align(8);
    cp.words_adj = (int32_t)b.w.size();
    if (fits && !b.ok) {
        *why = "plan index does not fit 16 bits";
        return false;
    }
    blob = std::move(b.w);
    cp.n = n;
    cp.nnz = nnz;
    cp.n_mos = nm;
    cp.n_src = ns;
    cp.nlin = nlin;
    cp.stamp_n = 3 * nm + ns;
    cp.nwd = nwd;
    cp.n_ea = (int32_t)ea.size() / 4;
    cp.n_eb = (int32_t)eb.size() / 4;
    cp.n_ec = (int32_t)ec.size() / 8;
    cp.n_ed = (int32_t)ed.size() / 8;
    cp.n_ez = (int32_t)ez.size();
    cp.n_items = (int32_t)items.size() / 8;
    cp.n_tsteps = n_tsteps;

    // pivot-order side arrays
    colnat.assign(n, 0);
    diffrow.assign(n, 0);
    probe.assign(n, -1);
    for (int32_t r = 0; r < n; r++) colnat[P.pcol[r]] = r;
    for (int32_t k = 0; k < n; k++) {
        diffrow[k] = P.is_diff[P.rownat[k]];
        probe[k] = P.probe_slot[colnat[k]];
    }
    dev.assign(4 * (size_t)nm, 0);
    for (int32_t m = 0; m < nm; m++) {
        for (int q = 0; q < 3; q++) {
            const int32_t v = P.mos[4 * m + q];
            dev[4 * m + q] = v >= 0 ? bU(P.pcol[v]) : Z;
        }
        dev[4 * m + 3] = P.mos[4 * m + 3];
    }
    devrow.assign(2 * (size_t)nm, 0);
    for (int32_t m = 0; m < nm; m++) {
        const int32_t d = P.mos[4 * m], s = P.mos[4 * m + 2];
        devrow[2 * m] = d >= 0 ? P.prow[d] : (int32_t)CP_GROUND;
        devrow[2 * m + 1] = s >= 0 ? P.prow[s] : (int32_t)CP_GROUND;
    }
    return true;
}

std::vector<std::vector<PackSeg>> pack_chunks(const std::vector<int32_t>& cs, const std::vector<size_t>& img,
                                              const std::vector<size_t>& dblb, std::vector<size_t> rem,
                                              int waves, int segs, size_t cap, size_t* need) {
    std::vector<std::vector<PackSeg>> chunks;
    *need = 0;
    for (int32_t c : cs)
        if (rem[c] && img[c] + dblb[c] > cap) return chunks;
    for (size_t hi = 0, lo = cs.size();;) {
        while (hi < cs.size() && rem[cs[hi]] == 0) hi++;
        if (hi == cs.size()) break;
        while (lo > hi + 1 && rem[cs[lo - 1]] == 0) lo--;   // the smallest circuits left end at lo
        const int32_t L = cs[hi];
        const size_t kfit = std::min<size_t>({rem[L], (size_t)waves, (cap - img[L]) / dblb[L]});
        std::vector<PackSeg> best;
        int best_w = -1;
        size_t best_b = 0;
        for (size_t k = kfit; k >= 1; k--) {
            std::vector<PackSeg> sg{{L, (int32_t)k}};
            size_t bytes = img[L] + k * dblb[L];
            int w = (int)k;
            for (size_t q = lo; q-- > hi + 1 && w < waves && (int)sg.size() < segs;) {
                const int32_t c = cs[q];
                if (rem[c] == 0 || bytes + img[c] + dblb[c] > cap) continue;
                const size_t t = std::min<size_t>({rem[c], (size_t)(waves - w), (cap - bytes - img[c]) / dblb[c]});
                sg.push_back({c, (int32_t)t});
                bytes += img[c] + t * dblb[c];
                w += (int)t;
            }
            if (w > best_w) { best = sg; best_w = w; best_b = bytes; }
            if (w == waves) break;
        }
        for (const PackSeg& g : best) rem[g.c] -= g.cnt;
        *need = std::max(*need, best_b);
        chunks.push_back(best);
    }
    return chunks;
}

}  // namespace cedar
