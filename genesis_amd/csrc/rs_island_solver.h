// Constraint rows and Newton / conjugate-gradient solve of one environment on one wavefront, for models with 25 to 128
// dofs whose constraint rows are short and that have no collision pairs (the rule is takes_islands in rs_lib.hip;
// constraint/solver.py: rows :580-1286, solve :2936-3261, line search :2034-2597).
//
// A constraint row touches the dofs above the (at most) two links it acts on: 12 of the 120 dofs of a pile of 20 free
// boxes. So a row is kept as its W = FusedArgs::row_width first entries, the dofs' columns in ascending order (columns
// that do not exist hold 0), with one column list per group of rows (the four rows of a contact, or a single equality,
// friction-loss or limit row). Entities joined by rows form islands; the Hessian M + J^T D J has no entry between two
// islands, so every island's block is stored alone (a packed lower triangle) and all islands are assembled, factored
// and solved side by side: lane l owns dofs l and l + 64 and follows the pivots of its own island, so the number of
// steps is the size of the largest island. Leaving out zero terms changes no sum: rows, Hessian entries, factor and
// forward substitution are summed in the reference's order; the cost and line-search sums run across the lanes and the
// backward substitution takes its columns last to first. The factor is formed anew in every Newton iteration (the
// reference updates it row by row, solver.py:1782-1822: the same matrix up to rounding).
//
// Measured while it still took models with contacts, against dense 120-column rows and rank-1 updates through memory:
// pile of 20 boxes x1024, the first four steps from a reset (320 rows, 5 Newton iterations), 6.0 -> 0.94 ms per step. Of
// the old step's 9.4 M cycles per environment 4.3 M were the rank-1 updates, 1.0 M each the Hessian and the line
// searches, 0.8 M the triangular solves, 0.6 M each the row builder and the updates of the row forces. The dense solver
// as it is now takes 2.8 ms per step.
#pragma once
#include "rs_constraint.h"
#include "rs_gjk.h"
#include "rs_wave.h"
#include "rs_wave_dyn.h"
#include "rs_wave_solver.h"

namespace rs {

#define LF(field, row) FP(loc, field)[(row)]

// The row groups of one environment (all in its slice of the work field): g < n1 a single equality or friction-loss row,
// then one group per contact, then single limit rows.
struct RowGroups {
    float* J;         // [c * W + p]: entry of row c in its group's p-th column
    uint8_t* idx;     // [g * W + p]: the p-th column of group g (a dof, later its position), n_dofs where there is none
    uint32_t* mask;   // [4 g + k]: the dofs of group g, 32 per word
    int* ent;         // [g]: first dofs of the entities it joins, a | b << 8 (255: none)
    int* list;        // [k * D + d]: the k-th group that touches dof d, g << 5 | p
    float* dense;     // dense rows of the equality / friction-loss rows or of the limit rows while they are built
    int W, n1, ncont;
    __device__ __forceinline__ int row0(int g) const {
        return g < n1 ? g : g < n1 + ncont ? n1 + 4 * (g - n1) : g + 3 * ncont;
    }
    __device__ __forceinline__ bool four(int g) const { return g >= n1 && g < n1 + ncont; }
    __device__ __forceinline__ int group(int c) const {
        return c < n1 ? c : c < n1 + 4 * ncont ? n1 + ((c - n1) >> 2) : c - 3 * ncont;
    }
};

__device__ __forceinline__ RowGroups row_groups(const DModel& m, float* wk, const FusedArgs& fa) {
    const int W = fa.row_width;
    float* p = wk + fa.off_jac;
    RowGroups g;
    g.W = W;
    g.n1 = g.ncont = 0;
    g.J = p;
    p += (size_t)m.CMAX * W;
    const size_t G = row_group_max(m.NE, m.D, m.KMAX);
    g.idx = (uint8_t*)p;
    p += G * W / 4;
    g.mask = (uint32_t*)p;
    p += 4 * G;
    g.ent = (int*)p;
    p += G;
    g.list = (int*)p;
    p += G * m.D;
    g.dense = p;
    return g;
}

// rows base, base + 1, ... of the row builders, dense, one after the other; the other row arrays are the environment's
struct DenseRows {
    float* J;
    const WorkRows& R;
    int base, D;
    __device__ __forceinline__ float& jac(int c, int d) const { return J[(size_t)(c - base) * D + d]; }
    __device__ __forceinline__ float& diag(int c) const { return R.diag(c); }
    __device__ __forceinline__ float& aref(int c) const { return R.aref(c); }
    __device__ __forceinline__ float& efc_D(int c) const { return R.efc_D(c); }
    __device__ __forceinline__ float& fl(int c) const { return R.fl(c); }
};

// entities joined by a group whose dofs are (lo, hi): those of its first and of its last dof
__device__ __forceinline__ int group_entities(const DModel& m, uint64_t lo, uint64_t hi) {
    if (!(lo | hi)) return 0xffff;
    const int first = lo ? __builtin_ctzll(lo) : kWave + __builtin_ctzll(hi);
    const int last = hi ? 2 * kWave - 1 - __builtin_clzll(hi) : kWave - 1 - __builtin_clzll(lo);
    return m.entity_dof_start[m.dof_entity[first]] | m.entity_dof_start[m.dof_entity[last]] << 8;
}

// rows c0 .. c1 - 1 (single-row groups from g0 on) from the dense rows to their groups
__device__ inline void compact_rows(const DModel& m, const WorkRows& R, const RowGroups& Q, const DenseRows& dr, int c0,
                                    int c1, int g0, int lane) {
    const int D = m.D, W = Q.W;
    for (int c = c0; c < c1; c++) {
        const int g = g0 + c - c0;
        const float v0 = lane < D ? dr.jac(c, lane) : 0.f;
        const float v1 = lane + kWave < D ? dr.jac(c, lane + kWave) : 0.f;
        const uint64_t lo = wave_ballot(v0 != 0.f), hi = wave_ballot(v1 != 0.f);
        const uint64_t below = (1ull << lane) - 1;
        const int n0 = __popcll(lo), n = n0 + __popcll(hi);
        const int p0 = __popcll(lo & below), p1 = n0 + __popcll(hi & below);
        if (v0 != 0.f && p0 < W) {
            Q.J[(size_t)c * W + p0] = v0;
            Q.idx[(size_t)g * W + p0] = (uint8_t)lane;
        }
        if (v1 != 0.f && p1 < W) {
            Q.J[(size_t)c * W + p1] = v1;
            Q.idx[(size_t)g * W + p1] = (uint8_t)(lane + kWave);
        }
        if (lane >= n && lane < W) {
            Q.J[(size_t)c * W + lane] = 0.f;
            Q.idx[(size_t)g * W + lane] = (uint8_t)D;
        }
        if (lane < 4) Q.mask[4 * (size_t)g + lane] = (uint32_t)((lane < 2 ? lo : hi) >> (32 * (lane & 1)));
        if (lane == 0) Q.ent[g] = group_entities(m, lo, hi);
    }
}

// a staged row written as its group's columns
struct GroupJac : ChainJac {
    const DModel& m;
    const RowGroups& Q;
    __device__ __forceinline__ GroupJac(float* col, const uint32_t* chains, const DModel& model, const RowGroups& groups)
        : ChainJac{col, chains, groups.W, 0, 0, 0, 0}, m(model), Q(groups) {}
    template <class R>
    __device__ __forceinline__ void flush(const R&, int c, int D) const {
        for (int p = 0; p < Q.W; p += 4)
            *(float4*)(Q.J + (size_t)c * Q.W + p) = make_float4(col[p * kTileStride], col[(p + 1) * kTileStride],
                                                                col[(p + 2) * kTileStride], col[(p + 3) * kTileStride]);
        const int g = Q.group(c);
        if (((c - Q.n1) & 3) != 0) return;  // the first of the contact's four rows writes what they share
        uint64_t l = lo(), h = hi();
        *(uint4*)(Q.mask + 4 * (size_t)g) = make_uint4(m0, m1, m2, m3);
        Q.ent[g] = group_entities(m, l, h);
        for (int p = 0; p < Q.W; p++) {
            int d = D;
            if (l) {
                d = __builtin_ctzll(l);
                l &= l - 1;
            } else if (h) {
                d = kWave + __builtin_ctzll(h);
                h &= h - 1;
            }
            Q.idx[(size_t)g * Q.W + p] = (uint8_t)d;
        }
    }
};

// solver.py:580-1286: equality, friction-loss and limit rows uniformly (few rows), contact rows one lane per row.
// tile: max(W, kTileMinRows) tile rows, then 4 words per link.
__device__ __forceinline__ void island_constraints(const DModel& m, const LState& loc, const DState& st, int b,
                                          const WorkRows& R, RowGroups& Q, int lane, float* tile) {
    const int D = m.D;
    const DenseRows dr{Q.dense, R, 0, D};
    int nc = equality_rows(m, loc, 0, dr);
    const int neq = nc;
    const int nfl = frictionloss_rows(m, loc, 0, dr, nc);
    nc += nfl;
    wave_sync();
    if (nc > 0) compact_rows(m, R, Q, dr, 0, nc, 0, lane);
    Q.n1 = nc;
    Q.ncont = m.enable_collision ? LF(n_contacts, 0) : 0;
    if (Q.ncont > 0) {
        uint32_t* chains = (uint32_t*)(tile + island_tile_rows(Q.W) * kTileStride);
        link_chains(m, chains, lane);
        const GroupJac gj(tile + lane, chains, m, Q);
        for (int r = lane; r < 4 * Q.ncont; r += kWave)
            contact_row(m, loc, 0, st, b, R, r >> 2, r & 3, nc, gj);
        nc += 4 * Q.ncont;
    }
    if (m.enable_joint_limit) {
        const DenseRows dl{Q.dense, R, nc, D};
        wave_sync();  // the dense rows above have been read
        const int c1 = limit_rows(m, loc, 0, dl, nc);
        wave_sync();
        if (c1 > nc) compact_rows(m, R, Q, dl, nc, c1, Q.n1 + Q.ncont, lane);
        nc = c1;
    }
    LF(n_con, 0) = nc;
    LF(n_con_eq, 0) = neq;
    LF(n_con_fl, 0) = nfl;
    wave_sync();
}

// the packed triangles in the private region's nt_H, whose D * D words hold them from the first 16-byte boundary on (the
// region itself starts on one)
__device__ __forceinline__ float* triangles_in_record(const LState& loc) {
    return loc.base + (loc.off[FID_nt_H] + 3) / 4 * 4;
}

// What a lane knows of its dofs lane and lane + 64 (h = 0, 1).
struct IslandDofs {
    bool own[2];
    int e0[2], e1[2];  // dofs of its entity
    int li[2], n[2];   // index in its island, size of the island
    int pos[2];        // position: islands one after the other
    int cb[2], hb[2];  // offset of the island's packed triangle, and of the dof's row in it
    int cnt[2];        // groups that touch the dof
    int steps;         // size of the largest island (uniform)
};

// Islands: every group joins its entities; labels (the smallest first dof of an entity reached) spread over the groups
// until none changes. lds: island_words(D) words.
__device__ __forceinline__ void find_islands(const DModel& m, const RowGroups& Q, int n_groups, int lane, int* lds,
                                    IslandDofs& I) {
    const int D = m.D;
    int* lab = lds;
    uint32_t* cm = (uint32_t*)(lds + 2 * kWave);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + h * kWave;
        I.own[h] = d < D;
        I.e0[h] = I.e1[h] = I.cnt[h] = 0;
        if (I.own[h]) {
            const int e = m.dof_entity[d];
            I.e0[h] = m.entity_dof_start[e];
            I.e1[h] = m.entity_dof_end[e];
            lab[d] = I.e0[h];
#pragma unroll
            for (int k = 0; k < 4; k++) cm[4 * d + k] = 0;
        }
    }
    // the groups of each dof, in group order: 64 groups at a time, one per lane, their masks read lane by lane
    const int wi = lane >> 5;
    for (int g0 = 0; g0 < n_groups; g0 += kWave) {
        const uint4 mk = g0 + lane < n_groups ? ((const uint4*)Q.mask)[g0 + lane] : make_uint4(0, 0, 0, 0);
        const int n = min(kWave, n_groups - g0);
        for (int j = 0; j < n; j++) {
            const uint32_t a0 = __builtin_amdgcn_readlane(mk.x, j), a1 = __builtin_amdgcn_readlane(mk.y, j);
            const uint32_t a2 = __builtin_amdgcn_readlane(mk.z, j), a3 = __builtin_amdgcn_readlane(mk.w, j);
            const uint32_t bit = 1u << (lane & 31), below = bit - 1;
            const uint32_t x0 = wi ? a1 : a0, x1 = wi ? a3 : a2;
            if (x0 & bit) {
                const int p = __popc(x0 & below) + (wi ? __popc(a0) : 0);
                Q.list[(size_t)I.cnt[0] * D + lane] = (g0 + j) << 5 | p;
                I.cnt[0]++;
            }
            if (x1 & bit) {
                const int p = __popc(x1 & below) + __popc(a0) + __popc(a1) + (wi ? __popc(a2) : 0);
                Q.list[(size_t)I.cnt[1] * D + lane + kWave] = (g0 + j) << 5 | p;
                I.cnt[1]++;
            }
        }
    }
    wave_sync();
    bool changed;
    do {  // every pass that goes on has lowered a label, so the loop ends
        changed = false;
        for (int g = lane; g < n_groups; g += kWave) {
            const int e = Q.ent[g], a = e & 0xff, c = (e >> 8) & 0xff;
            if (a == c || a == 0xff || c == 0xff) continue;
            const int la = lab[a], lc = lab[c], lo = min(la, lc), up = max(la, lc);
            if (lo == up) continue;
            atomicMin(&lab[a], lo);
            atomicMin(&lab[c], lo);
            atomicMin(&lab[up], lo);
            changed = true;
        }
        wave_sync();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int d = lane + h * kWave;
            if (I.own[h] && d == I.e0[h]) {
                const int l = lab[d], ll = lab[l];
                if (ll < l) {
                    lab[d] = ll;
                    changed = true;
                }
            }
        }
        wave_sync();
    } while (wave_ballot(changed) != 0);
    int root[2] = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + h * kWave;
        if (I.own[h]) {
            root[h] = lab[I.e0[h]];
            atomicOr(&cm[4 * root[h] + (d >> 5)], 1u << (d & 31));
        }
    }
    wave_sync();
    int sizes[2] = {0, 0}, words[2] = {0, 0};
    int big = 0;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + h * kWave;
        I.li[h] = I.n[h] = 0;
        if (I.own[h]) {
            int n = 0, li = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t w = cm[4 * root[h] + k];
                n += __popc(w);
                li += 32 * k + 32 <= d ? __popc(w) : 32 * k <= d ? __popc(w & ((1u << (d & 31)) - 1)) : 0;
            }
            I.li[h] = li;
            I.n[h] = n;
            if (d == root[h]) {
                sizes[h] = n;
                words[h] = tri4(n);
            }
            big = max(big, n);
        }
    }
    wave_sync();
    int t0, t1, w0, w1;
    const int s0 = wave_excl_scan(sizes[0], lane, t0), s1 = wave_excl_scan(sizes[1], lane, t1) + t0;
    const int o0 = wave_excl_scan(words[0], lane, w0), o1 = wave_excl_scan(words[1], lane, w1) + w0;
    int* at = (int*)cm;  // an island's first position and first word, at its root
    if (I.own[0] && lane == root[0]) {
        at[4 * lane] = s0;
        at[4 * lane + 1] = o0;
    }
    if (I.own[1] && lane + kWave == root[1]) {
        at[4 * (lane + kWave)] = s1;
        at[4 * (lane + kWave) + 1] = o1;
    }
    wave_sync();
#pragma unroll
    for (int h = 0; h < 2; h++) {
        I.pos[h] = I.cb[h] = I.hb[h] = 0;
        if (I.own[h]) {
            I.pos[h] = at[4 * root[h]] + I.li[h];
            I.cb[h] = at[4 * root[h] + 1];
            I.hb[h] = I.cb[h] + tri4(I.li[h]);
        }
    }
    I.steps = (int)wave_max_f((float)big);
    wave_sync();
    // the groups' columns become positions (position n_dofs holds 0 in every gathered vector)
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (I.own[h]) lab[lane + h * kWave] = I.pos[h];
    wave_sync();
    for (int t = lane; t < n_groups * (Q.W / 4); t += kWave) {
        uint32_t w = ((uint32_t*)Q.idx)[t], r = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int d = (w >> (8 * u)) & 0xff;
            r |= (uint32_t)(d < D ? lab[d] : D) << (8 * u);
        }
        ((uint32_t*)Q.idx)[t] = r;
    }
    wave_sync();
}

// The solver's state on a lane: its dofs' vectors, and the sums of the line search. Rows of up to 4 kQ entries. One
// wavefront per SIMD is all a batch of 1024 gives, so nothing hides a load but other loads: the loops below load what
// they need for both of a lane's dofs, for several rows, or one step ahead, before they use any of it (Hessian 120 k ->
// 81 k cycles a call, factor 36 k -> 35 k, line search 29 k -> 21 k, row builder 250 k -> 113 k on 1024 box piles).
template <bool kHLds, int kQ>
struct IslandSolver {
    const DModel& m;
    const LState& loc;
    const WorkRows& R;
    const RowGroups& Q;
    const IslandDofs& I;
    float* H;  // the islands' packed triangles, first the Hessian, then its factor
    float* xv; // vector in position order: D + 1 words, xv[D] = 0
    int lane, nc, ne, nef;
    static constexpr int kRows = kQ <= 3 ? 5 : 1;     // rows of a lane taken together
    static constexpr int kQuads = kQ <= 3 ? kQ : 1;   // quads of a row taken together
    float qacc[2], Ma[2], force[2], acc0[2], qfc[2], grad[2], Mgrad[2], search[2], mv[2];
    float gauss, qg[3], es[3];

    // xv[pos] = v, for all dofs
    __device__ __forceinline__ void put(const float (&v)[2]) const {
        wave_sync();
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (I.own[h]) xv[I.pos[h]] = v[h];
        wave_sync();
    }
    // M x of this lane's dofs, x in xv (an entity's dofs have consecutive positions)
    __device__ __forceinline__ void mass_mul(float (&out)[2]) const {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            out[h] = 0.f;
            if (!I.own[h]) continue;
            const int d = lane + h * kWave;
            const float* row = FP(loc, mass_mat) + (size_t)d * m.D;
            const float* x = xv + I.pos[h] - d;
            out[h] = seq_sum<6>(0.f, I.e0[h], I.e1[h], [&](int j) { return row[j] * x[j]; });
        }
    }
    // out[u] = init[u] + J x for rows c0 + lane + 64 u (the last row again past the end), in column order, x in xv
    template <int U>
    __device__ __forceinline__ void row_dots(int c0, float (&out)[U]) const {
        const int W = Q.W;
        for (int q0 = 0; 4 * q0 < W; q0 += kQuads) {
            float4 v[U][kQuads];
            uint32_t k[U][kQuads];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = min(c0 + u * kWave + lane, nc - 1);
                const float4* j = (const float4*)(Q.J + (size_t)c * W) + q0;
                const uint32_t* ix = (const uint32_t*)(Q.idx + (size_t)Q.group(c) * W) + q0;
#pragma unroll
                for (int q = 0; q < kQuads; q++) {  // past the row's last quad: that quad again, left out below
                    const int qq = min(q, W / 4 - 1 - q0);
                    v[u][q] = j[qq];
                    k[u][q] = ix[qq];
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int q = 0; q < kQuads; q++)
                    if (4 * (q0 + q) < W) {
                        out[u] = out[u] + v[u][q].x * xv[k[u][q] & 0xff];
                        out[u] = out[u] + v[u][q].y * xv[(k[u][q] >> 8) & 0xff];
                        out[u] = out[u] + v[u][q].z * xv[(k[u][q] >> 16) & 0xff];
                        out[u] = out[u] + v[u][q].w * xv[k[u][q] >> 24];
                    }
        }
    }
    // Jaref = J qacc - aref, qacc in xv
    __device__ __forceinline__ void init_rows() const {
        for (int c0 = 0; c0 < nc; c0 += kRows * kWave) {
            float s[kRows];
#pragma unroll
            for (int u = 0; u < kRows; u++) s[u] = -R.aref(min(c0 + u * kWave + lane, nc - 1));
            row_dots(c0, s);
#pragma unroll
            for (int u = 0; u < kRows; u++)
                if (c0 + u * kWave + lane < nc) R.Jaref(c0 + u * kWave + lane) = s[u];
        }
        wave_sync();
    }
    // the k-th group of this lane's dof h; any valid entry (the environment's first group) when there is none
    __device__ __forceinline__ int entry(int h, int k) const {
        return k < I.cnt[h] ? Q.list[(size_t)k * m.D + lane + h * kWave] : 0;
    }
    __device__ __forceinline__ float dof_sum(float a, float b) const {
        return wave_sum_f((I.own[0] ? a : 0.f) + (I.own[1] ? b : 0.f));
    }

    // solver.py:2620-2694 after a step of alpha along jv (first: none): Jaref, active flags, row forces, J^T force, cost
    __device__ __forceinline__ float update(bool first, float alpha) {
        float pf = 0.f, pq = 0.f;
        constexpr int U = 4;
        for (int c0 = 0; c0 < nc; c0 += U * kWave) {
            float ja[U], jv[U], Dc[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = min(c0 + u * kWave + lane, nc - 1);
                ja[u] = R.Jaref(c);
                jv[u] = first ? 0.f : R.jv(c);
                Dc[u] = R.efc_D(c);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + u * kWave + lane;
                if (c >= nc) continue;
                const float x = first ? ja[u] : ja[u] + jv[u] * alpha;
                int act = 1;
                float ff = 0.f, fc = 0.f;
                if (ne <= c && c < nef) {
                    const float f = R.fl(c), rf = R.diag(c) * f;
                    const bool ln = x <= -rf, lp = x >= rf;
                    act = !(ln || lp);
                    ff = (float)ln * f + (float)lp * -f;
                    fc = (float)ln * f * (-0.5f * rf - x);
                    fc = fc + (float)lp * f * (-0.5f * rf + x);
                } else if (nef <= c) {
                    act = x < 0.f;
                }
                R.Jaref(c) = x;
                R.active(c) = act;
                R.force(c) = ff + (-x * Dc[u] * (float)act);
                pf = pf + fc;
                pq = pq + 0.5f * (x * x * Dc[u] * (float)act);
            }
        }
        wave_sync();
        qfc[0] = qfc[1] = 0.f;
        const int most = max(I.cnt[0], I.cnt[1]);
        int e[2] = {entry(0, 0), entry(1, 0)};
        for (int k = 0; k < most; k++) {
            float v[2][4], f[2][4];
            const int en[2] = {entry(0, k + 1), entry(1, k + 1)};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int g = e[h] >> 5, c = Q.row0(g), last = Q.four(g) ? 3 : 0;
                const float* j = Q.J + (size_t)c * Q.W + (e[h] & 31);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    v[h][r] = j[min(r, last) * Q.W];
                    f[h][r] = R.force(c + min(r, last));
                }
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const bool four = Q.four(e[h] >> 5);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (k < I.cnt[h] && (r == 0 || four)) qfc[h] = qfc[h] + v[h][r] * f[h][r];
                e[h] = en[h];
            }
        }
        float cost = wave_sum_f(pf);
        gauss = dof_sum(0.5f * (Ma[0] - force[0]) * (qacc[0] - acc0[0]), 0.5f * (Ma[1] - force[1]) * (qacc[1] - acc0[1]));
        return cost + gauss + wave_sum_f(pq);
    }

    // solver.py:1395-1452: the lower triangle's row of each of this lane's dofs, its groups in order
    __device__ __forceinline__ void hessian() const {
        const float eps = m.eps;
        const int W = Q.W;
        wave_sync();
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (I.own[h])
                for (int j = 0; j <= I.li[h]; j += 4) *(float4*)(H + I.hb[h] + j) = make_float4(0.f, 0.f, 0.f, 0.f);
        const int most = max(I.cnt[0], I.cnt[1]);
        int e[2] = {entry(0, 0), entry(1, 0)};
        for (int k = 0; k < most; k++) {
            float ji[2][4], Dc[2][4];
            int act[2][4];
            const int en[2] = {entry(0, k + 1), entry(1, k + 1)};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int g = e[h] >> 5, p = e[h] & 31, c = Q.row0(g), last = Q.four(g) ? 3 : 0;
                const float* J = Q.J + (size_t)c * W;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int rr = min(r, last);
                    ji[h][r] = J[rr * W + p];
                    Dc[h][r] = R.efc_D(c + rr);
                    act[h][r] = R.active(c + rr);
                }
            }
            // kQuads columns' quads at a time
            for (int q0 = 0; 4 * q0 < W; q0 += kQuads) {
                uint32_t ix[2][kQuads];
                float4 v[2][kQuads][4];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int g = e[h] >> 5, c = Q.row0(g), last = Q.four(g) ? 3 : 0;
                    const float* J = Q.J + (size_t)c * W + 4 * q0;
                    const uint8_t* id = Q.idx + (size_t)g * W + 4 * q0;
#pragma unroll
                    for (int q = 0; q < kQuads; q++) {  // past the row's last quad: that quad again, never used
                        const int qq = 4 * min(q, W / 4 - 1 - q0);
                        ix[h][q] = *(const uint32_t*)(id + qq);
#pragma unroll
                        for (int r = 0; r < 4; r++) v[h][q][r] = *(const float4*)(J + min(r, last) * W + qq);
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int p = e[h] & 31;
                    if (k >= I.cnt[h] || 4 * q0 > p) continue;
                    const bool four = Q.four(e[h] >> 5);
                    float* row = H + I.hb[h];
                    float* at = row + I.li[h] - I.pos[h];  // the island's position 0 in this row
#pragma unroll
                    for (int q = 0; q < kQuads; q++) {
                        const int n = p - 4 * (q0 + q);  // columns 0 .. n of the quad are at or left of the dof
                        if (n < 0) continue;
                        float* s[4];
                        float x[4];
#pragma unroll
                        for (int u = 0; u < 4; u++) {
                            s[u] = u <= n ? at + ((ix[h][q] >> (8 * u)) & 0xff) : row;
                            x[u] = *s[u];
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++) {
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                const float4 w = v[h][q][r];
                                const float jj = u == 0 ? w.x : u == 1 ? w.y : u == 2 ? w.z : w.w;
                                const float t = jj * ji[h][r] * Dc[h][r] * (float)act[h][r];
                                if (fabsf(ji[h][r]) > eps && (r == 0 || four)) x[u] = x[u] + t;
                            }
                        }
#pragma unroll
                        for (int u = 0; u < 4; u++)
                            if (u <= n) *s[u] = x[u];
                    }
                }
            }
            e[0] = en[0];
            e[1] = en[1];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (!I.own[h]) continue;
            const int d = lane + h * kWave;
            const float* mass = FP(loc, mass_mat) + (size_t)d * m.D;
            float* row = H + I.hb[h] + I.li[h] - d;
            int j = I.e0[h];
            for (; j + 3 <= d + 1; j += 3) {
                const float a = mass[j], b = mass[j + 1], c = mass[j + 2];
                row[j] = row[j] + a;
                row[j + 1] = row[j + 1] + b;
                row[j + 2] = row[j + 2] + c;
            }
            for (; j <= d; j++) row[j] = row[j] + mass[j];
        }
        wave_sync();
    }

    // solver.py:1595-1621 func_cholesky_factor_direct_batch for all islands at once: in step t every lane below or at
    // pivot t of its island forms the pivot and its own entry (the sums over k in order)
    __device__ __forceinline__ void factor() const {
        for (int t = 0; t < I.steps; t++) {
            const bool on[2] = {I.own[0] && I.li[0] >= t, I.own[1] && I.li[1] >= t};
            float val[2] = {0.f, 0.f};
            if (on[0] || on[1]) {
                const float *Lk[2], *Lr[2];
                float s[2], hr[2], dt[2] = {0.f, 0.f};
#pragma unroll
                for (int h = 0; h < 2; h++) {  // a dof with nothing to do repeats the lane's other one
                    const int g = on[h] ? h : 1 - h;
                    Lk[h] = H + (g ? I.cb[1] : I.cb[0]) + tri4(t);
                    Lr[h] = H + (g ? I.hb[1] : I.hb[0]);
                    s[h] = Lk[h][t];
                    hr[h] = Lr[h][t];
                }
                int j = 0;
                for (; j + 4 <= t; j += 4) {
                    float4 a[2], c[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        a[h] = *(const float4*)(Lk[h] + j);
                        c[h] = *(const float4*)(Lr[h] + j);
                    }
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        s[h] = s[h] - a[h].x * a[h].x;
                        s[h] = s[h] - a[h].y * a[h].y;
                        s[h] = s[h] - a[h].z * a[h].z;
                        s[h] = s[h] - a[h].w * a[h].w;
                        dt[h] = dt[h] + c[h].x * a[h].x;
                        dt[h] = dt[h] + c[h].y * a[h].y;
                        dt[h] = dt[h] + c[h].z * a[h].z;
                        dt[h] = dt[h] + c[h].w * a[h].w;
                    }
                }
                if (j < t) {  // the row's last, partly filled quad
                    float4 a[2], c[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        a[h] = *(const float4*)(Lk[h] + j);
                        c[h] = *(const float4*)(Lr[h] + j);
                    }
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        s[h] = s[h] - a[h].x * a[h].x;
                        dt[h] = dt[h] + c[h].x * a[h].x;
                        if (j + 1 < t) {
                            s[h] = s[h] - a[h].y * a[h].y;
                            dt[h] = dt[h] + c[h].y * a[h].y;
                        }
                        if (j + 2 < t) {
                            s[h] = s[h] - a[h].z * a[h].z;
                            dt[h] = dt[h] + c[h].z * a[h].z;
                        }
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const float dii = sqrtf(fmaxf(s[h], m.eps));
                    const float inv = 1.f / dii;
                    val[h] = I.li[h] == t ? dii : (hr[h] - dt[h]) * inv;
                }
            }
            wave_sync();
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (on[h]) H[I.hb[h] + t] = val[h];
            wave_sync();
        }
    }

    // solver.py:2722-2751 + :1893-1910: Mgrad = (L L^T)^-1 grad, column by column, all islands side by side
    __device__ __forceinline__ void newton_direction() {
        float cur[2], dg[2];
        int x0[2];  // the island's first position
#pragma unroll
        for (int h = 0; h < 2; h++) {
            cur[h] = grad[h];
            dg[h] = I.own[h] ? H[I.hb[h] + I.li[h]] : 1.f;
            x0[h] = I.pos[h] - I.li[h];
        }
        auto below = [&](int h, int t) { return (I.own[h] && I.li[h] > t) ? H[I.hb[h] + t] : 0.f; };
        auto beside = [&](int h, int t) {
            return (I.own[h] && I.li[h] < t && t < I.n[h]) ? H[I.cb[h] + tri4(t) + I.li[h]] : 0.f;
        };
        wave_sync();
        float l[2] = {below(0, 0), below(1, 0)};
        for (int t = 0; t < I.steps; t++) {
            const float ln[2] = {below(0, t + 1), below(1, t + 1)};
            const float c[2] = {cur[0] / dg[0], cur[1] / dg[1]};
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (I.own[h] && I.li[h] == t) xv[I.pos[h]] = cur[h] = c[h];
            wave_sync();
            float x[2];
#pragma unroll
            for (int h = 0; h < 2; h++) x[h] = (I.own[h] && I.li[h] > t) ? xv[x0[h] + t] : 0.f;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (I.own[h] && I.li[h] > t) cur[h] = cur[h] - l[h] * x[h];
                l[h] = ln[h];
            }
            wave_sync();
        }
        l[0] = beside(0, I.steps - 1);
        l[1] = beside(1, I.steps - 1);
        for (int t = I.steps - 1; t >= 0; t--) {
            const float ln[2] = {beside(0, t - 1), beside(1, t - 1)};
            const float c[2] = {cur[0] / dg[0], cur[1] / dg[1]};
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (I.own[h] && I.li[h] == t) xv[I.pos[h]] = cur[h] = c[h];
            wave_sync();
            float x[2];
            bool on[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                on[h] = I.own[h] && I.li[h] < t && t < I.n[h];
                x[h] = on[h] ? xv[x0[h] + t] : 0.f;
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (on[h]) cur[h] = cur[h] - l[h] * x[h];
                l[h] = ln[h];
            }
            wave_sync();
        }
#pragma unroll
        for (int h = 0; h < 2; h++) Mgrad[h] = cur[h];
    }

    // solver.py:2722-2751: the gradient and the preconditioned direction
    __device__ __forceinline__ void gradient(bool cg) {
#pragma unroll
        for (int h = 0; h < 2; h++) grad[h] = Ma[h] - force[h] - qfc[h];
        if (!cg) {
            newton_direction();
            return;
        }
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (I.own[h]) LF(grad, lane + h * kWave) = grad[h];
        wave_sync();
        wave_solve_mass(m, loc, lane, FP(loc, grad), FP(loc, Mgrad));
#pragma unroll
        for (int h = 0; h < 2; h++) Mgrad[h] = I.own[h] ? LF(Mgrad, lane + h * kWave) : 0.f;
    }

    // the two coefficients of a friction-loss row outside its quadratic range
    __device__ __forceinline__ static void friction_line(float f, float rf, float ja, float jv, bool ln, bool lp,
                                                         float& a0, float& a1, float& a2) {
        a0 = (float)ln * f * (-0.5f * rf - ja) + (float)lp * f * (-0.5f * rf + ja);
        a1 = (float)ln * (-f * jv) + (float)lp * (f * jv);
        a2 = 0.f;
    }

    // solver.py:2034-2152
    __device__ __forceinline__ LsP ls_init(int& ls_it) {
        put(search);
        mass_mul(mv);
        qg[0] = gauss;
        qg[1] = dof_sum(search[0] * Ma[0] - search[0] * force[0], search[1] * Ma[1] - search[1] * force[1]);
        qg[2] = dof_sum(0.5f * search[0] * mv[0], 0.5f * search[1] * mv[1]);
        float t[3] = {0.f, 0.f, 0.f}, e[3] = {0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < nc; c0 += kRows * kWave) {
            float jr[kRows], dr[kRows], vr[kRows];
#pragma unroll
            for (int u = 0; u < kRows; u++) {
                const int c = min(c0 + u * kWave + lane, nc - 1);
                jr[u] = R.Jaref(c);
                dr[u] = R.efc_D(c);
                vr[u] = 0.f;
            }
            row_dots(c0, vr);
#pragma unroll
            for (int u = 0; u < kRows; u++) {
                const int c = c0 + u * kWave + lane;
                if (c >= nc) continue;
                const float ja = jr[u], Dc = dr[u], jv = vr[u];
                R.jv(c) = jv;
                float f0 = Dc * (0.5f * ja * ja), f1 = Dc * (jv * ja), f2 = Dc * (0.5f * jv * jv);
                if (c < ne) {
                    e[0] = e[0] + f0;
                    e[1] = e[1] + f1;
                    e[2] = e[2] + f2;
                } else if (c < nef) {
                    const float f = R.fl(c), rf = R.diag(c) * f;
                    const bool ln = ja <= -rf, lp = ja >= rf;
                    if (ln || lp) friction_line(f, rf, ja, jv, ln, lp, f0, f1, f2);
                } else {
                    const float a = (float)(ja < 0.f);
                    f0 = f0 * a;
                    f1 = f1 * a;
                    f2 = f2 * a;
                }
                t[0] = t[0] + f0;
                t[1] = t[1] + f1;
                t[2] = t[2] + f2;
            }
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            t[k] = qg[k] + wave_sum_f(t[k]);
            es[k] = ne > 0 ? wave_sum_f(e[k]) : 0.f;
        }
        float h = 2.f * t[2];
        if (h <= 0.f) h = m.eps;
        ls_it = 1;
        wave_sync();
        return {0.f, t[0], t[1], h};
    }

    // solver.py:2155-2355 for N = 1 or 3 candidate steps: one pass over the rows, their values loaded together
    template <int N>
    __device__ __forceinline__ void ls_eval(const float* al, LsP* out, int& ls_it) const {
        float T[3 * N];
#pragma unroll
        for (int q = 0; q < 3 * N; q++) T[q] = 0.f;
        constexpr int U = 5;
        for (int c0 = 0; c0 < nc; c0 += U * kWave) {
            float ja[U], jv[U], Dc[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = min(c0 + u * kWave + lane, nc - 1);
                ja[u] = R.Jaref(c);
                jv[u] = R.jv(c);
                Dc[u] = R.efc_D(c);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + u * kWave + lane;
                if (c < ne || c >= nc) continue;
                const float f0 = Dc[u] * (0.5f * ja[u] * ja[u]), f1 = Dc[u] * (jv[u] * ja[u]),
                            f2 = Dc[u] * (0.5f * jv[u] * jv[u]);
                if (c < nef) {
                    const float f = R.fl(c), rf = R.diag(c) * f;
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const float x = ja[u] + al[k] * jv[u];
                        const bool ln = x <= -rf, lp = x >= rf;
                        float a0 = f0, a1 = f1, a2 = f2;
                        if (ln || lp) friction_line(f, rf, ja[u], jv[u], ln, lp, a0, a1, a2);
                        T[3 * k] = T[3 * k] + a0;
                        T[3 * k + 1] = T[3 * k + 1] + a1;
                        T[3 * k + 2] = T[3 * k + 2] + a2;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const float a = (float)(ja[u] + al[k] * jv[u] < 0.f);
                        T[3 * k] = T[3 * k] + f0 * a;
                        T[3 * k + 1] = T[3 * k + 1] + f1 * a;
                        T[3 * k + 2] = T[3 * k + 2] + f2 * a;
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 3 * N; q++) T[q] = (qg[q % 3] + es[q % 3]) + wave_sum_f(T[q]);
#pragma unroll
        for (int k = 0; k < N; k++) {
            const float a = al[k];
            float h = 2.f * T[3 * k + 2];
            if (h <= 0.f) h = m.eps;
            out[k] = {a, a * a * T[3 * k + 2] + a * T[3 * k + 1] + T[3 * k], 2.f * a * T[3 * k + 2] + T[3 * k + 1], h};
        }
        ls_it += N;
    }
};

// solver.py:2936-3059 (init), :3063-3139 (Newton or conjugate-gradient iteration), :3164-3190 (body), :3241-3261,
// :3199-3237. tile: at least island_words(D) words; H: the packed triangles (LDS, or the record's nt_H).
template <bool kHLds, int kQ>
__device__ __forceinline__ void island_solve_rows(const DModel& m, const LState& loc, const DState& st, int b, const WorkRows& R,
                                    const RowGroups& Q, int lane, float* tile, float* H) {
    const int D = m.D;
    const int nc = LF(n_con, 0), ne = LF(n_con_eq, 0), nef = ne + LF(n_con_fl, 0);
    IslandDofs I;
    find_islands(m, Q, nc - 3 * Q.ncont, lane, (int*)tile, I);
    IslandSolver<kHLds, kQ> S{m, loc, R, Q, I, H, tile, lane, nc, ne, nef};
    const bool ws = nc > 0 && LF(is_warmstart, 0);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + h * kWave;
        S.qacc[h] = S.force[h] = S.acc0[h] = 0.f;
        if (I.own[h]) {
            S.acc0[h] = LF(acc_smooth, d);
            S.qacc[h] = ws ? LF(qacc_ws, d) : S.acc0[h];
            S.force[h] = LF(force, d);
        }
    }
    if (lane == 0) S.xv[D] = 0.f;
    S.put(S.qacc);
    S.mass_mul(S.Ma);
    S.init_rows();
    const bool cg = m.solver_type == RS_SOLVER_CG;
    float prev = LF(cost, 0);
    float cost = S.update(true, 0.f);
    int improved = nc > 0;
    if (!cg) {
        S.hessian();
        S.factor();
    }
    S.gradient(cg);
#pragma unroll
    for (int h = 0; h < 2; h++) S.search[h] = -S.Mgrad[h];
    S.mv[0] = S.mv[1] = 0.f;
    int n_iter = 0;
    if (nc > 0) {
        const float tol = (m.meaninertia * (float)max(1, D)) * m.tolerance;
        for (int it = 0; it < m.iterations; it++) {
            n_iter++;
            const float sn = sqrtf(S.dof_sum(S.search[0] * S.search[0], S.search[1] * S.search[1]));
            const float alpha = linesearch_body(m, loc, sn, S);
            if (fabsf(alpha) < m.eps) {
                improved = 0;
            } else {
                float pg[2] = {S.grad[0], S.grad[1]}, pM[2] = {S.Mgrad[0], S.Mgrad[1]};
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    S.qacc[h] = S.qacc[h] + S.search[h] * alpha;
                    S.Ma[h] = S.Ma[h] + S.mv[h] * alpha;
                }
                prev = cost;
                cost = S.update(false, alpha);
                if (!cg) {
                    S.hessian();
                    S.factor();
                }
                S.gradient(cg);
                const float gn = sqrtf(S.dof_sum(S.grad[0] * S.grad[0], S.grad[1] * S.grad[1]));
                improved = gn > tol && (prev - cost) > tol;
                if (improved && !cg) {
#pragma unroll
                    for (int h = 0; h < 2; h++) S.search[h] = -S.Mgrad[h];
                } else if (improved) {  // solver.py:2865-2884 Polak-Ribiere direction
                    float beta = S.dof_sum(S.grad[0] * (S.Mgrad[0] - pM[0]), S.grad[1] * (S.Mgrad[1] - pM[1]));
                    const float pgM = S.dof_sum(pM[0] * pg[0], pM[1] * pg[1]);
                    beta = fmaxf(beta / fmaxf(m.eps, pgM), 0.f);
                    FV(st, cg_pg_dot_pMg, b)[0] = pgM;
                    FV(st, cg_beta, b)[0] = beta;
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const int d = lane + h * kWave;
                        if (I.own[h]) {
                            FV(st, cg_prev_grad, b)[d] = pg[h];
                            FV(st, cg_prev_Mgrad, b)[d] = pM[h];
                        }
                        S.search[h] = -S.Mgrad[h] + beta * S.search[h];
                    }
                }
            }
            if (!improved) break;
        }
    } else {
        improved = 0;
    }
    LF(cost, 0) = cost;
    LF(prev_cost, 0) = prev;
    LF(gauss, 0) = S.gauss;
    LF(improved, 0) = improved;
    LF(n_iter, 0) = n_iter;
    bool nan_seen = false;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int d = lane + h * kWave;
        if (!I.own[h]) continue;
        const float qa = S.qacc[h];
        LF(qacc, d) = qa;
        LF(acc, d) = qa;
        LF(qacc_ws, d) = qa;
        LF(Ma, d) = S.Ma[h];
        LF(grad, d) = S.grad[h];
        LF(Mgrad, d) = S.Mgrad[h];
        LF(search, d) = S.search[h];
        LF(mv, d) = S.mv[h];
        LF(qfrc_constraint, d) = S.qfc[h];
        LF(qf_constraint, d) = S.qfc[h];
        LF(force, d) = LF(qf_smooth, d) + S.qfc[h];
        nan_seen = nan_seen || isnan(qa);
    }
    if (wave_ballot(nan_seen) != 0) LF(errbits, 0) = LF(errbits, 0) | RS_ERR_INVALID_FORCE_NAN;
    LF(is_warmstart, 0) = 1;
    wave_sync();
    export_row_forces(m, loc, st, b, R, lane);
    wave_sync();
}

// rows of up to 12 entries (free bodies and short chains) hold all their loads in registers; longer ones take fewer at once
template <bool kHLds>
__device__ __forceinline__ void island_solve(const DModel& m, const LState& loc, const DState& st, int b, const WorkRows& R,
                                    const RowGroups& Q, int lane, float* tile, float* H) {
    if (Q.W <= 12) island_solve_rows<kHLds, 3>(m, loc, st, b, R, Q, lane, tile, H);
    else island_solve_rows<kHLds, kRowWidthMax / 4>(m, loc, st, b, R, Q, lane, tile, H);
}

#undef LF

}  // namespace rs
