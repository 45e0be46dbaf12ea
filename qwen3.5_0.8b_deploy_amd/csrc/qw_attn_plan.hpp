// qw_attn_plan.hpp -- how the INT8 attention prefill in 64-token blocks (attn_pf)
// cuts a segment of sequences and tokens into units of work.  The kernels compute
// the plan (only they know the positions); the host sizes the grid and the
// partials for any plan.  Both use this one header, which a plain C++ compiler
// takes as well.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#if defined(__HIPCC__)
#define QW_HD __host__ __device__ __forceinline__
#else
#define QW_HD inline
#endif

namespace qwk {

constexpr int PF_Q = 64;    // tokens per query block
constexpr int PF_KT = 32;   // keys per tile
constexpr int PF_SC = 128;  // floats per tile of scales: 32 K | 32 V | raise threshold | padding
constexpr int PF_MIN = 4;   // fewest tiles per unit

// The query blocks of one sequence, longest first: block j (tokens 64 (nblk - 1
// - j) .. of the segment's [tb, tb + ntok)) has tiles(j) key tiles (up to two more
// than its last query needs; at least one).  pend: positions stay below it, P0:
// the sequence's position, valid or not.  The host bounds the segment's total
// tiles below 2^31.
struct PfSeq {
    uint32_t nblk, c, tmax;
    QW_HD PfSeq(int pend, int tb, int ntok, int P0) {
        const int p = P0 < 0 ? 0 : P0 > pend ? pend : P0;
        nblk = (uint32_t)(ntok + PF_Q - 1) / PF_Q;
        tmax = (uint32_t)(pend + PF_KT - 1) / PF_KT;
        c = ((uint32_t)p + tb + PF_KT - 1) / PF_KT;
    }
    QW_HD uint32_t tiles(uint32_t j) const {
        const uint32_t t = c + 2 * (nblk - j);
        return t < tmax ? t : tmax;
    }
    QW_HD uint32_t all() const {  // sum over the blocks, c + 2, c + 4, .. clamped to tmax
        const uint32_t below = tmax > c ? (tmax - c) / 2 : 0u, k = below < nblk ? below : nblk;
        return k * c + k * (k + 1) + (nblk - k) * tmax;
    }
};

// Longest unit, in tiles, of a plan for `units` CUs over `total` tiles:
// 1.3 (floor(total / units) + 1), rounded up, so strictly above 1.3 total / units
// for every total -- pf_most_units and pf_most_shares rest on that.
QW_HD uint32_t pf_unit_tiles(uint32_t total, uint32_t units) {
    const uint32_t k = total / units + 1, ut = k + (3 * k + 9) / 10;
    return ut < PF_MIN ? PF_MIN : ut;
}

// Units of block j
QW_HD uint32_t pf_shares(const PfSeq& q, uint32_t ut, uint32_t j) { return (q.tiles(j) + ut - 1) / ut; }

// Most units of any plan for `units` CUs over `blocks` blocks: a block of t tiles
// has less than t / ut + 1.
inline int64_t pf_most_units(int units, int64_t blocks) { return (int64_t)units * 10 / 13 + 1 + blocks; }
// Most that belong to blocks of more than one: at most 2 t / (ut + 1) each.
inline int64_t pf_most_shares(int units, int64_t blocks) {
    return std::min((int64_t)units * 20 / 13 + 1, pf_most_units(units, blocks));
}

// A call's shape, as far as the plan needs it.  keys: per sequence of the
// expanded cache, a multiple of 64.
struct PfCall {
    int nh, nkv, hd, cus, batch, tokens;
    int64_t keys;
    size_t ws;  // bytes for the f16 queries, the expanded cache and the partials

    size_t row_bytes() const { return (size_t)nh * hd * 2; }
    size_t seq_bytes() const { return (size_t)nkv * keys * (2 * hd * 2 + PF_SC * 4 / PF_KT); }
    size_t piece_bytes() const { return (size_t)(nh / nkv) * PF_Q * (hd + 2) * 4; }  // one share's partial
    static int64_t blocks(int64_t ntok) { return (ntok + PF_Q - 1) / PF_Q; }
};

// Segments of nb sequences x ntok tokens, each planned for at least min_units CUs;
// ntok < 32: the workspace holds none.
struct PfSegments {
    int64_t nb, ntok;
    int min_units;
};

inline PfSegments pf_segments(const PfCall& p) {
    PfSegments s{0, 0, std::min(p.cus, 32)};
    if (p.keys > (1 << 21)) return s;
    // a segment's rows, keys and the shares of a plan for min_units fit, and its
    // tiles count in 31 bits
    auto fits = [&] {
        return s.nb * (p.seq_bytes() + (size_t)s.ntok * p.row_bytes()) +
                       pf_most_shares(s.min_units, s.nb * p.nkv * p.blocks(s.ntok)) * p.piece_bytes() <= p.ws &&
               (double)s.nb * p.nkv * p.blocks(s.ntok) * (p.keys / PF_KT + 1) < 2147483648.0;
    };
    for (;;) {
        s.nb = std::min<int64_t>(p.batch, 65535), s.ntok = p.tokens;
        while (s.nb > 1 && !fits()) s.nb = (s.nb + 1) / 2;
        while (s.ntok >= 32 && !fits()) s.ntok = s.ntok / 2 / 32 * 32;
        if (s.ntok >= 32 || s.min_units < 32) return s;
        s.min_units = 4;  // small workspaces
    }
}

// One segment's launch.  Workspace: rows of f16 queries | K | V | scales | partials.
struct PfSegment {
    int units;    // CUs the plan aims at
    int lone;     // uncut blocks write the output themselves
    int room;     // workgroups that any plan's units (of all KV heads) fit into
    int grid;     // workgroups launched: one more per KV head, which finds no unit
    int pieces;   // partials that the workspace holds
    size_t k_off, v_off, s_off, part_off;
};

inline PfSegment pf_segment(const PfCall& p, int min_units, int64_t nb, int64_t ntok) {
    PfSegment g;
    const size_t rows = (size_t)(nb * ntok) * p.row_bytes(), kb = (size_t)nb * p.nkv * p.keys * p.hd * 2;
    g.k_off = rows;
    g.v_off = rows + kb;
    g.s_off = rows + 2 * kb;
    g.part_off = rows + nb * p.seq_bytes();
    g.pieces = (int)std::min<size_t>((p.ws - g.part_off) / p.piece_bytes(), 1u << 30);
    const int64_t nblk = nb * p.nkv * p.blocks(ntok);
    g.units = p.cus;
    while (g.units > min_units && pf_most_shares(g.units, nblk) > g.pieces) g.units /= 2;
    g.units = std::max(g.units, min_units);
    g.lone = nblk > g.units || pf_most_units(g.units, nblk) > g.pieces;
    g.room = (int)(pf_most_units(g.units, nblk) / p.nkv * p.nkv);
    g.grid = g.room + p.nkv;
    return g;
}

}  // namespace qwk
