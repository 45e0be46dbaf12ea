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

// Whether the segments' launches take less time than the 16-token-block kernel,
// which cuts each block's keys into nsplit splits of `split`.  len: the keys per
// sequence that the launch is sized for; known: that is the caller's bound of the
// sequences' lengths, not just the cache's capacity.  Measured (us, 8 heads over 2
// KV heads of 256, 256 CUs; the 64-token blocks against the 16-token ones):
// - one split: the 16-token kernel writes the outputs itself, without a merge
//   (64 x 96 tokens alone 114 : 93, 200 x 32 after 224 188 : 162, 64 x 160 182 : 179).
// - Four launches per segment cost ~43 before the keys count, the other kernel ~12
//   and 0.08 per key of a split while its workgroups are one per CU: worth it from
//   288 keys x 16-token blocks per CU and segment (1 x 512 after 500: 65 K, 54 : 44;
//   1 x 777: 76 K, 53 : 70; 8 x 128 after 500: 80 K, 57 : 58; 8 x 512: 512 K, 95 :
//   157), and where one split is long (1 x 64 after 2000 58 : 40, after 8000 88 : 94,
//   after 30000 125 : 303).
// - Of a run of one or two blocks per sequence each expanded key is used little.
//   For half a block over many keys, and once the expanded keys outgrow the
//   memory-side cache (from ~144 MB), fits of both sides decide: 30 per segment, 0.8
//   per sequence and the expanded bytes at 1.15 TB/s, 0.6 times that again for a
//   second block, against rounds of workgroups of 13 + 0.08 per key (8 x 32 after 8000
//   113 : 97, after 30000 535 : 308, 16 x 32 after 30000 1073 : 597, 16 x 80 1698 : 1480,
//   8 x 64 after 10000 189 : 221, 3 x 32 after 28000 231 : 279, 4 x 32 after 14000 99 : 151;
//   from 96 tokens on the blocks win, 8 x 96 after 30000 850 : 900).
// - Keys not known: only the run's own are certain, and the other kernel, its splits
//   sized for the capacity, walks them in one: worth it from 72 keys x blocks per CU
//   and segment (position 0, capacity 32768: 1 x 256 44 : 38, 1 x 400 49 : 73, 8 x 256
//   in four segments 196 : 177, 8 x 100 180 : 62, 64 x 100 1465 : 412; capacity 2048: 64
//   x 100 157 : 412), and not for a block that is half empty (100 x 32, 130 : 102).
inline bool pf_pays(const PfCall& p, const PfSegments& s, int64_t len, bool known, int64_t split, int64_t nsplit) {
    if (nsplit <= 1) return false;
    const int64_t nseg = (p.batch + s.nb - 1) / s.nb * ((p.tokens + s.ntok - 1) / s.ntok);
    const int64_t blocks = (int64_t)p.batch * p.nkv * ((p.tokens + 15) / 16);
    if (!known) return p.tokens >= 48 && blocks * std::min<int64_t>(p.tokens, len) >= 72 * p.cus * nseg;
    if (split < 832 && blocks * len < 288 * p.cus * nseg) return false;
    const double bytes = (double)p.batch * p.seq_bytes();
    if (p.tokens >= 96 || (bytes <= 144e6 && (p.tokens > PF_Q / 2 || split < 832))) return true;
    const double rounds = std::max(1.0, (double)blocks * nsplit / p.cus);
    return 30.0 * nseg + 0.8 * p.batch + bytes * (p.tokens > PF_Q ? 1.6 : 1.0) / 1.15e6 < rounds * (13.0 + 0.08 * split);
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
    // as many CUs as the partials allow, where the blocks alone do not fill the chip
    // (8 x 100 tokens after 8000, room for 160: 367 us for 128 CUs, 266 for 165)
    while (g.units > min_units && pf_most_shares(g.units, nblk) > g.pieces)
        g.units -= nblk >= g.units ? (g.units + 1) / 2 : (g.units + 15) / 16;
    g.units = std::max(g.units, min_units);
    g.lone = nblk > g.units || pf_most_units(g.units, nblk) > g.pieces;
    g.room = (int)(pf_most_units(g.units, nblk) / p.nkv * p.nkv);
    g.grid = g.room + p.nkv;
    return g;
}

}  // namespace qwk
