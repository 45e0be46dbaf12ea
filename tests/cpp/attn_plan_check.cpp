// Runs the plan of the 64-token-block INT8 attention prefill (qw_attn_plan.hpp, the
// header that the kernels and the host share) over sequences, tokens, contexts and
// workspaces, and checks that what the kernels will need never exceeds what the
// host provides: units <= workgroups (but the last of each head), cut units <=
// partials, everything inside the workspace.  Prints the first violation, or "ok".
#include <cstdio>
#include <cmath>
#include <random>
#include <vector>

#include "qw_attn_plan.hpp"

using namespace qwk;

static long plans = 0, units_seen = 0;

static bool check_segment(const PfCall& p, const PfSegments& s, int64_t nb, int tb, int ntok, int pend, const int* pos) {
    const PfSegment g = pf_segment(p, s.min_units, nb, ntok);
    uint64_t total = 0, walked = 0, units = 0, cut = 0;
    for (int64_t b = 0; b < nb; ++b) total += PfSeq(pend, tb, ntok, pos[b]).all();
    total *= p.nkv;
    const uint32_t ut = pf_unit_tiles((uint32_t)total, g.units);
    bool good = total < (1ull << 31);
    for (int64_t b = 0; b < nb; ++b) {
        const PfSeq q(pend, tb, ntok, pos[b]);
        good = good && (int64_t)q.tmax * PF_KT <= p.keys;
        for (uint32_t j = 0; j < q.nblk; ++j) {
            const uint32_t n = pf_shares(q, ut, j), t = q.tiles(j);
            good = good && t >= 1 && n >= 1 && (n - 1) * ut < t && t <= n * ut;
            // the tiles reach the block's last valid query
            const int64_t P = pos[b], last = std::min<int64_t>(P + tb + ntok - 1 - (int64_t)j * PF_Q + (int64_t)(q.nblk * PF_Q - ntok), pend - 1);
            good = good && (P < 0 || P >= pend || (int64_t)t * PF_KT > std::min<int64_t>(last, P + tb + ntok - 1));
            walked += t;
            units += n;
            cut += n > 1 || !g.lone ? n : 0;
        }
    }
    ++plans;
    units_seen += units;
    good = good && walked * p.nkv == total && g.units >= 1 && (int64_t)units * p.nkv <= g.room && g.grid == g.room + p.nkv &&
           (int64_t)cut * p.nkv <= g.pieces && g.part_off + (size_t)g.pieces * p.piece_bytes() <= p.ws &&
           g.k_off >= (size_t)(nb * ntok) * p.row_bytes() &&
           g.part_off >= g.s_off + (size_t)nb * p.nkv * (p.keys / PF_KT) * PF_SC * 4;
    if (!good)
        printf("violation: heads %d/%d hd %d cus %d batch %ld tb %d ntok %d pend %d pos %d ws %zu: tiles %lu, ut %u, units %lu "
               "x %d, grid %d, cut %lu, pieces %d\n", p.nh, p.nkv, p.hd, p.cus, (long)nb, tb, ntok, pend, pos[0], p.ws,
               (unsigned long)total, ut, (unsigned long)units, p.nkv, g.grid, (unsigned long)cut, g.pieces);
    return good;
}

// every segment of a call; false on a violation
static bool check_call(int nh, int nkv, int hd, int cus, size_t ws, int batch, int tokens, int pend, const int* pos) {
    const PfCall p{nh, nkv, hd, cus, batch, tokens, ((int64_t)pend + 63) / 64 * 64, ws};
    const PfSegments s = pf_segments(p);
    if (s.ntok < 32) return true;  // the 16-token kernels
    for (int64_t b0 = 0; b0 < batch; b0 += s.nb)
        for (int64_t tb = 0; tb < tokens; tb += s.ntok)
            if (!check_segment(p, s, std::min(s.nb, batch - b0), (int)tb, (int)std::min(s.ntok, tokens - tb), pend, pos + b0))
                return false;
    return true;
}

// the route of a call of 8 heads over 2 KV heads of 256 on 256 CUs, its splits cut
// as qw_attn_forward cuts them
static bool route(int batch, int tokens, int len, bool known, size_t ws = 180u << 20) {
    const int split = std::max(256, ((len + 7) / 8 + 31) / 32 * 32), nsplit = (len + split - 1) / split;
    const PfCall p{8, 2, 256, 256, batch, tokens, ((int64_t)len + 63) / 64 * 64, ws};
    const PfSegments s = pf_segments(p);
    return s.ntok >= 32 && pf_pays(p, s, len, known, split, nsplit);
}

// A cache's spare capacity takes no call to the 64-token blocks that its keys do not.
static bool check_routes() {
    struct R { int batch, tokens, len; bool known, blocks; };
    std::vector<R> rs;
    for (int cap : {4096, 8192, 32768})
        for (const R& r : {R{1, 64, 0, false, false}, R{1, 144, 0, false, false}, R{1, 256, 0, false, false},
                           R{8, 100, 0, false, false}, R{1, 777, 0, false, true}, R{1, 4096, 0, false, true}})
            rs.push_back({r.batch, r.tokens, std::max(cap, r.tokens), false, r.blocks});
    for (const R& r : {R{64, 100, 8192, false, false}, R{64, 100, 32768, false, false}, R{64, 100, 2048, false, true},
                       R{100, 32, 1024, false, false}, R{1, 64, 64, true, false}, R{8, 100, 100, true, false},
                       R{1, 64, 30064, true, true}, R{1, 512, 1012, true, false}, R{1, 777, 777, true, true},
                       R{8, 512, 512, true, true}, R{16, 32, 30032, true, false}, R{8, 32, 8032, true, false}, R{4, 32, 14032, true, true},
                       R{8, 32, 10532, true, false}, R{16, 80, 30080, true, false}, R{8, 64, 10064, true, true}, R{8, 100, 32100, true, true},
                       R{1, 4096, 4096, true, true}})
        rs.push_back(r);
    for (const R& r : rs)
        if (route(r.batch, r.tokens, r.len, r.known) != r.blocks) {
            printf("violation: route of %d x %d, %d keys (%sknown): not the %d-token blocks\n", r.batch, r.tokens, r.len,
                   r.known ? "" : "not ", r.blocks ? 64 : 16);
            return false;
        }
    // a bound at its loosest makes no difference to calls whose keys are not known
    for (int batch : {1, 2, 5, 8, 30, 64})
        for (int tokens = 32; tokens <= 512; tokens += 16)
            for (int len = 1024; len <= 65536; len *= 2)
                if (route(batch, tokens, 2 * len, false) && !route(batch, tokens, len, false)) {
                    printf("violation: %d x %d takes the 64-token blocks for a capacity of %d, not of %d\n", batch, tokens,
                           2 * len, len);
                    return false;
                }
    return true;
}

int main() {
    if (!check_routes()) return 1;
    const size_t big = 180u << 20;
    // one sequence, and several at one position, at every position up to 32768:
    // a cache just long enough, and one of 32768
    for (int cus : {256, 304, 80})
        for (int nkv : {1, 2, 4})
            for (int tokens : {32, 64, 96, 128, 192, 320})
                for (int batch : {1, 2, 4})
                    for (int P = 0; P + tokens <= 32768; P += batch == 1 ? 1 : 7) {
                        const int pos[4] = {P, P, P, P};
                        if (!check_call(4 * nkv, nkv, 256, cus, big, batch, tokens, P + tokens, pos)) return 1;
                        if (P % 5 == 0 && !check_call(4 * nkv, nkv, 256, cus, big, batch, tokens, 32768, pos)) return 1;
                    }
    // ragged batches, invalid positions, workspaces down to where no segment fits
    std::mt19937 rng(1);
    auto upto = [&](int lo, int hi) {  // spread over the logarithm
        const double u = std::uniform_real_distribution<double>(0, 1)(rng);
        return std::min(hi, (int)(lo * std::pow((double)(hi + 1) / lo, u)));
    };
    for (int i = 0; i < 200000; ++i) {
        const int nkv = 1 << (rng() % 3), G = 1 + rng() % 4, hd = rng() % 2 ? 256 : 128, batch = upto(1, 100);
        const int tokens = upto(32, 6000 / batch + 32), pend = upto(64, 40000);
        std::vector<int> pos(batch);
        const int base = (int)(rng() % pend);
        for (int& x : pos) x = rng() % 4 ? (rng() % 2 ? base : (int)(rng() % pend)) : rng() % 8 ? base / 2 : rng() % 2 ? -5 : pend + 9;
        const size_t ws = (size_t)upto(1 << 10, 200 << 10) << 10;
        if (!check_call(G * nkv, nkv, hd, rng() % 4 ? 256 : upto(1, 400), ws, batch, tokens, pend, pos.data())) return 1;
    }
    printf("ok: %ld plans, %ld units\n", plans, units_seen);
    return 0;
}
