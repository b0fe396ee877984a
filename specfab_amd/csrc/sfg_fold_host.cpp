// Host layout of the folded operator (sfg_fold.h), from the real-basis terms.
#include <algorithm>
#include <array>
#include <cmath>
#include <map>
#include <mutex>
#include <stdexcept>

#include "sfg_fold.h"
#include "sfg_internal.h"

namespace sfg {

namespace {
// weight pairs (Re, Im) of the operator's parameters, -1 where real
const int kWeight[14][2] = {{0, -1}, {1, 2}, {3, 4}, {5, -1}, {6, 7}, {8, -1}, {9, -1},
                            {10, 11}, {12, 13}, {14, -1}, {15, 16}, {17, 18}, {19, 20}, {21, 22}};
// threads per workgroup and sources per thread: whole waves that the chunks
// fill to 80-99 % (L = 8: 62 of 64, L = 12: 220 of 256, L = 20: 452 of 512)
void shape(int L, int* threads, int* slots) {
    static const int s[9][2] = {{64, 2}, {64, 5}, {64, 9}, {128, 8}, {256, 6}, {256, 8}, {512, 5}, {512, 7}, {512, 9}};
    *threads = s[L / 2 - 2][0];
    *slots = s[L / 2 - 2][1];
}
}  // namespace

// (A + B s) / (C + s) through the crossings measured at s = 1, 2, 4, 12, 40 and
// 120 stages per launch, within 10 % of each (250 to 13,000 parcels, LROT + REG +
// DDRX; the parameters' launch counted).  FP64, L = 12: 1,595 parcels at one
// stage (1,500: 19 us against 19; 5,000: 56 against 39 at four), 3,234 at four,
// 7,424 at forty (5,000: 183 against 264; 8,000: 283 against 264); L = 4, one
// stage: 3,050 (5,000: 21.5 us against 13.3).
int64_t fold_limit(int L, int prec, int64_t stages) {
    static const double A[2][9] = {{138400, 73400, 21200, 21400, 7600, 6600, 6400, 6400, 5700},
                                   {36700, 11100, 1400, 23700, 32300, 23800, 8400, 9900, 11500}};
    static const double B[2][9] = {{5600, 10000, 10500, 12300, 8900, 9900, 6700, 8500, 8200},
                                   {8300, 10500, 14500, 13000, 12700, 12800, 8600, 5900, 7700}};
    static const double C[2][9] = {{45.5, 27.7, 13.4, 15.7, 9.3, 10.8, 9.5, 10.1, 10.7},
                                   {85.7, 34.5, 19.2, 27.6, 34.1, 34.1, 18.7, 18.6, 21.9}};
    if (L < 4 || L > 20 || L % 2 || stages < 0) return 0;
    const int i = L / 2 - 2;
    const double s = (double)(stages > 0 ? stages : 1);
    return (int64_t)((A[prec][i] + B[prec][i] * s) / (C[prec][i] + s));
}

namespace {
FoldLayout build(int L) {
    if (L < 4 || L > 20 || L % 2) throw std::invalid_argument("L must be even, 4 <= L <= 20");
    const RealOperator& op = real_operator(L);
    FoldLayout f;
    f.L = L;
    f.n = op.n;
    shape(L, &f.threads, &f.slots);
    std::vector<int> pair_of(op.n), part_of(op.n);
    int np = -1;
    for (int r = 0; r < op.n; r++) {
        if (op.ridx[r].c == 0) np++;
        pair_of[r] = np;
        part_of[r] = op.ridx[r].c;
        f.pos.push_back(2 * np + op.ridx[r].c);
        f.blk.push_back(op.ridx[r].l / 2);
    }
    f.npairs = np + 1;
    int wk[23];
    for (int k = 0; k < 14; k++)
        for (int q = 0; q < 2; q++)
            if (kWeight[k][q] >= 0) wk[kWeight[k][q]] = k;
    // (target pair, source pair) -> weight pair -> the four cells' signed parameters and the value
    typedef std::array<int, 4> Code;
    struct Entry { double c; Code code; };
    std::map<std::pair<int, int>, std::map<int, Entry>> blocks;
    for (int r = 0; r < op.n; r++)
        for (int g = op.rows[r].g0; g < op.rows[r].g1; g++) {
            const int p = op.groups[g].param;
            for (int t = op.groups[g].t0; t < op.groups[g].t1; t++) {
                const int col = op.terms[t].col;
                const double v = op.terms[t].val;
                auto& m = blocks[{pair_of[r], pair_of[col]}];
                auto it = m.find(wk[p]);
                if (it == m.end()) it = m.emplace(wk[p], Entry{v, Code{0, 0, 0, 0}}).first;
                if (std::fabs(v) != std::fabs(it->second.c))
                    throw std::runtime_error("a coupling is not a complex product");
                it->second.code[2 * part_of[r] + part_of[col]] = (v == it->second.c ? 1 : -1) * (p + 1);
            }
        }
    // <D>: sum over the first 15 rows of omega_q x_q
    const int gt = f.npairs;
    for (int q = 0; q < std::min(op.n, 15); q++) {
        auto& m = blocks[{gt, pair_of[q]}];
        auto it = m.find(14);
        if (it == m.end()) it = m.emplace(14, Entry{1.0, Code{0, 0, 0, 0}}).first;
        it->second.code[part_of[q]] = 23 + q + 1;
    }
    std::map<Code, int> pats;
    pats[Code{0, 0, 0, 0}] = 0;   // entries past a thread's own
    struct Slot { int src; std::vector<Entry> e; };
    std::vector<std::vector<Slot>> lanes;
    std::vector<int> c0(f.npairs + 1), cn(f.npairs + 1);
    for (int t = 0; t <= f.npairs; t++) {
        std::vector<Slot> all;
        for (auto b = blocks.lower_bound({t, 0}); b != blocks.end() && b->first.first == t; ++b) {
            Slot s{b->first.second, {}};
            for (auto& e : b->second) s.e.push_back(e.second);
            all.push_back(s);
        }
        // most entries first, dealt round the chunks: a wave's slots then
        // need similar entry counts
        std::stable_sort(all.begin(), all.end(), [](const Slot& a, const Slot& b) { return a.e.size() > b.e.size(); });
        const int nc = ((int)all.size() + f.slots - 1) / f.slots;
        c0[t] = (int)lanes.size();
        cn[t] = nc;
        std::vector<std::vector<Slot>> ch(nc);
        for (size_t i = 0; i < all.size(); i++) ch[i % nc].push_back(all[i]);
        if (t != gt) f.chunks = std::max(f.chunks, nc);
        lanes.insert(lanes.end(), ch.begin(), ch.end());
    }
    if (f.n > f.threads || cn[gt] > FOLD_G) throw std::runtime_error("rows or <D> chunks outnumber the threads");
    if ((int)lanes.size() > f.threads) throw std::runtime_error("the chunks outnumber the threads");
    f.g0 = c0[gt];
    f.gn = cn[gt];
    for (int r = 0; r < op.n; r++) {
        f.chunk0.push_back(c0[pair_of[r]]);
        f.chunkn.push_back(cn[pair_of[r]]);
    }
    lanes.resize(f.threads);
    // a thread's slots past its own sources read the pair after the last, which
    // stays zero: a coefficient that is not finite reaches only what it couples to
    f.src.assign((size_t)f.slots * f.threads, f.npairs);
    for (int w = 0; w < f.threads / 64; w++)
        for (int j = 0; j < f.slots; j++) {
            int most = 0;
            for (int l = 0; l < 64; l++) {
                auto& ln = lanes[64 * w + l];
                if (j < (int)ln.size()) {
                    most = std::max(most, (int)ln[j].e.size());
                    f.src[(size_t)j * f.threads + 64 * w + l] = ln[j].src;
                }
            }
            f.cnt.push_back(most);
            f.base.push_back((int)(f.c.size() / 64));
            for (int e = 0; e < most; e++)
                for (int l = 0; l < 64; l++) {
                    auto& ln = lanes[64 * w + l];
                    const bool on = j < (int)ln.size() && e < (int)ln[j].e.size();
                    const Code code = on ? ln[j].e[e].code : Code{0, 0, 0, 0};
                    auto it = pats.emplace(code, (int)pats.size()).first;
                    f.c.push_back(on ? ln[j].e[e].c : 0.0);
                    f.pat.push_back((unsigned char)it->second);
                }
        }
    f.npat = (int)pats.size();
    if (f.npat > FOLD_PATTERNS) throw std::runtime_error("too many weight patterns");
    f.pcode.assign(4 * f.npat, 0);
    for (auto& p : pats)
        for (int q = 0; q < 4; q++) f.pcode[4 * p.second + q] = (signed char)p.first[q];
    return f;
}

}  // namespace

// once per truncation and process (4 ms at L = 20), as real_operator
const FoldLayout& fold_layout(int L) {
    static std::mutex mu;
    static std::map<int, FoldLayout> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(L);
    if (it == cache.end()) it = cache.emplace(L, build(L)).first;
    return it->second;
}

}  // namespace sfg
