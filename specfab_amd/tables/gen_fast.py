#!/usr/bin/env python3
"""Generate the register-resident stepping kernels (HIP, gfx950).

For each truncation L in FAST_L and each precision, this writes
csrc/generated/sfg_fast_L{L}_{f64|f32}_v{variant}.hip: one kernel that steps
64 parcels per group (one parcel per lane, a few waves per group) through all
its time steps.  Every coupling value is compiled into the instruction stream
as a literal constant (FP32: a 32-bit literal of the FMA itself; FP64: two
s_mov_b32 on the scalar unit, or a literal high word), so the operator costs
no memory traffic.  Per output row a the rate is

    f_a = sum_p theta_p (sum_b R_p[a][b] x_b) + (s_l(a) - Gamma0 <D>(x)) x_a

gen_kernel_pair evaluates it over complex couplings with the state resident in
registers and LDS; gen_kernel row by row, one FMA per coupling value, with the
stage data in SoA buffers (the plain form: a check of the term count, and of
the pair kernels, at the two most used truncations).

The sparsity structure and the values come from a dump of the host builder
(specfab_amd/tables/dump_basis.cpp), i.e. the same term array that the
generic stepper reads at run time (sfg::real_operator(L).terms).

FP32 variant ("FP32 stepping, compensated state update"): the operator
application and the RK increments run in FP32 (constants rounded to float);
the state x0 is kept and updated in FP64 (x1 = x0 + sum of FP32 increments).

Usage: gen_fast.py OUTDIR
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "csrc")
FAST_L = (4, 6, 8, 10, 12, 14, 16, 18, 20)

# Kernel variants (the library's autotuner times them and keeps the fastest):
#   lit   row by row, coupling values as literals, the RK increment sum and
#         the next-stage input in SoA buffers; `chunk` output rows accumulated
#         together
#   pair  complex couplings, state resident (gen_kernel_pair): `split` waves
#         per 64-parcel group, `waves` waves per SIMD asked of the register
#         allocator, `gb` target pairs per basic block (the code generator
#         materialises a constant once per block for all its uses there; over
#         a whole stage those shared constants outgrow the scalar registers)
#         and `ahead`: a block's LDS loads issued one block early
# Measured per RK4 step (us, 2^18 parcels, L = 12, FP64; the row-by-row form
# with split rows it replaced: 509): split 4: 329 with loads ahead, 339
# without; 8 waves of 256 registers, one group per CU: 413; 8 waves of 128
# registers, two groups per CU, 34 registers spilled: 338; 6 waves: 520 (they
# do not spread evenly over four SIMDs).  gb 2 / 4 / 8 / 16: 336 / 329 / 328 /
# 322.  FP32 operator, L = 12: split 4 with loads ahead 181 against 217.
# L = 8 FP64, ten-step launches, v1 .. v7: 20,000 parcels 23.3 23.2 26.3 34.7
# 23.1 22.0 25.1, 2^18 parcels 150 147 200 190 149 161 156; one-step launches of
# 2^20 parcels 739 788 1,151 900 730 869 816: three waves per SIMD (v5) and two
# eight-wave groups per CU (v6) win by up to 5 % in between and are left to the
# autotuner, two waves per group (v4) and no loads ahead (v7) are the other ends
# of what it compares.  lit is three to five times slower throughout.
# L = 20 FP64 holds one group per CU (its stage input takes 118 KB of LDS):
# eight waves, no registers left for loads ahead: 1,053 against 1,202.
LIT = dict(mode="lit", chunk=8, waves=2, block=64)
Pr = lambda split, waves, gb, ahead=True: dict(mode="pair", split=split, waves=waves, gb=gb, ahead=ahead,
                                               block=64 * split)


def variants(L, prec):
    """(variants, index for large batches, index for small ones)."""
    if prec == "f64":
        if L >= 18:
            return [Pr(8, 2, 3, False), Pr(8, 2, 6, False), Pr(8, 2, 32, False)], 2, 2
        if L >= 14:
            return [Pr(8, 2, 8)], 0, 0
        vs = [Pr(4, 2, 16), Pr(8, 2, 8)]
        if L == 12:
            return [LIT, Pr(4, 2, 8)] + vs, 2, 3
        if L == 8:
            return [LIT, Pr(4, 2, 8)] + vs + [Pr(2, 2, 8), Pr(4, 3, 8), Pr(8, 4, 8), Pr(4, 2, 6, False)], 2, 3
        return vs, 0, 1
    if L >= 18:
        return [Pr(16, 4, 64), Pr(12, 3, 64), Pr(8, 2, 64)], 0, 0
    return [Pr(4, 2, 64), Pr(8, 4, 64), Pr(4, 3, 64)], 0, 1


def dump(L, exe):
    out = subprocess.check_output([exe, str(L)]).decode().split("\n")
    L_, n, nrows, ngroups, nterms = map(int, out[0].split())
    rows = []
    i = 1
    while i < len(out) and out[i]:
        tok = out[i].split()
        assert tok[0] == "R"
        l, ng = int(tok[1]), int(tok[2])
        i += 1
        groups = []
        for _ in range(ng):
            g = out[i].split()
            assert g[0] == "G"
            p, nt = int(g[1]), int(g[2])
            i += 1
            terms = []
            for _ in range(nt):
                t = out[i].split()
                terms.append((int(t[1]), int(t[2]), float.fromhex(t[3])))
                i += 1
            groups.append((p, terms))
        rows.append((l, groups))
    assert len(rows) == n
    return n, rows


def lit(v, prec):
    """Exact C literal of a term value (FP32: rounded to float)."""
    if prec == "f64":
        return "(%s)" % float(v).hex()
    import struct
    f = struct.unpack("f", struct.pack("f", v))[0]
    return "(%sf)" % float(f).hex()


def gen_kernel(L, prec, n, rows, cfg, vid):
    """Row-by-row stepper ("lit" mode): per output row and parameter one FMA
    per coupling value, x (n FP64 values) in registers, the step-start state,
    the RK increment sum YS and the next-stage input XN in SoA buffers."""
    assert prec == "f64"
    name = "evolve_fast_L%d_%s_v%d" % (L, prec, vid)
    CHUNK, B = cfg["chunk"], cfg["block"]
    used_p = sorted({p for (_, gs) in rows for (p, _) in gs})
    pidx = {q: i for i, q in enumerate(used_p)}
    nq = min(n, 15)
    nblk = L // 2 + 1
    o = []
    w = o.append
    w("// Generated by specfab_amd/tables/gen_fast.py -- do not edit.")
    w("// Row-by-row stepper, L = %d (n = %d), FP64; variant %d: %s." %
      (L, n, vid, ", ".join("%s=%s" % kv for kv in sorted(cfg.items()))))
    w('#include "../sfg_kernels.h"')
    w("namespace sfg {")
    w("__global__ void __launch_bounds__(%d, %d) %s(EvolveArgs a) {" % (B, cfg["waves"], name))
    w("    const int64_t P = a.P;")
    w("    const int64_t p = (int64_t)blockIdx.x * %d + threadIdx.x;" % B)
    w("    if (p >= P) return;")
    w("    // SoA rows through buffer resources: row r of an array is at byte")
    w("    // r * P * 8 [scalar] + p * 8 [one lane offset]")
    w("    const uint32_t P8 = (uint32_t)P * 8u, v8 = (uint32_t)p * 8u;")
    w("    const sfg_rsrc RX = make_rsrc(a.X, P8 * %du);" % n)
    w("    const sfg_rsrc RYS = make_rsrc(a.YS, P8 * %du);" % n)
    w("    const sfg_rsrc RXN = make_rsrc(a.XA, P8 * %du);" % n)
    w("    const sfg_rsrc ROM = make_rsrc(a.omega, P8 * 15u);")
    w("    const sfg_rsrc RSL = make_rsrc(a.sl, P8 * %du);" % nblk)
    w("    const int nstage = a.scheme ? 4 : 1;")
    w("    const int rem = a.steps ? a.steps[p] : a.nsteps;")
    w("    const int ns = (a.steps && a.steps_dec) ? (rem < a.nsteps ? rem : a.nsteps) : rem;")
    w("    const double h = a.dt;")
    w("    // per-parcel operator parameters in LDS ([param][lane]), read once per")
    w("    // (row chunk, parameter)")
    w("    __shared__ double thl[%d][%d];" % (len(used_p), B))
    for q in used_p:
        w("    thl[%d][threadIdx.x] = a.theta[(int64_t)%d * P + p];" % (pidx[q], q))
    w("    double %s;" % ", ".join("x%d" % b for b in range(n)))
    w("    for (int step = 0; step < ns; step++) {")
    for b in range(n):
        w("        x%d = bld64(RX, v8, %du * P8);" % (b, b))
    w("        for (int s = 0; s < nstage; s++) {")
    w("            const bool first = (s == 0), last = (s == nstage - 1), euler = (nstage == 1);")
    w("            // a.zero is 0 at run time but unknown to the compiler: it keeps the")
    w("            // LDS parameter reads of different row chunks apart")
    w("            const int z = (int)a.zero * (step * 4 + s);")
    w("            const double cy = euler ? h : ((s == 0 || s == 3) ? h / 6 : h / 3);")
    w("            const double cx = (s == 2) ? h : h / 2;")
    w("            double gD = 0.0;")
    w("            if (a.use_ddrx) {")
    w("                gD = (%s) / x0;" % " + ".join("bld64(ROM, v8, %du * P8) * x%d" % (q, q) for q in range(nq)))
    w("            }")
    for c0 in range(0, n, CHUNK):
        chunk = list(range(c0, min(n, c0 + CHUNK)))
        w("            {   // rows %d..%d" % (chunk[0], chunk[-1]))
        w("                double %s;" % ", ".join("acc%d = 0.0" % r for r in chunk))
        byp = {}
        for r in chunk:
            for (pp, tl) in rows[r][1]:
                byp.setdefault(pp, []).append((r, tl))
        for pp in sorted(byp):
            w("                {")
            w("                    const double th = thl[%d][threadIdx.x + z * %d];" % (pidx[pp], c0 // CHUNK + 1))
            for (r, tl) in byp[pp]:
                col, ti, v = tl[0]
                w("                    double u%d = %s * x%d;" % (r, lit(v, prec), col))
                for (col, ti, v) in tl[1:]:
                    w("                    u%d = fma(%s, x%d, u%d);" % (r, lit(v, prec), col, r))
                w("                    acc%d = fma(th, u%d, acc%d);" % (r, r, r))
            w("                }")
        for r in chunk:
            l = rows[r][0]
            w("                {")
            w("                    const double f = fma(bld64(RSL, v8, %du * P8) - gD, x%d, acc%d);" % (l // 2, r, r))
            w("                    const double x0a = bld64(RX, v8, %du * P8);" % r)
            w("                    if (euler) {")
            w("                        bst64(RX, v8, %du * P8, x0a + cy * f);" % r)
            w("                    } else {")
            w("                        const double ys = first ? cy * f : fma(cy, f, bld64(RYS, v8, %du * P8));" % r)
            w("                        if (last) {")
            w("                            bst64(RX, v8, %du * P8, x0a + ys);" % r)
            w("                        } else {")
            w("                            bst64(RYS, v8, %du * P8, ys);" % r)
            w("                            bst64(RXN, v8, %du * P8, fma(cx, f, x0a));" % r)
            w("                        }")
            w("                    }")
            w("                }")
        w("            }")
    w("            if (!last) {")
    for b in range(n):
        w("                x%d = bld64(RXN, v8, %du * P8);" % (b, b))
    w("            }")
    w("        }")
    w("    }")
    w("    if (a.steps && a.steps_dec) a.steps[p] = rem - ns;")
    w("    if (a.status) {")
    w("        int st = 0;")
    w("        for (int r = 0; r < %d; r++) st |= isfinite(bld64(RX, v8, (uint32_t)r * P8)) ? 0 : 1;" % n)
    w("        a.status[p] |= st;")
    w("    }")
    w("}")
    w("#ifndef SFG_HOST_EMUL")
    w("hipError_t launch_%s(const EvolveArgs& a, hipStream_t s) {" % name)
    w("    hipLaunchKernelGGL(%s, dim3((unsigned)((a.P + %d) / %d)), dim3(%d), 0, s, a);" % (name, B - 1, B, B))
    w("    return hipGetLastError();")
    w("}")
    w("#endif")
    w("}  // namespace sfg")
    return "\n".join(o) + "\n"


# (l, m, part) couples: real index of each row pair, and the parameter pairs
# (real, imaginary) of the operator's complex weights with their harmonic order
PARAM_PAIRS = ((0, None), (1, 2), (3, 4), (5, None), (6, 7), (8, None), (9, None), (10, 11), (12, 13), (14, None),
               (15, 16), (17, 18), (19, 20), (21, 22))


def row_pairs(L):
    """(l, m, real row, imaginary row or None) in state order."""
    out, i = [], 0
    for l in range(0, L + 1, 2):
        for m in range(l + 1):
            out.append((l, m, i, i + 1 if m else None))
            i += 1 if m == 0 else 2
    return out


def pair_blocks(L, rows):
    """The operator as couplings of complex coefficients.

    Every coupling value of a row pair (Re, Im of n_l^m), a weight pair (Re,
    Im of theta_k) and a source pair (Re, Im of n_l'^m') occurs up to four
    times with one magnitude, since the products are real times complex times
    complex: {(target, m'): [(k, cells, {l': value})]}, where cells maps
    (row part, weight part, source part) to its sign relative to the value,
    the same for every l' of the entry (checked)."""
    lp = row_pairs(L)
    R = [{p: {c: v for c, _, v in tl} for p, tl in gs} for _, gs in rows]
    blocks, found = {}, 0
    for t, (l, m, a, b) in enumerate(lp):
        for k, (p, q) in enumerate(PARAM_PAIRS):
            for (l2, m2, c, d) in lp:
                cells = {}
                for rp, r in ((0, a), (1, b)):
                    for wp, w in ((0, p), (1, q)):
                        for cp, col in ((0, c), (1, d)):
                            v = None if None in (r, w, col) else R[r].get(w, {}).get(col)
                            if v is not None:
                                cells[rp, wp, cp] = v
                if not cells:
                    continue
                found += len(cells)
                first = cells[min(cells)]
                if any(abs(v) != abs(first) for v in cells.values()):
                    raise ValueError("coupling of (%d,%d) to (%d,%d) is not a complex product" % (l, m, l2, m2))
                sg = {x: (1 if v == first else -1) for x, v in cells.items()}
                ent = blocks.setdefault((t, m2), {}).setdefault(k, (sg, {}))
                if ent[0] != sg:
                    raise ValueError("coupling signs of (%d,%d) differ over l'" % (l, m))
                ent[1][l2] = first
    if found != sum(len(tl) for _, gs in rows for _, tl in gs):
        raise ValueError("couplings outside the known weight pairs")
    return lp, {key: [(k, sg, d) for k, (sg, d) in sorted(v.items())] for key, v in blocks.items()}


def weight_cells(sg):
    """{(row part, source part): (weight part, sign, anchor, sign relative to
    the anchor)}: cells with the same weight part share the weight of their
    first cell, the anchor, up to a sign; and the key of entries whose weights
    may be added (the same cells, anchors and relative signs)."""
    W = {(r, c): (w, s) for (r, w, c), s in sg.items()}
    out = {}
    for x in sorted(W):
        an = min(y for y in W if W[y][0] == W[x][0])
        out[x] = (W[x][0], W[x][1], an, W[x][1] * W[an][1])
    return out, tuple((x, v[2], v[3]) for x, v in sorted(out.items()))


def block_plan(entries):
    """How one (target pair, m') block is evaluated: entries (k, cells, {l':
    c}) are covered either by weight k (the source sum over l' first, then the
    product with theta_k) or by source l' (the weights sum over k first, then
    the product with the source), whichever needs fewer products: a minimum
    vertex cover of the (k, l') pairs, per class of entries whose weights may
    be added.  Returns ([entries summed over l'], [(class cells, l', [(k,
    cells, c)])])."""
    import itertools
    classes = {}
    for e in entries:
        classes.setdefault(weight_cells(e[1])[1], []).append(e)
    byk, byl = [], []
    for es in classes.values():
        best = None
        for r in range(len(es) + 1):
            for S in itertools.combinations(range(len(es)), r):
                rest = sorted({l for i, e in enumerate(es) if i not in S for l in e[2]})
                if best is None or r + len(rest) < best[0]:
                    best = (r + len(rest), S, rest)
        _, S, rest = best
        for i, e in enumerate(es):
            if i in S:
                byk.append(e)
        for l in rest:
            byl.append((es[0][1], l, [(e[0], e[1], e[2][l]) for i, e in enumerate(es) if i not in S and l in e[2]]))
    return byk, byl


def block_cost(plan):
    byk, byl = plan
    c = 0
    for k, sg, d in byk:
        c += len(d) * len({x[2] for x in sg}) + len(sg)
    for sg, l, ks in byl:
        W, _ = weight_cells(sg)
        c += len(ks) * len({v[2] for v in W.values()}) + len(W)
    return c


def gen_kernel_pair(L, prec, n, rows, cfg, vid):
    """Split resident stepper over complex couplings ("pair" mode).

    S waves share one group of 64 parcels (one per lane); the state and the RK
    increment sums of a wave's row pairs (Re, Im of n_l^m, sorted by m and
    split by operation count) stay in its registers over the whole launch, the
    stage input of the group lives in LDS.  A stage walks the source orders m'
    that couple to the wave's pairs (|m - m'| <= 4 or m + m' <= 4): it loads
    the columns of one m' from LDS once and adds their contribution to all of
    the wave's pairs.  Couplings are evaluated as real values times complex
    coefficients times complex weights (pair_blocks), so that one constant
    serves the real and the imaginary part and the sum over l' is formed once
    for both rows of a pair (or the weights once, block_plan): 0.73 of the
    FP64 instructions of the row-by-row form at L = 12 and 0.3 of its
    constants.  The last wave also forms Gamma0 <D>, which the others read
    after the stage's first barrier.  launch_bounds' second number (cfg
    "waves") sets the registers per wave, and with them how many groups a CU
    holds: with two, one group's barriers and LDS loads hide behind the
    other's arithmetic.
    """
    F64 = prec == "f64"
    T = "double" if F64 else "float"
    cv = (lambda e: e) if F64 else (lambda e: "(float)(%s)" % e)
    zero = "0.0" if F64 else "0.0f"
    S = cfg["split"]
    B = 64 * S
    name = "evolve_fast_L%d_%s_v%d" % (L, prec, vid)
    lp, blocks = pair_blocks(L, rows)
    plans = {key: block_plan(v) for key, v in blocks.items()}
    nq, nblk, NPU = min(n, 15), L // 2 + 1, 23
    OMC, SLC = NPU + nblk, NPU
    order = sorted(range(len(lp)), key=lambda t: (lp[t][1], lp[t][0]))
    cost = {t: sum(block_cost(pl) for (tt, _), pl in plans.items() if tt == t) + 8 * (1 if lp[t][3] is None else 2)
            for t in order}

    # contiguous shares of the order with the least largest cost; the last
    # wave's extra work is <D>
    def split(limit):
        out, cur, acc = [], [], 0
        for t in order:
            extra = 60 if len(out) == S - 1 else 0
            if cur and acc + cost[t] + extra > limit and len(out) < S - 1:
                out.append(cur)
                cur, acc = [], 0
            cur.append(t)
            acc += cost[t]
        out.append(cur)
        worst = max(sum(cost[t] for t in s) + (60 if i == S - 1 else 0) for i, s in enumerate(out))
        return out, worst
    shares = min((split(lim) for lim in range(max(cost.values()), sum(cost.values()) + 64,
                                              max(1, sum(cost.values()) // 400))), key=lambda r: r[1])[0]
    shares += [[] for _ in range(S - len(shares))]
    srcs = {}
    for (l2, m2, c, d) in lp:
        srcs.setdefault(m2, []).append((l2, c, d))
    o = []
    w = o.append
    w("// Generated by specfab_amd/tables/gen_fast.py -- do not edit.")
    w("// Split resident stepper over complex couplings, L = %d (n = %d), %s; variant %d: %s; operations per share %s." %
      (L, n, "FP64" if F64 else "FP32 stepping, FP64 state", vid, ", ".join("%s=%s" % kv for kv in sorted(cfg.items())),
       ", ".join(str(sum(cost[t] for t in s)) for s in shares)))
    w('#include "../sfg_kernels.h"')
    w("namespace sfg {")
    w("__global__ void __launch_bounds__(%d, %d) %s(EvolveArgs a) {" % (B, cfg["waves"], name))
    w("    const int64_t P = a.P;")
    w("    const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;   // wv is uniform per wave")
    w("    const int64_t p = (int64_t)blockIdx.x * 64 + lane;")
    w("    const bool valid = p < P;")
    w("    const uint32_t P8 = (uint32_t)P * 8u;")
    w("    // lanes past the batch stay for the barriers: loads return 0, stores are dropped")
    w("    const uint32_t v8 = valid ? (uint32_t)p * 8u : 0x80000000u;")
    w("    const sfg_rsrc RX = make_rsrc(a.X, P8 * %du);" % n)
    w("    const int nstage = a.scheme ? 4 : 1;")
    w("    const int rem = valid ? (a.steps ? a.steps[p] : a.nsteps) : 0;")
    w("    const int ns = (a.steps && a.steps_dec) ? (rem < a.nsteps ? rem : a.nsteps) : rem;")
    w("    const double h = a.dt;")
    w("    // launch constants ([column][lane]: theta_p, s_l, omega_q), Gamma0 <D> and the stage input")
    w("    __shared__ %s thl[%d][64];" % (T, NPU + nblk + nq))
    w("    __shared__ %s gs[64];" % T)
    w("    __shared__ %s xs[%d][64];" % (T, n))
    cols = [("a.theta", q, q) for q in range(NPU)] + [("a.sl", b, SLC + b) for b in range(nblk)] + \
           [("a.omega", q, OMC + q) for q in range(nq)]
    for k in range(S):
        w("    %sif (wv == %d && valid) {" % ("" if k == 0 else "} else ", k))
        for (arr, q, c) in cols[k::S]:
            w("        thl[%d][lane] = %s;" % (c, cv("%s[(int64_t)%d * P + p]" % (arr, q))))
    w("    }")
    uid = [0]

    def nid():
        uid[0] += 1
        return uid[0]

    def val(v):
        return lit(v, prec)

    def emit_block(t, m2, ind, tag):
        """accumulate block (t, m2) into acc{row}; the columns are c{row}"""
        l, m, a, b = lp[t]
        byk, byl = plans[t, m2]
        col = {l2: (c, d) for (l2, c, d) in srcs[m2]}
        rowof = (a, b)
        for k, sg, d in byk:
            u = nid()
            parts = sorted({x[2] for x in sg})
            for j, (l2, c) in enumerate(sorted(d.items())):
                for cp in parts:
                    src = "c%d" % col[l2][cp]
                    if j == 0:
                        w("%s%s u%d_%d = %s * %s;" % (ind, T, u, cp, val(c), src))
                    else:
                        w("%su%d_%d = fma(%s, %s, u%d_%d);" % (ind, u, cp, val(c), src, u, cp))
            for (rp, wp, cp), s in sorted(sg.items()):
                th = "th%d%s" % (PARAM_PAIRS[k][wp], tag)
                w("%sacc%d = fma(%s%s, u%d_%d, acc%d);" % (ind, rowof[rp], "-" if s < 0 else "", th, u, cp, rowof[rp]))
        for sg, l2, ks in byl:
            W, _ = weight_cells(sg)
            u = nid()
            anchors = sorted({v[2] for v in W.values()})
            for i, an in enumerate(anchors):
                for j, (k, sgk, c) in enumerate(ks):
                    wp, sk = weight_cells(sgk)[0][an][:2]
                    th = "th%d%s" % (PARAM_PAIRS[k][wp], tag)
                    if j == 0:
                        w("%s%s w%d_%d = %s * %s;" % (ind, T, u, i, val(sk * c), th))
                    else:
                        w("%sw%d_%d = fma(%s, %s, w%d_%d);" % (ind, u, i, val(sk * c), th, u, i))
            for (rp, cp), (_, _, an, sign) in sorted(W.items()):
                w("%sacc%d = fma(%sw%d_%d, c%d, acc%d);" % (ind, rowof[rp], "-" if sign < 0 else "", u,
                                                          anchors.index(an), col[l2][cp], rowof[rp]))

    for sh, mine in enumerate(shares):
        myrows = [r for t in mine for r in lp[t][2:] if r is not None]
        w("    %sif (wv == %d) {" % ("" if sh == 0 else "} else ", sh))
        for r in myrows:
            w("        double s%d = bld64(RX, v8, %du * P8);" % (r, r))
            w("        xs[%d][lane] = %s;" % (r, cv("s%d" % r)))
        if myrows:
            w("        %s %s;" % (T, ", ".join("y%d = %s" % (r, zero) for r in myrows)))
        w("        __syncthreads();")
        w("        for (int step = 0; step < ns; step++) {")
        w("            for (int s = 0; s < nstage; s++) {")
        w("                const bool last = (s == nstage - 1);")
        w("                const %s cy = %s;" % (T, cv("(nstage == 1) ? h : ((s == 0 || s == 3) ? h / 6 : h / 3)")))
        w("                const %s cx = %s;" % (T, cv("(s == 2) ? h : h / 2")))
        w("                // a.zero is 0 at run time but unknown to the compiler: z keeps the LDS")
        w("                // reads of different blocks apart and bounds the basic blocks")
        w("                const int z = (int)a.zero * (step * 4 + s);")
        if sh == S - 1:
            w("                {")
            w("                    %s g = %s;" % (T, zero))
            w("                    if (a.use_ddrx)")
            w("                        g = (%s) / xs[0][lane];" % " + ".join(
                "thl[%d][lane] * xs[%d][lane]" % (OMC + q, q) for q in range(nq)))
            w("                    gs[lane] = g;")
            w("                }")
        if myrows:
            w("                %s %s;" % (T, ", ".join("acc%d = %s" % (r, zero) for r in myrows)))
        # units: the targets of one m against one source order m'; a unit's
        # columns and weights are loaded while the previous unit computes
        units = []
        for m2 in sorted(srcs):
            todo = [t for t in mine if (t, m2) in plans]
            cols_in = sorted({r for t in todo for k, sg, d in blocks[t, m2] for l2 in d for (ll, c, dd) in srcs[m2]
                              if ll == l2 for r in ({c, dd} if dd is not None else {c})})
            for m in sorted({lp[t][1] for t in todo}):
                grp = [t for t in todo if lp[t][1] == m]
                ths = sorted({PARAM_PAIRS[k][x[1]] for t in grp for k, sg, d in blocks[t, m2] for x in sg})
                units.append((m2, m, grp, cols_in, ths))
                cols_in = []
        cnt = 0

        def loads(i):
            m2, m, grp, cols_in, ths = units[i]
            w("                const int lo%d = lane + z * %d;" % (i, nid()))
            if cols_in:
                w("                const %s %s;" % (T, ", ".join("c%d = xs[%d][lo%d]" % (r, r, i) for r in cols_in)))
            w("                const %s %s;" % (T, ", ".join("th%d_%d = thl[%d][lo%d]" % (q, i, q, i) for q in ths)))

        if units and cfg["ahead"]:
            loads(0)
        for i, (m2, m, grp, _, ths) in enumerate(units):
            if not cfg["ahead"]:
                loads(i)
            elif i + 1 < len(units):
                loads(i + 1)
            w("                {   // m = %d from m' = %d" % (m, m2))
            dirty = []
            for t in grp:
                w("                    {   // (%d, %d)" % lp[t][:2])
                emit_block(t, m2, "                        ", "_%d" % i)
                w("                    }")
                cnt += 1
                dirty += [r for r in lp[t][2:] if r is not None]
                if cnt % cfg["gb"] == 0 or t == grp[-1]:
                    # the sums so far are used here: the compiler cannot move their
                    # arithmetic past the block, away from the loads
                    for d0 in range(0, len(dirty), 14):
                        w("                    if (z) asm volatile(\"\" :: %s);" %
                          ", ".join('"v"(acc%d)' % r for r in dirty[d0:d0 + 14]))
                    dirty = []
            w("                }")
        w("                __syncthreads();   // every wave has read the stage input; gs is written")
        if myrows:
            w("                {")
            w("                    const int lo = lane + z * %d;" % nid())
            w("                    const %s gD = gs[lane];" % T)
            if F64:
                w("                    const double lastf = last ? 1.0 : 0.0, keepf = last ? 0.0 : 1.0, cxe = last ? 0.0 : cx;")
            for t in mine:
                l = lp[t][0]
                w("                    {")
                w("                        const %s d = thl[%d][lo] - gD;" % (T, SLC + l // 2))
                for r in [r for r in lp[t][2:] if r is not None]:
                    w("                        {")
                    w("                            const %s f = fma(d, xs[%d][lo], acc%d);" % (T, r, r))
                    w("                            const %s yv = fma(cy, f, y%d);" % (T, r))
                    if F64:
                        # s + yv in the last stage (fma with 1: one rounding), s unchanged before it;
                        # the next stage input s + cx f before the last stage, the new state in it
                        w("                            s%d = fma(yv, lastf, s%d);" % (r, r))
                        w("                            y%d = yv * keepf;" % r)
                        w("                            xs[%d][lane] = fma(cxe, f, s%d);" % (r, r))
                    else:
                        w("                            s%d = last ? s%d + (double)yv : s%d;" % (r, r, r))
                        w("                            y%d = last ? 0.0f : yv;" % r)
                        w("                            xs[%d][lane] = last ? (float)s%d : fma(cx, f, (float)s%d);" % (r, r, r))
                    w("                        }")
                w("                    }")
            w("                }")
        w("                __syncthreads();   // the next stage input is complete")
        w("            }")
        w("        }")
        if myrows:
            w("        int st = 0;")
            for r in myrows:
                w("        bst64(RX, v8, %du * P8, s%d); st |= isfinite(s%d) ? 0 : 1;" % (r, r, r))
            w("        if (a.status && valid && st) atomicOr(a.status + p, st);")
    w("    }")
    w("    if (wv == 0 && valid && a.steps && a.steps_dec) a.steps[p] = rem - ns;")
    w("}")
    w("#ifndef SFG_HOST_EMUL")
    w("hipError_t launch_%s(const EvolveArgs& a, hipStream_t s) {" % name)
    w("    hipLaunchKernelGGL(%s, dim3((unsigned)((a.P + 63) / 64)), dim3(%d), 0, s, a);" % (name, B))
    w("    return hipGetLastError();")
    w("}")
    w("#endif")
    w("}  // namespace sfg")
    return "\n".join(o) + "\n"


def gen_dispatch(kinds):
    """kinds: list of (L, prec, variant configs, large, small)."""
    pn = lambda prec: 0 if prec == "f64" else 1
    o = ["// Generated by specfab_amd/tables/gen_fast.py -- do not edit.",
         '#include "../sfg_fast.h"', "namespace sfg {"]
    for (L, prec, cfgs, _, _) in kinds:
        for v in range(len(cfgs)):
            o.append("hipError_t launch_evolve_fast_L%d_%s_v%d(const EvolveArgs& a, hipStream_t s);" % (L, prec, v))
    o.append("int fast_variants(int L, int prec) {")
    for (L, prec, cfgs, _, _) in kinds:
        o.append("    if (L == %d && prec == %d) return %d;" % (L, pn(prec), len(cfgs)))
    o.append("    return 0;")
    o.append("}")
    o.append("int fast_default(int L, int prec, int64_t P) {")
    for (L, prec, _, large, small) in kinds:
        o.append("    if (L == %d && prec == %d) return P <= FAST_SMALL ? %d : %d;" % (L, pn(prec), small, large))
    o.append("    return 0;")
    o.append("}")
    o.append("#ifndef SFG_HOST_EMUL")
    for (L, prec, cfgs, _, _) in kinds:
        for v in range(len(cfgs)):
            o.append("__global__ void evolve_fast_L%d_%s_v%d(EvolveArgs a);" % (L, prec, v))
    o.append("const void* fast_kernel(int L, int prec, int variant, int* block, int* parcels) {")
    for (L, prec, cfgs, _, _) in kinds:
        for v, cfg in enumerate(cfgs):
            o.append("    if (L == %d && prec == %d && variant == %d) { *block = %d; *parcels = 64; "
                     "return (const void*)&evolve_fast_L%d_%s_v%d; }" % (L, pn(prec), v, cfg["block"], L, prec, v))
    o.append("    return nullptr;")
    o.append("}")
    o.append("#endif")
    o.append("int fast_buffers(int L, int prec, int variant) {")
    for (L, prec, cfgs, _, _) in kinds:
        for v, cfg in enumerate(cfgs):
            if cfg["mode"] == "lit":
                o.append("    if (L == %d && prec == %d && variant == %d) return BUF_YS | BUF_XA;" % (L, pn(prec), v))
    o.append("    return 0;   // the state stays in registers and LDS")
    o.append("}")
    o.append("hipError_t launch_evolve_fast(int L, int prec, int variant, const EvolveArgs& a, hipStream_t s) {")
    o.append("    if (a.P == 0) return hipSuccess;")
    for (L, prec, cfgs, _, _) in kinds:
        for v in range(len(cfgs)):
            o.append("    if (L == %d && prec == %d && variant == %d) return launch_evolve_fast_L%d_%s_v%d(a, s);"
                     % (L, pn(prec), v, L, prec, v))
    o.append("    return hipErrorInvalidValue;")
    o.append("}")
    o.append("}  // namespace sfg")
    return "\n".join(o) + "\n"


def gen_moment_maps(exe):
    """Mandel a2 / a4 of the l <= 4 block of a state as literal FMAs over the
    maps' nonzero coefficients (in increasing row order, so the sums equal
    those of a loop over all 15 rows)."""
    a2, a4 = {}, {}
    for line in subprocess.check_output([exe, "maps"]).decode().split("\n"):
        if not line:
            continue
        tag, i, q, v = line.split()
        (a2 if tag == "A2" else a4).setdefault(int(i), []).append((int(q), float.fromhex(v)))
    o = ["// Generated by specfab_amd/tables/gen_fast.py -- do not edit.",
         "// Mandel a2 and a4 of the l <= 4 block of a real-basis state x (xq[q] = row q):",
         "// a2v[i] = a2s[i] / x0 + (i < 3 ? 1/3 : 0), a4v[i][j] = a4s[i][j] / x0, with the",
         "// nonzero coefficients of the maps of src/moments.f90:164-178 as literals.",
         "#pragma once", "namespace sfg {",
         "__device__ __forceinline__ void moment_maps(const double (&xq)[15], double (&a2s)[6], double (&a4s)[6][6]) {"]
    for i in range(6):
        terms = sorted(a2.get(i, []))
        o.append("    { double s = 0.0;" + "".join(" s = fma(%s, xq[%d], s);" % (v.hex(), q) for q, v in terms)
                 + " a2s[%d] = s; }" % i)
    for i in range(6):
        for j in range(i, 6):
            terms = sorted(a4.get(6 * i + j, []))
            assert terms == sorted(a4.get(6 * j + i, [])), "a4 map not symmetric"
            o.append("    { double s = 0.0;" + "".join(" s = fma(%s, xq[%d], s);" % (v.hex(), q) for q, v in terms)
                     + " a4s[%d][%d] = s;%s }" % (i, j, "" if i == j else " a4s[%d][%d] = s;" % (j, i)))
    o.append("}")
    o.append("}  // namespace sfg")
    return "\n".join(o) + "\n"


def write_if_changed(path, text):
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path + ".tmp", "w") as f:
        f.write(text)
    os.replace(path + ".tmp", path)


def main():
    outdir = sys.argv[1]
    os.makedirs(outdir, exist_ok=True)
    exe = os.path.join(outdir, "dump_basis")
    srcs = [os.path.join(HERE, "dump_basis.cpp"), os.path.join(CSRC, "sfg_basis.cpp")]
    if not os.path.exists(exe) or any(os.path.getmtime(s) > os.path.getmtime(exe) for s in srcs):
        subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, "-I", outdir] + srcs + ["-o", exe])
    kinds = []
    for prec in ("f64", "f32"):
        for L in FAST_L:
            n, rows = dump(L, exe)
            vs, large, small = variants(L, prec)
            for vid, cfg in enumerate(vs):
                gen = gen_kernel_pair if cfg["mode"] == "pair" else gen_kernel
                write_if_changed(os.path.join(outdir, "sfg_fast_L%d_%s_v%d.hip" % (L, prec, vid)),
                                 gen(L, prec, n, rows, cfg, vid))
            kinds.append((L, prec, vs, large, small))
    # drop generated kernels of an older variant list
    keep = {"sfg_fast_L%d_%s_v%d.hip" % (L, prec, v) for (L, prec, cfgs, _, _) in kinds for v in range(len(cfgs))}
    for f in os.listdir(outdir):
        if f.startswith("sfg_fast_L") and f.endswith(".hip") and f not in keep:
            os.remove(os.path.join(outdir, f))
    write_if_changed(os.path.join(outdir, "sfg_fast_dispatch.hip"), gen_dispatch(kinds))
    write_if_changed(os.path.join(outdir, "sfg_moment_maps.h"), gen_moment_maps(exe))
    print("generated %d fast kernels" % sum(len(k[2]) for k in kinds))


if __name__ == "__main__":
    main()
