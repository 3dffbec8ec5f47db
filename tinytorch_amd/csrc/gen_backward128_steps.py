#!/usr/bin/env python3
"""Writes backward128_steps.inc: the hand-ordered instruction streams of the head_dim-128 attention backward
(sdpa_backward_d128.hip), one string per (tile of the unrolled body, element type).

    python3 gen_backward128_steps.py > backward128_steps.inc

As in the forward (gen_prefill128_steps.py) a stream is a fixed sequence of slots, one matrix instruction each, with the vector work
spread over them so that no instruction waits for the one before it, and the LDS operand of the slot PD places ahead requested
into a ring of operand registers.

dq, a step of key tile i (32 keys), 24 slots:
    0 .. 7    dq^T += K(i-1)^T . dS(i-1)    (two key steps of 16 x four head_dim blocks)
    8 .. 23   S^T(i+1) = K(i+1) . Q^T and dP^T(i+1) = V(i+1) . dout^T, k-steps in turn: two chains of dependent products
while the vector ALU turns S(i) and dP(i) into dS(i): P = exp2(S c - mc), its sum, (dP - delta) P, converted in pairs into the
first eight registers of dP(i)'s accumulator.  The slots that come first read what the last two steps read, so the ring's requests
cross the barrier between steps without tile i+1 having to be in place before it.

Register plan of a lane (fixed, named in the statements' constraints by the kernel):
    v[82:87]    temporaries       v[88:91]  row operand addresses r (index k-step / 2)     v[92:95]  transposed operand addresses t
                                  (index head_dim block); LDS bytes
    v[96:127]   Q operands        v[128:159]  dout operands, 8 k-steps x 4 registers
    v[160:175], v[176:191]  S of even, odd tiles      v[192:207], v[208:223]  dP of even, odd tiles (then dS)
    v[224:255]  operand ring, 8 x 4
Named operands: o0-o3 the dq accumulators (read-write), ps the lane's sum of the step's probabilities (out), c = scale*log2(e)
(scalar register), mc = maximum*c, dl = delta of the lane's row.

dk/dv, a tile of 32 query rows against the wavefront's 32 keys (K in registers), 32 slots:
    0 .. 7    S = Q . K^T, a chain of dependent products
    8 .. 15   dP - delta = dout . V^T - delta (the chain's first accumulator)      P = exp2(S c - lse) from slot 9
    16 .. 23  dv^T += dout^T . P                                                                      dS = (dP - delta) P from slot 18
    24 .. 31  dk^T += Q^T . dS
    Fixed registers: v[128:131] addresses of V's rows, v[136:139] transposed, v[140:143] row operand addresses
    v[144:151]  lse of rows, quads 0 and 1 (2 and 3 lie in v[152:159] before P does)     v[152:159] P in pairs of 16 bits
    v[160:175]  dP (then dS)      v[176:191]  S (then P)      v[192:223]  K, 8 k-steps x 4 registers      v[224:255]  operand ring
    Named: o0-o3 dk, o4-o7 dv (read-write), c = scale*log2(e), st = the stage's start,
    adv = the next stage's from there, more = whether the step has asked for a tile (scalar registers).  One stream for all stages: with one
    each, a workgroup's first steps waited for their instructions (of 36 to 90 us on 165 to 480 rows, 2 to 5).

LDS: a tile is 8 groups of 4 rows of 256 bytes, a group every GROUP bytes (the 16 bytes between them spread the banks); chunk c of
16 bytes of row i of a group sits at slot c ^ 4i.
"""

KST, NDB = 8, 4
GROUP = 1040
TILE = 8 * GROUP
STAGES = 4          # of K and of V
PD, RING = 6, 8
T0, R0, TR0, Q0, G0, S0, D0, RING0 = 82, 88, 92, 96, 128, 160, 192, 224


def vr(lo, n=1):
    return "v%d" % lo if n == 1 else "v[%d:%d]" % (lo, lo + n - 1)


def row_operand(r, ks, base):
    """k-step ks of a tile's rows (b128): bits 1 and 2 of the k-step are in the address register."""
    return ["ds_read_b128 %s, %s offset:%d" % (vr(r, 4), vr(R0 + ks // 2), base + 32 * (ks & 1))]


def transposed_operand(r, t, db, base):
    """Rows 16t .. 16t+15, head_dim block db."""
    return ["ds_read_b64_tr_b16 %s, %s offset:%d" % (vr(r + 2 * ld, 2), vr(TR0 + db), base + (4 * t + 2 * ld) * GROUP) for ld in range(2)]


# ---- dq ------------------------------------------------------------------------------------------------------------------
DQ_SLOTS = 24


def dq_fetch(G):
    G %= DQ_SLOTS * STAGES
    u, s = G // DQ_SLOTS, G % DQ_SLOTS  # the step of tile i, i % STAGES = (u + 1) % STAGES
    r = RING0 + 4 * (G % RING)
    if s < 8:
        return transposed_operand(r, s // NDB, s % NDB, (u % STAGES) * TILE)
    ks, of_v = (s - 8) // 2, (s - 8) % 2
    return row_operand(r, ks, (STAGES if of_v else 0) * TILE + ((u + 2) % STAGES) * TILE)


def pending_after(G, fetch):
    """LDS requests issued after the operand of slot G and before slot G's matrix instruction."""
    return sum(len(fetch(g)) for g in range(G + 1, G + PD))


def spread(work, slots):
    """Vector instructions to slots by the cycles they take to issue (exponentials four times the others')."""
    cost = [4 if "v_exp" in w else 1 for w in work]
    total, at, out = sum(cost), 0, [[] for _ in range(slots)]
    for w, c in zip(work, cost):
        out[min(slots - 1, at * slots // total)].append(w)
        at += c
    return out


def dq_step(u, elem):
    mfma, cvt = "v_mfma_f32_32x32x16_%s" % elem, "v_cvt_pk_%s_f32" % elem
    cur = (u + 1) & 1  # buffers of tile i; those of i-1 and i+1 are the others
    s_cur, s_new = S0 + 16 * cur, S0 + 16 * (cur ^ 1)
    d_cur, d_new = D0 + 16 * cur, D0 + 16 * (cur ^ 1)
    F, T = [T0, T0 + 1], [T0 + 2 + i for i in range(4)]
    fma = lambda n: "v_fma_f32 %s, %s, %%[c], -%%[mc]" % (vr(F[n & 1]), vr(s_cur + n))
    pack = lambda j: "%s %s, %s, %s" % (cvt, vr(d_cur + j), vr(d_cur + 2 * j), vr(d_cur + 2 * j + 1))
    work = [fma(0)]
    for n in range(17):
        if n < 16:
            work.append("v_exp_f32 %s, %s" % (vr(T[n & 3]), vr(F[n & 1])))
            if n < 15:
                work.append(fma(n + 1))
            work.append("v_sub_f32 %s, %s, %%[dl]" % (vr(d_cur + n), vr(d_cur + n)))
        if n == 2:
            work.append("v_add_f32 %%[ps], %s, %s" % (vr(T[0]), vr(T[1])))
        elif n > 2:
            work.append("v_add_f32 %%[ps], %%[ps], %s" % vr(T[(n - 1) & 3]))
        if n >= 1:
            work.append("v_mul_f32 %s, %s, %s" % (vr(d_cur + n - 1), vr(T[(n - 1) & 3]), vr(d_cur + n - 1)))
        if n % 2 == 1 and n >= 3:
            work.append(pack((n - 3) // 2))
    work.append(pack(7))
    per_slot = spread(work, DQ_SLOTS)
    out = []
    for s in range(DQ_SLOTS):
        G = DQ_SLOTS * u + s
        r = RING0 + 4 * (G % RING)
        out.append("s_waitcnt lgkmcnt(%d)" % pending_after(G, dq_fetch))
        if s < 8:
            out.append("%s %%[o%d], %s, %s, %%[o%d]" % (mfma, s % NDB, vr(r, 4), vr(d_new + 4 * (s // NDB), 4), s % NDB))
        else:
            ks, of_v = (s - 8) // 2, (s - 8) % 2
            acc, own = (d_new, G0) if of_v else (s_new, Q0)
            out.append("%s %s, %s, %s, %s" % (mfma, vr(acc, 16), vr(r, 4), vr(own + 4 * ks, 4), "0" if ks == 0 else vr(acc, 16)))
        out += dq_fetch(G + PD)
        out += per_slot[s]
    return out


# ---- dk/dv -----------------------------------------------------------------------------------------------------------------
KV_SLOTS = 32
KV, KTR, KR, KL, KPB, KD, KS, KK = 128, 136, 140, 144, 152, 160, 176, 192
# operands of a step in the order of their use: the slots' counts
KV_OPS = [1] * 8 + [2] * 8 + [1] * 16
KV_ENTRIES = sum(KV_OPS)  # a multiple of RING: the same registers in every step


# All reads of the step's tile have arrived, and so has the next tile (what was asked for last, %[more], may still be on its way: five
# loads of a wavefront); the next tile's first operands follow.
KV_BARRIER, KV_NEXT = 28, {28: 2, 29: 3, 30: 5, 31: 6}
KV_SYNC = ["s_cmp_lg_u32 %[more], 0", "s_cbranch_scc1 1f", "s_waitcnt vmcnt(0)", "1:", "s_waitcnt vmcnt(5) lgkmcnt(0)", "s_barrier"]


def kv_row(r, address, ks, base):
    return "ds_read_b128 %s, %s offset:%d" % (vr(r, 4), vr(address), base + 32 * (ks & 1))


def kv_fetch(e):
    """Requests of entry e of a step (entries behind the last are the next one's: the addresses have moved on by then)."""
    e %= KV_ENTRIES
    r = RING0 + 4 * (e % RING)
    if e < 8:
        return [kv_row(r, KR + e // 2, e, 0)]
    if e < 24:
        ks, of_v = (e - 8) // 2, (e - 8) % 2
        if not of_v:
            return [kv_row(r, KR + ks // 2, ks, TILE)]
        return [kv_row(r, KV + ks // 2, ks, 0)]
    t, db = (e - 24) % 8 // NDB, e % NDB
    tile = TILE if e < 32 else 0
    return ["ds_read_b64_tr_b16 %s, %s offset:%d" % (vr(r + 2 * ld, 2), vr(KTR + db), tile + (4 * t + 2 * ld) * GROUP) for ld in range(2)]


def kv_statistics():
    """Requests of the row statistics, by slot: lse's four quads, -delta into dP's accumulator (their address in one of its registers)."""
    at, adr = 2 * TILE, KD + 12
    lse = ["ds_read_b128 %s, v%d offset:%d" % (vr(r, 4), adr, at + 32 * q) for q, r in enumerate((KL, KL + 4, KPB, KPB + 4))]
    delta = ["ds_read_b128 %s, v%d offset:%d" % (vr(KD + 4 * q, 4), adr, at + 128 + 32 * q) for q in range(4)]
    address = ["v_mbcnt_lo_u32_b32 v%d, -1, 0" % adr, "v_bfe_u32 v%d, v%d, 5, 1" % (adr, adr), "v_lshl_add_u32 v%d, v%d, 4, %%[st]" % (adr, adr)]
    return {1: address + lse[:1], 2: lse[1:2], 3: lse[2:], 4: delta[:1], 5: delta[1:2], 6: delta[2:]}


def kv_vector_work(elem):
    """The vector instructions of the slots."""
    cvt = "v_cvt_pk_%s_f32" % elem
    lse = [KL, KPB]
    fma = lambda n: "v_fma_f32 %s, %s, %%[c], -%s" % (vr(KS + n), vr(KS + n), vr(lse[n // 8] + n % 8))
    exp = lambda n: "v_exp_f32 %s, %s" % (vr(KS + n), vr(KS + n))
    mul = lambda n: "v_mul_f32 %s, %s, %s" % (vr(KD + n), vr(KD + n), vr(KS + n))
    pack = lambda to, frm, j: "%s %s, %s, %s" % (cvt, vr(to + j), vr(frm + 2 * j), vr(frm + 2 * j + 1))
    p, ds = lambda j: pack(KPB, KS, j), lambda j: pack(KD, KD, j)
    first = sum(([fma(2 * n), fma(2 * n + 1), exp(n)] for n in range(8)), []) + [exp(8)] + [p(j) for j in range(4)]
    second = [exp(9), exp(10), p(4), exp(11), exp(12), p(5), exp(13), exp(14), p(6), exp(15), mul(0), mul(1), p(7)]
    third = [mul(2), mul(3), ds(0), mul(4), mul(5), ds(1), mul(6), mul(7), ds(2), mul(8), mul(9), ds(3)]
    third += [mul(10), mul(11), ds(4), mul(12), mul(13), ds(5), mul(14), mul(15), ds(6), ds(7)]
    out = [[] for _ in range(KV_SLOTS)]
    for lo, work, slots in ((9, first, 6), (15, second, 4), (19, third, 4)):
        out[lo:lo + slots] = spread(work, slots)
    advance = lambda r: "v_add_u32 v%d, %%[adv], v%d" % (r, r)  # to the next stage, behind their last use in this one
    out[24], out[25] = [advance(KR), advance(KR + 1)], [advance(KR + 2), advance(KR + 3)]
    out[26], out[27] = [advance(KTR), advance(KTR + 1)], [advance(KTR + 2), advance(KTR + 3)]
    return out


def kv_step(elem):
    mfma = "v_mfma_f32_32x32x16_%s" % elem
    work, stat = kv_vector_work(elem), kv_statistics()
    # LDS requests in their order, those of the first PD entries from the step before
    order = [("e", e) for e in range(PD) for r in kv_fetch(e)]
    out, used, asked = [], 0, PD
    for s in range(KV_SLOTS):
        entries = range(used, used + KV_OPS[s])
        used += KV_OPS[s]
        needed = [("e", e) for e in entries] + ([("s", t) for t in range(1, 7)] if s == 8 else [])
        last = max(i for i, o in enumerate(order) if o in needed)
        out.append("s_waitcnt lgkmcnt(%d)" % min(15, len(order) - 1 - last))
        ring = [vr(RING0 + 4 * (e % RING), 4) for e in entries]
        if s < 8:
            out.append("%s %s, %s, %s, %s" % (mfma, vr(KS, 16), ring[0], vr(KK + 4 * s, 4), "0" if s == 0 else vr(KS, 16)))
        elif s < 16:
            out.append("%s %s, %s, %s, %s" % (mfma, vr(KD, 16), ring[0], ring[1], vr(KD, 16)))
        else:
            db, t, of_k = s % NDB, s % 8 // NDB, s >= 24
            out.append("%s %%[o%d], %s, %s, %%[o%d]" % (mfma, db if of_k else 4 + db, ring[0], vr((KD if of_k else KPB) + 4 * t, 4), db if of_k else 4 + db))
        if s == KV_BARRIER:
            out += KV_SYNC
        while asked < (used + PD if s < 26 else KV_ENTRIES + KV_NEXT.get(s, 0)):
            lines = kv_fetch(asked)
            out += lines
            order += [("e", asked)] * sum("ds_read" in x for x in lines)
            asked += 1
        out += stat.get(s, [])
        order += [("s", s)] * sum("ds_read" in x for x in stat.get(s, []))
        out += work[s]
    assert asked == KV_ENTRIES + PD == KV_ENTRIES + KV_NEXT[31] and KV_ENTRIES % RING == 0
    return out


def emit(name, lines):
    print("#define %s \\" % name)
    print(" \\\n".join('  "%s\\n\\t"' % l for l in lines))
    print()


def main():
    print("// Generated by gen_backward128_steps.py; do not edit.  Instruction streams of the head_dim-128 attention backward:")
    print("// TT_B128_DQ_<elem>_U<tile of the unrolled body>, TT_B128_DKV_<elem>.")
    print()
    for u in range(STAGES):  # the first requests of a step, where the step before was not a stream
        emit("TT_B128_DQ_PREFETCH_U%d" % u, sum((dq_fetch(DQ_SLOTS * u + g) for g in range(PD)), []))
    for elem in ("bf16", "f16"):
        for u in range(STAGES):
            emit("TT_B128_DQ_%s_U%d" % (elem.upper(), u), dq_step(u, elem))
    emit("TT_B128_DKV_PREFETCH", sum((kv_fetch(e) for e in range(PD)), []))
    for elem in ("bf16", "f16"):
        emit("TT_B128_DKV_%s" % elem.upper(), kv_step(elem))


if __name__ == "__main__":
    main()
