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


def emit(name, lines):
    print("#define %s \\" % name)
    print(" \\\n".join('  "%s\\n\\t"' % l for l in lines))
    print()


def main():
    print("// Generated by gen_backward128_steps.py; do not edit.  Instruction streams of the head_dim-128 attention backward:")
    print("// TT_B128_DQ_<elem>_U<tile of the unrolled body>.")
    print()
    for u in range(STAGES):  # the first requests of a step, where the step before was not a stream
        emit("TT_B128_DQ_PREFETCH_U%d" % u, sum((dq_fetch(DQ_SLOTS * u + g) for g in range(PD)), []))
    for elem in ("bf16", "f16"):
        for u in range(STAGES):
            emit("TT_B128_DQ_%s_U%d" % (elem.upper(), u), dq_step(u, elem))


if __name__ == "__main__":
    main()
