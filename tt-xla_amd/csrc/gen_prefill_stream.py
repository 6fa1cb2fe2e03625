#!/usr/bin/env python3
"""Writes the hand-scheduled loop of the streaming prefill kernel (32 query rows of one
head per wavefront, workgroups of four wavefronts) as one block of gfx950 assembly per head size and
form of the loop: build/prefill_stream_asm.h, included by prefill_stream_kernel.h.  Head sizes 64 (three
workgroups per CU), 128 (two) and 256 (one: its 128 accumulators are accumulation registers).  The forms: dense
K / V, dense with a sliding window, paged K / V in cache blocks of whole 64-key tiles, and in
cache blocks of whole 32-key blocks; at 128 also dense with keys of 128 + 64 features (the second part, the rotary
one, with base and strides of its own).  The numbers below are those of head size 128; at d, S(i) is d / 16
matrix instructions, PV(i) d / 16, a block 64 d bytes.

Why assembly: the loop wants the matrix pipe and the vector ALU of a SIMD busy at the same time
from one instruction stream, with every register chosen by hand (`Registers`) and every wait counted.  The unit of work is a BLOCK of 32 keys:

  S(i)   8 matrix instructions   S^T = K . Q^T of block i          (K fragments from LDS)
  sm(i)  ~56 vector instructions  p = exp2(s c - m), packed to bfloat16, row sum
  PV(i)  8 matrix instructions   O^T += V^T . P^T of block i       (V^T fragments from LDS)

Iteration i issues S(i + 1) and PV(i - 1) alternately, one slice of sm(i) and the LDS read of a
fragment 8 matrix instructions ahead behind each; the fragment reads run on across iterations.
Scores and probabilities alternate between two register banks by the parity of i, so nothing is
copied.

The running maximum is not tracked per block.  Probabilities are taken relative to a reference
m (kept as mc = m c + 7 in the exponent domain) that only moves when some probability of the
block reaches 2, which is one OR over the packed probabilities and one test of bit 14 of every
bfloat16: p >= 2 exactly when the score exceeds the reference's maximum by 2^8, the lazy rule of
the plain loop.  The block then takes the slow path at the end of the iteration: true row maximum over
it and the block behind it, new reference, accumulators and row sum rescaled, probabilities of the
block recomputed.  The first
block of a row always does: the reference starts at the lowest finite float, so that every real score
lies above it by more than any exponent, while a masked one (-inf) still becomes a zero and not a NaN
(a block may be masked for all keys of a row: wavefronts of one workgroup may hold different row
blocks, and a window may start behind the first block).

Masks: a lane holds the keys key0 + 4 h + {0..3, 8..11, 16..19, 24..27} of a block (h = lane / 32)
for query row lane % 32, and may see keys up to its limit (causal diagonal, end of K / V).  Blocks
from key `mask_from` on are masked in place, at the start of their iteration, before anything reads
the scores: 16 compares of the key constants against limit - 4 h - key0 and 16 selects of -inf.
Blocks in front of it skip that with one scalar branch.  With a sliding window a lane also has a
lowest key; blocks whose first key is below `low_to` are masked from below in the same way.

LDS: a ring of NS slots of 8 KiB (32 rows) for K blocks and one for V blocks (NS = 5; 4 at head size 256, whose five
would be past what an LDS instruction's offset reaches); block j lives in
slot j % NS.  Iteration i reads K block i + 1 and V block i - 1 and, through the running fragment
reads, the first fragments of K block i + 2 and V block i.  Its barrier, at its start, says that
nobody reads K block i and V block i - 2 any more; K block i + NS and V block i + NS - 2 are
requested into their slots (LDS-DMA loads, two per tensor and wavefront).  A request has to have
landed NS - 2 barriers later: the wait in front of a barrier lets the requests of the last NS - 3
barriers stay in flight (vmcnt(8), less near the end, where there are fewer), so a tile has three iterations to arrive with NS = 5, where
two stages of whole tiles gave it two.  Dense K / V: a block is `stride` bytes behind the one before.  Paged (block
size a multiple of 64): two blocks are a tile, a tile lies in one cache block; the table entry of
the tile K enters two iterations from now is requested in front of the tile requests of every
odd iteration (so the same wait covers it) and read at the next odd one.  Entries outside
[0, num_blocks) read cache block 0.  Cache blocks of a multiple of 32 keys: every block has an entry
of its own; the one of K block i + NS is read in iteration i and was requested in iteration i - 2 in
front of the tile requests, so the same wait covers it (vmcnt(8), not 10: near the end an iteration
requests no entry any more).  V follows two blocks behind K, so two byte offsets wait in a queue.

Keys of 128 + 64 features: S(i) is 12 matrix instructions, an iteration 20; a block of the second part
is 4 KiB (one load per wavefront), in a ring of its own behind the other two.  With rings of NS = 4
the three still fit 80 KiB, half of a CU's LDS, and a request has two iterations to arrive.

A workgroup may take only a part of the keys (paged forms): it starts at any block, and if the base
of a partial result is given, the accumulators go out as they are, with the reference and the sum of
every row, for a merge kernel.

A workgroup takes one or several ITEMS (blocks of 32 query rows of its four heads) one after the
other: item k of the workgroup in slot j of `spg` slots is row block nqt - 1 - d with
d = k spg + (k even ? j : spg - 1 - j), as long as d < nqt.  Row blocks are dealt heavy first and in
alternating direction, so that with causal masking every workgroup gets about the same number of
key blocks.  The launcher's default is one item per workgroup (spg = nqt: the hardware deals the
workgroups as slots free up, which measured faster than one static round), several when the row
blocks weigh the same and divide evenly over one round.  (Only where the four wavefronts share their
rows, and not with a window, whose row blocks start at different keys.)  Per item the block does everything
between the Q rows and the stored output rows: its first requests (K blocks 0..NS-1, V blocks
0..NS-3; for the first item they are a block of assembly of their own, one block less of each, in front of the
caller's set-up), all blocks, the last PV, normalisation and store; then the next item's Q fragments
and first requests go out in front of the store of the finished one.

Matrix-to-vector hazards the hardware does not interlock are kept by construction and checked in the
text of every form (check_distances): the vector instructions that read a score bank start two matrix
instructions or more after the last one that wrote it (a result is there about a dozen wait states after
its instruction, of which the next one's eight passes are eight; the mask waits explicitly); a register
of probabilities is rewritten five matrix instructions (head size 64), ten (128) or nineteen (256) after
the last one that read it, which read it as it started; the slow path and the exit wait out the
matrix pipe with s_nop.
"""

import re
import sys


# ---- vector registers ---------------------------------------------------------------------------
class Registers:
    """The vector register map of a head size; what is an operand of the block says `operands`."""

    def __init__(self, d, wide):
        self.acc_file = "a" if d == 256 else "v"   # file of the output accumulators
        at = 0

        def take(n):
            nonlocal at
            at += n
            return at - n

        # output accumulators, head-dim blocks 0 .. d / 32 - 1
        self.ACC = [16 * db for db in range(d // 32)] if d == 256 else [take(16) for _ in range(d // 32)]
        self.QF = take(d // 4)                     # Q fragments, k-step ks at QF + 4 ks
        self.S = [take(16), take(16)]              # score banks (these, P and RING in one piece: the epilogue's packed rows)
        self.P = [take(8), take(8)]                # probability banks (packed pairs)
        self.RING = take(4 * NSLOT)                # fragment slots of 4 registers
        self.KOFF = take(d // 16)                  # LDS byte address of the lane's K fragment in K slot 0, k-step ks
        self.VOFF = take(d // 32)                  # ... of the lane's V^T fragment in V slot 0, output block db
        self.LDK = take(d // 64)                   # per-lane global byte offsets of the K loads of a block
        self.LDV = take(d // 64)                   # ... of the V loads
        if d == 128:
            at = 196
        self.MC, self.LRUN, self.LSUM, self.ALPHA = (take(1) for _ in range(4))
        self.T = [take(1) for _ in range(4)]
        self.ORV, self.MLOC, self.MB, self.MCN = (take(1) for _ in range(4))
        self.PTREQ = take(1)                       # paged: the requested block-table entry
        self.LOWEST, self.LOWREL = take(1), take(1)  # window: first visible key of the lane's row, minus 4 h; relative to the block
        self.PTREQ2 = take(1)                      # blocks of 32: the entry requested in odd iterations
        self.LIMIT = take(1)                       # last visible key of the lane's row, minus 4 h
        self.LIMREL, self.NEGINF, self.VZERO = (take(1) for _ in range(3))
        # items: per lane, 64-bit: q / out of row 0 of the lane's head, at the lane's 8 h elements
        self.QBASE, self.OUTBASE = take(2), take(2)
        self.VN, self.V4H = take(1), take(1)       # lane % 32 and 4 (lane / 32)
        self.OUTP, self.PTMP = take(2), take(2)
        self.VT0, self.VROW = take(1), take(1)
        if wide:                                   # keys of 128 + 64: Q fragments, LDS addresses and global offsets of the second part
            self.QFP, self.KOFFP, self.LDKP = take(16), take(4), take(1)
        self.count = at


NSLOT = 8

# ---- scalar registers ---------------------------------------------------------------------------
S_KBASE = "s[64:65]"           # dense: next K block to request; paged: the K cache (both minus 1024, see dma)
S_VBASE = "s[66:67]"
S_STRIDE = "s68"               # dense: bytes from one block to the next; paged: bytes of one (cache block, head) slab
S_C = "s69"                    # softmax scale times log2(e)
S_NB = "s70"                   # blocks left
S_KLEFT = "s71"                # K blocks left to request
S_M0B = "s72"                  # LDS address of this wavefront's first 1 KiB segment in K slot 0
S_VLEFT = "s73"                # V blocks left to request
S_MASKFROM = "s74"             # blocks whose first key is >= this are masked
S_KEY0 = "s75"                 # first key of the block whose softmax comes next (input: of the first block)
S_STATS, S_PART = "s[36:37]", "s[38:39]"  # paged: where (reference, sum) and the accumulators of a part go (0: the whole result)
S_LOWTO = "s34"                # window: blocks whose first key is < this are masked from below (input)
# keys of 128 + 64 only: the second part of K, its bytes per block and the LDS address of the wavefront's segment; V's bytes per block
S_PBASE, S_PSTRIDE, S_M0P, S_VSTRIDE = "s[30:31]", "s32", "s33", "s35"
# paged only
S_HKV, S_HK, S_NCB, S_TPB = "s76", "s77", "s78", "s79"  # kv heads, this kv head, cache blocks, tiles per cache block
S_CIN = "s80"                  # tile-in-cache-block index of the tile whose entry is read next
S_RIN = "s81"                  # ... of the tile whose entry is requested next
S_RPTR = "s[82:83]"            # address of that entry
S_OFFV = "s[84:85]"            # byte offset in a cache of the tile V requests from (on entry: tile 1)
S_OFFK = "s[86:87]"            # ... K requests from (on entry: tile 2)
S_RLEFT = "s96"                # entries left to request
S_OFF0 = "s[98:99]"            # byte offset of tile 0
# items
S_K, S_J, S_SPG, S_NQT = "s40", "s41", "s42", "s43"      # item counter, slot of the workgroup, slots, row blocks
S_SQ, S_SKV, S_OFFSET, S_CAUSAL = "s44", "s45", "s46", "s47"
S_QTS, S_OTS = "s48", "s49"    # bytes from a query / output row to the next
# dense: s[50:51], s[52:53] K / V block 0 (minus 1024); paged: tile 1 and 2 offsets, s54 entry of tile 3,
# s55 / s56 tile-in-cache-block of tiles 3 / 4, s[58:59] address of tile 4's entry
# blocks of 32: s[50:51], s[52:53], s[58:59] byte offsets of blocks 0, 1, 2, s[84:85] and s[98:99] of blocks 3
# and 4 (later: the next two V blocks), s[86:87] the K block's; S_TPB, S_CIN, S_RIN count 32-key blocks
S_ROW0 = "s57"                 # first query row of the item
S_STOREMASK = "s[60:61]"
# LDS offset of the slot with the wavefront's Q rows; LDS offset and address of the slot its output rows go through; output of the
# wavefront's head, row 0
S_QSLOT, S_OUTSLOT, S_OUTADDR, S_OUT = "s25", "s26", "s27", "s[28:29]"
# temporaries s[88:95], s[62:63]

PSLOT = 4096                   # bytes of a block of the second part of K
KEY_CONST = [8 * (r // 4) + r % 4 for r in range(16)]


class Form:
    """What one block of assembly serves."""

    def __init__(self, name, d=128, paged=0, window=False, wide=False):
        self.name, self.d = f"{name}_{d}", d
        self.paged, self.window = paged, window  # paged: 0 or the keys that share a table entry
        self.wide = wide                    # keys of 128 + 64 features
        self.ns = 4 if wide or d == 256 else 5  # slots per ring
        self.unroll = 4 if self.ns == 4 else 10  # lcm(2, ns): score bank and slots repeat
        self.SLOT = 64 * d                  # bytes of a block of K or V
        self.tensor_loads = d // 64         # loads per wavefront of a block of K or V
        self.__dict__.update(vars(Registers(d, wide)))
        self.vring = self.ns * self.SLOT    # LDS offset of the V ring (VOFF carries it), of the second part's ring (KOFFP)
        self.pring = 2 * self.vring
        self.loads = 2 * self.tensor_loads + wide  # tile loads of an iteration
        self.items = d == 128 and not window and not wide and paged != 32  # several row blocks in turn
        self.parts = paged > 0  # may take a part of the keys


FORMS = [Form("DENSE_WIDE", wide=True)] + [
    form for d in (64, 128, 256)
    for form in (Form("DENSE", d), Form("DENSE_WINDOW", d, window=True), Form("PAGED", d, paged=64), Form("PAGED32", d, paged=32))]
START_REFERENCE = "0xff7fffff"  # the lowest finite float


class Out:
    def __init__(self):
        self.lines = []

    def e(self, s):
        self.lines.append(s)

    def label(self, name):
        self.lines.append(name + "%=:")


def vr(a, n=1, file="v"):
    return f"{file}{a}" if n == 1 else f"{file}[{a}:{a + n - 1}]"


def frag_reads(f, frag, slot):
    """LDS read instructions of a fragment into ring slot `slot`.
    ("K", LDS slot, k-step) or ("V", LDS slot, key step 0 / 1, output block)."""
    base = f.RING + 4 * slot
    if frag[0] == "K" and frag[2] >= f.d // 16:
        return [f"ds_read_b128 {vr(base, 4)}, v{f.KOFFP + frag[2] - f.d // 16} offset:{frag[1] * PSLOT}"]
    if frag[0] == "K":
        _, ls, ks = frag
        return [f"ds_read_b128 {vr(base, 4)}, v{f.KOFF + ks} offset:{ls * f.SLOT}"]
    _, ls, k4, db = frag
    off = ls * f.SLOT + k4 * f.SLOT // 2
    return [f"ds_read_b64_tr_b16 {vr(base, 2)}, v{f.VOFF + db} offset:{off}",
            f"ds_read_b64_tr_b16 {vr(base + 2, 2)}, v{f.VOFF + db} offset:{off + f.SLOT // 4}"]


def mfma(f, m, slot):
    a = vr(f.RING + 4 * slot, 4)
    if m[0] == "S":
        _, bank, ks = m
        d = vr(f.S[bank], 16)
        q = f.QF + 4 * ks if ks < f.d // 16 else f.QFP + 4 * (ks - f.d // 16)
        return f"v_mfma_f32_32x32x16_bf16 {d}, {a}, {vr(q, 4)}, {'0' if ks == 0 else d}"
    _, db, bank, k4p = m
    d = vr(f.ACC[db], 16, f.acc_file)
    return f"v_mfma_f32_32x32x16_bf16 {d}, {a}, {vr(f.P[bank] + 4 * k4p, 4)}, {d}"


def softmax_ops(f, q, test=True):
    """Vector instructions of sm(i) on bank q, in an order that keeps one instruction between a
    transcendental and its first use."""
    s, p = f.S[q], f.P[q]
    A = lambda r: f"v_fma_f32 v{f.T[r % 4]}, v{s + r}, {S_C}, -v{f.MC}"
    B = lambda r: f"v_exp_f32 v{f.T[r % 4]}, v{f.T[r % 4]}"
    C = lambda j: f"v_cvt_pk_bf16_f32 v{p + j}, v{f.T[(2 * j) % 4]}, v{f.T[(2 * j + 1) % 4]}"
    D = lambda j: f"v_dot2c_f32_bf16 v{f.LSUM}, 0x3f803f80, v{p + j}"
    ops = [f"v_mov_b32 v{f.LSUM}, 0", A(0), A(1), B(0), B(1)]
    for j in range(8):
        if j < 7:
            ops += [A(2 * j + 2), A(2 * j + 3)]
        ops.append(C(j))
        if j < 7:
            ops += [B(2 * j + 2), B(2 * j + 3)]
        ops.append(D(j))
    if test:
        ops += [f"v_or3_b32 v{f.ORV}, v{p}, v{p + 1}, v{p + 2}",
                f"v_or3_b32 v{f.ORV}, v{f.ORV}, v{p + 3}, v{p + 4}",
                f"v_or3_b32 v{f.ORV}, v{f.ORV}, v{p + 5}, v{p + 6}",
                f"v_or_b32 v{f.ORV}, v{f.ORV}, v{p + 7}",
                f"v_and_b32 v{f.ORV}, 0x40004000, v{f.ORV}",
                f"v_cmp_ne_u32 vcc, 0, v{f.ORV}"]
    for i, op in enumerate(ops[:-1]):  # a transcendental's result is not read by the next instruction
        if op.startswith("v_exp_f32"):
            dst = op.split()[1].rstrip(",")
            assert dst not in [t.rstrip(",") for t in ops[i + 1].split()[2:]], (op, ops[i + 1])
    return ops


def spread(ops, nslots, first=0):
    """ops cut into nslots consecutive chunks of nearly equal size; slots before `first` get none."""
    n = nslots - first
    out = [[] for _ in range(nslots)]
    for k, op in enumerate(ops):
        out[first + (k * n) // len(ops)].append(op)
    return out


def stream(o, f, pairs, valu_chunks, phase, in_flight, tail):
    """pairs: [(matrix instruction, fragment)].  Per pair: wait for its fragment, the matrix
    instruction, the read of the fragment NSLOT pairs on, the vector chunk.  phase: the ring slot of the
    first pair's fragment; in_flight: the first NSLOT fragments have been requested by the code in front
    (else they are requested here); tail: the fragments requested behind the last NSLOT pairs (the next
    iteration's first ones).  Returns the next phase."""
    frags = [f for _, f in pairs] + list(tail)
    n = len(pairs)
    count = lambda k: len(frag_reads(f, frags[k], 0))
    if not in_flight:
        for k in range(min(NSLOT, len(frags))):
            for x in frag_reads(f, frags[k], (phase + k) % NSLOT):
                o.e(x)
    for j in range(n):
        after = sum(count(k) for k in range(j + 1, min(j + NSLOT, len(frags))))
        assert after <= 15
        o.e(f"s_waitcnt lgkmcnt({after})")
        o.e(mfma(f, pairs[j][0], (phase + j) % NSLOT))
        if j + NSLOT < len(frags):
            for x in frag_reads(f, frags[j + NSLOT], (phase + j) % NSLOT):
                o.e(x)
        for x in valu_chunks[j]:
            o.e(x)
    return (phase + n) % NSLOT


def score_pairs(bank, slot, f):
    return [(("S", bank, x), ("K", slot, x)) for x in range(f.d // 16 + 4 * f.wide)]


def iteration_pairs(p, f, has_pv=True):
    """Iteration i = p (mod f.unroll): S(i + 1) into bank 1 - q from K block i + 1, PV(i - 1) from
    bank 1 - q of the probabilities and V block i - 1."""
    q = p % 2
    scores = score_pairs(1 - q, (p + 1) % f.ns, f)
    if not has_pv:
        return scores
    db = f.d // 32
    pv = [(("PV", x % db, 1 - q, x // db), ("V", (p - 1) % f.ns, x // db, x % db)) for x in range(2 * db)]
    order = "SPSSPSPSSPSPSSPSPSSP" if f.wide else "SP" * len(pv)
    assert order.count("S") == len(scores) and order.count("P") == len(pv)
    scores, pv = iter(scores), iter(pv)
    return [next(scores if x == "S" else pv) for x in order]


def mask_selects(o, f, bank):
    """-inf in place of the scores of the block at S_KEY0 that a lane may not see; the bank has been written."""
    s = f.S[bank]
    o.e(f"v_subrev_u32 v{f.LIMREL}, {S_KEY0}, v{f.LIMIT}")  # limit - 4 h - key0
    o.e(f"v_mov_b32 v{f.NEGINF}, 0xff800000")
    sel = lambda r: f"v_cndmask_b32_e64 v{s + r}, v{s + r}, v{f.NEGINF}, s[{88 + 2 * (r % 4)}:{89 + 2 * (r % 4)}]"
    sides = [("v_cmp_gt_i32_e64", f.LIMREL)]
    if f.window:
        o.e(f"v_subrev_u32 v{f.LOWREL}, {S_KEY0}, v{f.LOWEST}")
        sides.append(("v_cmp_lt_i32_e64", f.LOWREL))
    for compare, bound in sides:
        for r in range(16):
            o.e(f"{compare} s[{88 + 2 * (r % 4)}:{89 + 2 * (r % 4)}], {KEY_CONST[r]}, v{bound}")
            if r >= 3:  # a select reads its mask three instructions after the compare that wrote it
                o.e(sel(r - 3))
        o.e("s_nop 1")
        for r in range(13, 16):
            o.e(sel(r))


def skip_unless_masked(o, f, tag):
    """Branches to L_nomask_<tag> if no lane needs a mask for the block at S_KEY0."""
    if f.window:
        o.e(f"s_cmp_lt_i32 {S_KEY0}, {S_LOWTO}")
        o.e(f"s_cbranch_scc1 L_mask_{tag}%=")
    o.e(f"s_cmp_lt_i32 {S_KEY0}, {S_MASKFROM}")
    o.e(f"s_cbranch_scc1 L_nomask_{tag}%=")
    if f.window:
        o.label(f"L_mask_{tag}")


def mask_block(o, f, q, tag):
    """Start of the iteration whose softmax reads bank q: masks the block in place if it needs it."""
    skip_unless_masked(o, f, tag)
    o.e("s_nop 15")  # the last matrix instruction into this bank has written
    mask_selects(o, f, q)
    o.label(f"L_nomask_{tag}")
    o.e(f"s_add_u32 {S_KEY0}, {S_KEY0}, 32")


def accumulators(f):
    return range(f.ACC[0], f.ACC[0] + f.d // 2)


def scale_accumulators(o, f):
    """All of them by ALPHA."""
    for r in accumulators(f):
        if f.acc_file == "v":
            o.e(f"v_mul_f32 v{r}, v{f.ALPHA}, v{r}")
        else:  # (accumulation registers are the matrix instructions': a round trip through four registers in turn)
            t = f.T[r % 4]
            o.e(f"v_accvgpr_read_b32 v{t}, a{r}")
            o.e(f"v_mul_f32 v{t}, v{f.ALPHA}, v{t}")
            o.e(f"v_accvgpr_write_b32 a{r}, v{t}")


def slow_path(o, f, q, name, join, first=False):
    """Bank q: true row maximum, new reference, rescale, probabilities again.  The scores of the next block are there
    already (bank 1 - q, S_KEY0 is its first key): the maximum is taken over both.  The weight that equals the
    reference is exact in bfloat16, and it is the row's largest one more often for 64 keys than for 32: the output's
    relative error against 64 bits at 16 / 8 heads, 512 tokens 2.019e-3 -> 1.999e-3 (the plain loop, whose tiles hold 64
    keys: 1.999e-3), 768 tokens in a window of 256 2.078e-3 -> 2.058e-3 (2.064e-3).  The first block of a row has nothing to rescale
    (`first`), which makes up for the time: a prompt of 128 tokens 7.66 us before, 7.70 with the second block's maximum,
    7.59 this way."""
    def row_max(bank, regs):
        for r in regs:
            o.e(f"v_max3_f32 v{f.MLOC}, v{f.MLOC}, v{f.S[bank] + r}, v{f.S[bank] + r + 1}")

    o.label(name)
    o.e("s_nop 15")
    o.e("s_nop 15")
    o.e(f"v_max_f32 v{f.MLOC}, v{f.S[q]}, v{f.S[q] + 1}")
    row_max(q, range(2, 16, 2))
    o.e(f"s_cmp_lt_u32 {S_NB}, 2")              # no next block: its bank holds products of whatever the slot held
    o.e(f"s_cbranch_scc1 L_one_{name}%=")
    skip_unless_masked(o, f, name)
    mask_selects(o, f, 1 - q)                   # (the next iteration masks it again: the same selects)
    o.label(f"L_nomask_{name}")
    row_max(1 - q, range(0, 16, 2))
    o.label(f"L_one_{name}")
    o.e(f"v_mov_b32 v{f.MB}, v{f.MLOC}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{f.MLOC}, v{f.MB}")
    o.e("s_nop 1")
    o.e(f"v_max_f32 v{f.MLOC}, v{f.MLOC}, v{f.MB}")                 # row maximum (raw score)
    o.e(f"v_fma_f32 v{f.MB}, v{f.MLOC}, {S_C}, -v{f.MC}")           # how far above the reference's zero
    o.e(f"v_cmp_le_f32 vcc, 1.0, v{f.MB}")                      # p >= 2 somewhere in the row: move
    o.e(f"v_mul_f32 v{f.MCN}, {S_C}, v{f.MLOC}")
    o.e(f"v_add_f32 v{f.MCN}, 0x40e00000, v{f.MCN}")              # m c + 7
    o.e("s_nop 1")
    o.e(f"v_cndmask_b32 v{f.MCN}, v{f.MC}, v{f.MCN}, vcc")
    if first:  # nothing is accumulated yet: no rescale
        o.e(f"v_mov_b32 v{f.MC}, v{f.MCN}")
    else:
        o.e(f"v_sub_f32 v{f.ALPHA}, v{f.MC}, v{f.MCN}")             # 0 where the reference stays
        keep_zeros = f.window and f.acc_file == "a"
        if keep_zeros:
            # A row whose window starts at this block or behind it has only zeros to rescale: with two row blocks in a
            # workgroup, the second one's rows find their first keys blocks later than the first one's.  By position,
            # not by the reference (a score may be the lowest float); S_KEY0 is the first key of the next block.  At
            # head size 256 a rescale is three instructions for each of 128 registers: 16 / 8 heads, 6 x 4032 tokens in a
            # window of 512 365 -> 358 us, 1024 tokens 20.7 -> 20.0, 352 in 100 12.7 -> 12.1.  Where it is one for each of
            # 32 or 64, the test does not pay: 4 x 2048 tokens, 16 / 8 of 128 in 512 51.5 -> 50.5, 64 / 8 of 64 in
            # 128 47.4 -> 48.5.
            o.e(f"v_subrev_u32 v{f.LOWREL}, {S_KEY0}, v{f.LOWEST}")
            o.e(f"v_add_u32 v{f.LOWREL}, v{f.V4H}, v{f.LOWREL}")
            o.e(f"v_cmp_le_i32 vcc, 0xffffffe0, v{f.LOWREL}")
            o.e("s_nop 1")
            o.e(f"v_cndmask_b32 v{f.ALPHA}, v{f.ALPHA}, 0, vcc")
        o.e(f"v_exp_f32 v{f.ALPHA}, v{f.ALPHA}")
        o.e(f"v_mov_b32 v{f.MC}, v{f.MCN}")
        o.e("s_nop 0")
        o.e(f"v_mul_f32 v{f.LRUN}, v{f.LRUN}, v{f.ALPHA}")
        if keep_zeros:
            o.e(f"v_cmp_neq_f32 vcc, 1.0, v{f.ALPHA}")
            o.e(f"s_cbranch_vccz L_kept_{name}%=")
        scale_accumulators(o, f)
        if keep_zeros:
            o.label(f"L_kept_{name}")
    for x in softmax_ops(f, q, test=False):
        o.e(x)
    o.e("s_nop 4")
    o.e(f"s_branch {join}%=")


def block_loads(o, f, lane_regs, base):
    """The instruction offset moves the LDS address as well as the global one: load j lands 1024 j
    bytes behind M0 and reads base + lane offset + 1024 j, so the lane offsets carry
    1024 - 1024 j and the bases - 1024."""
    for j in range(f.tensor_loads):
        o.e(f"global_load_lds_dwordx4 v{lane_regs + j}, {base} offset:{1024 * j}")


def request_block(o, f, which, slot, tag, half):
    """One K or V block into LDS slot `slot` of its ring, if there is one left to request.
    paged: the block is half `half` of the tile at S_OFFK / S_OFFV."""
    paged = f.paged
    left, lane, base, ring = (S_KLEFT, f.LDK, S_KBASE, 0) if which == "K" else (S_VLEFT, f.LDV, S_VBASE, f.vring)
    o.e(f"s_cmp_eq_u32 {left}, 0")
    o.e(f"s_cbranch_scc1 L_no{which}_{tag}%=")
    if paged:
        lo, hi = (86, 87) if which == "K" else (84, 85)
        b0 = int(base[2:4])
        o.e(f"s_add_u32 s90, s{b0}, s{lo}")
        o.e(f"s_addc_u32 s91, s{b0 + 1}, s{hi}")
        if half:
            o.e(f"s_add_u32 s90, s90, {f.SLOT}")
            o.e("s_addc_u32 s91, s91, 0")
    o.e(f"s_add_u32 m0, {S_M0B}, {ring + slot * f.SLOT}")
    o.e("s_nop 0")
    block_loads(o, f, lane, "s[90:91]" if paged else base)
    if not paged:
        b0 = int(base[2:4])
        o.e(f"s_add_u32 s{b0}, s{b0}, {S_VSTRIDE if f.wide and which == 'V' else S_STRIDE}")
        o.e(f"s_addc_u32 s{b0 + 1}, s{b0 + 1}, 0")
    if f.wide and which == "K":
        o.e(f"s_add_u32 m0, {S_M0P}, {slot * PSLOT}")
        o.e("s_nop 0")
        o.e(f"global_load_lds_dwordx4 v{f.LDKP}, {S_PBASE}")
        o.e(f"s_add_u32 s30, s30, {S_PSTRIDE}")
        o.e("s_addc_u32 s31, s31, 0")
    o.e(f"s_sub_u32 {left}, {left}, 1")
    o.label(f"L_no{which}_{tag}")


def next_tile(o, f, tag):
    """paged, odd iterations: V moves on to the tile K was in, K to the tile whose entry has
    arrived; the entry after that is requested."""
    o.e("s_mov_b64 s[84:85], s[86:87]")
    o.e(f"v_readfirstlane_b32 s88, v{f.PTREQ}")
    o.e(f"s_cmp_lt_u32 s88, {S_NCB}")
    o.e("s_cselect_b32 s88, s88, 0")
    o.e(f"s_mul_i32 s88, s88, {S_HKV}")
    o.e(f"s_add_u32 s90, s88, {S_HK}")            # cache block * kv_heads + kv_head
    o.e(f"s_mul_hi_u32 s87, s90, {S_STRIDE}")
    o.e(f"s_mul_i32 s86, s90, {S_STRIDE}")
    o.e(f"s_lshl_b32 s90, {S_CIN}, {f.SLOT.bit_length()}")  # 64 tokens per tile inside the cache block
    o.e("s_add_u32 s86, s86, s90")
    o.e("s_addc_u32 s87, s87, 0")
    o.e(f"s_add_u32 {S_CIN}, {S_CIN}, 1")
    o.e(f"s_cmp_eq_u32 {S_CIN}, {S_TPB}")
    o.e(f"s_cselect_b32 {S_CIN}, 0, {S_CIN}")
    o.e(f"s_cmp_eq_u32 {S_RLEFT}, 0")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"global_load_dword v{f.PTREQ}, v{f.VZERO}, {S_RPTR}")
    o.e(f"s_sub_u32 {S_RLEFT}, {S_RLEFT}, 1")
    o.e(f"s_add_u32 {S_RIN}, {S_RIN}, 1")
    o.e(f"s_cmp_lg_u32 {S_RIN}, {S_TPB}")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"s_mov_b32 {S_RIN}, 0")
    o.e("s_add_u32 s82, s82, 4")
    o.e("s_addc_u32 s83, s83, 0")
    o.label(f"L_noreq_{tag}")


def next_block(o, f, p, tag):
    """Blocks of 32, every iteration: the byte offset of the K block from its table entry; the entry of
    the K block two iterations on is requested."""
    req = f.PTREQ2 if p % 2 else f.PTREQ
    o.e(f"v_readfirstlane_b32 s88, v{req}")
    o.e(f"s_cmp_lt_u32 s88, {S_NCB}")
    o.e("s_cselect_b32 s88, s88, 0")
    o.e(f"s_mul_i32 s88, s88, {S_HKV}")
    o.e(f"s_add_u32 s90, s88, {S_HK}")
    o.e(f"s_mul_hi_u32 s87, s90, {S_STRIDE}")
    o.e(f"s_mul_i32 s86, s90, {S_STRIDE}")
    o.e(f"s_lshl_b32 s90, {S_CIN}, {f.SLOT.bit_length() - 1}")  # 32 tokens per block inside the cache block
    o.e("s_add_u32 s86, s86, s90")
    o.e("s_addc_u32 s87, s87, 0")
    o.e(f"s_add_u32 {S_CIN}, {S_CIN}, 1")
    o.e(f"s_cmp_eq_u32 {S_CIN}, {S_TPB}")
    o.e(f"s_cselect_b32 {S_CIN}, 0, {S_CIN}")
    o.e(f"s_cmp_eq_u32 {S_RLEFT}, 0")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"global_load_dword v{req}, v{f.VZERO}, {S_RPTR}")
    o.e(f"s_sub_u32 {S_RLEFT}, {S_RLEFT}, 1")
    o.e(f"s_add_u32 {S_RIN}, {S_RIN}, 1")
    o.e(f"s_cmp_lg_u32 {S_RIN}, {S_TPB}")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"s_mov_b32 {S_RIN}, 0")
    o.e("s_add_u32 s82, s82, 4")
    o.e("s_addc_u32 s83, s83, 0")
    o.label(f"L_noreq_{tag}")


def in_flight(f, left):
    """Loads of the ns - 3 iterations in front of one with `left` blocks left (itself among them): iteration j has requested K block
    j + ns and V block j + ns - 2 if they exist."""
    k, v = f.loads - f.tensor_loads, f.tensor_loads
    return sum(k * (left > f.ns - back) + v * (left > f.ns - 2 - back) for back in range(1, f.ns - 2))


def iteration_head(o, f, p, tag):
    """Mask, barrier and requests of iteration i = p (mod f.unroll)."""
    paged, ns = f.paged, f.ns
    mask_block(o, f, p % 2, tag)
    # requests of the last ns - 3 iterations may stay in flight; near the end they are fewer.  (Iteration 0 needs blocks that have landed
    # in front of it.)  A wait for everything from the last K request on cost a workgroup three waits of half a memory trip.
    if tag != "i0":
        o.e(f"s_cmp_ge_u32 {S_NB}, {ns}")
        o.e(f"s_cbranch_scc0 L_few_{tag}%=")
        o.e(f"s_waitcnt vmcnt({in_flight(f, ns)})")
        o.label(f"L_bar_{tag}")
    o.e("s_barrier")
    if paged == 64 and (p + ns) % 2 == 0:
        next_tile(o, f, tag)
    if paged == 32:
        next_block(o, f, p, tag)
    # K block i + NS is half (i + NS) % 2 of its tile, V block i + NS - 2 the same half of its own
    half = (p + ns) % 2 if paged == 64 else 0
    request_block(o, f, "K", p % ns, tag, half)
    request_block(o, f, "V", (p + ns - 2) % ns, tag, half)
    if paged == 32:
        o.e("s_mov_b64 s[84:85], s[98:99]")
        o.e("s_mov_b64 s[98:99], s[86:87]")


def few_left(o, f, tag):
    """The wait of an iteration with less than ns blocks left."""
    o.label(f"L_few_{tag}")
    for left in range(1, f.ns - 1):
        o.e(f"s_cmp_lg_u32 {S_NB}, {left}")
        o.e(f"s_cbranch_scc1 L_few{left}_{tag}%=")
        o.e(f"s_waitcnt vmcnt({in_flight(f, left)})")
        o.e(f"s_branch L_bar_{tag}%=")
        o.label(f"L_few{left}_{tag}")
    o.e(f"s_waitcnt vmcnt({in_flight(f, f.ns - 1)})")
    o.e(f"s_branch L_bar_{tag}%=")


def iteration_tail(o, f, tag, exit_label):
    o.e(f"s_cbranch_vccnz L_slow_{tag}%=")
    o.label(f"L_join_{tag}")
    o.e(f"v_add_f32 v{f.LRUN}, v{f.LRUN}, v{f.LSUM}")
    o.e(f"s_sub_u32 {S_NB}, {S_NB}, 1")
    o.e(f"s_cmp_eq_u32 {S_NB}, 0")
    o.e(f"s_cbranch_scc1 {exit_label}%=")


def first_frags(p, f):
    """The first NSLOT fragments of iteration p (mod f.unroll)."""
    return [frag for _, frag in iteration_pairs(p % f.unroll, f)[:NSLOT]]


def item_setup(o, f, tag):
    """Per-item state from S_ROW0: output pointers, the rows' key limits, the mask threshold, cleared
    accumulators and softmax state."""
    o.e(f"v_add_u32 v{f.VROW}, {S_ROW0}, v{f.VN}")                                   # the lane's query row
    if f.items:
        o.e(f"v_mad_u64_u32 v[{f.OUTP}:{f.OUTP + 1}], s[92:93], v{f.VROW}, {S_OTS}, v[{f.OUTBASE}:{f.OUTBASE + 1}]")
        o.e(f"v_cmp_gt_i32_e64 {S_STOREMASK}, {S_SQ}, v{f.VROW}")                  # rows that exist are stored
    o.e(f"s_sub_u32 s88, {S_SQ}, 1")
    o.e(f"v_min_i32 v{f.VT0}, s88, v{f.VROW}")                                       # rows past the end repeat the last one
    o.e(f"v_add_u32 v{f.VT0}, {S_OFFSET}, v{f.VT0}")
    o.e(f"s_sub_u32 s89, {S_SKV}, 1")
    o.e(f"v_min_i32 v{f.VT0}, s89, v{f.VT0}")                                        # causal: min(offset + row, skv - 1)
    o.e(f"s_add_u32 s88, {S_OFFSET}, {S_ROW0}")
    o.e("s_min_i32 s88, s88, s89")
    o.e(f"s_cmp_eq_u32 {S_CAUSAL}, 0")
    o.e("s_cselect_b32 s88, s89, s88")                                           # the first row's limit
    o.e(f"s_cbranch_scc0 L_causal_{tag}%=")
    o.e(f"v_mov_b32 v{f.VT0}, s89")                                                # not causal: skv - 1 for every row
    o.label(f"L_causal_{tag}")
    o.e(f"v_sub_u32 v{f.LIMIT}, v{f.VT0}, v{f.V4H}")
    o.e(f"s_sub_u32 {S_MASKFROM}, s88, 30")
    if tag != "first":  # (several row blocks in turn: all of them start at key 0)
        o.e(f"s_mov_b32 {S_KEY0}, 0")
    o.e(f"v_mov_b32 v{f.MC}, {START_REFERENCE}")
    o.e(f"v_mov_b32 v{f.LRUN}, 0")
    for r in accumulators(f):
        o.e(f"v_mov_b32 v{r}, 0" if f.acc_file == "v" else f"v_accvgpr_write_b32 a{r}, 0")


def item_blocks(o):
    """S_NB / requests left from S_ROW0: the 32-key blocks any row of the item can see."""
    o.e(f"s_add_u32 s88, {S_ROW0}, 32")
    o.e(f"s_min_i32 s88, s88, {S_SQ}")
    o.e(f"s_add_u32 s88, s88, {S_OFFSET}")
    o.e(f"s_min_i32 s88, s88, {S_SKV}")
    o.e(f"s_cmp_eq_u32 {S_CAUSAL}, 0")
    o.e(f"s_cselect_b32 s88, {S_SKV}, s88")
    o.e("s_max_i32 s88, s88, 1")                        # (at least one block: they are counted down to zero)
    o.e("s_add_u32 s88, s88, 31")
    o.e(f"s_lshr_b32 {S_NB}, s88, 5")
    o.e(f"s_mov_b32 {S_KLEFT}, {S_NB}")
    o.e(f"s_mov_b32 {S_VLEFT}, {S_NB}")


def normalise(o, f):
    """Normalises the item's accumulators and packs them: lane (n, h) holds, in accumulator
    register 16 db + 4 j + i, head-dim element 32 db + 8 j + 4 h + i of query row n, and ends with 16-byte chunk 4 db + 2 jp + h
    of the row in registers S[0] + 8 db + 4 jp ...  (The plain loop divides; v_rcp_f32 and the product are within two units of float of
    that, and the results are rounded to bfloat16, whose unit is 2^16 of those.)"""
    o.e(f"v_mov_b32 v{f.MB}, v{f.LRUN}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{f.LRUN}, v{f.MB}")
    o.e("s_nop 1")
    o.e(f"v_add_f32 v{f.ALPHA}, v{f.LRUN}, v{f.MB}")          # the row's sum: both halves of its keys
    o.e(f"v_rcp_f32 v{f.ALPHA}, v{f.ALPHA}")
    o.e("s_nop 1")
    if f.acc_file == "v":
        scale_accumulators(o, f)
        for i in range(f.d // 4):
            o.e(f"v_cvt_pk_bf16_f32 v{f.S[0] + i}, v{f.ACC[0] + 2 * i}, v{f.ACC[0] + 2 * i + 1}")
    else:
        for i in range(f.d // 4):
            t = (f.T[2 * (i % 2)], f.T[2 * (i % 2) + 1])
            for k in range(2):
                o.e(f"v_accvgpr_read_b32 v{t[k]}, a{f.ACC[0] + 2 * i + k}")
                o.e(f"v_mul_f32 v{t[k]}, v{f.ALPHA}, v{t[k]}")
            o.e(f"v_cvt_pk_bf16_f32 v{f.S[0] + i}, v{t[0]}, v{t[1]}")
    o.e("s_nop 1")
    # The two lanes of a row trade halves, so that each holds 16 consecutive bytes: lane (n, 0) keeps its block j and
    # takes (n, 1)'s, lane (n, 1) ends with both blocks j + 1.
    for db in range(f.d // 32):
        for jp in range(2):
            x = f.S[0] + 8 * db + 4 * jp
            o.e(f"v_permlane32_swap_b32 v{x}, v{x + 2}")
            o.e(f"v_permlane32_swap_b32 v{x + 1}, v{x + 3}")
    o.e("s_nop 3")


def direct_store(o, f):
    """From the lanes as they are, a row's 32 bytes per instruction (the rings belong to the next item already).  The output pointer of
    lane (n, h) is row n's plus 16 h bytes."""
    o.e(f"s_and_saveexec_b64 s[62:63], {S_STOREMASK}")
    o.e("s_nop 1")
    for db in range(f.d // 32):
        for jp in range(2):
            src = f.S[0] + 8 * db + 4 * jp
            o.e(f"global_store_dwordx4 v[{f.OUTP}:{f.OUTP + 1}], v[{src}:{src + 3}], off offset:{64 * db + 32 * jp} nt")   # written once, read by a later kernel
    o.e("s_mov_b64 exec, s[62:63]")
    o.e("s_nop 1")


def store_rows(o, f):
    """The packed rows through LDS, so that a store writes whole rows (1 KiB) and not 32 bytes of each of 32 rows: a short pass waited
    0.85 us for those.  Slot w of the K ring (nobody reads it behind the last barrier) takes the 32 rows of wavefront w in the layout of a K
    block: chunk 2 s + h of row n lies where the lane's K fragment s does."""
    rpi, chunks = 512 // f.d, f.d // 8  # rows per instruction, 16-byte chunks per row
    swizzle = lambda r: r & 15 if f.d >= 128 else r >> 1 & 7
    for s in range(f.d // 16):
        o.e(f"v_add_u32 v{f.T[s % 4]}, {S_OUTSLOT}, v{f.KOFF + s}")
        o.e(f"ds_write_b128 v{f.T[s % 4]}, {vr(f.S[0] + 4 * s, 4)}")
    # lane l reads and stores chunk l % chunks of row rpi i + l / chunks
    lane, row, off = f.LIMREL, f.VROW, f.VT0
    o.e(f"v_lshl_add_u32 v{lane}, v{f.V4H}, 3, v{f.VN}")
    o.e(f"v_lshrrev_b32 v{row}, {chunks.bit_length() - 1}, v{lane}")
    o.e(f"v_and_b32 v{off}, {chunks - 1}, v{lane}")
    if f.d >= 128:
        o.e(f"v_xor_b32 v{f.MB}, v{off}, v{row}")
    else:
        o.e(f"v_lshrrev_b32 v{f.MB}, 1, v{row}")
        o.e(f"v_xor_b32 v{f.MB}, v{off}, v{f.MB}")
    o.e(f"v_lshlrev_b32 v{f.MB}, 4, v{f.MB}")
    o.e(f"v_lshl_add_u32 v{f.MB}, v{row}, {(2 * f.d).bit_length() - 1}, v{f.MB}")
    o.e(f"v_add_u32 v{f.MB}, {S_OUTADDR}, v{f.MB}")
    n = 32 // rpi
    for i in range(n):
        x = 16 * swizzle(rpi * i)
        if x:
            o.e(f"v_xor_b32 v{f.T[i % 4]}, 0x{x:x}, v{f.MB}")
        o.e(f"ds_read_b128 {vr(f.S[0] + 4 * i, 4)}, v{f.T[i % 4] if x else f.MB} offset:{1024 * i}")
    o.e(f"v_add_u32 v{f.MCN}, {S_ROW0}, v{row}")
    o.e(f"v_mov_b32 v{f.PTMP}, s28")
    o.e(f"v_mov_b32 v{f.PTMP + 1}, s29")
    o.e(f"v_mad_u64_u32 v[{f.PTMP}:{f.PTMP + 1}], s[92:93], v{f.MCN}, {S_OTS}, v[{f.PTMP}:{f.PTMP + 1}]")
    o.e(f"v_mad_u64_u32 v[{f.PTMP}:{f.PTMP + 1}], s[92:93], v{off}, 16, v[{f.PTMP}:{f.PTMP + 1}]")
    o.e(f"s_mul_hi_u32 s89, {S_OTS}, {rpi}")
    o.e(f"s_mul_i32 s88, {S_OTS}, {rpi}")
    o.e(f"s_sub_u32 s94, {S_SQ}, {S_ROW0}")                       # rows that exist
    o.e("s_mov_b64 s[62:63], exec")
    o.e("s_cmp_lt_i32 s94, 32")
    o.e("s_cbranch_scc1 L_some_rows%=")
    for some in (False, True):
        for i in range(n):
            if some:
                o.e(f"v_cmp_gt_i32_e64 s[92:93], s94, v{row}")
                o.e(f"s_sub_u32 s94, s94, {rpi}")
            o.e(f"s_waitcnt lgkmcnt({min(n - 1 - i, 15)})" if not some or i == 0 else "s_nop 0")
            if some:
                o.e("s_mov_b64 exec, s[92:93]")
                o.e("s_nop 1")
            o.e(f"global_store_dwordx4 v[{f.PTMP}:{f.PTMP + 1}], {vr(f.S[0] + 4 * i, 4)}, off nt")   # written once, read by a later kernel
            if some:
                o.e("s_mov_b64 exec, s[62:63]")
            o.e(f"v_lshl_add_u64 v[{f.PTMP}:{f.PTMP + 1}], v[{f.PTMP}:{f.PTMP + 1}], 0, s[88:89]")
        if not some:
            o.e("s_branch L_stored%=")
            o.label("L_some_rows")
            o.e("s_waitcnt lgkmcnt(0)")
    o.label("L_stored")
    o.e("s_nop 1")


def partial_epilogue(o, f):
    """The accumulators of a part of the keys as floats, register group by register group in the order in
    which the lanes hold them (a store writes 1 KiB), and (reference, sum) per row."""
    o.e(f"v_mov_b32 v{f.MB}, v{f.LRUN}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{f.LRUN}, v{f.MB}")
    o.e("s_nop 1")
    o.e(f"v_add_f32 v{f.S[0] + 1}, v{f.LRUN}, v{f.MB}")
    o.e(f"v_mov_b32 v{f.S[0]}, v{f.MC}")
    o.e(f"v_lshlrev_b32 v{f.VT0}, 3, v{f.VN}")
    o.e(f"v_lshlrev_b32 v{f.PTMP}, 4, v{f.VN}")
    o.e(f"v_lshl_add_u32 v{f.PTMP}, v{f.V4H}, 7, v{f.PTMP}")      # 16 times the lane
    for g in range(f.d // 8):
        if g and g % 4 == 0:
            o.e("s_add_u32 s38, s38, 4096")
            o.e("s_addc_u32 s39, s39, 0")
        o.e(f"global_store_dwordx4 v{f.PTMP}, {vr(f.ACC[0] + 4 * g, 4, f.acc_file)}, {S_PART} offset:{1024 * (g % 4)}")
    o.e(f"global_store_dwordx2 v{f.VT0}, v[{f.S[0]}:{f.S[0] + 1}], {S_STATS}")   # (both lanes of a row: the same values)


def last_epilogue(o, f):
    if f.parts:
        o.e(f"s_cmp_lg_u64 {S_PART}, 0")
        o.e("s_cbranch_scc1 L_partial%=")
    normalise(o, f)
    store_rows(o, f)
    if f.parts:
        o.e("s_branch L_done%=")
        o.label("L_partial")
        partial_epilogue(o, f)
        o.label("L_done")


def next_item(o, f):
    """Behind the last PV of an item: is there another one?  Its Q fragments and first requests go
    out first, then the finished item is stored, then the state of the new one is set up."""
    paged = f.paged
    o.e(f"s_add_u32 {S_K}, {S_K}, 1")
    o.e(f"s_mul_i32 s88, {S_K}, {S_SPG}")
    o.e(f"s_sub_u32 s89, {S_SPG}, 1")
    o.e(f"s_sub_u32 s89, s89, {S_J}")
    o.e(f"s_bitcmp1_b32 {S_K}, 0")
    o.e(f"s_cselect_b32 s89, s89, {S_J}")               # odd items are dealt in the other direction
    o.e("s_add_u32 s88, s88, s89")                      # d: the item's rank among the row blocks, heavy first
    o.e(f"s_cmp_ge_u32 s88, {S_NQT}")
    o.e("s_cbranch_scc1 L_last_item%=")
    o.e(f"s_sub_u32 s88, {S_NQT}, s88")
    o.e("s_sub_u32 s88, s88, 1")
    o.e(f"s_lshl_b32 {S_ROW0}, s88, 5")                 # (the finished item's pointers and store mask stay in registers)
    o.e("s_barrier")                                    # everybody has left the rings
    o.e(f"v_add_u32 v{f.VROW}, {S_ROW0}, v{f.VN}")
    o.e(f"s_sub_u32 s88, {S_SQ}, 1")
    o.e(f"v_min_i32 v{f.VROW}, s88, v{f.VROW}")
    o.e(f"v_mad_u64_u32 v[{f.PTMP}:{f.PTMP + 1}], s[92:93], v{f.VROW}, {S_QTS}, v[{f.QBASE}:{f.QBASE + 1}]")
    for ks in range(f.d // 16):
        o.e(f"global_load_dwordx4 {vr(f.QF + 4 * ks, 4)}, v[{f.PTMP}:{f.PTMP + 1}], off offset:{32 * ks}")
    item_blocks(o)
    if paged:
        o.e("s_mov_b64 s[84:85], s[50:51]")
        o.e("s_mov_b64 s[86:87], s[52:53]")
        o.e(f"v_mov_b32 v{f.PTREQ}, s54")
        o.e(f"s_mov_b32 {S_CIN}, s55")
        o.e(f"s_mov_b32 {S_RIN}, s56")
        o.e("s_mov_b64 s[82:83], s[58:59]")
        o.e(f"s_sub_u32 s88, {S_NB}, 1")
        o.e("s_lshr_b32 s88, s88, 1")
        o.e("s_sub_u32 s88, s88, 3")
        o.e("s_max_i32 s88, s88, 0")
        o.e(f"s_mov_b32 {S_RLEFT}, s88")
    else:
        o.e("s_mov_b64 s[64:65], s[50:51]")
        o.e("s_mov_b64 s[66:67], s[52:53]")
    for ln in generate_first(f, "nx", f.ns):
        o.lines.append(ln)
    normalise(o, f)
    direct_store(o, f)
    item_setup(o, f, "nx")
    o.e("s_branch L_item_top%=")
    o.label("L_last_item")
    last_epilogue(o, f)


def first_offsets(f):
    """Paged: the registers of the first byte offsets, one per tile of 64 keys (`paged` 64) or per block of 32.  The loop
    goes on with the last two: K's and V's tiles, or the next two V blocks."""
    if f.paged == 64:
        return ([S_OFF0] if f.ns == 5 else []) + [S_OFFV, S_OFFK]
    return ["s[50:51]", "s[52:53]"] + (["s[58:59]"] if f.ns == 5 else []) + [S_OFFV, S_OFF0]


def first_request(o, f, which, j, tag):
    """K or V block j, one of the first, into slot j."""
    if not f.paged:
        request_block(o, f, which, j, tag, 0)
        return
    left, lane, base, ring = (S_KLEFT, f.LDK, 64, 0) if which == "K" else (S_VLEFT, f.LDV, 66, f.vring)
    lo = int(first_offsets(f)[j // 2 if f.paged == 64 else j][2:4])
    o.e(f"s_cmp_eq_u32 {left}, 0")
    o.e(f"s_cbranch_scc1 L_no{which}_{tag}%=")
    o.e(f"s_add_u32 s90, s{base}, s{lo}")
    o.e(f"s_addc_u32 s91, s{base + 1}, s{lo + 1}")
    if j % 2 and f.paged == 64:
        o.e(f"s_add_u32 s90, s90, {f.SLOT}")
        o.e("s_addc_u32 s91, s91, 0")
    o.e(f"s_add_u32 m0, {S_M0B}, {ring + j * f.SLOT}")
    o.e("s_nop 0")
    block_loads(o, f, lane, "s[90:91]")
    o.e(f"s_sub_u32 {left}, {left}, 1")
    o.label(f"L_no{which}_{tag}")


def generate_first(f, suffix="", blocks=0):
    """The first requests: K blocks 0 .. blocks - 1, V blocks 0 .. blocks - 3 (a block of assembly of its own, so that the caller can
    put its set-up behind them).  At first ns - 1: the slots of the next ones, and those that no V block is in yet, hold Q rows."""
    o = Out()
    blocks = blocks or f.ns - 1
    for j in range(blocks):
        first_request(o, f, "K", j, f"pro{j}{suffix}")
    for j in range(blocks - 2):
        first_request(o, f, "V", j, f"pro{j}{suffix}")
    return o.lines


READ_AFTER_WRITE, WRITE_AFTER_READ = 2, 2  # matrix instructions in between, at least (see the top)


def vector_registers(operand):
    """The numbers of the vector registers that an operand names."""
    m = re.match(r"-?v(?:(\d+)|\[(\d+):(\d+)\])$", operand)
    return range(0) if not m else range(int(m[1]), int(m[1]) + 1) if m[1] else range(int(m[2]), int(m[3]) + 1)


def check_distances(f, lines):
    """(fewest matrix instructions between the last write of a score register and a vector instruction that reads it, and between
    the last read of a probability register and one that writes it) in the unrolled iterations, taken twice round.  The mask of a block, behind its
    branch, waits by itself."""
    top, end = lines.index("L_it1%=:"), lines.index("s_branch L_it1%=")
    scores = {r for bank in f.S for r in range(bank, bank + 16)}
    probabilities = {r for bank in f.P for r in range(bank, bank + 8)}
    written, read, n, masked = {}, {}, 0, False
    fewest = [len(lines), len(lines)]
    for line in lines[top:end] * 2:
        if line.startswith("s_cbranch_scc1 L_nomask"):
            masked = True
        if line.startswith("L_nomask"):
            masked = False
        name, _, rest = line.partition(" ")
        operands = [x.strip() for x in rest.split(",")]
        if name.startswith("v_mfma"):
            n += 1
            written.update((r, n) for r in vector_registers(operands[0]) if r in scores)
            read.update((r, n) for r in vector_registers(operands[2]) if r in probabilities)
        elif name.startswith("v_") and not masked:
            for r in (r for x in operands[1:] for r in vector_registers(x) if r in written):
                fewest[0] = min(fewest[0], n - written[r])
            for r in (r for r in vector_registers(operands[0]) if r in read):
                fewest[1] = min(fewest[1], n - read[r])
    assert fewest[0] >= READ_AFTER_WRITE and fewest[1] >= WRITE_AFTER_READ, (f.name, fewest)
    return tuple(fewest)


def generate(f):
    o = Out()
    assert (f.ns, f.unroll) in ((5, 10), (4, 4))
    o.e(f"v_mov_b32 v{f.VZERO}, 0")
    item_setup(o, f, "first")
    # The Q rows of wavefront w lie, in the layout of a K block, in the slot of K block ns - 1 or of V blocks ns - 3 ...: fragment ks at
    # the lane's K fragment's place.  Once all wavefronts have them, the blocks of those slots are requested.
    o.e("s_waitcnt vmcnt(0)")
    for ks in range(f.d // 16):
        o.e(f"v_add_u32 v{f.T[ks % 4]}, {S_QSLOT}, v{f.KOFF + ks}")
        o.e(f"ds_read_b128 {vr(f.QF + 4 * ks, 4)}, v{f.T[ks % 4]}")
    o.e("s_waitcnt lgkmcnt(0)")
    o.e("s_barrier")
    first_request(o, f, "K", f.ns - 1, "late")
    first_request(o, f, "V", f.ns - 3, "late")
    if f.items:
        o.e("s_branch L_start%=")
        o.label("L_item_top")
        o.e("s_waitcnt vmcnt(0)")
        o.e("s_barrier")
        o.label("L_start")
    # ---- S(0) from K block 0; behind it the fragments of iteration 0 (K block 1) ------------------
    pairs = score_pairs(0, 0, f)
    it0 = iteration_pairs(0, f, has_pv=False)
    behind = [frag for _, frag in it0] + first_frags(1, f)
    phase = stream(o, f, pairs, [[] for _ in pairs], 0, False, behind[:NSLOT])
    # ---- iteration 0: S(1), sm(0) ---------------------------------------------------------------
    o.e("s_nop 7")
    iteration_head(o, f, 0, "i0")
    phase = stream(o, f, it0, spread(softmax_ops(f, 0), len(it0)), phase, True, first_frags(1, f))
    iteration_tail(o, f, "i0", "L_exit0")
    phases = {0: phase}  # ring slot of the next iteration's first fragment, behind iteration p
    # ---- iterations 1 .. : `unroll` in a row, then round again -----------------------------------------
    for k in range(f.unroll):
        p = (k + 1) % f.unroll
        o.label(f"L_it{p}")
        iteration_head(o, f, p, f"p{p}")
        pairs = iteration_pairs(p, f)
        phase = stream(o, f, pairs, spread(softmax_ops(f, p % 2), len(pairs)), phase, True, first_frags(p + 1, f))
        assert phases.setdefault(p, phase) == phase  # (iteration 0 and iteration `unroll` share an exit)
        iteration_tail(o, f, f"p{p}", f"L_exit{p}")
    o.e("s_branch L_it1%=")

    # ---- exits: PV of the last block i = p (mod unroll) -----------------------------------------------
    # The ring holds the first fragments of the iteration that is not coming, some of V block i among
    # them; the others take the slots of the K fragments nobody needs.
    for p in range(f.unroll):
        o.label(f"L_exit{p}")
        o.e("s_waitcnt lgkmcnt(0)")
        held = {frag: (phases[p] + j) % NSLOT for j, frag in enumerate(first_frags(p + 1, f)) if frag[0] == "V"}
        db = f.d // 32
        wanted = [("V", p % f.ns, x // db, x % db) for x in range(2 * db)]
        free = [x for x in range(NSLOT) if x not in held.values()]
        missing = [frag for frag in wanted if frag not in held]
        slots = dict(held)
        for k, frag in enumerate(missing[:len(free)]):
            slots[frag] = free[k]
            for x in frag_reads(f, frag, slots[frag]):
                o.e(x)
        for frag in sorted(held, key=wanted.index):
            o.e(mfma(f, ("PV", frag[3], p % 2, frag[2]), slots[frag]))
        batch, rest = missing[:len(free)], missing[len(free):]
        while batch:
            o.e("s_waitcnt lgkmcnt(0)")
            for frag in batch:
                o.e(mfma(f, ("PV", frag[3], p % 2, frag[2]), slots[frag]))
            batch, rest = rest[:NSLOT], rest[NSLOT:]
            for k, frag in enumerate(batch):
                slots[frag] = k
                for x in frag_reads(f, frag, k):
                    o.e(x)
        o.e("s_branch L_end%=")

    slow_path(o, f, 0, "L_slow_i0", "L_join_i0", first=True)
    for p in range(f.unroll):
        slow_path(o, f, p % 2, f"L_slow_p{p}", f"L_join_p{p}")
        few_left(o, f, f"p{p}")
    o.label("L_end")
    o.e("s_nop 15")
    o.e("s_nop 15")
    if f.items:
        next_item(o, f)
    else:
        last_epilogue(o, f)
    check_distances(f, o.lines)
    return o.lines


def bind(reg, value, inout=False, file="v", n=1):
    """An operand bound to a register (a name like "s[64:65]", or the first of `n` of a file)."""
    return f'"{"+" if inout else ""}{{{vr(reg, n, file) if isinstance(reg, int) else reg}}}"({value})'


def operands(f):
    """(outputs, inputs) of the first requests and of the block behind them, by the names that prefill_kernel
    in prefill_stream_kernel.h gives the values."""
    io = lambda reg, value, n=1: bind(reg, value, True, n=n)
    i = lambda reg, value, n=1: bind(reg, value, n=n)
    offs = [(reg, f"off[{k}]") for k, reg in enumerate(first_offsets(f))] if f.paged else []
    loads = [i(f.LDK, "ldk", f.tensor_loads), i(f.LDV, "ldv", f.tensor_loads)]
    wide_in = [i(f.LDKP, "ldp"), i(S_PSTRIDE, "wide.stride"), i(S_M0P, "wide.m0"), i(S_VSTRIDE, "wide.v_stride")] if f.wide else []
    wide_io = [io(S_PBASE, "wide.base")] if f.wide else []
    bases = [(S_KBASE, "req.kbase"), (S_VBASE, "req.vbase")]
    counts = [io(S_KLEFT, "req.k_requests"), io(S_VLEFT, "req.v_requests")]
    if f.paged:
        first = counts, loads + [i(*b) for b in bases] + [i(S_M0B, "req.m0_base")] + [i(*x) for x in offs]
    else:
        first = [io(*b) for b in bases] + counts + wide_io, loads + [i(S_STRIDE, "req.stride"), i(S_M0B, "req.m0_base")] + wide_in
    outs = [io(*b) for b in bases] + counts + wide_io
    outs += [io(S_NB, "nblk"), io(S_K, "it.k"), io(S_ROW0, "it.row0"), io(S_KEY0, "it.key0")]
    ins = [i(f.KOFF, "ko", f.d // 16), i(f.VOFF, "vo", f.d // 32)] + loads + wide_in
    ins += [i(f.VN, "n"), i(f.V4H, "h4"), i(S_QSLOT, "q_slot"), i(S_OUTSLOT, "out_slot"), i(S_OUTADDR, "out_address"), i(S_OUT, "out_row0")]
    if f.items:
        ins += [i(f.QBASE, "q_base", 2), i(f.OUTBASE, "out_base", 2)]
    ins += [i(S_STRIDE, "req.stride"), i(S_C, "a.scale_log2e"), i(S_M0B, "req.m0_base"), i(S_J, "it.j"), i(S_SPG, "it.spg"), i(S_NQT, "it.nqt"),
            i(S_SQ, "it.sq"), i(S_SKV, "it.skv"), i(S_OFFSET, "it.offset"), i(S_CAUSAL, "it.causal"), i(S_QTS, "it.q_row_bytes"),
            i(S_OTS, "it.out_row_bytes")]
    if f.wide:
        ins += [i(f.QFP, "q_second", 16), i(f.KOFFP, "po", 4)]
    if f.window:
        ins += [i(f.LOWEST, "lowest"), i(S_LOWTO, "low_to")]
    if f.paged:
        outs += [io(S_CIN, "tab.read_in_block"), io(S_RIN, "tab.request_in_block"), io(S_RPTR, "tab.entry_ptr"), io(S_RLEFT, "tab.entry_requests"),
                 io(f.PTREQ, "tab.entry"), io(S_PART, "out_part.acc")] + [io(*x) for x in offs[-2:]]
        ins += [i(S_HKV, "tab.kv_heads"), i(S_HK, "tab.kv_head"), i(S_NCB, "tab.num_blocks"), i(S_TPB, "tab.per_block"), i(S_STATS, "out_part.stats")]
        if f.paged == 32:
            outs += [io(f.PTREQ2, "tab.entry2")]
            ins += [i(*offs[f.ns - 3])]
    if f.items and f.paged:  # where the items that follow start
        ins += [i(S_OFF0, "off[0]"), i("s[50:51]", "off[1]"), i("s[52:53]", "off[2]"), i("s54", "tab.entry"), i("s55", "tab.read_in_block"),
                i("s56", "tab.request_in_block"), i("s[58:59]", "tab.entry_ptr")]
    elif f.items:
        ins += [i("s[50:51]", "kbase0"), i("s[52:53]", "vbase0")]
    return first, (outs, ins)


def registers(text):
    """Every vector, accumulation and scalar register that a text names."""
    found = set()
    for file, single, lo, hi in re.findall(r"\b([vas])(?:(\d+)|\[(\d+):(\d+)\])", text):
        found |= {f"{file}{r}" for r in (range(int(single), int(single) + 1) if single else range(int(lo), int(hi) + 1))}
    return found


def write_asm(out, macro, lines, outs, ins):
    """An asm statement's text, operands and clobbers (whatever the text names and no operand is bound to)."""
    bound = [registers(x.split("(")[0]) for x in outs + ins]
    for k, x in enumerate(bound):
        assert not any(x & y for y in bound[:k]), (macro, (outs + ins)[k])
    clobbers = registers("\n".join(lines)) - set().union(*bound)
    out.write(f"#define {macro} \\\n")
    for ln in lines:
        out.write(f'  "{ln}\\n\\t" \\\n')
    named = sorted(clobbers, key=lambda r: (r[0], int(r[1:])))
    out.write(f'  "" : {", ".join(outs)} : {", ".join(ins)} : "memory", "vcc", "scc", "m0"' + "".join(f', "{r}"' for r in named) + "\n")


def main():
    with open(sys.argv[1] if len(sys.argv) > 1 else "/dev/stdout", "w") as out:
        out.write("// Generated by gen_prefill_stream.py; do not edit.\n#pragma once\n")
        for form in FORMS:
            first, loop = operands(form)
            write_asm(out, f"TTPA_STREAM_FIRST_{form.name}", generate_first(form), *first)
            write_asm(out, f"TTPA_STREAM_LOOP_{form.name}", generate(form), *loop)
        out.write(f"#define TTPA_STREAM_SLOTS(d, wide) ((wide) || (d) == 256 ? 4 : 5)\n")
        for form in FORMS:
            assert form.ns == (4 if form.wide or form.d == 256 else 5)


if __name__ == "__main__":
    main()
