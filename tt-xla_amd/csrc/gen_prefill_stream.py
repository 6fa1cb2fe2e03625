#!/usr/bin/env python3
"""Writes the hand-scheduled loop of the streaming prefill kernel (head size 128, 32 query rows of one
head per wavefront, two workgroups of four wavefronts per CU) as one block of gfx950 assembly per
form of the loop: build/prefill_stream_asm.h, included by prefill_stream.hip.  The forms: dense
K / V, dense with a sliding window, dense with keys of 128 + 64 features (the second part, the rotary
one, with base and strides of its own), paged K / V in cache blocks of whole 64-key tiles, and in
cache blocks of whole 32-key blocks.

Why assembly: the loop wants the matrix pipe and the vector ALU of a SIMD busy at the same time
from one instruction stream, with every register chosen by hand (256 per wavefront at two
wavefronts per SIMD) and every wait counted.  The unit of work is a BLOCK of 32 keys:

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

LDS: a ring of NS slots of 8 KiB (32 rows) for K blocks and one for V blocks; block j lives in
slot j % NS.  Iteration i reads K block i + 1 and V block i - 1 and, through the running fragment
reads, the first fragments of K block i + 2 and V block i.  Its barrier, at its start, says that
nobody reads K block i and V block i - 2 any more; K block i + NS and V block i + NS - 2 are
requested into their slots (LDS-DMA loads, two per tensor and wavefront).  A request has to have
landed NS - 2 barriers later: the wait in front of a barrier lets the requests of the last NS - 3
barriers stay in flight (vmcnt(8)), so a tile has three iterations to arrive with NS = 5, where
two stages of whole tiles gave it two.  Once requests have been skipped (no such block) the wait
is for everything.  Dense K / V: a block is `stride` bytes behind the one before.  Paged (block
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
between the Q fragments and the stored output rows: its first requests (K blocks 0..NS-1, V blocks
0..NS-3; for the first item they are a block of assembly of their own, so that the caller's Q loads
overlap them), all blocks, the last PV, normalisation and store; then the next item's Q fragments
and first requests go out in front of the store of the finished one.

Matrix-to-vector hazards the hardware does not interlock are kept by construction: the vector
instructions that read a score bank start two matrix instructions after the last one that wrote
it (the mask waits explicitly); a bank of probabilities is rewritten three matrix instructions
after the last one that read it; the slow path and the exit wait out the matrix pipe with s_nop.
"""

import sys


# ---- register map (vector registers) ---------------------------------------------------------
ACC = [0, 16, 32, 48]          # output accumulators, head-dim blocks 0..3 (inputs / outputs)
QF = 64                        # Q fragments, k-step ks at QF + 4 ks (inputs)
S = [96, 112]                  # score banks
P = [128, 136]                 # probability banks (8 packed pairs each)
RING = 144                     # 8 fragment slots of 4 registers
NSLOT = 8
KOFF = 176                     # LDS byte address of the lane's K fragment in K slot 0, k-step ks (inputs)
VOFF = 184                     # ... of the lane's V^T fragment in V slot 0, output block db (inputs)
LDK = 188                      # per-lane global byte offsets of the 2 K loads of a block (inputs)
LDV = 190                      # ... of the 2 V loads
MC, LRUN, LSUM, ALPHA = 196, 197, 198, 199   # MC, LRUN: inputs / outputs
T = [200, 201, 202, 203]
ORV, MLOC, MB, MCN = 204, 205, 206, 207
PTREQ = 208                    # paged: the requested block-table entry (input)
PTREQ2 = 211                   # blocks of 32: the entry requested in odd iterations (input)
LOWEST, LOWREL = 209, 210      # window: first visible key of the lane's row, minus 4 h (input); relative to the block
LIMIT = 212                    # last visible key of the lane's row, minus 4 h (input)
LIMREL, NEGINF, VZERO = 213, 214, 215
QBASE, OUTBASE = 216, 218      # per lane, 64-bit: q / out of row 0 of the lane's head, at the lane's 8 h / 4 h elements (inputs)
VN, V4H = 220, 221             # lane % 32 and 4 (lane / 32) (inputs)
QFP, KOFFP, LDKP = 228, 244, 248  # keys of 128 + 64: Q fragments, LDS addresses and global offsets of the second part (inputs)
OUTP, PTMP, VT0, VROW = 222, 224, 226, 227
CLOBBERED = (list(range(0, QF)) + list(range(S[0], RING + 4 * NSLOT)) + list(range(MC, MCN + 1)) + [LOWREL, LIMIT, LIMREL, NEGINF, VZERO]
             + list(range(OUTP, VROW + 1)))

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
# temporaries s[88:95], s[62:63]
SCALAR_CLOBBERS = [f"s{r}" for r in list(range(88, 96)) + [60, 61, 62, 63, 74]]

SLOT, PSLOT = 8192, 4096       # bytes of a block of K or V, of the second part of K
KEY_CONST = [8 * (r // 4) + r % 4 for r in range(16)]


class Form:
    """What one block of assembly serves."""

    def __init__(self, name, paged=0, window=False, wide=False):
        self.name, self.paged, self.window = name, paged, window  # paged: 0 or the keys that share a table entry
        self.wide = wide                    # keys of 128 + 64 features
        self.ns = 4 if wide else 5          # slots per ring
        self.unroll = 4 if wide else 10     # lcm(2, ns): score bank and slots repeat
        self.vring = self.ns * SLOT         # LDS offset of the V ring (VOFF carries it), of the second part's ring (KOFFP)
        self.pring = 2 * self.vring
        self.loads = 5 if wide else 4       # tile loads of an iteration
        self.items = not window and not wide and paged != 32  # several row blocks in turn
        self.parts = paged > 0  # may take a part of the keys


FORMS = [Form("DENSE"), Form("DENSE_WINDOW", window=True), Form("DENSE_WIDE", wide=True), Form("PAGED", paged=64),
         Form("PAGED32", paged=32)]
START_REFERENCE = "0xff7fffff"  # the lowest finite float


class Out:
    def __init__(self):
        self.lines = []

    def e(self, s):
        self.lines.append(s)

    def label(self, name):
        self.lines.append(name + "%=:")


def vr(a, n=1):
    return f"v{a}" if n == 1 else f"v[{a}:{a + n - 1}]"


def frag_reads(frag, slot):
    """LDS read instructions of a fragment into ring slot `slot`.
    ("K", LDS slot, k-step) or ("V", LDS slot, key step 0 / 1, output block)."""
    base = RING + 4 * slot
    if frag[0] == "K" and frag[2] >= 8:
        return [f"ds_read_b128 {vr(base, 4)}, v{KOFFP + frag[2] - 8} offset:{frag[1] * PSLOT}"]
    if frag[0] == "K":
        _, ls, ks = frag
        return [f"ds_read_b128 {vr(base, 4)}, v{KOFF + ks} offset:{ls * SLOT}"]
    _, ls, k4, db = frag
    off = ls * SLOT + k4 * 4096
    return [f"ds_read_b64_tr_b16 {vr(base, 2)}, v{VOFF + db} offset:{off}",
            f"ds_read_b64_tr_b16 {vr(base + 2, 2)}, v{VOFF + db} offset:{off + 2048}"]


def mfma(m, slot):
    a = vr(RING + 4 * slot, 4)
    if m[0] == "S":
        _, bank, ks = m
        d = vr(S[bank], 16)
        q = QF + 4 * ks if ks < 8 else QFP + 4 * (ks - 8)
        return f"v_mfma_f32_32x32x16_bf16 {d}, {a}, {vr(q, 4)}, {'0' if ks == 0 else d}"
    _, db, bank, k4p = m
    d = vr(ACC[db], 16)
    return f"v_mfma_f32_32x32x16_bf16 {d}, {a}, {vr(P[bank] + 4 * k4p, 4)}, {d}"


def softmax_ops(q, test=True):
    """Vector instructions of sm(i) on bank q, in an order that keeps one instruction between a
    transcendental and its first use."""
    s, p = S[q], P[q]
    A = lambda r: f"v_fma_f32 v{T[r % 4]}, v{s + r}, {S_C}, -v{MC}"
    B = lambda r: f"v_exp_f32 v{T[r % 4]}, v{T[r % 4]}"
    C = lambda j: f"v_cvt_pk_bf16_f32 v{p + j}, v{T[(2 * j) % 4]}, v{T[(2 * j + 1) % 4]}"
    D = lambda j: f"v_dot2c_f32_bf16 v{LSUM}, 0x3f803f80, v{p + j}"
    ops = [f"v_mov_b32 v{LSUM}, 0", A(0), A(1), B(0), B(1)]
    for j in range(8):
        if j < 7:
            ops += [A(2 * j + 2), A(2 * j + 3)]
        ops.append(C(j))
        if j < 7:
            ops += [B(2 * j + 2), B(2 * j + 3)]
        ops.append(D(j))
    if test:
        ops += [f"v_or3_b32 v{ORV}, v{p}, v{p + 1}, v{p + 2}",
                f"v_or3_b32 v{ORV}, v{ORV}, v{p + 3}, v{p + 4}",
                f"v_or3_b32 v{ORV}, v{ORV}, v{p + 5}, v{p + 6}",
                f"v_or_b32 v{ORV}, v{ORV}, v{p + 7}",
                f"v_and_b32 v{ORV}, 0x40004000, v{ORV}",
                f"v_cmp_ne_u32 vcc, 0, v{ORV}"]
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


def stream(o, pairs, valu_chunks, phase, in_flight, tail):
    """pairs: [(matrix instruction, fragment)].  Per pair: wait for its fragment, the matrix
    instruction, the read of the fragment NSLOT pairs on, the vector chunk.  phase: the ring slot of the
    first pair's fragment; in_flight: the first NSLOT fragments have been requested by the code in front
    (else they are requested here); tail: the fragments requested behind the last NSLOT pairs (the next
    iteration's first ones).  Returns the next phase."""
    frags = [f for _, f in pairs] + list(tail)
    n = len(pairs)
    count = lambda f: len(frag_reads(frags[f], 0))
    if not in_flight:
        for f in range(min(NSLOT, len(frags))):
            for x in frag_reads(frags[f], (phase + f) % NSLOT):
                o.e(x)
    for j in range(n):
        after = sum(count(f) for f in range(j + 1, min(j + NSLOT, len(frags))))
        assert after <= 15
        o.e(f"s_waitcnt lgkmcnt({after})")
        o.e(mfma(pairs[j][0], (phase + j) % NSLOT))
        if j + NSLOT < len(frags):
            for x in frag_reads(frags[j + NSLOT], (phase + j) % NSLOT):
                o.e(x)
        for x in valu_chunks[j]:
            o.e(x)
    return (phase + n) % NSLOT


def score_pairs(bank, slot, f):
    return [(("S", bank, x), ("K", slot, x)) for x in range(12 if f.wide else 8)]


def iteration_pairs(p, f, has_pv=True):
    """Iteration i = p (mod f.unroll): S(i + 1) into bank 1 - q from K block i + 1, PV(i - 1) from
    bank 1 - q of the probabilities and V block i - 1."""
    q = p % 2
    scores = score_pairs(1 - q, (p + 1) % f.ns, f)
    if not has_pv:
        return scores
    pv = [(("PV", x % 4, 1 - q, x // 4), ("V", (p - 1) % f.ns, x // 4, x % 4)) for x in range(8)]
    order = "SPSSPSPSSPSPSSPSPSSP" if f.wide else "SP" * 8
    assert order.count("S") == len(scores) and order.count("P") == 8
    scores, pv = iter(scores), iter(pv)
    return [next(scores if x == "S" else pv) for x in order]


def mask_selects(o, f, bank):
    """-inf in place of the scores of the block at S_KEY0 that a lane may not see; the bank has been written."""
    s = S[bank]
    o.e(f"v_subrev_u32 v{LIMREL}, {S_KEY0}, v{LIMIT}")  # limit - 4 h - key0
    o.e(f"v_mov_b32 v{NEGINF}, 0xff800000")
    sel = lambda r: f"v_cndmask_b32_e64 v{s + r}, v{s + r}, v{NEGINF}, s[{88 + 2 * (r % 4)}:{89 + 2 * (r % 4)}]"
    sides = [("v_cmp_gt_i32_e64", LIMREL)]
    if f.window:
        o.e(f"v_subrev_u32 v{LOWREL}, {S_KEY0}, v{LOWEST}")
        sides.append(("v_cmp_lt_i32_e64", LOWREL))
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
            o.e(f"v_max3_f32 v{MLOC}, v{MLOC}, v{S[bank] + r}, v{S[bank] + r + 1}")

    o.label(name)
    o.e("s_nop 15")
    o.e("s_nop 15")
    o.e(f"v_max_f32 v{MLOC}, v{S[q]}, v{S[q] + 1}")
    row_max(q, range(2, 16, 2))
    o.e(f"s_cmp_lt_u32 {S_NB}, 2")              # no next block: its bank holds products of whatever the slot held
    o.e(f"s_cbranch_scc1 L_one_{name}%=")
    skip_unless_masked(o, f, name)
    mask_selects(o, f, 1 - q)                   # (the next iteration masks it again: the same selects)
    o.label(f"L_nomask_{name}")
    row_max(1 - q, range(0, 16, 2))
    o.label(f"L_one_{name}")
    o.e(f"v_mov_b32 v{MB}, v{MLOC}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{MLOC}, v{MB}")
    o.e("s_nop 1")
    o.e(f"v_max_f32 v{MLOC}, v{MLOC}, v{MB}")                 # row maximum (raw score)
    o.e(f"v_fma_f32 v{MB}, v{MLOC}, {S_C}, -v{MC}")           # how far above the reference's zero
    o.e(f"v_cmp_le_f32 vcc, 1.0, v{MB}")                      # p >= 2 somewhere in the row: move
    o.e(f"v_mul_f32 v{MCN}, {S_C}, v{MLOC}")
    o.e(f"v_add_f32 v{MCN}, 0x40e00000, v{MCN}")              # m c + 7
    o.e("s_nop 1")
    o.e(f"v_cndmask_b32 v{MCN}, v{MC}, v{MCN}, vcc")
    if first:  # nothing is accumulated yet: no rescale
        o.e(f"v_mov_b32 v{MC}, v{MCN}")
    else:
        o.e(f"v_sub_f32 v{ALPHA}, v{MC}, v{MCN}")             # 0 where the reference stays
        o.e(f"v_exp_f32 v{ALPHA}, v{ALPHA}")
        o.e(f"v_mov_b32 v{MC}, v{MCN}")
        o.e("s_nop 0")
        o.e(f"v_mul_f32 v{LRUN}, v{LRUN}, v{ALPHA}")
        for r in range(64):
            o.e(f"v_mul_f32 v{r}, v{ALPHA}, v{r}")
    for x in softmax_ops(q, test=False):
        o.e(x)
    o.e("s_nop 4")
    o.e(f"s_branch {join}%=")


def two_loads(o, lane_regs, base):
    """The instruction offset moves the LDS address as well as the global one: load j lands 1024 j
    bytes behind M0 and reads base + lane offset + 1024 j, so the lane offsets carry
    1024 - 1024 j and the bases - 1024."""
    for j in range(2):
        o.e(f"global_load_lds_dwordx4 v{lane_regs + j}, {base} offset:{1024 * j}")


def request_block(o, f, which, slot, tag, half):
    """One K or V block into LDS slot `slot` of its ring, if there is one left to request.
    paged: the block is half `half` of the tile at S_OFFK / S_OFFV."""
    paged = f.paged
    left, lane, base, ring = (S_KLEFT, LDK, S_KBASE, 0) if which == "K" else (S_VLEFT, LDV, S_VBASE, f.vring)
    o.e(f"s_cmp_eq_u32 {left}, 0")
    o.e(f"s_cbranch_scc1 L_no{which}_{tag}%=")
    if paged:
        lo, hi = (86, 87) if which == "K" else (84, 85)
        b0 = int(base[2:4])
        o.e(f"s_add_u32 s90, s{b0}, s{lo}")
        o.e(f"s_addc_u32 s91, s{b0 + 1}, s{hi}")
        if half:
            o.e(f"s_add_u32 s90, s90, {SLOT}")
            o.e("s_addc_u32 s91, s91, 0")
    o.e(f"s_add_u32 m0, {S_M0B}, {ring + slot * SLOT}")
    o.e("s_nop 0")
    two_loads(o, lane, "s[90:91]" if paged else base)
    if not paged:
        b0 = int(base[2:4])
        o.e(f"s_add_u32 s{b0}, s{b0}, {S_VSTRIDE if f.wide and which == 'V' else S_STRIDE}")
        o.e(f"s_addc_u32 s{b0 + 1}, s{b0 + 1}, 0")
    if f.wide and which == "K":
        o.e(f"s_add_u32 m0, {S_M0P}, {slot * PSLOT}")
        o.e("s_nop 0")
        o.e(f"global_load_lds_dwordx4 v{LDKP}, {S_PBASE}")
        o.e(f"s_add_u32 s30, s30, {S_PSTRIDE}")
        o.e("s_addc_u32 s31, s31, 0")
    o.e(f"s_sub_u32 {left}, {left}, 1")
    o.label(f"L_no{which}_{tag}")


def next_tile(o, tag):
    """paged, odd iterations: V moves on to the tile K was in, K to the tile whose entry has
    arrived; the entry after that is requested."""
    o.e("s_mov_b64 s[84:85], s[86:87]")
    o.e(f"v_readfirstlane_b32 s88, v{PTREQ}")
    o.e(f"s_cmp_lt_u32 s88, {S_NCB}")
    o.e("s_cselect_b32 s88, s88, 0")
    o.e(f"s_mul_i32 s88, s88, {S_HKV}")
    o.e(f"s_add_u32 s90, s88, {S_HK}")            # cache block * kv_heads + kv_head
    o.e(f"s_mul_hi_u32 s87, s90, {S_STRIDE}")
    o.e(f"s_mul_i32 s86, s90, {S_STRIDE}")
    o.e(f"s_lshl_b32 s90, {S_CIN}, 14")           # 64 tokens of 256 bytes per tile inside the cache block
    o.e("s_add_u32 s86, s86, s90")
    o.e("s_addc_u32 s87, s87, 0")
    o.e(f"s_add_u32 {S_CIN}, {S_CIN}, 1")
    o.e(f"s_cmp_eq_u32 {S_CIN}, {S_TPB}")
    o.e(f"s_cselect_b32 {S_CIN}, 0, {S_CIN}")
    o.e(f"s_cmp_eq_u32 {S_RLEFT}, 0")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"global_load_dword v{PTREQ}, v{VZERO}, {S_RPTR}")
    o.e(f"s_sub_u32 {S_RLEFT}, {S_RLEFT}, 1")
    o.e(f"s_add_u32 {S_RIN}, {S_RIN}, 1")
    o.e(f"s_cmp_lg_u32 {S_RIN}, {S_TPB}")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"s_mov_b32 {S_RIN}, 0")
    o.e("s_add_u32 s82, s82, 4")
    o.e("s_addc_u32 s83, s83, 0")
    o.label(f"L_noreq_{tag}")


def next_block(o, p, tag):
    """Blocks of 32, every iteration: the byte offset of the K block from its table entry; the entry of
    the K block two iterations on is requested."""
    req = PTREQ2 if p % 2 else PTREQ
    o.e(f"v_readfirstlane_b32 s88, v{req}")
    o.e(f"s_cmp_lt_u32 s88, {S_NCB}")
    o.e("s_cselect_b32 s88, s88, 0")
    o.e(f"s_mul_i32 s88, s88, {S_HKV}")
    o.e(f"s_add_u32 s90, s88, {S_HK}")
    o.e(f"s_mul_hi_u32 s87, s90, {S_STRIDE}")
    o.e(f"s_mul_i32 s86, s90, {S_STRIDE}")
    o.e(f"s_lshl_b32 s90, {S_CIN}, 13")           # 32 tokens of 256 bytes per block inside the cache block
    o.e("s_add_u32 s86, s86, s90")
    o.e("s_addc_u32 s87, s87, 0")
    o.e(f"s_add_u32 {S_CIN}, {S_CIN}, 1")
    o.e(f"s_cmp_eq_u32 {S_CIN}, {S_TPB}")
    o.e(f"s_cselect_b32 {S_CIN}, 0, {S_CIN}")
    o.e(f"s_cmp_eq_u32 {S_RLEFT}, 0")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"global_load_dword v{req}, v{VZERO}, {S_RPTR}")
    o.e(f"s_sub_u32 {S_RLEFT}, {S_RLEFT}, 1")
    o.e(f"s_add_u32 {S_RIN}, {S_RIN}, 1")
    o.e(f"s_cmp_lg_u32 {S_RIN}, {S_TPB}")
    o.e(f"s_cbranch_scc1 L_noreq_{tag}%=")
    o.e(f"s_mov_b32 {S_RIN}, 0")
    o.e("s_add_u32 s82, s82, 4")
    o.e("s_addc_u32 s83, s83, 0")
    o.label(f"L_noreq_{tag}")


def iteration_head(o, f, p, tag):
    """Mask, barrier and requests of iteration i = p (mod f.unroll)."""
    paged, ns = f.paged, f.ns
    mask_block(o, f, p % 2, tag)
    # requests of the last ns - 3 barriers may stay in flight, unless some were skipped
    o.e(f"s_cmp_eq_u32 {S_KLEFT}, 0")
    o.e(f"s_cbranch_scc1 L_all_{tag}%=")
    o.e(f"s_waitcnt vmcnt({(ns - 3) * f.loads})")
    o.e(f"s_branch L_bar_{tag}%=")
    o.label(f"L_all_{tag}")
    o.e("s_waitcnt vmcnt(0)")
    o.label(f"L_bar_{tag}")
    o.e("s_barrier")
    if paged == 64 and p % 2 == 1:
        next_tile(o, tag)
    if paged == 32:
        next_block(o, p, tag)
    # K block i + NS is half (i + NS) % 2 of its tile, V block i + NS - 2 the same half of its own
    half = (p + ns) % 2 if paged == 64 else 0
    request_block(o, f, "K", p % ns, tag, half)
    request_block(o, f, "V", (p + ns - 2) % ns, tag, half)
    if paged == 32:
        o.e("s_mov_b64 s[84:85], s[98:99]")
        o.e("s_mov_b64 s[98:99], s[86:87]")


def iteration_tail(o, tag, exit_label):
    o.e(f"s_cbranch_vccnz L_slow_{tag}%=")
    o.label(f"L_join_{tag}")
    o.e(f"v_add_f32 v{LRUN}, v{LRUN}, v{LSUM}")
    o.e(f"s_sub_u32 {S_NB}, {S_NB}, 1")
    o.e(f"s_cmp_eq_u32 {S_NB}, 0")
    o.e(f"s_cbranch_scc1 {exit_label}%=")


def first_frags(p, f):
    """The first NSLOT fragments of iteration p (mod f.unroll)."""
    return [frag for _, frag in iteration_pairs(p % f.unroll, f)[:NSLOT]]


def item_setup(o, tag):
    """Per-item state from S_ROW0: output pointers, the rows' key limits, the mask threshold, cleared
    accumulators and softmax state."""
    o.e(f"v_add_u32 v{VROW}, {S_ROW0}, v{VN}")                                   # the lane's query row
    o.e(f"v_mad_u64_u32 v[{OUTP}:{OUTP + 1}], s[92:93], v{VROW}, {S_OTS}, v[{OUTBASE}:{OUTBASE + 1}]")
    o.e(f"v_cmp_gt_i32_e64 {S_STOREMASK}, {S_SQ}, v{VROW}")                      # rows that exist are stored
    o.e(f"s_sub_u32 s88, {S_SQ}, 1")
    o.e(f"v_min_i32 v{VT0}, s88, v{VROW}")                                       # rows past the end repeat the last one
    o.e(f"v_add_u32 v{VT0}, {S_OFFSET}, v{VT0}")
    o.e(f"s_sub_u32 s89, {S_SKV}, 1")
    o.e(f"v_min_i32 v{VT0}, s89, v{VT0}")                                        # causal: min(offset + row, skv - 1)
    o.e(f"s_add_u32 s88, {S_OFFSET}, {S_ROW0}")
    o.e("s_min_i32 s88, s88, s89")
    o.e(f"s_cmp_eq_u32 {S_CAUSAL}, 0")
    o.e("s_cselect_b32 s88, s89, s88")                                           # the first row's limit
    o.e(f"s_cbranch_scc0 L_causal_{tag}%=")
    o.e(f"v_mov_b32 v{VT0}, s89")                                                # not causal: skv - 1 for every row
    o.label(f"L_causal_{tag}")
    o.e(f"v_sub_u32 v{LIMIT}, v{VT0}, v{V4H}")
    o.e(f"s_sub_u32 {S_MASKFROM}, s88, 30")
    if tag != "first":  # (several row blocks in turn: all of them start at key 0)
        o.e(f"s_mov_b32 {S_KEY0}, 0")
    o.e(f"v_mov_b32 v{MC}, {START_REFERENCE}")
    o.e(f"v_mov_b32 v{LRUN}, 0")
    for r in range(64):
        o.e(f"v_mov_b32 v{r}, 0")


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


def epilogue(o):
    """Normalises the item's accumulators and stores its rows: lane (n, h) holds, in accumulator
    register 16 db + 4 j + i, head-dim element 32 db + 8 j + 4 h + i of query row n.  The output pointer
    of lane (n, h) is row n's plus 16 h bytes."""
    o.e(f"v_mov_b32 v{MB}, v{LRUN}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{LRUN}, v{MB}")
    o.e("s_nop 1")
    o.e(f"v_add_f32 v{ALPHA}, v{LRUN}, v{MB}")          # the row's sum: both halves of its keys
    o.e(f"v_rcp_f32 v{ALPHA}, v{ALPHA}")
    o.e("s_nop 1")
    for r in range(64):
        o.e(f"v_mul_f32 v{r}, v{ALPHA}, v{r}")
    for i in range(32):
        o.e(f"v_cvt_pk_bf16_f32 v{S[0] + i}, v{2 * i}, v{2 * i + 1}")
    o.e("s_nop 1")
    # The two lanes of a row trade halves, so that each stores 16 consecutive bytes (a row's 32 bytes per
    # instruction): lane (n, 0) keeps its block j and takes (n, 1)'s, lane (n, 1) ends with both blocks j + 1.
    for db in range(4):
        for jp in range(2):
            x = S[0] + 8 * db + 4 * jp
            o.e(f"v_permlane32_swap_b32 v{x}, v{x + 2}")
            o.e(f"v_permlane32_swap_b32 v{x + 1}, v{x + 3}")
    o.e("s_nop 3")
    o.e(f"s_and_saveexec_b64 s[62:63], {S_STOREMASK}")
    o.e("s_nop 1")
    for db in range(4):
        for jp in range(2):
            src = S[0] + 8 * db + 4 * jp
            o.e(f"global_store_dwordx4 v[{OUTP}:{OUTP + 1}], v[{src}:{src + 3}], off offset:{64 * db + 32 * jp} nt")   # written once, read by a later kernel
    o.e("s_mov_b64 exec, s[62:63]")
    o.e("s_nop 1")


def partial_epilogue(o):
    """The accumulators of a part of the keys as floats, register group by register group in the order in
    which the lanes hold them (a store writes 1 KiB), and (reference, sum) per row."""
    o.e(f"v_mov_b32 v{MB}, v{LRUN}")
    o.e("s_nop 1")
    o.e(f"v_permlane32_swap_b32 v{LRUN}, v{MB}")
    o.e("s_nop 1")
    o.e(f"v_add_f32 v{S[0] + 1}, v{LRUN}, v{MB}")
    o.e(f"v_mov_b32 v{S[0]}, v{MC}")
    o.e(f"v_lshlrev_b32 v{VT0}, 3, v{VN}")
    o.e(f"v_lshlrev_b32 v{PTMP}, 4, v{VN}")
    o.e(f"v_lshl_add_u32 v{PTMP}, v{V4H}, 7, v{PTMP}")      # 16 times the lane
    for g in range(16):
        if g and g % 4 == 0:
            o.e("s_add_u32 s38, s38, 4096")
            o.e("s_addc_u32 s39, s39, 0")
        o.e(f"global_store_dwordx4 v{PTMP}, v[{4 * g}:{4 * g + 3}], {S_PART} offset:{1024 * (g % 4)}")
    o.e(f"global_store_dwordx2 v{VT0}, v[{S[0]}:{S[0] + 1}], {S_STATS}")   # (both lanes of a row: the same values)


def last_epilogue(o, f):
    if f.parts:
        o.e(f"s_cmp_lg_u64 {S_PART}, 0")
        o.e("s_cbranch_scc1 L_partial%=")
    epilogue(o)
    if f.parts:
        o.e("s_branch L_done%=")
        o.label("L_partial")
        partial_epilogue(o)
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
    o.e(f"v_add_u32 v{VROW}, {S_ROW0}, v{VN}")
    o.e(f"s_sub_u32 s88, {S_SQ}, 1")
    o.e(f"v_min_i32 v{VROW}, s88, v{VROW}")
    o.e(f"v_mad_u64_u32 v[{PTMP}:{PTMP + 1}], s[92:93], v{VROW}, {S_QTS}, v[{QBASE}:{QBASE + 1}]")
    for ks in range(8):
        o.e(f"global_load_dwordx4 {vr(QF + 4 * ks, 4)}, v[{PTMP}:{PTMP + 1}], off offset:{32 * ks}")
    item_blocks(o)
    if paged:
        o.e("s_mov_b64 s[84:85], s[50:51]")
        o.e("s_mov_b64 s[86:87], s[52:53]")
        o.e(f"v_mov_b32 v{PTREQ}, s54")
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
    for ln in generate_first(f, "nx"):
        o.lines.append(ln)
    epilogue(o)
    item_setup(o, "nx")
    o.e("s_branch L_item_top%=")
    o.label("L_last_item")
    last_epilogue(o, f)


FIRST32 = ("s[50:51]", "s[52:53]", "s[58:59]", "s[84:85]", "s[98:99]")  # blocks of 32: the first five byte offsets


def generate_first(f, suffix=""):
    """The first requests: K blocks 0 .. ns - 1, V blocks 0 .. ns - 3 (a block of its own, so that
    the caller can put its Q loads behind them)."""
    o = Out()
    paged = f.paged
    for j in range(f.ns):
        if paged:  # tiles 0, 1, 2 at S_OFF0, S_OFFV, S_OFFK; blocks of 32: 0 .. 4
            src = ("s[98:99]", S_OFFV, S_OFFK)[j // 2] if paged == 64 else FIRST32[j]
            lo = int(src[2:4])
            o.e(f"s_cmp_eq_u32 {S_KLEFT}, 0")
            o.e(f"s_cbranch_scc1 L_noK_pro{j}{suffix}%=")
            o.e(f"s_add_u32 s90, s64, s{lo}")
            o.e(f"s_addc_u32 s91, s65, s{lo + 1}")
            if j % 2 and paged == 64:
                o.e(f"s_add_u32 s90, s90, {SLOT}")
                o.e("s_addc_u32 s91, s91, 0")
            o.e(f"s_add_u32 m0, {S_M0B}, {j * SLOT}")
            o.e("s_nop 0")
            two_loads(o, LDK, "s[90:91]")
            o.e(f"s_sub_u32 {S_KLEFT}, {S_KLEFT}, 1")
            o.label(f"L_noK_pro{j}{suffix}")
        else:
            request_block(o, f, "K", j, f"pro{j}{suffix}", 0)
    for j in range(f.ns - 2):
        if paged:
            src = ("s[98:99]", S_OFFV)[j // 2] if paged == 64 else FIRST32[j]
            lo = int(src[2:4])
            o.e(f"s_cmp_eq_u32 {S_VLEFT}, 0")
            o.e(f"s_cbranch_scc1 L_noV_pro{j}{suffix}%=")
            o.e(f"s_add_u32 s90, s66, s{lo}")
            o.e(f"s_addc_u32 s91, s67, s{lo + 1}")
            if j % 2 and paged == 64:
                o.e(f"s_add_u32 s90, s90, {SLOT}")
                o.e("s_addc_u32 s91, s91, 0")
            o.e(f"s_add_u32 m0, {S_M0B}, {f.vring + j * SLOT}")
            o.e("s_nop 0")
            two_loads(o, LDV, "s[90:91]")
            o.e(f"s_sub_u32 {S_VLEFT}, {S_VLEFT}, 1")
            o.label(f"L_noV_pro{j}{suffix}")
        else:
            request_block(o, f, "V", j, f"pro{j}{suffix}", 0)
    return o.lines


def generate(f):
    o = Out()
    assert (f.ns, f.unroll) in ((5, 10), (4, 4))
    o.e(f"v_mov_b32 v{VZERO}, 0")
    item_setup(o, "first")
    o.label("L_item_top")
    o.e("s_waitcnt vmcnt(0)")
    o.e("s_barrier")
    # ---- S(0) from K block 0; behind it the fragments of iteration 0 (K block 1) ------------------
    pairs = score_pairs(0, 0, f)
    it0 = iteration_pairs(0, f, has_pv=False)
    phase = stream(o, pairs, [[] for _ in pairs], 0, False, [frag for _, frag in it0[:NSLOT]])
    # ---- iteration 0: S(1), sm(0) ---------------------------------------------------------------
    o.e("s_nop 7")
    iteration_head(o, f, 0, "i0")
    phase = stream(o, it0, spread(softmax_ops(0), len(it0)), phase, True, first_frags(1, f))
    iteration_tail(o, "i0", "L_exit0")
    phases = {0: phase}  # ring slot of the next iteration's first fragment, behind iteration p
    # ---- iterations 1 .. : `unroll` in a row, then round again -----------------------------------------
    for k in range(f.unroll):
        p = (k + 1) % f.unroll
        o.label(f"L_it{p}")
        iteration_head(o, f, p, f"p{p}")
        pairs = iteration_pairs(p, f)
        phase = stream(o, pairs, spread(softmax_ops(p % 2), len(pairs)), phase, True, first_frags(p + 1, f))
        assert phases.setdefault(p, phase) == phase  # (iteration 0 and iteration `unroll` share an exit)
        iteration_tail(o, f"p{p}", f"L_exit{p}")
    o.e("s_branch L_it1%=")

    # ---- exits: PV of the last block i = p (mod unroll) -----------------------------------------------
    # The ring holds the first fragments of the iteration that is not coming, some of V block i among
    # them; the others take the slots of the K fragments nobody needs.
    for p in range(f.unroll):
        o.label(f"L_exit{p}")
        o.e("s_waitcnt lgkmcnt(0)")
        held = {frag: (phases[p] + j) % NSLOT for j, frag in enumerate(first_frags(p + 1, f)) if frag[0] == "V"}
        wanted = [("V", p % f.ns, x // 4, x % 4) for x in range(8)]
        free = [x for x in range(NSLOT) if x not in held.values()]
        missing = [frag for frag in wanted if frag not in held]
        slots = dict(held)
        for frag in missing:
            slots[frag] = free.pop(0)
            for x in frag_reads(frag, slots[frag]):
                o.e(x)
        for frag in sorted(held, key=wanted.index):
            o.e(mfma(("PV", frag[3], p % 2, frag[2]), slots[frag]))
        o.e("s_waitcnt lgkmcnt(0)")
        for frag in missing:
            o.e(mfma(("PV", frag[3], p % 2, frag[2]), slots[frag]))
        o.e("s_branch L_end%=")

    slow_path(o, f, 0, "L_slow_i0", "L_join_i0", first=True)
    for p in range(f.unroll):
        slow_path(o, f, p % 2, f"L_slow_p{p}", f"L_join_p{p}")
    o.label("L_end")
    o.e("s_nop 15")
    o.e("s_nop 15")
    if f.items:
        next_item(o, f)
    else:
        last_epilogue(o, f)
    return o.lines


def main():
    out = sys.argv[1] if len(sys.argv) > 1 else "/dev/stdout"
    with open(out, "w") as f:
        f.write("// Generated by gen_prefill_stream.py; do not edit.\n#pragma once\n")
        for form in FORMS:
            for macro, lines in ((f"TTPA_STREAM_FIRST_TEXT_{form.name}", generate_first(form)),
                                 (f"TTPA_STREAM_LOOP_TEXT_{form.name}", generate(form))):
                f.write(f"#define {macro} \\\n")
                for ln in lines:
                    f.write(f'  "{ln}\\n\\t" \\\n')
                f.write('  ""\n')
        regs = ", ".join([f'"v{r}"' for r in CLOBBERED] + [f'"{r}"' for r in SCALAR_CLOBBERS])
        f.write(f"#define TTPA_STREAM_LOOP_CLOBBERS {regs}\n")
        lds = {form.pring + (form.ns * PSLOT if form.wide else 0) for form in FORMS}
        assert len(lds) == 1  # every form takes half of a CU's LDS
        wide = next(form for form in FORMS if form.wide)
        f.write(f"#define TTPA_STREAM_LDS_BYTES {lds.pop()}\n#define TTPA_STREAM_V_RING {FORMS[0].vring}\n"
                f"#define TTPA_STREAM_WIDE_V_RING {wide.vring}\n#define TTPA_STREAM_WIDE_P_RING {wide.pring}\n")


if __name__ == "__main__":
    main()
