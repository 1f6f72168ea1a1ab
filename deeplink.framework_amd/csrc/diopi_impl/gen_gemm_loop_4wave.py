#!/usr/bin/env python3
"""Writes gemm_loop_4wave.inc: the K loop of the 4-wave 256 x 256 x 64 GEMM kernel (gemm.hip,
gemmMfma4WaveKernel) as inline-assembly text for gfx950.

Why a generator: with one wave per SIMD nothing hides a stall, so every instruction of the loop is placed by hand:
which MFMA an LDS fragment read or a tile load follows, and the exact s_waitcnt before the first MFMA that needs a
fragment. The compiler cannot be told to keep 256 accumulators in fixed accumulation registers across iterations
and to leave the order alone, so the loop is emitted as text with physical register names.

Registers (per lane):   a[0:255]    accumulators, tile (i, j) of the wave's 8 x 8 grid of 16 x 16 at a[4 (8 i + j) ..]
                        v[120:183]  A fragments, two buffers of 8 (one per 32-wide k-step)
                        v[184:247]  B fragments, two buffers of 8
Operands of each block: %[voA0..7] %[voB0..7]  lane byte offsets of the 8 + 8 tile loads of this wave
                        %[adA0] %[adA1] %[adB0] %[adB1]  LDS byte addresses of this lane's fragment chunk for k-step 0 / 1
                        %[rsA] %[rsB]  buffer descriptors, %[lds] LDS address of this wave's 1 KiB slot in stage 0 of A
                        %[kcur]  K byte offset of the tile whose loads are issued next, %[m0s]  the caller's M0

One tile of the loop (stage s = tile & 1), 128 MFMAs, two barriers:
  k-step 0, MFMAs 0-22    out of fragment buffer 0 | the 16 fragment reads of k-step 1 (stage s) into buffer 1, one per MFMA
  s_waitcnt lgkmcnt(0); s_barrier (B1)    every wave is done reading stage s: it may be refilled
  k-step 0, MFMAs 23-63   | the loads of tile t + 2 into stage s start here, one per five MFMAs, and run on into k-step 1
  s_waitcnt vmcnt(loads of tile t + 2 issued so far); s_barrier (B2)    tile t + 1 has landed in stage s ^ 1
  k-step 1, 64 MFMAs out of buffer 1 | the 16 fragment reads of tile t + 1, k-step 0 into buffer 0 | the rest of the loads
A load is needed at B2 of the next tile, so the youngest has more than a whole tile (128 MFMAs, about 1.3 us) to
arrive, at half the issue rate of a schedule that packs the loads between one barrier per tile and the next k-step
boundary: 16.9 cycles per MFMA against 18.2 on 8192 x 4096 x 11008 (16.3 with no tile loads at all). The kernel runs at
the power limit, where the cycles saved come back as a lower clock (1.59 against 1.65 GHz, the same time per launch); they
count when the clock is not what limits it.
Fragment reads are issued in the order the MFMAs need them (B0, A0..A7, B1..B7; the MFMAs run B-major) and LDS
returns them in order, so the wait before an MFMA is a count of younger reads that may still be outstanding.
Within a k-step the A fragments are walked forth for even B fragments and back for odd ones, so consecutive MFMAs
always share one operand (with A0..A7 restarted for every B, both operands change at each turn). At the power limit
that is measurable: 8192 x 4096 x 12288 550.4 -> 545.9 us, x 22016 985.9 -> 978.2 us, same box, same results bit for bit.
Measured and not used: K tiles of 32 in a four-stage ring (loads three tiles ahead) is 10 % slower, because a tile
load then fetches 64-byte row pieces, twice the cache lines per byte; issuing the loads twice as densely (to gain
slack) stalls the wave at issue. The same tile out of v_mfma_f32_32x32x16 (4 x 4 blocks per wave, four 16-wide k-steps,
the same number of fragment reads) takes 1.5 % fewer cycles and 9 % more time (592 -> 646 us on 8192 x 4096 x 12288): that
instruction reads and writes twice the accumulator registers per multiply-add, and at the power limit this is paid in
clock. Register-only loops of either instruction over the whole chip (no memory traffic at all) sustain 2160 TFLOP/s at
2.12 GHz (16x16x32, 16.4 cycles per instruction) against 1940 TFLOP/s at 1.87 GHz (32x32x16, 32.4 cycles): the first
figure is the ceiling that the power limit leaves to any bf16 GEMM here, 0.86 of the nominal peak.

The forms with 7 instead of 8 A fragments (T7, tiles of 224 x 256; `rows` below) leave out a[4 (56 + j) ..] and their MFMAs, reads and loads: 112
MFMAs a tile, 15 loads a wave, the same slots otherwise.

The form for int8 weights (the macros with W8): the second operand lies in LDS as it does in memory, rows of 128 bytes that are
the K of a PAIR of tiles, so its loads (8 per pair instead of 16) and its two stages go by pairs, and a load still fetches
whole 128-byte lines. A lane reads the 8 bytes of a fragment (ds_read_b64, K order and swizzle as in the 16-bit form: half
the LDS bytes) into v[104:119] and converts them between the MFMAs of the k-step before the one that needs them, exactly:
bf16 by a conversion to fp32 per byte and a permutation that joins two high halves (12 instructions a fragment), fp16 by one
conversion per byte into the half it belongs to (8). The matrix pipe leaves room for three vector instructions an MFMA and
this takes one and a half of it. Of each k-step's reads the raw ones come first:
  k-step 0, MFMAs 0-15    raw B0..B7, then A0..A7 of k-step 1 | 23-62  the conversions (all reads are done at B1)
  k-step 1, MFMAs 65-95   raw B0..B7, then A0..A7 of the next tile's k-step 0, one per two MFMAs | 79-126 the conversions
Operands besides those above: %[adB01] %[adB10] %[adB11] LDS addresses in this pair's stage of (tile of the pair, k-step),
%[adN00] of the first in the next pair's stage; %[kcurB] K byte offset of the pair whose B loads come next, %[ldsB] LDS address of
this wave's 1 KiB slot in this pair's stage, %[sel] the permutation's selector."""
import os
import sys

def read_order(rows):
    return [("B", 0)] + [("A", i) for i in range(rows)] + [("B", j) for j in range(1, 8)]


VA0, VB0 = 120, 184


def va(b, i):
    r = VA0 + b * 32 + i * 4
    return f"v[{r}:{r + 3}]"


def vb(b, j):
    r = VB0 + b * 32 + j * 4
    return f"v[{r}:{r + 3}]"


def acc(i, j):
    r = 4 * (8 * i + j)
    return f"a[{r}:{r + 3}]"


def tile_loads(rows, stage):
    """The loads of a K tile into a stage, as (operand, pass of 32 rows, stage)."""
    return [("A", d, stage) for d in range(rows)] + [("B", d, stage) for d in range(8)]


def load_m0(out, load):
    kind, d, stage = load
    out.append(f"s_add_u32 m0, %[lds], {stage * 32768 + (65536 if kind == 'B' else 0) + d * 4096}")


def load_issue(out, load):
    kind, d, _ = load
    out.append(f"buffer_load_dwordx4 %[vo{kind}{d}], %[rs{kind}], %[kcur] offen lds")
    if kind == "B" and d == 7:
        out.append("s_add_u32 %[kcur], %[kcur], 128")


def read_fragment(out, kind, idx, buf, stage, ks):
    reg = va(buf, idx) if kind == "A" else vb(buf, idx)
    out.append(f"ds_read_b128 {reg}, %[ad{kind}{ks}] offset:{idx * 2048 + stage * 32768}")


B1_SLOT = 22       # B1 follows this MFMA of k-step 0
LOAD_STEP = 5      # MFMAs between two tile loads


def tile(out, rows, s, loads, next_tile, next_output=False):
    """16 `rows` MFMAs of one K tile in stage s; loads: issue the loads of tile t + 2; next_tile: read tile t + 1's first
    fragments during k-step 1; next_output (last K tile of an output tile only): once B1 has freed both stages, issue
    the loads of the first two K tiles of the workgroup's next output tile (the caller passes that tile's lane
    offsets), so that they land while the epilogue runs."""
    step, order = 8 * rows, read_order(rows)               # MFMAs of a k-step
    after = {m: [] for m in range(2 * step)}
    for r in range(len(order)):                            # this tile's k-step 1 fragments, right away
        after[r].append(("read1", r))
    after[B1_SLOT].append(("B1", None))
    loads_before_b2 = 0
    if loads:
        for n, load in enumerate(tile_loads(rows, s)):
            slot = B1_SLOT + 1 + n * LOAD_STEP
            if slot + 1 < step:
                loads_before_b2 += 1
            after[slot].append(("m0", load))               # M0 is written one MFMA before the load that reads it
            after[slot + 1].append(("load", load))
    if next_output:
        after[B1_SLOT].append(("rewind", None))
        for n, load in enumerate(tile_loads(rows, 0) + tile_loads(rows, 1)):
            slot = B1_SLOT + 1 + n * 3
            after[slot].append(("m0", load))
            after[slot + 1].append(("load", load))
    if next_tile:
        for r in range(len(order)):
            after[step + 1 + 3 * r].append(("read0", r))
    for m in range(2 * step):
        ks, mm = divmod(m, step)
        j, pos = divmod(mm, rows)
        i = pos if j % 2 == 0 else rows - 1 - pos          # A fragments back and forth: one operand changes per MFMA
        if m == 0:
            out.append("s_waitcnt lgkmcnt(7)")             # B0 and A of buffer 0 (read during the previous k-step 1)
        elif ks == 0 and pos == 0 and j >= 1 and m <= B1_SLOT:
            # B_j of buffer 0: 7 - j reads of its set are younger, and so are this tile's reads issued so far
            out.append(f"s_waitcnt lgkmcnt({min(7 - j + min(m, len(order)), 15)})")
        if m == step and next_tile:                        # B2; the last K tile has no successor to wait for
            out.append(f"s_waitcnt vmcnt({loads_before_b2}) lgkmcnt(0)")
            out.append("s_barrier")
        out.append(f"MFMA {acc(i, j)}, {vb(ks, j)}, {va(ks, i)}, {acc(i, j)}")
        for what, arg in after[m]:
            if what == "read1":
                read_fragment(out, order[arg][0], order[arg][1], 1, s, 1)
            elif what == "read0":
                read_fragment(out, order[arg][0], order[arg][1], 0, s ^ 1, 0)
            elif what == "B1":
                out.append("s_waitcnt lgkmcnt(0)")
                out.append("s_barrier")
            elif what == "m0":
                load_m0(out, arg)
            elif what == "rewind":
                out.append("s_mov_b32 %[kcur], 0")
            else:
                load_issue(out, arg)


def prologue(out, rows, issue_loads):
    """issue_loads: issue the loads of K tiles 0 and 1 (otherwise the workgroup's previous output tile did, before its
    epilogue). The wait that follows allows one K tile's loads to be outstanding. Loads return in order, so whatever else
    is still counted (K tile 1's loads, the previous epilogue's stores), K tile 0 has landed: if one of its
    loads were pending, all younger loads of K tile 1 would be too."""
    out.append("s_mov_b32 %[m0s], m0")
    if issue_loads:
        for load in tile_loads(rows, 0) + tile_loads(rows, 1):
            load_m0(out, load)
            out.append("s_nop 0")
            load_issue(out, load)
    for r in range(256):                            # while the loads are in flight
        out.append(f"v_accvgpr_write_b32 a{r}, 0")
    out.append(f"s_waitcnt vmcnt({rows + 8})")
    out.append("s_barrier")
    for kind, idx in read_order(rows):
        read_fragment(out, kind, idx, 0, 0, 0)


RAW0, TMP0 = 104, 100   # raw bytes of a k-step's 8 fragments (2 registers each); 4 temporaries


def convert(kind, buf, j):
    """The instructions that turn the raw bytes of fragment j into buffer buf."""
    d, r = VB0 + buf * 32 + j * 4, RAW0 + 2 * j
    ops = []
    if kind == "F16":
        for half in (0, 1):      # (a register's two halves well apart: the second write keeps the first)
            for q in range(4):
                b = 2 * q + half
                unused = "UNUSED_PAD" if half == 0 else "UNUSED_PRESERVE"
                ops.append(f"v_cvt_f16_i16_sdwa v{d + q}, sext(v{r + b // 4}) dst_sel:WORD_{half} dst_unused:{unused} src0_sel:BYTE_{b % 4}")
    else:
        for q in range(4):
            t = TMP0 + 2 * (q % 2)
            for half in (0, 1):
                b = 2 * q + half
                ops.append(f"v_cvt_f32_i32_sdwa v{t + half}, sext(v{r + b // 4}) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_{b % 4}")
            ops.append(f"v_perm_b32 v{d + q}, v{t + 1}, v{t}, %[sel]")
    return ops


def read8(out, kind, idx, buf, stage, ks, ad):
    """Fragment read of the int8 form; ad: the address operand of B."""
    if kind == "A":
        read_fragment(out, "A", idx, buf, stage, ks)
    else:
        out.append(f"ds_read_b64 v[{RAW0 + 2 * idx}:{RAW0 + 2 * idx + 1}], %[{ad}] offset:{idx * 2048}")


def order8(rows):
    return [("B", j) for j in range(8)] + [("A", i) for i in range(rows)]


def m0_8(out, load):
    kind, d, stage = load
    if stage is None:
        out.append(f"s_add_u32 m0, %[ldsB], {d * 4096}")
    else:
        load_m0(out, load)


def issue8(out, load, rows):
    kind, d, _ = load
    k = "kcur" if kind == "A" else "kcurB"
    out.append(f"buffer_load_dwordx4 %[vo{kind}{d}], %[rs{kind}], %[{k}] offen lds")
    if d == (rows if kind == "A" else 8) - 1:
        out.append(f"s_add_u32 %[{k}], %[{k}], 128")


def tile8(out, rows, kind, h, load_a, load_b, younger, next_tile, next_output=False):
    """One K tile of the int8 form, the pair's tile h (its stage of A too). load_a: issue the A loads of tile t + 2, load_b: then
    the B loads of the pair after the next (h == 1); younger: loads issued before this tile that its B2 may leave in flight."""
    step, order = 8 * rows, order8(rows)
    after = {m: [] for m in range(2 * step)}
    for r in range(len(order)):
        after[r].append(("read", (r, 1, h, 1, f"adB{h}1")))
    after[B1_SLOT].append(("B1", None))
    loads = [("A", d, h) for d in range(rows)] * load_a + [("B", d, None) for d in range(8)] * load_b
    spacing = LOAD_STEP
    if next_output:
        after[B1_SLOT].append(("rewind", None))
        loads = tile_loads(rows, 0) + tile_loads(rows, 1)
        spacing = 3
    before_b2 = younger
    for n, load in enumerate(loads):
        slot = B1_SLOT + 1 + n * spacing
        before_b2 += slot + 1 < step
        after[slot].append(("m0", load))
        after[slot + 1].append(("load", load))
    vector = {m: [] for m in range(2 * step)}
    for j in range(8):
        ops = convert(kind, 1, j)
        for n, op in enumerate(ops):
            vector[23 + 5 * j + n * 5 // len(ops)].append(op)
    if next_tile:
        for r in range(len(order)):
            after[step + 1 + 2 * r].append(("read", (r, 0, h ^ 1, 0, "adB10" if h == 0 else "adN00")))
        begin, width = (15, 6) if rows == 8 else (13, 5)
        for j in range(8):
            first, ops = step + begin + width * j, convert(kind, 0, j)
            issued = min(len(order), (first - step) // 2)     # reads issued behind MFMAs before `first`
            vector[first].append(f"s_waitcnt lgkmcnt({issued - j - 1})")
            for n, op in enumerate(ops):
                vector[first + n * width // len(ops)].append(op)
    for m in range(2 * step):
        ks, mm = divmod(m, step)
        j, pos = divmod(mm, rows)
        i = pos if j % 2 == 0 else rows - 1 - pos
        if m == 0:
            out.append("s_waitcnt lgkmcnt(0)")           # A of buffer 0, read a good while ago
        if m == step and next_tile:
            out.append(f"s_waitcnt vmcnt({before_b2}) lgkmcnt(0)")
            out.append("s_barrier")
        out.append(f"MFMA {acc(i, j)}, {vb(ks, j)}, {va(ks, i)}, {acc(i, j)}")
        out += vector[m]
        for what, arg in after[m]:
            if what == "read":
                r, buf, stage, rks, ad = arg
                read8(out, order[r][0], order[r][1], buf, stage, rks, ad)
            elif what == "B1":
                out.append("s_waitcnt lgkmcnt(0)")
                out.append("s_barrier")
            elif what == "m0":
                m0_8(out, arg)
            elif what == "rewind":
                out.append("s_mov_b32 %[kcur], 0")
                out.append("s_mov_b32 %[kcurB], 0")
            else:
                issue8(out, arg, rows)


def prologue8(out, rows, kind, issue_loads):
    """As prologue(); K tile 0 is A's first loads and B's first pair, and K tile 1 and the second pair are those after them."""
    out.append("s_mov_b32 %[m0s], m0")
    if issue_loads:
        for stage in (0, 1):
            for load in tile_loads(rows, stage):
                m0_8(out, load)
                out.append("s_nop 0")
                issue8(out, load, rows)
    for r in range(256):
        out.append(f"v_accvgpr_write_b32 a{r}, 0")
    out.append(f"s_waitcnt vmcnt({rows + 8})")
    out.append("s_barrier")
    for k, idx in order8(rows):
        read8(out, k, idx, 0, 0, 0, "adB00")
    out.append(f"s_waitcnt lgkmcnt({rows})")
    for j in range(8):
        out += convert(kind, 0, j)


def macros(text, prefix, kind, mnemonic, blocks):
    for name, lines in blocks:
        text.append(f"#define GEMM4W_{prefix}{name}_{kind} \\\n")
        text.append(" \\\n".join('  "' + l.replace("MFMA", mnemonic) + '\\n\\t"' for l in lines) + "\n\n")


def finished(block):
    """The end of an output tile: the last MFMAs have written their accumulators."""
    return block + ["s_nop 15", "s_nop 15", "s_mov_b32 m0, %[m0s]"]


def main():
    text = ["// Generated by gen_gemm_loop_4wave.py (see there for the schedule); do not edit.\n"]

    def block(fn, *calls):
        out = []
        for args in calls:
            fn(out, *args)
        return out

    for rows, t7 in ((8, ""), (7, "T7_")):
        for kind, mnemonic in (("BF16", "v_mfma_f32_16x16x32_bf16"), ("F16", "v_mfma_f32_16x16x32_f16")):
            macros(text, t7, kind, mnemonic, (
                ("PROLOGUE", block(prologue, (rows, True))),
                ("PROLOGUE_LOADED", block(prologue, (rows, False))),
                ("BODY", block(tile, (rows, 0, True, True), (rows, 1, True, True))),
                ("TAIL", finished(block(tile, (rows, 0, False, True), (rows, 1, False, False)))),
                ("TAIL_NEXT", finished(block(tile, (rows, 0, False, True), (rows, 1, False, False, True))))))
            # int8: B2 of a pair's first tile waits for the A loads of the tile before it; that tile's B loads, issued behind
            # them, are waited for by B2 of the second
            macros(text, "W8_" + t7, kind, mnemonic, (
                ("PROLOGUE", block(prologue8, (rows, kind, True))),
                ("PROLOGUE_LOADED", block(prologue8, (rows, kind, False))),
                ("BODY", block(tile8, (rows, kind, 0, True, False, 8, True), (rows, kind, 1, True, True, 0, True))),
                ("BODY_LAST", block(tile8, (rows, kind, 0, True, False, 8, True), (rows, kind, 1, True, False, 0, True))),
                ("TAIL", finished(block(tile8, (rows, kind, 0, False, False, 0, True), (rows, kind, 1, False, False, 0, False)))),
                ("TAIL_NEXT", finished(block(tile8, (rows, kind, 0, False, False, 0, True), (rows, kind, 1, False, False, 0, False, True))))))
    clobbers = ", ".join(f'"v{r}"' for r in range(VA0, VA0 + 128)) + ", " + ", ".join(f'"a{r}"' for r in range(256))
    text.append(f"#define GEMM4W_CLOBBERS {clobbers}\n")
    clobbers = ", ".join(f'"v{r}"' for r in range(TMP0, VA0))
    text.append(f"#define GEMM4W_W8_CLOBBERS {clobbers}, GEMM4W_CLOBBERS\n")
    path = sys.argv[1] if len(sys.argv) > 1 else os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_loop_4wave.inc")
    with open(path, "w") as f:
        f.write("".join(text))


if __name__ == "__main__":
    main()
