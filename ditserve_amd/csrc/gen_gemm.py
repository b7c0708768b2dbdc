"""Generate the main loop of the one-wave-per-SIMD GEMM (gemm.hip:
gemm_kernel_l4) as gfx950 assembly, for each of its tile configurations.

The workgroup computes a tile of C^T = W A^T with four waves, one per SIMD, each
owning a wave tile of 16 FI features x 16 FJ tokens: FI x FJ accumulator tiles of
v_mfma_f32_16x16x32_bf16 (256 accumulators, all of the AGPRs, at 128 x 128).  The
compiler cannot hold that working set without copies, so the registers are placed
here:

  AGPR a0..a255    acc[i][j] (4 each): features w_row0 + 16 i + 4 (lane / 16) + e,
                   token a_row0 + 16 j + lane % 16
  VGPR v0..v63     operand set 0: W fragments i (v[4i..4i+3]), then token
                   fragments j (v[32+4j..])
  VGPR v64..v127   operand set 1
  VGPR v128..v137  epilogue temporaries, the weight prefetch's offsets
  SGPR s40..s53    loop state

K advances in 64-k stages through NBUF LDS buffers (A rows then W rows, 128 bytes
per row -- one L2 line of each operand row per stage -- with 16-byte units
XOR-swizzled by row) filled by direct global->LDS DMA.  A stage is two 32-k chunks
of FI x FJ MFMAs; each chunk runs on the operand set read during the chunk before
and reads the next chunk's fragments into the other set.  One barrier per stage,
between its chunks, after this wave's DMA of the next stage and its reads of
chunk 1 landed: after it every wave may read the next stage, and this stage's
buffer is free, so chunk 1 issues the DMA of stage min(s + NBUF, nk - 1) into it,
spread over its MFMAs.  The smaller tiles' stages are short (512 MFMA cycles at
128 x 128), so they take more buffers: the operands of 3-4 stages in flight.  The
first chunk runs peeled, its MFMAs starting from 0.  After the last stage the
accumulators plus bias are rounded to bf16 and staged in LDS for the C++ epilogue.

A tile may also prefetch its launch's weights (%[pfn] > 0): each lane touches a
share of the weight matrix's lines a few stages ahead of their use, so that the
workgroups, which run in step, do not all wait for HBM at the first touch of
every line.

Every output element accumulates the same MFMAs over the same k order as the
C++ kernels (gemm_kernel), and the bias add and rounding are the same
instructions, so the results are bitwise theirs.

Usage: python gen_gemm.py [dir/any]  (writes gemm_l4_<tokens>x<features>_body.inc
per configuration and gemm_l4_clobbers.h into that directory, default beside this
file)
"""
import os
import sys

# the generated wave tiles: (feature fragments, token fragments, stage buffers)
VARIANTS = [(8, 8, 2), (6, 8, 2), (8, 4, 3), (6, 4, 3), (4, 4, 4), (3, 4, 5)]


def name_of(fi, fj):
    return f"gemm_l4_{32 * fj}x{32 * fi}"


def configure(fi, fj, nbuf):
    """fi feature and fj token fragments of 16 per wave tile (workgroup tile
    32 fj tokens x 32 fi features), nbuf stage buffers."""
    global FI, FJ, NBUF, BUF, WOFF, STG_ROW, ND, DMA_SLOTS, READ_STEP
    FI, FJ, NBUF = fi, fj, nbuf
    WOFF = 32 * fj * 128               # stage buffer: A rows, then W rows
    BUF = WOFF + 32 * fi * 128
    STG_ROW = 32 * fi + 16             # staging row: 16 fi bf16 features + 16 bytes
    ND = fj + fi                       # DMA instructions per wave and stage (A groups, then W)
    n = fi * fj                        # MFMAs per chunk
    step = n // ND                     # chunk-1 MFMA slots of the stage's DMAs, evenly spread
    DMA_SLOTS = [step * k + min(2, step - 1) for k in range(ND)]
    # fragment reads: one every other MFMA slot while that leaves the last of them
    # 8 MFMAs (128 cycles) to land, else one every slot
    READ_STEP = 2 if 2 * (ND - 1) + 8 <= n else 1
    assert DMA_SLOTS[-1] < n and READ_STEP * ND <= n and nbuf * BUF + 1024 <= 160 * 1024


configure(*VARIANTS[0])
ROW = 128               # bytes per LDS row (64 k of bf16)

S_A, S_W = 40, 42       # s[40:41], s[42:43] DMA bases of the stage being fetched
S_S, S_NK1, S_SW = 44, 45, 46   # stage index, nk - 1, LDS + 1 KiB wave slice
S_T0, S_T1 = 47, 48
S_PFN, S_PFS = 49, 50    # weight prefetch: batches left, the stage the next one is due at
S_PF = 52                # s[52:53] the weight matrix
SGPRS = list(range(40, 54))
LAST_VGPR, LAST_AGPR = 139, 255
TMP = 128
PF_OFF = 136             # weight prefetch: this lane's next byte offset, and a temporary


def acc(i, j):
    return (i * FJ + j) * 4


def wreg(p, i):
    return p * 64 + i * 4


def xreg(p, j):
    return p * 64 + 32 + j * 4


class Gen:
    def __init__(self):
        self.lines = []
        self.label_n = 0
        self.tails = []

    def __call__(self, s):
        self.lines.append(s)

    def label(self, name):
        self.lines.append(f"{name}:")

    def new_label(self, stem):
        self.label_n += 1
        return f"L_{stem}_{self.label_n}_%="


def set_dma_bases(g, stage_expr):
    """S_A / S_W = tile bases + min(stage, nk - 1) * 128 bytes."""
    g(f"s_min_u32 s{S_T0}, {stage_expr}, s{S_NK1}")
    g(f"s_lshl_b32 s{S_T0}, s{S_T0}, 7")
    g(f"s_add_u32 s{S_A}, %[a_lo], s{S_T0}")
    g(f"s_addc_u32 s{S_A + 1}, %[a_hi], 0")
    g(f"s_add_u32 s{S_W}, %[w_lo], s{S_T0}")
    g(f"s_addc_u32 s{S_W + 1}, %[w_hi], 0")


def dma_m0(g, k, buf):
    """DMA instruction k (0..FJ-1: A groups, then W groups) of this wave into buffer buf."""
    base = buf * BUF + (WOFF + (k - FJ) * 4096 if k >= FJ else k * 4096)
    g(f"s_add_u32 m0, s{S_SW}, {base}")


def dma_go(g, k):
    if k < FJ:
        g(f"global_load_lds_dwordx4 %[aoff{k}], s[{S_A}:{S_A + 1}]")
    else:
        g(f"global_load_lds_dwordx4 %[woff{k - FJ}], s[{S_W}:{S_W + 1}]")


def dma_block(g, buf):
    for k in range(ND):
        dma_m0(g, k, buf)
        g("s_nop 0")
        dma_go(g, k)


def read_frag(g, kind, idx, p, buf, c):
    reg = wreg(p, idx) if kind == "w" else xreg(p, idx)
    base = f"%[rd{kind}{buf}{c}]"
    g(f"ds_read_b128 v[{reg}:{reg + 3}], {base} offset:{idx * 16 * ROW}")


def read_order():
    return [("w", 0), ("x", 0)] + [("w", i) for i in range(1, FI)] + [("x", j) for j in range(1, FJ)]


def chunk(g, p, first, reads, dmas):
    """FI x FJ MFMAs on operand set p; reads: (buffer, chunk) of the fragments to
    read into set 1 - p (one every READ_STEP slots); dmas: (buffer) the stage's
    DMA goes to, spread over the chunk, or None."""
    order = read_order()
    for m in range(FI * FJ):
        j, i = m // FI, m % FI
        k = DMA_SLOTS.index(m) if dmas is not None and m in DMA_SLOTS else None
        if k is not None:
            dma_m0(g, k, dmas)
        src_c = "0" if first else f"a[{acc(i, j)}:{acc(i, j) + 3}]"
        g(f"v_mfma_f32_16x16x32_bf16 a[{acc(i, j)}:{acc(i, j) + 3}], v[{wreg(p, i)}:{wreg(p, i) + 3}], "
          f"v[{xreg(p, j)}:{xreg(p, j) + 3}], {src_c}")
        if m % READ_STEP == 0 and m // READ_STEP < len(order):
            kind, idx = order[m // READ_STEP]
            read_frag(g, kind, idx, 1 - p, *reads)
        if k is not None:
            dma_go(g, k)


def stage(g, buf, first=False, last_check=None):
    """One 64-k stage s (s % NBUF == buf): chunk 0 on operand set 0 (read during
    the previous stage) while reading chunk 1 into set 1; the barrier that
    publishes stage s + 1 (this wave's DMA of it landed; the NBUF - 2 later
    stages may still fly) and frees buffer buf (every wave's reads of it done);
    chunk 1 on set 1 while reading stage s + 1's chunk 0 into set 0 and DMAing
    stage min(s + NBUF, nk - 1) into buffer buf."""
    chunk(g, 0, first, (buf, 1), None)
    g(f"s_waitcnt vmcnt({(NBUF - 2) * ND}) lgkmcnt(0)")
    g("s_barrier")
    g(f"s_add_u32 s{S_T1}, s{S_S}, {NBUF}")
    set_dma_bases(g, f"s{S_T1}")
    prefetch_due(g)
    chunk(g, 1, False, ((buf + 1) % NBUF, 0), buf)
    g(f"s_add_u32 s{S_S}, s{S_S}, 1")
    g("s_waitcnt lgkmcnt(0)")
    if last_check is not None:
        g(f"s_cmp_gt_u32 s{S_S}, s{S_NK1}")
        g(f"s_cbranch_scc1 {last_check}")


def prefetch_batch(g):
    """One batch of the weight prefetch: a 4-byte load per lane from its next
    line (the byte offset in PF_OFF, none past %[pfmax]) into a spare LDS line
    that nothing reads."""
    g(f"s_add_u32 m0, %[lds], {NBUF * BUF}")
    g(f"v_min_u32 v{PF_OFF + 1}, %[pfmax], v{PF_OFF}")
    g(f"v_add_u32 v{PF_OFF}, %[pfstep], v{PF_OFF}")
    g(f"global_load_lds_dword v{PF_OFF + 1}, s[{S_PF}:{S_PF + 1}]")


def prefetch_start(g):
    """The first %[pfn0] of the tile's %[pfn] prefetch batches; the others follow
    one every %[pflpr] stages (prefetch_due)."""
    skip, loop = g.new_label("nopf"), g.new_label("pf")
    g(f"s_mov_b32 s{S_PFS}, -1")
    g("s_cmp_eq_u32 %[pfn], 0")
    g(f"s_cbranch_scc1 {skip}")
    g(f"s_mov_b32 s{S_PF}, %[pf_lo]")
    g(f"s_mov_b32 s{S_PF + 1}, %[pf_hi]")
    g(f"s_mov_b32 s{S_T0}, %[pfn0]")
    g(f"v_mov_b32 v{PF_OFF}, %[pfoff]")
    g.label(loop)
    prefetch_batch(g)
    g(f"s_sub_u32 s{S_T0}, s{S_T0}, 1")
    g(f"s_cmp_lg_u32 s{S_T0}, 0")
    g(f"s_cbranch_scc1 {loop}")
    g(f"s_sub_u32 s{S_PFN}, %[pfn], %[pfn0]")
    g(f"s_cmp_eq_u32 s{S_PFN}, 0")
    g(f"s_cselect_b32 s{S_PFS}, -1, %[pflpr]")
    g.label(skip)


def prefetch_due(g):
    """The next prefetch batch, out of line, when stage S_S is the one it is due at."""
    go, back = g.new_label("pfgo"), g.new_label("pfback")
    g(f"s_cmp_eq_u32 s{S_S}, s{S_PFS}")
    g(f"s_cbranch_scc1 {go}")
    g.label(back)
    g.tails.append((go, back))


def prefetch_tails(g):
    for go, back in g.tails:
        g.label(go)
        prefetch_batch(g)
        g(f"s_sub_u32 s{S_PFN}, s{S_PFN}, 1")
        g(f"s_add_u32 s{S_PFS}, s{S_PFS}, %[pflpr]")
        g(f"s_cmp_eq_u32 s{S_PFN}, 0")
        g(f"s_cselect_b32 s{S_PFS}, -1, s{S_PFS}")
        g(f"s_branch {back}")


def prologue(g):
    # a persistent workgroup's previous tile: every wave's reads of its staged
    # rows are done before the stage DMAs overwrite them
    g("s_waitcnt lgkmcnt(0)")
    g("s_barrier")
    g(f"s_add_u32 s{S_SW}, %[lds], %[wave1k]")
    g(f"s_sub_u32 s{S_NK1}, %[nk], 1")
    g(f"s_mov_b32 s{S_S}, 0")
    # the first NBUF stages into their buffers (clamped to the last stage)
    for st in range(NBUF):
        g(f"s_mov_b32 s{S_T1}, {st}")
        set_dma_bases(g, f"s{S_T1}")
        dma_block(g, st)
    g(f"s_waitcnt vmcnt({(NBUF - 1) * ND})")
    g("s_barrier")
    prefetch_start(g)
    for kind, idx in read_order():
        read_frag(g, kind, idx, 0, 0, 0)
    g("s_waitcnt lgkmcnt(0)")


def epilogue(g):
    """acc + bias -> bf16 pairs -> this wave's staging rows: token row j*16 + lane%16,
    8-byte unit i*4 + lane/16 (features 4 apart)."""
    g("s_waitcnt vmcnt(0) lgkmcnt(0)")
    g("s_barrier")
    g("s_nop 7")
    g("s_nop 7")
    g("s_nop 7")
    for i in range(FI):
        for j in range(FJ):
            a = acc(i, j)
            for e in range(4):
                g(f"v_accvgpr_read_b32 v{TMP + e}, a{a + e}")
            for e in range(4):
                g(f"v_add_f32 v{TMP + e}, v{TMP + e}, %[b{i * 4 + e}]")
            g(f"v_cvt_pk_bf16_f32 v{TMP + 4}, v{TMP}, v{TMP + 1}")
            g(f"v_cvt_pk_bf16_f32 v{TMP + 5}, v{TMP + 2}, v{TMP + 3}")
            g(f"ds_write_b64 %[stg], v[{TMP + 4}:{TMP + 5}] offset:{j * 16 * STG_ROW + i * 32}")
    g("s_waitcnt lgkmcnt(0)")


def generate():
    g = Gen()
    prologue(g)
    done = g.new_label("done")
    loop = g.new_label("loop")
    # stage 0 peeled (its MFMAs start from 0), then the buffers in turn
    stage(g, 0, first=True, last_check=done)
    g.label(loop)
    for b in range(1, NBUF + 1):
        stage(g, b % NBUF, last_check=done)
    g(f"s_branch {loop}")
    prefetch_tails(g)
    g.label(done)
    epilogue(g)
    return g.lines


def clobbers():
    regs = ([f"v{i}" for i in range(LAST_VGPR + 1)] + [f"a{i}" for i in range(LAST_AGPR + 1)] +
            [f"s{i}" for i in SGPRS])
    rows = [", ".join(f'"{r}"' for r in regs[i:i + 16]) for i in range(0, len(regs), 16)]
    return ("// Registers the generated gemm_kernel_l4 body owns (gen_gemm.py register map).\n"
            "#define DITK_GEMM_L4_CLOBBERS \\\n" + "".join(f"  {r}, \\\n" for r in rows) + "\n")


def write_body(path):
    lines = generate()
    with open(path, "w") as f:
        f.write(f"// Generated by gen_gemm.py -- the instruction body of gemm_kernel_l4<FI = {FI}, FJ = {FJ}>.\n")
        for line in lines:
            esc = line.replace("\\", "\\\\").replace('"', '\\"')
            f.write(f'"{esc}\\n"\n')


def main(argv):
    here = os.path.dirname(os.path.abspath(__file__))
    out = os.path.dirname(os.path.abspath(argv[1])) if len(argv) > 1 else here
    for v in VARIANTS:
        configure(*v)
        write_body(os.path.join(out, name_of(v[0], v[1]) + "_body.inc"))
    configure(*VARIANTS[0])
    with open(os.path.join(out, "gemm_l4_clobbers.h"), "w") as f:
        f.write(clobbers())
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv))
