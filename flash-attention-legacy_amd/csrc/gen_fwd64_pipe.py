"""Generates fal_fwd64_pipe.inc: the key-tile loop of the head_dim-64 forward kernel for
small grids (fwd_kernel with SMALL), 32 query rows per wave at two waves per SIMD, as one
inline-asm block.

What bounds this head dim is the vector ALU: per 64-key tile a wave issues 512 cycles of
MFMAs but about 600 of softmax (32 exponentials at 8 cycles, 32 score
FMAs, 32 sums and 16 packs at 4).  The C++ loop runs the products and the softmax of a tile
one after the other, so a wave needs about 1800 cycles per tile and three waves per SIMD
still 1150 each.  Here the loop is software-pipelined inside the wave: iteration j runs
  * the PV products of tile j-1 (V^T from LDS by transposed reads), then
  * the S products of tile j+1 (K fragments from LDS), and
  * beside both, spread between the MFMAs, the softmax of tile j.
The LDS reads run ahead of their MFMAs across the products and across iterations (an
iteration ends with the first V^T reads of the next one's PV), so the MFMAs of an
iteration form one stream without a gap for LDS latency.

Semantics are those of fwd_kernel's C++ tile loop: scores s = q.k, exponent s * c - m with
c = scale * log2(e) > 0 and m the row's reference max (log2 domain); m moves only when a
tile's per-lane P sum could leave fp16 range (> 2^15) or the row has no max yet, and then O
and l are rescaled by 2^(m_old - m_new); masked scores (key > row for causal, key >= nk)
are -inf.

LDS: a ring of 4 slots (K tile, then V tile, 64 rows each, XOR-swizzled as SwizzledTile<D>);
tile jbeg + i goes to slot i % 4.  The loop is unrolled over the four slots, so slot offsets
are immediates of the LDS reads.  One barrier opens an iteration: behind it tile j+1's K and
tile j's V are readable, and the slots of K tile j-1 and V tile j-2 are free, so iteration j
copies K tile j+3 and V tile j+2 (buffer->LDS loads, two iterations before their barrier).
After the last tile the wave writes its O accumulators to LDS (blocks of 1 KB, OSTR bytes
apart, from the `olds` address) for the C++ epilogue.

Waves of a workgroup can own different tile ranges (causal: each wave stops at its diagonal
tile); every wave runs every iteration's copy and barrier.  Tiles before `jf` need no mask
and are followed by another tile of the wave: they run the loop's short path.

Registers (per lane; VGPRs only):
  O     O^T accumulators, db*16 + i
  SA    S^T of two consecutive tiles, kb*16 + i; a tile's P^T (fp16/bf16 pairs) is
        packed in place into the first 8 registers of each 16-register block
  KF, VF  K fragment ring (2*KS x 4), V^T fragment ring (8 x 4)
  LT per-lane P sums, NM -m, T0..T3 temporaries
  s[84:85] compare mask, s86 caller's m0, s87 rows left from the next V tile to copy,
  s[88:91]/s[92:95] K/V copy resources, s96 tile j, s98/s99 temporaries
  lower VGPRs and s0..s83 are left to the compiler.

The output is deterministic text, tracked under csrc/gen/; build.py checks the tracked
file against render() and rewrites it only when asked (--regen).
"""

import os
import sys

NBUF = 4            # LDS ring slots
OSTR = 1040         # bytes between a wave's O blocks in the LDS hand-off (kPipeOStr in fal_fwd.hip)
D = 64
# Knobs (set by configure(); the values here are the product kernel's)
DEFAULTS = {
    "DIST": 8,        # LDS reads issued ahead of the MFMA that needs them
    "PRE": 8,         # V^T reads of the next PV issued at an iteration's end (2 per product)
    "LEAD": 24,       # softmax issue cycles placed before an iteration's first MFMA
}
DIST, PRE, LEAD = 8, 8, 24
MEASURE = False
DEFAULT_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gen", "fal_fwd64_pipe.inc")

VRING = 8
SM, SM0, SR = 84, 86, 87
SK, SV = 88, 92
SJ, ST, ST2 = 96, 98, 99
NEG_INF = "0xff800000"


def v(n):
    return f"v{n}"


def vr(n, k):
    return f"v[{n}:{n + k - 1}]"


def operands(d=D):
    """(name, constraint, C++ expression) of the block's outputs and inputs."""
    ks, db, ipt = d // 16, d // 32, d // 32
    outs = [("m", "+v", "m_run[0]"), ("l", "+v", "l_run[0]")]
    ins = [(f"Q{t}", "v", f"qreg[0][{t}]") for t in range(ks)]
    ins += [(f"kvo{i}", "v", f"kvo[{i}]") for i in range(ipt)]
    ins += [(f"vvo{i}", "v", f"vvo[{i}]") for i in range(ipt)]
    ins += [(f"ka{t}", "v", f"p_ka[{t}]") for t in range(ks)]
    ins += [(f"va{hf}{b}", "v", f"p_va[{hf}][{b}]") for hf in range(2) for b in range(db)]
    ins += [("row", "v", "p_row[0]"), ("hh4", "v", "p_hh4"), ("olds", "v", "p_olds")]
    ins += [(f"kr{i}", "s", f"pk_rs[{i}]") for i in range(4)]
    ins += [(f"vr{i}", "s", f"pv_rs[{i}]") for i in range(4)]
    ins += [("c", "s", "c"), ("jbeg", "s", "p_jbeg"), ("jend", "s", "p_jend"), ("jl", "s", "p_jl"),
            ("jf", "s", "p_jf"), ("wrow", "s", "p_wrow"), ("nk", "s", "p_nk"), ("ktb", "s", "p_ktb"),
            ("vtb", "s", "p_vtb"), ("krb", "s", "p_krb"), ("vrb", "s", "p_vrb"), ("rows", "s", "p_rows"),
            ("lbase", "s", "p_lbase"), ("npre", "s", "p_npre")]
    return outs, ins


class Emitter:
    def __init__(self, bf16, d=D):
        self.lines = []
        self.mf = "v_mfma_f32_32x32x16_bf16" if bf16 else "v_mfma_f32_32x32x16_f16"
        self.cvt = "v_cvt_pk_bf16_f32" if bf16 else "v_cvt_pk_f16_f32"
        self.ks, self.db, self.ipt = d // 16, d // 32, d // 32
        self.rowb = d * 2                 # bytes of a tile row
        self.voff = 64 * self.rowb        # V tile inside a slot
        self.slotb = 2 * self.voff
        self.O, self.SA, self.KF, self.VF = 224, (160, 192), 128, 96
        self.LT, self.NM, self.T, self.vlow = 95, 94, (90, 91, 92, 93), 90
        outs, ins = operands(d)
        self.idx = {name: i for i, (name, _, _) in enumerate(outs + ins)}
        self.counter = 0

    def op(self, name):
        return f"%{self.idx[name]}"

    def e(self, s):
        self.lines.append(s)

    def es(self, xs):
        for x in xs:
            self.e(x)

    def label(self, name):
        self.counter += 1
        return f"{name}{self.counter}_%="

    # -- instruction streams -------------------------------------------------
    def softmax_ops(self, par, fma=True):
        """Softmax of the tile whose scores are in SA[par]: exponent FMA, exp2, per-lane P
        sum (fp32 adds of the exponentials), packing into P^T (in place).
        Streamed element by element (e = 2*i + kb over the two 16-score blocks): the FMA
        runs two elements ahead, an element is summed one step after its exponential, and a
        pair is packed one step after its second exponential."""
        op, b0, lt = self.op, self.SA[par], v(self.LT)
        ops = [f"v_mov_b32 {lt}, 0"]
        reg = lambda e: b0 + (e % 2) * 16 + e // 2
        fmas = [f"v_fma_f32 {v(reg(e))}, {v(reg(e))}, {op('c')}, {v(self.NM)}" for e in range(32)] if fma else []
        cvt_at = {}
        for kb in range(2):
            for k in range(8):
                last = 4 * k + 2 + kb           # element index of the pair's second exponential
                b = b0 + kb * 16
                cvt_at.setdefault(last + 1, []).append(f"{self.cvt} {v(b + k)}, {v(b + 2 * k)}, {v(b + 2 * k + 1)}")
        ops += fmas[:2]
        for e in range(36):
            if e + 2 < len(fmas):
                ops.append(fmas[e + 2])
            if e < 32:
                ops.append(f"v_exp_f32 {v(reg(e))}, {v(reg(e))}")
            if 0 <= e - 1 < 32:
                ops.append(f"v_add_f32 {lt}, {lt}, {v(reg(e - 1))}")
            ops += cvt_at.get(e, [])
        return ops

    def load(self, part, slot):
        """Copy of one K (part 0) or V (part 1) tile into `slot`: IPT buffer->LDS loads, each
        behind its m0 (a wait state or another instruction in between)."""
        rs, vo = ((SK, "kvo"), (SV, "vvo"))[part]
        return [(f"s_add_u32 m0, {self.op('lbase')}, {slot * self.slotb + part * self.voff + i * 4096}",
                 f"buffer_load_dwordx4 {self.op(f'{vo}{i}')}, s[{rs}:{rs + 3}], 0 offen lds")
                for i in range(self.ipt)]

    def records(self, part, ahead):
        """Record count of the copy of the tile `ahead` tiles past s87's: its rows inside the
        copy range (0..64) times the row stride, so rows past the range read as zeros."""
        r = (SK, SV)[part] + 2
        return [f"s_sub_i32 s{r}, s{SR}, {64 * ahead}", f"s_max_i32 s{r}, s{r}, 0", f"s_min_i32 s{r}, s{r}, 64",
                f"s_mul_i32 s{r}, s{r}, {self.op(('krb', 'vrb')[part])}"]

    def advance(self, part):
        r = (SK, SV)[part]
        return [f"s_add_u32 s{r}, s{r}, {self.op(('ktb', 'vtb')[part])}", f"s_addc_u32 s{r + 1}, s{r + 1}, 0"]

    def iter_records(self):
        """Record counts of iteration j's copies (K tile j+3, V tile j+2; s87 counts the
        rows left from V's).  Tiles of the short path (j < jf) keep the full count that an
        earlier iteration set."""
        self.es(self.records(0, 1) + self.records(1, 0))

    def dma_groups(self, u):
        """Iteration j (slot u): copies of K tile j+3 and V tile j+2, as (before, after)
        instructions of an MFMA."""
        g = [([a], [b]) for a, b in self.load(0, (u + 3) % NBUF) + self.load(1, (u + 2) % NBUF)]
        return g + [(self.advance(0), self.advance(1) + [f"s_sub_i32 s{SR}, s{SR}, 64"])]

    def s_prod(self, par, slot):
        """S^T = K Q^T of the tile in `slot`, into SA[par]: reads, and (MFMA, its read)."""
        reads, mf = [], []
        for t in range(self.ks):
            for kb in range(2):
                k = 2 * t + kb
                f = vr(self.KF + 4 * k, 4)
                reads.append(f"ds_read_b128 {f}, {self.op(f'ka{t}')} offset:{slot * self.slotb + kb * 32 * self.rowb}")
                d = vr(self.SA[par] + kb * 16, 16)
                mf.append((f"{self.mf} {d}, {f}, {self.op(f'Q{t}')}, {d if t else 0}", k))
        return reads, mf

    def pv_prod(self, par, slot):
        """O^T += V^T P^T of the tile in `slot` whose P^T is packed in SA[par]: reads, and
        (MFMA, its last read)."""
        reads, mf = [], []
        k = 0
        for ks in range(4):
            kb, t2 = ks // 2, ks % 2
            for db in range(self.db):
                p = self.VF + 4 * (k % VRING)
                for hf in range(2):
                    reads.append(f"ds_read_b64_tr_b16 {vr(p + 2 * hf, 2)}, {self.op(f'va{hf}{db}')} "
                                 f"offset:{slot * self.slotb + self.voff + ks * 16 * self.rowb}")
                o = vr(self.O + db * 16, 16)
                pb = vr(self.SA[par] + kb * 16 + 4 * t2, 4)
                mf.append((f"{self.mf} {o}, {vr(p, 4)}, {pb}, {o}", 2 * k + 1))
                k += 1
        assert k <= VRING                # no fragment of a tile overwrites another
        return reads, mf

    @staticmethod
    def cost(ins):
        """Issue cycles of a VALU instruction (measured: an exponential 8, the others 4)."""
        return 8 if ins.startswith("v_exp") else 4

    def stream(self, reads, mf, issued=0, valu=(), groups=(), lead=0):
        """The MFMAs `mf` with their LDS reads DIST ahead, and the VALU stream and instruction
        groups spread between them (the VALU by issue cycles, `lead` cycles of it before the
        first MFMA).  `reads` are (instruction, number of MFMAs to issue before it); the first
        `issued` of them are in flight already.  LDS reads complete in issue order, so the
        wait before an MFMA lets the reads issued after its last one stay in flight."""
        valu, groups = list(valu), list(groups)
        total = sum(self.cost(x) for x in valu)
        done, ready = 0.0, -1

        def issue(limit, k):
            nonlocal issued
            while issued < min(limit, len(reads)) and reads[issued][1] <= k:
                self.e(reads[issued][0])
                issued += 1

        def spend(goal):
            nonlocal done
            while valu and done < goal:
                x = valu.pop(0)
                done += self.cost(x)
                self.e(x)

        for k, (ins, need) in enumerate(mf):
            issue(need + 1 + DIST, k)
            if k == 0:
                spend(lead)
            before, after = groups.pop(0) if groups else ((), ())
            self.es(before)
            assert issued > need
            if need > ready:
                self.e(f"s_waitcnt lgkmcnt({min(issued - need - 1, 15)})")
                ready = need
            self.e(ins)
            self.es(after)
            spend(lead + (total - lead) * (k + 1) / len(mf))
        self.plain(groups)
        spend(total + 1)
        issue(len(reads), len(mf))
        assert not valu and issued == len(reads)

    def plain(self, groups):
        for before, after in groups:
            self.es(list(before) + ["s_nop 0"] + list(after))

    # -- blocks ----------------------------------------------------------------
    def mask_block(self, par):
        """Scores of tile j in SA[par] set to -inf where key > row (causal) or key >= nk.
        Skipped when no key of the tile can be masked for this wave."""
        e, op, (t0, t1, _, t3) = self.e, self.op, self.T
        lbl = self.label("nomask")
        e(f"s_lshl_b32 s{ST}, s{SJ}, 6")                  # n0 = j * 64
        e(f"s_add_u32 s{ST2}, s{ST}, 63")
        e(f"s_cmp_gt_i32 s{ST2}, {op('wrow')}")
        e(f"s_cselect_b32 s{SM}, 1, 0")
        e(f"s_cmp_ge_i32 s{ST2}, {op('nk')}")
        e(f"s_cselect_b32 s{SM + 1}, 1, 0")
        e(f"s_or_b32 s{SM}, s{SM}, s{SM + 1}")
        e(f"s_cmp_eq_u32 s{SM}, 0")
        e(f"s_cbranch_scc1 {lbl}")
        e("s_nop 7")
        e("s_nop 7")
        e(f"v_mov_b32 {v(t3)}, {NEG_INF}")
        e(f"s_sub_u32 s{ST2}, {op('nk')}, s{ST}")
        e(f"s_sub_u32 s{ST2}, s{ST2}, 1")                 # last valid key of the tile, local
        # thr = min(row - n0, nk - 1 - n0) - hh*4: key kb*32 + c_i (+ hh*4) is kept iff
        # c_i + kb*32 <= thr
        e(f"v_subrev_u32 {v(t0)}, s{ST}, {op('row')}")
        e(f"v_min_i32 {v(t0)}, s{ST2}, {v(t0)}")
        e(f"v_sub_u32 {v(t0)}, {v(t0)}, {op('hh4')}")
        for kb in range(2):
            e(f"v_subrev_u32 {v(t1)}, {kb * 32}, {v(t0)}")
            for i in range(16):
                ci = (i // 4) * 8 + i % 4
                r = self.SA[par] + kb * 16 + i
                e(f"v_cmp_le_i32 vcc, {ci}, {v(t1)}")
                e(f"v_cndmask_b32 {v(r)}, {v(t3)}, {v(r)}, vcc")
        e(f"{lbl}:")

    def init_max(self):
        """Rows without a max yet (m = -inf) take the max of the first tile's scaled
        scores (SA[0])."""
        e, op, (t0, t1, t2, t3) = self.e, self.op, self.T
        lbl = self.label("noinit")
        e(f"v_cmp_eq_f32 vcc, {NEG_INF}, {op('m')}")
        e(f"s_cbranch_vccz {lbl}")
        b0 = self.SA[0]
        e(f"v_mov_b32 {v(t2)}, {NEG_INF}")
        for i in range(0, 32, 2):
            e(f"v_mul_f32 {v(t0)}, {op('c')}, {v(b0 + i)}")
            e(f"v_mul_f32 {v(t1)}, {op('c')}, {v(b0 + i + 1)}")
            e(f"v_max3_f32 {v(t2)}, {v(t2)}, {v(t0)}, {v(t1)}")
        e(f"v_mov_b32 {v(t3)}, {v(t2)}")
        e("s_nop 1")                                           # VALU write -> permlane swap read
        e(f"v_permlane32_swap_b32 {v(t2)}, {v(t3)}")
        e(f"v_max_f32 {v(t2)}, {v(t2)}, {v(t3)}")
        e(f"v_mov_b32 {op('m')}, {v(t2)}")
        e(f"v_cmp_eq_f32 vcc, {NEG_INF}, {v(t2)}")
        e(f"v_cndmask_b32_e64 {v(self.NM)}, -{v(t2)}, 0, vcc")
        e(f"{lbl}:")

    def s_simple(self, par, slot):
        """S of the tile in `slot` into SA[par], not interleaved (first tile, redo)."""
        reads, mf = self.s_prod(par, slot)
        self.stream([(r, 0) for r in reads], mf)
        for _ in range(4):
            self.e("s_nop 15")

    def fix_block(self, u):
        """Tile j redone with a new row max: S recomputed from its K slot, masked, the
        max taken, O and l rescaled, P and its sums recomputed."""
        e, op, par, (t0, t1, t2, t3) = self.e, self.op, u & 1, self.T
        e(f"fix{u}_%=:")
        e("s_nop 15")
        e("s_waitcnt lgkmcnt(0)")
        self.s_simple(par, u)
        self.mask_block(par)
        e("s_nop 4")
        b0, m, nm = self.SA[par], op("m"), v(self.NM)
        for i in range(32):
            e(f"v_fma_f32 {v(b0 + i)}, {v(b0 + i)}, {op('c')}, {nm}")
        e(f"v_mov_b32 {v(t0)}, {NEG_INF}")
        for i in range(0, 32, 2):
            e(f"v_max3_f32 {v(t0)}, {v(t0)}, {v(b0 + i)}, {v(b0 + i + 1)}")
        e(f"v_mov_b32 {v(t1)}, {v(t0)}")
        e("s_nop 1")
        e(f"v_permlane32_swap_b32 {v(t0)}, {v(t1)}")
        e(f"v_max_f32 {v(t0)}, {v(t0)}, {v(t1)}")             # mx (log2 domain, relative to m)
        # first row: dlt = mx, m = mx, alpha = 1; otherwise dlt = max(mx, 0), m += dlt,
        # alpha = 2^-dlt; mx = -inf: dlt = 0
        e(f"v_max_f32 {v(t1)}, 0, {v(t0)}")
        e(f"v_cmp_class_f32_e64 s[{SM}:{SM + 1}], {m}, 4")        # first: m = -inf
        e("s_nop 1")
        e(f"v_cndmask_b32_e64 {v(t1)}, {v(t1)}, {v(t0)}, s[{SM}:{SM + 1}]")
        e(f"v_cmp_eq_f32 vcc, {NEG_INF}, {v(t0)}")
        e(f"v_cndmask_b32_e64 {v(t1)}, {v(t1)}, 0, vcc")          # dlt
        e(f"v_add_f32 {v(t2)}, {m}, {v(t1)}")
        e(f"v_cndmask_b32_e64 {m}, {v(t2)}, {v(t0)}, s[{SM}:{SM + 1}]")
        e(f"v_exp_f32_e64 {v(t2)}, -{v(t1)}")
        e("s_nop 0")
        e(f"v_cndmask_b32_e64 {v(t2)}, {v(t2)}, 1.0, s[{SM}:{SM + 1}]")   # alpha
        e(f"v_mul_f32 {op('l')}, {op('l')}, {v(t2)}")
        for k in range(16 * self.db):
            o = self.O + k
            e(f"v_mul_f32 {v(o)}, {v(o)}, {v(t2)}")
        for i in range(32):
            e(f"v_sub_f32 {v(b0 + i)}, {v(b0 + i)}, {v(t1)}")
        e(f"v_cmp_eq_f32 vcc, {NEG_INF}, {m}")
        e(f"v_cndmask_b32_e64 {nm}, -{m}, 0, vcc")
        self.es(self.softmax_ops(par, fma=False))
        e(f"s_branch cont{u}_%=")

    def fix_check(self, u):
        """Redo the tile if some lane's P sum exceeds 2^15 or a row still has no max."""
        e = self.e
        e(f"s_mov_b32 s{ST2}, 0x47000000")                # 2^15
        e(f"v_cmp_nge_f32 vcc, s{ST2}, {v(self.LT)}")
        e(f"v_cmp_class_f32_e64 s[{SM}:{SM + 1}], {self.op('m')}, 4")   # m = -inf
        e(f"s_or_b64 vcc, vcc, s[{SM}:{SM + 1}]")
        e(f"s_cbranch_vccnz fix{u}_%=")

    def open_iteration(self):
        """All copies but those of the last iteration are done, in every wave."""
        self.e(f"s_waitcnt vmcnt({2 * self.ipt})")
        self.e("s_barrier")

    def soft_iteration(self, u, pv, snext):
        """Iteration j (slot u) with the softmax of tile j, its scores in SA[u & 1]: PV of
        tile j-1 (its first reads in flight), S of tile j+1, the first V^T reads of tile j."""
        par = u & 1
        ops = self.softmax_ops(par)
        reads, mf = [], []
        if pv:
            r, m = self.pv_prod(par ^ 1, (u - 1) % NBUF)
            reads += [(x, 0) for x in r]
            mf += m
        npv, nr = len(mf), len(reads)
        if snext:
            r, m = self.s_prod(par ^ 1, (u + 1) % NBUF)
            reads += [(x, 0) for x in r]
            mf += [(x, need + nr) for x, need in m]
        # (they overwrite fragments of this iteration's PV: after its products)
        r, _ = self.pv_prod(par, u)
        reads += [(x, npv) for x in r[:PRE]]
        start = len(self.lines)
        if not (pv and snext):
            self.es(["s_nop 7", "s_nop 7"])
        if mf:
            self.stream(reads, mf, PRE if pv else 0, ops, self.dma_groups(u), LEAD)
        else:
            self.plain(self.dma_groups(u))
            self.es(ops + [x for x, _ in reads])
        self.fix_check(u)
        if snext:
            # scores of tile j+1: 12 wait states between their last MFMA and the first VALU
            # read, which comes in the next iteration, 6 instructions on at the earliest
            # (sum of l, tile index, compare, branch, copy wait, barrier)
            last = max(i for i in range(start, len(self.lines)) if "mfma" in self.lines[i])
            assert len(self.lines) - 1 - last + 6 >= 16

    def last_pv(self, u, groups=()):
        """PV of tile j-1 (slot u - 1), the wave's last one; its first reads are in flight."""
        r, mf = self.pv_prod((u & 1) ^ 1, (u - 1) % NBUF)
        self.stream([(x, 0) for x in r], mf, PRE, (), groups)

    def program(self):
        e, op = self.e, self.op
        e("s_nop 7")
        e(f"s_mov_b32 s{SM0}, m0")
        for i in range(4):
            e(f"s_mov_b32 s{SK + i}, {op(f'kr{i}')}")
            e(f"s_mov_b32 s{SV + i}, {op(f'vr{i}')}")
        e(f"s_mov_b32 s{SJ}, {op('jbeg')}")
        e(f"s_mov_b32 s{SR}, {op('rows')}")
        # the first two tiles (K then V of each), unless the caller already issued their
        # copies (npre = 2: the copy resources and the row count then start two tiles on)
        e(f"s_cmp_eq_u32 {op('npre')}, 0")
        e("s_cbranch_scc0 pre_%=")
        for slot in range(2):
            self.es(self.records(0, 0) + self.records(1, 0))
            for part in range(2):
                self.plain([([a], [b]) for a, b in self.load(part, slot)])
                self.es(self.advance(part))
            e(f"s_sub_i32 s{SR}, s{SR}, 64")
        e("pre_%=:")
        self.es(self.records(0, 0))
        self.plain([([a], [b]) for a, b in self.load(0, 2)])
        self.es(self.advance(0))
        for a in range(16 * self.db):
            e(f"v_mov_b32 {v(self.O + a)}, 0")
        e(f"v_cmp_eq_f32 vcc, {NEG_INF}, {op('m')}")
        e(f"v_cndmask_b32_e64 {v(self.NM)}, -{op('m')}, 0, vcc")
        # S of the first tile (if this wave has any tile), masked, then the first max
        e(f"s_waitcnt vmcnt({4 * self.ipt})")
        e("s_barrier")
        e(f"s_cmp_gt_i32 s{SJ}, {op('jl')}")
        e("s_cbranch_scc1 disp0_%=")
        self.s_simple(0, 0)
        self.mask_block(0)
        e("s_nop 4")
        self.init_max()
        e("s_branch disp0_%=")
        # ---- the loop's short path: tiles below jf, slot after slot ----
        for u in range(NBUF):
            e(f"main{u}_%=:")
            self.open_iteration()
            self.soft_iteration(u, True, True)
            e(f"cont{u}_%=:")
            e(f"v_add_f32 {op('l')}, {op('l')}, {v(self.LT)}")
            e(f"s_add_u32 s{SJ}, s{SJ}, 1")
            e(f"s_cmp_lt_i32 s{SJ}, {op('jf')}")
            e(f"s_cbranch_scc0 slow{u}_%=")
        e("s_branch main0_%=")
        for u in range(NBUF):
            n = (u + 1) % NBUF
            e(f"next{u}_%=:")
            e(f"s_add_u32 s{SJ}, s{SJ}, 1")
            e(f"slow{u}_%=:")
            e(f"s_cmp_lt_i32 s{SJ}, {op('jend')}")
            e(f"s_cbranch_scc0 fin{n}_%=")
            # ---- dispatch of iteration j, slot n (uniform per wave) ----
            e(f"disp{n}_%=:")
            self.iter_records()
            e(f"s_cmp_gt_i32 s{SJ}, {op('jl')}")
            e(f"s_cbranch_scc1 nosoft{n}_%=")
            if n == 0:
                e(f"s_cmp_eq_u32 s{SJ}, {op('jbeg')}")
                e("s_cbranch_scc1 first_%=")
            e(f"s_cmp_eq_u32 s{SJ}, {op('jl')}")
            e(f"s_cbranch_scc1 last{n}_%=")
            self.mask_block(n & 1)
            e(f"s_branch main{n}_%=")
        for u in range(NBUF):
            e(f"last{u}_%=:")
            self.mask_block(u & 1)
            self.open_iteration()
            self.soft_iteration(u, True, False)
            e(f"s_branch cont{u}_%=")
            # no softmax: PV of the wave's last tile (j = jl + 1), or nothing
            e(f"nosoft{u}_%=:")
            self.open_iteration()
            e(f"s_add_u32 s{ST}, {op('jl')}, 1")
            e(f"s_cmp_eq_u32 s{SJ}, s{ST}")
            e(f"s_cbranch_scc0 idle{u}_%=")
            e(f"s_cmp_gt_i32 s{SJ}, {op('jbeg')}")
            e(f"s_cbranch_scc0 idle{u}_%=")
            self.last_pv(u, self.dma_groups(u))
            e(f"s_branch next{u}_%=")
            e(f"idle{u}_%=:")
            self.plain(self.dma_groups(u))
            e(f"s_branch next{u}_%=")
            # tile j's P could leave fp16 range, or a row had no max: redo it
            self.fix_block(u)
            # ---- after the last iteration (j = jend, slot u): PV of the wave's last tile
            # if it is the workgroup's last tile ----
            e(f"fin{u}_%=:")
            e(f"s_add_u32 s{ST}, {op('jl')}, 1")
            e(f"s_cmp_eq_u32 s{SJ}, s{ST}")
            e("s_cbranch_scc0 out_%=")
            e(f"s_cmp_gt_i32 s{SJ}, {op('jbeg')}")
            e("s_cbranch_scc0 out_%=")
            self.last_pv(u)
            e("s_branch out_%=")
        e("first_%=:")
        self.open_iteration()
        e(f"s_cmp_eq_u32 s{SJ}, {op('jl')}")
        e("s_cbranch_scc1 firstlast_%=")
        self.soft_iteration(0, False, True)
        e("s_branch cont0_%=")
        e("firstlast_%=:")
        self.soft_iteration(0, False, False)
        e("s_branch cont0_%=")
        e("out_%=:")
        # every wave is done with the ring: O goes to this wave's blocks of LDS
        for _ in range(2):
            e("s_nop 15")
        e("s_waitcnt vmcnt(0) lgkmcnt(0)")
        e("s_barrier")
        for g in range(4 * self.db):
            e(f"ds_write_b128 {op('olds')}, {vr(self.O + 4 * g, 4)} offset:{g * OSTR}")
        e("s_waitcnt lgkmcnt(0)")
        e(f"s_mov_b32 m0, s{SM0}")
        return self.lines


def configure(knobs=None, measure=False):
    """Set the generator's knobs.  `knobs` maps names of DEFAULTS to values; nothing
    is read from the environment."""
    knobs = dict(knobs or {})
    bad = set(knobs) - set(DEFAULTS)
    if bad:
        raise ValueError(f"unknown generator knobs {sorted(bad)}; known: {sorted(DEFAULTS)}")
    cfg = {**DEFAULTS, **knobs}
    g = globals()
    for k in DEFAULTS:
        g[k] = type(DEFAULTS[k])(cfg[k])
    g["MEASURE"] = bool(measure)


def render(knobs=None, measure=False):
    """The generated text for the given knobs (defaults: the product kernel)."""
    configure(knobs, measure)
    try:
        return _render()
    finally:
        configure()


def _render():
    out = ["// Generated by gen_fwd64_pipe.py; do not edit.", "#pragma once", ""]
    for bf16, name in ((False, "F16"), (True, "BF16")):
        em = Emitter(bf16)
        lines = em.program()
        out.append(f"#define FAL_PIPE64_ASM_{name} \\")
        for ln in lines:
            out.append(f'  "{ln}\\n" \\')
        out.append("")
    outs, ins = operands()
    fmt = lambda ops: ", ".join(f'"{c}"({x})' for _, c, x in ops)
    clob = ", ".join([f'"v{i}"' for i in range(em.vlow, 256)] + [f'"s{i}"' for i in range(84, 100)] +
                     ['"vcc"', '"scc"', '"memory"'])
    out.append(f"#define FAL_PIPE64_OUTS {fmt(outs)}")
    out.append(f"#define FAL_PIPE64_INS {fmt(ins)}")
    out.append(f"#define FAL_PIPE64_CLOBBERS {clob}")
    out.append("")
    return "\n".join(out)


def main(path=None):
    """Write the default text to `path` (the tracked file when None)."""
    path = path or DEFAULT_PATH
    with open(path, "w") as f:
        f.write(render())
    return path


if __name__ == "__main__":
    print(main(sys.argv[1] if len(sys.argv) > 1 else None))
