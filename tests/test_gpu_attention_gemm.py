"""GPU parity: dense contractions, prefill / decode attention, int8 weight-only linear and the
fp32 decoder block vs the CPU oracle."""
import contextlib
import math

import pytest
import torch

from oracle import cpu_fallback as oracle
from tests.decoder import run_decoder_block, run_decomposed_decoder_block
from tests.parity import assert_close, assert_exact, assert_fp32, assert_half

pytestmark = pytest.mark.gpu


def g(seed):
    return torch.Generator().manual_seed(seed)


@contextlib.contextmanager
def own_context(ops, pkg):
    """A context for the calls within, outside of every scope: its workspace tells which form a product took."""
    ops._ctx = ctx = pkg.diopi.Context()
    try:
        yield ctx
        torch.cuda.synchronize()
    finally:
        ops._ctx = 0
        ctx.close()


# ------------------------------------------------------------------ contractions
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(256, 256, 64), (512, 768, 4096), (300, 200, 136), (1, 64, 64), (129, 257, 8),
                                   (1024, 1536, 512), (64, 11008, 4096)])
def test_linear_mfma_shapes(ops, dev, dtype, m, n, k):
    x = torch.randn(m, k, generator=g(0)).to(dtype)
    w = (torch.randn(n, k, generator=g(1)) * 0.05).to(dtype)
    b = torch.randn(n, generator=g(2)).to(dtype)
    want = x.float() @ w.float().t()
    assert_half(ops.linear(x.to(dev), w.to(dev)), want)
    assert_half(ops.linear(x.to(dev), w.to(dev), b.to(dev)), want + b.float())


def test_linear_known_answer_and_batched(ops, dev):
    # dipu/tests/python/unittests/test_linear.py:14-46: weight = bias = 1, x = arange
    for shape in [(3, 3), (2, 2, 3), (2, 2, 2, 3)]:
        x = torch.arange(math.prod(shape), dtype=torch.float).reshape(shape)
        y = ops.linear(x.to(dev), torch.ones(2, 3, device=dev), torch.ones(2, device=dev))
        assert_exact(y, x.sum(-1, keepdim=True).expand(*shape[:-1], 2) + 1)
    x = torch.randn(4, 96, 256, generator=g(3)).bfloat16()
    w = (torch.randn(320, 256, generator=g(4)) * 0.05).bfloat16()
    assert_half(ops.linear(x.to(dev), w.to(dev)), x.float() @ w.float().t())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_mm_bmm_matmul_addmm_baddbmm(ops, dev, dtype):
    chk = assert_fp32 if dtype == torch.float32 else assert_half
    a = torch.randn(130, 72, generator=g(5)).to(dtype)
    b = (torch.randn(72, 200, generator=g(6)) * 0.1).to(dtype)
    ref = a.float() @ b.float()
    chk(ops.mm(a.to(dev), b.to(dev)), ref)                                   # row-major mat2
    chk(ops.mm(a.to(dev), b.t().contiguous().to(dev).t()), ref)              # mat2 = W.t() view
    chk(ops.mm(a.t().contiguous().to(dev).t(), b.to(dev)), ref)              # column-major mat1
    ba = torch.randn(6, 40, 64, generator=g(7)).to(dtype)
    bb = (torch.randn(6, 64, 48, generator=g(8)) * 0.1).to(dtype)
    chk(ops.bmm(ba.to(dev), bb.to(dev)), torch.bmm(ba.float(), bb.float()))
    chk(ops.bmm(ba.to(dev), bb.transpose(1, 2).contiguous().to(dev).transpose(1, 2)), torch.bmm(ba.float(), bb.float()))
    # matmul: vector/matrix/batched/broadcast forms (test_matmul.py:8-71)
    v = torch.randn(64, generator=g(9)).to(dtype)
    chk(ops.matmul(v.to(dev), v.to(dev)), (v.float() @ v.float()))
    chk(ops.matmul(ba[0].to(dev), v.to(dev)), ba[0].float() @ v.float())
    chk(ops.matmul(v.to(dev), bb[0].to(dev)), v.float() @ bb[0].float())
    chk(ops.matmul(ba.to(dev), bb[0].to(dev)), ba.float() @ bb[0].float())
    chk(ops.matmul(ba.to(dev), bb.to(dev)), ba.float() @ bb.float())
    b4 = (torch.randn(2, 1, 64, 48, generator=g(10)) * 0.1).to(dtype)
    a4 = torch.randn(1, 3, 40, 64, generator=g(11)).to(dtype)
    chk(ops.matmul(a4.to(dev), b4.to(dev)), a4.float() @ b4.float())
    # addmm / baddbmm with broadcast addends and scalars
    c = torch.randn(200, generator=g(12)).to(dtype)
    chk(ops.addmm(c.to(dev), a.to(dev), b.to(dev), beta=0.5, alpha=2), 0.5 * c.float() + 2 * ref)
    c2 = torch.randn(130, 200, generator=g(13)).to(dtype)
    chk(ops.addmm(c2.to(dev), a.to(dev), b.to(dev)), c2.float() + ref)
    c3 = torch.randn(6, 40, 48, generator=g(14)).to(dtype)
    chk(ops.baddbmm(c3.to(dev), ba.to(dev), bb.to(dev), beta=2, alpha=0.5), 2 * c3.float() + 0.5 * torch.bmm(ba.float(), bb.float()))
    chk(ops.baddbmm(c3[:, :1].to(dev), ba.to(dev), bb.to(dev)), c3[:, :1].float() + torch.bmm(ba.float(), bb.float()))


@pytest.mark.parametrize("m,n,k,form", [
    (2048, 2048, 64, "linear"),      # 256 tiles of 128 x 128, operands straight into LDS
    (2048, 2048, 64, "mm"),          # the same with a row-major [K, N] second operand
    (1000, 1030, 96, "linear"),      # 64 x 64 tiles, ragged rows and columns
    (200, 328, 96, "linear"),        # the same in 32 x 32 tiles: fewer than 192 of 64 x 64
    (200, 328, 96, "mm"),
    (1100, 2100, 32, "addmm"),       # one stage; alpha, beta and a matrix addend in the epilogue
    (1000, 1030, 72, "linear"),      # K no multiple of 32: tiles staged through registers
    (130, 200, 72, "linear"),        # 32 x 32 tiles, a K that ends inside a stretch
    (130, 200, 72, "mm"),
    (136, 200, 36, "mm_at"),         # transposed first operand (row-contiguous along M)
    (2304, 2048, 40, "mm"),          # staged, 128 x 128 tiles, ragged last stage
    (64, 64, 4100, "bmm"),           # long K, batch 3
    (33, 40, 8, "linear"),           # one partial tile
    (31, 64, 64, "linear"),          # fewer than 32 rows
    (31, 12300, 64, "linear"),       # the same over 193 tiles: the FMA engine
    (64, 8200, 64, "linear"),        # 514 tiles of 32 x 32, more than two on a compute unit: 64 x 64 at a short K ...
    (64, 8200, 256, "linear"),       # ... and 32 x 32 at a longer one
])
def test_fp32_gemm_on_the_matrix_cores(ops, dev, m, n, k, form):
    """fp32 operands through the fp32 MFMA kernels (both tile sizes, operands straight into LDS or staged through
    registers, either layout of the second operand) against the product in float64: true fp32 products and sums, so
    only the summation order differs (1e-5 of the largest sum)."""
    x, w = torch.randn(m, k, generator=g(40)), torch.randn(n, k, generator=g(41))
    want = x.double() @ w.double().t()
    if form == "linear":
        b = torch.randn(n, generator=g(42))
        assert_fp32(ops.linear(x.to(dev), w.to(dev)), want)
        assert_fp32(ops.linear(x.to(dev), w.to(dev), b.to(dev)), want + b.double())
    elif form == "mm":
        assert_fp32(ops.mm(x.to(dev), w.t().contiguous().to(dev)), want)
    elif form == "mm_at":
        assert_fp32(ops.mm(x.t().contiguous().to(dev).t(), w.t().contiguous().to(dev)), want)
    elif form == "addmm":
        c = torch.randn(m, n, generator=g(43))
        assert_fp32(ops.addmm(c.to(dev), x.to(dev), w.to(dev).t(), beta=0.5, alpha=2), 0.5 * c.double() + 2 * want)
    else:
        xb, wb = torch.randn(3, m, k, generator=g(44)), torch.randn(3, k, n, generator=g(45))
        assert_fp32(ops.bmm(xb.to(dev), wb.to(dev)), torch.bmm(xb.double(), wb.double()))
    # a one-hot row picks one weight column exactly, whatever the tiling
    if form == "linear":
        onehot = torch.zeros(m, k)
        onehot[torch.arange(m), torch.arange(m) % k] = 1.0
        assert_exact(ops.linear(onehot.to(dev), w.to(dev)), w.t()[torch.arange(m) % k])


@pytest.mark.parametrize("batch,m,n,k", [(1, 256, 512, 1376), (1, 1, 33, 4), (1, 31, 100, 516), (3, 65, 64, 1024 + 28), (1, 700, 512, 96)])
def test_fp32_gemm_with_few_tiles(ops, dev, batch, m, n, k):
    """32 x 32 tiles with K dealt over the waves: fewer stretches of 32 than waves, none at all, a K that ends inside one,
    ragged rows and columns, a batch, bias and addend; and exactly on one-hot rows."""
    x, w = torch.randn(batch, m, k, generator=g(95)), torch.randn(n, k, generator=g(96))
    bias, c = torch.randn(n, generator=g(97)), torch.randn(batch, m, n, generator=g(98))
    want = x.double() @ w.double().t()
    dx, dw = x.to(dev), w.to(dev)
    assert_fp32(ops.linear(dx, dw, bias.to(dev)), want + bias.double())
    wb = dw.t().unsqueeze(0).expand(batch, k, n)
    assert_fp32(ops.baddbmm(c.to(dev), dx, wb, beta=0.5, alpha=2), 0.5 * c.double() + 2 * want)
    onehot = torch.zeros(m, k)
    cols = torch.randint(0, k, (m,), generator=g(99))
    cols[-1] = k - 1
    onehot[torch.arange(m), cols] = 1
    assert_exact(ops.linear(onehot.to(dev), dw), w[:, cols].t().contiguous())


def test_gemm_linearity_at_7b_shapes(ops, dev):
    # size-independent property at the full prefill shape: f(x1 + x2) = f(x1) + f(x2), and a
    # one-hot row selects a weight column exactly
    w = (torch.randn(11008, 4096, generator=g(15)) * 0.02).bfloat16().to(dev)
    x1 = torch.randn(8192, 4096, generator=g(16)).bfloat16().to(dev)
    y1 = ops.linear(x1, w)
    want = x1[:32].float().cpu() @ w.float().cpu().t()
    assert_half(y1[:32], want)
    assert_half(y1[-32:], x1[-32:].float().cpu() @ w.float().cpu().t())
    onehot = torch.zeros(256, 4096, dtype=torch.bfloat16, device=dev)
    cols = torch.randint(0, 4096, (256,), generator=g(17)).to(dev)
    onehot[torch.arange(256, device=dev), cols] = 1
    assert_exact(ops.linear(onehot, w), w[:, cols].t().contiguous().cpu())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(3500, 3700, 128), (3500, 3700, 192), (3841, 3585, 320), (4096, 4096, 1088)])
def test_large_tile_gemm_edges_and_k_tile_counts(ops, dev, dtype, m, n, k):
    """At least 144 tiles of 256 x 256 and K a multiple of 64 select the 8-wave kernel whose tiles are loaded
    straight into LDS: two, three, five and seventeen K tiles (even and odd ring positions at the end),
    ragged last tile rows / columns, bias, and the alpha / beta epilogue."""
    x = torch.randn(m, k, generator=g(40)).to(dtype)
    w = (torch.randn(n, k, generator=g(41)) * 0.05).to(dtype)
    b = torch.randn(n, generator=g(42)).to(dtype)
    want = x.float() @ w.float().t()
    dx, dw = x.to(dev), w.to(dev)
    assert_half(ops.linear(dx, dw), want)
    assert_half(ops.linear(dx, dw, b.to(dev)), want + b.float())
    c = torch.randn(m, n, generator=g(43)).to(dtype)
    assert_half(ops.addmm(c.to(dev), dx, dw.t(), beta=0.5, alpha=2), 0.5 * c.float() + 2 * want)


def test_large_tile_gemm_batched_and_row_strided_operands(ops, dev):
    # 4 batches of 8 x 8 tiles; A rows taken out of a wider buffer (row stride > K), B shared by all batches
    wide = torch.randn(4, 2000, 512, generator=g(44)).bfloat16().to(dev)
    a = wide[:, :, 128:128 + 320]
    assert not a.is_contiguous()
    w = (torch.randn(1900, 320, generator=g(45)) * 0.05).bfloat16()
    want = a.float().cpu() @ w.float().t()
    assert_half(ops.matmul(a, w.to(dev).t()), want)
    bb = (torch.randn(4, 1900, 320, generator=g(46)) * 0.05).bfloat16()
    assert_half(ops.bmm(a, bb.to(dev).transpose(1, 2)), torch.bmm(a.float().cpu(), bb.float().transpose(1, 2)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,m,k,n", [(1, 4096, 512, 4096),      # 256 x 256 tiles
                                         (1, 1024, 4096, 4096),     # 128 x 128 tiles
                                         (1, 200, 1024, 520),       # 128 x 128 tiles, K split, ragged edges
                                         (3, 700, 128, 136),        # batched, two K tiles, a narrow matrix
                                         (16, 2048, 2048, 128),     # the P . V product of decomposed attention
                                         (2, 2304, 192, 2048)])     # batched 256 x 256 tiles, three K tiles
def test_second_operand_read_in_place_as_k_by_n(ops, dev, dtype, batch, m, k, n):
    """mm / bmm / matmul with the right-hand side as the caller holds it, [K, N] row-major: the tile kernels read it in
    place. Checked against the fp32 product, and exactly: one-hot rows on the left select rows of the right."""
    g0 = g(91)
    a = torch.randn(batch, m, k, generator=g0).to(dtype)
    b = (torch.randn(batch, k, n, generator=g0) * 0.05).to(dtype)
    want = a.float() @ b.float()
    got = ops.bmm(a.to(dev), b.to(dev)) if batch > 1 else ops.mm(a[0].to(dev), b[0].to(dev)).unsqueeze(0)
    assert_half(got, want)
    rows = torch.randint(0, k, (batch, m), generator=g0)
    onehot = torch.zeros(batch, m, k, dtype=dtype)
    onehot.scatter_(2, rows.unsqueeze(-1), 1)
    sel = torch.gather(b, 1, rows.unsqueeze(-1).expand(batch, m, n))
    got = ops.bmm(onehot.to(dev), b.to(dev)) if batch > 1 else ops.mm(onehot[0].to(dev), b[0].to(dev)).unsqueeze(0)
    assert_exact(got, sel)
    if batch == 1:
        # a column slice of a wider matrix as the right-hand side (row stride above N), through matmul with a broadcast left side
        wide = (torch.randn(k, n + 64, generator=g0) * 0.05).to(dtype)
        a3 = torch.randn(2, m, k, generator=g0).to(dtype)
        got = ops.matmul(a3.to(dev), wide.to(dev)[:, 8:8 + n])
        assert_half(got, a3.float() @ wide[:, 8:8 + n].float())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epilogue", ["linear", "bias", "addend", "addend_ragged", "addend_in_place_scaled", "addend_batched", "rotary",
                                      "rotary_bias", "rotary_conj", "rotary_f32_tables", "rotary_ragged_rows", "silu_mul"])
def test_four_wave_gemm_every_instantiation_exact(ops, dev, dtype, epilogue):
    """Every instantiation of the 4-wave large-tile kernel (two dtypes x plain, bias, addend (the form that finds a quarter of
    each tile's addend in LDS; also with rows and columns that end inside the last tiles and an addend with a longer row
    pitch, with the output written over the addend under alpha and beta, and batched), rotary without a bias and
    with 16-bit tables (the form whose table entries wait in LDS; also with the conjugate rotation and with rows that
    end inside the last tile), rotary with fp32 tables (the wave-uniform form), rotary with a bias (the general form)
    and gated epilogues) by name, on a problem of 288 tiles of 256 x 256 so that every workgroup walks at least one tile after
    its first (the path that requests the next tile's operands before the epilogue) and K = 256 (a prologue, one loop
    body and the tail). The kernel keeps its accumulators and operand fragments in registers the compiler only knows
    as clobbered: a change of register allocation around the loop would show here. Activations are one-hot rows, so
    every product is one weight element and the expected result is exact."""
    g0 = g(77)
    m, n, k = 8192, 2304, 256
    if epilogue in ("rotary_ragged_rows", "addend_ragged"):
        m -= 64                                         # 31 whole tile rows and 192 rows of the last one
    if epilogue == "addend_ragged":
        n -= 40                                         # 8 whole tile columns and 216 columns of the last one
    cols = torch.randint(0, k, (m,), generator=g0)
    x = torch.zeros(m, k, dtype=dtype)
    x[torch.arange(m), cols] = 1
    if epilogue == "silu_mul":
        w = torch.randn(2 * n, k, generator=g0).to(dtype)
        got = ops.linear_silu_mul(x.to(dev), w.to(dev))
        y = w.float()[:, cols].t().reshape(m, n // 32, 2, 32)
        want = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(m, n)
        assert_half(got, want)      # silu goes through exp: not an exact case, but every element is one known product
        return
    w = torch.randn(n, k, generator=g0).to(dtype)
    sel = w.float()[:, cols].t()                        # [m, n]: out[i] = w[:, cols[i]]
    if epilogue == "linear":
        assert_exact(ops.linear(x.to(dev), w.to(dev)), sel.to(dtype))
    elif epilogue == "bias":
        b = torch.randn(n, generator=g0).to(dtype)
        assert_exact(ops.linear(x.to(dev), w.to(dev), b.to(dev)), (sel + b.float()).to(dtype))
    elif epilogue == "addend":
        c = torch.randn(m, n, generator=g0).to(dtype)
        assert_exact(ops.addmm(c.to(dev), x.to(dev), w.to(dev).t()), (c.float() + sel).to(dtype))
    elif epilogue == "addend_ragged":
        wide = torch.randn(m, n + 24, generator=g0).to(dtype)      # the addend is a column slice: its rows are 24 elements apart
        got = ops.addmm(wide.to(dev)[:, 8:8 + n], x.to(dev), w.to(dev).t())
        assert_exact(got, (wide[:, 8:8 + n].float() + sel).to(dtype))
    elif epilogue == "addend_batched":
        # two batches of the same problem through baddbmm: the addend and the output of batch 1 lie a batch stride further on
        c = torch.randn(2, m, n, generator=g0).to(dtype)
        x2 = torch.stack([x, x.flip(0)])
        sel2 = torch.stack([sel, sel.flip(0)])
        got = ops.baddbmm(c.to(dev), x2.to(dev), w.to(dev).t().unsqueeze(0).expand(2, k, n))
        assert_exact(got, (c.float() + sel2).to(dtype))
    elif epilogue == "addend_in_place_scaled":
        c = torch.randn(m, n, generator=g0).to(dtype)
        dc = c.to(dev)
        got = ops.addmm(dc, x.to(dev), w.to(dev).t(), beta=0.5, alpha=2, out=dc)     # powers of two: still one rounding
        assert got.data_ptr() == dc.data_ptr()
        assert_exact(got, (0.5 * c.float() + 2 * sel).to(dtype))
    else:
        # tables of signed powers of two: each rotated value is a sum of two exactly scaled terms, rounded once
        hd, rows = 128, 64
        e = torch.randint(-3, 1, (rows, hd // 2), generator=g0).float()
        sg = torch.randint(0, 2, (rows, hd // 2), generator=g0).float() * 2 - 1
        tdt = torch.float32 if epilogue == "rotary_f32_tables" else dtype
        cos, sin = (2.0 ** e).to(tdt), (sg * 2.0 ** (e - 1)).to(tdt)
        rot = n - 2 * hd                                # the last two heads pass through, like v
        conj = epilogue == "rotary_conj"
        b = (torch.randint(-4, 5, (n,), generator=g0).float() / 4).to(dtype) if epilogue == "rotary_bias" else None
        got = ops.linear_rotary(x.to(dev), w.to(dev), cos.to(dev), sin.to(dev), rot, hd, None if b is None else b.to(dev),
                                conj=conj, interleaved=True)
        if b is not None:
            sel = sel + b.float()                       # quarters added to 8- or 11-bit values: exact in fp32
        v = sel.clone().reshape(m, n // hd, hd // 2, 2)
        cf = cos.float()[torch.arange(m) % rows][:, None, :]
        sf = sin.float()[torch.arange(m) % rows][:, None, :] * (-1.0 if conj else 1.0)
        out = torch.stack([v[..., 0] * cf - v[..., 1] * sf, v[..., 0] * sf + v[..., 1] * cf], dim=-1)
        out[:, rot // hd:] = v[:, rot // hd:]
        assert_exact(got, out.reshape(m, n).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epilogue,m,n,k,left,slices,other", [
    ("linear", 1554, 11000, 4096, 45, 4, 0),          # 301 tiles: a whole round, then 45 tiles in slices; ragged rows and columns
    ("bias", 1554, 11008, 4096 + 128, 45, 5, 0),      # 33 K-tile pairs: slices of unequal length
    ("linear", 4525, 4096, 4096, 32, 4, 0), ("linear", 4525, 4096, 14336, 32, 8, 0), ("linear", 6001, 4096, 4096, 128, 2, 0),
    ("linear", 882, 5120, 5120, 80, 3, 0),            # 80 tiles: slices only
    ("addend", 882, 5120, 13824, 80, 3, 0),
    ("addend", 300, 8192, 8192, 0, 0, 0),             # 64 tiles: 128 x 128 ones instead
    ("linear", 512, 4096, 11008, 0, 0, 2 * 512 * 4096 * 4),                      # the same, split over K
    ("addend", 5000, 5120, 13824, 144, 3, 0),         # 400 tiles, 144 left: more slices than workgroups
    ("rotary", 1554, 12288, 4096, 80, 3, 0), ("rotary", 203, 22016, 4096, 86, 2, 0),
    ("silu_mul", 1554, 22016, 4096, 90, 2, 0), ("silu_mul", 400, 12288, 4096, 96, 2, 0),
    ("column_scale", 882, 5120, 13824, 80, 3, 0),      # int8 weights as they are
    ("column_scale", 3000, 6144, 4096, 32, 4, 6144 * 4096 * 2)])                 # and the weight in 16 bits
def test_four_wave_gemm_last_round_split_along_k_exact(ops, dev, pkg, dtype, epilogue, m, n, k, left, slices, other):
    """The tiles of a partly filled last round in slices of K (the 4-wave kernel's accumulators as fp32 partial sums, added
    and given the epilogue by a second launch): as many as the workspace tells, with whole rounds before them and without.
    One-hot activations over the whole of K: every product is one weight element, found by exactly one slice, and the
    expected result is exact."""
    ops._ctx = ctx = pkg.diopi.Context()             # outside a scope, whose products take no such workspace
    try:
        check_last_round(ops, dev, dtype, epilogue, m, n, k)
        assert ctx.workspace()[1] == left * slices * 256 * 1024 + other
        torch.cuda.synchronize()
    finally:
        ops._ctx = 0
        ctx.close()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.int16])
@pytest.mark.parametrize("shape", [(8, 8), (9, 65), (3, 7, 64), (2, 64, 64), (5, 63, 129), (2, 777, 128), (1, 1000, 9)])
def test_transposing_copy_of_two_byte_elements(ops, dev, shape, dtype):
    """Blocks of 8 x 8 in registers, the last ones overlapping those before; fewer than 8 rows take the other kernel. Rows of
    a wider matrix, from an odd element on; what lies around the destination stays."""
    wide = torch.randint(-30000, 30000, (*shape[:-1], shape[-1] + 5), generator=g(81)).to(torch.int16)
    if dtype != torch.int16:
        wide = torch.randn(wide.shape, generator=g(82)).to(dtype)
    src = wide.to(dev)[..., 3:3 + shape[-1]]
    want = src.transpose(-1, -2).contiguous()
    buf = torch.zeros(want.numel() + 2, dtype=dtype, device=dev)
    out = buf[1:-1].view(want.shape)
    ops.copy_(out, src.transpose(-1, -2))
    assert_exact(out, want)
    assert buf[0] == 0 and buf[-1] == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(129, 131, 128), (300, 7, 192), (70, 777, 128), (2310, 4101, 256), (128, 255, 320)])
def test_outputs_without_whole_pieces(ops, dev, dtype, m, n, k):
    """Rows of an odd number of columns, stored 8 columns at a time at element alignment, the last ones one by one: exact on
    one-hot activations, with a bias and with an addend whose columns are not contiguous, in both tile sizes."""
    g0 = g(83)
    cols = torch.randint(0, k, (m,), generator=g0)
    x = torch.zeros(m, k, dtype=dtype)
    x[torch.arange(m), cols] = 1
    w = torch.randn(n, k, generator=g0).to(dtype)
    sel = w[:, cols].float().t()
    b, c = torch.randn(n, generator=g0).to(dtype), torch.randn(n, m, generator=g0).to(dtype)
    assert_exact(ops.linear(x.to(dev), w.to(dev)), sel.to(dtype))
    assert_exact(ops.linear(x.to(dev), w.to(dev), b.to(dev)), (sel + b.float()).to(dtype))
    assert_exact(ops.addmm(c.to(dev).t(), x.to(dev), w.to(dev).t()), (c.t().float() + sel).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epilogue,m,n,k", [
    ("linear", 224, 40960, 256),                      # one row of whole tiles, full
    ("linear", 225, 40960, 256),                      # one row too many: 256
    ("bias", 447, 20488, 384), ("silu_mul", 448, 22016, 256), ("addend", 1344, 8192, 256), ("rotary", 1121, 12288, 256),
    ("rotary", 1120, 12288, 256),                     # 5 rows of tiles each, the first of them just above what 224 rows hold
    ("linear", 1568, 11008, 1024),                    # a whole round, then slices
    ("silu_mul", 193, 28672, 4096), ("column_scale", 440, 12288, 4096), ("column_scale", 1100, 10240, 256),
    ("addend", 400, 12288, 4096), ("rotary", 210, 22016, 4096)])         # slices only
def test_four_wave_gemm_tiles_of_224_rows_exact(ops, dev, dtype, epilogue, m, n, k):
    """Row counts at and around those that fill tiles of 224 rows, in every epilogue, whole tiles and slices of K."""
    check_last_round(ops, dev, dtype, epilogue, m, n, k)


def check_last_round(ops, dev, dtype, epilogue, m, n, k):
    g0 = g(78)
    cols = torch.randint(0, k, (m,), generator=g0)
    cols[:4] = torch.tensor([0, k - 1, 127, 128])
    x = torch.zeros(m, k, dtype=dtype)
    x[torch.arange(m), cols] = 1
    if epilogue == "column_scale":
        w = torch.randint(-127, 128, (n, k), generator=g0, dtype=torch.int8)
        scale = (0.001 + 0.019 * torch.rand(n, generator=g0)).to(torch.float16)
        assert_exact(ops.weight_only_int8_linear(x.to(dev), w.to(dev), scale.to(dev)),
                     (w[:, cols].float() * scale.float()[:, None]).t().to(dtype))
        return
    w = torch.randn(n, k, generator=g0).to(dtype)
    sel = w[:, cols].float().t()
    if epilogue == "linear":
        assert_exact(ops.linear(x.to(dev), w.to(dev)), sel.to(dtype))
    elif epilogue == "bias":
        b = torch.randn(n, generator=g0).to(dtype)
        assert_exact(ops.linear(x.to(dev), w.to(dev), b.to(dev)), (sel + b.float()).to(dtype))
    elif epilogue == "addend":
        c = torch.randn(m, n, generator=g0).to(dtype)
        assert_exact(ops.addmm(c.to(dev), x.to(dev), w.to(dev).t(), beta=0.5, alpha=2), (0.5 * c.float() + 2 * sel).to(dtype))
    elif epilogue == "silu_mul":
        y = sel.reshape(m, n // 64, 2, 32)
        assert_half(ops.linear_silu_mul(x.to(dev), w.to(dev)), (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(m, n // 2))
    else:
        hd, rot = 128, n - 256
        e = torch.randint(-3, 1, (m, hd // 2), generator=g0).float()
        cos, sin = 2.0 ** e, 2.0 ** (e - 1)             # powers of two: a sum of two exactly scaled terms, rounded once
        v = sel.clone().reshape(m, n // hd, hd // 2, 2)
        out = torch.stack([v[..., 0] * cos[:, None] - v[..., 1] * sin[:, None], v[..., 0] * sin[:, None] + v[..., 1] * cos[:, None]], dim=-1)
        out[:, rot // hd:] = v[:, rot // hd:]
        got = ops.linear_rotary(x.to(dev), w.to(dev), cos.to(dtype).to(dev), sin.to(dtype).to(dev), rot, hd, interleaved=True)
        assert_exact(got, out.reshape(m, n).to(dtype))


@pytest.mark.parametrize("m,n,k", [(70, 136, 192), (70, 136, 256), (129, 264, 320), (129, 264, 384), (65, 136, 448), (100, 136, 512), (130, 264, 2752), (100, 4096, 11008)])
def test_products_with_few_tiles_four_stage_ring_exact(ops, dev, m, n, k):
    """K no longer than the four-stage ring (two stages), two slices as long as it, and one to three K tiles longer; K slices of unequal length; the [K, N]
    operand in place and the K-contiguous one. One-hot rows over the whole of K: exact."""
    g0 = g(79)
    cols = torch.randint(0, k, (m,), generator=g0)
    cols[:3] = torch.tensor([0, k - 1, k - 64])
    x = torch.zeros(m, k, dtype=torch.bfloat16)
    x[torch.arange(m), cols] = 1
    w = torch.randn(n, k, generator=g0).to(torch.bfloat16)
    want = w[:, cols].t().contiguous()
    assert_exact(ops.linear(x.to(dev), w.to(dev)), want)
    assert_exact(ops.mm(x.to(dev), w.t().contiguous().to(dev)), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,bias", [
    (203, 12288, 256, False),          # 192 tiles of 128: one round of the 128 x 128 kernel
    (65, 17408 + 64, 192, True),       # K shorter than its ring, a last tile of half the columns, the general rotary form
    (300, 13312, 320, False),          # 312 tiles: two workgroups per CU
    (203, 22016, 4096, False),         # 86 tiles of 256 in two K slices each
    (130, 1024, 1024, False)])         # a product split over K: the separate pass
def test_gate_and_rotation_in_the_epilogue_at_a_few_hundred_rows(ops, dev, dtype, m, n, k, bias):
    """One-hot activations: every product is one weight element, so the rotation by powers of two is exact."""
    g0 = g(81)
    cols = torch.randint(0, k, (m,), generator=g0)
    cols[:2] = torch.tensor([0, k - 1])
    x = torch.zeros(m, k, dtype=dtype)
    x[torch.arange(m), cols] = 1
    w = torch.randn(n, k, generator=g0).to(dtype)
    sel = w[:, cols].float().t()
    y = sel.reshape(m, n // 64, 2, 32)
    assert_half(ops.linear_silu_mul(x.to(dev), w.to(dev)), (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(m, n // 2))
    hd = 64
    rot = n - 256
    b = torch.zeros(n, dtype=dtype)
    if bias:
        b[rot:] = 1
    e = torch.randint(-3, 1, (m, hd // 2), generator=g0).float()
    cos, sin = 2.0 ** e, 2.0 ** (e - 1)
    v = sel.clone().reshape(m, n // hd, hd // 2, 2)
    out = torch.stack([v[..., 0] * cos[:, None] - v[..., 1] * sin[:, None], v[..., 0] * sin[:, None] + v[..., 1] * cos[:, None]], dim=-1)
    out[:, rot // hd:] = v[:, rot // hd:]
    want = out.reshape(m, n) + b.float()
    got = ops.linear_rotary(x.to(dev), w.to(dev), cos.to(dtype).to(dev), sin.to(dtype).to(dev), rot, hd, b.to(dev) if bias else None,
                            interleaved=True)
    assert_exact(got, want.to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,m,n,k", [(3, 777, 128, 777), (2, 129, 131, 65), (1, 1, 1, 1), (5, 128, 127, 7), (1, 300, 500, 4097),
                                           (1, 130, 257, 1031), (2, 127, 129, 390), (1, 2048, 2048, 33)])
def test_products_over_a_k_that_is_no_multiple_of_eight(ops, dev, dtype, batch, m, n, k):
    """Rows that start at any element: K ends inside a 16-byte piece, inside a 64-wide K tile and one element into one, and
    lies inside the first; a K of which the matrix kernel has too little (65 and below) on the FMA engine;
    the [K, N] and the transposed second operand, a K-strided first one, and a linear with a bias. The fp32 product, and
    exactly on one-hot rows. The operands end where their allocations do: nothing may be read past them."""
    a, b = torch.randn(batch, m, k, generator=g(91)).to(dtype), torch.randn(batch, k, n, generator=g(92)).to(dtype)
    want = a.float() @ b.float()
    da, db = a.to(dev), b.to(dev)
    assert_half(ops.bmm(da, db), want)
    assert_half(ops.bmm(da, db.transpose(1, 2).contiguous().transpose(1, 2)), want)
    assert_half(ops.bmm(da.transpose(1, 2).contiguous().transpose(1, 2), db), want)
    bias = torch.randn(n, generator=g(93)).to(dtype)
    assert_half(ops.linear(da, db[0].t().contiguous(), bias.to(dev)), a.float() @ b[0].float() + bias.float())
    onehot = torch.zeros(batch, m, k, dtype=dtype)
    cols = torch.randint(0, k, (batch, m), generator=g(94))
    cols[:, -1] = k - 1
    onehot.scatter_(2, cols[:, :, None], 1)
    assert_exact(ops.bmm(onehot.to(dev), db), torch.gather(b, 1, cols[:, :, None].expand(batch, m, n)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1024, 4096, 4096), (300, 520, 1024), (65, 4096, 4096 + 64), (2047, 2048, 576),
                                   (512, 768, 4096)])
def test_split_k_gemm(ops, dev, dtype, m, n, k):
    """More than 64 rows but fewer than 144 tiles of 256 x 256, K a multiple of 64 with at least eight K tiles: the
    large-tile kernel with K split over the grid (4, 4, 13, 2 and 16 ways here; 65 K tiles in splits of 5, 9 in splits
    of 5 + 4), fp32 partial products and a reduction pass that applies bias and the alpha / beta epilogue; ragged
    last tile rows and columns."""
    x = torch.randn(m, k, generator=g(60)).to(dtype)
    w = (torch.randn(n, k, generator=g(61)) * 0.05).to(dtype)
    b = torch.randn(n, generator=g(62)).to(dtype)
    want = x.float() @ w.float().t()
    dx, dw = x.to(dev), w.to(dev)
    assert_half(ops.linear(dx, dw), want)
    assert_half(ops.linear(dx, dw, b.to(dev)), want + b.float())
    c = torch.randn(m, n, generator=g(63)).to(dtype)
    assert_half(ops.addmm(c.to(dev), dx, dw.t(), beta=0.5, alpha=2), 0.5 * c.float() + 2 * want)
    onehot = torch.zeros(m, k, dtype=dtype, device=dev)
    cols = torch.randint(0, k, (m,), generator=g(64)).to(dev)
    onehot[torch.arange(m, device=dev), cols] = 1
    assert_exact(ops.linear(onehot, dw), dw[:, cols].t().contiguous().cpu())


@pytest.mark.parametrize("m,n,k,ways", [(600, 4096, 11008, 3), (300, 4096, 11008, 5), (512, 4096, 11008, 2), (203, 4096, 4096, 4),
                                        (1024, 4096, 4096, 1), (1300, 2048, 512, 1)])
def test_slices_of_k_for_one_or_two_workgroups_on_a_compute_unit(ops, dev, pkg, m, n, k, ways):
    """Tiles of 128 x 128 against a [K, N] operand: K in slices for two workgroups on a CU where a long K would leave too few
    of one (the first two), for one, and not at all, which the workspace of the partial sums tells. Sums of small whole
    numbers, exact in fp32."""
    gen = torch.Generator().manual_seed(65)
    x, w = (torch.randint(-2, 3, s, generator=gen).to(torch.bfloat16).to(dev) for s in ((m, k), (k, n)))
    out = torch.empty(m, n, dtype=torch.bfloat16, device=dev)
    with pkg.diopi.Context() as ctx:
        handles = [pkg.diopi.handle(t) for t in (out, x, w)]
        pkg.diopi.call("diopiMm", ctx, *[p for _, p in handles])
        assert ctx.workspace() == ((1, ways * m * n * 4) if ways > 1 else (0, 0))
        torch.cuda.synchronize()
    assert torch.equal(out, (x.float() @ w.float()).to(torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (5, 100, 8192 + 128), (16, 11008, 4096), (17, 4096, 11008),
                                   (40, 16 * 7 + 3, 384), (64, 16000, 128), (1, 16, 128), (64, 4096, 4096),
                                   (48, 12288, 1024 + 768), (33, 2056, 11008),
                                   (64, 12288, 4096), (33, 12296, 4096 + 128), (50, 16384, 4096 + 384), (64, 22016, 4096), (64, 9216, 4096),
                                   (64, 4096, 8192), (40, 4104, 11008), (64, 6144, 4096 + 640),
                                   (20, 8200, 640), (1, 12288, 256), (32, 32000, 384), (7, 8192, 128)])
def test_skinny_m_linear_and_addmm(ops, dev, dtype, m, n, k):
    """(Where few columns come on a compute unit the kernel of the test below takes the product by now: 1 x 4096 x 4096, 64 x 4096 x 4096, 64 x
    6144 x 4736 and others. What follows is of the shapes that it leaves.)
    At most 64 rows against a K-contiguous weight with K a multiple of 128 select the weight-streaming kernel:
    one, two and four 16-column tiles per workgroup (N = 4096, 11008, 32000), K in one and in two staged chunks
    and down to a single step per wave, row groups of 16 with a ragged last group, ragged N, bias, and the
    alpha / beta epilogue with a full and a broadcast addend. With more than 32 rows K is also split over the grid
    in slices of 1024 (4, 2 with a ragged second, and 11 slices here; N = 16 * 7 + 3 is not a multiple of 8 and
    stays unsplit) and a reduction pass applies the epilogue. Five cases (more than 32 rows, at least 512
    column tiles, K from 4096) take the whole-K form with double-buffered activations: three and four tiles per
    workgroup, a last chunk of one and of three steps, a ragged last tile and a last workgroup with a tile past N;
    the three after them run it on K slices (four even slices, four with a short last one, two with a ragged
    second) that meet in the reduction pass. Weights at least 5120 columns wide (4096 at 17 to 32 rows) take the
    form that stages both operands through LDS (columns dealt evenly over the CUs, up to 64 or 128 per workgroup,
    walking K in stages of 128 from a staggered start): one to four row groups, column shares that are no multiple
    of 16, a last workgroup with fewer columns, K of one, two, three and five stages (fewer than the ring holds)
    up to 86. Two cases (more than 32 rows, 4096 and 4104 columns, K of 8192 and 11008) take that form with K split two
    ways over the grid and the reduction pass."""
    x = torch.randn(m, k, generator=g(50)).to(dtype)
    w = (torch.randn(n, k, generator=g(51)) * 0.05).to(dtype)
    b = torch.randn(n, generator=g(52)).to(dtype)
    want = x.float() @ w.float().t()
    dx, dw = x.to(dev), w.to(dev)
    assert_half(ops.linear(dx, dw), want)
    assert_half(ops.linear(dx, dw, b.to(dev)), want + b.float())
    c = torch.randn(m, n, generator=g(53)).to(dtype)
    assert_half(ops.addmm(c.to(dev), dx, dw.t(), beta=0.5, alpha=2), 0.5 * c.float() + 2 * want)
    assert_half(ops.addmm(b.to(dev), dx, dw.t()), b.float() + want)
    # a one-hot row selects a weight column exactly
    onehot = torch.zeros(m, k, dtype=dtype, device=dev)
    cols = torch.randint(0, k, (m,), generator=g(54)).to(dev)
    onehot[torch.arange(m, device=dev), cols] = 1
    assert_exact(ops.linear(onehot, dw), dw[:, cols].t().contiguous().cpu())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(3, 16, 16), (1, 250, 16904), (16, 4096, 520), (5, 4098, 1032), (16, 8192, 512), (4, 8190, 8208), (17, 4096, 1544),
                                   (32, 250, 8192), (32, 300, 48), (2, 4100, 1528), (33, 4096, 264), (48, 250, 3080), (49, 8192, 1288), (64, 4104, 4096),
                                   (17, 8190, 1032)])
def test_few_columns_for_a_compute_unit(ops, dev, dtype, m, n, k):
    # the kernel that streams few columns for each compute unit over the whole of K: ragged column shares, a last stage that
    # is not whole, fewer stages than ring places, one and two row groups; rows lie in a wider matrix of NaNs. (16 x 8192 x 512 in int8 is
    # declined, and K that is no multiple of 16 goes to the kernel with one output a lane there: int8 forms in the test below)
    wide = torch.full((m, k + 24), float("nan"), dtype=dtype)
    wide[:, :k] = torch.randn(m, k, generator=g(1)).to(dtype)
    x, xd = wide[:, :k], wide.to(dev)[:, :k]
    w = (torch.randn(n, k, generator=g(2)) / k**0.5).to(dtype)
    c, b = torch.randn(m, n, generator=g(3)).to(dtype), torch.randn(n, generator=g(4)).to(dtype)
    want = x.double() @ w.double().t()
    assert_half(ops.linear(xd, w.to(dev)), want)
    assert_half(ops.linear(xd, w.to(dev), b.to(dev)), want + b.double())
    assert_half(ops.addmm(c.to(dev), xd, w.to(dev).t(), beta=0.5, alpha=2.0), 0.5 * c.double() + 2 * want)
    q = torch.randint(-127, 128, (n, k), generator=g(5), dtype=torch.int8)
    scale = (torch.rand(n, generator=g(6)) + 0.5) / (73 * k**0.5)
    want = (x.double() @ q.double().t()) * scale.half().double()
    assert_half(ops.weight_only_int8_linear(xd, q.to(dev), scale.half().to(dev)), want)
    assert_half(ops.weight_only_int8_linear(xd, q.to(dev), scale.half().to(dev), b.to(dev)), want + b.double())


def check_rotations(ops, gen, x, w, b, want, hd):
    """The rotated projection of x by w, whose exact value is `want`, in its forms: either way, with a bias, with tables of both types, of a row
    for each row of x and of half as many. They hold signed powers of two, so that every result is rounded once."""
    (m, n), dev, dtype = want.shape, want.device, x.dtype
    cols = n * 3 // 4 // hd * hd
    fewer = m // 2 if m % 2 == 0 else m
    for rows, table_dtype, conj, bias in ((m, dtype, False, None), (fewer, torch.float32, True, b), (fewer, dtype, True, b)):
        e, sign = (torch.randint(low, high, (rows, hd // 2), generator=gen, device=dev) for low, high in ((-3, 1), (0, 2)))
        cos, sin = 2.0 ** e, (sign * 2.0 - 1) * 2.0 ** (e - 1)
        got = ops.linear_rotary(x, w, cos.to(table_dtype), sin.to(table_dtype), cols, hd, bias=bias, conj=conj)
        v = want if bias is None else want + bias.double()
        pairs, co, si = v[:, :cols].reshape(m // rows, rows, cols // hd, hd // 2, 2), cos.double()[:, None], sin.double()[:, None] * (-1 if conj else 1)
        rotated = torch.stack([pairs[..., 0] * co - pairs[..., 1] * si, pairs[..., 0] * si + pairs[..., 1] * co], -1).reshape(m, cols)
        assert_exact(got, torch.cat([rotated, v[:, cols:]], 1).to(dtype))


# int8 weights or not, groups of 16 rows, column tiles of 16 of a workgroup
NARROW_STREAMS = [
    (False, 1, 1, 5, 4090, 1032), (False, 1, 2, 16, 8186, 1544), (False, 2, 1, 17, 4090, 1544), (False, 2, 2, 32, 8190, 1032), (False, 3, 1, 33, 4090, 1288),
    (False, 3, 2, 48, 6144, 4096), (False, 3, 2, 47, 8190, 1288), (False, 4, 1, 64, 4090, 1288), (False, 4, 2, 49, 8190, 1288),
    (True, 1, 1, 3, 4090, 1040), (True, 1, 2, 16, 8190, 2064), (True, 1, 3, 12, 12280, 2064), (True, 2, 1, 17, 4090, 1040), (True, 2, 2, 32, 8190, 2064),
    (True, 3, 1, 33, 4090, 1040), (True, 3, 2, 48, 6144, 4096), (True, 3, 2, 47, 8190, 2064), (True, 4, 1, 64, 4090, 1040), (True, 4, 2, 49, 8190, 2064),
    (False, 1, 1, 6, 4030, 1152), (False, 1, 2, 10, 8190, 1152), (False, 2, 1, 20, 4030, 1152), (False, 2, 2, 32, 8190, 1152), (False, 3, 1, 34, 4030, 1152),
    (False, 3, 2, 48, 6144, 4096), (False, 4, 1, 64, 4030, 1152), (False, 4, 2, 50, 8190, 1152),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("int8,groups,tiles,m,n,k", NARROW_STREAMS)
def test_every_form_of_the_narrow_streams_exact(ops, dev, pkg, dtype, int8, groups, tiles, m, n, k):
    """Every form of the kernel that streams few columns for each compute unit, with a last stage of K that is not whole: plain, with
    a bias, with an addend and written over it; rotated where K is a multiple of 128, either way, with tables of either type, of a row for each
    and of half as many; int8 weights with scales and biases in fp32 and in 16 bits. Sums of small whole numbers, which fp32 holds
    exactly in any order, rounded once. That the forms are these is checked without a GPU, in the build's checks."""
    gen = torch.Generator(dev).manual_seed(83)
    whole = lambda *s, scale=1.0: torch.randint(-3, 4, s, generator=gen, device=dev).to(dtype) * scale
    x, b = whole(m, k), whole(n)
    with own_context(ops, pkg) as ctx:
        if int8:
            w = torch.randint(-127, 128, (n, k), generator=gen, device=dev, dtype=torch.int8)
            scale = 2.0 ** torch.randint(-12, -8, (n,), generator=gen, device=dev)
            want = x.double() @ w.double().t() * scale.double()
            assert_exact(ops.weight_only_int8_linear(x, w, scale.half()), want.to(dtype))
            assert_exact(ops.weight_only_int8_linear(x, w, scale.float(), b), (want + b.double()).to(dtype))
            assert_exact(ops.weight_only_int8_linear(x, w, scale.float(), b.float()), (want + b.double()).to(dtype))
        else:
            w, c = whole(n, k, scale=2.0 ** -6), whole(m, n)
            want = x.double() @ w.double().t()
            assert_exact(ops.linear(x, w), want.to(dtype))
            assert_exact(ops.linear(x, w, b), (want + b.double()).to(dtype))
            assert_exact(ops.addmm(b, x, w.t(), beta=-1), (want - b.double()).to(dtype))
            total = (0.5 * c.double() + 2 * want).to(dtype)
            assert_exact(ops.addmm(c, x, w.t(), beta=0.5, alpha=2), total)
            assert_exact(ops.addmm(c, x, w.t(), beta=0.5, alpha=2, out=c), total)
            if k % 128 == 0:
                check_rotations(ops, gen, x, w, b, want, 64)
        assert ctx.workspace()[1] == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,slices", [(64, 512, 3968, 4), (33, 1024, 3456, 4), (49, 16, 3584, 4), (64, 512, 3328, 0), (64, 1032, 3968, 0),
                                          (48, 516, 3968, 0), (33, 512, 3936, 0), (32, 512, 3968, 0), (64, 512, 4096, 4)])
def test_k_slices_or_a_stream_where_k_is_a_little_less_than_4096(ops, dev, pkg, dtype, m, n, k, slices):
    """33 to 64 rows and at most 64 column tiles: K slices, which the workspace of their sums tells, from 3329 columns on; a row fewer, a
    column tile more, and sizes that the slices do not take stay with the kernel that streams the whole of K."""
    x, w = torch.randn(m, k, generator=g(1)).to(dtype), (torch.randn(n, k, generator=g(2)) / k**0.5).to(dtype)
    with own_context(ops, pkg) as ctx:
        got = ops.linear(x.to(dev), w.to(dev))
        assert ctx.workspace()[1] == slices * m * n * 4
    assert_half(got, x.double() @ w.double().t())


@pytest.mark.parametrize("table_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,heads,hd,vcols,k", [(3, 10, 128, 2 * 128, 4096), (16, 40, 64, 1000, 1032), (17, 6, 128, 256, 768), (5, 33, 64, 130 * 8, 2048 + 128), (40, 10, 128, 2 * 128, 1152), (64, 40, 64, 1000, 1536)])
def test_rotation_with_few_columns_for_a_compute_unit(ops, dev, table_dtype, m, heads, hd, vcols, k):
    # (K = 1032, no multiple of 128: the product and the rotation in launches of their own)
    n, cols = heads * hd + vcols, heads * hd
    x = torch.randn(m, k, generator=g(1)).bfloat16()
    w = (torch.randn(n, k, generator=g(2)) / k**0.5).bfloat16()
    b = torch.randn(n, generator=g(3)).bfloat16()
    angle = torch.rand(m, hd // 2, generator=g(4)) * 6
    cos, sin = angle.cos().to(table_dtype), angle.sin().to(table_dtype)
    for bias in (None, b):
        want = x.double() @ w.double().t() + (0 if bias is None else b.double())
        pairs = want[:, :cols].reshape(m, heads, hd // 2, 2)
        c, s = cos.double()[:, None], sin.double()[:, None]
        rotated = torch.stack([pairs[..., 0] * c - pairs[..., 1] * s, pairs[..., 0] * s + pairs[..., 1] * c], -1).reshape(m, cols)
        got = ops.linear_rotary(x.to(dev), w.to(dev), cos.to(dev), sin.to(dev), cols, hd, bias=None if bias is None else b.to(dev))
        assert_half(got, torch.cat([rotated, want[:, cols:]], 1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(65, 512, 1024), (128, 4096, 1024), (97, 11008, 1088), (704, 1536, 1152), (257, 11008, 1088), (257, 14336, 4096), (257, 22016, 4096),
                                   (704, 6144, 1088), (704, 8192, 4096), (203, 22016, 4096), (300, 3072, 1088), (451, 1040, 1024), (600, 2560, 1216)])
def test_rectangles_cut_to_the_chip(ops, dev, dtype, m, n, k):
    # the kernel of 65 to 704 rows whose rectangles are cut to the chip, on drawn numbers: ragged last rows and column tiles,
    # 16 stages of K and more; rows lie in a wider matrix of NaNs (every tile of it: the test below)
    wide = torch.full((m, k + 24), float("nan"), dtype=dtype)
    wide[:, :k] = torch.randn(m, k, generator=g(1)).to(dtype)
    x, xd = wide[:, :k], wide.to(dev)[:, :k]
    w = (torch.randn(n, k, generator=g(2)) / k**0.5).to(dtype)
    c, b = torch.randn(m, n, generator=g(3)).to(dtype), torch.randn(n, generator=g(4)).to(dtype)
    want = (x.float() @ w.float().t()).double()
    assert_half(ops.linear(xd, w.to(dev)), want)
    assert_half(ops.linear(xd, w.to(dev), b.to(dev)), want + b.double())
    assert_half(ops.addmm(c.to(dev), xd, w.to(dev).t(), beta=0.5, alpha=2.0), 0.5 * c.double() + 2 * want)
    if n % 64 == 0:
        blocks = want.view(m, n // 64, 2, 32)
        assert_half(ops.linear_silu_mul(xd, w.to(dev)), (torch.nn.functional.silu(blocks[:, :, 0]) * blocks[:, :, 1]).reshape(m, n // 2))
    for table_dtype in (dtype, torch.float32):
        hd, cols = 64, n * 2 // 3 // 64 * 64
        angle = torch.rand(m, hd // 2, generator=g(5)) * 6
        cos, sin = angle.cos().to(table_dtype), angle.sin().to(table_dtype)
        pairs = (want + b.double())[:, :cols].reshape(m, cols // hd, hd // 2, 2)
        co, si = cos.double()[:, None], sin.double()[:, None]
        rotated = torch.stack([pairs[..., 0] * co - pairs[..., 1] * si, pairs[..., 0] * si + pairs[..., 1] * co], -1).reshape(m, cols)
        got = ops.linear_rotary(xd, w.to(dev), cos.to(dev), sin.to(dev), cols, hd, bias=b.to(dev))
        assert_half(got, torch.cat([rotated, (want + b.double())[:, cols:]], 1))


# (TM, TN): an output tile is 32 TM rows by 32 TN columns. The last entry: the other form would take workspace.
RECTANGLES = [
    (4, 1, "gated", 70, 2944, 1280, True), (4, 1, "plain", 67, 144, 1088, True), (4, 1, "rotated", 66, 144, 1024, True),
    (4, 2, "gated", 114, 4160, 1024, True), (4, 2, "plain", 118, 4192, 1024, True), (4, 2, "rotated", 116, 4304, 1024, True),
    (4, 3, "gated", 103, 8576, 1024, True), (4, 3, "plain", 97, 8576, 1024, True), (4, 3, "rotated", 102, 8352, 1024, True),
    (4, 4, "gated", 110, 32576, 3904, False), (4, 4, "plain", 79, 32736, 6592, False), (4, 4, "rotated", 80, 31296, 10240, False),
    (4, 6, "gated", 147, 16640, 1024, False), (4, 6, "plain", 146, 17024, 1152, False), (4, 6, "rotated", 152, 16592, 1856, False),
    (5, 1, "gated", 257, 3328, 2624, True), (5, 1, "plain", 529, 1648, 1024, True), (5, 1, "rotated", 514, 1680, 1024, True),
    (5, 2, "gated", 640, 3520, 3520, False), (5, 2, "plain", 130, 16352, 9216, True), (5, 2, "rotated", 284, 6928, 5632, True),
    (5, 3, "gated", 131, 16512, 1024, False), (5, 3, "plain", 133, 16544, 1088, False), (5, 3, "rotated", 134, 22688, 3712, True),
    (5, 4, "gated", 129, 24960, 3840, True), (5, 4, "plain", 131, 25888, 3584, True), (5, 4, "rotated", 130, 30240, 3840, True),
    (5, 6, "gated", 257, 18304, 1024, False), (5, 6, "plain", 264, 18576, 1408, False), (5, 6, "rotated", 258, 17776, 10752, True),
    (6, 1, "plain", 481, 2704, 1024, True), (6, 1, "rotated", 482, 2704, 1024, True), (6, 2, "gated", 340, 6720, 5952, True),
    (6, 2, "plain", 383, 8080, 8704, False), (6, 3, "gated", 641, 5632, 3712, True), (6, 3, "plain", 168, 22624, 3584, True),
    (6, 3, "rotated", 168, 23968, 4480, True), (6, 4, "gated", 163, 26240, 3584, True), (6, 4, "plain", 162, 26944, 3840, True),
    (6, 4, "rotated", 166, 31888, 4096, True), (7, 1, "plain", 577, 2704, 1024, True), (7, 1, "rotated", 578, 2704, 1024, True),
    (7, 2, "gated", 650, 5440, 1088, False), (7, 2, "plain", 641, 5392, 3840, True), (7, 2, "rotated", 642, 5392, 1408, False),
    (7, 3, "gated", 583, 6592, 1024, False), (7, 3, "plain", 660, 7088, 3328, True), (7, 3, "rotated", 204, 24400, 6400, True),
    (7, 4, "gated", 199, 28160, 3840, True), (7, 4, "plain", 199, 29472, 3968, True), (7, 4, "rotated", 200, 31440, 4736, True),
    (8, 2, "gated", 697, 5440, 1216, False), (8, 2, "plain", 673, 5408, 3840, True), (8, 2, "rotated", 674, 5392, 1536, False),
    (8, 3, "gated", 701, 7616, 3328, True), (8, 3, "plain", 673, 7568, 3328, True), (8, 3, "rotated", 686, 6592, 2944, False),
    (8, 4, "gated", 230, 28992, 3968, True), (8, 4, "plain", 226, 31328, 4096, True), (8, 4, "rotated", 236, 31936, 8064, True),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tm,tn,form,m,n,k,told", RECTANGLES)
def test_every_form_of_the_rectangles_exact(ops, dev, pkg, dtype, tm, tn, form, m, n, k, told):
    """Every tile of the kernel whose rectangles are cut to the chip: plain, with a bias, with an addend and written over it; gated; rotated either
    way, with tables of either type, of a row for each and of half as many. Sums of small whole numbers, which fp32 holds exactly in
    any order, rounded once (but for the gate). That the cuts are these is checked without a GPU, in the build's checks."""
    gen = torch.Generator(dev).manual_seed(82)
    whole = lambda *s, scale=1.0: torch.randint(-3, 4, s, generator=gen, device=dev).to(dtype) * scale
    x, w = whole(m, k), whole(n, k, scale=2.0 ** -6)
    want = torch.cat([x.double() @ part.double().t() for part in w.split(4096)], 1)
    with own_context(ops, pkg) as ctx:
        if form == "plain":
            b, c = whole(n), whole(m, n)
            assert_exact(ops.linear(x, w), want.to(dtype))
            assert_exact(ops.linear(x, w, b), (want + b.double()).to(dtype))
            assert_exact(ops.addmm(b, x, w.t(), beta=-1), (want - b.double()).to(dtype))
            total = (0.5 * c.double() + 2 * want).to(dtype)
            assert_exact(ops.addmm(c, x, w.t(), beta=0.5, alpha=2), total)
            assert_exact(ops.addmm(c, x, w.t(), beta=0.5, alpha=2, out=c), total)
        elif form == "gated":
            blocks = want.view(m, n // 64, 2, 32)
            assert_half(ops.linear_silu_mul(x, w), (torch.nn.functional.silu(blocks[:, :, 0]) * blocks[:, :, 1]).reshape(m, n // 2))
        else:
            check_rotations(ops, gen, x, w, whole(n), want, 8 if n < 512 else 64)
        assert not told or ctx.workspace()[1] == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("form,m,n,k,slices", [("gated", 111, 448, 3072, 12), ("rotated", 111, 448, 3072, 12), ("gated", 362, 832, 4608, 12), ("rotated", 416, 2368, 3840, 3),
                                               ("gated", 300, 3072, 1088, 0), ("rotated", 300, 3072, 1088, 0), ("gated", 65, 5632, 1024, 0)])
def test_gate_and_rotation_in_a_rectangle_or_behind_k_slices(ops, dev, pkg, dtype, form, m, n, k, slices):
    """What a gate or a rotation in a launch of its own costs decides between rectangles, which take no workspace, and K slices, whose
    sums (and the two halves before the gate) lie in it."""
    x, w = torch.randn(m, k, generator=g(1)).to(dtype), (torch.randn(n, k, generator=g(2)) / k**0.5).to(dtype)
    want = x.double() @ w.double().t()
    with own_context(ops, pkg) as ctx:
        if form == "gated":
            got = ops.linear_silu_mul(x.to(dev), w.to(dev))
            blocks = want.view(m, n // 64, 2, 32)
            want = (torch.nn.functional.silu(blocks[:, :, 0]) * blocks[:, :, 1]).reshape(m, n // 2)
        else:
            cols = n * 2 // 3 // 64 * 64
            angle = torch.rand(m, 32, generator=g(3)) * 6
            got = ops.linear_rotary(x.to(dev), w.to(dev), angle.cos().to(dev), angle.sin().to(dev), cols, 64)
            pairs, co, si = want[:, :cols].reshape(m, cols // 64, 32, 2), angle.double().cos()[:, None], angle.double().sin()[:, None]
            rotated = torch.stack([pairs[..., 0] * co - pairs[..., 1] * si, pairs[..., 0] * si + pairs[..., 1] * co], -1).reshape(m, cols)
            terms = torch.stack([(pairs[..., 0] * co).abs() + (pairs[..., 1] * si).abs(), (pairs[..., 0] * si).abs() + (pairs[..., 1] * co).abs()], -1).reshape(m, cols)
            want = torch.cat([rotated, want[:, cols:]], 1)
        assert ctx.workspace()[1] == slices * m * n * 4 + (m * n * 2 if slices and form == "gated" else 0)
    if form == "gated":
        assert_half(got, want)
    else:  # each term of a rotation behind slices is rounded to 16 bits before, the result after it: half a last place; fp32 sums
        half = 1.01 * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
        bound = half * want.abs() + 1e-4
        bound[:, :cols] += half * terms
        assert ((got.cpu().double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,f,k", [(4096, 3584, 256), (3700, 4000 - 32, 192), (96, 64, 80), (1, 32, 8),
                                   (5, 2048, 256), (33, 5536, 384), (48, 16384, 128), (64, 11008, 640), (20, 8224, 256)])
def test_linear_silu_mul(ops, dev, dtype, m, f, k):
    """silu(x Wg^T) * (x Wu^T) from the interleaved weight: the single-launch path (at least 144 tiles, K a
    multiple of 64, 16-bit dtypes) and the two-pass path, against the reference's four-op form in fp32. The last five
    cases (at most 64 rows, K a multiple of 128, at least 4096 stacked columns, 16-bit dtypes) take the decode-sized
    kernel with the gate applied to its sums: one to four row groups, workgroups of 64 and of 128 columns, a last
    workgroup with a single block of 64, K of one to five stages."""
    x = torch.randn(m, k, generator=g(60)).to(dtype)
    wg = (torch.randn(f, k, generator=g(61)) * 0.08).to(dtype)
    wu = (torch.randn(f, k, generator=g(62)) * 0.08).to(dtype)
    gate, up = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    want = torch.nn.functional.silu(gate) * up
    w = ops.interleave_gate_up(wg.to(dev), wu.to(dev))
    assert_exact(w[32:64], wu[:32])  # block 0: 32 gate rows, then 32 up rows
    got = ops.linear_silu_mul(x.to(dev), w)
    (assert_fp32 if dtype == torch.float32 else assert_half)(got, want)
    if m >= 96:  # batch dims and a strided destination
        x3 = x[:96].reshape(2, 48, k)
        dst = torch.zeros(2, 48, 2 * f, dtype=dtype, device=dev)
        ops.linear_silu_mul(x3.to(dev), w, out=dst[..., :f])
        (assert_fp32 if dtype == torch.float32 else assert_half)(dst[..., :f], want[:96].reshape(2, 48, f))
        assert_exact(dst[..., f:], torch.zeros(2, 48, f, dtype=dtype))
    elif f >= 2048:  # the decode-sized kernel into a strided destination
        dst = torch.zeros(m, 2 * f, dtype=dtype, device=dev)
        ops.linear_silu_mul(x.to(dev), w, out=dst[:, :f])
        assert_exact(dst[:, :f], got.cpu())
        assert_exact(dst[:, f:], torch.zeros(m, f, dtype=dtype))


# ------------------------------------------------------------------ prefill attention
@pytest.mark.parametrize("dtype,table_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("m,heads,hd,vcols,k,interleaved,conj,bias", [
    (2304, 16, 128, 2048, 256, True, False, False),   # 9 x 16 tiles: one launch; q and k rotated, v through
    (2400, 57, 64, 0, 192, True, True, True),         # ragged rows and columns, all columns rotated, negative angle, bias
    (2304, 16, 128, 2048, 256, False, False, False),  # half-split pairs: projection + rotary kernel
    (40, 4, 64, 128, 128, True, False, True),         # small: projection + rotary kernel
    (64, 64, 128, 4096, 256, True, False, False),     # decode-sized, 12288 columns: the LDS-staged kernel rotates its sums (48 columns per workgroup)
    (7, 45, 128, 640, 384, True, True, True),         # one row group, 25 columns per workgroup made 26, negative angle, bias
    (33, 96, 64, 22016 - 6144, 128, True, False, True),  # 22016 columns: workgroups of 86 columns, three row groups
])
def test_linear_rotary(ops, dev, dtype, table_dtype, m, heads, hd, vcols, k, interleaved, conj, bias):
    """The stacked projection with the rotary embedding in its epilogue against the oracle's projection followed by
    the oracle's rotation (half-split: ext_ops.py:24-33; interleaved: model.py:58-69), and against this backend's
    own two separate ops."""
    rot = heads * hd
    n = rot + vcols
    x = torch.randn(m, k, generator=g(70)).to(dtype)
    w = (torch.randn(n, k, generator=g(71)) * 0.05).to(dtype)
    b = torch.randn(n, generator=g(72)).to(dtype) if bias else None
    cos, sin = oracle.precompute_freqs(hd, m)
    cos_t, sin_t = cos.to(table_dtype), sin.to(table_dtype)
    y = x.float() @ w.float().t() + (b.float() if bias else 0)
    sgn = -1.0 if conj else 1.0
    yr = y[:, :rot].reshape(m, heads, hd)
    want_rot = (oracle.rotary_emb_interleaved if interleaved else oracle.rotary_emb)(yr, cos_t.float(), sgn * sin_t.float())
    want = torch.cat([want_rot.reshape(m, rot), y[:, rot:]], dim=1)
    db = b.to(dev) if bias else None
    got = ops.linear_rotary(x.to(dev), w.to(dev), cos_t.to(dev), sin_t.to(dev), rot, hd, db, conj=conj, interleaved=interleaved)
    assert_half(got, want)
    # tables of any shape that holds [t, head_dim / 2] values are read the same way by both forms
    flat = ops.linear_rotary(x.to(dev), w.to(dev), cos_t.reshape(-1).to(dev), sin_t.reshape(-1).to(dev), rot, hd, db, conj=conj,
                             interleaved=interleaved)
    assert_exact(flat, got.cpu())
    # this backend's separate ops (one rounding more between them)
    sep = ops.linear(x.to(dev), w.to(dev), db)
    q = sep[:, :rot].view(m, heads, hd)
    ops.rotary_emb(q, cos_t.to(dev), sin_t.to(dev), conj=conj, interleaved=interleaved, out=q)
    assert_half(got, sep.float().cpu(), rel=2e-2, abs_=3e-2)   # two device results, each with its own roundings (not an oracle comparison)


def test_rotary_row_permutation_keeps_attention_scores(ops, dev):
    """A half-split checkpoint through the interleaved single-launch form: with the q / k weight rows of every head
    permuted (row 2i <- row i, row 2i + 1 <- row i + d / 2) the rotated q and k are the same permutation of the
    half-split results, so every q . k is unchanged."""
    m, heads, hd, k = 2304, 16, 128, 256
    x = torch.randn(m, k, generator=g(73)).bfloat16().to(dev)
    w = (torch.randn(2 * heads * hd, k, generator=g(74)) * 0.05).bfloat16()
    cos, sin = oracle.precompute_freqs(hd, m)
    cos, sin = cos.bfloat16().to(dev), sin.bfloat16().to(dev)
    half_split = ops.linear_rotary(x, w.to(dev), cos, sin, 2 * heads * hd, hd, interleaved=False)
    wp = ops.interleave_rotary_rows(w, hd).to(dev)
    inter = ops.linear_rotary(x, wp, cos, sin, 2 * heads * hd, hd, interleaved=True)
    perm = inter.view(m, 2 * heads, hd // 2, 2).transpose(2, 3).reshape(m, 2 * heads * hd)  # back to half-split order
    assert_half(perm, half_split.float().cpu(), rel=2e-2, abs_=3e-2)   # two device results (see above)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float16, 128), (torch.bfloat16, 64),
                                     (torch.float32, 64), (torch.float32, 40)])
def test_context_attention(ops, dev, dtype, d):
    lens = [200, 1, 130, 64, 333]
    starts, total = [], 0
    for n in lens:
        starts.append(total)
        total += n
    heads = 4
    q = torch.randn(total, heads, d, generator=g(20)).to(dtype)
    k = torch.randn(total, heads, d, generator=g(21)).to(dtype)
    v = torch.randn(total, heads, d, generator=g(22)).to(dtype)
    st, ln = torch.tensor(starts, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    want = oracle.context_attention(q.float(), k.float(), v.float(), st, ln)
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), st.to(dev), ln.to(dev), max(lens))
    (assert_fp32 if dtype == torch.float32 else assert_half)(got, want)
    # first row of every sequence equals its V row; int64 index tensors give the same result
    for s in starts:
        assert_close(got[s], v[s])
    got64 = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), st.long().to(dev), ln.long().to(dev), max(lens))
    assert_exact(got64, got.cpu())


def test_context_attention_gqa_and_strided_inputs(ops, dev):
    total, heads, kvh, d = 257, 8, 2, 128
    qkv = torch.randn(total, (heads + 2 * kvh) * d, generator=g(23)).bfloat16()
    q, k, v = qkv.split([heads * d, kvh * d, kvh * d], -1)
    q, k, v = q.reshape(total, heads, d), k.reshape(total, kvh, d), v.reshape(total, kvh, d)
    st, ln = torch.tensor([0, 100]), torch.tensor([100, 157])
    want = oracle.context_attention(q.float(), k.float(), v.float(), st, ln)
    dq = qkv.to(dev).split([heads * d, kvh * d, kvh * d], -1)
    got = ops.context_attention(dq[0].reshape(total, heads, d), dq[1].reshape(total, kvh, d), dq[2].reshape(total, kvh, d),
                                st.to(dev), ln.to(dev), 157)
    assert_half(got, want)


@pytest.mark.parametrize("heads,kvh,d,lens", [(8, 8, 64, [128, 128]), (8, 2, 128, [1, 15, 16, 17, 33]), (4, 4, 64, [64, 65, 200]), (2, 1, 128, [130])])
def test_context_attention_fp32_on_the_matrix_cores(ops, dev, heads, kvh, d, lens):
    """16 queries per workgroup, key tiles dealt over its four waves: fewer key tiles than waves, one and several rounds of
    them, lengths around a tile's edge, shared K/V heads, and q, k, v as slices of one projection."""
    total = sum(lens)
    qkv = torch.randn(total, heads + 2 * kvh, d, generator=g(43))
    starts = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32)
    ln = torch.tensor(lens, dtype=torch.int32)
    dq = qkv.to(dev)
    q, k, v = qkv[:, :heads], qkv[:, heads:heads + kvh], qkv[:, heads + kvh:]
    got = ops.context_attention(dq[:, :heads], dq[:, heads:heads + kvh], dq[:, heads + kvh:], starts.to(dev), ln.to(dev), max(lens),
                                out=torch.empty(total, heads, d, device=dev))
    want = torch.empty(total, heads, d, dtype=torch.float64)
    for s, n in zip(starts.tolist(), lens):
        kk = k[s:s + n].double().repeat_interleave(heads // kvh, 1)
        vv = v[s:s + n].double().repeat_interleave(heads // kvh, 1)
        sc = torch.einsum("qhd,khd->hqk", q[s:s + n].double(), kk) / d ** 0.5
        sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), float("-inf"))
        want[s:s + n] = torch.einsum("hqk,khd->qhd", torch.softmax(sc, -1), vv)
    assert_fp32(got, want)


@pytest.mark.parametrize("d,n", [(64, 44), (128, 100)])
def test_context_attention_fp32_keeps_later_keys_and_overflowed_scores_out(ops, dev, d, n):
    """A V row that is infinite or NaN reaches the queries from its own position on and no earlier one, and a key whose score
    is -inf has weight 0 even if it is the first that a wave meets."""
    q, k, v = (torch.randn(n, 2, d, generator=g(44)) for _ in range(3))
    at = n - 9
    v[at, 0, 3], v[at, 1, 5] = float("inf"), float("nan")
    q[:, :, 0] = q[:, :, 0].abs() + 1
    k[17:32, :, 0] = float("-inf")
    k[16, :, 0] = float("-inf")
    starts, ln = torch.zeros(1, dtype=torch.int32, device=dev), torch.full((1,), n, dtype=torch.int32, device=dev)
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), starts, ln, n, out=torch.empty(n, 2, d, device=dev)).cpu()
    clean = v.clone()
    clean[at] = 0
    sc = torch.einsum("qhd,khd->hqk", q.double(), k.double()) / d ** 0.5
    sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(sc, -1)
    want = torch.einsum("hqk,khd->qhd", p, clean.double()) + torch.einsum("hq,hd->qhd", p[:, :, at], v[at].double().nan_to_num(0, 0))
    assert_fp32(torch.where(got.isfinite(), got, want.float()), want)
    assert got[:at].isfinite().all() and (got[at:, 0, 3] == float("inf")).all() and got[at:, 1, 5].isnan().all()
    assert (~got.isfinite()).sum() == 2 * (n - at)


def test_context_attention_uniform_keys_give_running_mean_at_length_2048(ops, dev):
    # property that holds at the full sequence length: identical keys -> uniform weights
    n, heads, d = 2048, 2, 128
    q = torch.randn(n, heads, d, generator=g(24)).bfloat16()
    k = torch.randn(1, heads, d, generator=g(25)).bfloat16().expand(n, -1, -1).contiguous()
    v = torch.randn(n, heads, d, generator=g(26)).bfloat16()
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), torch.tensor([0], dtype=torch.int32).to(dev),
                                torch.tensor([n], dtype=torch.int32).to(dev), n)
    run_mean = torch.cumsum(v.float(), 0) / torch.arange(1, n + 1).view(-1, 1, 1)
    assert_half(got, run_mean)

@pytest.mark.parametrize("heads,kvh,lens", [(8, 2, [1000, 2048, 517]), (16, 16, [1300, 90, 700]), (4, 4, [900, 1100]),
                                            (4, 2, [600, 1025, 130])])
def test_context_attention_long_ragged_batch_paired_blocks(ops, dev, heads, kvh, lens):
    """Ragged sequences up to 2048 tokens: exercises the heavy + light query-block pairing (odd and even block counts,
    sequences shorter than the longest one) and the three ways a workgroup finds its (sequence, head): a head count
    that is a multiple of 8 (one or two heads of every sequence per XCD), heads x sequences a multiple of 8, neither."""
    d = 128
    starts = [sum(lens[:i]) for i in range(len(lens))]
    total = sum(lens)
    q = torch.randn(total, heads, d, generator=g(27)).bfloat16()
    k = torch.randn(total, kvh, d, generator=g(28)).bfloat16()
    v = torch.randn(total, kvh, d, generator=g(29)).bfloat16()
    st, ln = torch.tensor(starts, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    want = oracle.context_attention(q.float(), k.float(), v.float(), st, ln)
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), st.to(dev), ln.to(dev), max(lens))
    assert_half(got, want)


@pytest.mark.parametrize("heads,kvh,d,dtype,lens", [(32, 32, 128, torch.bfloat16, [512]), (8, 2, 128, torch.bfloat16, [1000]),
                                                    (16, 4, 64, torch.float16, [700, 129, 5]), (8, 8, 128, torch.float16, [257, 256, 255, 1]),
                                                    (28, 4, 128, torch.bfloat16, [600]), (6, 3, 64, torch.bfloat16, [300, 1025])])
def test_context_attention_one_query_block_per_workgroup(ops, dev, heads, kvh, d, dtype, lens):
    """Launches too small for the paired schedule to fill the chip evenly: every 128-query block is a workgroup of its
    own, heaviest first (a single short prompt; a few ragged sequences; block counts of 4, 8, 6 and 3)."""
    starts = [sum(lens[:i]) for i in range(len(lens))]
    total = sum(lens)
    q = torch.randn(total, heads, d, generator=g(40)).to(dtype)
    k = torch.randn(total, kvh, d, generator=g(41)).to(dtype)
    v = torch.randn(total, kvh, d, generator=g(42)).to(dtype)
    st, ln = torch.tensor(starts, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    want = oracle.context_attention(q.float(), k.float(), v.float(), st, ln)
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), st.to(dev), ln.to(dev), max(lens))
    assert_half(got, want)
    assert_exact(got[starts[-1]].cpu(), v[starts[-1]].repeat_interleave(heads // kvh, dim=0))   # a sequence's first query sees one key


@pytest.mark.parametrize("heads,kvh,d,dtype,lens", [(8, 8, 96, torch.bfloat16, [300, 1, 130, 64, 333]), (8, 2, 80, torch.float16, [700, 129]),
                                                    (4, 4, 40, torch.bfloat16, [200, 513]), (4, 2, 256, torch.bfloat16, [260, 900, 64]),
                                                    (16, 16, 256, torch.float16, [1300, 2048, 517]), (8, 4, 192, torch.bfloat16, [1000]),
                                                    (32, 8, 112, torch.bfloat16, [2048, 2048])])
def test_context_attention_other_head_sizes_on_the_matrix_pipe(ops, dev, heads, kvh, d, dtype, lens):
    """Head sizes that are a multiple of 8 other than 64 and 128 take the tile layout of the next of 64 / 128 / 256, the
    pieces of a row past the head size read as zeros and never stored: sizes under 64, between 64 and 128, 256 itself
    and one between 128 and 256; both schedules (pairs of query blocks and a block per workgroup), grouped K/V heads,
    ragged batches. The neighbours of every row (the next head, the next token) hold other values, so a piece read past
    the head size would show."""
    starts = [sum(lens[:i]) for i in range(len(lens))]
    total = sum(lens)
    q = torch.randn(total, heads, d, generator=g(43)).to(dtype)
    k = torch.randn(total, kvh, d, generator=g(44)).to(dtype)
    v = torch.randn(total, kvh, d, generator=g(45)).to(dtype)
    st, ln = torch.tensor(starts, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    want = oracle.context_attention(q.float(), k.float(), v.float(), st, ln)
    out = torch.full((total, heads, d), 7.0, dtype=dtype, device=dev)
    got = ops.context_attention(q.to(dev), k.to(dev), v.to(dev), st.to(dev), ln.to(dev), max(lens), out=out)
    assert_half(got, want)
    assert_exact(got[starts[-1]].cpu(), v[starts[-1]].repeat_interleave(heads // kvh, dim=0))   # a sequence's first query sees one key


# ------------------------------------------------------------------ decode attention
@pytest.mark.parametrize("dtype,d,idt", [(torch.bfloat16, 128, torch.int32), (torch.float16, 64, torch.int64),
                                          (torch.float32, 64, torch.int32), (torch.bfloat16, 256, torch.int32)])
def test_token_attention_fused_and_two_call(ops, dev, pkg, dtype, d, idt):
    w = pkg.workloads.paged_decode(seed=1, batch=7, heads=4, head_dim=d, min_len=1, max_len=1300, pool_slots=8192,
                                   dtype=dtype, index_dtype=idt)
    kp, vp = w["k_pool"].clone(), w["v_pool"].clone()
    oracle.dest_index_copy_kv(kp, w["k_new"], w["dest_loc"])
    oracle.dest_index_copy_kv(vp, w["v_new"], w["dest_loc"])
    dk, dv = w["k_pool"].to(dev), w["v_pool"].to(dev)
    ops.dest_index_copy_kv(w["k_new"].to(dev), w["dest_loc"].to(dev), dk)
    ops.dest_index_copy_kv(w["v_new"].to(dev), w["dest_loc"].to(dev), dv)
    assert_exact(dk, kp)
    assert_exact(dv, vp)
    want = oracle.token_attention(w["q"].float(), kp.float(), vp.float(), w["b_loc"], w["b_seq_len"], w["max_input_len"])
    args = (w["b_loc"].to(dev), w["b_start_loc"].to(dev), w["b_seq_len"].to(dev), w["max_input_len"])
    got = ops.token_decode_attention(w["q"].to(dev), dk, dv, *args)
    chk = assert_fp32 if dtype == torch.float32 else assert_half
    chk(got, want)
    # the DIOPI two-call form: logits, then softmax . V
    att = torch.zeros(4, w["total_tokens"], dtype=torch.float32, device=dev)
    ops.token_attention(w["q"].to(dev), dk, att, *args)
    want_att = oracle.token_logits(w["q"], kp, w["b_loc"], w["b_start_loc"], w["b_seq_len"], w["max_input_len"], w["total_tokens"])
    assert_fp32(att, want_att, rel=1e-5)       # fp32 logits from either dtype: only the order of the d additions differs
    out2 = torch.empty_like(got)
    ops.token_softmax_reducev(att, dv, out2, *args)
    chk(out2, want)


@pytest.mark.parametrize("dtype,d,kvh,rep", [(torch.bfloat16, 80, 4, 2), (torch.float16, 32, 2, 1), (torch.float32, 96, 1, 4),
                                             (torch.bfloat16, 40, 8, 1), (torch.float32, 300, 2, 1)])
def test_token_attention_any_head_size(ops, dev, pkg, dtype, d, kvh, rep):
    """Head rows that are not 128, 256 or 512 bytes long: whole 16-byte pieces up to 512 bytes ride on the lanes of the
    next of those sizes with the lanes past the row's end masked (160, 64, 384 and 80 bytes here), longer rows take the
    generic kernels (1200 bytes): the fused form, the entry point that allocates nothing and the two-call form against
    the oracle (ext_ops.py:100-133), with a sequence of one token and one longer than a block of 256."""
    heads = kvh * rep
    w = pkg.workloads.paged_decode(seed=11, batch=5, heads=kvh, head_dim=d, min_len=1, max_len=700, pool_slots=4096, dtype=dtype)
    w["b_seq_len"][0] = 1                                    # b_loc is right-aligned: the last column is the token
    gq = torch.Generator().manual_seed(12)
    q = torch.randn(5, heads, d, generator=gq).to(dtype)
    want = oracle.token_attention(q.float(), w["k_pool"].float(), w["v_pool"].float(), w["b_loc"], w["b_seq_len"], w["max_input_len"])
    dk, dv = w["k_pool"].to(dev), w["v_pool"].to(dev)
    args = (w["b_loc"].to(dev), w["b_start_loc"].to(dev), w["b_seq_len"].to(dev), w["max_input_len"])
    chk = assert_fp32 if dtype == torch.float32 else assert_half
    got = ops.token_decode_attention(q.to(dev), dk, dv, *args)
    chk(got, want)
    assert_exact(ops.token_decode_attention(q.to(dev), dk, dv, *args, no_alloc=True), got.cpu())
    att = torch.zeros(heads, w["total_tokens"], dtype=torch.float32, device=dev)
    ops.token_attention(q.to(dev), dk, att, *args)
    want_att = oracle.token_logits(q, w["k_pool"], w["b_loc"], w["b_start_loc"], w["b_seq_len"], w["max_input_len"], w["total_tokens"])
    for b in range(5):                                       # only the columns of live tokens are defined
        s0, n = int(w["b_start_loc"][b]), int(w["b_seq_len"][b])
        assert_fp32(att[:, s0:s0 + n], want_att[:, s0:s0 + n], rel=1e-5)
    out2 = torch.empty_like(got)
    ops.token_softmax_reducev(att, dv, out2, *args)
    chk(out2, want)


@pytest.mark.parametrize("dtype,d,heads,kvh", [(torch.bfloat16, 96, 8, 8), (torch.float16, 112, 12, 4), (torch.bfloat16, 192, 4, 2),
                                               (torch.bfloat16, 80, 5, 5)])
def test_token_attention_masked_head_rows_over_split_sequences(ops, dev, pkg, dtype, d, heads, kvh):
    """Head sizes between the powers of two at lengths that are split into chunks and merged, on a pool whose every slot
    is in use (the lanes past a row's end must not reach past the pool's last row): four heads of a token per wave
    load, four and two query heads per K/V head, and a head count that keeps a workgroup per head."""
    w = pkg.workloads.paged_decode(seed=21, batch=9, heads=kvh, head_dim=d, min_len=700, max_len=3000, pool_slots=15285, dtype=dtype)   # exactly the tokens drawn
    gq = torch.Generator().manual_seed(22)
    q = torch.randn(9, heads, d, generator=gq).to(dtype)
    want = oracle.token_attention(q.float(), w["k_pool"].float(), w["v_pool"].float(), w["b_loc"], w["b_seq_len"], w["max_input_len"])
    dk, dv = w["k_pool"].to(dev), w["v_pool"].to(dev)
    args = (w["b_loc"].to(dev), w["b_start_loc"].to(dev), w["b_seq_len"].to(dev), w["max_input_len"])
    got = ops.token_decode_attention(q.to(dev), dk, dv, *args)
    assert_half(got, want)
    assert_exact(ops.token_decode_attention(q.to(dev), dk, dv, *args, no_alloc=True), got.cpu())
    att = torch.zeros(heads, w["total_tokens"], dtype=torch.float32, device=dev)
    ops.token_attention(q.to(dev), dk, att, *args)
    out2 = torch.empty_like(got)
    ops.token_softmax_reducev(att, dv, out2, *args)
    assert_half(out2, want)


@pytest.mark.parametrize("heads,kvh", [(8, 2), (6, 3)])
def test_token_attention_len_one_and_gqa(ops, dev, heads, kvh):
    """Grouped-query decode: four query heads per K/V head (served from one read of its rows) and two."""
    slots, d = 64, 128
    kp = torch.randn(slots, kvh, d, generator=g(30)).bfloat16()
    vp = torch.randn(slots, kvh, d, generator=g(31)).bfloat16()
    q = torch.randn(3, heads, d, generator=g(32)).bfloat16()
    lens = torch.tensor([1, 5, 1], dtype=torch.int32)
    b_loc = torch.zeros(3, 5, dtype=torch.int32)
    b_loc[0, 4] = 17
    b_loc[1] = torch.tensor([3, 60, 9, 41, 22])
    b_loc[2, 4] = 63
    starts = torch.tensor([0, 1, 6], dtype=torch.int32)
    got = ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), b_loc.to(dev), starts.to(dev), lens.to(dev), 5)
    want = oracle.token_attention(q.float(), kp.float(), vp.float(), b_loc, lens, 5)
    assert_half(got, want)
    # a single cached token: the output is that token's V row for the mapped kv head
    assert_exact(got[0].cpu(), vp[17].repeat_interleave(heads // kvh, dim=0))
    assert_exact(got[2].cpu(), vp[63].repeat_interleave(heads // kvh, dim=0))


@pytest.mark.parametrize("heads,kvh,dtype,d,idt", [
    (32, 8, torch.bfloat16, 128, torch.int32),    # 16-bit rows so few: the matrix pipe, here four of its 16 columns in use
    (16, 8, torch.float16, 64, torch.int64),      # two, 128-byte rows
    (64, 8, torch.bfloat16, 128, torch.int32),    # eight
    (8, 1, torch.float32, 64, torch.int32),       # fp32 rows: the lanes; one K/V head for all, two workgroups of four heads
    (8, 2, torch.float16, 256, torch.int32),      # 512-byte rows
    (12, 4, torch.bfloat16, 128, torch.int32),    # three
    (28, 4, torch.bfloat16, 128, torch.int64),    # seven
    (10, 2, torch.float16, 128, torch.int32),     # five
])
def test_token_attention_grouped_query_layouts(ops, dev, heads, kvh, dtype, d, idt):
    """Fused and two-call decode attention with fewer K/V heads than query heads, over sequences of 1 to 1500 tokens
    (one to several chunks, ragged ends), against the oracle's repeat-interleaved K/V."""
    slots = 4096
    lens = [1, 1500, 777, 64, 513, 130, 1024]
    batch, width, total = len(lens), max(lens), sum(lens)
    kp = torch.randn(slots, kvh, d, generator=g(90)).to(dtype)
    vp = torch.randn(slots, kvh, d, generator=g(91)).to(dtype)
    q = torch.randn(batch, heads, d, generator=g(92)).to(dtype)
    b_loc = torch.zeros(batch, width, dtype=idt)
    for b, n in enumerate(lens):
        b_loc[b, width - n:] = torch.randint(0, slots, (n,), generator=g(93 + b)).to(idt)
    ln = torch.tensor(lens, dtype=idt)
    st = torch.zeros(batch, dtype=idt)
    st[1:] = torch.cumsum(ln, 0)[:-1]
    want = oracle.token_attention(q.float(), kp.float(), vp.float(), b_loc, ln, width)
    chk = assert_fp32 if dtype == torch.float32 else assert_half
    args = (b_loc.to(dev), st.to(dev), ln.to(dev), width)
    got = ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), *args)
    chk(got, want)
    att = torch.zeros(heads, total, dtype=torch.float32, device=dev)
    ops.token_attention(q.to(dev), kp.to(dev), att, *args)
    assert_fp32(att, oracle.token_logits(q, kp, b_loc, st, ln, width, total), rel=1e-5)
    out2 = torch.empty_like(got)
    ops.token_softmax_reducev(att, vp.to(dev), out2, *args)
    chk(out2, want)
    if dtype != torch.float32:   # scores kept in the 16-bit dtype between the two calls
        att16 = torch.zeros(heads, total, dtype=dtype, device=dev)
        ops.token_attention(q.to(dev), kp.to(dev), att16, *args)
        assert_half(att16, oracle.token_logits(q, kp, b_loc, st, ln, width, total))
        out3 = torch.empty_like(got)
        ops.token_softmax_reducev(att16, vp.to(dev), out3, *args)
        assert_half(out3, want, rel=3e-2, abs_=2e-2)   # softmax of scores rounded to 8 (11) bits


@pytest.mark.parametrize("heads,kvh,d,dtype", [
    (5, 5, 128, torch.bfloat16),     # a head count that is no multiple of four heads per wave load: the matrix pipe below 2048 pairs
    (8, 8, 64, torch.float16),       # few pairs of whole rows
    (16, 1, 128, torch.float16),     # all 16 columns of the products in use
    (17, 1, 128, torch.bfloat16),    # two workgroups of 9 and 8 heads
    (6, 2, 8, torch.float16),        # one 16-byte piece per row
    (4, 2, 200, torch.bfloat16),     # rows laid out for 512 bytes
    (2, 1, 256, torch.float16),
])
def test_token_attention_tiles_of_sixteen_tokens(ops, dev, heads, kvh, d, dtype):
    """Sequence lengths around the edges of a tile (16 tokens), of a wave's and of a workgroup's share, scores that grow by
    more than 2^8 along a sequence (the running maximum has to follow), and slots outside the pool, which are skipped."""
    lens = [1, 15, 16, 17, 63, 64, 65, 127, 129, 511, 513, 0]
    slots, width, total = 1500, 513, sum(lens)
    kp = torch.randn(slots, kvh, d, generator=g(60)).to(dtype)
    vp = torch.randn(slots, kvh, d, generator=g(61)).to(dtype)
    q = (3 * torch.randn(len(lens), heads, d, generator=g(62))).to(dtype)
    b_loc = torch.zeros(len(lens), width, dtype=torch.int32)
    for b, n in enumerate(lens):
        b_loc[b, width - n:] = torch.randperm(slots, generator=g(63 + b))[:n].to(torch.int32)
    kp[b_loc[9, width - 100:].long()] *= 6          # the last 100 tokens of the sequence of 511
    ln = torch.tensor(lens, dtype=torch.int32)
    st = torch.zeros(len(lens), dtype=torch.int32)
    st[1:] = torch.cumsum(ln, 0)[:-1]
    want = oracle.token_attention(q[:-1].float(), kp.float(), vp.float(), b_loc[:-1], ln[:-1], width)
    args = (b_loc.to(dev), st.to(dev), ln.to(dev), width)
    got = ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), *args)
    assert_half(got[:-1], want)
    assert_exact(got[-1].cpu(), torch.zeros(heads, d, dtype=dtype))
    assert_exact(ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), *args, no_alloc=True), got.cpu())
    att = torch.full((heads, total), float("nan"), dtype=torch.float32, device=dev)
    ops.token_attention(q.to(dev), kp.to(dev), att, *args)
    assert_fp32(att, oracle.token_logits(q, kp, b_loc, st, ln, width, total), rel=1e-5)
    out2 = torch.empty_like(got)
    ops.token_softmax_reducev(att, vp.to(dev), out2, *args)
    assert_half(out2[:-1], want)
    # the sequence of 65 tokens without every third one: as if it were the shorter sequence
    bad = b_loc.clone()
    bad[6, width - 65::3] = torch.tensor([-1, slots] * 11, dtype=torch.int32)
    kept = b_loc[6, width - 65:][torch.arange(65) % 3 != 0]
    short = oracle.token_attention(q[6:7].float(), kp.float(), vp.float(), kept[None], torch.tensor([len(kept)]), len(kept))
    got = ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), bad.to(dev), *args[1:])
    assert_half(got[6:7], short)


@pytest.mark.parametrize("heads,kvh,d", [(8, 2, 128), (8, 2, 200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_token_attention_values_that_are_not_finite(ops, dev, heads, kvh, d, dtype):
    """NaN in slot 0, which no sequence holds, changes nothing where slots outside the pool are skipped; an infinity in V
    stays an infinity in its column, in the last token of a partial tile too; a key whose score is -inf weighs nothing."""
    slots, width = 100, 37
    kp = torch.randn(slots, kvh, d, generator=g(75)).to(dtype)
    vp = torch.randn(slots, kvh, d, generator=g(76)).to(dtype)
    q = torch.randn(2, heads, d, generator=g(77)).abs().to(dtype)
    b_loc = torch.randperm(slots - 1, generator=g(78))[:2 * width].view(2, width).to(torch.int32) + 1
    b_loc[0, 3::5] = torch.tensor([-1, slots, -7, slots + 1, -1, slots, -1], dtype=torch.int32)
    kept = b_loc[0][(b_loc[0] >= 0) & (b_loc[0] < slots)].long()
    cut = b_loc[1, 5].long()                        # (every query component is positive: its scores are -inf)
    kp[0], vp[0] = float("nan"), float("nan")
    vp[b_loc[0, 36].long(), :, 3], vp[b_loc[0, 20].long(), :, 5], vp[b_loc[1, 0].long(), :, 0] = float("inf"), -float("inf"), float("inf")
    kp[cut, :, 0] = -float("inf")
    one = lambda loc, i: oracle.token_attention(q[i:i + 1].float(), kp.float(), vp.float(), loc[None].to(torch.int32), torch.tensor([len(loc)]), len(loc))
    want = torch.cat([one(kept, 0), one(b_loc[1][b_loc[1] != cut], 1)])
    ln, st = torch.tensor([width, width], dtype=torch.int32).to(dev), torch.tensor([0, width], dtype=torch.int32).to(dev)
    args = (b_loc.to(dev), st, ln, width)
    att = torch.empty(heads, 2 * width, dtype=torch.float32, device=dev)
    out2 = torch.empty(2, heads, d, dtype=dtype, device=dev)
    ops.token_attention(q.to(dev), kp.to(dev), att, *args)
    ops.token_softmax_reducev(att, vp.to(dev), out2, *args)
    finite = torch.isfinite(want)
    assert not finite[0, :, 3].any() and not finite[0, :, 5].any() and not finite[1, :, 0].any()
    for got in (ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), *args), out2):
        got = got.cpu()
        assert torch.equal(got[~finite].float(), want[~finite].float())
        assert_half(got[finite], want[finite])


@pytest.mark.parametrize("heads,kvh", [(4, 4), (8, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_token_attention_weights_are_held_in_full(ops, dev, heads, kvh, dtype):
    """What a probability holds beyond its rounding to 16 bits, and below the smallest 16-bit number, reaches the result. In
    twelve sequences three tokens, in different tiles, have values that cancel to about 2^-13 of their terms and the others
    have none; in the last one every 16th token weighs 4e7 times as much as those between but has no values. K picks the
    scores: q is 8 in its first element, d = 64."""
    d, n, batch = 64, 200, 13
    gen = g(79)
    score = -torch.randint(0, 64, (batch, n), generator=gen).float() / 64
    score[-1] = -17.5
    score[-1, ::16] = 0
    p = torch.exp(score.double()).view(batch, n, 1, 1)
    v = torch.zeros(batch, n, kvh, d, dtype=torch.float64)
    v[:, 20] = torch.randn(batch, kvh, d, generator=gen).to(dtype).double()
    v[:, 77] = (-v[:, 20] * p[:, 20] / p[:, 77]).to(dtype).double()
    v[:, 150] = (-(v[:, 20] * p[:, 20] + v[:, 77] * p[:, 77]) * 15 / 16 / p[:, 150]).to(dtype).double()
    v[-1] = (torch.rand(n, kvh, d, generator=gen) * 20000 + 100).to(dtype).double()
    v[-1, ::16] = 0
    q = torch.zeros(batch, heads, d, dtype=dtype)
    q[:, :, 0] = 8
    kp = torch.zeros(batch * n, kvh, d, dtype=dtype)
    kp[:, :, 0] = score.view(-1, 1).to(dtype)
    vp = v.view(batch * n, kvh, d).to(dtype)
    want, terms = ((p * t).sum(1).div(p.sum(1)).repeat_interleave(heads // kvh, dim=1) for t in (v, v.abs()))
    # Bound: the rounding of the result, and fp32 arithmetic on each term: an exponent of at most 1.5 (25.3 in the last
    # sequence) to 2^-24 of itself twice over, exp2 to 2^-23, the sums to a few 2^-24.
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    fp32 = torch.full((batch, 1, 1), 2.0 ** -21)
    fp32[-1] = 2.0 ** -17
    bound = 1.01 * half_ulp * want.abs() + fp32 * terms + 2.0 ** -25
    ln, st = torch.full((batch,), n, dtype=torch.int32), torch.arange(batch, dtype=torch.int32) * n
    args = (torch.arange(batch * n, dtype=torch.int32).view(batch, n).to(dev), st.to(dev), ln.to(dev), n)
    out2 = torch.empty(batch, heads, d, dtype=dtype, device=dev)
    ops.token_softmax_reducev(score.view(1, -1).expand(heads, -1).contiguous().to(dev), vp.to(dev), out2, *args)
    fused = ops.token_decode_attention(q.to(dev), kp.to(dev), vp.to(dev), *args)
    for name, got in (("two-call", out2), ("fused", fused)):
        worst = ((got.cpu().double() - want).abs() / bound).amax(dim=(1, 2))
        assert worst.max() <= 1, (name, worst)



@pytest.mark.parametrize("infinite", [False, True])
@pytest.mark.parametrize("batch,heads,kvh", [(21, 32, 32), (20, 32, 8)])
def test_token_attention_fp16_weights_far_below_the_largest(ops, dev, batch, heads, kvh, infinite):
    """fp16 probabilities of about 2^-45.5 are held as precisely as larger ones: every 128th token weighs nearly all and has no values, and those
    between, alike in weight and value, bring results next to the middle between two of the type's smallest numbers, which are rounded
    to the right side wherever they are no closer to it than fp32 arithmetic errs. Infinities in one column of V change nothing in the
    others. K picks the scores: q is 32 in its first two elements."""
    d, n, gen = 128, 512, g(81)
    live = torch.ones(n, dtype=torch.bool)
    live[::128] = False
    first = -torch.randint(177, 180, (batch, kvh), generator=gen).half() / 16
    second = -torch.randint(0, 512, (batch, kvh), generator=gen).half() / 4096
    score = 32 * (first.double() + second.double())
    p = torch.exp(score / d ** 0.5)
    middle = torch.randint(0, 2, (batch, kvh, d), generator=gen) + 0.5      # in units of the smallest number
    value = (middle * 2.0 ** -24 * (4 / 508) / p[..., None]).half().double()
    kp, vp = torch.zeros(2, batch, n, kvh, d, dtype=torch.float16)
    kp[:, live, :, 0], kp[:, live, :, 1] = first[:, None], second[:, None]
    vp[:, live] = value.half()[:, None]
    q = torch.zeros(batch, heads, d, dtype=torch.float16)
    q[:, :, :2] = 32
    units = (508 * p[..., None] * value / (4 + 508 * p[..., None]) * 2.0 ** 24).repeat_interleave(heads // kvh, dim=1)
    # fp32: an exponent of 46 to three roundings of 2^-19, exp2 to 2^-22, 512 sums to 2^-24 each: 2^-14.6 of the result
    off = units - middle.repeat_interleave(heads // kvh, dim=1)
    clear = off.abs() > units * 2.0 ** -14
    if infinite:
        vp[:, 5::128, :, 7], units[:, :, 7], clear[:, :, 7] = math.inf, math.inf, True
        off[:, :, 7] = 0
    assert clear.float().mean() > 0.7 and (off.abs() < units * 2.0 ** -10).all()
    ln, st = torch.full((batch,), n, dtype=torch.int32), torch.arange(batch, dtype=torch.int32) * n
    args = (torch.arange(batch * n, dtype=torch.int32).view(batch, n).to(dev), st.to(dev), ln.to(dev), n)
    kd, vd = kp.view(batch * n, kvh, d).to(dev), vp.view(batch * n, kvh, d).to(dev)
    att = torch.zeros(heads, batch, n)
    att[:, :, live] = (score / d ** 0.5).float().t().repeat_interleave(heads // kvh, dim=0)[..., None]
    out2 = torch.empty(batch, heads, d, dtype=torch.float16, device=dev)
    ops.token_softmax_reducev(att.view(heads, batch * n).to(dev), vd, out2, *args)
    for name, got in (("fused", ops.token_decode_attention(q.to(dev), kd, vd, *args)), ("two-call", out2)):
        wrong = (got.cpu().double() * 2.0 ** 24 != units.round()) & clear
        assert not bool(wrong.any()), (name, int(wrong.sum()), int(clear.sum()))



@pytest.mark.parametrize("heads,kvh", [(4, 4), (8, 2)])
def test_token_attention_values_near_the_largest(ops, dev, heads, kvh):
    """A later key that weighs 2^7 times what the first tile's do and has values near the type's largest: the weighted sum
    stays in range as it does with weights of at most one."""
    d, n, late = 64, 100, 85                         # (a wave takes tokens 64 ... 95, in two tiles)
    score = torch.zeros(n)
    score[late] = 4.875                               # log2: 7.03, less than what replaces the running maximum
    sign = torch.randint(0, 2, (kvh, d), generator=g(84)).double() * 2 - 1
    v = (torch.randn(n, kvh, d, generator=g(85)) * 1e34).bfloat16()
    v[late] = (sign * 2e38).bfloat16()
    kp = torch.zeros(n, kvh, d, dtype=torch.bfloat16)
    kp[:, :, 0] = score[:, None]
    q = torch.zeros(1, heads, d, dtype=torch.bfloat16)
    q[:, :, 0] = 8
    p = torch.softmax(score.double(), 0).view(n, 1, 1)
    want = (p * v.double()).sum(0).repeat_interleave(heads // kvh, dim=0)
    args = (torch.arange(n, dtype=torch.int32).view(1, n).to(dev), torch.zeros(1, dtype=torch.int32, device=dev), torch.full((1,), n, dtype=torch.int32, device=dev), n)
    out2 = torch.empty(1, heads, d, dtype=torch.bfloat16, device=dev)
    ops.token_softmax_reducev(score.expand(heads, n).contiguous().to(dev), v.to(dev), out2, *args)
    for got in (out2, ops.token_decode_attention(q.to(dev), kp.to(dev), v.to(dev), *args)):
        assert_half(got[0].cpu().double() / 1e38, want / 1e38)



@pytest.mark.parametrize("batch,heads,kvh,d,dtype", [
    (3, 8, 8, 64, torch.float32), (3, 8, 2, 64, torch.float32), (3, 4, 2, 48, torch.float32),
    (170, 4, 4, 128, torch.bfloat16), (3, 4, 4, 80, torch.float16), (3, 5, 5, 128, torch.bfloat16), (3, 8, 2, 128, torch.float16)])
def test_token_attention_what_slot_zero_holds(ops, dev, batch, heads, kvh, d, dtype):
    """NaN in slot 0, which no sequence holds, changes nothing: not where a slot outside the pool is skipped, nor in the places
    past a sequence's end. Rows on the lanes (fp32, many pairs, rows of other lengths) and on the matrix pipe."""
    slots, width = 120, 37
    kp = torch.randn(slots, kvh, d, generator=g(86)).to(dtype)
    vp = torch.randn(slots, kvh, d, generator=g(87)).to(dtype)
    q = torch.randn(batch, heads, d, generator=g(88)).to(dtype).to(dev)
    b_loc = torch.randint(1, slots, (batch, width), generator=g(89)).to(torch.int32)
    b_loc[0, 3::5] = torch.tensor([-1, slots, -7, slots + 1, -1, slots, -1], dtype=torch.int32)
    ln = torch.full((batch,), width, dtype=torch.int32)
    ln[1], ln[2] = 1, 30
    args = (b_loc.to(dev), torch.arange(batch, dtype=torch.int32).to(dev) * width, ln.to(dev), width)

    def both():
        k, v = kp.to(dev), vp.to(dev)
        att = torch.zeros(heads, batch * width, dtype=torch.float32, device=dev)
        out2 = torch.empty(batch, heads, d, dtype=dtype, device=dev)
        ops.token_attention(q, k, att, *args)
        ops.token_softmax_reducev(att, v, out2, *args)
        return ops.token_decode_attention(q, k, v, *args).cpu(), out2.cpu()

    kp[0], vp[0] = 0, 0
    want = both()
    kp[0], vp[0] = float("nan"), float("nan")
    for got, w in zip(both(), want):
        assert torch.isfinite(w).all()
        assert torch.equal(got, w)



@pytest.mark.parametrize("batch,heads,kvh,d,width,dtype", [
    (128, 8, 8, 128, 24, torch.bfloat16),      # a head to itself: all three forms on the lanes
    (24, 32, 32, 64, 1500, torch.float16),     # (not many, but longer)
    (128, 9, 9, 64, 40, torch.float16),        # a head count that leaves wave loads incomplete
    (4, 3, 3, 200, 700, torch.bfloat16),       # and rows of other lengths, in splits
    (128, 32, 16, 128, 30, torch.bfloat16),    # two heads per row
    (256, 16, 8, 96, 20, torch.float16),
    (2, 8, 4, 256, 8300, torch.bfloat16),      # long sequences of rows of 512 bytes: the fused form
    (128, 32, 8, 256, 24, torch.float16),      # four
    (512, 56, 8, 192, 10, torch.bfloat16),     # seven
    (520, 12, 4, 128, 32, torch.bfloat16),     # three
    (9, 30, 30, 128, 62, torch.bfloat16),      # short sequences: a head to itself, from few rows on
    (3, 8, 8, 128, 24, torch.float16),
    (5, 64, 64, 256, 12, torch.bfloat16),
    (3, 16, 8, 256, 16, torch.float16),        # two
    (140, 64, 8, 256, 30, torch.float16),      # eight
])
def test_token_attention_many_rows_on_the_lanes(ops, dev, batch, heads, kvh, d, width, dtype):
    """16-bit rows that are many for their length, short ones, and those of 512 bytes: fused, and the two calls with scores in fp32 and in
    the type of the rows, sequences of one token up to the widest."""
    gen = g(90)
    slots = batch * width + 5
    kp, vp = (torch.randn(slots, kvh, d, generator=gen).to(dtype) for _ in range(2))
    q = torch.randn(batch, heads, d, generator=gen).to(dtype)
    ln = torch.randint(1, width + 1, (batch,), generator=gen)
    ln[0], ln[1] = width, 1
    b_loc = torch.randperm(slots, generator=gen)[:batch * width].view(batch, width)
    st = torch.arange(batch) * width
    rows = b_loc.to(dev)                              # right-aligned: the last ln[b] columns count
    rep = lambda t: t.to(dev)[rows].float().repeat_interleave(heads // kvh, dim=2)     # [batch, width, heads, d]
    score = (q.to(dev).float()[:, None] * rep(kp)).sum(-1) / d ** 0.5
    live = torch.arange(width, device=dev)[None, :] >= width - ln.to(dev)[:, None]
    p = torch.softmax(score.masked_fill(~live[..., None], float("-inf")), dim=1)
    want = (p[..., None] * rep(vp)).sum(1)
    i32 = lambda t: t.to(torch.int32).to(dev)
    args = (i32(b_loc), i32(st), i32(ln), width)
    q, kp, vp = q.to(dev), kp.to(dev), vp.to(dev)
    got = ops.token_decode_attention(q, kp, vp, *args)
    assert_half(got, want, rel=1e-2, abs_=2e-3)
    assert_exact(ops.token_decode_attention(q, kp, vp, *args, no_alloc=True), got)
    for st_type, tight in ((torch.float32, True), (dtype, False)):
        att = torch.full((heads, batch * width), float("nan"), dtype=st_type, device=dev)
        ops.token_attention(q, kp, att, *args)
        for b in (0, 1, batch - 1):
            n = int(ln[b])
            col, ref = att[:, b * width:b * width + n], score[b, width - n:].t()
            assert_fp32(col, ref, rel=1e-5) if tight else assert_half(col, ref)
        out2 = torch.empty_like(got)
        ops.token_softmax_reducev(att, vp, out2, *args)
        assert_half(out2, want, rel=1e-2, abs_=2e-3) if tight else assert_half(out2, want, rel=3e-2, abs_=2e-2)



@pytest.mark.parametrize("batch,heads,kvh,d,width,dtype", [
    (2, 8, 2, 128, 256, torch.bfloat16), (2, 8, 2, 128, 257, torch.float16),           # any number of workgroups
    (20, 32, 8, 128, 512, torch.bfloat16), (19, 32, 8, 128, 512, torch.bfloat16), (20, 32, 8, 128, 513, torch.float16),
    (28, 32, 8, 128, 768, torch.float16), (28, 16, 8, 64, 768, torch.bfloat16),        # (rows of 128 bytes: chunks)
    (44, 32, 8, 128, 768, torch.bfloat16), (44, 32, 8, 128, 769, torch.bfloat16),
    (52, 32, 8, 64, 1024, torch.float16), (52, 32, 8, 128, 1025, torch.bfloat16), (65, 16, 8, 128, 600, torch.bfloat16),
    (20, 18, 1, 96, 512, torch.float16),                                               # two workgroups a row
    # many rows with a query head to itself: on the pipe, and past each line of that on the lanes
    (24, 32, 32, 128, 64, torch.bfloat16), (25, 32, 32, 128, 64, torch.bfloat16), (20, 40, 40, 128, 250, torch.float16),
    (64, 32, 32, 128, 130, torch.bfloat16), (21, 32, 32, 128, 512, torch.float16), (21, 32, 32, 128, 513, torch.bfloat16), (64, 32, 32, 128, 385, torch.bfloat16),
])
def test_token_attention_one_chunk_or_several(ops, dev, batch, heads, kvh, d, width, dtype):
    """Both sides of the lines up to which sequences are walked whole by the matrix pipe: longest sequence against workgroups."""
    test_token_attention_many_rows_on_the_lanes(ops, dev, batch, heads, kvh, d, width, dtype)


@pytest.mark.parametrize("heads,kvh,dtype", [(4, 4, torch.bfloat16), (8, 2, torch.float16), (2, 1, torch.bfloat16), (4, 1, torch.float32)])
def test_token_attention_slots_beyond_32_bits(ops, dev, heads, kvh, dtype):
    """A pool of more slots than 31 bits number (here all of them one row, by a stride of zero) is the lanes' in every form."""
    d, n, slots = 64, 300, (1 << 31) + 1000
    row_k, row_v = torch.randn(1, kvh, d, generator=g(91)).to(dtype).to(dev), torch.randn(1, kvh, d, generator=g(92)).to(dtype).to(dev)
    k, v = row_k.expand(slots, kvh, d), row_v.expand(slots, kvh, d)
    q = torch.randn(2, heads, d, generator=g(93)).to(dtype).to(dev)
    b_loc = torch.randint(0, slots, (2, n), generator=g(94))
    b_loc[0, :3] = torch.tensor([slots - 1, slots, -1])                     # two of them outside the pool
    args = (b_loc.to(dev), torch.tensor([0, n], device=dev), torch.tensor([n, 7], device=dev), n)
    want = row_v[0].repeat_interleave(heads // kvh, dim=0).cpu()            # a mean of equal rows
    score = (q * row_k[0].repeat_interleave(heads // kvh, dim=0)).float().sum(-1) / 8
    att = torch.zeros(heads, 2 * n, dtype=torch.float32, device=dev)
    ops.token_attention(q, k, att, *args)
    assert (att[:, 1:3] == -float("inf")).all()
    out2 = torch.empty(2, heads, d, dtype=dtype, device=dev)
    ops.token_softmax_reducev(att, v, out2, *args)
    for got in (out2, ops.token_decode_attention(q, k, v, *args)):
        for b in range(2):
            assert_half(got[b], want, rel=1e-2, abs_=1e-5)
    assert_half(att[:, 0], score[0])
    assert_half(att[:, n + 6], score[1])


# ------------------------------------------------------------------ int8 weight-only linear
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [
    (2305, 4360, 256),      # whole tiles only (a workgroup walks two: the loads of the next one), the fewest K tiles, ragged rows and columns
    (2560, 4096, 384),      # an odd number of K-tile pairs
    (65, 2056, 8192),       # one row of tiles in slices of K
    (97, 4096, 4096), (129, 4104, 4096), (257, 4096, 4224),
    (1025, 17160, 1152),    # whole tiles, then slices of the last round
])
def test_weight_only_int8_linear_converted_in_the_large_tiles(ops, dev, m, n, k, dtype):
    """Products of small whole numbers: every sum is exact in fp32, the scales are powers of two, so the result is the exact
    sum rounded once. Weights are rows of a wider matrix; with and without bias."""
    x = torch.randint(-4, 5, (m, k), generator=g(70)).to(dtype)
    wide = torch.randint(-128, 128, (n, k + 16), generator=g(71), dtype=torch.int8)
    w = wide[:, :k]
    scale = 2.0 ** torch.randint(-12, -8, (n,), generator=g(72)).float()
    bias = torch.randint(-8, 9, (n,), generator=g(73)).float()
    want = torch.matmul(x.to(dev).double(), w.to(dev).double().t()) * scale.to(dev).double()
    for b in (None, bias):
        got = ops.weight_only_int8_linear(x.to(dev), wide.to(dev)[:, :k], scale.to(dev), None if b is None else b.to(dev))
        # (sums of at most 2^22 plus a bias: exact in fp32, and in float64, until the one rounding)
        assert_exact(got, (want if b is None else want + b.to(dev).double()).float().to(dtype))


@pytest.mark.parametrize("m", [1, 4, 16, 33])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weight_only_int8_linear(ops, dev, pkg, m, dtype):
    w = pkg.workloads.int8_linear(seed=2, m=m, k=4096, n=1000, dtype=dtype)
    want = oracle.weight_only_int8_linear(w["x"], w["w"], w["scale"])
    got = ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev))
    assert_half(got, want)
    bias = torch.randn(1000, generator=g(33)).to(dtype)
    got = ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].float().to(dev), bias.to(dev))
    assert_half(got, want + bias.float())
    # odd K takes the scalar path
    w2 = pkg.workloads.int8_linear(seed=3, m=m, k=200, n=37, dtype=dtype)
    assert_half(ops.weight_only_int8_linear(w2["x"].to(dev), w2["w"].to(dev), w2["scale"].to(dev)),
                oracle.weight_only_int8_linear(w2["x"], w2["w"], w2["scale"]))


@pytest.mark.parametrize("m", [1, 4, 16])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weight_only_int8_full_shape(ops, dev, pkg, m, dtype):
    """K = 4096, N = 11008 at every row count the workload names, against the oracle and against an exact case: a
    one-hot activation row selects one weight column, so the result is w * scale rounded once."""
    w = pkg.workloads.int8_linear(seed=4, m=m, k=4096, n=11008, dtype=dtype)
    got = ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev))
    assert_half(got, oracle.weight_only_int8_linear(w["x"], w["w"], w["scale"]))
    x = torch.zeros(m, 4096, dtype=dtype)
    cols = torch.randint(0, 4096, (m,), generator=g(34))
    x[torch.arange(m), cols] = 1
    got = ops.weight_only_int8_linear(x.to(dev), w["w"].to(dev), w["scale"].to(dev))
    want = (w["w"][:, cols].float() * w["scale"].float()[:, None]).t().to(dtype)
    assert_exact(got, want)


@pytest.mark.parametrize("m,k,n", [(1, 11008, 4096), (5, 8192 + 128, 100), (37, 4096, 16 * 7 + 3), (16, 4096, 22016),
                                   (64, 4096, 4096), (100, 1024 + 256, 520), (29, 2048 + 128, 11008),
                                   (40, 2048, 11008), (20, 1024, 6200), (100, 512, 12288), (33, 768, 22016 + 8),
                                   (24, 256, 30000), (3, 256, 10240)])
def test_weight_only_int8_linear_chunked_k_row_groups_and_tile_counts(ops, dev, pkg, m, k, n):
    """K beyond one staged activation chunk (4096 columns), more than 16 rows (row groups), channel counts that leave
    partly filled workgroups, and an N large enough to use the widest workgroup. Wide weights with K a multiple of
    256 take the form that stages both operands through LDS (the last six cases, and N = 22016 above): one, two and four
    row groups, channel shares of up to 64 and up to 128 per workgroup that are no multiple of 16, more than 64 rows
    (a second workgroup row), K of one to eight stages."""
    w = pkg.workloads.int8_linear(seed=5, m=m, k=k, n=n)
    got = ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev))
    assert_half(got, oracle.weight_only_int8_linear(w["x"], w["w"], w["scale"]))



@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n", [(64, 14336, 4096), (33, 4096, 4096), (17, 2048 + 256, 5120), (48, 11008, 4100), (64, 2048, 200),
                                   (4, 8192, 4096), (16, 8192, 8192)])
def test_weight_only_int8_linear_narrow_weights_split_over_k(ops, dev, pkg, m, k, n, dtype):
    """Weights of fewer than 10240 channels with few columns for each compute unit: K split over workgroups for 48 and 64 rows with a long K (4 and
    3 slices, the latter with a ragged last channel block), unscaled fp32 sums reduced by a second launch that applies scale and bias; the
    others stream the whole of K. Against the oracle, with a bias in float32, and exactly on one-hot rows."""
    w = pkg.workloads.int8_linear(seed=8, m=m, k=k, n=n, dtype=dtype)
    want = oracle.weight_only_int8_linear(w["x"], w["w"], w["scale"])
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev)), want)
    bias = torch.randn(n, generator=g(37))
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev), bias.to(dev)), want + bias)
    x = torch.zeros(m, k, dtype=dtype)
    cols = torch.randint(0, k, (m,), generator=g(38))
    x[torch.arange(m), cols] = 1
    got = ops.weight_only_int8_linear(x.to(dev), w["w"].to(dev), w["scale"].to(dev))
    assert_exact(got, (w["w"][:, cols].float() * w["scale"].float()[:, None]).t().to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n,slices", [(16, 28672, 8192, 2), (17, 13824, 5120, 3), (32, 11008, 4096, 4), (24, 11008, 4100, 3), (31, 8448, 200, 11), (48, 11008, 4100, 3),
                                          (64, 14336, 4096, 4), (17, 8192, 5120, 0)])
def test_weight_only_int8_linear_k_slices_for_one_to_four_row_groups(ops, dev, pkg, m, k, n, slices, dtype):
    """K split over workgroups, as the workspace of the slices' sums tells, at 13 to 64 rows: one, two and four row groups, a shorter last
    slice, a ragged last channel block (and one shape that is left whole). Sums of whole numbers below 2^24, exact in fp32, scaled by
    powers of two and rounded once."""
    gen = torch.Generator(dev).manual_seed(39)
    x = torch.randint(-3, 4, (m, k), generator=gen, device=dev).to(dtype)
    w = torch.randint(-127, 128, (n, k), generator=gen, device=dev, dtype=torch.int8)
    scale, bias = 2.0 ** torch.randint(-12, -8, (n,), generator=gen, device=dev), torch.randint(-4, 5, (n,), generator=gen, device=dev).float()
    want = x.double() @ w.double().t() * scale.double()
    with own_context(ops, pkg) as ctx:
        assert_exact(ops.weight_only_int8_linear(x, w, scale.half()), want.to(dtype))
        assert ctx.workspace()[1] == slices * m * n * 4
        assert_exact(ops.weight_only_int8_linear(x, w, scale.float(), bias), (want + bias.double()).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n", [(129, 4096, 1000), (300, 1024 + 16, 520), (1024, 4096, 4096), (4608, 384, 4096),
                                   (4568, 512, 4072)])
def test_weight_only_int8_linear_many_rows(ops, dev, pkg, m, k, n, dtype):
    """From 129 rows on, without a bias, the weights are expanded once and the product goes to the dense GEMM, the
    channel scale in a pass over the result or, where the product takes the large-tile kernel (the last two shapes:
    288 tiles, the second with ragged last tiles), in that kernel's epilogue: against the oracle, with a bias (the
    streaming kernels, or that epilogue), with a float32 scale, and exactly on one-hot rows, where the result is
    w * scale (+ bias) rounded once on every route."""
    w = pkg.workloads.int8_linear(seed=6, m=m, k=k, n=n, dtype=dtype)
    want = oracle.weight_only_int8_linear(w["x"], w["w"], w["scale"])
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev)), want)
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].float().to(dev)), want)
    bias = torch.randn(n, generator=g(35)).to(dtype)
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].to(dev), bias.to(dev)), want + bias.float())
    assert_half(ops.weight_only_int8_linear(w["x"].to(dev), w["w"].to(dev), w["scale"].float().to(dev), bias.float().to(dev)),
                want + bias.float())
    x = torch.zeros(m, k, dtype=dtype)
    cols = torch.randint(0, k, (m,), generator=g(36))
    x[torch.arange(m), cols] = 1
    got = ops.weight_only_int8_linear(x.to(dev), w["w"].to(dev), w["scale"].to(dev))
    assert_exact(got, (w["w"][:, cols].float() * w["scale"].float()[:, None]).t().to(dtype))
    # and with a bias: w * scale is exact in fp32, the bias is added there, one rounding on every route
    got = ops.weight_only_int8_linear(x.to(dev), w["w"].to(dev), w["scale"].to(dev), bias.to(dev))
    assert_exact(got, ((w["w"][:, cols].float() * w["scale"].float()[:, None]).t() + bias.float()).to(dtype))


# ------------------------------------------------------------------ decoder block
def test_tiny_decoder_block_fp32_every_intermediate(ops, dev, pkg):
    x, p, cfg = pkg.workloads.tiny_block(seed=0)
    want, wi = oracle.decoder_block(x, p, cfg["heads"], cfg["eps"], cfg["theta"])
    got, gi = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg)
    for name in ["norm1", "qkv", "q_rot", "k_rot", "attn", "o", "res1", "norm2", "act", "down", "out"]:
        a, b = gi[name].cpu(), wi[name]
        assert_fp32(a.reshape(b.shape), b, rel=1e-5)
    got2, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_ffn=True)
    assert_fp32(got2, want)
    # gate and up as the column halves of one stacked projection: the same numbers, op for op
    got3, gi3 = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_ffn=True, stacked_gate_up=True)
    assert_fp32(gi3["act"].cpu().reshape(wi["act"].shape), wi["act"], rel=1e-5)
    assert_fp32(got3, want)
    got4, gi4 = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, stacked_gate_up="interleaved")
    assert_fp32(gi4["act"].cpu().reshape(wi["act"].shape), wi["act"], rel=1e-5)
    assert_fp32(got4, want)
    # rotary inside the stacked projection, on q / k weight rows permuted to the adjacent-pair convention
    got5, gi5 = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_rotary=True)
    assert_fp32(gi5["attn"].cpu().reshape(wi["attn"].shape), wi["attn"], rel=1e-5)
    assert_fp32(got5, want, rel=1e-5)


def test_small_decoder_block_bf16(ops, dev, pkg):
    x, p, cfg = pkg.workloads.llama7b_layer(seed=0, batch=2, seq=256, hidden=512, heads=4, ffn=1408)
    want, _ = oracle.decoder_block(x.float(), {k: v.float() for k, v in p.items()}, cfg["heads"], cfg["eps"], cfg["theta"])
    got, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_ffn=True)
    # eleven chained bf16 roundings: 3e-2 relative / 3e-2 absolute on an O(1) output
    assert_half(got, want, rel=3e-2, abs_=3e-2)
    got, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_ffn=True, stacked_gate_up=True)
    assert_half(got, want, rel=3e-2, abs_=3e-2)
    got, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, stacked_gate_up="interleaved")
    assert_half(got, want, rel=3e-2, abs_=3e-2)
    got, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, stacked_gate_up="interleaved", fused_rotary=True)
    assert_half(got, want, rel=3e-2, abs_=3e-2)


def test_decoder_block_bf16_with_both_fused_projections_in_one_launch_each(ops, dev, pkg):
    """The benchmark's configuration of the layer at a size where both fused projections take their single-launch
    form (2304 tokens, hidden 2048: 216 and 198 tiles of 256 x 256): rotary in the QKV epilogue on permuted weight
    rows, silu * mul in the gate / up epilogue, residuals through addmm-free adds."""
    x, p, cfg = pkg.workloads.llama7b_layer(seed=3, batch=3, seq=768, hidden=2048, heads=16, ffn=2816)
    want, _ = oracle.decoder_block(x.float(), {k: v.float() for k, v in p.items()}, cfg["heads"], cfg["eps"], cfg["theta"])
    got, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, stacked_gate_up="interleaved", fused_rotary=True)
    assert_half(got, want, rel=3e-2, abs_=3e-2)
    ref, _ = run_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg, fused_ffn=True)
    assert_half(got, ref.float().cpu(), rel=3e-2, abs_=3e-2)


def test_decoder_block_from_primitive_ops_only(ops, dev, pkg):
    """No fused ext op: RMSNorm, rotary tables and rotation, causal mask and attention all come from primitive
    diopi ops (pow, mean, rsqrt, arange, exp, cos, sin, cat, comparisons, masked_fill, softmax, bmm, strided copies)."""
    x, p, cfg = pkg.workloads.tiny_block(seed=1)
    want, _ = oracle.decoder_block(x, p, cfg["heads"], cfg["eps"], cfg["theta"])
    got = run_decomposed_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg)
    # the decomposed rotary tables come from exp() on the device instead of pow() on the host: 2e-5 on the tensor scale
    assert_fp32(got, want, rel=2e-5)
    x, p, cfg = pkg.workloads.llama7b_layer(seed=2, batch=2, seq=128, hidden=512, heads=4, ffn=1408)
    want, _ = oracle.decoder_block(x.float(), {k: v.float() for k, v in p.items()}, cfg["heads"], cfg["eps"], cfg["theta"])
    got = run_decomposed_decoder_block(ops, x.to(dev), {k: v.to(dev) for k, v in p.items()}, cfg)
    assert_half(got, want, rel=3e-2, abs_=3e-2)
