"""Each kernel alone against a plain 32-bit (or 64-bit) reference of the same
operation, at sizes other than the engine's, with inputs made so that a fault
shows: a far key among hundreds, a window's edge, a slot of the cache, pages
out of order."""

import math

import numpy as np
import pytest
import torch

import plain_llama as P
from nnis_amd.errors import KernelError
from nnis_amd.kernels.ops import GEMM_F32_NORM_ROWS, GEMM_F32_VARIANTS

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def _ops():
    from nnis_amd.kernels import ops

    return ops


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_embed(dtype):
    ops = _ops()
    table = torch.randn(777, 130).to(DT[dtype])
    ids = [0, 776, 5, 5, -1, 777, 300]
    out = torch.full((len(ids), 130), 9.0, device="cuda")
    ops.embed(_i32(ids), table.cuda(), out)
    want = torch.stack([table[i].float() if 0 <= i < 777 else torch.zeros(130) for i in ids])
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("width", [5, 64, 576, 1020, 4100, 8192, 9000])
@pytest.mark.parametrize("x_dtype, w_dtype, out_dtype", [("float32", "float32", "float32"), ("float32", "bfloat16", "bfloat16"),
                                                         ("bfloat16", "float32", "bfloat16"), ("float32", "float32", "bfloat16")])
def test_rmsnorm(width, x_dtype, w_dtype, out_dtype):
    ops = _ops()
    torch.manual_seed(width)
    x = (torch.randn(7, width) * 4).to(DT[x_dtype])
    w = (1 + 0.2 * torch.randn(width)).to(DT[w_dtype])
    out = torch.empty(7, width, dtype=DT[out_dtype], device="cuda")
    ops.rmsnorm(x.cuda(), w.cuda(), 1e-6, out)
    want = P.rms_norm(x.double(), w.double(), 1e-6)
    tol = 1e-6 if out_dtype == "float32" else 1e-2
    assert ((out.cpu().double() - want).abs() <= tol * (1 + want.abs())).all()
    if x_dtype == "bfloat16":
        with pytest.raises(KernelError, match="32-bit"):
            ops.rmsnorm(x.cuda(), w.cuda(), 1e-6, out, delta=x.cuda())


@pytest.mark.parametrize("m, n, k", [(1, 1, 1), (1, 960, 576), (7, 63, 17), (65, 130, 176), (200, 70, 600), (3, 1000, 96)])
@pytest.mark.parametrize("x_dtype, w_dtype, y_dtype", [("float32", "float32", "float32"), ("bfloat16", "bfloat16", "bfloat16"),
                                                       ("bfloat16", "bfloat16", "float32"), ("bfloat16", "float32", "bfloat16")])
def test_gemm_ordered(m, n, k, x_dtype, w_dtype, y_dtype):
    ops = _ops()
    torch.manual_seed(m * 1000 + n + k)
    x = torch.randn(m, k).to(DT[x_dtype])
    w = torch.randn(n, k).to(DT[w_dtype])
    y = torch.empty(m, n, dtype=DT[y_dtype], device="cuda")
    ops.gemm_ordered(x.cuda(), w.cuda(), y)
    want = x.double() @ w.double().t()
    scale = (x.double().abs() @ w.double().abs().t())  # bounds the rounding of a sum of k products
    tol = 2e-7 * math.sqrt(k) if y_dtype == "float32" else 4e-3
    assert ((y.cpu().double() - want).abs() <= tol * scale + 1e-30).all()
    if (x_dtype, w_dtype, y_dtype) == ("float32", "float32", "float32"):
        # one ascending chain of fused multiply-adds per element: reproduce it exactly for one row
        chain = np.zeros(n, dtype=np.float64)
        for kk in range(k):  # float64 holds every 32-bit product exactly; round after each step
            chain = (x[0, kk].double().item() * w[:, kk].double().numpy() + chain).astype(np.float32).astype(np.float64)
        assert np.array_equal(y[0].cpu().numpy().astype(np.float64), chain)
    # a row's result does not depend on the other rows
    if m > 1:
        alone = torch.empty(1, n, dtype=DT[y_dtype], device="cuda")
        ops.gemm_ordered(x[m - 1:].contiguous().cuda(), w.cuda(), alone)
        assert torch.equal(alone[0], y[m - 1])


@pytest.mark.parametrize("variant", range(-1, GEMM_F32_VARIANTS))
@pytest.mark.parametrize("m, n, k", [(1, 1, 4), (8, 40, 52), (7, 130, 548), (17, 33, 100), (65, 130, 176), (131, 257, 612), (5, 17, 2052)])
def test_gemm_f32_on_the_matrix_cores(m, n, k, variant):
    """Every form of the product at sizes with tails in every dimension (K a multiple of 4 and of nothing more), against 64
    bits: a sum of k products in chains is off by at most k roundings of the sum of magnitudes, sqrt(k) where they are
    as random as here."""
    ops = _ops()
    if variant == 13 and m > 8:
        with pytest.raises(KernelError, match="no variant"):
            ops.gemm_f32(torch.zeros(m, k, device="cuda"), torch.zeros(n, k, device="cuda"), torch.zeros(m, n, device="cuda"), variant)
        return
    torch.manual_seed(m + n + k)
    x, w = torch.randn(m, k), torch.randn(n, k)
    want, scale = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    y = torch.full((m + 1, n), 7.0, device="cuda")
    ops.gemm_f32(x.cuda(), w.cuda(), y[:m], variant)
    assert ((y[:m].cpu().double() - want).abs() <= 2e-7 * math.sqrt(k) * scale).all() and (y[m] == 7).all()
    if 4 <= variant <= 12:
        return  # tiles take 32-bit rows
    x = x.bfloat16()
    for dtype, tol in ((torch.float32, 2e-7 * math.sqrt(k)), (torch.bfloat16, 4e-3)):
        y = torch.empty(m, n, dtype=dtype, device="cuda")
        ops.gemm_f32(x.cuda(), w.cuda(), y, variant)
        assert ((y.cpu().double() - x.double() @ w.double().t()).abs() <= tol * (x.double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("variant", range(4, 13))
@pytest.mark.parametrize("k", [36, 100, 612])
def test_gemm_f32_tiles_split_any_number(k, variant):
    """The tiles multiply the bfloat16 parts that a 32-bit number is the sum of.  Rows of every magnitude come out as
    accurate as ordinary ones: the bound as above, and the smallest 32-bit number for each product that falls below
    it.  Rows and columns with infinities and numbers that are none come out as the 32-bit chain has them, and change
    nothing beside them."""
    ops = _ops()
    torch.manual_seed(k)
    m, n = 70, 65
    x, w = torch.randn(m, k), torch.randn(n, k)
    x[1] *= 1e-36  # (their last parts are below bfloat16's smallest number)
    x[2] *= 1e-25
    x[3] *= 1e30
    x[4] = torch.where(x[4] > 0, 3.4e38, -3.4e38) * (torch.arange(k) == k - 1)  # rounds up to infinity in bfloat16
    x[5] = 0.0
    w[3] *= 1e-20
    w[4] *= torch.logspace(-18, 18, k)
    want, scale = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    y = torch.empty(m, n, device="cuda")
    ops.gemm_f32(x.cuda(), w.cuda(), y, variant)
    got = y.cpu().double()
    scale = 2e-7 * math.sqrt(k) * scale + 1.5e-45 * k
    fits = scale < 3.4e38 * 2e-7  # (a sum of terms beyond it may be infinite, or cancel, in one order and not in another)
    bad = ((got - want).abs() > scale) & fits
    assert not bad.any() and (got[5] == 0).all(), (bad.nonzero()[:8], (got - want)[bad][:8], scale[bad][:8], want[bad][:8])
    x[6, k - 1], x[7, 3], w[9, 0] = float("inf"), float("nan"), float("-inf")
    ops.gemm_f32(x.cuda(), w.cuda(), y, variant)
    now, chain = y.cpu(), torch.empty(m, n, device="cuda")
    ops.gemm_ordered(x.cuda(), w.cuda(), chain)
    chain = chain.cpu()
    for got_line, want_line in ((now[6], chain[6]), (now[7], chain[7]), (now[:, 9], chain[:, 9])):
        assert torch.equal(got_line.isnan(), want_line.isnan()) and torch.equal(got_line.isinf(), want_line.isinf())
        assert torch.equal(got_line.sign()[got_line.isinf()], want_line.sign()[got_line.isinf()])
    assert not now[:, 9].isfinite().any()
    rest = [r for r in range(m) if r not in (6, 7)]
    columns = [c for c in range(n) if c != 9]
    # (bits: a sum whose terms are beyond the largest number with either sign is none, in both)
    assert torch.equal(now[rest][:, columns].view(torch.int32), got.float()[rest][:, columns].view(torch.int32))


@pytest.mark.parametrize("variant", range(4, 13))
@pytest.mark.parametrize("m, n, k", [(70, 65, 4), (129, 130, 100), (64, 64, 612)])
def test_gemm_f32_tiles_keep_every_bit_of_tiny_factors(m, n, k, variant):
    """Numbers below 2^-110 are not the sum of their bfloat16 parts, and below 2^-134 all of these are zero: times large numbers they
    come out as accurate as any others, on either side, and change no other row or column."""
    ops = _ops()
    torch.manual_seed(k)
    x, w = torch.randn(m, k), torch.randn(n, k)
    y, plain = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda")
    ops.gemm_f32(x.cuda(), w.cuda(), plain, variant)
    for row, magnitude in ((0, -112), (17, -118), (38, -126), (62, -135), (m - 1, -142)):
        x[row] *= 2.0 ** magnitude
    for column, magnitude in ((1, 40), (20, 70), (39, 110), (50, -114), (n - 1, -130)):
        w[column] *= 2.0 ** magnitude
    x[40, 1:], x[40, 0], w[40, 1:], w[40, 0] = 0.0, 4e-41, 0.0, 1e20  # (one term, whose sum of parts is zero)
    x[41, 1:], x[41, 0] = 0.0, 3e35
    want, scale = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    ops.gemm_f32(x.cuda(), w.cuda(), y, variant)
    error = (y.cpu().double() - want).abs()
    bad = (error > 2e-7 * math.sqrt(k) * scale + 1.5e-45 * k) & (scale < 3e38)  # (row 41 beside the large columns is beyond the largest number)
    assert not bad.any(), (bad.nonzero()[:8], error[bad][:8], want[bad][:8])
    rows = [r for r in range(m) if r not in (0, 17, 38, 62, m - 1, 40, 41)]
    columns = [c for c in range(n) if c not in (1, 20, 39, 50, n - 1, 40)]
    assert torch.equal(y[rows][:, columns], plain[rows][:, columns])


@pytest.mark.parametrize("variant", range(4, 13))
def test_gemm_f32_tiles_of_no_numbers_take_no_age(variant):
    """Rows that are no numbers, and tiny sums, are multiplied again in 32 bits by the whole wave.  A product of nothing else reads
    its operands twice and multiplies them a second time at the 32-bit instruction's rate: a few times as long as an ordinary one
    (about 4 here), where one lane's chain for each sum took 80 to 208 times."""
    ops = _ops()
    torch.manual_seed(variant)
    m, n, k = 256, 512, 2048
    w, y = torch.randn(n, k).cuda(), torch.empty(m, n, device="cuda")
    times = []
    for x in (torch.randn(m, k).cuda(), torch.full((m, k), float("nan"), device="cuda"), 1e-30 * torch.randn(m, k).cuda()):
        for _ in range(3):
            ops.gemm_f32(x, w, y, variant)
        best = math.inf
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                ops.gemm_f32(x, w, y, variant)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end) * 100)
        times.append(best)
    assert max(times[1:]) < 10 * times[0], times


def _f32_forms(rows, normed):
    """The forms that take a product of so many 32-bit rows, with the norm before it or without."""
    few = (-1, 0, 1, 13, 14, 15)  # (13: half strips, up to 8 rows)
    return [v for v in range(-1, GEMM_F32_VARIANTS) if (v != 13 or rows <= 8) and not (normed and (rows > GEMM_F32_NORM_ROWS or v not in few))]


UNPAIRED_F32_FORMS = (0, 6, 8, 11)  # a wave of theirs has no whole pair of strips: no gate, no rotation


@pytest.mark.parametrize("m, n, k, normed, variant", [
    (*sizes, normed, variant) for sizes in [(1, 2, 4), (8, 70, 52), (5, 2 * 130, 548), (16, 34, 100), (65, 2 * 67, 176), (131, 256, 612)]
    for normed in (False, True) for variant in _f32_forms(sizes[0], normed)])
def test_gemm_f32_with_what_comes_behind_it(m, n, k, normed, variant):
    """The gate, the sum into the stream and the plain store behind the product, with the norm before it or without, in
    every form that takes them, against 64 bits: the bound of the plain product, carried through the gate (whose slopes
    are below 1.1 times the other factor) and with the norm's own few roundings."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x, w, gain = torch.randn(m, k), torch.randn(n, k), 1 + 0.2 * torch.randn(k)
    rows = P.rms_norm(x.double(), gain.double(), 1e-5) if normed else x.double()
    product, scale = rows @ w.double().t(), 4e-7 * math.sqrt(k) * (rows.abs() @ w.double().abs().t()) + 1e-7
    norm = (gain.cuda(), 1e-5) if normed else ()
    out = torch.full((m + 1, n // 2), 7.0, device="cuda")
    if variant in UNPAIRED_F32_FORMS:
        with pytest.raises(KernelError, match="no variant"):
            ops.gemm_f32_fused(x.cuda(), w.cuda(), out[:m], ops.EPILOGUE_SILU, *norm, variant=variant)
    else:
        ops.gemm_f32_fused(x.cuda(), w.cuda(), out[:m], ops.EPILOGUE_SILU, *norm, variant=variant)
        gate, up = product[:, :n // 2], product[:, n // 2:]
        bound = 1.1 * (scale[:, :n // 2] * up.abs() + gate.abs() * scale[:, n // 2:]) + 1e-6 * (1 + (gate * up).abs()) + scale[:, :n // 2] * scale[:, n // 2:]
        assert ((out[:m].cpu().double() - gate * torch.sigmoid(gate) * up).abs() <= bound).all() and (out[m] == 7).all()
    out = torch.full((m + 1, n), 7.0, device="cuda")
    ops.gemm_f32_fused(x.cuda(), w.cuda(), out[:m], ops.EPILOGUE_STORE, *norm, variant=variant)
    assert ((out[:m].cpu().double() - product).abs() <= scale).all() and (out[m] == 7).all()
    if not normed:
        stream = torch.randn(m + 1, n)
        out = stream.cuda()
        ops.gemm_f32_fused(x.cuda(), w.cuda(), out[:m], ops.EPILOGUE_RESIDUAL, variant=variant)
        assert ((out[:m].cpu().double() - stream[:m].double() - product).abs() <= scale + 1e-6).all() and torch.equal(out[m].cpu(), stream[m])


@pytest.mark.parametrize("tokens, heads, kv_heads, head_dim, normed, tables, variant", [
    (*case, variant) for case in [(1, 9, 3, 64, True, True), (7, 3, 1, 32, True, False), (13, 4, 4, 96, False, True), (70, 4, 2, 64, False, False)]
    for variant in _f32_forms(case[0], case[4]) if variant not in UNPAIRED_F32_FORMS])
def test_gemm_f32_rotates_and_writes_the_cache(tokens, heads, kv_heads, head_dim, normed, tables, variant):
    """The rotation and the cache write behind the product against the kernels of their own on the plain product."""
    ops = _ops()
    torch.manual_seed(tokens + head_dim)
    k, n = 100, (heads + 2 * kv_heads) * head_dim
    x, w, gain = torch.randn(tokens, k).cuda(), torch.randn(n, k).cuda(), (1 + 0.2 * torch.randn(k)).cuda()
    cos, sin = (torch.from_numpy(t).cuda() for t in P.rope_tables(256, head_dim, 10000.0))
    slots = [t % 3 if t % 5 != 4 else -1 for t in range(tokens)]
    positions = [(t // 3) * 3 + 60 for t in range(tokens)]
    table = torch.tensor([[3, 0], [9, 4], [2, 7]], dtype=torch.int32).cuda()
    slot, pos = _i32(slots), _i32(positions)
    pages = [_empty_pages(10, kv_heads, head_dim, torch.float32, 7.0, 7.0, "cuda") for _ in range(2)]
    rows = ops.rmsnorm(x, gain, 1e-5, torch.empty_like(x)) if normed else x
    plain, want, got = torch.empty(tokens, n, device="cuda"), torch.zeros(tokens, heads * head_dim, device="cuda"), torch.zeros(tokens, heads * head_dim, device="cuda")
    ops.gemm_f32(rows, w, plain)
    ops.rope_kv_write(plain, want, cos, sin, head_dim, slot, pos, *pages[0], table, heads, kv_heads, head_dim)
    rope = dict(cos=cos, sin=sin, tok_slot=slot, tok_pos=pos, k_pages=pages[1][0], v_pages=pages[1][1], block_table=table, heads=heads,
                kv_heads=kv_heads, head_dim=head_dim, tables=ops.step_tables(slot, pos, tokens, cos, sin, table) if tables else None)
    ops.gemm_f32_fused(x, w, got, ops.EPILOGUE_ROPE, *((gain, 1e-5) if normed else ()), rope=rope, variant=variant)
    live = torch.tensor([s >= 0 for s in slots])
    bound = 1e-6 * k  # both sides sum k products of normal values in 32 bits
    assert (got - want)[live.cuda()].abs().max().item() <= bound
    for mine, theirs in zip(pages[1], pages[0]):
        assert (mine - theirs).abs().max().item() <= bound


def test_a_32_bit_product_whose_rows_cannot_be_loaded_16_bytes_at_a_time_takes_the_ordered_kernel():
    ops = _ops()
    w = torch.randn(24, 36, device="cuda")
    for x, weight in ((torch.randn(5, 34, device="cuda"), w.flatten()[:24 * 34].view(24, 34)),  # a width that is no multiple of 4
                      (torch.randn(5 * 36 + 1, device="cuda")[1:].view(5, 36), w)):  # rows on no 16-byte boundary
        y, ordered = torch.empty(5, 24, device="cuda"), torch.empty(5, 24, device="cuda")
        assert not ops.gemm_f32_takes(x, weight, y)
        ops.linear(x, weight, y)
        assert torch.equal(y, ops.gemm_ordered(x, weight, ordered))
        with pytest.raises(KernelError):
            ops.gemm_f32(x, weight, y)
    for count in (5, 70):  # the last chunk's lanes beyond K count as zeros whatever the row begins with
        x = torch.randn(count, 36, device="cuda")
        x[2, 0] = float("inf")
        y = torch.empty(count, 24, device="cuda")
        ops.linear(x, w, y)
        assert torch.isfinite(y[[0, 1, 3, 4]]).all() and torch.isinf(y[2]).all()


@pytest.mark.parametrize("m", [1, 8, 16, 17, 40, 64, 65, 130, 300])
@pytest.mark.parametrize("n, k", [(576, 576), (960, 576), (1000, 96), (70, 176), (3072, 64), (64, 1536), (17, 8), (200, 1096),
                                  (2050, 2312)])  # the last: large weights, few columns -- K is cut among blocks beyond 16 tokens
@pytest.mark.parametrize("y_dtype", ["bfloat16", "float32"])
def test_gemm_bf16_on_the_matrix_cores(m, n, k, y_dtype):
    """Skinny (M <= 64) and tiled kernels at sizes with tails in every
    dimension.  Integer-valued operands make the 32-bit sums exact, so any
    misplaced or dropped product shows as a whole-number error."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randint(-3, 4, (m, k)).to(torch.bfloat16)
    w = torch.randint(-3, 4, (n, k)).to(torch.bfloat16)
    y = torch.full((m, n), 7.0, dtype=DT[y_dtype], device="cuda")
    ops.gemm_bf16(x.cuda(), ops.pack_weight(w.cuda()), y)
    want = x.double() @ w.double().t()
    if y_dtype == "float32":
        assert torch.equal(y.cpu().double(), want)
    else:
        assert torch.equal(y.cpu(), want.to(torch.bfloat16))
    # and with ordinary values, against the 64-bit product
    x = torch.randn(m, k).to(torch.bfloat16)
    w = torch.randn(n, k).to(torch.bfloat16)
    ops.gemm_bf16(x.cuda(), ops.pack_weight(w.cuda()), y)
    want = x.double() @ w.double().t()
    scale = x.double().abs() @ w.double().abs().t()
    tol = 1e-6 * math.sqrt(k) if y_dtype == "float32" else 4e-3
    assert ((y.cpu().double() - want).abs() <= tol * scale + 1e-30).all()


@pytest.mark.parametrize("n,k", [(16, 64), (5, 8), (37, 88), (130, 200), (960, 576)])
def test_packed_weight_order(n, k):
    """Element (row, c) of a weight lies in strip row / 16, chunk c / 64, half c % 16 / 8, lane
    16 * (c % 64 / 16) + row % 16, place c % 8; what pads the last strip and chunk is zeros."""
    ops = _ops()
    w = torch.randn(n, k).bfloat16()
    packed = ops.pack_weight(w.cuda())
    assert packed.shape == (n, k) and packed.data.numel() == ops.packed_weight_elems(n, k)
    strips, chunks = (n + 15) // 16, ((k + 63) // 64) | 1  # a strip is padded to an odd number of chunks
    got = packed.data.cpu().view(strips, chunks, 2, 4, 16, 8)  # [strip][chunk][half][k group][row][8]
    padded = torch.zeros(strips * 16, chunks * 64, dtype=torch.bfloat16)
    padded[:n, :k] = w
    want = padded.view(strips, 16, chunks, 4, 2, 8).permute(0, 2, 4, 3, 1, 5)  # [strip][row][chunk][k group][half][8] ->
    assert torch.equal(got, want.contiguous())


def test_gemm_bf16_refuses_what_it_cannot_load():
    ops = _ops()
    x = torch.zeros(4, 12, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(6, 12, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(KernelError, match="multiple of 8"):
        ops.pack_weight(w)
    assert not ops.packs(w)
    with pytest.raises(KernelError, match="must be packed"):  # a weight in the checkpoint's order is not taken for a packed one
        ops.gemm_bf16(x, w, torch.zeros(4, 6, dtype=torch.bfloat16, device="cuda"))
    out = torch.zeros(4, 6, dtype=torch.bfloat16, device="cuda")
    ops.linear(x + 1, w + 1, out)  # a weight that is not packed takes the ordered product
    assert (out == 12).all()


MFMA_SHAPES = [(4, 2, 16), (3, 3, 16), (3, 1, 32), (6, 2, 48), (6, 6, 48), (4, 2, 48), (9, 3, 64), (2, 2, 64), (5, 5, 80),
               (4, 1, 112), (8, 2, 128), (32, 1, 64), (40, 2, 16), (8, 1, 64), (12, 2, 32), (2, 1, 192), (3, 3, 256)]


def _small_decode_call(heads, kv_heads, head_dim):
    """Arguments of a one-token decode call over one page (for calls that are to be refused)."""
    k_pages, v_pages = _empty_pages(1, kv_heads, head_dim, torch.bfloat16, 0.0, 0.0, "cuda")
    q = torch.zeros(1, heads * head_dim, dtype=torch.bfloat16, device="cuda")
    return (q, torch.empty_like(q), k_pages, v_pages, _i32([[0]]), _i32([0]), _i32([0]), heads, kv_heads, head_dim, 1.0)


def _plain_rows(q_rows, ks, vs, scale, window=0):
    """q_rows: list of (slot, pos, q[heads, hd]) -> plain attention output per row."""
    out = []
    for slot, pos, q in q_rows:
        lo = max(0, pos + 1 - window) if window else 0
        full_q = torch.zeros(pos + 1 - lo, *q.shape)
        full_q[-1] = q
        out.append(P.causal_attention(full_q, ks[slot][lo:pos + 1], vs[slot][lo:pos + 1], scale)[-1])
    return torch.stack(out)


@pytest.mark.parametrize("heads, kv_heads, head_dim", MFMA_SHAPES)
@pytest.mark.parametrize("splits, waves", [(1, 1), (4, 1), (16, 2), (1, 8), (2, 4)])
@pytest.mark.parametrize("kernel", ["columns", "keys"])
def test_decode_attention_on_the_matrix_cores(heads, kv_heads, head_dim, splits, waves, kernel):
    ops = _ops()
    if kernel == "keys" and (heads // kv_heads > 4 or head_dim > 128):  # refused, in words
        with pytest.raises(Exception, match="keys on lanes"):
            ops.attention_decode_bf16(*_small_decode_call(heads, kv_heads, head_dim), kernel="keys")
        return
    torch.manual_seed(heads + head_dim)
    lengths = [700, 1, 65, 33]
    ks = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    vs = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    scale = 1.0 / math.sqrt(head_dim)
    q_last = torch.randn(heads, head_dim)
    ks[0][3, 0] = (q_last[0] * (12.0 / scale / q_last[0].pow(2).sum())).bfloat16().float()  # a far key among hundreds
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim)
    rows = [(0, 699, q_last), (1, 0, torch.randn(heads, head_dim)), (-1, 9, torch.randn(heads, head_dim)),
            (2, 64, torch.randn(heads, head_dim)), (3, 31, torch.randn(heads, head_dim))]
    rows = [(s, p, q.bfloat16().float()) for s, p, q in rows]
    q = torch.stack([q for _, _, q in rows]).bfloat16().reshape(len(rows), -1).cuda()
    out = torch.full((len(rows), heads * head_dim), 3.0, dtype=torch.bfloat16, device="cuda")
    partial = torch.full((len(rows) * heads * splits * (head_dim + 4),), float("nan"), dtype=torch.float32, device="cuda")
    waves = min(waves, ops.decode_max_waves(heads, kv_heads, head_dim))
    ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32([s for s, _, _ in rows]), _i32([p for _, p, _ in rows]),
                              heads, kv_heads, head_dim, scale, 0, splits, partial, waves, kernel)
    got = out.cpu().float().view(len(rows), heads, head_dim)
    live = [i for i, (s, _, _) in enumerate(rows) if s >= 0]
    want = _plain_rows([rows[i] for i in live], ks, vs, scale)
    assert (got[live] - want).abs().max().item() <= 2e-2
    assert (got[2] == 3.0).all()  # the padding row is left alone
    assert (got[0, 0] - vs[0][3, 0]).abs().max().item() < 0.05
    # a window: the row at position 699 reads keys 600..699 only
    ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32([s for s, _, _ in rows]), _i32([p for _, p, _ in rows]),
                              heads, kv_heads, head_dim, scale, 100, splits, partial, waves, kernel)
    got = out.cpu().float().view(len(rows), heads, head_dim)
    want = _plain_rows([rows[i] for i in live], ks, vs, scale, window=100)
    assert (got[live] - want).abs().max().item() <= 2e-2


@pytest.mark.parametrize("heads, kv_heads, head_dim", MFMA_SHAPES)
def test_prefill_attention_on_the_matrix_cores(heads, kv_heads, head_dim):
    """Three sequences in one step: a whole prompt, a continuation that starts
    at position 70, and a single token; every new row against the plain
    attention over its sequence's keys up to its own position."""
    ops = _ops()
    torch.manual_seed(heads * 3 + head_dim)
    sequences = [(2, 0, 130), (0, 70, 37), (1, 0, 1)]  # (slot, first new position, new tokens)
    total = {slot: pos0 + n for slot, pos0, n in sequences}
    ks = [torch.randn(total[s], kv_heads, head_dim).bfloat16().float() for s in range(3)]
    vs = [torch.randn(total[s], kv_heads, head_dim).bfloat16().float() for s in range(3)]
    scale = 1.0 / math.sqrt(head_dim)
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim)
    rows = [(slot, pos0 + i, torch.randn(heads, head_dim).bfloat16().float()) for slot, pos0, n in sequences for i in range(n)]
    # one loud key: row 100 of the first sequence must find key 17 (head 0)
    loud_q = rows[100][2][0]
    ks[2][17, 0] = (loud_q * (12.0 / scale / loud_q.pow(2).sum())).bfloat16().float()
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim)
    q = torch.stack([q for _, _, q in rows]).bfloat16().reshape(len(rows), -1).cuda()
    out = torch.full((len(rows), heads * head_dim), 3.0, dtype=torch.bfloat16, device="cuda")
    tile = ops.prefill_tile_rows(heads, kv_heads, head_dim)
    assert tile in (16, 32, 64)
    items = [(seq, row0) for seq, (_, _, n) in enumerate(sequences) for row0 in range(0, n, tile)]
    starts = [0, 130, 167, 168]
    starts = [0, 130, 167, 168]
    for window, waves, columns in ((0, 1, 0), (40, 1, 0), (0, 8, 0), (40, 2, 0), (0, 8, 1), (40, 4, 2), (0, 1, 2)):
        waves = min(waves, ops.prefill_max_waves(heads, kv_heads, head_dim, columns))
        tile = ops.prefill_tile_rows(heads, kv_heads, head_dim, columns)
        items = [(seq, row0) for seq, (_, _, n) in enumerate(sequences) for row0 in range(0, n, tile)]
        ops.attention_prefill_bf16(q, out, k_pages, v_pages, table, _i32([s for s, _ in items]), _i32([r for _, r in items]),
                                   _i32([s for s, _, _ in sequences]), _i32(starts), _i32([p for _, p, _ in sequences]),
                                   heads, kv_heads, head_dim, scale, window, waves, columns)
        got = out.cpu().float().view(len(rows), heads, head_dim)
        want = _plain_rows(rows, ks, vs, scale, window=window)
        error = (got - want).abs().amax(dim=(1, 2))
        assert error.max().item() <= 2e-2, (window, int(error.argmax()), error.max().item())
        if window == 0:
            assert (got[100, 0] - vs[2][17, 0]).abs().max().item() < 0.05


@pytest.mark.parametrize("heads, kv_heads, head_dim, splits, rows_out", [(9, 3, 64, 4, 576), (4, 2, 16, 8, 70), (8, 2, 128, 2, 1024),
                                                                         (5, 5, 80, 3, 200)])
def test_residual_projection_adds_up_key_runs(heads, kv_heads, head_dim, splits, rows_out):
    """A decode attention that leaves its runs of keys, and the projection that
    adds them up on its way: the stream, the prepared norm and its sums are
    those of the path with the kernel of its own between the two, bit for bit
    (a padding row's aside: nobody reads it)."""
    ops = _ops()
    torch.manual_seed(heads + head_dim + splits)
    lengths = [700, 1, 65, 33]
    ks = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    vs = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim)
    slots, positions = [0, 1, -1, 2, 3], [699, 0, 9, 64, 31]
    live = [i for i, s in enumerate(slots) if s >= 0]
    m, k = len(slots), heads * head_dim
    q = torch.randn(m, k).bfloat16().cuda()
    out = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda")
    partial = torch.full((m * heads * splits * (head_dim + 4),), float("nan"), dtype=torch.float32, device="cuda")
    waves = min(2, ops.decode_max_waves(heads, kv_heads, head_dim))
    runs = ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32(slots), _i32(positions), heads, kv_heads, head_dim,
                                     1.0 / math.sqrt(head_dim), 0, splits, partial, waves, keep_runs=True)
    assert isinstance(runs, ops.KeyRuns) and runs.shape == (m, k) and runs.fits(rows_out)
    w = (torch.randn(rows_out, k) / math.sqrt(k)).bfloat16().cuda()
    packed = ops.pack_weight(w)
    gain = (1 + 0.3 * torch.randn(rows_out)).bfloat16().cuda()
    resid = torch.randn(m, rows_out).cuda()

    def project(x):
        mine = resid.clone()
        scaled = torch.zeros(m, rows_out, dtype=torch.bfloat16, device="cuda")
        ss = torch.zeros(ops.gemm_residual_parts(m, rows_out), m, device="cuda")
        parts = ops.gemm_residual(x, packed, mine, gain, scaled, ss)
        return mine[live].cpu(), scaled[live].cpu(), ss[:parts][:, live].cpu()

    fused = project(runs)
    added = runs.combine()
    assert added.data_ptr() == out.data_ptr()
    want = _plain_rows([(slots[i], positions[i], q[i].float().cpu().view(heads, head_dim)) for i in live], ks, vs, 1.0 / math.sqrt(head_dim))
    assert (added[live].cpu().float().view(len(live), heads, head_dim) - want).abs().max().item() <= 2e-2
    apart = project(added)
    for got, expected in zip(fused, apart):
        assert torch.equal(got, expected)
    # runs that the projection does not take: too many of them, or too many tokens
    assert not ops.KeyRuns(partial, 9, m, heads, head_dim, _i32(slots), out).fits(rows_out)
    assert not ops.KeyRuns(partial, splits, 65, heads, head_dim, _i32(slots), out).fits(rows_out)


@pytest.mark.parametrize("heads, kv_heads, head_dim, lengths", [(9, 3, 64, (1500, 700, 90)), (8, 8, 16, (1300, 1000, 100))])
def test_prefill_attention_with_more_items_than_compute_units(heads, kv_heads, head_dim, lengths):
    """Steps of so many tiles that a block takes two of them, a long one and
    then a short one.  The second sequence goes on from position 100.  One
    loud key far back for a row of the shortest tiles and one for a row of
    the longest."""
    ops = _ops()
    torch.manual_seed(heads + head_dim)
    sequences = [(1, 0, lengths[0]), (2, 100, lengths[1]), (0, 0, lengths[2])]  # (slot, first new position, new tokens)
    total = {slot: pos0 + n for slot, pos0, n in sequences}
    ks = [torch.randn(total[s], kv_heads, head_dim).bfloat16().float() for s in range(3)]
    vs = [torch.randn(total[s], kv_heads, head_dim).bfloat16().float() for s in range(3)]
    scale = 1.0 / math.sqrt(head_dim)
    queries = {slot: torch.zeros(total[slot], heads, head_dim) for slot in total}
    for slot, pos0, n in sequences:
        queries[slot][pos0:] = torch.randn(n, heads, head_dim).bfloat16().float()
    loud = [(0, 40, 3), (1, lengths[0] - 2, 70)]  # (slot, position of the row, position of the key), head 0
    for slot, row, key in loud:
        loud_q = queries[slot][row, 0]
        ks[slot][key, 0] = (loud_q * (14.0 / scale / loud_q.pow(2).sum())).bfloat16().float()
    pages = sum((n + 63) // 64 for n in total.values())
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim, pages=pages, max_pages=max(total.values()) // 64 + 1)
    q = torch.cat([queries[slot][pos0:] for slot, pos0, _ in sequences]).bfloat16().reshape(sum(lengths), -1).cuda()
    want = torch.cat([P.causal_attention(queries[slot], ks[slot], vs[slot], scale)[pos0:] for slot, pos0, _ in sequences])
    starts = [0, lengths[0], lengths[0] + lengths[1], sum(lengths)]
    tile = ops.prefill_tile_rows(heads, kv_heads, head_dim)
    items = sorted(((pos0 + min(row0 + tile, n), seq, row0) for seq, (_, pos0, n) in enumerate(sequences)
                    for row0 in range(0, n, tile)), reverse=True)  # longest first, as the engine hands them over
    group_chunks = kv_heads * -(-(heads // kv_heads) // max(1, min(heads // kv_heads, 4)))
    assert len(items) * group_chunks > 256 + 32  # more than the compute units of the chip: the grid folds
    for waves in (8, 2, 1):  # (one wave: each item whole, a block's two one after the other)
        waves = min(waves, ops.prefill_max_waves(heads, kv_heads, head_dim))
        out = torch.full((sum(lengths), heads * head_dim), 3.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_prefill_bf16(q, out, k_pages, v_pages, table, _i32([s for _, s, _ in items]), _i32([r for _, _, r in items]),
                                   _i32([s for s, _, _ in sequences]), _i32(starts), _i32([p for _, p, _ in sequences]),
                                   heads, kv_heads, head_dim, scale, 0, waves)
        got = out.cpu().float().view(sum(lengths), heads, head_dim)
        error = (got - want).abs().amax(dim=(1, 2))
        assert error.max().item() <= 2e-2, (waves, int(error.argmax()), error.max().item())
        for slot, row, key in loud:
            seq = [s for s, _, _ in sequences].index(slot)
            packed = starts[seq] + row - sequences[seq][1]
            assert (got[packed, 0] - vs[slot][key, 0]).abs().max().item() < 0.05


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(9, 3, 64), (32, 4, 64), (4, 4, 32)])
def test_attention_beyond_64_pages(heads, kv_heads, head_dim):
    """A sequence of 4,500 tokens (71 pages: a wave that walks them all comes
    to the end of its first run of page numbers and has to fetch the next),
    with a loud key in the very first page and one beyond page 64, for one
    token of a decode step (one wave and one run, several waves, several runs,
    both kernels) and for the last rows of a prompt step."""
    ops = _ops()
    torch.manual_seed(heads + head_dim)
    length = 4500
    scale = 1.0 / math.sqrt(head_dim)
    ks = [torch.randn(length, kv_heads, head_dim).bfloat16().float(), torch.randn(70, kv_heads, head_dim).bfloat16().float()]
    vs = [torch.randn(length, kv_heads, head_dim).bfloat16().float(), torch.randn(70, kv_heads, head_dim).bfloat16().float()]
    group = heads // kv_heads
    q_last = torch.randn(heads, head_dim).bfloat16().float()
    # head 0 finds key 5 (page 0); the first head of the last group finds key 4,230 (page 66)
    far_head = heads - group
    ks[0][5, 0] = (q_last[0] * (14.0 / scale / q_last[0].pow(2).sum())).bfloat16().float()
    ks[0][4230, kv_heads - 1] = (q_last[far_head] * (14.0 / scale / q_last[far_head].pow(2).sum())).bfloat16().float()
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim, pages=80, max_pages=72)
    rows = [(0, length - 1, q_last), (1, 69, torch.randn(heads, head_dim).bfloat16().float())]
    q = torch.stack([q for _, _, q in rows]).bfloat16().reshape(len(rows), -1).cuda()
    want = _plain_rows(rows, ks, vs, scale)
    kernels = ["columns"] + (["keys"] if group <= 4 else [])
    for kernel in kernels:
        for splits, waves in ((1, 1), (1, 4), (8, 4), (2, 1)):
            waves = min(waves, ops.decode_max_waves(heads, kv_heads, head_dim))
            out = torch.full((len(rows), heads * head_dim), 3.0, dtype=torch.bfloat16, device="cuda")
            partial = torch.full((len(rows) * heads * splits * (head_dim + 4),), float("nan"), dtype=torch.float32, device="cuda")
            ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32([0, 1]), _i32([length - 1, 69]), heads, kv_heads,
                                      head_dim, scale, 0, splits, partial, waves, kernel)
            got = out.cpu().float().view(len(rows), heads, head_dim)
            assert (got - want).abs().max().item() <= 2e-2, (kernel, splits, waves, (got - want).abs().max().item())
            assert (got[0, 0] - vs[0][5, 0]).abs().max().item() < 0.05, (kernel, splits, waves)
            assert (got[0, far_head] - vs[0][4230, kv_heads - 1]).abs().max().item() < 0.05, (kernel, splits, waves)
    # a prompt step: the sequence's last 40 tokens are new, the 4,460 before them are in the cache
    new = 40
    pos0 = length - new
    q_rows = torch.randn(new, heads, head_dim).bfloat16().float()
    q_rows[-1] = q_last
    prompt_rows = [(0, pos0 + i, q_rows[i]) for i in range(new)]
    want = _plain_rows(prompt_rows, ks, vs, scale)
    qp = q_rows.bfloat16().reshape(new, -1).cuda()
    for waves in (1, 8):
        waves = min(waves, ops.prefill_max_waves(heads, kv_heads, head_dim))
        tile = ops.prefill_tile_rows(heads, kv_heads, head_dim)
        items = [(0, row0) for row0 in range(0, new, tile)]
        out = torch.full((new, heads * head_dim), 3.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_prefill_bf16(qp, out, k_pages, v_pages, table, _i32([s for s, _ in items]), _i32([r for _, r in items]),
                                   _i32([0]), _i32([0, new]), _i32([pos0]), heads, kv_heads, head_dim, scale, 0, waves)
        got = out.cpu().float().view(new, heads, head_dim)
        assert (got - want).abs().max().item() <= 2e-2, (waves, (got - want).abs().max().item())
        assert (got[-1, 0] - vs[0][5, 0]).abs().max().item() < 0.05
        assert (got[-1, far_head] - vs[0][4230, kv_heads - 1]).abs().max().item() < 0.05


def test_step_tables_and_the_kernels_that_read_them():
    """The step's tables against plain indexing, padding rows included; the decode attention reading each token's
    pages from them gives what it gives through slots and the block table; the rotating projection that takes
    rotation rows and pages from them writes the same queries and the same cache."""
    ops = _ops()
    torch.manual_seed(11)
    heads, kv_heads, head_dim = 6, 2, 64
    half = head_dim // 2
    lengths = [300, 70, 1, 129]
    ks = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    vs = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim)
    cos, sin = (torch.from_numpy(t).cuda() for t in P.rope_tables(512, head_dim, 10000.0))
    slots, positions = [2, -1, 0, 3, 1, -1], [0, 0, 299, 128, 69, 0]
    tables = ops.step_tables(_i32(slots), _i32(positions), len(slots), cos, sin, table, sequence_pages=True)
    host_table = table.cpu()
    for row, (slot, pos) in enumerate(zip(slots, positions)):
        if slot < 0:
            assert tables.page[row].item() == -1 and tables.pages[row, 0].item() == 0
            assert bool((tables.cos[row] == 1).all()) and bool((tables.sin[row] == 0).all())
            continue
        assert torch.equal(tables.cos[row], cos[pos]) and torch.equal(tables.sin[row], sin[pos])
        assert tables.page[row].item() == host_table[slot, pos // 64].item()
        assert torch.equal(tables.pages[row, :pos // 64 + 1].cpu(), host_table[slot, :pos // 64 + 1])
    only_pages = ops.step_tables(_i32(slots), _i32(positions), len(slots), block_table=table)
    assert only_pages.cos is None and only_pages.pages is None and torch.equal(only_pages.page, tables.page)

    scale = 1.0 / math.sqrt(head_dim)
    q = torch.randn(len(slots), heads * head_dim).bfloat16().cuda()
    for kernel in ("keys", "columns"):
        for splits, waves in ((1, 1), (4, 2)):
            outs = []
            for token_pages in (None, tables.pages):
                out = torch.zeros(len(slots), heads * head_dim, dtype=torch.bfloat16, device="cuda")
                partial = torch.zeros(len(slots) * heads * splits * (head_dim + 4), dtype=torch.float32, device="cuda")
                ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32(slots), _i32(positions), heads, kv_heads, head_dim,
                                          scale, 0, splits, partial, waves, kernel, token_pages=token_pages)
                outs.append(out.cpu())
            live = [i for i, s in enumerate(slots) if s >= 0]
            assert torch.equal(outs[0][live], outs[1][live]), (kernel, splits, waves)

    # the rotating projection: 6 tokens, one a padding row, written at the positions above
    m, k, eps = len(slots), 96, 1e-5
    n = (heads + 2 * kv_heads) * head_dim
    x = torch.randn(m, k)
    gain = (1 + 0.1 * torch.randn(k)).bfloat16()
    w = ops.pack_weight((torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda())
    results = []
    for with_tables in (False, True):
        kp, vp = k_pages.clone(), v_pages.clone()
        rope = dict(cos=cos, sin=sin, tok_slot=_i32(slots), tok_pos=_i32(positions), k_pages=kp, v_pages=vp, block_table=table,
                    heads=heads, kv_heads=kv_heads, head_dim=head_dim, tables=tables if with_tables else None)
        y = torch.zeros(m, heads * head_dim, dtype=torch.bfloat16, device="cuda")
        ops.gemm_fused(x.cuda(), None, None, gain.cuda(), eps, w, y, ops.EPILOGUE_ROPE, rope)
        results.append((y.cpu(), kp.cpu(), vp.cpu()))
    live = [i for i, s in enumerate(slots) if s >= 0]
    assert torch.equal(results[0][0][live], results[1][0][live])
    assert torch.equal(results[0][1], results[1][1]) and torch.equal(results[0][2], results[1][2])
    assert not torch.equal(results[1][1], k_pages.cpu())  # and the cache was written


@pytest.mark.parametrize("hint", [32, 48, 64, 80, 96, 112, 128])
def test_gemm_tiled_over_many_blocks(hint):
    """Each tile of the tiled kernel (64 x 128, 64 x 64, 256 x 256, 256 x 192, 128 x 128, 256 x 128, 128 x 192) over a grid of hundreds of blocks in
    bands and groups, with a ragged edge in every dimension; whole-number
    operands, so a block that took another's rows or columns shows."""
    ops = _ops()
    torch.manual_seed(hint)
    m, n, k = 2300, 1100, 584
    x = torch.randint(-3, 4, (m, k)).to(torch.bfloat16)
    w = torch.randint(-3, 4, (n, k)).to(torch.bfloat16)
    y = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
    ops.gemm_bf16(x.cuda(), ops.pack_weight(w.cuda()), y, hint)
    assert torch.equal(y.cpu().double(), x.double() @ w.double().t())


@pytest.mark.parametrize("m", [1, 8, 19, 64, 67, 100, 300])
@pytest.mark.parametrize("n, k", [(576, 576), (100, 72), (2048, 1536), (48, 8), (64, 176), (3072, 576), (2080, 2304)])
@pytest.mark.parametrize("gain_dtype", ["bfloat16", "float32"])
def test_residual_projection_prepares_the_norm(m, n, k, gain_dtype):
    """resid += x . w^T in place; scaled = bfloat16(resid * gain); the parts of
    ss add up to each row's sum of squares."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m, k).bfloat16()
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    resid = torch.randn(m, n) * 2
    gain = (1 + 0.3 * torch.randn(n)).to(DT[gain_dtype])
    want = resid.double() + x.double() @ w.double().t()
    resid_gpu = resid.cuda()
    scaled = torch.full((m, n), 9.0, dtype=torch.bfloat16, device="cuda")
    rows = ops.gemm_residual_parts(m, n)
    ss = torch.full((rows + 1, m), 7.0, device="cuda")
    parts = ops.gemm_residual(x.cuda(), ops.pack_weight(w.cuda()), resid_gpu, gain.cuda(), scaled, ss)
    assert 0 < parts <= rows
    assert (ss[parts:] == 7.0).all()  # nothing beyond the parts it names
    got = resid_gpu.cpu().double()
    assert ((got - want).abs() <= 1e-5 * (1 + want.abs())).all(), (got - want).abs().max().item()
    # scaled is the rounding of the 32-bit product of the new residual and the gain
    exact = (resid_gpu.cpu() * gain.float()).bfloat16()
    assert torch.equal(scaled.cpu(), exact)
    total = ss[:parts].cpu().double().sum(dim=0)
    assert ((total - got.pow(2).sum(dim=1)).abs() <= 1e-5 * got.pow(2).sum(dim=1)).all()


@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("n, k", [(2048, 5632), (1990, 5128), (48, 8192), (2048, 5120)])
def test_residual_projection_with_two_blocks_a_strip(m, n, k):
    """Up to 16 tokens on few strips and a long K (from 5,120 on): two blocks share each strip, and the second
    to be done adds the sums of the first to its own.  Three calls in a row on the same stream, with a tiled
    product that cuts its K into parts (and fills the workspace they share) between them: each is right, and
    the strips' counts are back at zero."""
    ops = _ops()
    assert ops.gemm_takes_pair(m, n, k)  # the kernel under test is the one that runs (and not at sizes beside its rule)
    assert not ops.gemm_takes_pair(17, n, k) and not ops.gemm_takes_pair(m, n, 5056) and not ops.gemm_takes_pair(m, 2064, k)
    torch.manual_seed(m + n + k)
    gain = (1 + 0.3 * torch.randn(n)).bfloat16()
    other_x = torch.randn(64, 4096).bfloat16().cuda()
    other_w = ops.pack_weight((torch.randn(2048, 4096) / 64).bfloat16().cuda())
    other_y = torch.empty(64, 2048, dtype=torch.bfloat16, device="cuda")
    rows = ops.gemm_residual_parts(m, n)
    for call in range(3):
        x = torch.randn(m, k).bfloat16()
        w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
        resid = torch.randn(m, n) * 2
        want = resid.double() + x.double() @ w.double().t()
        resid_gpu = resid.cuda()
        scaled = torch.full((m, n), 9.0, dtype=torch.bfloat16, device="cuda")
        ss = torch.full((rows + 1, m), 7.0, device="cuda")
        parts = ops.gemm_residual(x.cuda(), ops.pack_weight(w.cuda()), resid_gpu, gain.cuda(), scaled, ss)
        ops.gemm_bf16(other_x, other_w, other_y)  # 64 tokens on 2048 x 4096: K in parts, through the workspace
        assert 0 < parts <= rows and (ss[parts:] == 7.0).all()
        got = resid_gpu.cpu().double()
        assert ((got - want).abs() <= 1e-5 * (1 + want.abs())).all(), (call, (got - want).abs().max().item())
        assert torch.equal(scaled.cpu(), (resid_gpu.cpu() * gain.float()).bfloat16())
        total = ss[:parts].cpu().double().sum(dim=0)
        assert ((total - got.pow(2).sum(dim=1)).abs() <= 1e-5 * got.pow(2).sum(dim=1)).all()
        counts = ops.gemm_pair_counts(resid_gpu.device)
        assert counts.numel() == ops.PAIR_COUNTS and int(counts.abs().sum()) == 0


@pytest.mark.parametrize("tile", ["TILE_64x128", "TILE_64x64", "TILE_256x256", "TILE_256x192", "TILE_128x128", "TILE_256x128", "TILE_128x192"])
@pytest.mark.parametrize("m, n, k", [(70, 600, 136), (530, 300, 72), (300, 1100, 584), (300, 1100, 1800), (70, 600, 1992)])
def test_residual_projection_with_every_tile(tile, m, n, k):
    """The tiled kernel's residual epilogue with each tile shape (several row
    and column blocks, ragged edges): the stream, the prepared operand and the
    parts of the sums of squares, one per wave column."""
    ops = _ops()
    torch.manual_seed(m + n)
    x = torch.randn(m, k).bfloat16()
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    resid = torch.randn(m, n) * 2
    gain = (1 + 0.3 * torch.randn(n)).bfloat16()
    want = resid.double() + x.double() @ w.double().t()
    resid_gpu = resid.cuda()
    scaled = torch.full((m, n), 9.0, dtype=torch.bfloat16, device="cuda")
    rows = ops.gemm_residual_parts(m, n)
    ss = torch.full((rows + 1, m), 7.0, device="cuda")
    parts = ops.gemm_residual(x.cuda(), ops.pack_weight(w.cuda()), resid_gpu, gain.cuda(), scaled, ss, getattr(ops, tile))
    width = {"TILE_64x128": 64, "TILE_64x64": 32, "TILE_256x256": 128, "TILE_256x192": 96, "TILE_128x128": 64, "TILE_256x128": 64, "TILE_128x192": 96}[tile]  # columns of a part
    if parts != 2 * ((n + 2 * width - 1) // (2 * width)):  # few tiles and a long K: K went in parts, summed per 64 columns
        assert tile in ("TILE_64x128", "TILE_64x64") and k >= 512 and parts == (n + 63) // 64
        width = 64
    assert (ss[parts:] == 7.0).all()
    got = resid_gpu.cpu().double()
    assert ((got - want).abs() <= 1e-5 * (1 + want.abs())).all(), (got - want).abs().max().item()
    assert torch.equal(scaled.cpu(), (resid_gpu.cpu() * gain.float()).bfloat16())
    for part in range(parts):
        columns = got[:, part * width:(part + 1) * width]
        assert ((ss[part].cpu().double() - columns.pow(2).sum(dim=1)).abs() <= 1e-5 * (1e-3 + columns.pow(2).sum(dim=1))).all(), part


@pytest.mark.parametrize("m", [1, 8, 16, 17, 40, 64, 65, 200, 300])
@pytest.mark.parametrize("k", [64, 96, 576, 1096])
@pytest.mark.parametrize("with_delta", [False, True, "prepared"])
@pytest.mark.parametrize("gain_dtype", ["bfloat16", "float32"])
def test_fused_norm_projection(m, k, with_delta, gain_dtype):
    """Residual sum + RMSNorm + projection in one kernel, with each epilogue,
    against the plain functions one after another.  "prepared": the sum and
    the first half of the norm are taken by the projection before (here one by
    the identity, so that it adds ``delta`` itself), the second half by the
    kernel under test."""
    ops = _ops()
    prepared = with_delta == "prepared"
    with_delta = bool(with_delta)
    if m > 64 and not prepared:
        pytest.skip("the kernel that takes the sum and the norm itself is for up to 64 tokens")
    torch.manual_seed(m * 7 + k)
    eps = 2e-5
    x = torch.randn(m, k) * 2
    delta = torch.randn(m, k).bfloat16() if with_delta else None
    gain = (1 + 0.3 * torch.randn(k)).to(DT[gain_dtype])
    summed = x + (delta.float() if with_delta else 0)
    normed = P.rms_norm(summed.double(), gain.double(), eps)

    if prepared:
        resid = x.cuda()
        scaled = torch.empty(m, k, dtype=torch.bfloat16, device="cuda")
        ss = torch.empty(ops.gemm_residual_parts(m, k), m, device="cuda")
        parts = ops.gemm_residual(delta.cuda(), ops.pack_weight(torch.eye(k).bfloat16().cuda()), resid, gain.cuda(), scaled, ss)
        assert torch.equal(resid.cpu(), summed)

    def run(w, y, epilogue, rope=None):
        if prepared:
            ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, epilogue, rope)
            return y.cpu().double()
        x_out = torch.full((m, k), 9.0, device="cuda") if with_delta else None
        ops.gemm_fused(x.cuda(), delta.cuda() if with_delta else None, x_out, gain.cuda(), eps, ops.pack_weight(w.cuda()), y, epilogue, rope)
        if with_delta:
            assert torch.equal(x_out.cpu(), summed)  # the residual sum, exactly, written once
        return y.cpu().double()

    def close(got, want, what):
        assert ((got - want).abs() <= 2e-2 * (1 + want.abs())).all(), (what, (got - want).abs().max().item())

    # store, with a ragged last strip
    n = 70
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    close(run(w, torch.empty(m, n, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_STORE), normed @ w.double().t(), "store")
    # gate rows, then up rows
    inner = 88
    w = (torch.randn(2 * inner, k) / math.sqrt(k)).bfloat16()
    both = normed @ w.double().t()
    close(run(w, torch.empty(m, inner, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_SILU),
          P.silu(both[:, :inner]) * both[:, inner:], "silu")
    # queries, keys, values: rotation and the cache
    heads, kv_heads, head_dim = 3, 2, 32
    w = (torch.randn((heads + 2 * kv_heads) * head_dim, k) / math.sqrt(k)).bfloat16()
    qkv = (normed @ w.double().t()).view(m, heads + 2 * kv_heads, head_dim)
    cos_np, sin_np = P.rope_tables(512, head_dim, 10000.0)
    slots = [(i * 5) % 7 - (1 if i % 9 == 4 else 0) * 100 for i in range(m)]  # some padding rows
    slots = [s if s >= 0 else -1 for s in slots]
    positions = [(i * 37) % 320 for i in range(m)]  # no two tokens at one position (37 and 320 share no factor)
    table = torch.arange(7 * 5, dtype=torch.int32).view(7, 5).flip(0).contiguous()
    k_pages, v_pages = _empty_pages(35, kv_heads, head_dim, torch.bfloat16, 7.0, 7.0, "cuda")
    rope = dict(cos=torch.from_numpy(cos_np).cuda(), sin=torch.from_numpy(sin_np).cuda(), tok_slot=_i32(slots),
                tok_pos=_i32(positions), k_pages=k_pages, v_pages=v_pages, block_table=table.cuda(), heads=heads,
                kv_heads=kv_heads, head_dim=head_dim)
    got_q = run(w, torch.empty(m, heads * head_dim, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_ROPE, rope)
    pos = torch.tensor(positions)
    turned = P.rope_rotate_half(qkv[:, :heads + kv_heads], torch.from_numpy(cos_np)[pos].double(), torch.from_numpy(sin_np)[pos].double())
    close(got_q.view(m, heads, head_dim), turned[:, :heads], "queries")
    seen = {}
    for t in range(m):  # a later token of the same slot and position overwrites an earlier one
        if slots[t] >= 0:
            seen[(slots[t], positions[t])] = t
    k_plain, v_plain = _read_pages(k_pages, v_pages, head_dim)
    for (slot, position), t in seen.items():
        page, inside = table[slot, position // 64].item(), position % 64
        close(k_plain[page, :, inside, :].double(), turned[t, heads:], "keys")
        close(v_plain[page, :, inside, :].double(), qkv[t, heads + kv_heads:], "values")
    written = sum(1 for _ in seen)
    assert int((k_plain != 7.0).any(dim=-1).sum()) <= written * kv_heads
    assert int((v_plain != 7.0).any(dim=-1).sum()) <= written * kv_heads


@pytest.mark.parametrize("hint", [32, 48, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("m", [65, 200, 530])
def test_scaled_projection_with_every_tile(hint, m):
    """The tiled kernel's epilogues with each of its tile shapes (the hint picks
    one): pairs of strips in a wave, one or two of them."""
    ops = _ops()
    torch.manual_seed(hint + m)
    k, eps = 96, 1e-5
    v = torch.randn(m, k) * 2
    gain = (1 + 0.3 * torch.randn(k)).bfloat16()
    normed = P.rms_norm(v.double(), gain.double(), eps)
    resid = v.cuda()
    scaled = torch.empty(m, k, dtype=torch.bfloat16, device="cuda")
    ss = torch.empty(ops.gemm_residual_parts(m, k), m, device="cuda")
    parts = ops.gemm_residual(torch.zeros(m, 8, dtype=torch.bfloat16, device="cuda"), ops.pack_weight(torch.zeros(k, 8, dtype=torch.bfloat16, device="cuda")),
                              resid, gain.cuda(), scaled, ss)

    def close(got, want, what):
        assert ((got - want).abs() <= 2e-2 * (1 + want.abs())).all(), (what, (got - want).abs().max().item())

    n = 300
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    y = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    close(ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, ops.EPILOGUE_STORE, None, hint).cpu().double(), normed @ w.double().t(), "store")
    inner = 200
    w = (torch.randn(2 * inner, k) / math.sqrt(k)).bfloat16()
    both = normed @ w.double().t()
    y = torch.empty(m, inner, dtype=torch.bfloat16, device="cuda")
    close(ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, ops.EPILOGUE_SILU, None, hint).cpu().double(),
          P.silu(both[:, :inner]) * both[:, inner:], "silu")
    heads, kv_heads, head_dim = 5, 2, 64
    w = (torch.randn((heads + 2 * kv_heads) * head_dim, k) / math.sqrt(k)).bfloat16()
    qkv = (normed @ w.double().t()).view(m, heads + 2 * kv_heads, head_dim)
    cos_np, sin_np = P.rope_tables(1024, head_dim, 10000.0)
    positions = [(i * 37) % 1024 for i in range(m)]  # no two tokens at one place
    slots = [0 if i % 11 else -1 for i in range(m)]
    table = _i32([[3, 1, 0, 2, 15, 14, 4, 5, 13, 6, 12, 7, 11, 8, 10, 9]])
    k_pages, v_pages = _empty_pages(16, kv_heads, head_dim, torch.bfloat16, 7.0, 7.0, "cuda")
    rope = dict(cos=torch.from_numpy(cos_np).cuda(), sin=torch.from_numpy(sin_np).cuda(), tok_slot=_i32(slots),
                tok_pos=_i32(positions), k_pages=k_pages, v_pages=v_pages, block_table=table, heads=heads,
                kv_heads=kv_heads, head_dim=head_dim)
    y = torch.empty(m, heads * head_dim, dtype=torch.bfloat16, device="cuda")
    got_q = ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, ops.EPILOGUE_ROPE, rope, hint).cpu().double()
    pos = torch.tensor(positions)
    turned = P.rope_rotate_half(qkv[:, :heads + kv_heads], torch.from_numpy(cos_np)[pos].double(), torch.from_numpy(sin_np)[pos].double())
    close(got_q.view(m, heads, head_dim), turned[:, :heads], "queries")
    k_plain, v_plain = _read_pages(k_pages, v_pages, head_dim)
    written = 0
    for t in range(m):
        if slots[t] < 0:
            continue
        written += 1
        page, inside = table[0, positions[t] // 64].item(), positions[t] % 64
        close(k_plain[page, :, inside, :].double(), turned[t, heads:], "keys")
        close(v_plain[page, :, inside, :].double(), qkv[t, heads + kv_heads:], "values")
    assert int((k_plain != 7.0).any(dim=-1).sum()) <= written * kv_heads  # padding rows wrote nothing


@pytest.mark.parametrize("m", [1, 8, 16, 30])
@pytest.mark.parametrize("n, paired", [(8192, False), (11264, False), (32000, False), (2 * 4096, True), (2 * 5632, True), (2 * 14336, True)])
def test_prepared_projection_on_wide_weights(n, paired, m):
    """Few tokens on a prepared operand over hundreds to thousands of strips of 16 weight rows, where the
    number of waves that share a strip's K goes from 8 to 4, 2 and 1 with the width: every width the rule
    tells apart, with the sizes' own choice."""
    ops = _ops()
    torch.manual_seed(n + m)
    k, eps = 2048, 1e-5
    v = torch.randn(m, k) * 2
    gain = (1 + 0.3 * torch.randn(k)).bfloat16()
    normed = P.rms_norm(v.double(), gain.double(), eps)
    scaled = torch.empty(m, k, dtype=torch.bfloat16, device="cuda")
    ss = torch.empty(ops.gemm_residual_parts(m, k), m, device="cuda")
    parts = ops.gemm_residual(torch.zeros(m, 8, dtype=torch.bfloat16, device="cuda"), ops.pack_weight(torch.zeros(k, 8, dtype=torch.bfloat16, device="cuda")),
                              v.cuda(), gain.cuda(), scaled, ss)
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    both = normed @ w.double().t()
    if paired:
        want = P.silu(both[:, :n // 2]) * both[:, n // 2:]
        y = torch.empty(m, n // 2, dtype=torch.bfloat16, device="cuda")
        got = ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, ops.EPILOGUE_SILU).cpu().double()
    else:
        want = both
        y = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        got = ops.gemm_scaled(scaled, ss, parts, eps, ops.pack_weight(w.cuda()), y, ops.EPILOGUE_STORE).cpu().double()
    assert ((got - want).abs() <= 2e-2 * (1 + want.abs())).all(), (got - want).abs().max().item()


def _k_index(head_dim):
    """[64 tokens, head_dim] -> offset of each (token, channel) in a page's keys of one head."""
    t = torch.arange(64).view(64, 1)
    c = torch.arange(head_dim).view(1, head_dim)
    return (c // 8) * 512 + t * 8 + c % 8


def _v_index(head_dim):
    t = torch.arange(64).view(64, 1)
    c = torch.arange(head_dim).view(1, head_dim)
    return ((((c // 16) * 2 + t // 32) * 4 + (t % 32) // 8) * 16 + c % 16) * 8 + t % 8


def _empty_pages(pages, kv_heads, head_dim, dtype, k_fill, v_fill, device="cpu"):
    k_pages = torch.full((pages, kv_heads, (head_dim + 7) // 8, 64, 8), k_fill, dtype=dtype, device=device)
    v_pages = torch.full((pages, kv_heads, (head_dim + 15) // 16, 2, 4, 16, 8), v_fill, dtype=dtype, device=device)
    return k_pages, v_pages


def _read_pages(k_pages, v_pages, head_dim):
    """Pages back in plain order: keys and values as [pages, kv_heads, 64 tokens, head_dim]."""
    pages, kv_heads = k_pages.shape[:2]
    k = k_pages.cpu().float().reshape(pages, kv_heads, -1)[:, :, _k_index(head_dim)]
    v = v_pages.cpu().float().reshape(pages, kv_heads, -1)[:, :, _v_index(head_dim)]
    return k, v


def _paged(k_seqs, v_seqs, dtype, kv_heads, head_dim, page_order=None, pages=32, max_pages=12):
    """Lays sequences out in pages the way the cache does.  k_seqs[i]: [len, kv_heads, head_dim]."""
    k_pages, v_pages = _empty_pages(pages, kv_heads, head_dim, dtype, 77.0, -55.0)
    k_flat, v_flat = k_pages.view(pages, kv_heads, -1), v_pages.view(pages, kv_heads, -1)
    k_index, v_index = _k_index(head_dim), _v_index(head_dim)
    table = torch.zeros(len(k_seqs), max_pages, dtype=torch.int32)
    order = list(page_order or range(pages))
    for slot, (k, v) in enumerate(zip(k_seqs, v_seqs)):
        for page_index in range((k.shape[0] + 63) // 64):
            page = order.pop()
            table[slot, page_index] = page
            chunk = slice(page_index * 64, min(k.shape[0], page_index * 64 + 64))
            n = chunk.stop - chunk.start
            k_flat[page][:, k_index[:n]] = k[chunk].transpose(0, 1).to(dtype)
            v_flat[page][:, v_index[:n]] = v[chunk].transpose(0, 1).to(dtype)
    return k_pages.cuda(), v_pages.cuda(), table.cuda()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads, kv_heads, head_dim", [(4, 2, 16), (3, 1, 32), (9, 3, 64), (5, 5, 80), (8, 2, 128), (2, 1, 192), (3, 3, 256)])
def test_attention_over_pages(dtype, heads, kv_heads, head_dim):
    """Queries at the end of three sequences of unequal length (and one in the
    middle of a sequence), pages handed out in reverse order."""
    ops = _ops()
    torch.manual_seed(heads * head_dim)
    lengths = [700, 1, 65]
    ks = [torch.randn(n, kv_heads, head_dim) for n in lengths]
    vs = [torch.randn(n, kv_heads, head_dim) for n in lengths]
    scale = 1.0 / math.sqrt(head_dim)
    # a far key among hundreds: position 3 of sequence 0 answers the last query of head 0 and nothing else does
    q_last = torch.randn(heads, head_dim)
    ks[0][3, 0] = q_last[0] * (12.0 / scale / q_last[0].pow(2).sum())
    if dtype == "bfloat16":
        ks = [k.bfloat16().float() for k in ks]
        vs = [v.bfloat16().float() for v in vs]
    k_pages, v_pages, table = _paged(ks, vs, DT[dtype], kv_heads, head_dim)
    queries = [(0, 699, q_last), (1, 0, torch.randn(heads, head_dim)), (2, 64, torch.randn(heads, head_dim)),
               (0, 130, torch.randn(heads, head_dim)), (-1, 5, torch.randn(heads, head_dim))]
    q = torch.stack([qq for _, _, qq in queries]).to(DT[dtype])
    out = torch.full((len(queries), heads * head_dim), 3.0, dtype=DT[dtype], device="cuda")
    ops.attention_rows(q.reshape(len(queries), -1).cuda(), out, k_pages, v_pages, table, _i32([s for s, _, _ in queries]),
                       _i32([p for _, p, _ in queries]), heads, kv_heads, head_dim, scale)
    out = out.cpu().float().view(len(queries), heads, head_dim)
    tol = 2e-5 if dtype == "float32" else 2e-2
    for row, (slot, pos, _) in enumerate(queries):
        if slot < 0:
            assert (out[row] == 0).all()  # a padding row
            continue
        full_q = torch.zeros(pos + 1, heads, head_dim)
        full_q[pos] = q[row].float()
        want = P.causal_attention(full_q, ks[slot][:pos + 1], vs[slot][:pos + 1], scale)[pos]
        assert (out[row] - want).abs().max().item() <= tol, (row, (out[row] - want).abs().max().item())
    # the far key dominates head 0 of the first query: its value comes back almost alone
    assert (out[0, 0] - vs[0][3, 0]).abs().max().item() < 0.05


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_attention_window_edge(dtype):
    """With a window of w the query at p reads keys p-w+1 .. p: a loud key just
    outside changes nothing, the same key just inside takes over."""
    ops = _ops()
    heads, kv_heads, head_dim, window, pos = 2, 1, 32, 100, 300
    torch.manual_seed(5)
    scale = 1.0 / math.sqrt(head_dim)
    q = torch.randn(1, heads, head_dim)
    loud = q[0, 0] * (15.0 / scale / q[0, 0].pow(2).sum())
    for where, inside in ((pos - window, False), (pos - window + 1, True)):
        k, v = torch.randn(pos + 1, kv_heads, head_dim), torch.randn(pos + 1, kv_heads, head_dim)
        k[where, 0] = loud
        if dtype == "bfloat16":
            k, v = k.bfloat16().float(), v.bfloat16().float()
        k_pages, v_pages, table = _paged([k], [v], DT[dtype], kv_heads, head_dim)
        out = torch.empty(1, heads * head_dim, dtype=DT[dtype], device="cuda")
        ops.attention_rows(q.reshape(1, -1).to(DT[dtype]).cuda(), out, k_pages, v_pages, table, _i32([0]), _i32([pos]), heads,
                           kv_heads, head_dim, scale, window=window)
        lo = pos - window + 1
        full_q = torch.zeros(window, heads, head_dim)
        full_q[-1] = q[0].to(DT[dtype]).float()
        want = P.causal_attention(full_q, k[lo:], v[lo:], scale)[-1]
        got = out.cpu().float().view(heads, head_dim)
        assert (got - want).abs().max().item() <= (2e-5 if dtype == "float32" else 2e-2)
        assert ((got[0] - v[where, 0]).abs().max().item() < 0.05) == inside


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads, kv_heads, head_dim, rot_dim", [(4, 2, 16, 16), (3, 1, 32, 32), (2, 2, 48, 16), (1, 1, 64, 0)])
def test_rope_and_cache_write(dtype, heads, kv_heads, head_dim, rot_dim):
    ops = _ops()
    torch.manual_seed(rot_dim + heads)
    tokens = 6
    slots = [2, 2, 0, -1, 1, 2]
    positions = [63, 64, 5, 9, 130, 200]
    width = (heads + 2 * kv_heads) * head_dim
    qkv = torch.randn(tokens, width).to(DT[dtype])
    table = torch.tensor([[3, 0, 0, 0], [9, 4, 6, 0], [1, 7, 2, 5]], dtype=torch.int32)
    k_pages, v_pages = _empty_pages(10, kv_heads, head_dim, DT[dtype], 7.0, 7.0, "cuda")
    q_out = torch.full((tokens, heads * head_dim), 5.0, dtype=DT[dtype], device="cuda")
    cos = sin = None
    if rot_dim:
        c, s = P.rope_tables(256, rot_dim, 10000.0)
        cos, sin = torch.from_numpy(c).cuda(), torch.from_numpy(s).cuda()
    ops.rope_kv_write(qkv.cuda(), q_out, cos, sin, rot_dim, _i32(slots), _i32(positions), k_pages, v_pages, table.cuda(),
                      heads, kv_heads, head_dim)
    x = qkv.float().view(tokens, heads + 2 * kv_heads, head_dim)
    rotated = x[:, :heads + kv_heads].clone()
    if rot_dim:
        pos = torch.tensor(positions)
        turned = P.rope_rotate_half(rotated[..., :rot_dim], torch.from_numpy(c)[pos], torch.from_numpy(s)[pos])
        rotated = torch.cat([turned, rotated[..., rot_dim:]], dim=-1)
    tol = 1e-6 if dtype == "float32" else 1e-2
    touched_k = torch.zeros(10, 64, dtype=torch.bool)
    k_plain, v_plain = _read_pages(k_pages, v_pages, head_dim)  # [pages, kv_heads, 64, head_dim]
    for t in range(tokens):
        if slots[t] < 0:
            assert (q_out[t] == 5.0).all()
            continue
        assert (q_out[t].cpu().float().view(heads, head_dim) - rotated[t, :heads]).abs().max() <= tol
        page, inside = table[slots[t], positions[t] // 64].item(), positions[t] % 64
        touched_k[page, inside] = True
        assert (k_plain[page, :, inside, :] - rotated[t, heads:]).abs().max() <= tol
        assert torch.equal(v_plain[page, :, inside, :], x[t, heads + kv_heads:])  # values are copied as they are
    # nothing else in the cache was written (padding of a page's last chunk included)
    assert (k_plain[~touched_k.unsqueeze(1).expand(-1, kv_heads, -1)] == 7.0).all()
    assert (v_plain[~touched_k.unsqueeze(1).expand(-1, kv_heads, -1)] == 7.0).all()
    assert int((k_pages != 7.0).sum()) <= int(touched_k.sum()) * kv_heads * head_dim
    assert int((v_pages != 7.0).sum()) <= int(touched_k.sum()) * kv_heads * head_dim
    # a run that keeps no cache rotates the queries only
    q_only = torch.empty_like(q_out)
    ops.rope_kv_write(qkv.cuda(), q_only, cos, sin, rot_dim, _i32([0] * tokens), _i32(positions), None, None, None,
                      heads, kv_heads, head_dim)
    assert (q_only.cpu().float().view(tokens, heads, head_dim) - rotated[:, :heads]).abs().max() <= tol


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_silu_mul(dtype):
    ops = _ops()
    gate_up = (torch.randn(13, 2 * 177) * 3).to(DT[dtype])
    out = torch.empty(13, 177, dtype=DT[dtype], device="cuda")
    ops.silu_mul(gate_up.cuda(), out)
    want = P.silu(gate_up[:, :177].double()) * gate_up[:, 177:].double()
    assert ((out.cpu().double() - want).abs() <= (1e-6 if dtype == "float32" else 1e-2) * (1 + want.abs())).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("columns, rest, k", [(16, 1, 8), (16, 16, 64), (128, 32, 4096), (48, 33, 200), (3072, 8, 2048)])
def test_two_products_in_one_launch(columns, rest, k, dtype):
    """The same numbers as apart."""
    from nnis_amd.parts.linear import ProjectionPair
    from nnis_amd.engine.runtime import Runtime

    rt = Runtime(dtype="bfloat16")
    torch.manual_seed(columns + k)
    weights = [torch.randn(n, k, device="cuda").bfloat16() for n in (columns, rest)]
    pair = ProjectionPair(*weights, rt)
    assert pair.joined is not None
    for rows in (1, 4, 16, 17):
        x = torch.randn(rows, k, device="cuda").bfloat16()
        first, second = pair(x, rt, second_dtype=dtype)
        assert torch.equal(first, pair.first(x, rt)) and torch.equal(second, pair.second(x, rt, out_dtype=dtype))
        assert torch.allclose(second.float(), x.float() @ weights[1].float().t(), rtol=0.02, atol=0.02 * k ** 0.5)  # (2^-8 of a result and more)
    with pytest.raises(KernelError):
        rt.ops.gemm_two(x, pair.joined, first, second)  # 17 rows


@pytest.mark.parametrize("vocab", [1, 63, 1000, 49152, 50001])
def test_argmax(vocab):
    ops = _ops()
    torch.manual_seed(vocab)
    logits = torch.randn(5, vocab)
    if vocab >= 63:
        logits[0, 40] = logits[0, 7] = 9.0  # a tie: the lower index wins
        logits[1, vocab - 1] = 11.0
        logits[2] = 0.5  # all equal: index 0
        logits[3, 3] = float("nan")
        logits[3, 20] = 30.0
    if vocab > 9000:
        logits[4, 8999] = logits[4, 100] = 12.0  # a tie between two blocks' shares of the row
    out = torch.empty(5, dtype=torch.int32, device="cuda")
    ops.argmax(logits.cuda(), out)
    want = [int(np.nanargmax(row)) for row in logits.numpy()]
    assert out.cpu().tolist() == want
    if vocab >= 63:
        assert want[:3] == [7, vocab - 1, 0]
    if vocab > 9000:
        assert want[4] == 100


def test_refusals():
    ops = _ops()
    f = lambda *shape, dtype=torch.float32: torch.zeros(*shape, dtype=dtype, device="cuda")  # noqa: E731
    with pytest.raises(KernelError, match="ss has 1 rows"):  # scratch too small for the parts it would write
        ops.gemm_residual(f(70, 176, dtype=torch.bfloat16), ops.pack_weight(f(64, 176, dtype=torch.bfloat16)), f(70, 64),
                          f(64, dtype=torch.bfloat16), f(70, 64, dtype=torch.bfloat16), f(1, 70))
    with pytest.raises(KernelError):
        ops.gemm_ordered(f(3, 8), f(5, 9), f(3, 5))
    with pytest.raises(KernelError, match="GPU"):
        ops.gemm_ordered(torch.zeros(3, 8), f(5, 8), f(3, 5))
    with pytest.raises(KernelError, match="float32 or bfloat16"):
        ops.gemm_ordered(f(3, 8, dtype=torch.float16), f(5, 8), f(3, 5))
    from nnis_amd.errors import Unsupported

    for head_dim in (258, 0, -2):  # a size nobody runs: said as such (the model's check at load raises the same)
        with pytest.raises(Unsupported, match="head_dim"):
            ops.attention_module(head_dim)
    with pytest.raises(KernelError):
        ops.silu_mul(f(4, 11), f(4, 5))
    with pytest.raises(KernelError):
        ops.argmax(f(4, 11), torch.zeros(4, dtype=torch.int64, device="cuda"))


def test_the_tiles_that_products_are_given():
    """The tiled kernel's choice of tile by the product's sizes, at the sizes its rules were measured on (the
    library's own host code: no launch)."""
    ops = _ops()
    T = ops
    for (m, n, k), tile in {
        (2048, 16384, 2048): T.TILE_256x256,  # two full rounds of large tiles
        (2048, 6144, 2048): T.TILE_256x192,   # 256 blocks of 192 columns, where 256 columns make 192
        (1024, 11264, 2048): T.TILE_256x192,  # 236 blocks
        (512, 16384, 2048): T.TILE_256x128,   # 256 blocks where tiles of 256 x 192 make 172
        (384, 16384, 2048): T.TILE_256x128,   # rows that fill three quarters of their blocks: enough for a three-stage tile
        (320, 16384, 2048): T.TILE_64x128,    # ... and rows that do not (the blocks of 128 rows would be 384: a round and a half)
        (4096, 4096, 4096): T.TILE_256x256,   # a large tile that fills its round stays
        (4096, 2048, 8192): T.TILE_256x128,   # 256 blocks, one a compute unit, where large tiles would be 176
        (2048, 4096, 14336): T.TILE_256x128,
        (2048, 2048, 8192): T.TILE_128x128,   # 256 blocks of 128 rows where 256 rows make 128
        (2048, 2048, 512): T.TILE_64x128,     # ... over a short K the small tiles
        (2048, 2560, 2048): T.TILE_128x192,   # 224 tiles, where 256 x 128 makes 160 and 128 x 128 a round and a quarter
        (1536, 2560, 2048): T.TILE_128x128,
        (2048, 3072, 2048): T.TILE_128x192,   # a full round of 128 x 192 before three quarters of one of 256 x 128
        (1536, 4096, 4096): T.TILE_256x128,   # three quarters of a round (eleven sixteenths are enough)
        (1024, 6144, 2048): T.TILE_128x192,
        (2048, 1536, 2048): T.TILE_128x128,
        (3072, 2048, 4096): T.TILE_256x128,   # (192 blocks, where 128 x 128 would make a round and a half)
        (1024, 2048, 2048): T.TILE_64x64,     # no more than one wide block a compute unit: the narrow tile
        (2048, 576, 1536): T.TILE_64x64,
        (2048, 3072, 576): T.TILE_64x128,
    }.items():
        assert ops.gemm_tile(m, n, k) == tile, (m, n, k, ops.gemm_tile(m, n, k))


def test_the_tile_of_a_product_into_the_stream_by_the_parts_it_leaves():
    ops = _ops()
    for m, n, k, width in ((4096, 4096, 14336, 128), (2048, 8192, 2048, 256)):  # (another tile than a product that is stored takes, and the same)
        assert {ops.TILE_256x128: 128, ops.TILE_256x256: 256}[ops.gemm_tile(m, n, k, residual=True)] == width
        x, w = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda"), ops.pack_weight(torch.zeros(n, k, dtype=torch.bfloat16, device="cuda"))
        resid, scaled = torch.ones(m, n, device="cuda"), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        ss = torch.empty(ops.gemm_residual_parts(m, n), m, device="cuda")
        parts = ops.gemm_residual(x, w, resid, torch.ones(n, dtype=torch.bfloat16, device="cuda"), scaled, ss)
        assert parts == 2 * (n // width) and (ss[:parts].sum(0) == n).all()


F32_ATTENTION = [
    # heads, key/value heads, key channels, value channels, options
    (9, 3, 64, 64, {}), (4, 4, 16, 16, {}), (32, 1, 64, 64, {}), (40, 2, 16, 16, {}), (5, 5, 80, 80, {}), (8, 2, 128, 128, {}), (3, 3, 256, 256, {}),
    (6, 2, 48, 48, dict(window=70)), (4, 1, 112, 112, dict(window=-96)), (6, 3, 32, 16, dict(window=33, keep_first=21, bias=True, sink=True)),
    (4, 2, 16, 48, dict(window=64, softcap=3.0, sink=True, pool=16)), (8, 2, 32, 16, dict(softcap=2.0, bias=True, decay=True, gated=True)),
    (4, 4, 96, 64, dict(bias=True, sink=True)),
]


@pytest.mark.parametrize("heads, kv_heads, head_dim, value_dim, options", F32_ATTENTION)
def test_attention_in_32_bits_on_the_matrix_cores(heads, kv_heads, head_dim, value_dim, options):
    """Single tokens (their keys in one block or several) and a step of prompts, some behind tokens held already, in every
    option, against the row kernel.  Both are 32-bit: a score below 16 is rounded at each of its ``head_dim`` products, by up
    to 2^-21 a time, of which about the square root adds up, and moves an output by as much of the values' spread, 4."""
    ops = _ops()
    torch.manual_seed(heads * head_dim + value_dim)
    rand = lambda *shape: torch.randn(*shape)  # noqa: E731
    first, new = [0, 250, 63, 0], [37, 50, 1, 130]
    ends = [f + n for f, n in zip(first, new)]
    k_pages, v_pages, table = _paged([rand(n, kv_heads, head_dim) for n in ends], [rand(n, kv_heads, value_dim) for n in ends], torch.float32,
                                     kv_heads, head_dim) if value_dim == head_dim else (None, None, None)
    if k_pages is None:
        k_pages, _, table = _paged([rand(n, kv_heads, head_dim) for n in ends], [rand(n, kv_heads, head_dim) for n in ends], torch.float32, kv_heads, head_dim)
        _, v_pages, _ = _paged([rand(n, kv_heads, value_dim) for n in ends], [rand(n, kv_heads, value_dim) for n in ends], torch.float32, kv_heads, value_dim)
    pooled = terms = None
    extras = ops.ScoreExtras(options.get("keep_first", 0), rand(heads, 41).cuda() if options.get("bias") else None,
                             rand(heads).cuda() if options.get("sink") else None)
    if options.get("pool"):
        pk = _paged([rand(64, kv_heads, head_dim) for _ in ends], [rand(64, kv_heads, head_dim) for _ in ends], torch.float32, kv_heads, head_dim)
        pv = _paged([rand(64, kv_heads, value_dim) for _ in ends], [rand(64, kv_heads, value_dim) for _ in ends], torch.float32, kv_heads, value_dim)
        pooled = ops.PooledBlocks(pk[0], pv[1], pk[2], options["pool"])
    if options.get("decay"):
        terms = ops.HeadTerms((torch.rand(heads).cuda(), torch.rand(heads).cuda()), gated=options.get("gated", False))
    common = (heads, kv_heads, head_dim, head_dim ** -0.5, options.get("window", 0), value_dim, options.get("softcap", 0.0), extras, pooled)

    def both(slots, positions, tiles=None, splits=1):
        tokens = len(slots)
        q = 3.0 * rand(tokens, heads * head_dim).cuda()  # (scores large enough for the softmax reference to move)
        own = terms.with_gate(rand(tokens, heads).cuda()) if terms is not None and terms.gated else terms
        want = torch.empty(tokens, heads * value_dim, device="cuda")
        got = torch.full((tokens, heads * value_dim), 9.0, device="cuda")
        ops.attention_rows(q, want, k_pages, v_pages, table, _i32(slots), _i32(positions), *common, own)
        ops.attention_f32(q, got, k_pages, v_pages, table, _i32(slots), _i32(positions), *common, own, tiles, splits)
        assert (got - want).abs().max().item() <= 4 * 2.0 ** -21 * max(head_dim, 32) ** 0.5, (tiles is not None, splits)
        return got

    for splits in (1, 3, ops.ATTENTION_F32_MOST_SPLITS):
        got = both([3, 1, -1, 0, 2], [129, 299, 0, 0, 63], splits=splits)
        assert (got[2] == 0).all()  # a padding row
    rows = ops.attention_module(head_dim, value_dim, options.get("softcap", 0.0), extras, pooled, terms).nnis_attention_f32_tile_rows(heads, kv_heads)
    starts = [0, *np.cumsum(new).tolist()]
    for padded in (None, (4, 256)):
        items = torch.from_numpy(ops.prefill_tile_list(new, first, padded, rows)).cuda()
        both([s for s, n in enumerate(new) for _ in range(n)], [f + i for f, n in zip(first, new) for i in range(n)],
             (items, _i32([0, 1, 2, 3]), _i32(starts), _i32(first)))
    with pytest.raises(KernelError):
        both([0], [0], splits=ops.ATTENTION_F32_MOST_SPLITS + 1)


@pytest.mark.parametrize("heads, kv_heads, head_dim, options", [
    (4, 4, 64, {}), (6, 2, 64, dict(window=20)), (2, 1, 128, dict(window=-24)), (3, 3, 256, {}), (20, 1, 16, dict(window=7, keep_first=5)),
    (4, 2, 32, dict(window=16, pool=8)), (8, 2, 80, {})])
def test_32_bit_attention_keeps_rows_from_values_that_they_do_not_see(heads, kv_heads, head_dim, options):
    """Values that are infinite or no numbers reach the rows that see their keys and no others, as in the row kernel, over a prompt and
    for single tokens: the same outputs are numbers, and those are equal to rounding (the bound of the test above)."""
    ops = _ops()
    torch.manual_seed(heads + head_dim)
    ends, window = [37, 50, 5], options.get("window", 0)
    keys, values = ([torch.randn(n, kv_heads, head_dim) for n in ends] for _ in range(2))
    values[0][20, 0, 3], values[0][22, -1, head_dim - 1], values[1][33, 0, 5], values[1][2, :, 1], values[2][4, 0, 0] = (
        float("nan"), float("inf"), float("-inf"), float("nan"), float("inf"))
    keys[1][40, 0, 2] = float("nan")
    k_pages, v_pages, table = _paged(keys, values, torch.float32, kv_heads, head_dim)
    pooled = None
    if options.get("pool"):
        entries = [torch.randn(8, kv_heads, head_dim) for _ in ends]
        entries[0][1, 0, 1] = float("inf")  # (a block that the first of a tile's rows do not see yet)
        pooled = ops.PooledBlocks(*_paged(entries, entries, torch.float32, kv_heads, head_dim), options["pool"])
    extras = ops.ScoreExtras(options.get("keep_first", 0), None, None)
    common = (heads, kv_heads, head_dim, head_dim ** -0.5, window, head_dim, 0.0, extras, pooled)

    def both(slots, positions, tiles=None, splits=1):
        q = torch.randn(len(slots), heads * head_dim).cuda()
        want, got = torch.empty_like(q), torch.empty_like(q)
        ops.attention_rows(q, want, k_pages, v_pages, table, _i32(slots), _i32(positions), *common)
        ops.attention_f32(q, got, k_pages, v_pages, table, _i32(slots), _i32(positions), *common, None, tiles, splits)
        numbers = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), numbers) and numbers.any() and not numbers.all()
        assert (got - want)[numbers].abs().max().item() <= 4 * 2.0 ** -21 * max(head_dim, 32) ** 0.5

    rows = ops.attention_module(head_dim, head_dim, 0.0, extras, pooled, None).nnis_attention_f32_tile_rows(heads, kv_heads)
    everywhere = [s for s, n in enumerate(ends) for _ in range(n)], [i for n in ends for i in range(n)]
    items = torch.from_numpy(ops.prefill_tile_list(ends, [0, 0, 0], None, rows)).cuda()
    both(*everywhere, (items, _i32([0, 1, 2]), _i32([0, *np.cumsum(ends).tolist()]), _i32([0, 0, 0])))
    for splits in (1, 2):
        both(*everywhere, splits=splits)


def _delta_in_64_bits(rows, ba, rate, dt_bias, q_scale, state, starts, heads, groups, d, e):
    rows, ba, S = rows.double(), ba.double(), state.double().transpose(-1, -2).clone()
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = (unit(rows[:, i * groups * d:(i + 1) * groups * d].view(-1, groups, d)).repeat_interleave(heads // groups, 1) for i in (0, 1))
    v = rows[:, 2 * groups * d:2 * groups * d + heads * e].view(-1, heads, e)
    beta, g = torch.sigmoid(ba[:, :heads]), torch.exp(-rate.double() * torch.log1p(torch.exp(ba[:, heads:] + dt_bias.double())))
    out = torch.empty(len(rows), heads, e, dtype=torch.float64)
    for b in range(len(starts) - 1):
        for t in range(starts[b], starts[b + 1]):
            S[b] *= g[t][:, None, None]
            S[b] += k[t][:, :, None] * (beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S[b])[:, 0]))[:, None]
            out[t] = torch.bmm(q[t][:, None] * q_scale, S[b])[:, 0]
    return out.view(len(rows), -1), S.transpose(-1, -2)


def _retention_in_64_bits(q, k, v, decay, scale, state, starts, positions, rotation, heads, d, e):
    S, out = state.double().clone(), torch.empty(len(q), heads, e, dtype=torch.float64)
    cos, sin = (table.double()[positions][:, None] for table in rotation[:2])
    half = rotation[2] // 2

    def turned(x):
        x = x.double().view(-1, heads, d)
        a, b = x[..., :half], x[..., half:2 * half]
        return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., 2 * half:]], dim=-1)

    q, k, v = turned(q), turned(k), v.double().view(-1, heads, e)
    for b in range(len(starts) - 1):
        for t in range(starts[b], starts[b + 1]):
            S[b] = decay.double()[:, None, None] * S[b] + k[t][:, :, None] * v[t][:, None]
            out[t] = torch.bmm(q[t][:, None] * scale, S[b])[:, 0]
    return out.view(len(q), -1), S


@pytest.mark.parametrize("lengths", [(63,), (64, 65, 1), (200, 7, 128, 2), (130,)])
@pytest.mark.parametrize("heads, groups, d, e, dtype", [(4, 2, 128, 128, torch.bfloat16), (2, 2, 16, 48, torch.float32), (3, 1, 112, 16, torch.bfloat16), (2, 1, 64, 256, torch.bfloat16)])
@pytest.mark.parametrize("delta", [True, False])
def test_matrix_states_in_chunks(delta, heads, groups, d, e, dtype, lengths, monkeypatch):
    """The delta rule (decays from slow to a state that is gone at once) and retention over prompts in chunks of 64 tokens and
    a token at a time, from states that hold something, against 64 bits.  A result is a sum over up to 64 tokens or 128
    channels that is rounded at each: 2^-24 of it, the square root of their number adding up."""
    import types

    ops = _ops()
    torch.manual_seed(sum(lengths) + d)
    tokens, batch, starts = sum(lengths), len(lengths), [0, *np.cumsum(lengths).tolist()]
    positions = [40 + i for n in lengths for i in range(n)]
    slots = list(range(batch, 0, -1))
    ctx = types.SimpleNamespace(decode=False, batch=batch, tokens=tokens, max_new=max(lengths), planned_new=max(lengths), planned_rows=max(lengths), seq_slot=_i32(slots), seq_start=_i32(starts),
                                tok_slot=_i32([s for s, n in zip(slots, lengths) for _ in range(n)]), tok_pos=_i32(positions))
    state = 0.3 * torch.randn(batch + 1, heads, *((e, d) if delta else (d, e)))
    if delta:
        wide = torch.randn(tokens, 2 * groups * d + heads * e + 8).to(dtype)  # (rows may be longer than what they hold)
        ba, rate, dt_bias = torch.randn(tokens, 2 * heads), 1 + torch.rand(heads), torch.linspace(-4.0, 3.0, heads)
        ba[tokens // 2, heads:] = 80.0  # (nothing of what was there before is left)
        want, after = _delta_in_64_bits(wide, ba, rate, dt_bias, d ** -0.5, state[slots], starts, heads, groups, d, e)
    else:
        wide = torch.randn(tokens, heads * (2 * d + e) + 8).to(dtype)
        q, k, v = wide[:, :heads * d], wide[:, heads * d:2 * heads * d], wide[:, 2 * heads * d:heads * (2 * d + e)]
        decay = torch.tensor([1 - 2.0 ** (-1 - 3 * h) for h in range(heads)])
        angle = torch.rand(300, d // 4 if d > 16 else 4) * 6
        rotation = (torch.cos(angle), torch.sin(angle), 2 * angle.shape[1])
        want, after = _retention_in_64_bits(q, k, v, decay, d ** -0.5, state[slots], starts, positions, rotation, heads, d, e)
    rooms = []

    def in_chunks(ctx, tokens, *sizes):  # (whatever the lengths; the floats that such a step asks for, and three chunks' behind them)
        need = lambda rows: ops.recurrent().nnis_chunked_scratch(rows, ctx.batch, *sizes[:4])  # noqa: E731
        rooms.append((torch.full((need(tokens + 192),), 7.0, device=sizes[4]), need(tokens)))
        return rooms[-1][0][:need(tokens)]

    for form in (in_chunks, lambda *sizes: None):
        monkeypatch.setattr(ops, "chunked_scratch", form)
        held, out = state.cuda(), torch.full((tokens, heads * e), 9.0, device="cuda")
        rows = wide.cuda()
        if delta:
            ops.gated_delta(rows, ba.cuda(), rate.cuda(), dt_bias.cuda(), d ** -0.5, held, ctx, heads, groups, d, e, out)
        else:
            q, k, v = rows[:, :heads * d], rows[:, heads * d:2 * heads * d], rows[:, 2 * heads * d:heads * (2 * d + e)]
            ops.gla_scan(q, k, v, None, d ** -0.5, held, ctx, heads, out, head_decay=torch.stack([decay, torch.log(decay)]).cuda(),
                         rotation=(rotation[0].cuda(), rotation[1].cuda(), rotation[2]))
        for got, exact in ((out.cpu(), want), (held.cpu()[slots], after)):
            error = (got.double() - exact).square().mean().sqrt() / exact.square().mean().sqrt()
            assert error.item() <= 2.0 ** -24 * 128 ** 0.5, form
        assert (held.cpu()[0] == state[0]).all()  # a slot that no sequence has
    assert len(rooms) == 1 and (rooms[0][0][rooms[0][1]:] == 7).all()  # nothing was written beyond what the step asks for


def _in_chunks(ops, monkeypatch):
    """Every step's matrix recurrences in chunks, whatever its lengths."""
    monkeypatch.setattr(ops, "chunked_scratch", lambda ctx, tokens, *sizes: torch.empty(
        ops.recurrent().nnis_chunked_scratch(tokens, ctx.batch, *sizes[:4]), device=sizes[4]))


def _prompts(lengths):
    import types

    starts = [0, *np.cumsum(lengths).tolist()]
    return types.SimpleNamespace(
        decode=False, batch=len(lengths), tokens=sum(lengths), max_new=max(lengths), planned_new=max(lengths), planned_rows=sum(lengths), seq_slot=_i32(range(len(lengths))),
        seq_start=_i32(starts), tok_slot=_i32([s for s, n in enumerate(lengths) for _ in range(n)]), tok_pos=_i32([i for n in lengths for i in range(n)]))


@pytest.mark.parametrize("rule", ["delta", "retention"])
def test_chunks_round_no_more_than_a_token_at_a_time(rule, monkeypatch):
    """Where states are forgotten within a few tokens, and over a prompt of a few, most of an output is its token's own update, which
    a chunk rounds as often as a token at a time does: the errors against 64 bits are equal (to 1%: both are averages over 2,000
    and more outputs of a few equal roundings and some that differ)."""
    ops = _ops()
    torch.manual_seed(11)
    heads, groups, d, e, tokens = (8, 4, 64, 128, 300) if rule == "delta" else (8, 8, 128, 256, 20)
    wide = torch.randn(tokens, 2 * groups * d + heads * e).bfloat16()
    if rule == "delta":
        ba, rate, dt_bias = 0.9 * torch.randn(tokens, 2 * heads), torch.arange(1.0, heads + 1), 2 + torch.randn(heads)
        state = 0.3 * torch.randn(1, heads, e, d)
        want = _delta_in_64_bits(wide, ba, rate, dt_bias, d ** -0.5, state, [0, tokens], heads, groups, d, e)[0]
    else:
        decay, state = torch.tensor([1 - 2.0 ** (-5 - h) for h in range(heads)]), 0.3 * torch.randn(1, heads, d, e)
        q, k, v = wide.split([heads * d, heads * d, heads * e], dim=1)
        still = (torch.ones(tokens, 0), torch.zeros(tokens, 0), 0)
        want = _retention_in_64_bits(q, k, v, decay, d ** -0.5, state, [0, tokens], list(range(tokens)), still, heads, d, e)[0]
    errors = []
    for chunks in (True, False):
        if chunks:
            _in_chunks(ops, monkeypatch)
        else:
            monkeypatch.setattr(ops, "chunked_scratch", lambda *sizes: None)
        held, out, rows = state.cuda(), torch.empty(tokens, heads * e, device="cuda"), wide.cuda()
        if rule == "delta":
            ops.gated_delta(rows, ba.cuda(), rate.cuda(), dt_bias.cuda(), d ** -0.5, held, _prompts([tokens]), heads, groups, d, e, out)
        else:
            ops.gla_scan(*rows.split([heads * d, heads * d, heads * e], dim=1), None, d ** -0.5, held, _prompts([tokens]), heads, out,
                         head_decay=torch.stack([decay, torch.log(decay)]).cuda())
        errors.append((out.cpu().double() - want).square().mean().sqrt().item())
    assert errors[0] <= 1.01 * errors[1]


@pytest.mark.parametrize("delta", [True, False])
def test_states_in_chunks_keep_tokens_from_those_behind_them(delta, monkeypatch):
    """Queries, keys, values and decays that are infinite or no numbers show in the outputs that they show in a token at a time, those
    from their token on, and in the same states; the others are equal to rounding."""
    ops = _ops()
    torch.manual_seed(5)
    heads, d, e, lengths = 3, 32, 48, [64, 100, 21, 130]
    tokens = sum(lengths)
    wide, ba = torch.randn(tokens, heads * (2 * d + e)), torch.randn(tokens, 2 * heads)
    q, k, v = wide[:, :heads * d], wide[:, heads * d:2 * heads * d], wide[:, 2 * heads * d:]
    nan, inf = float("nan"), float("inf")
    v[9, 3], v[60, e + 7], v[64 + 70, 2 * e + 1] = nan, inf, nan
    q[64 + 40, 5], k[64 + 90, d + 2] = nan, nan
    v[64 + 100 + 20, 2] = -inf  # (a sequence's last)
    if delta:
        ba[64 + 100 + 21 + 85, 0], ba[64 + 100 + 21 + 95, heads + 1] = nan, nan
    else:
        k[64 + 100 + 21 + 85, 3], v[64 + 100 + 21 + 95, e] = inf, inf
    rate, dt_bias, decay = 0.2 + torch.rand(heads).cuda(), torch.randn(heads).cuda(), torch.tensor([0.9, 0.99, 0.5])
    results = []
    for chunks in (True, False):
        if chunks:
            _in_chunks(ops, monkeypatch)
        else:
            monkeypatch.setattr(ops, "chunked_scratch", lambda *sizes: None)
        torch.manual_seed(6)
        held, out = torch.randn(4, heads, *((e, d) if delta else (d, e))).cuda(), torch.empty(tokens, heads * e, device="cuda")
        rows = wide.cuda()
        if delta:
            ops.gated_delta(rows, ba.cuda(), rate, dt_bias, d ** -0.5, held, _prompts(lengths), heads, heads, d, e, out)
        else:
            ops.gla_scan(*rows.split([heads * d, heads * d, heads * e], dim=1), None, d ** -0.5, held, _prompts(lengths), heads, out,
                         head_decay=torch.stack([decay, torch.log(decay)]).cuda())
        results.append((out, held))
    for got, want in zip(*results):
        numbers = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got), numbers) and numbers.any() and not numbers.all()
        error = (got - want)[numbers].double().square().mean().sqrt() / want[numbers].double().square().mean().sqrt()
        assert error.item() <= 2 * 2.0 ** -24 * 64 ** 0.5  # both sides sum over up to 64 tokens or channels, rounded at each


@pytest.mark.parametrize("logit", [200.0, 1e16, 1e20, float("inf")])
def test_decays_behind_a_decay_to_zero(logit, monkeypatch):
    """A decay of a chunk that is zero, however far below what a float holds, leaves the decays behind it as they are."""
    ops = _ops()
    torch.manual_seed(3)
    heads, d, e, lengths = 2, 32, 16, [64, 100]
    rows, ba, rate, dt_bias = torch.randn(164, 2 * heads * d + heads * e), torch.randn(164, 2 * heads), 1 + torch.rand(heads), torch.randn(heads)
    ba[[5, 6, 64 + 30, 64 + 70], heads:] = logit
    state = torch.randn(2, heads, e, d)
    want, after = _delta_in_64_bits(rows, ba, rate, dt_bias, d ** -0.5, state, [0, 64, 164], heads, heads, d, e)
    _in_chunks(ops, monkeypatch)
    held, out = state.cuda(), torch.empty(164, heads * e, device="cuda")
    ops.gated_delta(rows.cuda(), ba.cuda(), rate.cuda(), dt_bias.cuda(), d ** -0.5, held, _prompts(lengths), heads, heads, d, e, out)
    for got, exact in ((out.cpu(), want), (held.cpu(), after)):
        error = (got.double() - exact).square().mean().sqrt() / exact.square().mean().sqrt()
        assert error.item() <= 2.0 ** -24 * 64 ** 0.5  # sums over up to 64 tokens, rounded at each


@pytest.mark.parametrize("m, k", [(70, 72), (300, 392), (530, 8), (257, 136)])
@pytest.mark.parametrize("epilogue", ["store", "silu", "rope"])
def test_the_tile_whose_weights_go_into_registers(epilogue, m, k):
    """The 256 x 256 tile behind a prepared norm, at ragged rows and columns, gate rows that share a strip with up rows, and K
    of one step to seven: every sum takes its terms in the order of the other tiles, so the rows are the 64 x 128 tile's."""
    ops = _ops()
    torch.manual_seed(m + k)
    rope, heads, kv_heads, head_dim = None, 6, 2, 64
    n = {"store": 596, "silu": 2 * 300, "rope": (heads + 2 * kv_heads) * head_dim}[epilogue]
    code, width = {"store": (ops.EPILOGUE_STORE, n), "silu": (ops.EPILOGUE_SILU, n // 2), "rope": (ops.EPILOGUE_ROPE, heads * head_dim)}[epilogue]
    if epilogue == "rope":
        angle = torch.rand(64, head_dim // 2, device="cuda") * 6
        rope = dict(cos=torch.cos(angle), sin=torch.sin(angle), tok_slot=_i32([0] * m), tok_pos=_i32([i % 64 for i in range(m)]), heads=heads,
                    kv_heads=kv_heads, head_dim=head_dim)
    x, weight = torch.randn(m, k).bfloat16().cuda(), ops.pack_weight((torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda())
    ss = (1.0 + torch.rand(1, m)).cuda() * k
    rows = []
    for tile in (ops.TILE_256x256, ops.TILE_64x128):
        y = torch.full((m, width), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm_scaled(x, ss, 1, 1e-5, weight, y, code, rope, 16 * tile)
        rows.append(y)
    assert torch.equal(*rows)


@pytest.mark.parametrize("lengths", [[1, 1, 1], [5, 1, 9], [150, 1, 70]])
@pytest.mark.parametrize("channels, states", [(70, 4), (300, 16), (33, 20), (40, 6), (40, 128)])
def test_selective_scan_states_off_16_byte_boundaries(channels, states, lengths):
    """States and rates that lie where 16 bytes can be loaded at a time, and the same ones 4 bytes further on: equal results,
    with single tokens, whole runs and runs in pieces."""
    ops = _ops()
    torch.manual_seed(channels + states)
    tokens, slots = sum(lengths), len(lengths) + 1
    x, z, dt, bc = torch.randn(tokens, channels).cuda(), torch.randn(tokens, channels).cuda(), torch.randn(tokens, channels).cuda(), torch.randn(tokens, 2 * states).cuda()
    rates, D, bias, state = -torch.rand(channels, states).cuda(), torch.randn(channels).cuda(), torch.randn(channels).cuda(), torch.randn(slots, channels, states).cuda()
    results = []
    for shift in (0, 1):
        held, A = (torch.cat([t.new_zeros(shift), t.flatten()])[shift:].view(t.shape) for t in (state, rates))
        assert held.data_ptr() % 16 == 4 * shift
        out = torch.empty(tokens, channels, device="cuda")
        ops.selective_scan(x, dt, bc, z, A, D, bias, held, _prompts(lengths), out)
        results.append((out, held))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert torch.equal(results[0][1][-1], state[-1]) and not torch.equal(results[0][1][0], state[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch, heads, d, e", [(1, 8, 128, 256), (3, 2, 64, 36), (2, 3, 20, 4), (70, 4, 72, 132), (40, 8, 256, 64), (2, 2, 65, 30), (66, 4, 48, 128)])
def test_gla_single_tokens(batch, heads, d, e, dtype):
    """A step of single tokens against the scan over runs of one token: equal states, and outputs within the roundings of a
    sum of d products in another order; sequences without a slot leave everything as it was."""
    ops = _ops()
    torch.manual_seed(batch + d + e)
    rows = torch.randn(batch, heads * (2 * d + e) + 8).to(dtype).cuda()
    q, k, v = rows[:, :heads * d], rows[:, heads * d:2 * heads * d], rows[:, 2 * heads * d:heads * (2 * d + e)]
    state = torch.randn(batch + 1, heads, d, e).cuda()
    ctx = _prompts([1] * batch)
    ctx.seq_slot = _i32([-1 if b == 1 and batch > 2 else batch - b for b in range(batch)])
    ctx.tok_pos = _i32([(7 * b) % 50 for b in range(batch)])
    angle = torch.rand(50, d // 4).cuda() * 6
    fixed = torch.rand(heads).cuda()
    for decays in (dict(decay_logs=-torch.rand(batch, heads * d).cuda()),
                   dict(decay_logs=None, head_decay=torch.stack([fixed, fixed.log()]), rotation=(angle.cos(), angle.sin(), 2 * (d // 4)))):
        results = []
        for ctx.decode in (False, True):
            held, out = state.clone(), torch.full((batch, heads * e), 9.0, device="cuda")
            ops.gla_scan(q, k, v, scale=d ** -0.5, state=held, ctx=ctx, heads=heads, out=out, **decays)
            results.append((out, held))
        assert torch.equal(results[0][1], results[1][1]) and torch.equal(results[0][1][0], state[0])
        slots = ctx.seq_slot.long()
        live = slots >= 0
        size = torch.einsum("bhd,bhde->bhe", q.float().abs().reshape(batch, heads, d) * 1.5, results[0][1][slots.clamp(min=0)].abs()).reshape(batch, heads * e)
        error = (results[0][0] - results[1][0]).abs()  # (a rotation makes a channel at most sqrt(2) as large)
        assert (error[live] <= 2.0 ** -23 * (4 + d ** 0.5) * d ** -0.5 * size[live] + 1e-6).all() and (results[1][0][~live] == 9.0).all()


@pytest.mark.parametrize("lengths", [(700, 324), (33, 1, 1000)])
@pytest.mark.parametrize("d, e", [(128, 256), (128, 255)])
def test_matrix_states_of_a_prompt_are_cut_alike_beside_more_heads(lengths, d, e):
    """Where a run is cut says how its sums are rounded: heads of one prompt are the same bits together and a few at a time, however many
    bytes of state the pieces hand on (64 MB here, half of it, and a little less)."""
    ops = _ops()
    torch.manual_seed(len(lengths))
    heads, tokens = 8, sum(lengths)
    q, k, v = (torch.randn(tokens, heads, n).bfloat16().cuda() for n in (d, d, e))
    logs, state = -0.2 * torch.rand(tokens, heads, d).cuda(), torch.randn(len(lengths), heads, d, e).cuda()

    def scan(first, last):
        part = [t[:, first:last].clone() for t in (q, k, v, logs, state)]
        held, out = part.pop(), torch.empty(tokens, (last - first) * e, device="cuda")
        rows = [t.reshape(tokens, -1) for t in part]
        ops.gla_scan(*rows, d ** -0.5, held, _prompts(lengths), last - first, out)
        return out.view(tokens, last - first, e), held

    together, apart = scan(0, heads), [scan(0, 4), scan(4, heads)]
    for which in (0, 1):
        assert torch.equal(together[which], torch.cat([part[which] for part in apart], dim=1))


@pytest.mark.parametrize("width", [1028, 2048, 4096, 5000, 8192])
@pytest.mark.parametrize("count", [1, 5, 1023, 1024, 2046])
def test_rmsnorm_of_few_rows(width, count):
    """Rows that a block each norms (up to 1,023) and rows that a wave each does, with the weight asked for beside the row (up to 2,048; the
    last count has 2,049 without a row list) and behind its sum: with a row list, with a sum written back, with
    both, in both types; the last rows of the list out of order."""
    ops = _ops()
    torch.manual_seed(width + count)
    x, delta, weight = torch.randn(count + 3, width), torch.randn(count + 3, width), 1 + 0.2 * torch.randn(width)
    for dtype in (torch.float32, torch.bfloat16):
        d, w = delta.to(dtype), weight.to(dtype)
        rows = torch.arange(count + 2, 2, -1, dtype=torch.int32)
        total = x.double() + d.double()
        for picked, added in ((rows, None), (rows, d), (None, d), (None, None)):
            held = x.cuda()
            out = torch.full((count + 1 if picked is not None else count + 3, width), 9.0, device="cuda")
            ops.rmsnorm(held, w.cuda(), 1e-6, out[:count] if picked is not None else out, delta=None if added is None else added.cuda(),
                        rows=None if picked is None else picked.cuda())
            source = (total if added is not None else x.double())[picked.long() if picked is not None else slice(None)]
            want = source / torch.sqrt((source * source).mean(1, keepdim=True) + 1e-6) * w.double()
            got = out[:len(want)].cpu().double()
            assert ((got - want).abs() <= 2e-6 * (1 + want.abs())).all()
            assert picked is None or (out[count] == 9).all()
            written = added is not None and picked is None
            assert torch.equal(held.cpu(), (x + d.float()) if written else x)


@pytest.mark.parametrize("width, shift", [(24, 0), (24, 1), (2052, 0), (2052, 4), (30, 0), (4100, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embeddings_four_channels_at_a_time(width, shift, dtype):
    """Rows that can be loaded four channels at a time, tables that lie off such places, and widths that cannot: exact copies,
    and with a table of pairs exact sums, in every copy; ids outside the table give zeros."""
    ops = _ops()
    torch.manual_seed(width)
    table, pairs = torch.randn(shift + 40 * width).to(dtype)[shift:].view(40, width), torch.randn(6, width).to(dtype)
    held = torch.empty(shift + 40 * width, dtype=dtype, device="cuda")[shift:].view(40, width)
    held.copy_(table)
    ids = _i32([3, 39, -1, 40, 0])
    out = torch.full((5, width), 9.0, device="cuda")
    ops.embed(ids, held, out, scale=0.5)
    want = table.float()[[3, 39, 0, 0, 0]] * torch.tensor([0.5, 0.5, 0.0, 0.0, 0.5])[:, None]
    assert torch.equal(out.cpu(), want)
    both = torch.full((3, 5, width), 9.0, device="cuda")
    ops.embed_pair(ids, _i32([0, 1, 2, 3, -1]), _i32([0, 0, 0, 0, 0]), held, pairs.cuda(), 3, 5, _i32([-1] * 4), both)
    want = torch.zeros(5, width)
    want[:2] = table.float()[[3, 39]] + pairs.float()[5]
    assert torch.equal(both.cpu(), want.expand(3, 5, width))


@pytest.mark.parametrize("count", [1023, 1024])
@pytest.mark.parametrize("width", [64, 260, 2050, 2052])
def test_embeddings_of_many_rows(width, count):
    """The blocks that few and many rows take, for widths of less than a wave's channels, a few more than one wave's, and wide ones whose
    channels are copied four and one at a time."""
    ops = _ops()
    torch.manual_seed(width)
    table, pairs = torch.randn(50, width), torch.randn(4, width)
    ids = torch.randint(-1, 51, (count,), dtype=torch.int32)
    known = ((ids >= 0) & (ids < 50))[:, None]
    out = torch.full((count + 1, width), 9.0, device="cuda")
    ops.embed(ids.cuda(), table.cuda(), out[:count], scale=0.5)
    assert torch.equal(out[:count].cpu(), torch.where(known, table[ids.clamp(0, 49).long()] * 0.5, 0.0)) and (out[count] == 9).all()
    both = torch.full((2, count, width), 9.0, device="cuda")
    slots = torch.zeros(count, dtype=torch.int32)
    ops.embed_pair(ids.cuda(), slots.cuda(), slots.cuda(), table.cuda(), pairs.cuda(), 3, 5, _i32([-1] * 4), both)  # (each at position 0)
    want = torch.where(known, table[ids.clamp(0, 49).long()] + pairs[3], 0.0)
    assert torch.equal(both.cpu(), want.expand(2, count, width))


@pytest.mark.parametrize("rows", [255, 256])
@pytest.mark.parametrize("streams, width", [(2, 36), (4, 2048), (5, 4096), (2, 4100)])
def test_streams_of_few_and_many_rows(streams, width, rows):
    """Rows whose norm's vectors come beside them (up to 255, up to 4,096 channels) and behind their sums, after an update: streams and
    norms against 64 bits, a few roundings of the largest terms."""
    ops = _ops()
    torch.manual_seed(width)
    x, y, mix, gain, take = torch.randn(streams, rows, width), torch.randn(rows, width), torch.randn(streams, streams), torch.randn(streams), torch.rand(streams) + 0.5
    w, b = 1 + 0.2 * torch.randn(width), torch.randn(width)
    want = torch.einsum("st,srw->trw", mix.double(), x.double()) + gain.double()[:, None, None] * y.double()
    read = (take.double()[:, None, None] * want).sum(0)
    centred = read - read.mean(1, keepdim=True)
    normed = centred / torch.sqrt((centred * centred).mean(1, keepdim=True) + 1e-5) * w.double() + b.double()
    held, h = x.cuda(), torch.full((rows, width), 9.0, device="cuda")
    ops.stream_step(held, h, y.cuda(), mix.cuda(), gain.cuda(), take.cuda(), w.cuda(), b.cuda(), 1e-5)
    size = torch.einsum("st,srw->trw", mix.double().abs(), x.double().abs()) + gain.double().abs()[:, None, None] * y.double().abs()
    assert ((held.cpu().double() - want).abs() <= 1e-6 * size).all()
    assert ((h.cpu().double() - normed).abs() <= 2e-5 * (1 + normed.abs())).all()


@pytest.mark.parametrize("rows", [5, 1023, 1024])
@pytest.mark.parametrize("q_rank, kv_rank, rot, gates", [(224, 64, 32, 16), (0, 72, 16, 3), (40, 208, 0, 0)])
def test_latents_of_few_and_many_rows(q_rank, kv_rank, rot, gates, rows):
    """A channel a thread (up to 1,023 rows) and fewer threads, for latents whose widths the two part: query latent, cached latent and
    rotated channels, gates against 64 bits; a row without a slot leaves the cache as it was."""
    ops = _ops()
    torch.manual_seed(q_rank + kv_rank)
    proj = torch.randn(rows, q_rank + kv_rank + rot + gates)
    q_weight, c_weight = 1 + 0.2 * torch.randn(q_rank), 1 + 0.2 * torch.randn(kv_rank)
    angle = torch.rand(rows, rot // 2) * 6
    pages = (rows + 63) // 64
    k_pages, v_pages = _empty_pages(pages, 1, kv_rank + rot, torch.float32, 7.0, 7.0, "cuda")[0], _empty_pages(pages, 1, kv_rank, torch.float32, 7.0, 7.0, "cuda")[1]
    slots = torch.zeros(rows, dtype=torch.int32)
    slots[3] = -1
    cq = torch.full((rows, q_rank), 9.0, device="cuda") if q_rank else None
    gate = torch.full((rows, gates), 9.0, device="cuda") if gates else None
    ops.latent_prepare(proj.cuda(), q_rank, kv_rank, rot, gates, q_weight.cuda() if q_rank else None, c_weight.cuda(), 1e-5,
                       angle.cos().cuda() if rot else None, angle.sin().cuda() if rot else None, slots.cuda(), _i32(range(rows)), cq, k_pages, v_pages,
                       torch.arange(pages, dtype=torch.int32).flip(0)[None].cuda(), gate)
    def normed(x, w):
        return x.double() / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5) * w.double()

    latent = normed(proj[:, q_rank:q_rank + kv_rank], c_weight)
    u, v = proj[:, q_rank + kv_rank:q_rank + kv_rank + rot].double().view(rows, rot // 2, 2).unbind(2)
    cos, sin = angle.cos().double(), angle.sin().double()
    keys = torch.cat([latent, torch.stack([u * cos - v * sin, v * cos + u * sin], 2).view(rows, rot)], 1)
    held_k = k_pages.cpu().view(pages, -1)[:, _k_index(kv_rank + rot)].flip(0).reshape(pages * 64, -1)
    held_v = v_pages.cpu().view(pages, -1)[:, _v_index(kv_rank)].flip(0).reshape(pages * 64, -1)
    kept = [r for r in range(rows) if r != 3]
    assert ((held_k[:rows] - keys).abs()[kept] <= 2e-6 * (1 + keys.abs()[kept])).all() and ((held_v[:rows] - latent).abs()[kept] <= 2e-6 * (1 + latent.abs()[kept])).all()
    assert (held_k[3] == 7).all() and (held_k[rows:] == 7).all() and (held_v[rows:] == 7).all()
    if q_rank:
        want = normed(proj[:, :q_rank], q_weight)
        assert ((cq.cpu().double() - want).abs() <= 2e-6 * (1 + want.abs())).all()
    if gates:
        want = torch.sigmoid(proj[:, -gates:].double())
        assert ((gate.cpu().double() - want).abs() <= 1e-6).all()


@pytest.mark.parametrize("rows", [1, 5, 300])
@pytest.mark.parametrize("size", [1, 2, 3, 4])
def test_rows_in_16_bits_as_in_32(size, rows):
    """Kernels that know their types when compiled against the same ones on the same values in 32 bits, whose types are branches, around
    the sizes that part them: the same numbers but for the rounding that is stored, on whose edge a value may fall to either side."""
    ops = _ops()
    torch.manual_seed(10 * size + rows)
    half = lambda *shape: torch.randn(*shape, device="cuda").bfloat16()

    def alike(call, *shapes):  # call(type, outputs): the outputs of each type
        got, want = ([torch.full(shape, 7.0, device="cuda", dtype=kind) for shape in shapes] for kind in (torch.bfloat16, torch.float32))
        call(torch.bfloat16, *got)
        call(torch.float32, *want)
        for g, w in zip(got, want):
            assert ((g.float() - w).abs() <= 2.0 ** -7 * w.abs() + 1e-6).all()

    for dim in (64 * size, 64 * size + 1):  # (in registers up to 256 channels a head)
        o, gate, weight = torch.randn(rows, 3 * dim, device="cuda"), half(rows, 3 * dim + 8)[:, 8:], half(dim)
        for w in (weight, None):
            alike(lambda kind, y: ops.head_norm_gate(o, gate.to(kind), None if w is None else w.to(kind), 1e-5, 3, y), (rows, 3 * dim))
    for width in (4, 260 * size, 1024 * size):
        ys, ws, b = [half(rows, width) for _ in range(size)], [half(width) for _ in range(size)], half(width)
        alike(lambda kind, out: ops.branch_mean([y.to(kind) for y in ys], [w.to(kind) for w in ws], [b.to(kind)] + [None] * (size - 1), 1e-5, out), (rows, width))
        x, mix, gain = torch.randn(size, rows, width, device="cuda"), torch.randn(size, size, device="cuda"), torch.randn(size, device="cuda")

        def stream(kind, h, y, norm):
            held = x.clone()
            ops.stream_step(held, h, ys[0].to(kind) if y else None, mix if y else None, gain if y else None, None, ws[0].to(kind) if norm else None,
                            b.to(kind) if norm else None, 1e-5 if norm else 0.0)
        for y, norm in ((True, True), (True, False), (False, True)):
            alike(lambda kind, h: stream(kind, h, y, norm), (rows, width))
    heads, kv, dim, rot = 5 * size, size, 128, 64 if size % 2 else 128  # (112 to 480 items of four channels)
    if rows == 5:
        heads, kv = 16 * size, 8 * size  # (up to 2,560, beyond a block)
    qkv, angle, pages = half(rows, (heads + 2 * kv) * dim), torch.rand(512, rot // 2, device="cuda") * 6, (rows + 63) // 64
    slots = torch.zeros(rows, dtype=torch.int32, device="cuda")
    slots[3:4] = -1
    table = torch.arange(pages, dtype=torch.int32).flip(0)[None].cuda()
    places = [(pages, kv, dim // 8, 64, 8), (pages, kv, dim // 16, 2, 4, 16, 8)]
    alike(lambda kind, q, k, v: ops.rope_kv_write(qkv.to(kind), q, angle.cos(), angle.sin(), rot, slots, _i32(range(rows)), k, v, table, heads, kv, dim),
          (rows, heads * dim), *places)
    q_rank, kv_rank, gates = 96 * (size - 1), 72 * size, 3 * (size % 2)  # (up to 288 channels, beyond a block's threads)
    proj, q_weight, c_weight, gate = torch.randn(rows, q_rank + kv_rank + 32 + gates, device="cuda"), half(q_rank), half(kv_rank), torch.empty(rows, gates, device="cuda")
    alike(lambda kind, cq, k, v: ops.latent_prepare(proj, q_rank, kv_rank, 32, gates, q_weight.to(kind) if q_rank else None, c_weight.to(kind), 1e-5,
                                                    angle[:, :16].cos().contiguous(), angle[:, :16].sin().contiguous(), slots, _i32(range(rows)),
                                                    cq if q_rank else None, k, v, table, gate if gates else None),
          (rows, q_rank), *[_empty_pages(pages, 1, n, torch.float32, 0.0, 0.0, "cuda")[which].shape for which, n in ((0, kv_rank + 32), (1, kv_rank))])


@pytest.mark.parametrize("kernel, heads, kv_heads", [("columns", 16, 2), ("keys", 9, 3)])
@pytest.mark.parametrize("splits, waves", [(1, 4), (2, 2), (8, 4), (1, 1)])
def test_decode_attention_around_64_pages(kernel, heads, kv_heads, splits, waves):
    """Runs of keys that end within a sequence's first 64 pages, at the 64th, behind it and begin behind it, whole and in a
    window that leaves the first pages out."""
    ops = _ops()
    torch.manual_seed(splits * 8 + waves)
    head_dim, lengths = 64, [4200, 4096, 4097, 8300, 63 * 64, 5]
    ks = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    vs = [torch.randn(n, kv_heads, head_dim).bfloat16().float() for n in lengths]
    scale = 1.0 / math.sqrt(head_dim)
    k_pages, v_pages, table = _paged(ks, vs, torch.bfloat16, kv_heads, head_dim, pages=420, max_pages=131)
    rows = [(s, n - 1, torch.randn(heads, head_dim).bfloat16().float()) for s, n in enumerate(lengths)]
    q = torch.stack([r[2] for r in rows]).bfloat16().reshape(len(rows), -1).cuda()
    out = torch.empty(len(rows), heads * head_dim, dtype=torch.bfloat16, device="cuda")
    partial = torch.full((len(rows) * heads * splits * (head_dim + 4),), float("nan"), dtype=torch.float32, device="cuda")
    for window in (0, 4300):
        ops.attention_decode_bf16(q, out, k_pages, v_pages, table, _i32([s for s, _, _ in rows]), _i32([p for _, p, _ in rows]),
                                  heads, kv_heads, head_dim, scale, window, splits, partial, waves, kernel)
        want = _plain_rows(rows, ks, vs, scale, window=window) if window else _plain_rows(rows, ks, vs, scale)
        assert (out.cpu().float().view(len(rows), heads, head_dim) - want).abs().max().item() <= 1e-2


@pytest.mark.parametrize("group", [5, 8, 15, 16, 24, 32])
def test_the_order_of_a_blocks_weights(group):
    """A lane's eight weights of a block of keys are added one after the other; where every column has a head, the blocks in the middle of a
    run are added in pairs.  Weights of 1 and seven times 0.92 of half a unit in its last place say which: one after the other they are
    lost, in pairs they are three units."""
    ops = _ops()
    lengths, places = [1536, 1536], [256, 704]  # (a block in the middle of the first of two runs of 24 blocks, and among its last)
    ks = [torch.zeros(n, 1, 64) for n in lengths]
    for k, place in zip(ks, places):
        k[:, 0, 0] = -20000.0  # (a weight of 0 beside the others)
        k[place:place + 8, 0, 0] = torch.tensor([0.0] + 7 * [-24.125])
    k_pages, v_pages, table = _paged(ks, ks, torch.bfloat16, 1, 64, pages=50, max_pages=24)
    q = torch.zeros(2, group, 64, dtype=torch.bfloat16, device="cuda")
    q[:, :, 0] = 1.0
    out = torch.empty(2, group * 64, dtype=torch.bfloat16, device="cuda")
    partial = torch.full((2, group, 2, 68), float("nan"), device="cuda")
    ops.attention_decode_bf16(q.view(2, -1), out, k_pages, v_pages, table, _i32([0, 1]), _i32([1535, 1535]), group, 1, 64, math.log(2.0), 0, 2, partial, 1, "columns")
    middle, end = partial[:, :, 0, 65].cpu()
    assert (middle == (1.0 + 3 * 2.0 ** -23 if group % 16 == 0 else 1.0)).all() and (end == 1.0).all()


@pytest.mark.parametrize("heads", [3, 8, 24])
@pytest.mark.parametrize("splits", [1, 3])
def test_a_bias_that_hides_far_keys(heads, splits):
    """A bias by distance whose last row is minus infinity, or the lowest number, leaves the keys before it out."""
    ops = _ops()
    torch.manual_seed(heads)
    length, reach, scale = 3000, 40, 0.125
    k, v = (torch.randn(length, 1, 64).bfloat16().float() for _ in range(2))
    k_pages, v_pages, table = _paged([k], [v], torch.bfloat16, 1, 64, pages=48, max_pages=48)
    q = torch.randn(1, heads * 64).bfloat16()
    bias = torch.randn(heads, reach + 1)
    bias[::2, reach], bias[1::2, reach] = float("-inf"), torch.finfo(torch.float32).min
    out = torch.empty(1, heads * 64, dtype=torch.bfloat16, device="cuda")
    partial = torch.empty(heads * splits * 68, device="cuda")
    ops.attention_decode_bf16(q.cuda(), out, k_pages, v_pages, table, _i32([0]), _i32([length - 1]), heads, 1, 64, scale, 0, splits, partial, 4, "columns",
                              extras=ops.ScoreExtras(0, bias.cuda(), None))
    seen = slice(length - reach, length)
    scores = q.double().view(heads, 64) @ k[seen, 0].double().T * scale + bias[:, :reach].flip(1).double()
    want = scores.softmax(dim=1) @ v[seen, 0].double()
    assert (out.cpu().double().view(heads, 64) - want).abs().max().item() <= 2e-2  # (probabilities and outputs in 16 bits, values up to 4)


@pytest.mark.parametrize("heads, kv_heads", [(8, 1), (5, 1), (24, 1), (9, 3)])
def test_keys_whose_scores_are_minus_infinity(heads, kv_heads):
    """A sequence's first pages of keys score minus infinity: they have no weight, and the others theirs."""
    ops = _ops()
    torch.manual_seed(heads)
    length, hidden = 1500, 200
    k, v = (torch.randn(length, kv_heads, 64).bfloat16().float() for _ in range(2))
    k[:, :, 0], k[:hidden, :, 0] = 0.0, -2.0 ** 100
    k_pages, v_pages, table = _paged([k], [v], torch.bfloat16, kv_heads, 64, pages=24, max_pages=24)
    q = torch.randn(1, heads, 64).bfloat16()
    q[:, :, 0] = 2.0 ** 100
    out = torch.empty(1, heads * 64, dtype=torch.bfloat16, device="cuda")
    for waves in (1, 4):
        ops.attention_decode_bf16(q.view(1, -1).cuda(), out, k_pages, v_pages, table, _i32([0]), _i32([length - 1]), heads, kv_heads, 64, 0.125, 0, 1, None, waves)
        scores = torch.einsum("khd,tkd->kht", q.double().view(kv_heads, -1, 64), k[hidden:].double()) * 0.125
        want = torch.einsum("kht,tkd->khd", scores.softmax(dim=2), v[hidden:].double()).reshape(heads, 64)
        assert (out.cpu().double().view(heads, 64) - want).abs().max().item() <= 1e-2, waves  # (probabilities and outputs in 16 bits)


# the four-wave tiles: their hint to the products, their columns
FOUR_WAVE_TILES = [(48, 64), (32, 128)]


def _tiled_parts(m, n, k, columns):
    """Parts of K of a product in tiles of 64 rows: the rule of the kernels' launch, written once more."""
    col_blocks, steps = -(-n // columns), -(-k // 64)
    tiles, parts = col_blocks * -(-m // 64), 1
    while parts < 8 and tiles * parts * 2 <= 256 and steps // (parts * 2) >= 4:
        parts *= 2
    while parts > 1 and parts * m * col_blocks * columns * 4 > _ops().GEMM_WORKSPACE_BYTES:
        parts //= 2
    return parts if k - k // parts >= 900 else 1


class _PartsOfK:
    """Sees by the workspace in how many parts of ``size`` sums the product inside went (1: K whole, nothing written)."""

    def __init__(self, size):
        ops = _ops()
        self.size, self.workspace = size, ops._gemm_workspace(torch.device("cuda", torch.cuda.current_device()))[:ops.GEMM_WORKSPACE_BYTES // 4]

    def __enter__(self):
        self.workspace.fill_(-7.5e33)
        return self

    def __exit__(self, *error):
        written = (self.workspace != -7.5e33).nonzero()
        self.parts = 1 if written.numel() == 0 else written.max().item() // self.size + 1
        self.workspace.zero_()


# sizes whose tiles of 64 x 64 leave room for 2, 4 and 8 parts: a K just too short for them, and just long enough
PARTS_OF_K = {(130, 2000, 1792): 1, (130, 2000, 1800): 2, (300, 1500, 1800): 2, (70, 1900, 1192): 1, (70, 1900, 1200): 4, (19, 130, 1200): 4, (70, 500, 1984): 4,
              (70, 500, 1992): 8}


@pytest.mark.parametrize("hint, columns", FOUR_WAVE_TILES)
@pytest.mark.parametrize("m, n, k", list(PARTS_OF_K))
def test_products_around_the_k_from_which_it_goes_in_parts(m, n, k, hint, columns):
    """Products whose K is just too short to go in two, four or eight parts, and just long enough: stored and into the stream, with
    the sums of squares that either leaves, against 64 bits; that K went in so many parts, or whole, shows in the workspace."""
    ops = _ops()
    torch.manual_seed(m + k)
    x, w = torch.randn(m, k).bfloat16(), (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    want, scale = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    parts, width = _tiled_parts(m, n, k, columns), -(-n // columns) * columns
    assert columns != 64 or parts == PARTS_OF_K[m, n, k]
    packed = ops.pack_weight(w.cuda())
    for dtype, bound in ((torch.float32, 2e-7 * math.sqrt(k) * scale + 1e-6), (torch.bfloat16, 2.0 ** -8 * want.abs() + 1e-5)):
        y = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
        with _PartsOfK(m * width) as seen:
            ops.gemm_bf16(x.cuda(), packed, y[:m], hint)
        assert seen.parts == parts
        assert ((y[:m].cpu().double() - want).abs() <= bound).all() and (y[m] == 7).all()
    resid, gain = torch.randn(m, n) * 2, (1 + 0.3 * torch.randn(n)).bfloat16()
    held, scaled = resid.cuda(), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ss = torch.full((ops.gemm_residual_parts(m, n) + 1, m), 7.0, device="cuda")
    with _PartsOfK(m * width) as seen:
        squares = ops.gemm_residual(x.cuda(), packed, held, gain.cuda(), scaled, ss, hint // 16)
    assert seen.parts == parts
    each = 64 if parts > 1 else columns // 2
    assert squares == (-(-n // 64) if parts > 1 else 2 * -(-n // columns)) and (ss[squares:] == 7).all()
    got = held.cpu().double()
    assert ((got - resid.double() - want).abs() <= 2e-7 * math.sqrt(k) * scale + 2e-6).all()
    assert torch.equal(scaled.cpu(), (held.cpu() * gain.float()).bfloat16())
    for part in range(squares):
        of = got[:, part * each:(part + 1) * each].pow(2).sum(dim=1)
        assert ((ss[part].cpu().double() - of).abs() <= 1e-5 * (1e-3 + of)).all(), part


@pytest.mark.parametrize("hint, columns", FOUR_WAVE_TILES)
@pytest.mark.parametrize("m, k", [(65, 1200), (19, 1992), (130, 2304)])
def test_scaled_projection_with_k_in_parts(m, k, hint, columns):
    """The epilogues of products behind a prepared norm -- stored, gated, rotated with the write into the cache -- where K goes in
    parts, whose sums a kernel behind the product adds up: against the plain functions one after another."""
    ops = _ops()
    torch.manual_seed(hint + m + k)
    eps = 1e-5
    scaled = torch.randn(m, k).bfloat16()
    ss = (torch.rand(3, m) + 0.1) * k
    normed = scaled.double() / torch.sqrt(ss.double().sum(0) / k + eps)[:, None]

    def run(w, y, epilogue, covered, rope=None):  # (covered: weight rows that the grid has tiles for)
        with _PartsOfK(m * -(-covered // columns) * columns) as seen:
            ops.gemm_scaled(scaled.cuda(), ss.cuda(), 3, eps, ops.pack_weight(w.cuda()), y, epilogue, rope, hint)
        assert seen.parts == _tiled_parts(m, covered, k, columns) > 1
        return y.cpu().double()

    def close(got, want, what):
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all(), (what, (got - want).abs().max().item())

    n = 300
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    close(run(w, torch.empty(m, n, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_STORE, n), normed @ w.double().t(), "store")
    inner = 200
    w = (torch.randn(2 * inner, k) / math.sqrt(k)).bfloat16()
    both = normed @ w.double().t()
    close(run(w, torch.empty(m, inner, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_SILU, 32 * -(-inner // 16)), P.silu(both[:, :inner]) * both[:, inner:], "silu")
    heads, kv_heads, head_dim = 5, 2, 64
    n = (heads + 2 * kv_heads) * head_dim
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    qkv = (normed @ w.double().t()).view(m, heads + 2 * kv_heads, head_dim)
    cos, sin = (torch.from_numpy(a) for a in P.rope_tables(1024, head_dim, 10000.0))
    positions = torch.tensor([(i * 37) % 1024 for i in range(m)])
    table = torch.arange(16, dtype=torch.int32).flip(0)[None]
    k_pages, v_pages = _empty_pages(16, kv_heads, head_dim, torch.bfloat16, 7.0, 7.0, "cuda")
    rope = dict(cos=cos.cuda(), sin=sin.cuda(), tok_slot=_i32([0 if i % 11 else -1 for i in range(m)]), tok_pos=positions.int().cuda(), k_pages=k_pages, v_pages=v_pages,
                block_table=table.cuda(), heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    got = run(w, torch.empty(m, heads * head_dim, dtype=torch.bfloat16, device="cuda"), ops.EPILOGUE_ROPE, n, rope)
    turned = P.rope_rotate_half(qkv[:, :heads + kv_heads], cos[positions].double(), sin[positions].double())
    close(got.view(m, heads, head_dim), turned[:, :heads], "queries")
    held_k, held_v = _read_pages(k_pages, v_pages, head_dim)
    for i in range(m):
        page, inside = table[0, positions[i] // 64].item(), positions[i].item() % 64
        if i % 11:
            close(held_k[page, :, inside].double(), turned[i, heads:], "keys")
            close(held_v[page, :, inside].double(), qkv[i, heads + kv_heads:], "values")
        else:
            assert (held_k[page, :, inside] == 7).all() and (held_v[page, :, inside] == 7).all()


@pytest.mark.parametrize("m, n, height, k", [(300, 4096, 128, 264), (2285, 8192, 128, 264), (621, 16384, 160, 264), (2093, 8192, 160, 264), (741, 16384, 192, 264), (2257, 11264, 192, 264),
                                             (741, 16384, 192, 520), (5900, 2048, 192, 1032)])
def test_large_tiles_with_lower_ones_behind_them(m, n, height, k):
    """Rows of a product in tiles of 256 x 256 whose last are cut lower, with every epilogue: the bits of tiles of 64 x 128, which add a sum
    up in the same order, and the parts of the sums of squares."""
    ops = _ops()
    torch.manual_seed(m)
    assert ops.gemm_large_rows(m, n, k)[1] == height and (height != 192 or k == 264 or ops.gemm_large_rows(m, n, k, False)[1] == 192)
    x, weight = torch.randn(m, k).bfloat16().cuda(), ops.pack_weight((torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda())
    ss = (1.0 + torch.rand(1, m)).cuda() * k
    head_dim, kv_heads = 64, 4
    heads = n // head_dim - 2 * kv_heads
    angle = torch.rand(64, head_dim // 2, device="cuda") * 6
    rope = dict(cos=torch.cos(angle), sin=torch.sin(angle), tok_slot=_i32([0] * m), tok_pos=_i32([i % 64 for i in range(m)]), heads=heads,
                kv_heads=kv_heads, head_dim=head_dim)
    for epilogue, width in ((ops.EPILOGUE_STORE, n), (ops.EPILOGUE_SILU, n // 2), (ops.EPILOGUE_ROPE, heads * head_dim)):
        rows = []
        for tile in (ops.TILE_256x256, ops.TILE_64x128):
            y = torch.full((m, width), 9.0, dtype=torch.bfloat16, device="cuda")
            ops.gemm_scaled(x, ss, 1, 1e-5, weight, y, epilogue, rope if epilogue == ops.EPILOGUE_ROPE else None, 16 * tile)
            rows.append(y)
        assert torch.equal(*rows), epilogue
    for dtype in (torch.bfloat16, torch.float32):
        rows = [torch.full((m + 1, n), 9.0, dtype=dtype, device="cuda") for _ in range(2)]
        for tile, y in zip((ops.TILE_256x256, ops.TILE_64x128), rows):
            ops.gemm_bf16(x, weight, y[:m], 16 * tile)
        assert torch.equal(*rows) and (rows[0][m] == 9.0).all(), dtype
    stream, gain, got = torch.randn(m, n).cuda(), (1 + 0.3 * torch.randn(n)).bfloat16().cuda(), []
    for tile in (ops.TILE_256x256, ops.TILE_64x128):
        resid, scaled = stream.clone(), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        parts_of = torch.full((ops.gemm_residual_parts(m, n) + 1, m), 7.0, device="cuda")
        parts = ops.gemm_residual(x, weight, resid, gain, scaled, parts_of, tile)
        assert (parts_of[parts:] == 7.0).all()
        got.append((resid, scaled, parts_of[:parts].double().sum(dim=0)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    # (sums of n squares in 32 bits: sqrt(n) roundings of 2^-24 and a few more)
    assert ((got[0][2] - got[1][2]).abs() <= 1e-5 * got[1][2]).all()


@pytest.mark.parametrize("n, k, parts", [(2560, 2048, 4), (6144, 2048, 2), (4096, 1288, 4), (6080, 1992, 2), (2304, 3080, 4)])
@pytest.mark.parametrize("epilogue", ["store", "silu", "rope"])
@pytest.mark.parametrize("m", [33, 48, 64])
def test_products_whose_waves_share_k_in_groups(m, epilogue, n, k, parts):
    """33 to 64 rows whose K went in parts through memory: the same bits from groups of waves that meet in LDS, in tiles of 32 x 32 and, of
    many columns, 64 x 32."""
    ops = _ops()
    torch.manual_seed(m + k)
    head_dim, kv_heads = 64, 3
    heads = n // head_dim - 2 * kv_heads
    code, columns = {"store": (ops.EPILOGUE_STORE, n), "silu": (ops.EPILOGUE_SILU, n // 2), "rope": (ops.EPILOGUE_ROPE, heads * head_dim)}[epilogue]
    rope = None
    if epilogue == "rope":
        angle = torch.rand(64, head_dim // 2, device="cuda") * 6
        rope = dict(cos=torch.cos(angle), sin=torch.sin(angle), tok_slot=_i32([0] * m), tok_pos=_i32([i % 64 for i in range(m)]), heads=heads,
                    kv_heads=kv_heads, head_dim=head_dim)
    x, weight = torch.randn(m, k).bfloat16().cuda(), ops.pack_weight((torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda())
    norm_parts = 2 * -(-k // 64)
    ss = (1.0 + torch.rand(norm_parts, m)).cuda() * k / norm_parts
    assert ops.gemm_grouped(m, n, k) == (None if parts == 2 and m > 48 else (32 if n // 32 * -(-m // 32) <= 256 else 64, parts))
    rows = []
    for split in (0, 16 * ops.TILE_64x64):
        y = torch.full((m + 1, columns), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm_scaled(x, ss, norm_parts, 1e-5, weight, y[:m], code, rope, split)
        assert (y[m] == 9.0).all()
        rows.append(y[:m])
    assert torch.equal(*rows)
