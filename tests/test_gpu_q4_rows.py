"""Parity of the 4-bit projections of several activation rows (the matrix-core
kernels of nwd_q4_rows.hip) with float64, through the C ABI.

Bars: |y - y64| <= 1e-6 sum_k |w_k a_k| (the one-row kernels' bar; their
activations enter as fp16 high and low parts, within 2^-23 of the largest of
their 32, or in fp32, and 32 products are summed at a time); a row that holds
an infinity or a NaN is NaN, as on the one-row kernels; cache rows within one
fp16 ulp; the picked token is the largest logit.

Sizes: the smallest and largest row counts of each row tiling (packed up to
8, then 16, 32 and 64 rows, several groups of 64), column counts that leave a
remainder of the 16- and 32-column tiles, odd block counts, one block, and
the largest K. All are sizes that these kernels take (test_route).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nwd_attn as nw  # noqa: E402
from gpu_util import dev, host, pos_tensor, say  # noqa: E402
from argmax_cases import reference_rule  # noqa: E402
from q4_cases import dequant_f64, random_q4, rng  # noqa: E402

pytestmark = pytest.mark.gpu

TOL_REL = 1e-6
D = 128


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X")
    nw.load_library()


class Q4:
    def __init__(self, g, n, n_blocks):
        quant, scales, zp = random_q4(g, n, n_blocks)
        self.t = (dev(quant), dev(scales), dev(zp))
        self.w = nw.q4_weight(*self.t, n, n_blocks)
        self.dense = torch.from_numpy(dequant_f64(quant, scales, zp)).cuda()

    def f64(self, x):
        x = torch.from_numpy(np.asarray(x, np.float64)).cuda()
        return host(x @ self.dense.t()), host(x.abs() @ self.dense.abs().t())


def _ctx(H=32, Hkv=8, cap=512, B=64, q="f32", Dh=D):
    return nw.AttnContext(H, Hkv, cap, head_dim=Dh, max_batch=B, q_dtype=q, o_dtype="f32",
                          kv_dtype="f32")


@pytest.mark.parametrize("n,n_blocks,rows", [
    (8192, 98, 2),     # packed: the smallest
    (1953, 98, 8),     # packed, full; one column past a tile
    (2050, 97, 9),     # one tile of 16, odd block count
    (1000, 98, 16),
    (1607, 98, 17),    # two tiles
    (1032, 98, 32),
    (3136, 160, 33),   # four tiles, mostly padding; K = 5120
    (7168, 98, 64),    # two column tiles per workgroup
    (904, 98, 65),     # a second group of one row
    (5120, 98, 300),   # four wavefronts per workgroup
    (3136, 160, 200),  # a workgroup walks several groups
    (37, 130, 1200),   # few columns
    (520, 256, 130),   # the largest K
    (48, 1, 40000),    # one block: most wavefronts have none
    (777, 5, 500),
    (32790, 40, 8), (32790, 40, 16), (32790, 40, 32),  # two column tiles: wide, of short K
    (16400, 98, 8), (16400, 98, 20),                   # and of long K: one
])
def test_rows_match_float64(n, n_blocks, rows):
    say(f"q4 rows n={n} n_blocks={n_blocks} rows={rows}")
    g = rng(900 + n + rows)
    w = Q4(g, n, n_blocks)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    prev = g.standard_normal((rows, n)).astype(np.float32)
    y = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
    relu, acc = torch.empty_like(y), dev(prev)
    with _ctx() as ctx:
        ctx.q4_gemv(dev(x), w.w, y, rows)
        ctx.q4_gemv(dev(x), w.w, relu, rows, nw.NWD_Q4_RELU2)
        ctx.q4_gemv(dev(x), w.w, acc, rows, nw.NWD_Q4_ACCUMULATE)
        got = host(y)
    y64, bound = w.f64(x)
    assert np.all(np.abs(got - y64) <= TOL_REL * bound)
    t = np.maximum(got, np.float32(0))
    np.testing.assert_array_equal(host(relu), t * t)
    np.testing.assert_array_equal(host(acc), prev + got)


def _one_row(ctx, w, x, n):
    """Every row by itself, on the one-row kernels."""
    y = torch.empty((len(x), n), dtype=torch.float32, device="cuda")
    dx = dev(x)
    for b in range(len(x)):
        ctx.q4_gemv(dx[b:b + 1], w.w, y[b:b + 1], 1)
    return host(y)


@pytest.mark.parametrize("n,n_blocks,rows,several", [
    # long K, few columns: faster on the one-row kernels
    (64, 256, 96, False), (100, 256, 70, False), (256, 98, 64, False), (512, 256, 17, False),
    (100, 160, 96, False), (2048, 256, 3, False), (5120, 256, 2, False),
    # and the others
    (1953, 98, 8, True), (1607, 98, 17, True), (904, 98, 65, True), (37, 130, 1200, True),
    (520, 256, 130, True), (2048, 256, 4, True), (3136, 160, 3, True),
])
def test_route(n, n_blocks, rows, several):
    """The kind of kernel that a call takes, told by its bits: the one-row
    kernels give a row the same at every batch, those of several rows sum in
    another order."""
    say(f"q4 rows route n={n} n_blocks={n_blocks} rows={rows}")
    g = rng(990)
    w = Q4(g, n, n_blocks)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    y = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    with _ctx() as ctx:
        ctx.q4_gemv(dev(x), w.w, y, rows)
        same = np.array_equal(host(y), _one_row(ctx, w, x, n))
    assert same == (not several)


def _workspace(H, Hkv, cap, B):
    """Bytes of a context's split-K workspace at head size 128 (nwd_create)."""
    records = max(H * 256, H // Hkv * 512, B * H, min(2 * cap * H * B, 65536))
    return records * 512


def _launch_rows(n_blocks, rows, workspace, records=lambda rows: 0):
    """Rows per launch: all, a multiple of 64, 32, 16 or 8, the most whose
    operands, factors, picks and records the workspace holds (8 rows: high and
    low parts in one tile of 16 rows, 1 KiB a block; more: 2 KiB a block for
    each tile of a group of 1, 2 or 4)."""
    def need(r):
        tiles = 1 if r <= 16 else 2 if r <= 32 else -(-r // 64) * 4
        a = n_blocks * (1024 if r <= 8 else 2048 * tiles)
        return a + -(-r // 4) * 16 + -(-r // 2) * 16 + 16 + 8 * r * records(r)

    sizes = [rows] + list(range((rows - 1) // 64 * 64, 0, -64)) + [32, 16, 8]
    return next(r for r in sizes if r <= rows and need(r) <= workspace)


@pytest.mark.parametrize("heads,per", [(3, 8), (5, 16), (9, 32), (17, 64), (34, 128)])
def test_rows_in_small_workspace(heads, per):
    """A context whose workspace holds `per` activation rows: the call goes
    through it in several launches, the last one ragged, each with the bits
    that a call of its rows has in a roomy context."""
    n, n_blocks, rows = 2048, 256, 150
    say(f"q4 rows in a small workspace, {per} of {rows} rows a launch")
    assert _launch_rows(n_blocks, rows, _workspace(heads, heads, 16, 1)) == per
    g = rng(950)
    w = Q4(g, n, n_blocks)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    dx = dev(x)
    y = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
    parts = torch.empty_like(y)
    with _ctx(heads, heads, 16, 1) as ctx, _ctx() as roomy:
        ctx.q4_gemv(dx, w.w, y, rows)
        for b in range(0, rows, per):
            m = min(per, rows - b)
            roomy.q4_gemv(dx[b:b + m], w.w, parts[b:b + m], m)
        got = host(y)
        np.testing.assert_array_equal(got, host(parts))
        assert not np.array_equal(got, _one_row(ctx, w, x, n))
    y64, bound = w.f64(x)
    assert np.all(np.abs(got - y64) <= TOL_REL * bound)


def test_qkv_rows_in_small_workspace():
    """The same for q/k/v: queries, caches and positions of every launch, a
    wide row and a position outside the cache in later ones."""
    H, Hkv, cap, B, nb = 8, 4, 2, 60, 256
    say(f"qkv rows in a small workspace, B={B}")
    per = _launch_rows(nb, B, _workspace(H, Hkv, cap, B))
    assert per == 16
    g = rng(955)
    wq, wk, wv = Q4(g, H * D, nb), Q4(g, Hkv * D, nb), Q4(g, Hkv * D, nb)
    x = g.standard_normal((B, 32 * nb)).astype(np.float32)
    x[20, 7] = 1e9
    pos = [int(v) for v in g.integers(0, cap, size=B)]
    pos[37] = cap
    canary = -7.5

    def buffers():
        kc = torch.full((B, Hkv, cap, D), canary, dtype=torch.float16, device="cuda")
        return kc, kc.clone(), torch.zeros((B, H, D), dtype=torch.float32, device="cuda")

    whole, parts, dx = buffers(), buffers(), dev(x)
    with _ctx(H, Hkv, cap, B) as ctx:
        ctx.qkv_append(dx, wq.w, wk.w, wv.w, whole[2], whole[0], whole[1], pos_tensor(pos), B)
        assert ctx.device_status() == nw.NWD_ERR_DEVICE
        assert ctx.device_status() == nw.NWD_OK
    roomy_cap = 512  # a workspace for all rows; its caches' first rows are compared
    with _ctx(H, Hkv, roomy_cap, B) as roomy:
        for b in range(0, B, per):
            m = min(per, B - b)
            kc = torch.full((m, Hkv, roomy_cap, D), canary, dtype=torch.float16, device="cuda")
            vc = kc.clone()
            p = pos_tensor([v if v < cap else roomy_cap for v in pos[b:b + m]])
            roomy.qkv_append(dx[b:b + m], wq.w, wk.w, wv.w, parts[2][b:b + m], kc, vc, p, m)
            roomy.device_status()
            parts[0][b:b + m], parts[1][b:b + m] = kc[:, :, :cap], vc[:, :, :cap]
    for a, b in zip(whole, parts):
        np.testing.assert_array_equal(host(a), host(b))
    y64, bound = wq.f64(x)
    assert np.all(np.abs(host(whole[2]).reshape(B, -1) - y64) <= TOL_REL * bound)
    written = np.zeros((B, cap), bool)
    for b in range(B):
        if pos[b] < cap:
            written[b, pos[b]] = True
    for c in whole[:2]:
        at = host(c) != np.float16(canary)
        assert np.array_equal(at.any(axis=(1, 3)), written)


@pytest.mark.parametrize("n,nb,rows,heads,per,records", [
    (16384, 104, 48, 4, 32, lambda r: 256 if r <= 8 else 256 // -(-r // 16)),  # wide picks: 32 and 16 rows
    (8192, 256, 50, 5, 16, lambda r: 512),                                     # the other kernel's
])
def test_lm_head_rows_in_small_workspace(n, nb, rows, heads, per, records):
    say(f"lm_head rows in a small workspace n={n} n_blocks={nb} rows={rows}")
    # past 32 rows both go to the kernel of one record per 32 (here 16) columns
    many = 512 if n >= 16384 else 256
    assert _launch_rows(nb, rows, _workspace(heads, heads, 16, 1),
                        lambda r: records(r) if r <= 32 else many) == per
    g = rng(956)
    w = Q4(g, n, nb)
    x = g.standard_normal((rows, 32 * nb)).astype(np.float32)
    x[33, 7] = 1e9  # a wide row in the second launch
    dx = dev(x)
    logits = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
    parts = torch.empty_like(logits)
    token = torch.full((2, rows), -1, dtype=torch.int32, device="cuda")
    with _ctx(heads, heads, 16, 1) as ctx, _ctx() as roomy:
        ctx.lm_head_argmax(dx, w.w, token[0], logits, rows)
        for b in range(0, rows, per):
            m = min(per, rows - b)
            roomy.lm_head_argmax(dx[b:b + m], w.w, token[1, b:b + m], parts[b:b + m], m)
        got, tok = host(logits), host(token)
    np.testing.assert_array_equal(got, host(parts))
    np.testing.assert_array_equal(tok[0], np.argmax(got, axis=1))
    np.testing.assert_array_equal(tok[1], tok[0])
    y64, bound = w.f64(x)
    assert np.all(np.abs(got - y64) <= TOL_REL * bound)


@pytest.mark.parametrize("n,nb,rows", [(20480, 98, 5), (20480, 33, 17), (4096, 98, 30)])
def test_lm_head_rows_ties_and_non_finite(n, nb, rows):
    """Logits that tie (columns repeated), rows of NaN and of one value: the
    reference's tie order on every kernel."""
    say(f"lm_head rows: ties, NaN n={n} n_blocks={nb} rows={rows}")
    g = rng(957)
    quant, scales, zp = random_q4(g, n // 256, nb)
    cells = n // 256 * nb
    z = np.stack([zp & 15, zp >> 4], axis=1).reshape(-1)[:cells].reshape(n // 256, nb)
    quant, scales, z = (np.tile(a, (256,) + (1,) * (a.ndim - 1)) for a in (quant, scales, z))
    z = z.reshape(-1, 2)
    t = [dev(a) for a in (quant, scales, z[:, 0] | z[:, 1] << 4)]
    w = nw.q4_weight(*t, n, nb)
    x = g.standard_normal((rows, 32 * nb)).astype(np.float32)
    x[1, 40] = np.nan
    x[2, 3] = np.inf
    x[3] = 0
    x[4, 9] = 1e12  # a wide row
    logits = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    token = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
    with _ctx() as ctx:
        ctx.lm_head_argmax(dev(x), w, token, logits, rows)
    got, tok = host(logits), host(token)
    assert np.all(np.isnan(got[1:3])) and np.all(got[3] == 0)
    for b in range(rows):
        assert tok[b] == reference_rule(got[b]), b
        if b not in (1, 2):
            assert (got[b] == got[b].max()).sum() >= 256


def test_rows_ranges_and_non_finite():
    """Rows at the ends of float32's range, of zeros, and with an infinity or
    a NaN, beside ordinary ones."""
    say("q4 rows: ranges, infinities, NaN")
    n, n_blocks, rows = 1200, 98, 14
    g = rng(951)
    w = Q4(g, n, n_blocks)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    x[1] *= np.float32(1e30)
    x[2] *= np.float32(1e-30)
    x[3] = 0
    x[4, 7] = np.inf
    x[5, 3000] = np.nan
    x[6, 100] = -np.inf
    x[7] *= np.float32(1e-41) / np.float32(1e-3)  # subnormals
    x[8, 5] = 3e4  # one large element among small ones
    y = torch.zeros((rows, n), dtype=torch.float32, device="cuda")
    with _ctx() as ctx:
        ctx.q4_gemv(dev(x), w.w, y, rows)
        got = host(y)
    bad = [4, 5, 6]
    assert np.all(np.isnan(got[bad]))
    fine = [b for b in range(rows) if b not in bad]
    y64, bound = w.f64(x[fine])
    # a subnormal result is within half its last place, 2^-150
    assert np.all(np.abs(got[fine] - y64) <= TOL_REL * bound + 2.0 ** -149)


def _hide_block(w, n, n_blocks, blk):
    """Block blk of every column gets no weight: nibbles and zero point 0 in
    even columns (the form the one-row kernels keep exact), 9 in odd ones."""
    quant, _, zp = w.t
    value = torch.arange(n, device="cuda") % 2 * 9
    quant[:, blk] = (value * 17).to(torch.uint8).unsqueeze(1)
    cell = torch.arange(n, device="cuda") * n_blocks + blk
    for half in (0, 1):
        at = cell % 2 == half
        b = cell[at] // 2
        keep = zp[b] & (0xF0 if half == 0 else 0x0F)
        zp[b] = keep | (value[at] << (4 * half)).to(torch.uint8)
    w.dense[:, 32 * blk:32 * blk + 32] = 0


@pytest.mark.parametrize("n,n_blocks,rows,head", [
    (4096, 98, 8, False),     # packed
    (1007, 98, 16, False), (1007, 97, 32, False),
    (3136, 160, 64, False), (5120, 98, 130, False),
    (16400, 98, 7, True), (33001, 98, 48, True),  # wide picks
    (16400, 105, 16, True),                       # the other kernel's
])
def test_wide_rows(n, n_blocks, rows, head):
    """Rows with one activation far above the rest, in a block without
    weight: what the others lose beside it shows, and must be no more than
    on the one-row kernels (the even columns; those lose everything in the
    odd ones, where the large element's products cancel)."""
    say(f"q4 wide rows n={n} n_blocks={n_blocks} rows={rows}")
    g = rng(953 + rows)
    w = Q4(g, n, n_blocks)
    blk = n_blocks // 3
    _hide_block(w, n, n_blocks, blk)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    large = [1e4, 2e5, 1e6, 1e8, 1e20]
    for b in range(0, rows, 2):  # ordinary rows between them
        x[b, 32 * blk + b % 32] = large[b // 2 % len(large)]
    x[1, :32] *= np.float32(1e-6)  # the other way about: a block far below the rest
    y = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
    token = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
    dx = dev(x)
    with _ctx() as ctx:
        if head:
            ctx.lm_head_argmax(dx, w.w, token, y, rows)
        else:
            ctx.q4_gemv(dx, w.w, y, rows)
        got, one = host(y), _one_row(ctx, w, x, n)
    y64, bound = w.f64(x)  # the large elements are not in the bound
    assert np.all(np.abs(got - y64) <= TOL_REL * bound)

    def err(v):
        return np.linalg.norm((v - y64)[:, ::2], axis=1) / np.linalg.norm(y64[:, ::2], axis=1)

    # 2-norms over hundreds of columns of errors of one size: 1.25 is far
    # outside their spread, and the parts gave 2 (at 1e6) to 10^6 times
    assert np.all(err(got) <= 1.25 * err(one)), (err(got) / err(one)).max()
    if head:
        np.testing.assert_array_equal(host(token), np.argmax(got, axis=1))


@pytest.mark.parametrize("H,Hkv,q,Dh,B", [(40, 8, "f32", 128, 3), (32, 8, "f16", 128, 12),
                                          (14, 2, "f32", 64, 40), (6, 2, "f16", 96, 64)])
def test_qkv_rows(H, Hkv, q, Dh, B):
    """q, k and v through the fused projection; the last sequence's position
    is outside its cache: nothing is written there and it is reported."""
    say(f"qkv rows H={H} Hkv={Hkv} D={Dh} B={B}")
    g = rng(960 + B)
    cap, nb = 24, 98
    wq, wk, wv = Q4(g, H * Dh, nb), Q4(g, Hkv * Dh, nb), Q4(g, Hkv * Dh, nb)
    x = g.standard_normal((B, 32 * nb)).astype(np.float32)
    pos = [int(v) for v in g.integers(0, cap, size=B)]
    pos[-1] = cap
    canary = -7.5
    with _ctx(H, Hkv, cap, B, q, Dh) as ctx:
        kc = torch.full((B, Hkv, cap, Dh), canary, dtype=torch.float16, device="cuda")
        vc = kc.clone()
        qo = torch.empty((B, H, Dh), dtype=torch.float32 if q == "f32" else torch.float16, device="cuda")
        ctx.qkv_append(dev(x), wq.w, wk.w, wv.w, qo, kc, vc, pos_tensor(pos), B)
        assert ctx.device_status() == nw.NWD_ERR_DEVICE
        assert ctx.device_status() == nw.NWD_OK
        qh, kh, vh = host(qo).astype(np.float64), host(kc), host(vc)

    def ulp(v):
        h = v.astype(np.float16)
        return np.abs((np.nextafter(h, np.float16(np.inf)) - h).astype(np.float64))

    y64, bound = wq.f64(x)
    assert np.all(np.abs(qh.reshape(B, -1) - y64) <= TOL_REL * bound + (ulp(y64) if q == "f16" else 0))
    for w, c in ((wk, kh), (wv, vh)):
        y64, bound = w.f64(x)
        for b in range(B):
            row = slice(0, 0) if pos[b] == cap else slice(pos[b], pos[b] + 1)
            got = c[b, :, row, :].astype(np.float64).reshape(-1)
            if got.size:
                assert np.all(np.abs(got - y64[b]) <= TOL_REL * bound[b] + ulp(y64[b])), b
            assert np.all(np.delete(c[b], row, axis=1) == np.float16(canary)), b


@pytest.mark.parametrize("n,n_blocks,rows", [(20011, 98, 4), (20011, 98, 16), (16384, 97, 20), (33000, 33, 70),
                                                (33001, 104, 48), (20017, 104, 48), (17001, 8, 48),
                                                (20480, 105, 9), (16401, 130, 25), (16400, 160, 32)])
def test_lm_head_rows(n, n_blocks, rows):
    say(f"lm_head rows n={n} n_blocks={n_blocks} rows={rows}")
    g = rng(970 + rows)
    w = Q4(g, n, n_blocks)
    x = g.standard_normal((rows, 32 * n_blocks)).astype(np.float32)
    logits = torch.empty((rows, n), dtype=torch.float32, device="cuda")
    token = torch.full((2, rows), -1, dtype=torch.int32, device="cuda")
    with _ctx() as ctx:
        ctx.lm_head_argmax(dev(x), w.w, token[0], logits, rows)
        ctx.lm_head_argmax(dev(x), w.w, token[1], None, rows)
        got, tok = host(logits), host(token)
    y64, bound = w.f64(x)
    assert np.all(np.abs(got - y64) <= TOL_REL * bound)
    np.testing.assert_array_equal(tok[0], np.argmax(got, axis=1))
    np.testing.assert_array_equal(tok[1], tok[0])


@pytest.mark.parametrize("n,n_blocks,rows,wide", [(33001, 97, 33, True), (20011, 98, 33, False),
                                                  (33001, 20, 40, False)])
def test_pick_route(n, n_blocks, rows, wide):
    """Picks of 33 to 48 rows: on the wide pick kernel, which gives a row of
    every row tile the bits of its 16-row form, or on the other, whose
    64-row form sums in another order."""
    say(f"lm_head route n={n} n_blocks={n_blocks} rows={rows}")
    g = rng(981)
    w = Q4(g, n, n_blocks)
    dx = dev(g.standard_normal((rows, 32 * n_blocks)).astype(np.float32))
    many, few = (torch.empty((r, n), dtype=torch.float32, device="cuda") for r in (rows, 16))
    token = torch.empty(rows, dtype=torch.int32, device="cuda")
    with _ctx() as ctx:
        ctx.lm_head_argmax(dx, w.w, token, many, rows)
        ctx.lm_head_argmax(dx[16:32], w.w, token, few, 16)
        assert np.array_equal(host(many)[16:32], host(few)) == wide


def test_lm_head_fills_the_workspace():
    """Batches up to the largest that the workspace takes (128 rows of 1024
    records here, its 1 MiB) run the kernels of several rows as they do in a
    roomy context: the same bits. One row more is refused."""
    say("lm_head in a full workspace")
    n, nb = 16384, 20
    g = rng(980)
    w = Q4(g, n, nb)
    x = g.standard_normal((129, 32 * nb)).astype(np.float32)
    dx = dev(x)
    y64, bound = w.f64(x)
    with _ctx(4, 4, 256, 1) as small, _ctx() as roomy:
        for rows in (60, 100, 126, 128):
            got, tok = [], []
            for ctx in (small, roomy):
                logits = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
                token = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
                ctx.lm_head_argmax(dx, w.w, token, logits, rows)
                got.append(host(logits))
                tok.append(host(token))
            np.testing.assert_array_equal(got[0], got[1])
            np.testing.assert_array_equal(tok[0], np.argmax(got[0], axis=1))
            np.testing.assert_array_equal(tok[1], tok[0])
            assert np.all(np.abs(got[0] - y64[:rows]) <= TOL_REL * bound[:rows])
        with pytest.raises(nw.NwdError):
            small.lm_head_argmax(dx, w.w, torch.empty(129, dtype=torch.int32, device="cuda"), None, 129)


def test_rows_in_a_graph():
    """q/k/v, a projection onto it and the wide pick of several rows, captured
    once and replayed on new activations (wide rows in some), with eager calls
    between: every replay gives the eager bits."""
    say("q4 rows in a graph")
    H, Hkv, cap, B, nb = 8, 8, 16, 12, 98
    g = rng(995)
    wq, wk, wv = Q4(g, H * D, nb), Q4(g, Hkv * D, nb), Q4(g, Hkv * D, nb)
    wo, wl = Q4(g, 4096, H * D // 32), Q4(g, 16390, nb)
    x = torch.zeros((B, 32 * nb), dtype=torch.float32, device="cuda")
    pos = pos_tensor([b % cap for b in range(B)])

    def buffers():
        kc = torch.zeros((B, Hkv, cap, D), dtype=torch.float16, device="cuda")
        return (torch.zeros((B, H * D), device="cuda"), kc, kc.clone(), torch.zeros((B, 4096), device="cuda"),
                torch.zeros((B, 16390), device="cuda"), torch.zeros(B, dtype=torch.int32, device="cuda"))

    def run(ctx, stream, q, kc, vc, h, logits, token):
        ctx.qkv_append(x, wq.w, wk.w, wv.w, q, kc, vc, pos, B, stream=stream)
        ctx.q4_gemv(q, wo.w, h, B, stream=stream)
        ctx.lm_head_argmax(x, wl.w, token, logits, B, stream=stream)

    captured, eager = buffers(), buffers()
    with _ctx(H, Hkv, cap, B) as ctx, _ctx(H, Hkv, cap, B) as other:
        stream = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            run(ctx, stream, *captured)
        for i in range(4):
            v = g.standard_normal((B, 32 * nb)).astype(np.float32)
            if i % 2:
                v[i, 9] = 1e12
            x.copy_(dev(v))
            graph.replay()
            run(other, None, *eager)
            for a, b in zip(captured, eager):
                np.testing.assert_array_equal(host(a), host(b))
