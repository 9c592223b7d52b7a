"""The Q8_0 / Q4_0 products on the matrix cores (csrc/gemm_q32.hip) at the edges of their tiles, against
the oracle bit for bit: rows and tokens around 32, 64 and 128, row lengths of whole and partial
four-block stages, matrices at every even offset of a 16-byte piece, the wide form, infinite and NaN
scales, and expert lists longer than the launch's grid."""
import numpy as np
import pytest
import torch

from gpu_util import announce, assert_same, dev, host, require_gpu
from oracle import oracle as o

pytestmark = pytest.mark.gpu
BYTES = {o.Q8_0: 34, o.Q4_0: 18}


@pytest.fixture(scope="module")
def S():
    require_gpu()
    import syntropy_amd.gemv as S
    return S


def blocks(rs, ty, n_out, k):
    """Random codes, F16 scales of either sign with biased exponents 3..12."""
    nb = n_out * k // 32
    b = rs.integers(0, 256, (nb, BYTES[ty]), dtype=np.uint8)
    h = (rs.integers(0, 2, nb) << 15) | (rs.integers(3, 13, nb) << 10) | rs.integers(0, 1024, nb)
    b[:, :2] = h.astype(np.uint16).view(np.uint8).reshape(nb, 2)
    return b.reshape(-1)


def check(S, ty, w, n_out, k, x, rows, what):
    want = o.gemv(ty, w, n_out, k, x, rows, threads=16)
    announce(what)
    W = S.Weights(S.WeightType(ty), dev(w), n_out, k)
    assert_same(host(S.gemv(W, dev(x), rows)), want, what)
    assert_same(host(S.gemv(S.repack(W), dev(x), rows)), want, what + " split")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
@pytest.mark.parametrize("rows,n_out,k", [
    (8, 1, 32), (9, 31, 64), (17, 33, 96), (32, 64, 128), (33, 65, 160), (63, 63, 256), (64, 130, 288),
    (65, 32, 1056), (130, 97, 416), (40, 3, 2080), (35, 129, 4128), (1, 64, 160), (5, 64, 160)])
def test_tile_edges(S, ty, rows, n_out, k):
    rs = np.random.default_rng(rows * 131 + n_out + k)
    x = rs.standard_normal((rows, k)).astype(np.float32)
    check(S, ty, blocks(rs, ty, n_out, k), n_out, k, x, rows, f"q32 ty={ty} rows={rows} {n_out}x{k}")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
@pytest.mark.parametrize("rows,n_out,k", [(2100, 2053, 96), (1025, 4099, 160)])
def test_wide_form(S, ty, rows, n_out, k):
    """Two token tiles a wavefront, the last of them partial or empty."""
    rs = np.random.default_rng(rows + k)
    x = rs.standard_normal((rows, k)).astype(np.float32)
    check(S, ty, blocks(rs, ty, n_out, k), n_out, k, x, rows, f"q32 wide ty={ty} rows={rows} {n_out}x{k}")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
def test_offsets(S, ty):
    """GGUF rows from any address: every even offset of a 16-byte piece, and odd ones."""
    n_out, k, rows = 37, 224, 20
    rs = np.random.default_rng(5)
    w, x = blocks(rs, ty, n_out, k), rs.standard_normal((rows, k)).astype(np.float32)
    want = o.gemv(ty, w, n_out, k, x, rows)
    for at in (1, 2, 4, 6, 8, 10, 12, 13, 14):
        buf = torch.zeros(w.size + 32, dtype=torch.uint8, device="cuda")
        buf[at:at + w.size] = dev(w)
        announce(f"q32 ty={ty} at {at}")
        W = S.Weights(S.WeightType(ty), buf[at:at + w.size], n_out, k)
        assert_same(host(S.gemv(W, dev(x), rows)), want, f"at {at}")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
def test_infinite_and_nan_scales(S, ty):
    """An infinite weight scale or activation scale (past F16's range), a NaN one, a NaN activation, an
    all-zero row: the reference's infinities and NaNs, and every other output as it is."""
    n_out, k, rows = 70, 192, 40
    rs = np.random.default_rng(11)
    w = blocks(rs, ty, n_out, k).reshape(n_out, k // 32, BYTES[ty])
    w[3, 2, :2] = np.array([0x7C00], np.uint16).view(np.uint8)
    w[40, 0, :2] = np.array([0xFC00], np.uint16).view(np.uint8)
    w[66, 5, :2] = np.array([0x7E00], np.uint16).view(np.uint8)
    w[50, 1, :2] = 0
    x = rs.standard_normal((rows, k)).astype(np.float32)
    x[2, 33:64] *= 3e8   # the block's scale rounds to an infinity
    x[34, 70] = np.nan
    x[35, 5] = np.inf
    x[36] = 0.0
    x[37] *= 1e-6        # subnormal scales
    check(S, ty, w.reshape(-1), n_out, k, x, rows, f"q32 ty={ty} infinite scales")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
@pytest.mark.parametrize("rows,n_out,k", [(33, 40, 1056), (1025, 4099, 160)])  # one and two token tiles a wavefront
def test_many_infinite_scales(S, ty, rows, n_out, k):
    """Whole rows of infinite weight scales and activation scales, of one sign and of both, and infinities
    in the last block of a partial stage and past the first 16 blocks."""
    rs = np.random.default_rng(rows + 3)
    nb = k // 32
    w = blocks(rs, ty, n_out, k).reshape(n_out, nb, BYTES[ty])
    f16 = lambda h: np.array([h], np.uint16).view(np.uint8)
    w[0, :, :2] = f16(0x7C00)
    w[1, ::2, :2], w[1, 1::2, :2] = f16(0x7C00), f16(0xFC00)
    w[33, nb - 1, :2] = f16(0xFC00)
    w[35, :, 2:] = 0x88  # sums of one sign (Q8_0) or zero (Q4_0): an infinity times zero
    w[35, 1, :2] = f16(0x7C00)
    w[38, nb // 2, :2] = f16(0x7E01)
    x = rs.standard_normal((rows, k)).astype(np.float32)
    x[1] *= 1e9
    x[2] = np.abs(x[2]) * 1e9
    x[rows - 1, k - 3] = -4e9
    x[rows - 2, : 16 * 32 if nb > 16 else 64] = np.inf
    check(S, ty, w.reshape(-1), n_out, k, x, rows, f"q32 ty={ty} many infinities {rows} {n_out}x{k}")


@pytest.mark.parametrize("ty,split", [(o.Q8_0, False), (o.Q4_0, False), (o.Q8_0, True)])
def test_nan_and_infinity_take_no_longer(S, ty, split):
    """A NaN row of activations, an activation past the scales' range and an infinite weight scale, each
    at the end of a row: at most one more pass over the rows' blocks (measured up to 1.5 times the call
    without; the outputs one by one took 10 to 150 times it)."""
    n_out, k, rows = 2048, 8192, 1024 if split else 64
    rs = np.random.default_rng(29)
    w = blocks(rs, ty, n_out, k)
    x = rs.standard_normal((rows, k)).astype(np.float32)
    y = torch.empty(rows, n_out, device="cuda")

    def micros(w, x):
        W = S.Weights(S.WeightType(ty), dev(w), n_out, k)
        W, xd = S.repack(W) if split else W, dev(x)
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        best = float("inf")
        for _ in range(5):
            ev[0].record()
            for _ in range(4):
                S.gemv(W, xd, rows, y=y)
            ev[1].record()
            torch.cuda.synchronize()
            best = min(best, 250 * ev[0].elapsed_time(ev[1]))
        return best

    announce(f"q32 ty={ty} split={split} time with NaNs")
    clean = micros(w, x)
    nan, big, winf = x.copy(), x.copy(), w.copy()
    nan[3] = np.nan
    big[3, -1] = 1e9
    winf.reshape(n_out, k // 32, -1)[5, -1, :2] = np.array([0x7C00], np.uint16).view(np.uint8)
    for what, t in (("NaN row", micros(w, nan)), ("infinite token scale", micros(w, big)),
                    ("infinite weight scale", micros(winf, x))):
        assert t < 4 * clean, f"{what}: {t:.0f} us against {clean:.0f}"


@pytest.mark.parametrize("E,top_k,hidden,inter,rows,popular", [
    (4, 1, 160, 96, 300, 290),    # one expert's entries beyond the grid's tiles
    (3, 2, 64, 224, 70, 65), (6, 2, 288, 64, 90, 0), (16, 2, 96, 160, 33, 20), (1, 1, 32, 32, 129, 129)])
def test_experts(S, E, top_k, hidden, inter, rows, popular):
    import syntropy_amd.moe as M
    rs = np.random.default_rng(E * 7 + rows)
    gate, up, down = (blocks(rs, o.Q8_0, E * n, k) for n, k in ((inter, hidden), (inter, hidden), (hidden, inter)))
    up.reshape(E, inter, hidden // 32, 34)[0, 5, 0, :2] = np.array([0x7C00], np.uint16).view(np.uint8)
    x = rs.standard_normal((rows, hidden)).astype(np.float32)
    ids = np.stack([rs.permutation(E)[:top_k] for _ in range(rows)]).astype(np.int32)
    ids[:popular, 0] = 0
    if top_k > 1:
        ids[:popular, 1:] = 1 + np.arange(top_k - 1)
    want = o.moe_grouped(o.Q8_0, o.Q8_0, E, top_k, hidden, inter, gate, up, down, x, ids, threads=8)
    announce(f"q32 experts E={E} k={top_k} {hidden} {inter} rows={rows}")
    ex = M.Experts(M.WeightType.Q8_0, dev(gate), dev(up), dev(down))
    got = M.moe_grouped(M.MoeShape(E, top_k, hidden, inter), ex, dev(x), dev(ids))
    assert_same(host(got), want, "experts")


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
@pytest.mark.parametrize("rows,n_out,k,at", [(20, 100, 96, 1), (70, 68, 160, 2), (1025, 4100, 64, 3), (33, 31, 96, 0)])
def test_outputs_at_any_address(S, ty, rows, n_out, k, at):
    """Outputs that no row starts at 16 bytes of (the tile goes through LDS), one and two token tiles a
    wavefront: the values, and nothing written beside them."""
    rs = np.random.default_rng(rows + n_out + at)
    w, x = blocks(rs, ty, n_out, k), rs.standard_normal((rows, k)).astype(np.float32)
    want = o.gemv(ty, w, n_out, k, x, rows, threads=16)
    W = S.Weights(S.WeightType(ty), dev(w), n_out, k)
    for name, w_ in (("gguf", W), ("split", S.repack(W))):
        buf = torch.full((rows * n_out + 64,), 7.5, device="cuda")
        announce(f"q32 ty={ty} {name} {rows} {n_out}x{k} y at {at}")
        S.gemv(w_, dev(x), rows, y=buf[at:at + rows * n_out])
        got = host(buf)
        assert_same(got[at:at + rows * n_out], want, f"{name} y at {at}")
        assert (got[:at] == 7.5).all() and (got[at + rows * n_out:] == 7.5).all()


@pytest.mark.parametrize("ty", [o.Q8_0, o.Q4_0])
def test_ragged_outputs_take_no_longer(S, ty):
    """1411 rows of 4098 outputs against 4100, as many tiles (measured: up to 1.1 times; four bytes of 32
    rows at a time took 1.4 times)."""
    k, rows = 512, 1411
    rs = np.random.default_rng(31)
    x = dev(rs.standard_normal((rows, k)).astype(np.float32))
    Ws = [S.repack(S.Weights(S.WeightType(ty), dev(blocks(rs, ty, n, k)), n, k)) for n in (4100, 4098)]
    ys = [torch.empty(rows, W.n_out, device="cuda") for W in Ws]
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    best = [float("inf")] * 2
    announce(f"q32 ty={ty} ragged outputs")
    for _ in range(8):
        for i, W in enumerate(Ws):
            ev[0].record()
            for _ in range(10):
                S.gemv(W, x, rows, y=ys[i])
            ev[1].record()
            torch.cuda.synchronize()
            best[i] = min(best[i], 100 * ev[0].elapsed_time(ev[1]))
    print(f"4100: {best[0]:.1f} us, 4098: {best[1]:.1f} us")
    assert best[1] < 1.25 * best[0]


@pytest.mark.parametrize("k,rows", [(4128, 9), (4096, 40), (4128, 70), (4096, 130)])
def test_split_matrix_past_32_bit_offsets(S, k, rows):
    """A Q8_0 SPLIT matrix of more than 4 GiB, which the register-staged kernel takes (16 and 32 tokens a
    tile, rows of whole and of odd stages): slices at both ends and around the 4 GiB mark."""
    n_out, nb = 1_050_003, k // 32
    g = torch.Generator("cuda").manual_seed(k + rows)
    buf = torch.empty(n_out * nb * 34, dtype=torch.uint8, device="cuda")
    codes, scales = buf[:n_out * k], buf[n_out * k:].view(torch.int16)
    for a in range(0, codes.numel(), 1 << 30):
        codes[a:a + (1 << 30)].random_(0, 256, generator=g)
    scales.random_(3 << 10, 13 << 10, generator=g)
    x = torch.randn(rows, k, generator=g, device="cuda")
    announce(f"q8_0 split {n_out}x{k} rows {rows}")
    y = S.gemv(S.Weights(S.WeightType.Q8_0, buf, n_out, k, S.LAYOUT_SPLIT), x, rows)
    for a in (0, (1 << 32) // k - 16, n_out - 33):
        w = np.empty((33, nb, 34), np.uint8)
        w[:, :, 2:] = host(codes[a * k:(a + 33) * k]).reshape(33, nb, 32)
        w[:, :, :2] = host(scales[a * nb:(a + 33) * nb]).view(np.uint8).reshape(33, nb, 2)
        want = o.gemv(o.Q8_0, w.reshape(-1), 33, k, host(x), rows, threads=16)
        assert_same(host(y[:, a:a + 33].contiguous()), want, f"outputs from {a}")


@pytest.mark.parametrize("hidden,inter", [(61_696, 65_536), (61_728, 65_504)])  # rows of whole 16-byte pieces, or not
def test_expert_past_32_bit_offsets(S, hidden, inter):
    """One Q8_0 expert whose matrices hold about 4 GiB each, past gemm_q32.hip's 32-bit offsets, against the
    dense ops over row slices."""
    import syntropy_amd.moe as M
    rows, part = 3, 8192
    g = torch.Generator("cuda").manual_seed(41)

    def matrix(n, k):
        m = torch.empty(n * (k // 32) * 17, dtype=torch.int16, device="cuda")
        for a in range(0, m.numel(), 1 << 30):
            m[a:a + (1 << 30)].random_(generator=g)
        m.view(-1, 17)[:, 0].random_(1 << 10, 5 << 10, generator=g)
        return m.view(torch.uint8)

    gate, up, down = matrix(inter, hidden), matrix(inter, hidden), matrix(hidden, inter)
    assert gate.numel() >= (1 << 32) - 65536
    x = torch.randn(rows, hidden, generator=g, device="cuda")
    ids = torch.zeros(rows, 1, dtype=torch.int32, device="cuda")
    announce(f"q8_0 expert {inter}x{hidden}")
    got = M.moe_grouped(M.MoeShape(1, 1, hidden, inter), M.Experts(M.WeightType.Q8_0, gate, up, down), x, ids)
    assert torch.isfinite(got).all()
    h = torch.empty(rows, inter, device="cuda")
    rb = hidden // 32 * 34
    for a in range(0, inter, part):
        n = min(part, inter - a)
        w = torch.cat([gate[a * rb:(a + n) * rb], up[a * rb:(a + n) * rb]])
        h[:, a:a + n] = S.gate_up_act(S.Weights(S.WeightType.Q8_0, w, 2 * n, hidden), x, rows)
    rb = inter // 32 * 34
    for a in range(0, hidden, part):
        n = min(part, hidden - a)
        want = S.gemv(S.Weights(S.WeightType.Q8_0, down[a * rb:(a + n) * rb].clone(), n, inter), h, rows)
        assert_same(host(got.view(rows, hidden)[:, a:a + n].contiguous()), host(want), f"outputs from {a}")
