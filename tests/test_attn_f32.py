"""The fp32 attention kernels on the fp32 matrix cores (attn_f32.hip): every
block shape of the forward and the backward against the float64 closed forms,
with rows that do not start on 16-byte boundaries, grouped heads, ragged
tiles and bands; and the LDS layout's bank property (CPU)."""

import numpy as np
import pytest

from oracle import closed_forms as cf
from tests.test_lds_layout import _ways

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("D", [64, 128])
def test_lds_reads_hit_distinct_banks(D):
    """Slot x of row r is stored at x ^ (r & 15): row reads (lane 16 G + c:
    row c, chunk 4 s + G) under the measured b128 rule, feature reads (row
    4 G + j, float 16 f + c) over all 64 four-byte banks at once."""
    L = range(64)
    for s in range(D // 16):
        assert _ways([(l & 15) * D * 4 + (((4 * s + (l >> 4)) ^ (l & 15)) << 4) for l in L], 16) == 1
    for f in range(D // 16):
        for j in range(4):
            words = set()
            for l in L:
                row, col = 4 * (l >> 4) + j, 16 * f + (l & 15)
                words.add(((row * D * 4 + (((col >> 2) ^ row) << 4) + (col & 3) * 4) // 4) % 64)
            assert len(words) == 64


def _tensor(gen, shape, offset):
    """Standard normals, dense, starting ``offset`` elements into their storage."""
    n = int(np.prod(shape))
    flat = torch.randn(n + offset, generator=gen, device="cuda", dtype=torch.float32)
    return flat[offset:].view(shape)


# (B, Hq, Hkv, T, S, D, band): (rows of a forward block, rows of a backward block) the launcher picks
CASES = {
    # the smallest, one short tile each
    (1, 1, 1, 1, 1, 64, None): (16, 16),
    (1, 1, 1, 15, 17, 128, (None, 2)): (16, 16),
    # 16-row blocks, keys over the waves (forward) and rings (backward)
    (1, 2, 1, 100, 333, 64, (-70, 240)): (16, 16),
    (1, 3, 3, 65, 64, 128, (None, -1)): (16, 16),  # a fully masked row: no prune
    (2, 4, 1, 130, 130, 128, (None, 0)): (16, 16),  # a group's key blocks sweep four heads
    (2, 40, 40, 95, 95, 128, None): (16, 64),
    # 32-row blocks, two waves on the keys
    (2, 32, 8, 150, 270, 64, (None, 120)): (32, 16),
    (2, 40, 40, 128, 95, 128, None): (32, 64),
    (1, 40, 20, 201, 310, 128, (-30, 140)): (32, 16),
    # 64-row blocks
    (4, 64, 32, 100, 65, 64, (-20, None)): (64, 64),
    (4, 64, 32, 100, 65, 128, (None, 9)): (64, 64),
    # 128-row blocks of eight waves
    (4, 64, 32, 129, 65, 64, (-20, 3)): (128, 64),
    (8, 64, 64, 129, 65, 64, (None, 0)): (128, 64),
    (8, 64, 16, 70, 97, 128, (-60, None)): (128, 64),
}


def _block_rows(B, Hq, Hkv, T, S, D, cus=256):
    """launch_fwd's and launch_bwd's choice (attn_f32.hip)."""
    q = lambda rows: B * Hq * -(-T // rows)  # noqa: E731
    fwd = 128 if q(128) >= 2 * cus else 64 if q(64) >= 2 * cus else 32 if q(32) >= cus else 16
    limit = 2 * cus if D == 64 or Hq > Hkv else 3 * cus // 4
    return fwd, 16 if q(64) + B * Hkv * -(-S // 64) < limit else 64


def test_the_cases_reach_every_block_shape():
    reached = set()
    for (*shape, _band), want in CASES.items():
        assert _block_rows(*shape) == want, shape
        reached |= {(shape[-1], "forward", want[0]), (shape[-1], "backward", want[1])}
    assert reached == {(D, *x) for D in (64, 128) for x in (("forward", 16), ("forward", 32), ("forward", 64),
                                                            ("forward", 128), ("backward", 16), ("backward", 64))}


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("B,Hq,Hkv,T,S,D,band", CASES)
def test_forward_and_backward_match_the_closed_forms(B, Hq, Hkv, T, S, D, band, offset):
    """Sampled (batch, K / V head) groups, every query head of each: 1e-5 of
    scale, the fp32 bound of the other attention tests (sums of at most a few
    hundred fp32 products)."""
    from pdum_dsl_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(T * 31 + S + D)
    q, do = (_tensor(gen, (B, Hq, T, D), offset) for _ in range(2))
    k, v = (_tensor(gen, (B, Hkv, S, D), offset) for _ in range(2))
    out = _tensor(gen, (B, Hq, T, D), offset)
    kb = K.Band(*band) if band is not None else None
    scale = D**-0.5
    fw = K.flash_fwd(q, k, v, band=kb, want_artifacts=True, out=out)
    grads = [K.flash_bwd(q, k, v, fw.o, do, fw.lse, band=kb),
             K.flash_bwd(q, k, v, fw.o, do, fw.lse, m=fw.m, den=fw.den, band=kb)]
    torch.cuda.synchronize()
    h = lambda t: t.double().cpu().numpy()  # noqa: E731
    close = lambda got, want, what: np.testing.assert_allclose(  # noqa: E731
        h(got), want, rtol=0, atol=1e-5 * max(1.0, np.abs(want).max()), err_msg=what)
    group = Hq // Hkv
    for b, hk in {(0, 0), (B - 1, Hkv - 1)}:
        wk, wv = np.zeros((S, D)), np.zeros((S, D))
        for hq in range(hk * group, (hk + 1) * group):
            Q, Kh, V, dO = h(q[b, hq]), h(k[b, hk]), h(v[b, hk]), h(do[b, hq])
            o, m, den, lse = cf.attention(Q, Kh, V, scale=scale, band=band)
            for got, want, what in ((fw.o, o, "o"), (fw.lse, lse, "lse"), (fw.m, m, "m")):
                close(got[b, hq], want, what)
            np.testing.assert_allclose(h(fw.den[b, hq]), den, rtol=1e-5, err_msg="den")
            gq, gk, gv = cf.attention_bwd(Q, Kh, V, dO, scale=scale, band=band)
            wk += gk
            wv += gv
            for g in grads:
                close(g[0][b, hq], gq, "dq")
        for g in grads:
            close(g[1][b, hk], wk, "dk")
            close(g[2][b, hk], wv, "dv")


@pytest.mark.gpu
@pytest.mark.parametrize(
    "B,H,T,D,band,bound",
    [
        (2, 12, 1000, 64, (None, 0), (4.97e-7, 8.13e-7, 8.04e-7)),
        (2, 32, 700, 128, (-200, 0), (5.38e-7, 5.77e-7, 5.20e-7)),
    ],
)
def test_gradients_stay_as_close_to_64_bits_as_fp32_sums_in_order(B, H, T, D, band, bound):
    """The 64-row backward's relative errors (2-norm) of dQ, dK, dV against
    float64: no larger than those of the fp32 VALU kernels (bwd_rows_f32), one
    running sum per element, measured on inputs of this distribution."""
    from pdum_dsl_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(1)
    q, k, v, do = (_tensor(gen, (B, H, T, D), 0) for _ in range(4))
    fw = K.flash_fwd(q, k, v, band=K.Band(*band))
    got = K.flash_bwd(q, k, v, fw.o, do, fw.lse, band=K.Band(*band))
    torch.cuda.synchronize()
    err, size = np.zeros(3), np.zeros(3)
    for b in range(B):
        for h in range(0, H, 5):
            x = [t[b, h].double().cpu().numpy() for t in (q, k, v, do)]
            for i, want in enumerate(cf.attention_bwd(*x, scale=D**-0.5, band=band)):
                err[i] += ((got[i][b, h].double().cpu().numpy() - want) ** 2).sum()
                size[i] += (want**2).sum()
    assert (np.sqrt(err / size) <= bound).all(), np.sqrt(err / size)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,T,S,D", [(1, 2, 70, 400, 64), (2, 32, 100, 300, 128), (4, 64, 100, 190, 64),
                                       (4, 64, 100, 190, 128), (8, 64, 129, 200, 64)])
def test_a_pruned_window_is_bit_equal_to_the_full_sweep(B, H, T, S, D):
    """A window leaves dead keys on both sides of a block's range; in the full
    sweep their fill scores must vanish from every state."""
    from pdum_dsl_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(T)
    q = _tensor(gen, (B, H, T, D), 0)
    k, v = (_tensor(gen, (B, H, S, D), 0) for _ in range(2))
    band = K.Band(40, 90)
    full = K.flash_fwd(q, k, v, band=band, prune=False, want_artifacts=True)
    cut = K.flash_fwd(q, k, v, band=band, prune=True, want_artifacts=True)
    torch.cuda.synchronize()
    for x in ("o", "lse", "m", "den"):
        assert torch.equal(getattr(full, x), getattr(cut, x)), x


@pytest.mark.gpu
@pytest.mark.parametrize("fill", [float("-inf"), torch.finfo(torch.float32).min], ids=["-inf", "lowest"])
@pytest.mark.parametrize("H,T,S,D", [(2, 130, 321, 64), (40, 224, 300, 64), (2, 130, 321, 128), (3, 70, 200, 32), (2, 70, 200, 40)])
def test_the_lowest_fills_leave_live_rows_finite(H, T, S, D, fill):
    """Whole tiles a row sees only as masked, with fills whose score is -inf or
    the lowest value, on the matrix-core, row and generic kernels: they add
    nothing, pruned or not."""
    from pdum_dsl_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(D + T)
    q = _tensor(gen, (1, H, T, D), 0)
    k, v = (_tensor(gen, (1, H, S, D), 0) for _ in range(2))
    band = (65, 120)  # the last rows' first live key is past three 64-key chunks
    if T + band[0] > S:
        band = (65 - T, 10)
    outs = [K.flash_fwd(q, k, v, band=K.Band(*band), fill=fill, prune=p) for p in (True, False)]
    torch.cuda.synchronize()
    for out in outs:
        for h in (0, H - 1):
            x = [t[0, h].double().cpu().numpy() for t in (q, k, v)]
            o, _m, _den, lse = cf.attention(*x, scale=D**-0.5, band=band)
            np.testing.assert_allclose(out.o[0, h].double().cpu().numpy(), o, rtol=0, atol=1e-5)
            np.testing.assert_allclose(out.lse[0, h].double().cpu().numpy(), lse, rtol=0, atol=1e-5)


@pytest.mark.gpu
def test_strided_and_broadcast_operands():
    """Rows of a wider tensor (a stride that is no multiple of four), heads
    behind rows, and K / V rows repeated by a zero stride."""
    from pdum_dsl_amd import kernels as K

    gen = torch.Generator(device="cuda").manual_seed(3)
    wide = torch.randn((2, 90, 3, 67), generator=gen, device="cuda")
    q = wide[..., 1:65].transpose(1, 2)
    k = torch.randn((2, 50, 3, 64), generator=gen, device="cuda").transpose(1, 2)
    v = torch.randn((2, 3, 1, 64), generator=gen, device="cuda").expand(2, 3, 50, 64)
    r = K.flash_fwd(q, k, v)
    torch.cuda.synchronize()
    for b, hh in ((0, 0), (1, 2)):
        want = cf.attention(*(t[b, hh].double().cpu().numpy() for t in (q, k, v)), scale=0.125)[0]
        np.testing.assert_allclose(r.o[b, hh].double().cpu().numpy(), want, rtol=0, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "D,stride",
    [
        (64, 2**23 - 4),  # the widest rows the matrix-core kernels take: a staged tile spans just under 2 GiB
        (64, 2**23 - 3),  # the same, rows not 16-byte aligned
        (64, 2**23),  # past it: the row kernel
        (128, 2**24 - 4),
        (128, 2**24),  # past it: the wave-per-row kernel
    ],
)
@pytest.mark.parametrize("H", [2, 40])  # 16-row blocks; 32-row blocks, which stage the longest tiles
def test_rows_far_apart(D, stride, H):
    """K rows up to 64 MiB apart (one batch entry of a [rows][batch * heads * D]
    tensor), NaN between them."""
    from pdum_dsl_amd import kernels as K

    T, S, Hkv = 224, 67, 2
    gen = torch.Generator(device="cuda").manual_seed(D + H)
    q, kc, v = (_tensor(gen, (1, h, n, D), 0) for h, n in ((H, T), (Hkv, S), (Hkv, S)))
    flat = torch.full(((S - 1) * stride + Hkv * D,), float("nan"), device="cuda")
    k = flat.as_strided((1, Hkv, S, D), (0, D, stride, 1))
    k.copy_(kc)
    got = K.flash_fwd(q, k, v, band=K.Band(None, 0))
    torch.cuda.synchronize()
    for hq in (0, H - 1):
        hk = hq * Hkv // H
        o, _m, _den, lse = cf.attention(*(t.double().cpu().numpy() for t in (q[0, hq], kc[0, hk], v[0, hk])),
                                        scale=D**-0.5, band=(None, 0))
        np.testing.assert_allclose(got.o[0, hq].double().cpu().numpy(), o, rtol=0, atol=1e-5)
        np.testing.assert_allclose(got.lse[0, hq].double().cpu().numpy(), lse, rtol=0, atol=1e-5)
