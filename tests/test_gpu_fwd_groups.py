"""The 16-bit forward whose waves share a block's keys and merge their states
through LDS: every workgroup shape the launcher picks, at ragged rows and
keys, bands and grouped heads, against float64; pruned and unpruned sweeps bit
for bit; and which shapes still split their keys over workgroups (CPU)."""

import pytest

torch = pytest.importorskip("torch")


def test_key_splits_only_for_few_blocks_with_long_rows():
    from pdum_dsl_amd.kernels import Band, _fwd_splits, pick_fwd_splits

    causal, window = Band(None, 0), Band(-255, 0)
    for (n, t, s, d, band), want in {
        (12, 1024, 1024, 64, causal): 1,
        (64, 500, 3001, 128, None): 1,
        (38, 1024, 1024, 128, causal): 1,
        (12, 1024, 8192, 64, window): 1,  # under 384 live keys a row
    }.items():
        assert _fwd_splits(n, t, s, d, band, cus=256) == want
    for n, t, s, d, band in ((12, 1024, 8192, 64, None), (1, 4096, 4096, 128, causal), (38, 1024, 4096, 128, None),
                             (4, 255, 255, 64, None), (1, 1, 1, 64, None)):
        assert _fwd_splits(n, t, s, d, band, cus=256) == pick_fwd_splits(n, t, s, cus=256)


# (heads, t, keys, d, band): us of one launch and of the split, bf16, where they differ by a tenth
MEASURED = {
    (1, 1024, 1024, 64, None): (11.6, 16.4),
    (1, 512, 3000, 64, None): (23.2, 16.9),
    (1, 3000, 3000, 64, (None, 0)): (22.8, 20.5),
    (1, 1024, 6000, 64, (None, 4976)): (39.2, 25.6),
    (4, 256, 4096, 64, None): (28.0, 19.7),
    (4, 1024, 6000, 64, (None, 4976)): (39.5, 34.3),
    (8, 512, 6000, 64, None): (38.9, 33.4),
    (8, 1024, 3000, 64, None): (23.3, 26.4),
    (6, 3000, 3000, 64, None): (34.7, 30.7),
    (12, 2048, 6000, 64, (None, 3952)): (63.0, 53.3),
    (24, 1024, 6000, 64, None): (63.4, 54.2),
    (12, 1024, 1024, 64, (None, 0)): (12.4, 19.7),
    (8, 4096, 4096, 64, (None, 0)): (40.5, 45.4),
    (1, 1500, 1500, 128, (None, 0)): (23.7, 18.6),
    (1, 256, 2048, 128, None): (29.3, 17.5),
    (2, 3000, 3000, 128, (None, 0)): (41.5, 29.9),
    (4, 1024, 3000, 128, None): (42.0, 29.8),
    (4, 512, 512, 128, (None, 0)): (12.5, 16.5),
    (8, 2048, 6000, 128, None): (79.4, 65.7),
    (12, 1024, 4096, 128, (None, 3072)): (55.0, 47.2),
    (8, 2048, 2048, 128, None): (30.6, 39.5),
    (12, 2048, 6000, 128, (None, 3952)): (98.3, 86.0),
    (16, 2048, 2048, 128, None): (40.0, 54.7),
    (24, 2048, 2048, 128, (None, 0)): (46.4, 60.8),
    (24, 2048, 6000, 128, (None, 3952)): (161.0, 138.6),
    (4, 1024, 6000, 128, (3953, 4976)): (22.3, 40.4),
    (1, 4096, 4096, 128, (-1023, 0)): (20.6, 33.6),
    (2, 512, 6000, 64, (4465, 5488)): (14.9, 27.7),
    (4, 4177, 4177, 64, (None, 0)): (39.9, 34.6),
}


def test_the_faster_of_one_launch_and_a_split_is_taken():
    from pdum_dsl_amd.kernels import Band, _fwd_splits

    for (n, t, s, d, band), (one, split) in MEASURED.items():
        got = _fwd_splits(n, t, s, d, None if band is None else Band(*band), cus=256)
        assert (got == 1) == (one < split), (n, t, s, d, band, got)


def _exact(q, k, v, band, fill, scale):
    """(o, sum p |v|, largest sum |q| |k|, lse) in float64."""
    q, k, v = (x.double().cpu() for x in (q, k, v))
    r = q.shape[1] // k.shape[1]
    k, v = (x.repeat_interleave(r, 1) for x in (k, v))
    s = torch.matmul(q, k.transpose(2, 3)) * scale
    size = float((torch.matmul(q.abs(), k.abs().transpose(2, 3)) * scale).max())
    if band is not None:
        d = torch.arange(s.shape[3])[None] - torch.arange(s.shape[2])[:, None]
        dead = torch.zeros_like(d, dtype=torch.bool)
        if band.lo is not None:
            dead |= d < band.lo
        if band.hi is not None:
            dead |= d > band.hi
        s = s.masked_fill(dead, fill)
    p = torch.softmax(s, -1)
    return torch.matmul(p, v), torch.matmul(p, v.abs()), size, torch.logsumexp(s, -1)


# (B, H, Hkv, T, S, D, band): the (row, key) wave groups of the workgroup the launcher picks
CASES = {
    (1, 1, 1, 1, 1024, 64, None): (2, 4),
    (1, 2, 1, 65, 1055, 64, (None, 990)): (2, 4),
    (1, 3, 3, 1030, 1024, 64, (None, 0)): (2, 4),
    (1, 2, 2, 63, 256, 64, None): (2, 2),
    (1, 4, 1, 130, 321, 64, (None, 2)): (2, 2),
    (2, 2, 1, 200, 1500, 64, (-300, 5)): (2, 2),  # a window: fewer live keys than stored
    (1, 1, 1, 33, 257, 128, (None, -1)): (2, 2),  # a fully masked row: no prune
    (1, 8, 2, 300, 417, 128, (None, 0)): (2, 2),
    (1, 6, 6, 129, 300, 128, (120, None)): (2, 2),
    (3, 24, 12, 190, 287, 128, None): (4, 2),
    # uneven sweeps over more blocks than compute units: up to 1.5 a unit at 512 keys ...
    (1, 100, 100, 257, 515, 64, (None, 100)): (2, 2),
    (1, 100, 50, 257, 515, 128, (None, 100)): (2, 2),
    # ... and up to 4 (D = 64) or 2 (128) at 2048 keys
    (1, 36, 36, 2048, 2048, 64, (None, 0)): (2, 2),
    (1, 200, 100, 129, 2050, 128, (None, 1900)): (2, 2),
    # past those lines: one key group
    (2, 70, 70, 257, 515, 64, (None, 100)): (4, 1),
    (1, 100, 50, 400, 513, 128, (None, 0)): (4, 1),
}


def _workgroup(B, H, Hkv, T, S, D, band, cus=256):
    """launch_mfma's choice (flash_fwd.hip)."""
    blocks, (lo, hi) = B * H * -(-T // 128), band or (None, None)
    keys = S if lo is None or hi is None else min(S, hi - lo + 128)
    uneven = (lo is None) != (hi is None)
    if blocks <= cus and keys >= 256:
        if D == 64 and 2 * blocks <= cus and keys >= 1024:
            return 2, 4
        return (4, 2) if D == 128 and 2 * blocks > cus and not uneven else (2, 2)
    wide = (2 * blocks <= 3 * cus and keys >= 512) or (blocks <= (4 if D == 64 else 2) * cus and keys >= 2048)
    return (2, 2) if uneven and wide else (4, 1)


def test_the_cases_reach_every_workgroup_shape():
    for case, want in CASES.items():
        assert _workgroup(*case) == want, case
    assert {(c[5], w) for c, w in CASES.items()} == {(64, (2, 4)), (64, (2, 2)), (64, (4, 1)), (128, (2, 2)), (128, (4, 2)),
                                                     (128, (4, 1))}


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("B,H,Hkv,T,S,D,band", CASES)
def test_grouped_keys_match_float64(B, H, Hkv, T, S, D, band, dt):
    from pdum_dsl_amd import kernels as K

    dt = getattr(torch, dt)
    g = torch.Generator(device="cuda").manual_seed(T + S + D)
    q, k, v = (torch.randn(B, h, n, D, generator=g, device="cuda").to(dt) for h, n in ((H, T), (Hkv, S), (Hkv, S)))
    bnd, scale = (None if band is None else K.Band(*band)), D**-0.5
    got = K.flash_fwd(q, k, v, band=bnd, nsplit=1)
    full = K.flash_fwd(q, k, v, band=bnd, nsplit=1, prune=False)
    arts = K.flash_fwd(q, k, v, band=bnd, nsplit=1, want_artifacts=True)
    torch.cuda.synchronize()
    assert torch.equal(got.o, full.o) and torch.equal(got.lse, full.lse)
    want, mag, size, lse = _exact(q, k, v, bnd, -1e9, scale)
    # p and o round to 16 bits (half an ulp each); a score is a sum of D fp32 products, and its error
    # moves every p of the row (and the sum under it) by as much
    unit = 2.0**-8 if dt == torch.bfloat16 else 2.0**-11
    ds = (D + 16) * 2.0**-24 * size + 2.0**-20
    bound = 1.01 * unit * (mag + want.abs()) + 3 * ds * mag + 2.0**-24
    for out in (got, arts):
        err = (out.o.double().cpu() - want).abs()
        assert bool((err <= bound).all()), float((err / bound).max())
        # lse of a fully masked row is the fill's own: compare relative to its size
        assert bool(((out.lse.double().cpu() - lse).abs() <= 2 * ds + 2.0**-22 * lse.abs()).all())
    assert bool(((arts.m + torch.log(arts.den) - arts.lse).abs() <= 1e-5 + 2.0**-21 * arts.lse.abs()).all())


@pytest.mark.gpu
@pytest.mark.parametrize("fill", [float("-inf"), torch.finfo(torch.float32).min], ids=["-inf", "lowest"])
@pytest.mark.parametrize(
    "B,H,Hkv,T,S,D,band",
    [
        (1, 2, 1, 65, 1055, 64, (None, 990)),  # four key groups
        (1, 4, 1, 130, 321, 64, (None, 2)),  # two: a group's first tile is dead for some of a wave's rows
        (2, 2, 1, 200, 1500, 64, (-300, 5)),
        (1, 1, 1, 33, 257, 128, (None, -1)),  # a fully masked row
        (1, 6, 6, 129, 300, 128, (120, None)),
        (3, 24, 12, 190, 287, 128, (None, 97)),
        (2, 70, 70, 257, 230, 64, (-100, 2)),  # one key group
        (2, 2, 1, 200, 90, 128, (-70, 3)),
    ],
)
def test_the_lowest_fills_leave_live_rows_finite(B, H, Hkv, T, S, D, band, fill):
    """A masked score of -inf, or of a finite fill that overflows over the
    scale: a tile (or group, or split) in which a row sees nothing else adds
    nothing to it. A row with no live key is NaN for -inf, the mean of V else."""
    from pdum_dsl_amd import kernels as K

    g = torch.Generator(device="cuda").manual_seed(T + S + D)
    q, k, v = (torch.randn(B, h, n, D, generator=g, device="cuda").bfloat16() for h, n in ((H, T), (Hkv, S), (Hkv, S)))
    bnd, scale = K.Band(*band), D**-0.5
    kw = dict(band=bnd, fill=fill)
    outs = [K.flash_fwd(q, k, v, nsplit=1, **kw), K.flash_fwd(q, k, v, nsplit=1, prune=False, **kw),
            K.flash_fwd(q, k, v, nsplit=1, want_artifacts=True, **kw), K.flash_fwd(q, k, v, nsplit=3, **kw),
            K.flash_fwd(q, k, v, nsplit=3, prune=False, want_artifacts=True, **kw)]
    torch.cuda.synchronize()
    want, mag, size, lse = _exact(q, k, v, bnd, fill, scale)
    d = torch.arange(S)[None] - torch.arange(T)[:, None]
    live = torch.ones_like(d, dtype=torch.bool)
    if band[0] is not None:
        live &= d >= band[0]
    if band[1] is not None:
        live &= d <= band[1]
    live = live.any(1)  # rows with a live key
    unit, ds = 2.0**-8, (D + 16) * 2.0**-24 * size + 2.0**-20  # as in test_grouped_keys_match_float64
    bound = 1.01 * unit * (mag + want.abs()) + 3 * ds * mag + 2.0**-24
    for out in outs:
        o = out.o.double().cpu()
        assert bool(((o - want).abs() <= bound)[:, :, live].all())
        assert bool(((out.lse.double().cpu() - lse).abs() <= 2 * ds + 2.0**-22 * lse.abs())[:, :, live].all())
        if fill == float("-inf"):
            assert bool(torch.isnan(o[:, :, ~live]).all())
        else:
            assert bool(((o - want).abs() <= bound)[:, :, ~live].all())
    assert torch.equal(outs[0].o[:, :, live.cuda()], outs[1].o[:, :, live.cuda()])
    for art in (outs[2], outs[4]):
        assert bool(((art.m + torch.log(art.den) - art.lse).abs() <= 1e-5 + 2.0**-21 * art.lse.abs())[:, :, live.cuda()].all())
