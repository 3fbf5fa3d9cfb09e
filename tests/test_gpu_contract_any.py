"""The 16-bit contraction over operands stored either way round
(pdh_contract_any): every pair of layouts against float64, at tile edges, with
k slices, odd output widths and unaligned output buffers; what it leaves to the
packing path; and the LDS layout's bank property (CPU)."""

import ctypes as C

import numpy as np
import pytest

from tests.test_lds_layout import _ways

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("BM", [64, 128])
def test_transposed_reads_hit_distinct_banks(BM):
    """A rows-contiguous tile holds k row r of BM values, 16-byte slot s of it
    at s ^ swz(r): the transposing 8-byte read of 16-lane group G takes k rows
    8 (G / 2) + i4 of columns 32 t + 16 (G % 2) ..+15."""
    swz = (lambda r: 4 * (r & 3)) if BM == 128 else (lambda r: 4 * ((r >> 1) & 1))
    for q in range(2):
        for t in range(BM // 64):
            for ks in range(4):
                for hi in (0, 4):
                    offs = []
                    for l in range(64):
                        G, i4, c4 = l >> 4, (l >> 2) & 3, l & 3
                        row = 16 * ks + hi + 8 * (G >> 1) + i4
                        s = BM // 16 * q + 4 * t + 2 * (G & 1) + (c4 >> 1)
                        offs.append(row * 2 * BM + ((s ^ swz(row)) << 4) + ((c4 & 1) << 3))
                    assert _ways(offs, 8) == 1


def _program(B, M, N, bias):
    """out = acc, or out = acc + bias[n]."""
    from pdum_dsl_amd import _lib as L

    p = L.EwProgram()
    rows = [("ACC", 0, 0, 0)] + ([("LOAD", 1, 0, 0), ("ADD", 2, 0, 1)] if bias else [])
    p.n_insns, p.n_operands, p.ndim, p.out_reg = len(rows), int(bias), 3, 2 if bias else 0
    for d, (e, s) in enumerate(zip((B, M, N), (M * N, N, 1))):
        p.shape[d], p.out_stride[d] = e, s
    p.in_stride[0][2] = 1
    for j, (op, dst, a, b) in enumerate(rows):
        p.insns[j].op, p.insns[j].dst, p.insns[j].a, p.insns[j].b = L.EW[op], dst, a, b
    return p


def _case(B, M, N, Kd, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn(B, M, Kd, generator=g, device="cuda").to(dt)
    b = torch.randn(B, N, Kd, generator=g, device="cuda").to(dt)
    ad, bd = a.double().cpu().numpy(), b.double().cpu().numpy()
    return a, b, np.matmul(ad, bd.transpose(0, 2, 1)), np.matmul(np.abs(ad), np.abs(bd).transpose(0, 2, 1))


def _check(got, want, mag, Kd, dt):
    # the output's rounding (half an ulp: 8 and 11 significant bits), and a sum of Kd fp32 products in any order
    unit = 2.0**-8 if dt == torch.bfloat16 else 2.0**-11
    bound = unit * np.abs(want) * 1.01 + (Kd + 8) * 2.0**-24 * mag + 2.0**-24
    err = np.abs(got.double().cpu().numpy() - want)
    assert np.isfinite(err).all() and (err <= bound).all(), float((err / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("lay", [0, 1, 2, 3])
@pytest.mark.parametrize(
    "B,M,N,Kd",
    [
        (1, 8, 8, 8),  # the smallest
        (3, 64, 72, 56),  # one k tile, a ragged one
        (1, 65, 61, 136),  # odd rows (k-contiguous only)
        (2, 40, 136, 1032),  # k slices, the last short
        (1, 24, 48, 4096),  # the most slices
        (1, 264, 8, 2048),
        (17, 136, 520, 72),  # 128 x 128 tiles that are not: two k tiles
        (4, 1032, 1096, 200),  # 128 x 128 tiles, ragged in m, n and k
        (1, 2040, 2051, 328),  # an odd output width
    ],
)
def test_every_layout_matches_float64(B, M, N, Kd, lay, dt):
    from pdum_dsl_amd import kernels as K

    if (lay & 1 and M % 8) or (lay & 2 and N % 8):
        pytest.skip("rows-contiguous operands hold rows in whole 16-byte chunks")
    dt = getattr(torch, dt)
    a, b, want, mag = _case(B, M, N, Kd, dt, seed=M + Kd)
    sa, sb = (M * Kd, Kd, 1), (N * Kd, Kd, 1)
    if lay & 1:
        a, sa = a.transpose(1, 2).contiguous(), (M * Kd, 1, M)
    if lay & 2:
        b, sb = b.transpose(1, 2).contiguous(), (N * Kd, 1, N)
    bias = torch.randn(N, device="cuda").to(dt)
    for off, with_bias in ((0, False), (1, True)):  # the second output and bias start off 16-byte boundaries
        flat = torch.full((B * M * N + 9,), 7.0, device="cuda", dtype=dt)
        out = flat[off:off + B * M * N].view(B, M, N)
        bs = torch.cat([bias[:1], bias])[off:off + N]
        assert K.contract_any(a, sa, b, sb, (B, M, N, Kd), _program(B, M, N, with_bias), [bs] if with_bias else [], out)
        torch.cuda.synchronize()
        add = bs.double().cpu().numpy() if with_bias else 0.0
        _check(out, want + add, mag + np.abs(add), Kd + 1, dt)
        assert bool((flat[:off] == 7).all()) and bool((flat[off + B * M * N:] == 7).all())  # nothing past the ends


@pytest.mark.gpu
def test_a_wide_row_pitch_a_zero_batch_stride_and_refusals():
    from pdum_dsl_amd import _lib as L
    from pdum_dsl_amd import kernels as K

    dt, (B, M, N, Kd) = torch.bfloat16, (3, 72, 80, 264)
    a, b, want, mag = _case(B, M, N, Kd, dt, seed=1)
    wide = torch.full((B, M, Kd + 24), float("nan"), device="cuda", dtype=dt)
    wide[..., :Kd] = a
    shared = b[:1].clone()
    want = np.matmul(a.double().cpu().numpy(), shared.double().cpu().numpy().transpose(0, 2, 1))
    mag = np.matmul(np.abs(a.double().cpu().numpy()), np.abs(shared.double().cpu().numpy()).transpose(0, 2, 1))
    out = torch.empty(B, M, N, device="cuda", dtype=dt)
    p, sw, sb = _program(B, M, N, False), (M * (Kd + 24), Kd + 24, 1), (0, Kd, 1)
    assert K.contract_any(wide, sw, shared, sb, (B, M, N, Kd), p, [], out)
    torch.cuda.synchronize()
    _check(out, want, mag, Kd, dt)
    # left to the packing path: a k that is not whole chunks, a row off 16 bytes, a base off 16 bytes, both strided
    assert not K.contract_any(wide, sw, shared, sb, (B, M, N, Kd - 4), p, [], out)
    assert not K.contract_any(wide, (M * (Kd + 24), Kd + 20, 1), shared, sb, (B, M, N, Kd), p, [], out)
    assert not K.contract_any(wide.view(-1)[1:], sw, shared, sb, (B, M, N, 8), p, [], out)
    assert not K.contract_any(wide, (0, 2, 288), shared, sb, (B, M, N, 8), p, [], out)
    with pytest.raises(ValueError, match="reaches past"):
        K.contract_any(wide, sw, shared, (0, Kd + 8, 1), (B, M, N, Kd), p, [], out)
    # a slice's partial sums need their workspace
    code = L.lib().pdh_contract_any(wide.data_ptr(), 0, 4096, 1, shared.data_ptr(), 0, 4096, 1, 1, 8, 8, 4096,
                                    C.byref(_program(1, 8, 8, False)), None, out.data_ptr(), L.PDH_BF16, None, 0, None)
    assert code == L.PDH_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("T,D,F", [(1, 8, 8), (37, 70, 45), (72, 264, 40), (65, 2048, 72), (300, 1024, 1032)])
def test_the_linear_seat_reads_its_weight_in_place_or_packs_it(T, D, F, dtype):
    from pdum_dsl_amd.hip_tile import compile_tile_hip
    from pdum_dsl_amd.tl import fusion, zoo

    s = zoo.linear_gelu(T=T, D=D, F=F, seed=T + D)
    (g,) = fusion.plan_region(s.region).groups
    run = compile_tile_hip(g.kernel, dtype=dtype)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    ts = [torch.as_tensor(f.arr, dtype=torch.float32, device="cuda").to(dt) for f in s.inputs]
    want = s.oracle([t.double().cpu().numpy() for t in ts])
    # fp32: the seat tests' 1e-5 of scale (six bf16 products: under 2^-23 a term); 16-bit: the output's
    # rounding of gelu's result, and its input's sum in fp32
    tol = {"f32": 1e-5, "bf16": 2.0**-8, "f16": 2.0**-10}[dtype] * max(1.0, float(np.abs(want).max()))
    # the weight and the bias 2 (4) bytes off a 16-byte boundary, as is x where it is packed
    flats = [t if i == 0 and D % 64 == 0 else torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
             for i, t in enumerate(ts)]
    for vals in (ts, flats, ts):
        got = run.run_dev(vals)
        torch.cuda.synchronize()
        np.testing.assert_allclose(got.double().cpu().numpy(), want, rtol=0, atol=tol)


@pytest.mark.gpu
def test_replays_of_a_captured_split_match_the_eager_result():
    from pdum_dsl_amd import kernels as K

    B, M, N, Kd = 1, 40, 136, 4096
    a, b, want, mag = _case(B, M, N, Kd, torch.bfloat16, seed=9)
    out = torch.empty(B, M, N, device="cuda", dtype=torch.bfloat16)
    call = lambda: K.contract_any(a, (0, Kd, 1), b, (0, Kd, 1), (B, M, N, Kd), _program(B, M, N, False), [], out)  # noqa: E731
    assert call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    for _ in range(3):
        a.neg_()
        want = -want
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check(out, want, mag, Kd, torch.bfloat16)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_the_mlp_activation_is_the_up_projections_epilogue(dtype):
    """gpt2's nested MLP plan: a layernorm and one contraction whose epilogue
    holds the bias and the gelu, with the toy model's values unchanged by the
    merge (the GPU's sized-model tests)."""
    from pdum_dsl_amd.executor import PlanExecutor
    from pdum_dsl_amd.tl import zoo
    from pdum_dsl_amd.tl.partition import plan_model

    m = zoo.gpt2(zoo.GPT2Config(t=64, d=64, nh=2, hk=32, m=256, layers=2, v=128), seed=3)
    ex = PlanExecutor(plan_model(m.region), m.region, dtype)
    assert [[st.kind for st in n.steps] for n in ex.nested] == [["row-statistics", "contraction-epilogue"]] * 2
    assert all("epilogue=16" in n.steps[1].source for n in ex.nested)


@pytest.mark.parametrize("row_major", [False, True])
def test_an_operand_past_two_gib_is_left_to_the_packing_path(row_major):
    """any_layout says no exactly where pdh_contract_any refuses the span (its
    checks come before any launch: nothing runs here)."""
    from pdum_dsl_amd import _lib as L
    from pdum_dsl_amd import kernels as K

    def strides(n):  # a weight stored [k][n], or [n][k] with rows padded to 2^20 elements
        return (0, 1, n) if not row_major else (0, 1 << 20, 1)

    k, lo, hi = 64, 8, 1 << 25
    while hi - lo > 8:  # the largest n that is read in place
        mid = (lo + hi) // 16 * 8
        lo, hi = (mid, hi) if K.any_layout(k, mid, *strides(mid)) else (lo, mid)
    assert hi == lo + 8 and hi < 10_000_000
    p = _program(1, 100, hi, False)
    code = L.lib().pdh_contract_any(4096, 0, 64, 1, 4096, *strides(hi), 1, 100, hi, k, C.byref(p), None, 4096,
                                    L.PDH_BF16, None, 0, None)
    assert code == L.PDH_EINVAL and "2 GiB" in L.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,N", [("bf16", 10_000_000), ("f32", 8_300_000)])
def test_the_seat_packs_a_weight_past_two_gib_in_place(dtype, N):
    """A weight [k][n] whose in-place span is over 2 GiB while its packed rows
    (k columns each) are under: the packed product."""
    from pdum_dsl_amd.hip_tile import compile_tile_hip
    from pdum_dsl_amd.tl import fusion
    from pdum_dsl_amd.tl.dialect import OPS
    from pdum_dsl_amd.tl.ir import Builder, Region, tensor_type

    M, Kd = 8, 64
    bld = Builder(OPS)
    x, w = bld.param(0, tensor_type(("m", "k"), (M, Kd))), bld.param(1, tensor_type(("k", "n"), (Kd, N)))
    prod = bld.emit("tl.pointwise", bld.emit("tl.repeat_like", x, w), bld.emit("tl.repeat_like", w, x), f="mul")
    y = bld.emit("tl.reduce", prod, dims=("k",), f="sum")
    (grp,) = fusion.plan_region(Region(params=(x, w), body=(bld.emit("core.yield", y),))).groups
    run = compile_tile_hip(grp.kernel, dtype=dtype)
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}[dtype]
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(M, Kd, generator=g, device="cuda").to(dt)
    b = torch.randn(Kd, N, generator=g, device="cuda", dtype=dt)
    got = run.run_dev([a, b])
    torch.cuda.synchronize()
    cols = torch.tensor([0, 1, N // 2 + 1, N - 65, N - 1], device="cuda")
    ad, bd = a.double().cpu().numpy(), b[:, cols].double().cpu().numpy()
    want, mag = ad @ bd, np.abs(ad) @ np.abs(bd)
    # the output's rounding and 64 fp32 products (fp32: six bf16 products a term, under 2^-23 of it)
    bound = (2.0**-8 * np.abs(want) if dtype == "bf16" else 0) + 80 * 2.0**-23 * mag
    assert (np.abs(got[:, cols].double().cpu().numpy() - want) <= bound).all()
