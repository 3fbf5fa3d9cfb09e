"""Repeated calls through bound programs: a seat's second call takes the
program its first call made, and a launch finds its specialized kernel by a
short key; new buffers, layouts, types and neighbouring programs must each get
their own result."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _seat(subject, dtype="f32"):
    from pdum_dsl_amd.hip_tile import compile_tile_hip
    from pdum_dsl_amd.tl import fusion

    (g,) = fusion.plan_region(getattr(subject, "naive", None) or subject.region).groups
    return compile_tile_hip(g.kernel, dtype=dtype)


@pytest.mark.parametrize("name", ["stencil", "masked", "linear"])
def test_later_calls_match_the_oracle_on_other_buffers_layouts_and_types(name):
    from pdum_dsl_amd.tl import zoo

    s = {"stencil": lambda: zoo.stencil_tile(MI=33, NI=61), "masked": lambda: zoo.masked_activation(I=31, J=70),
         "linear": lambda: zoo.linear_gelu(T=37, D=70, F=45)}[name]()
    run = _seat(s)
    rng = np.random.default_rng(4)
    side = torch.cuda.Stream()
    forms = [
        lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda"),
        lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda"),  # new buffers
        lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda"),  # another type
        lambda a: torch.as_tensor(np.ascontiguousarray(a.T), dtype=torch.float32, device="cuda").t(),  # strided
        lambda a: torch.as_tensor(a, dtype=torch.float32),  # on the host
    ]
    for i, form in enumerate(forms):
        vals = [rng.standard_normal(f.arr.shape).astype(np.float32) for f in s.inputs]
        ts = [form(v) for v in vals]
        torch.cuda.synchronize()
        got = run.run_dev(ts, stream=side if i == 1 else None)
        torch.cuda.synchronize()
        want = s.oracle([v.astype(np.float64) for v in vals])
        # 1e-5 of scale: the fp32 bound of the seat's tests (sums of up to 70 products)
        np.testing.assert_allclose(got.double().cpu().numpy(), want, rtol=0, atol=1e-5 * max(1.0, np.abs(want).max()))


def test_programs_that_differ_in_one_field_keep_their_own_kernels():
    """out = x op c: the operation, the constant, the result register and a
    broadcast operand each make another kernel."""
    from pdum_dsl_amd import _lib as L
    from pdum_dsl_amd import kernels as K

    x = torch.arange(1, 65, device="cuda", dtype=torch.float32).reshape(8, 8)

    def prog(op, imm, out_reg, st):
        p = L.EwProgram()
        p.n_insns, p.n_operands, p.ndim, p.out_reg = 3, 1, 2, out_reg
        for d, (ext, o, i) in enumerate(zip((8, 8), (8, 1), st)):
            p.shape[d], p.out_stride[d], p.in_stride[0][d] = ext, o, i
        for j, (o, dst, a, b, im) in enumerate((("LOAD", 0, 0, 0, 0.0), ("CONST", 1, 0, 0, imm), (op, 2, 0, 1, 0.0))):
            p.insns[j].op, p.insns[j].dst, p.insns[j].a, p.insns[j].b, p.insns[j].imm = L.EW[o], dst, a, b, im
        return p

    col = x[:, :1].expand(8, 8)
    cases = [(("ADD", 2.0, 2, (8, 1)), x + 2), (("SUB", 2.0, 2, (8, 1)), x - 2), (("ADD", 3.0, 2, (8, 1)), x + 3),
             (("ADD", 2.0, 0, (8, 1)), x), (("ADD", 2.0, 2, (8, 0)), col + 2), (("ADD", 2.0, 2, (1, 8)), x.t() + 2)]
    for _ in range(2):
        for args, want in cases:
            out = torch.empty((8, 8), device="cuda")
            K.map_chain(prog(*args), [x], out)
            torch.cuda.synchronize()
            assert torch.equal(out, want), args
