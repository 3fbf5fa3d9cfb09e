"""Which map chains a nested plan merges into the contraction they read
(executor._chains_as_epilogues): a chain that one epilogue program holds is
merged, every other one stays a carve of its own and the plan builds (CPU)."""

import pytest

from pdum_dsl_amd.executor import PlanExecutor
from pdum_dsl_amd.tl.dialect import OPS
from pdum_dsl_amd.tl.ir import F64, Builder, Region, tensor_type
from pdum_dsl_amd.tl.partition import plan_model


class _B:
    """A region under construction: params and pointwise ops that broadcast."""

    def __init__(self):
        self.b, self.params = Builder(OPS), []

    def param(self, **dims):
        p = self.b.param(len(self.params), tensor_type(tuple(dims), tuple(dims.values())))
        self.params.append(p)
        return p

    def const(self, v):
        return self.b.emit("core.const", type=F64, value=float(v))

    def op(self, f, *args):
        return self.b.emit("tl.pointwise", *args, f=f)

    def over(self, x, like):
        return self.b.emit("tl.repeat_like", x, like)

    def contract(self, x, w, k):
        prod = self.op("mul", self.over(x, w), self.over(w, x))
        return self.b.emit("tl.reduce", prod, dims=k, f="sum")

    def run(self, y, n):
        return self.op("add", y, self.over(n, y))

    def executor(self, y, dtype):
        region = Region(params=tuple(self.params), body=(self.b.emit("core.yield", y),))
        return PlanExecutor(plan_model(region), region, dtype)


def _mlp(middle, dtype):
    """y[t, h] = sum_f middle(sum_d x[t, d] w1[f, d])[t, f] w2[f, h]."""
    b = _B()
    x, w1, w2 = b.param(t=512, d=16), b.param(f=512, d=16), b.param(f=512, h=16)
    return b.executor(b.contract(middle(b, b.contract(x, w1, ("d",))), w2, ("f",)), dtype)


def _kinds(ex):
    return [[st.kind for st in n.steps] for n in ex.nested]


def _gelu(b, z):
    return b.op("zoo.gelu", b.run(z, b.param(f=512)))


def _eleven_vectors(b, z):
    for _ in range(11):
        z = b.run(z, b.param(f=512))
    return z


def _two_long_runs(b, z):
    for _ in range(24):
        z = b.op("tanh", z)
    z = b.run(z, b.param(f=512))
    for _ in range(48):
        z = b.op("tanh", z)
    return z


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize(
    "middle,kinds,epilogue",
    [
        (_gelu, ["contraction-epilogue"], 16),
        # eight of the eleven chains: the operands one program reads
        (_eleven_vectors, ["contraction-epilogue"] + ["map-chain"] * 3, 17),
        # 64 instructions a program: the sum's own run stays its epilogue
        (_two_long_runs, ["contraction-epilogue", "map-chain"], 25),
    ],
)
def test_a_chain_is_merged_while_one_program_holds_it(middle, kinds, epilogue, dtype):
    ex = _mlp(middle, dtype)
    assert [[st.kind for st in n.steps] for n in ex.nested] == [kinds]
    assert f"epilogue={epilogue}" in ex.nested[0].steps[0].source


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("dims", [("f",), ("j",), ("f", "j")])
@pytest.mark.parametrize("first", ["square", "gelu"])
def test_a_chain_over_another_lattice_stays_apart(dims, first, dtype):
    """o = sum over dims of (broadcast(act(x w + b)[t, f] over j) + p[t, f, j])
    v: the wide chain is no epilogue of x w, and the activation under it, where
    it is a chain of its own, is merged all the same."""
    b = _B()
    x, w, bias = b.param(t=64, d=16), b.param(f=48, d=16), b.param(f=48)
    p = b.param(t=64, f=48, j=8)
    v = b.param(**{d: {"f": 48, "j": 8}[d] for d in dims}, h=16)
    z = b.run(b.contract(x, w, ("d",)), bias)
    act = b.op("tanh", b.op("mul", z, z)) if first == "square" else b.op("zoo.gelu", z)
    wide = b.op("add", b.over(act, p), p)
    ex = b.executor(b.contract(wide, v, dims), dtype)
    (nested,) = ex.nested
    assert [st.kind for st in nested.steps] == ["contraction-epilogue", "map-chain"]


@pytest.mark.gpu
@pytest.mark.parametrize("middle", [_gelu, _eleven_vectors, _two_long_runs])
def test_values_match_float64(middle):
    import numpy as np

    from tests.test_contraction_mapchain import _oracle

    ex = _mlp(middle, "f32")
    rng = np.random.default_rng(5)
    vals = [rng.standard_normal(p.type.shape) * 0.25 for p in ex.params]
    ex.bind(vals)
    got = ex.run().cpu().numpy().astype(np.float64)
    want = _oracle(ex.region, vals, ex.region.body[-1].args[0].type.names)
    # sums of 16 and 512 fp32 products, on six bf16 products a term
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-5 * np.abs(want).max())
