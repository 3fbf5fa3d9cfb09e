"""The process-wide fp32 contraction mode under threads: what one request
generates belongs to one mode, whatever another thread sets meanwhile."""

import ctypes as C
import threading

import pytest

from pdum_dsl_amd import _lib as L
from tests.test_gpu_contract_any import _program


def test_a_source_belongs_to_one_mode():
    """A request reads the mode once (CPU; the sources of modes 0 and 6 share
    no kernel text)."""
    lib = L.lib()
    p = _program(1, 64, 64, False)

    def source():
        buf = C.create_string_buffer(1 << 14)
        lib.pdh_ew_jit_source(C.byref(p), 1, L.PDH_F32, buf, len(buf))
        return buf.value

    prev = lib.pdh_contract_set_f32_mode(0)
    stop = threading.Event()
    try:
        want = {source()}
        lib.pdh_contract_set_f32_mode(6)
        want.add(source())
        assert len(want) == 2

        def flip():
            while not stop.is_set():
                lib.pdh_contract_set_f32_mode(0)
                lib.pdh_contract_set_f32_mode(6)

        threads = [threading.Thread(target=flip) for _ in range(2)]
        for t in threads:
            t.start()
        try:
            for _ in range(40000):
                assert source() in want
        finally:
            stop.set()
            for t in threads:
                t.join()
    finally:
        lib.pdh_contract_set_f32_mode(prev)


@pytest.mark.gpu
def test_threads_in_different_modes_get_their_kernels():
    """Launches of both modes from two threads, then each mode alone: every
    product is right to fp32 (which mode a concurrent launch runs in is open,
    that its kernel and grid belong together is not)."""
    torch = pytest.importorskip("torch")
    from pdum_dsl_amd import kernels as K

    B, M, N, Kd = 1, 96, 72, 256
    g = torch.Generator(device="cuda").manual_seed(2)
    a, b = (torch.randn(B, r, Kd, generator=g, device="cuda") for r in (M, N))
    want = (a.double() @ b.double().transpose(1, 2).contiguous()).cpu()
    mag = (a.double().abs() @ b.double().abs().transpose(1, 2).contiguous()).cpu()

    def call(mode):
        out = torch.empty(B, M, N, device="cuda")
        K.contract_views(a, (M * Kd, Kd, 1), b, (N * Kd, Kd, 1), (B, M, N, Kd), _program(B, M, N, False), [], out,
                         f32_mode=mode)
        torch.cuda.synchronize()
        return out

    outs, prev = [], K.set_f32_contract("bf16x6")
    try:
        ts = [threading.Thread(target=lambda m=m: outs.extend(call(m) for _ in range(200))) for m in ("fma", "bf16x6")]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert len(outs) == 400
        outs += [call("fma"), call("bf16x6")]
    finally:
        K.set_f32_contract(prev)
    bound = (Kd + 80) * 2.0**-23 * mag  # 256 fp32 products in any order, or six bf16 products a term
    for o in outs:
        assert bool(((o.double().cpu() - want).abs() <= bound).all())
