"""Slab entries of every form on an x aligned to 2 bytes only: the forms without 2-byte loads hand the call to the full
form of the same rows, so their output is that form's, bit for bit, at split 1 and with FP32 partials."""
import numpy as np
import pytest

import gie
import oracle as O
from gpu_helpers import Bundle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("rows", ["14r16", "8r16", "4r32"])
@pytest.mark.parametrize("split", [1, 2])
def test_slab_forms_on_two_byte_aligned_x(prec, rows, split):
    p = gie.Problem(2, 64, 14, 14, 40, 3, 3, 1, 1, 1, 1, precision=prec, has_bias=True, relu=True)
    b = Bundle(p, 0x51AB, O.NORMAL)
    x = gie.DeviceBuffer(b.t.dx.nbytes + 16)
    gie.check(gie.capi().gie_memcpy_d2d_async(x.addr + 2, b.t.dx.addr, b.t.dx.nbytes, None))
    gie.synchronize()
    names = [k for k in gie.registry() if k.startswith(f"slab_{prec}_3x3_32x{rows}_") and k.endswith(f"_sk{split}")]
    full = [k for k in names if not any(f in k for f in ("_l_", "_p_", "_ld_"))]
    outs = {}
    for k in names:
        plan = gie.Plan(p, k)
        ws = gie.DeviceBuffer(max(256, plan.workspace_bytes))
        b.t.poison()
        plan.execute_raw(x.addr + 2, b.t.dw.addr, b.t.bias_addr(), b.t.dy.addr, ws.addr, ws.nbytes)
        gie.synchronize()
        outs[k] = b.t.y()
        m = b.compare(outs[k])
        assert m.passed(), f"{k}: {m.summary()}"
    assert full and len(names) > len(full)
    for k in names:
        assert any(np.array_equal(outs[k], outs[f]) for f in full), k
