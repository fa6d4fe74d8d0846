"""The bias epilogue of the GEMM path at its edges: columns that do not fill a
workgroup, rows that do not fill its four-row step, widths and pointers that
take the one-element kernel.  With exact inputs (small integers, so that every
sum is exact in fp32 whatever its order) the result is one rounding of the
exact value: bit-equal to the oracle."""
import numpy as np
import pytest
import torch

from genllm_amd import paged, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,offset", [(5, 1028, 0), (6, 516, 0), (9, 4, 0), (70, 2048, 0), (7, 30, 0), (6, 516, 1)])
def test_linear_bias_epilogue(orc, rows, cols, offset):
    rng = np.random.default_rng(rows * cols)
    x, w, b = (synth.f32_to_bf16_bits(rng.integers(-4, 5, s).astype(np.float32)) for s in ((rows, 64), (cols, 64), (cols,)))
    buf = torch.zeros(rows * cols + 8, dtype=torch.bfloat16, device="cuda")
    out = buf[offset:offset + rows * cols].view(rows, cols)
    ws = torch.empty(paged.linear_workspace_bytes(rows, 64, cols), dtype=torch.uint8, device="cuda")
    paged.linear(*(paged.to_device_bf16(t) for t in (x, w)), out, paged.to_device_bf16(b), ws)
    assert np.array_equal(paged.to_host_bits(out), orc.linear(x, w, b))
    assert not buf[offset + rows * cols:].any() and not buf[:offset].any()
