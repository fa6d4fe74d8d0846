"""The bias epilogue of the GEMM path at its edges: columns that do not fill a
workgroup, rows that do not fill its four-row step, widths and pointers that
take the one-element kernel.  With exact inputs (small integers, so that every
sum is exact in fp32 whatever its order) the result is one rounding of the
exact value: bit-equal to the oracle, also where the sum is NaN, infinite,
subnormal or rounds up to infinity."""
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


@pytest.mark.parametrize("offset", [0, 1])  # four columns per thread; one
def test_linear_bias_epilogue_special_values(orc, offset):
    """Rows whose GEMM results are 0, 2^119 and -2^119 (half an ulp of the
    largest bf16) and infinite, against NaN, infinite, subnormal, largest and
    ordinary biases.  A NaN's sign is left open."""
    rows, cols = 6, 516
    x = np.zeros((rows, 64), dtype=np.float32)
    x[1, 0], x[2, 0], x[3, 0] = 2.0 ** 60, -(2.0 ** 60), np.inf
    w = np.zeros((cols, 64), dtype=np.float32)
    w[:, 0] = 2.0 ** 59
    special = np.array([0x7FC0, 0xFFC1, 0x7F80, 0xFF80, 0x0001, 0x807F, 0x7F7F, 0xFF7F, 0x8000, 0x3F80, 0xC2F7], dtype=np.uint16)
    b = np.resize(special, cols)
    x, w = synth.f32_to_bf16_bits(x), synth.f32_to_bf16_bits(w)
    buf = torch.zeros(rows * cols + 8, dtype=torch.bfloat16, device="cuda")
    out = buf[offset:offset + rows * cols].view(rows, cols)
    ws = torch.empty(paged.linear_workspace_bytes(rows, 64, cols), dtype=torch.uint8, device="cuda")
    paged.linear(*(paged.to_device_bf16(t) for t in (x, w)), out, paged.to_device_bf16(b), ws)
    got, want = paged.to_host_bits(out), orc.linear(x, w, b)
    nan = (want & 0x7FFF) > 0x7F80
    assert nan.any() and (want == 0x7F80).any() and (want == 0xFF80).any()
    assert np.array_equal(got & np.where(nan, 0x7FFF, 0xFFFF), want & np.where(nan, 0x7FFF, 0xFFFF))
