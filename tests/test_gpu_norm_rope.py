"""The stand-alone RMSNorm and RoPE ops at the edges of their kernels, bit for
bit against the oracle: row widths on both sides of each workgroup size (a
partial 32-block, an 8-block tail, a scalar tail), row counts that leave lane
groups empty, pointers that do not allow 16-byte accesses, in place, head
counts that do not divide into pairs, and partial rotations."""
import numpy as np
import pytest
import torch

from genllm_amd import paged, synth

pytestmark = pytest.mark.gpu


def at_offset(bits, elems):
    """The values on the GPU, `elems` elements past a 16-byte boundary."""
    buf = torch.zeros(bits.size + 16, dtype=torch.bfloat16, device="cuda")
    view = buf[elems:elems + bits.size]
    view.copy_(paged.to_device_bf16(bits).reshape(-1))
    return view


@pytest.mark.parametrize("hidden", [64, 128, 256, 8, 40, 512, 520, 1024, 1032, 2048, 2560, 4104, 8200, 32768, 36, 3])
@pytest.mark.parametrize("rows", [1, 33])
@pytest.mark.parametrize("offset", [0, 1])
def test_rms_norm_widths(orc, hidden, rows, offset):
    x = synth.normal_bf16(hidden + rows, (rows, hidden))
    w = synth.uniform_f32(hidden + 1, (hidden,), 0.5, 1.5)
    xd = at_offset(x, offset)
    out = at_offset(np.zeros_like(x), offset)
    paged.rms_norm(out, xd, torch.from_numpy(w).cuda(), 1e-6)
    paged.rms_norm(xd, xd, torch.from_numpy(w).cuda(), 1e-6)  # in place
    want = orc.rms_norm(x, w, 1e-6).reshape(-1)
    assert np.array_equal(paged.to_host_bits(out), want)
    assert np.array_equal(paged.to_host_bits(xd), want)


@pytest.mark.parametrize("H,S,D,rope_dim,offset", [
    (5, 13200, 128, 128, 0),  # two heads per thread, the last group of one
    (7, 700, 128, 128, 0),    # one head per thread, the last workgroup partly empty
    (3, 900, 256, 64, 0),     # 192 copied dims
    (2, 2100, 128, 48, 0),
    (7, 1, 128, 128, 0),      # a small call: one pair per thread
    (2, 2100, 128, 24, 0),    # rope_dim not a multiple of 16: one pair per thread
    (2, 2100, 128, 128, 1),   # pointers 2 bytes past a 16-byte boundary: likewise
    (4, 4000, 36, 36, 0),     # head_dim not a multiple of 8: likewise
])
def test_apply_rope_widths(orc, H, S, D, rope_dim, offset):
    x = synth.normal_bf16(H * S + D, (H, S, D))
    cos, sin = paged.rope_cache(1e6, rope_dim, S + 3)
    cd, sd = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    xd = at_offset(x, offset).view(H, S, D)
    out = at_offset(np.zeros_like(x), offset).view(H, S, D)
    paged.apply_rope(out, xd, cd, sd, 3)
    paged.apply_rope(xd, xd, cd, sd, 3)  # in place
    want = orc.apply_rope_partial(x, cos, sin, 3)
    assert np.array_equal(paged.to_host_bits(out), want)
    assert np.array_equal(paged.to_host_bits(xd), want)


def same_but_nan(got, want):
    """Bit-equal, NaNs in the same places (their sign and payload are not fixed)."""
    g, w = synth.bf16_bits_to_f32(got), synth.bf16_bits_to_f32(want)
    return np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(got[~np.isnan(w)], want[~np.isnan(w)])


SPECIALS = np.array([0x7FC0, 0xFF81, 0x7F80, 0xFF80, 0x0001, 0x8001, 0x007F, 0x0080, 0x7F7F, 0xFF7F, 0x8000], dtype=np.uint16)


def with_specials(seed, shape):
    x = synth.normal_bf16(seed, shape).reshape(-1)
    r = np.random.default_rng(seed)
    at = r.choice(x.size, 200, replace=False)
    x[at] = r.choice(SPECIALS, 200)
    return x.reshape(shape)


@pytest.mark.parametrize("hidden,rows", [(128, 500), (2560, 300), (520, 300)])
def test_rms_norm_special_values(orc, hidden, rows):
    x = with_specials(hidden, (rows, hidden))
    w = synth.uniform_f32(hidden + 1, (hidden,), 0.5, 1.5)
    out = torch.empty((rows, hidden), dtype=torch.bfloat16, device="cuda")
    paged.rms_norm(out, paged.to_device_bf16(x), torch.from_numpy(w).cuda(), 1e-6)
    assert same_but_nan(paged.to_host_bits(out), orc.rms_norm(x, w, 1e-6))


@pytest.mark.parametrize("H,S,D,rope_dim", [(5, 900, 128, 128), (3, 900, 256, 64)])
def test_apply_rope_special_values(orc, H, S, D, rope_dim):
    x = with_specials(H * S, (H, S, D))
    cos, sin = paged.rope_cache(1e6, rope_dim, S)
    out = torch.empty((H, S, D), dtype=torch.bfloat16, device="cuda")
    paged.apply_rope(out, paged.to_device_bf16(x), torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda(), 0)
    assert same_but_nan(paged.to_host_bits(out), orc.apply_rope_partial(x, cos, sin, 0))
