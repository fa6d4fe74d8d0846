"""Decode over contexts of a few pages: up to kOneSplitPages pages (12 at
head_dim 128, 5 at 256) one split writes the output itself, above that the
planned splits and their merge.  Both sides of the line against the oracle,
a workspace too small for the planned splits is refused on both, and an output
over the inputs is written only after every workgroup has read them."""
import numpy as np
import pytest
import torch

from genllm_amd import paged, synth
from genllm_amd._lib import ERR_INVALID, GenllmError
from helpers import assert_attn_close, scale_for
from test_gpu_decode import Context
from test_gpu_f16_batch import check_pools, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hkv,G,D,S,N,causal", [
    (8, 4, 128, 1, 192, True),    # 12 whole pages: one split
    (8, 4, 128, 1, 193, True),    # 13 pages: several splits
    (1, 16, 128, 1, 33, True),    # 16 rows, the last page holds one key
    (2, 4, 128, 4, 177, True),    # a chunk of 4 queries across two pages
    (2, 4, 256, 1, 80, True),     # 5 whole pages at head_dim 256: one split
    (2, 4, 256, 2, 81, False),    # 6 pages: several splits
])
def test_short_decode_vs_oracle(orc, Hkv, G, D, S, N, causal):
    ctx = Context(orc, Hkv, D, (N + 15) // 16 + 2, N, 8800 + N, nan_tail=True)
    q = synth.normal_bf16(8900 + N, (Hkv * G, S, D))
    got, _ = ctx.decode(q, causal=causal)
    assert_attn_close(got, ctx.oracle(q, causal), f"short decode Hkv{Hkv} G{G} D{D} S{S} N{N}")
    ctx.close()


@pytest.mark.parametrize("merge,heads,split", [("kernel", 4, True), ("fused", 0, True), ("kernel", 1, False), ("kernel", 0, False)])
def test_short_decode_takes_forced_settings(orc, merge, heads, split):
    """A forced merge form or 4 kv heads per workgroup keep the planned splits
    of a short context (their partials are in the workspace, past its 1 KiB of
    counters); the automatic plan, and one head, leave the workspace alone."""
    N = 64
    ctx = Context(orc, 8, 128, 8, N, 8850)
    q = synth.normal_bf16(8950, (32, 1, 128))
    got, ws = ctx.decode(q, merge=merge, heads=heads)
    assert_attn_close(got, ctx.oracle(q), f"forced {merge} heads{heads}")
    assert bool(ws[1024:].any()) == split
    ctx.close()


@pytest.mark.parametrize("N", [100, 300])
def test_short_decode_keeps_its_workspace_check(N):
    q = paged.to_device_bf16(synth.normal_bf16(1, (8, 1, 128)))
    pool = paged.to_device_bf16(np.zeros((20, 16, 2, 128), dtype=np.uint16))
    ids = paged.to_device_bf16(np.zeros(40, dtype=np.uint16))  # 20 int32 zeros
    small = paged.to_device_bf16(np.zeros(8, dtype=np.uint16))
    with pytest.raises(GenllmError) as e:
        paged.paged_decode(q, q.clone(), pool, pool, ids, ids, (N + 15) // 16, N, 2, scale_for(128), small)
    assert e.value.code == ERR_INVALID and "workspace too small" in str(e.value)


@pytest.mark.parametrize("step", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,S,N,over,merge", [
    (32, 8, 128, 1, 100, "k", "kernel"),  # 7 pages: one split but for the overlap
    (32, 8, 128, 1, 100, "v", "kernel"),
    (32, 8, 128, 1, 100, "q", "kernel"),  # a head further on in the same buffer
    (32, 8, 128, 2, 20, "k", "kernel"),   # 2 pages: one split is planned
    (16, 8, 128, 1, 5, "v", "fused"),     # one page
    (32, 8, 128, 1, 300, "k", "fused"),   # several splits
    (8, 2, 256, 1, 70, "v", "kernel"),
])
def test_decode_output_over_inputs(orc, Hq, Hkv, D, S, N, over, merge, step):
    """The op and its device-position step with the new K or V rows inside the
    output buffer, and with an output that starts one head before q: outputs
    and pools as with separate buffers."""
    mgr, ref = make(orc, Hkv, D, (N + 15) // 16, 9300 + N, orc.BF16)
    k, v = (synth.normal_bf16(9310 + N + i, (Hkv, N - S, D)) for i in (0, 1))
    mgr.append_kv_from_pos(0, paged.to_device_bf16(k), paged.to_device_bf16(v), 0)
    ref.append_kv_from_pos(0, k, v, 0)
    q, k, v = (synth.normal_bf16(9320 + N + i, (1, h, S, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    want, rc = ref.paged_attention(0, q, k, v, Hq // Hkv, scale_for(D), True)
    assert rc == 0
    buf = torch.zeros((1, Hq + 1, S, D), dtype=torch.bfloat16, device="cuda")
    out, qd, kd, vd = buf[:, :Hq], paged.to_device_bf16(q), paged.to_device_bf16(k), paged.to_device_bf16(v)
    if over == "q":
        qd = buf[:, 1:].copy_(qd)
    elif over == "k":
        kd = buf[:, Hq - Hkv:Hq].copy_(kd)
    else:
        vd = buf[:, Hq - Hkv:Hq].copy_(vd)
    with paged.decode_tuned(0, merge):
        if step:
            mgr.stage_decode(0, S)
            paged.paged_attention_step(mgr, 0, qd, kd, vd, out, Hq // Hkv, scale_for(D))
            assert mgr.sync_decode(0) == N
        else:
            paged.paged_attention(mgr, 0, qd, kd, vd, out, Hq // Hkv, scale_for(D))
    torch.cuda.synchronize()
    assert_attn_close(paged.to_host_bits(out), want, f"out over {over} D{D} S{S} N{N} {merge} step {step}")
    check_pools(mgr, ref, f"out over {over}")
    mgr.close()
