"""Prefill chunks of the op that are short against the cached keys: the op
splits their keys over workgroups and a second kernel merges the splits.
Against the oracle op, at the edges of that path: rows that do not fill a row
tile of 64 (query, q head) pairs, key counts on and off the 64-key tile, more
than 64 key tiles (page ids come 64 tiles at a time, and a split may start or
end inside such a block), fp16, several batch entries, not causal, NaN and
infinite inputs in the chunk's own rows, and splits whose keys are all NaN.  Tolerances as everywhere (max-abs <=
2^-7 max|ref| and rel-L2 <= 1e-2 in bf16, 2^-8 and 4e-3 in fp16)."""
import numpy as np
import pytest
import torch

from genllm_amd import paged, synth
from helpers import assert_attn_close, assert_attn_close_f16, f16 as as_f16, f32, scale_for
from test_gpu_decode import Context
from test_gpu_f16_batch import make
from test_gpu_prefill import run_prefill

pytestmark = pytest.mark.gpu


def chunk(orc, mgr, ref, Hq, Hkv, S, D, seed, f16=False, batch=1, causal=True, plant=None):
    gen = synth.normal_f16 if f16 else synth.normal_bf16
    dev = paged.to_device_f16 if f16 else paged.to_device_bf16
    q = gen(seed, (batch, Hq, S, D))
    k = gen(seed + 1, (batch, Hkv, S, D)).copy()
    v = gen(seed + 2, (batch, Hkv, S, D)).copy()
    if plant:
        plant(k, v)
    out = torch.zeros((batch, Hq, S, D), dtype=torch.float16 if f16 else torch.bfloat16, device="cuda")
    paged.paged_attention(mgr, 0, dev(q), dev(k), dev(v), out, Hq // Hkv, scale_for(D), causal)
    torch.cuda.synchronize()
    want, rc = ref.paged_attention(0, q, k, v, Hq // Hkv, scale_for(D), causal, dtype=orc.F16 if f16 else orc.BF16)
    assert rc == 0
    return paged.to_host_bits(out), want


def cached(orc, Hkv, D, N, S, seed, f16, plant=None):
    """A layer holding N - S tokens, written without attending over them."""
    mgr, ref = make(orc, Hkv, D, (N + 15) // 16 + 3, seed, orc.F16 if f16 else orc.BF16)
    gen = synth.normal_f16 if f16 else synth.normal_bf16
    dev = paged.to_device_f16 if f16 else paged.to_device_bf16
    k, v = gen(seed + 5, (Hkv, N - S, D)).copy(), gen(seed + 6, (Hkv, N - S, D))
    if plant:
        plant(k)
    mgr.append_kv_from_pos(0, dev(k), dev(v), 0)
    ref.append_kv_from_pos(0, k, v, 0)
    return mgr, ref


@pytest.mark.parametrize("Hq,Hkv,D,S,N,f16,batch,causal", [
    (2, 1, 128, 9, 640, False, 1, True),     # 18 rows: one row tile, mostly empty; 10 whole key tiles
    (4, 1, 128, 5, 1025, False, 1, True),    # 20 rows, the last key alone in its tile
    (8, 2, 256, 33, 703, False, 1, True),    # head_dim 256, 132 rows: 3 row tiles, the last of 4 rows
    (8, 2, 128, 130, 1200, False, 1, True),  # 520 rows: 9 row tiles
    (4, 2, 128, 20, 4200, False, 1, True),   # 66 key tiles: page ids of two blocks
    (2, 1, 256, 9, 4100, False, 1, False),   # not causal: every row sees all 65 tiles
    (3, 3, 128, 40, 1000, True, 1, True),    # fp16, odd head count
    (4, 2, 128, 17, 900, False, 3, True),    # three batch entries over one cache
    (16, 1, 128, 2, 2047, False, 1, True),   # 32 rows from two queries
])
def test_split_prefill_vs_oracle(orc, Hq, Hkv, D, S, N, f16, batch, causal):
    mgr, ref = cached(orc, Hkv, D, N, S, 3000 + N, f16)
    got, want = chunk(orc, mgr, ref, Hq, Hkv, S, D, 4000 + N, f16, batch, causal)
    label = f"split prefill Hq{Hq} Hkv{Hkv} D{D} S{S} N{N} f16 {f16} batch {batch} causal {causal}"
    (assert_attn_close_f16 if f16 else assert_attn_close)(got, want, label)
    mgr.close()


@pytest.mark.parametrize("D,S,N", [(128, 24, 1100), (256, 40, 1333)])
def test_split_prefill_special_values(orc, D, S, N):
    """A NaN and an infinity in V rows and a NaN in a K row of the chunk's own
    keys, seen by its later queries only: the same outputs are NaN and infinite
    as in the oracle (up to the sign of a NaN), the others stay in tolerance."""
    Hq, Hkv = 4, 2

    def plant(k, v):
        v[0, 0, S // 2, 3] = 0x7FC0
        v[0, 0, S // 3, 7] = 0x7F80
        k[0, 1, S - 4, 11] = 0xFFC0

    mgr, ref = cached(orc, Hkv, D, N, S, 5000 + N, False)
    got, want = chunk(orc, mgr, ref, Hq, Hkv, S, D, 6000 + N, plant=plant)
    nf = ~np.isfinite(f32(want))
    assert nf.any() and np.array_equal(nf, ~np.isfinite(f32(got)))
    assert np.array_equal(got[nf] & 0x7FFF, want[nf] & 0x7FFF)
    assert_attn_close(np.where(nf, 0, got).astype(np.uint16), np.where(nf, 0, want).astype(np.uint16), f"special D{D}")
    mgr.close()


@pytest.mark.parametrize("Hq,Hkv,D,S,N,f16,first,last", [
    (32, 8, 128, 8, 1089, False, 1088, 1088),   # 18 splits of a tile: the last one holds key 1088 alone
    (8, 2, 256, 8, 1089, False, 1088, 1088),
    (32, 8, 128, 8, 1089, True, 1088, 1088),
    (32, 8, 128, 8, 1089, False, 320, 383),     # every key of the split of key tile 5, seen by all queries
    (8, 2, 256, 8, 1089, True, 320, 383),
    (32, 8, 128, 64, 8256, False, 7168, 8255),  # splits of many tiles: from the last eighth's first tile on
    (32, 8, 128, 8, 1089, False, 0, 1088),      # no key with a score
])
def test_split_prefill_nan_split(orc, Hq, Hkv, D, S, N, f16, first, last):
    """NaN in the K rows first..last of one kv head, so that every key a row
    sees in one of the splits has a NaN score: no running maximum comes out of
    such a split, but its NaN reaches the output, as in the oracle (fp16 outputs
    hold an infinity for a NaN)."""
    nan, h = 0x7E00 if f16 else 0x7FC0, 1

    def old(k):
        k[h, first:last + 1, 3] = nan

    def new(k, v):
        k[0, h, max(first - (N - S), 0):max(last + 1 - (N - S), 0), 3] = nan

    mgr, ref = cached(orc, Hkv, D, N, S, 9000 + first, f16, plant=old)
    got, want = chunk(orc, mgr, ref, Hq, Hkv, S, D, 9100 + first, f16, plant=new)
    val = as_f16 if f16 else f32
    G, seen = Hq // Hkv, np.arange(N - S, N) >= first
    expect = np.zeros(want.shape, dtype=bool)
    expect[:, h * G:(h + 1) * G, seen] = True
    for x in (want, got):
        assert np.array_equal(~np.isfinite(val(x)), expect)
    assert np.array_equal(got[expect] & 0x7FFF, want[expect] & 0x7FFF)
    fin = [np.where(expect, 0, x).astype(np.uint16) for x in (got, want)]
    (assert_attn_close_f16 if f16 else assert_attn_close)(*fin, f"nan split D{D} N{N} keys {first}..{last}")
    mgr.close()


@pytest.mark.parametrize("D,tokens,most", [(128, 640, 0), (128, 1024, 9), (256, 384, 0)])
def test_split_scratch_fits_the_layer(D, tokens, most):
    """A layer whose chunks are never split reserves no scratch for it, one with
    few tokens what its largest plan needs (MB, on top of the page table and
    the decode workspace, which take less than 5 MB with their 2 MB pages)."""
    mgr = paged.PagedAttentionManager(2 * tokens * D * 2 + (1 << 20))
    mgr.init_layer(0, 1, D)
    free = torch.cuda.mem_get_info()[0]
    mgr.reserve_layer(0, tokens // 16)
    used = (free - torch.cuda.mem_get_info()[0]) / 1e6
    print(f"D{D} {tokens} tokens: {used:.1f} MB", flush=True)
    assert used <= most + 5
    mgr.close()


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [
    (3, 4, 2, 70, 128),   # the q heads of a kv head packed into row tiles
    (5, 2, 1, 1, 256),
    (2, 16, 4, 64, 128),  # a row tile for each q head, heads in multiples of 8
    (2, 6, 2, 127, 256),  # row tiles of single q heads, 6 of them
])
def test_flash_batch_in_one_launch(orc, B, Hq, Hkv, S, D):
    """Every batch entry of the non-paged op reads its own q, k and v rows."""
    q, k, v = (synth.normal_bf16(7000 + i, (B, h, S, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    out = torch.zeros((B, Hq, S, D), dtype=torch.bfloat16, device="cuda")
    paged.flash_attention(*(paged.to_device_bf16(x) for x in (q, k, v)), out, Hq // Hkv, scale_for(D))
    torch.cuda.synchronize()
    assert_attn_close(paged.to_host_bits(out), orc.flash_attention(q, k, v, Hq // Hkv, scale_for(D), True), f"flash B{B}")


@pytest.mark.parametrize("Hq,Hkv,S,D,over", [
    (4, 4, 70, 128, "q"),
    (4, 4, 70, 128, "k"),
    (4, 4, 33, 256, "v"),
    (2, 2, 300, 128, "q"),
])
def test_flash_batch_output_over_earlier_inputs(orc, Hq, Hkv, S, D, over):
    """Each entry's output over the q, k or v rows of the entry before it:
    right as long as the entries run one after another."""
    B = 4
    q, k, v = (synth.normal_bf16(7100 + i, (B, h, S, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    d = {"q": paged.to_device_bf16(q), "k": paged.to_device_bf16(k), "v": paged.to_device_bf16(v)}
    buf = torch.zeros((B + 1, Hq, S, D), dtype=torch.bfloat16, device="cuda")
    d[over] = buf[1:].copy_(d[over])
    paged.flash_attention(d["q"], d["k"], d["v"], buf[:B], Hq // Hkv, scale_for(D))
    torch.cuda.synchronize()
    want = orc.flash_attention(q, k, v, Hq // Hkv, scale_for(D), True)
    assert_attn_close(paged.to_host_bits(buf[:B]), want, f"flash out over {over}")


def test_op_batch_output_over_earlier_queries(orc):
    """The op's prefill chunk with each entry's output over the queries of the
    entry before it."""
    B, Hq, Hkv, D, S, N = 3, 4, 2, 128, 40, 200
    mgr, ref = cached(orc, Hkv, D, N, S, 7200, False)
    q, k, v = (synth.normal_bf16(7210 + i, (B, h, S, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    buf = torch.zeros((B + 1, Hq, S, D), dtype=torch.bfloat16, device="cuda")
    qd = buf[1:].copy_(paged.to_device_bf16(q))
    paged.paged_attention(mgr, 0, qd, paged.to_device_bf16(k), paged.to_device_bf16(v), buf[:B], Hq // Hkv, scale_for(D))
    torch.cuda.synchronize()
    want, rc = ref.paged_attention(0, q, k, v, Hq // Hkv, scale_for(D), True)
    assert rc == 0
    assert_attn_close(paged.to_host_bits(buf[:B]), want, "op out over q")
    mgr.close()


@pytest.mark.parametrize("Hq,Hkv,S,N,causal", [
    (4, 2, 33, 1280, True),   # 10 whole 128-key tiles
    (2, 1, 20, 1281, True),   # the last key alone in its tile
    (3, 3, 70, 1409, False),  # every key part of the last tile but one is empty
    (2, 2, 40, 8300, True),   # 65 tiles: page ids of two blocks
])
def test_wide_prefill_vs_oracle(orc, Hq, Hkv, S, N, causal):
    """The stateless entry point never splits; from 1280 keys on a launch with
    a workgroup or less for each CU runs 16 waves on 128-key tiles."""
    ctx = Context(orc, Hkv, 128, (N + 15) // 16 + 2, N, 8000 + N, nan_tail=True)
    q = synth.normal_bf16(8100 + N, (Hq, S, 128))
    assert_attn_close(run_prefill(ctx, q, causal), ctx.oracle(q, causal), f"wide Hq{Hq} Hkv{Hkv} S{S} N{N} causal {causal}")
    ctx.close()


@pytest.mark.parametrize("Hq,Hkv,D,S,N,causal", [
    (4, 4, 128, 17, 17, True),     # 17 rows: two tiles of 16, the second with one row
    (6, 2, 128, 27, 100, True),    # three q heads per kv head: 81 rows in tiles of 16
    (64, 32, 128, 80, 100, True),  # tiles of 32 rows: 16 would take more than a workgroup per CU
    (8, 2, 256, 45, 300, False),   # head_dim 256
])
def test_small_row_tiles_vs_oracle(orc, Hq, Hkv, D, S, N, causal):
    """Launches that leave CUs idle take row tiles of 16 or 32 rows."""
    ctx = Context(orc, Hkv, D, (N + 15) // 16 + 2, N, 8200 + N + S, nan_tail=True)
    q = synth.normal_bf16(8300 + N, (Hq, S, D))
    assert_attn_close(run_prefill(ctx, q, causal), ctx.oracle(q, causal), f"row tiles Hq{Hq} Hkv{Hkv} D{D} S{S} N{N}")
    ctx.close()


@pytest.mark.parametrize("Hq,Hkv,D,S,prefix,f16,over", [
    (4, 2, 128, 9, 7, False, None),      # the chunk starts and ends inside the first page
    (4, 2, 128, 33, 0, False, None),     # no earlier tokens
    (4, 1, 256, 40, 75, False, None),    # head_dim 256, starts inside a page
    (2, 2, 128, 1290, 24, False, None),  # 16-wave form, nearly every tile the chunk's own
    (2, 2, 128, 50, 1281, True, None),   # split, fp16: the last split holds the chunk
    (2, 1, 128, 16, 64, False, None),    # whole pages
    (1, 1, 128, 4120, 3, False, None),   # more pages than the launch arguments hold
    (8, 2, 256, 30, 1500, False, None),
    (2, 2, 128, 60, 100, False, "k"),    # the output over the chunk's K rows: appended before
    (2, 2, 128, 60, 100, False, "v"),
])
def test_chunk_append_and_attention(orc, Hq, Hkv, D, S, prefix, f16, over):
    """A chunk's rows reach their page slots and the table bit for bit, and the
    attention sees them, whether one launch does both or two."""
    N = prefix + S
    mgr, ref = make(orc, Hkv, D, (N + 15) // 16 + 1, 600 + N, orc.F16 if f16 else orc.BF16)
    gen = synth.normal_f16 if f16 else synth.normal_bf16
    dev = paged.to_device_f16 if f16 else paged.to_device_bf16
    if prefix:
        k, v = gen(610 + N, (Hkv, prefix, D)), gen(611 + N, (Hkv, prefix, D))
        mgr.append_kv_from_pos(0, dev(k), dev(v), 0)
        ref.append_kv_from_pos(0, k, v, 0)
    q, k, v = (gen(620 + N + i, (1, h, S, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    qd, kd, vd = dev(q), dev(k), dev(v)
    out = {None: torch.zeros_like(qd), "k": kd, "v": vd}[over]
    paged.paged_attention(mgr, 0, qd, kd, vd, out, Hq // Hkv, scale_for(D))
    torch.cuda.synchronize()
    want, rc = ref.paged_attention(0, q, k, v, Hq // Hkv, scale_for(D), True, dtype=orc.F16 if f16 else orc.BF16)
    assert rc == 0
    (assert_attn_close_f16 if f16 else assert_attn_close)(paged.to_host_bits(out), want, f"chunk S{S} prefix {prefix} D{D}")
    for which in (0, 1):
        assert np.array_equal(mgr.read_pool(0, which), ref.pool_array(0, which)), f"pool {which}"
    for got, table in zip(mgr.read_device_table(0), ref.page_table(0)):
        assert np.array_equal(got, table)
    mgr.close()
