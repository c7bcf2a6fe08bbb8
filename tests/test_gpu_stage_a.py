"""Stage (a) on the GPU -- fused q/k RMSNorm + MRoPE + f16 KV append -- is
bit-identical to the oracle (cpu_decoder.rs:274-290, 398-423): roped Q, the
K rows written to the cache and the V rows copied, for prefill segments,
decode batches (one row per slot) and chunked segments at kv_start > 0."""
from __future__ import annotations

import numpy as np
import pytest

from workloads import HD, NKVH, SEED_BASE, TOT, Layer, OracleSeq, tables

pytestmark = pytest.mark.gpu


def test_stage_a_prefill_config2_bitexact(O, gpu):
    from gpu_helpers import Gpu, say

    from oracle import Rng

    rng = Rng(SEED_BASE + 2)
    lay = Layer(rng)
    s = 420
    qkv = rng.normal_f16((s, TOT))
    say(f"stage_a prefill s={s}")
    g = Gpu(slots=1, cap=1024)
    q_gpu = g.append(0, lay, [(0, 0, s)], qkv)
    ref = OracleSeq(O, 1024, lay, tables(O))
    q_ref = ref.append(qkv, 0)
    assert np.array_equal(q_gpu, q_ref)
    k_gpu, v_gpu = g.cache(0, 0, s)
    k_ref, v_ref = ref.cache_f16()
    assert np.array_equal(k_gpu, k_ref[:, :s])
    assert np.array_equal(v_gpu, v_ref[:, :s])
    g.close()


def test_stage_a_decode_batch_and_chunks_bitexact(O, gpu):
    from gpu_helpers import Gpu, say

    from oracle import Rng

    rng = Rng(SEED_BASE + 100)
    lay = Layer(rng)
    slots, cap, layers = 5, 4352, 3
    g = Gpu(slots=slots, cap=cap, layers=layers)
    refs = [OracleSeq(O, cap, lay, tables(O)) for _ in range(slots)]
    # chunked prefill per slot at growing offsets, into layer 2
    pos = [0] * slots
    for rnd, size in enumerate((37, 1, 300, 129)):
        segs, rows = [], []
        for sl in range(slots):
            n = size + sl
            segs.append((sl, pos[sl], n))
            rows.append(rng.normal_f16((n, TOT), 0.0, 1.0 + 0.5 * sl))
        qkv = np.concatenate(rows)
        say(f"stage_a segments round {rnd} rows={qkv.shape[0]}")
        q_gpu = g.append(2, lay, segs, qkv)
        q_ref = np.concatenate([refs[sl].append(rows[sl], pos[sl]) for sl in range(slots)])
        assert np.array_equal(q_gpu, q_ref)
        for sl in range(slots):
            pos[sl] += size + sl
    # a decode batch at the end: one row per slot, slots in scrambled order
    order = [3, 0, 4, 1, 2]
    rows = rng.normal_f16((slots, TOT))
    say("stage_a decode batch")
    q_gpu = g.append(2, lay, [(sl, pos[sl], 1) for sl in order], rows)
    q_ref = np.concatenate([refs[sl].append(rows[i:i + 1], pos[sl]) for i, sl in enumerate(order)])
    assert np.array_equal(q_gpu, q_ref)
    for sl in range(slots):
        n = pos[sl] + 1
        k_gpu, v_gpu = g.cache(sl, 2, n)
        k_ref, v_ref = refs[sl].cache_f16()
        assert np.array_equal(k_gpu, k_ref[:, :n]), sl
        assert np.array_equal(v_gpu, v_ref[:, :n]), sl
        # the other layers were not touched
        k0, v0 = g.cache(sl, 0, n)
        assert not k0.any() and not v0.any()
    g.close()


def test_stage_a_extreme_inputs_bitexact(O, gpu):
    """Large, tiny and subnormal-producing rows round exactly like the oracle."""
    from gpu_helpers import Gpu, say

    from oracle import Rng

    rng = Rng(SEED_BASE + 101)
    lay = Layer(rng)
    rows = []
    for scale in (1e-4, 1e-2, 1.0, 30.0, 3000.0):
        rows.append(rng.normal_f16((4, TOT), 0.0, scale))
    z = np.zeros((1, TOT), np.uint16)  # all-zero heads: inv = 1/sqrt(eps)
    qkv = np.concatenate(rows + [z])
    n = qkv.shape[0]
    say(f"stage_a extremes rows={n}")
    g = Gpu(slots=1, cap=1024)
    q_gpu = g.append(0, lay, [(0, 5000 - 1024 * 4, n)], qkv)
    ref = OracleSeq(O, 1024, lay, tables(O))
    q_ref = ref.append(qkv, 5000 - 1024 * 4)
    assert np.array_equal(q_gpu, q_ref)
    k_gpu, _ = g.cache(0, 0, 1024)
    k_ref, _ = ref.cache_f16()
    assert np.array_equal(k_gpu, k_ref)
    g.close()


@pytest.mark.parametrize("nqh,nkvh", [(16, 8), (2, 1), (10, 5), (32, 16)])
@pytest.mark.parametrize("segments", [[(0, 0, 800)], [(1, 37, 801), (0, 5, 3)],
                                      [(i, 11 * i, 1 + 13 * i) for i in range(12)]])
def test_many_rows_equal_few_rows(gpu, nqh, nkvh, segments):
    """From 800 rows one wave does a row; below, a workgroup does.  Both round
    where the reference rounds, so one call of many rows gives, bit for bit,
    what calls of a few rows each give, subnormal, large and all-zero heads
    among them."""
    import torch

    import qasr_attn
    from gpu_helpers import say

    hd = 128
    rows = sum(n for _, _, n in segments)
    slots = max(s for s, _, _ in segments) + 1
    g = torch.Generator(device="cuda").manual_seed(81 + nqh + rows)
    qkv = torch.randn((rows, (nqh + 2 * nkvh) * hd), generator=g, device="cuda").half()
    qkv[1::7, :hd] *= 2.0 ** -20   # subnormal f16
    qkv[2::7, hd:2 * hd] *= 1000.0
    qkv[3::7, :hd] = 0
    gains = [(torch.randn(hd, generator=g, device="cuda") * 0.1 + 1).half() for _ in range(2)]
    cos, sin = qasr_attn.mrope_text_tables(2048)
    ctx = qasr_attn.Context(nqh, nkvh, hd, 1, 1e-6, 2048, 0)
    ctx.set_rope_tables(cos, sin)
    got = []
    for chunk in (10 ** 9, 150):
        kv = qasr_attn.KVPool(ctx, slots, 1024)
        kv.tensor().zero_()
        q = torch.empty((rows, nqh * hd), dtype=torch.float16, device="cuda")
        say(f"stage (a) {nqh}+{nkvh} heads, {rows} rows, {len(segments)} segments, calls of {chunk}")
        if chunk > rows:
            qasr_attn.qk_norm_rope_append(ctx, kv, 0, segments, qkv, *gains, q)
        else:
            r0 = 0
            for slot, pos, n in segments:
                for a in range(0, n, chunk):
                    m = min(chunk, n - a)
                    qasr_attn.qk_norm_rope_append(ctx, kv, 0, [(slot, pos + a, m)], qkv[r0 + a:r0 + a + m],
                                                  *gains, q[r0 + a:r0 + a + m])
                r0 += n
        torch.cuda.synchronize()
        got.append((q.view(torch.int16).cpu(), kv.tensor().clone().view(torch.int16).cpu()))
        kv.close()
    ctx.close()
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])
