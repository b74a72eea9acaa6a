"""GPU parity of the fused stage-1 + max-pool entry point (fused in the
LDS-resident kernel for rows of at most 512 keys, in the decode kernel or the
K-streaming kernels for longer rows).

The pooled scores must equal, bit for bit, the max-pool the oracle computes
from the scores the same kernel wrote (``return_scores``), and the scores must
match the stage-1 oracle at atol 1e-3 / rtol 1e-2; without ``return_scores``
the pooled output must be the same bits.
"""

import numpy as np
import pytest
import torch

from oracle.maxpool import max_pooling_1d_varlen as oracle_pool
from oracle.stage1 import infllmv2_attn_stage1 as oracle_stage1, visible_counts
import workloads
from unum_ops_amd import _lib
from unum_ops_amd.infllm_v2 import (infllmv2_attn_stage1, infllmv2_attn_stage1_maxpool,
                                    max_pooling_1d_varlen)
from unum_ops_amd.pipeline import topk_blocks

pytestmark = pytest.mark.gpu


def _check(d, dev, max_context_len, local_blocks=1, init_blocks=1, causal=True):
    args = (d["q"].to(dev), d["k"].to(dev), d["cu_seqlens_q"].to(dev), d["cu_seqlens_k"].to(dev),
            max_context_len)
    kw = dict(max_seqlen_k=d["max_seqlen_k"], causal=causal, local_blocks=local_blocks,
              init_blocks=init_blocks)
    pooled, scores = infllmv2_attn_stage1_maxpool(*args, return_scores=True, **kw)
    pooled_only = infllmv2_attn_stage1_maxpool(*args, **kw)
    torch.cuda.synchronize()
    exp_s = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                          max_seqlen_k=d["max_seqlen_k"], causal=causal)
    torch.testing.assert_close(scores.cpu(), exp_s, atol=1e-3, rtol=1e-2)
    B = d["cu_seqlens_q"].numel() - 1
    exp_p = oracle_pool(scores.cpu(), d["cu_seqlens_q"], d["cu_seqlens_k"],
                        torch.zeros(B, dtype=torch.int32), 16 * scores.shape[-1],
                        max_context_len, local_blocks, init_blocks)
    np.testing.assert_array_equal(pooled.cpu().numpy(), exp_p)
    assert torch.equal(pooled_only, pooled)


@pytest.mark.parametrize("local_blocks,init_blocks", [(1, 1), (2, 3)])
def test_lds_path_prefill(local_blocks, init_blocks, dev):
    d = workloads.stage1_inputs([300, 64, 1000], [8192, 3000, 8192], seed=31)
    _check(d, dev, 8192, local_blocks, init_blocks)


def test_lds_path_cfg3_slice(dev):
    d = workloads.stage1_inputs([8192], [8192], seed=32)
    _check(d, dev, 8192)


@pytest.mark.parametrize("ctx_extra", [0, 8, 70, 2000])
@pytest.mark.parametrize("ctx", [8200, 9000])
def test_pool_width_vs_score_width(ctx, ctx_extra, dev):
    # max_context_len at or above the keys' span: pooled blocks past the
    # computed columns (the tail) hold at most the carried last tap.  8200
    # tokens (511 keys) take the LDS-resident kernel, 9000 (561) the
    # streaming one; ctx_extra 2000 puts pooled blocks past the score row.
    d = workloads.stage1_inputs([40, 17], [2000, ctx], seed=33)
    _check(d, dev, ctx + ctx_extra)


def test_stream_path_long_context(dev):
    d = workloads.stage1_inputs([96, 7], [40000, 135168], seed=34, raw_keys=False)
    _check(d, dev, 135168)


def test_non_causal_and_orphans(dev):
    d = workloads.stage1_inputs([20, 30], [3000, 600], seed=35)
    q = torch.cat([torch.randn(5, 32, 128).to(torch.bfloat16), d["q"]])
    d["q"] = q
    d["cu_seqlens_q"] = d["cu_seqlens_q"] + 5
    _check(d, dev, 3000, causal=False)


@pytest.mark.parametrize("q_len", [2500, 9000])
def test_prefill_rows_see_fewer_keys_than_the_pool(q_len, dev):
    # A prefill over 561 keys (the fused kernel): early tokens see few keys,
    # so blocks past the columns their piece computes lie over zero scores
    # below the key count and pool to 0, not -inf.
    d = workloads.stage1_inputs([q_len], [9000], seed=34)
    _check(d, dev, 9000)


def _fused_c(d, dev, max_context_len, local_blocks, init_blocks, causal, workspace):
    """The fused entry point through the C-ABI, with the key-split workspace
    (key splits, pooling in their second pass) or without it (whole rows)."""
    lib = _lib.load()
    q, k = d["q"].to(dev), d["k"].to(dev)
    cu_q = d["cu_seqlens_q"].to(torch.int32).to(dev)
    cu_k = d["cu_seqlens_k"].to(torch.int32).to(dev)
    B = cu_q.numel() - 1
    Tq, Hq, D = q.shape
    Tk, Hkv, _ = k.shape
    msk = int(d["max_seqlen_k"])
    cols = (msk + 127) // 128 * 128
    nb = (max_context_len + 63) // 64
    scores = torch.empty(Hkv, Tq, cols, device=dev, dtype=torch.float32)
    pooled = torch.empty(Hkv, Tq, nb, device=dev, dtype=torch.float32)
    ws_bytes = lib.unum_infllmv2_attn_stage1_workspace_size(B, Tq, Hq, Hkv, D, msk) if workspace else 0
    assert (ws_bytes > 0) == workspace
    ws = torch.empty(ws_bytes, device=dev, dtype=torch.uint8) if workspace else None
    with torch.cuda.device(dev):
        st = lib.unum_infllmv2_attn_stage1_maxpool(
            _lib.ptr(q), q.stride(0), q.stride(1), _lib.ptr(k), k.stride(0), k.stride(1),
            _lib.ptr(cu_q), _lib.ptr(cu_k), _lib.ptr(scores), _lib.ptr(pooled),
            B, Tq, Tk, Hq, Hkv, D, msk, cols, D ** -0.5, 1 if causal else 0, nb,
            local_blocks, init_blocks, _lib.ptr(ws), ws_bytes, _lib.stream_ptr(dev))
    _lib.check(st, "infllmv2_attn_stage1_maxpool")
    torch.cuda.synchronize()
    return pooled.cpu(), scores.cpu()


@pytest.mark.parametrize("workspace", [False, True])
@pytest.mark.parametrize("q_lens,ctx_lens,causal,local_blocks,init_blocks", [
    ([2500], [9000], True, 1, 1),             # prefill: early pieces see few keys
    ([64, 300, 17], [20000, 9000, 70000], True, 2, 3),
    ([40, 33], [5000, 30000], False, 1, 1),
])
def test_key_splits_and_whole_rows(q_lens, ctx_lens, causal, local_blocks, init_blocks,
                                   workspace, dev):
    # Pooling in the key-split kernels' second pass (each later split first
    # computes the chunk before its own to carry in the -1 tap; the split
    # whose chunks end a piece's columns writes the blocks past them) and in
    # the whole-row kernel: the pooled blocks are the max-pool of the scores
    # the same launch wrote, bit for bit.
    d = workloads.stage1_inputs(q_lens, ctx_lens, seed=36, raw_keys=False)
    max_context_len = max(ctx_lens)
    pooled, scores = _fused_c(d, dev, max_context_len, local_blocks, init_blocks, causal,
                              workspace)
    exp_s = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                          max_seqlen_k=d["max_seqlen_k"], causal=causal)
    torch.testing.assert_close(scores, exp_s, atol=1e-3, rtol=1e-2)
    B = d["cu_seqlens_q"].numel() - 1
    exp_p = oracle_pool(scores, d["cu_seqlens_q"], d["cu_seqlens_k"],
                        torch.zeros(B, dtype=torch.int32), 16 * scores.shape[-1],
                        max_context_len, local_blocks, init_blocks)
    np.testing.assert_array_equal(pooled.numpy(), exp_p)


@pytest.mark.parametrize("q_lens,k_lens", [
    ([1], [4096]), ([1], [513]), ([2], [4095]), ([1, 1], [4096, 64]), ([0, 3, 1, 0, 2], [600, 577, 1, 9, 2049]),
    ([1] * 70, [3000 + 16 * i for i in range(60)] + [1, 2, 63, 64, 65, 127, 128, 129, 640, 0]),
])
@pytest.mark.parametrize("causal,local,init", [(True, 1, 1), (False, 3, 0)])
def test_decode_rows_pooled(q_lens, k_lens, causal, local, init, dev):
    # Batches of at most two tokens a sequence on average, rows of 513 to 4096
    # keys: the one-launch decode kernel, from waves without keys to eight
    # quads each, sequences without tokens and without keys.
    ctx = [16 * (n - 1) + 32 if n > 0 else 8 for n in k_lens]
    d = workloads.stage1_inputs(q_lens, ctx, seed=sum(q_lens) + len(k_lens), raw_keys=False)
    assert 512 < d["max_seqlen_k"] <= 4096 and sum(q_lens) <= 2 * len(q_lens)
    args = [d[n].to(dev) for n in ("q", "k", "cu_seqlens_q", "cu_seqlens_k")]
    kw = dict(max_seqlen_k=d["max_seqlen_k"], causal=causal, local_blocks=local, init_blocks=init)
    mcl = max(ctx) + 333
    pooled, scores = infllmv2_attn_stage1_maxpool(*args, mcl, return_scores=True, **kw)
    only = infllmv2_attn_stage1_maxpool(*args, mcl, **kw)
    assert torch.equal(pooled, only)
    exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                        max_seqlen_k=d["max_seqlen_k"], causal=causal)
    torch.testing.assert_close(scores.cpu(), exp, atol=1e-3, rtol=1e-2)
    cache = torch.zeros(len(q_lens), dtype=torch.int32)
    exp_p = oracle_pool(scores.cpu(), d["cu_seqlens_q"], d["cu_seqlens_k"], cache,
                        16 * scores.shape[-1], mcl, local, init, oob="absent")
    np.testing.assert_array_equal(pooled.cpu().numpy(), exp_p)


@pytest.mark.parametrize("causal", [True, False])
def test_decode_rows_orphans_and_offsets(causal, dev):
    # The decode kernel with tokens before the first sequence and after the
    # last, and a first sequence whose keys lie before k (they read as zero
    # keys: every visible score is 16 / vis).
    k_lens = [700, 600, 900, 3000, 1500, 1400]
    d = workloads.stage1_inputs([1, 2, 1, 0, 1, 1], [16 * (n - 1) + 32 for n in k_lens], seed=40,
                                raw_keys=False)
    d["q"] = torch.cat([d["q"], d["q"]])[:11]            # 2 + 6 + 3 tokens, at most 2 a sequence
    d["cu_seqlens_q"] = d["cu_seqlens_q"] + 2
    d["cu_seqlens_k"] = d["cu_seqlens_k"].clone()
    d["cu_seqlens_k"][0] = -5
    ctx = 16 * 1500
    args = [d[n].to(dev) for n in ("q", "k", "cu_seqlens_q", "cu_seqlens_k")]
    kw = dict(max_seqlen_k=1500, causal=causal)
    pooled, scores = infllmv2_attn_stage1_maxpool(*args, ctx, return_scores=True, **kw)
    assert torch.equal(infllmv2_attn_stage1_maxpool(*args, ctx, **kw), pooled)
    exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"].clamp(min=0),
                        max_seqlen_k=1500, causal=causal)
    vis = 705 if not causal else int(visible_counts(np.arange(1), 1, 705)[0])
    exp[:, 2] = 0.0
    exp[:, 2, :vis] = 16.0 / vis
    scores = scores.cpu()
    torch.testing.assert_close(scores, exp, atol=1e-3, rtol=1e-2)
    assert not scores[:, :2].any() and not scores[:, 8:].any()
    exp_p = oracle_pool(scores, d["cu_seqlens_q"], d["cu_seqlens_k"], torch.zeros(6, dtype=torch.int32),
                        16 * scores.shape[-1], ctx, 1, 1, oob="absent")
    np.testing.assert_array_equal(pooled.cpu().numpy(), exp_p)


def test_decode_ids_against_the_two_ops(dev):
    # Plain stage 1 keeps a decode row's probabilities as f16 exponentials times
    # f16 weights, the fused entry rounds each probability to f16.  On nearly
    # flat rows of up to 3800 keys, as here, all of them are normal f16 values
    # (2^-10 truncated, 2^-11 for a weight; below 2^-14 a probability is off by
    # 2^-24, 16 of them by 2^-20): the two are within 2^-8 of a score and 2^-20,
    # and select the same blocks but for those that near to the K-th score.
    d = workloads.stage1_inputs([1] * 64, [16384 + 700 * i for i in range(64)], seed=41, raw_keys=False)
    args = [d[n].to(dev) for n in ("q", "k", "cu_seqlens_q", "cu_seqlens_k")]
    ctx, K = 16384 + 700 * 63, 64
    fused = infllmv2_attn_stage1_maxpool(*args, ctx, max_seqlen_k=d["max_seqlen_k"], causal=True)
    sc = infllmv2_attn_stage1(args[0], args[1], None, *args[2:], max_seqlen_k=d["max_seqlen_k"], causal=True)
    chain = max_pooling_1d_varlen(sc, *args[2:], torch.zeros(64, dtype=torch.int32, device=dev),
                                  16 * sc.shape[-1], ctx, 1, 1)
    fin = torch.isfinite(chain)
    assert torch.equal(fin, torch.isfinite(fused)) and torch.equal(chain[~fin], fused[~fin])
    far = (fused - chain).abs() - (2 ** -8 * chain + 2 ** -20)
    assert float(far[fin].max()) <= 0
    a, b = topk_blocks(fused, K).cpu(), topk_blocks(chain, K).cpu()
    chain = chain.cpu()
    for h in range(2):
        for t in range(64):
            kth = float(chain[h, t, b[h, t].long()].min())
            for i in set(a[h, t].tolist()) ^ set(b[h, t].tolist()):
                assert abs(float(chain[h, t, i]) - kth) <= 2 ** -7 * kth + 2 ** -19, (h, t, i)


@pytest.mark.parametrize("q_lens,splits", [
    ([1] * 64, False), ([300] + [0] * 255, False), ([1] * 400, False), ([500] + [0] * 511, True),
    ([4] * 64, True),
])
def test_decode_kernel_or_key_splits(q_lens, splits, dev):
    # The decode kernel reads a row's keys for every row: a batch padded with
    # empty sequences that holds one long chunk runs the key splits, which write
    # their workspace; the decode kernel leaves it alone.
    B, T, keys = len(q_lens), sum(q_lens), 600
    g = torch.Generator().manual_seed(T)
    q = torch.randn(T, 32, 128, generator=g).to(torch.bfloat16).to(dev)
    k = torch.randn(B * keys, 2, 128, generator=g).to(torch.bfloat16).to(dev)
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32, device=dev)
    cu_k = torch.arange(B + 1, dtype=torch.int32, device=dev) * keys
    lib = _lib.load()
    need = lib.unum_infllmv2_attn_stage1_workspace_size(B, T, 32, 2, 128, keys)
    assert need > 0
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=dev)
    nb = -(-(16 * keys + 16) // 64)
    pooled = torch.empty(2, T, nb, device=dev)
    st = lib.unum_infllmv2_attn_stage1_maxpool(
        _lib.ptr(q), q.stride(0), q.stride(1), _lib.ptr(k), k.stride(0), k.stride(1),
        _lib.ptr(cu_q), _lib.ptr(cu_k), None, _lib.ptr(pooled), B, T, B * keys, 32, 2, 128, keys,
        640, 128 ** -0.5, 1, nb, 1, 1, _lib.ptr(ws), need, _lib.stream_ptr(q.device))
    _lib.check(st, "infllmv2_attn_stage1_maxpool")
    assert bool((ws != 0xA5).any()) == splits
