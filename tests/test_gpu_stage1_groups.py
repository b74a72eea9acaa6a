"""GPU parity of stage 1 with three and four kv groups of 16 query heads.

The MFMA kernels take a (token, group) row's 16 heads as one 4 KiB run of q,
group g's keys at column g of each key row, and write group g's scores at
``out[g]``; the other tests run them with one or two groups.  Here every MFMA
path -- the LDS-resident kernel (rows of at most 512 keys), the streaming
kernel's whole rows and key splits, and the decode kernel -- runs Hq/Hkv = 48/3
and 64/4 against the fp32 oracle (atol 1e-3 / rtol 1e-2), and the fused
stage-1 + max-pool entry is checked bit for bit against the oracle's pool of
the scores it returns.
"""

import numpy as np
import pytest
import torch

from oracle.maxpool import max_pooling_1d_varlen as oracle_pool
from oracle.stage1 import infllmv2_attn_stage1 as oracle_stage1
import workloads
from unum_ops_amd.infllm_v2 import infllmv2_attn_stage1, infllmv2_attn_stage1_maxpool

pytestmark = pytest.mark.gpu

ATOL, RTOL = 1e-3, 1e-2

# (Hq, Hkv, new tokens per sequence, context per sequence); the comment names
# the kernel the shape takes.
CASES = {
    "lds_3": (48, 3, [200, 64], [6000, 8192]),           # <= 512 keys: LDS-resident
    "lds_4": (64, 4, [96, 33], [3000, 8000]),
    "split_3": (48, 3, [40, 9, 1], [9000, 30000, 12000]),  # few tokens, long rows: key splits
    "rows_4": (64, 4, [300], [12000]),                    # one long prefill piece set
    "decode_3": (48, 3, [1] * 6, [20000] * 6),            # Tq <= 2B, <= 4096 keys: decode
    "decode_4": (64, 4, [1, 2, 1, 1], [9000, 16000, 7000, 12000]),
}


def _inputs(name):
    Hq, Hkv, q_lens, ctx = CASES[name]
    return workloads.stage1_inputs(q_lens, ctx, Hq=Hq, Hkv=Hkv, seed=Hq + 7 * Hkv + len(q_lens))


@pytest.mark.parametrize("name", sorted(CASES))
def test_stage1_groups(name, dev):
    d = _inputs(name)
    out = infllmv2_attn_stage1(d["q"].to(dev), d["k"].to(dev), None, d["cu_seqlens_q"].to(dev),
                               d["cu_seqlens_k"].to(dev), max_seqlen_k=d["max_seqlen_k"],
                               causal=True)
    torch.cuda.synchronize()
    exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                        max_seqlen_k=d["max_seqlen_k"], causal=True)
    assert out.shape == exp.shape and out.shape[0] == CASES[name][1]
    torch.testing.assert_close(out.cpu(), exp, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("name", ["lds_3", "split_3", "rows_4"])
def test_stage1_maxpool_groups(name, dev):
    d = _inputs(name)
    ctx = max(CASES[name][3])
    args = (d["q"].to(dev), d["k"].to(dev), d["cu_seqlens_q"].to(dev), d["cu_seqlens_k"].to(dev), ctx)
    kw = dict(max_seqlen_k=d["max_seqlen_k"], causal=True, local_blocks=1, init_blocks=1)
    pooled, scores = infllmv2_attn_stage1_maxpool(*args, return_scores=True, **kw)
    pooled_only = infllmv2_attn_stage1_maxpool(*args, **kw)
    torch.cuda.synchronize()
    exp_s = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                          max_seqlen_k=d["max_seqlen_k"], causal=True)
    torch.testing.assert_close(scores.cpu(), exp_s, atol=ATOL, rtol=RTOL)
    B = d["cu_seqlens_q"].numel() - 1
    exp_p = oracle_pool(scores.cpu(), d["cu_seqlens_q"], d["cu_seqlens_k"],
                        torch.zeros(B, dtype=torch.int32), 16 * scores.shape[-1], ctx, 1, 1)
    np.testing.assert_array_equal(pooled.cpu().numpy(), exp_p)
    assert torch.equal(pooled_only, pooled)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("G,D", [(1, 128), (2, 64), (3, 96), (4, 128), (5, 72), (7, 128), (8, 128),
                                 (8, 256), (9, 32), (12, 64), (16, 64), (16, 8), (17, 128), (32, 64),
                                 (32, 256), (33, 64), (8, 100), (2, 264)])
def test_other_groups_and_head_sizes(G, D, causal, dev):
    # Every token packing of the M tile (1 to 16 tokens), two tiles a token
    # (G 17..32), head sizes on and between its 32-element steps, and beside
    # them shapes that only the scalar kernel takes (G 33, D 100, D 264).
    # Pieces of every length, rows around the 64-key chunks, an empty sequence,
    # a sequence without keys.  32-bit products and sums: the oracle's and the
    # kernel's exponents (|x| below about 40) each round by 2^-24 |x| or so.
    lens = [1, 130, 0, 37, 200, 5]
    ctx = [1100, 2100, 600, 20, 1040, 1024]
    d = workloads.stage1_inputs(lens, ctx, Hq=2 * G, Hkv=2, D=D, seed=1000 * G + D, peaky=True)
    out = infllmv2_attn_stage1(d["q"].to(dev), d["k"].to(dev), None, d["cu_seqlens_q"].to(dev),
                               d["cu_seqlens_k"].to(dev), max_seqlen_k=d["max_seqlen_k"],
                               causal=causal).cpu()
    exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                        max_seqlen_k=d["max_seqlen_k"], causal=causal)
    torch.testing.assert_close(out, exp, atol=1e-6, rtol=2e-5)


@pytest.mark.parametrize("scale", [-0.05, 0.0, 0.3])
def test_other_groups_any_scale_and_bf16(scale, dev):
    d = workloads.stage1_inputs([70, 3], [1500, 3000], Hq=24, Hkv=3, D=64, seed=5)
    for dt, tol in ((torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8)):
        out = infllmv2_attn_stage1(d["q"].to(dev), d["k"].to(dev), None, d["cu_seqlens_q"].to(dev),
                                   d["cu_seqlens_k"].to(dev), max_seqlen_k=d["max_seqlen_k"],
                                   causal=True, softmax_scale=scale, out_dtype=dt).cpu().float()
        exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"],
                            max_seqlen_k=d["max_seqlen_k"], causal=True, softmax_scale=scale)
        torch.testing.assert_close(out, exp, atol=1e-6, rtol=tol)


@pytest.mark.parametrize("Hq,Hkv,D", [(32, 4, 128), (24, 3, 64), (34, 2, 96)])
def test_other_groups_strided_inputs(Hq, Hkv, D, dev):
    # q and k as slices of wider tensors (16-byte aligned rows and heads): the
    # same bits as packed copies; and one element further on, where the scalar
    # kernel runs, the oracle's values.
    d = workloads.stage1_inputs([90, 33], [2500, 1800], Hq=Hq, Hkv=Hkv, D=D, seed=Hq)
    cu_q, cu_k = d["cu_seqlens_q"].to(dev), d["cu_seqlens_k"].to(dev)
    kw = dict(max_seqlen_k=d["max_seqlen_k"], causal=True)
    exp = oracle_stage1(d["q"], d["k"], None, d["cu_seqlens_q"], d["cu_seqlens_k"], **kw)
    base = infllmv2_attn_stage1(d["q"].to(dev), d["k"].to(dev), None, cu_q, cu_k, **kw)
    for off in (8, 1):
        q = torch.zeros(d["q"].shape[0], Hq + 2, D + 24, dtype=torch.bfloat16, device=dev)
        k = torch.zeros(d["k"].shape[0], Hkv + 1, D + 16, dtype=torch.bfloat16, device=dev)
        qs, ks = q[:, 1:Hq + 1, off:off + D], k[:, :Hkv, off:off + D]
        qs.copy_(d["q"])
        ks.copy_(d["k"])
        out = infllmv2_attn_stage1(qs, ks, None, cu_q, cu_k, **kw)
        if off == 8:
            assert torch.equal(out, base)
        torch.testing.assert_close(out.cpu(), exp, atol=1e-6, rtol=2e-5)


def test_grid_of_2_to_24_pieces(dev):
    # 65535 kv heads x (1 token piece + 256 sequences): more four-wave
    # workgroups than a launch takes, so the scalar kernel runs.
    Hkv, G, D, B, T, lk = 65535, 32, 8, 256, 2, 20
    g = torch.Generator(device=dev).manual_seed(3)
    q = torch.randn(T, Hkv * G, D, generator=g, device=dev).to(torch.bfloat16)
    k = torch.randn(lk, Hkv, D, generator=g, device=dev).to(torch.bfloat16)
    cu_q = torch.full((B + 1,), T, dtype=torch.int32, device=dev)
    cu_k = torch.full((B + 1,), lk, dtype=torch.int32, device=dev)
    cu_q[0] = cu_k[0] = 0
    out = infllmv2_attn_stage1(q, k, None, cu_q, cu_k, max_seqlen_k=lk, causal=False)
    x = (q.float().view(T, Hkv, G, 1, D) * k.float().permute(1, 0, 2).reshape(1, Hkv, 1, lk, D)).sum(-1)
    exp = torch.softmax(x * D ** -0.5, -1).sum(2).transpose(0, 1)
    torch.testing.assert_close(out[:, :, :lk], exp, atol=1e-6, rtol=2e-5)
    assert not out[:, :, lk:].any()
