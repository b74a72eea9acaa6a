#!/usr/bin/env python3
"""Benchmark of the InfLLM-v2 selection path on one MI355X.

Metric: "stage1 TFLOP/s (% bf16 MFMA peak); maxpool+block-table
GB/s (% HBM) @32K".  One step runs the three kernels on their "@32K" headline
configurations with inputs resident in HBM:

* stage 1   : cfg3, 4 x 8192-token causal prefill, Hq=32/Hkv=2/D=128, bf16 in,
              fp32 scores [2, 32768, 512];
* max-pool  : cfg2, 34816 rows of 1024 fp32 scores -> [2, 34816, 256];
* block tab.: the block-table stage of cfg5 (4096 query tokens of a 131072-token
              context, H=2, top-64) -> int32 [4096, 2, 4096] (134 MB).

``value`` is the stage-1 useful TFLOP/s (QK^T over the visible keys, counted
once); the max-pool and block-table bandwidths are in ``components``.  Each
kernel's average duration comes from HIP events recorded on torch's current
stream, the stream the kernels are launched on.  ``cpu_baseline`` times the CPU
oracle (the reference algorithm restated in torch/numpy) on a bounded sample on
this host's cores.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline]
"""

import argparse
import json
import os
import sys
import time

PEAK_HBM_GBS = 8000.0       # MI355X HBM3E
PEAK_BF16_TFLOPS = 2500.0   # MI355X dense bf16 MFMA
METRIC = ("stage1 TFLOP/s (% bf16 MFMA peak); maxpool+block-table GB/s (% HBM) @32K")


# Components whose kernel is shorter than the Python wrapper's host time per
# call (measured: 4.3, 5.3 and 12.0 us of GPU time against 11-16 us between
# eager launches); their calls allocate with torch.empty and never sync with the
# host, so they are captured in a HIP graph and timed without the launch gaps.
# The other components' kernels outlast the host time per call (graph and
# eager timings agree within a few percent), so they are timed eagerly.
GRAPH_TIMED = ("block_table_cfg5_h16", "block_table_cfg4", "ref_block_table_256")


# Untimed back-to-back run of each kernel before its timed launches.  After
# idle the GPU's clock takes about 25 ms of load to settle: stage 1 on cfg3
# measured 128-136 us per launch in its first 2 ms and 104-108 us from 25 ms
# on, batches of 20 launches read by HIP events.
KERNEL_WARM_S = 0.03


def warm(fn, seconds):
    """Run `fn` back to back for `seconds` of wall time, untimed."""
    import torch
    t0 = time.perf_counter()
    while True:
        for _ in range(8):
            fn()
        torch.cuda.synchronize()
        if time.perf_counter() - t0 >= seconds:
            return


def graph_ms(fn, steps):
    """Milliseconds per call of `fn` as a HIP graph of `steps` captured calls."""
    import torch
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # torch's capture wants the work seen once off the capture
        fn()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(steps):
            fn()
    g.replay()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    g.replay()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / steps
    del g
    return ms


def parse():
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=100)
    ap.add_argument("--no-cpu-baseline", action="store_true",
                    help="skip the CPU oracle timing (e.g. under a profiler)")
    ap.add_argument("--only", choices=["stage1", "maxpool", "block_table", "stage1_cfg5",
                                       "maxpool_cfg5", "maxpool_topk", "maxpool_topk_cfg5",
                                       "compress_keys_cfg5", "stage1_maxpool",
                                       "stage1_maxpool_cfg5", "stage1_cfg4", "stage1_decode",
                                       "stage1_maxpool_decode", "stage1_group8",
                                       "stage2_decode", "stage1_peaky", "stage1_cfg5_h16", "maxpool_cfg5_h16",
                                       "block_table_cfg5_h16", "block_table_cfg4",
                                       "stage1_maxpool_cfg4", "stage2_cfg5", "stage2_cfg4",
                                       "topk_cfg5", "select_cfg5", "stage2_gather_cfg5",
                                       "stage2_gather_cfg4", "stage1_bf16", "ref_stage1_1024",
                                       "ref_maxpool_8192", "ref_block_table_256", "copy"],
                    default=None,
                    help="run a single kernel (profiling); 'copy' runs a plain 256 MiB device "
                         "copy, the calibration for the FETCH_SIZE / WRITE_SIZE counters")
    return ap.parse_args()


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def build_inputs(dev):
    import torch

    from tests import workloads
    from unum_ops_amd.infllm_v2 import (infllmv2_attn_stage1, infllmv2_attn_stage1_maxpool,
                                        max_pooling_1d_varlen)
    from unum_ops_amd.pipeline import topk_blocks

    t0 = time.time()
    s1 = workloads.cfg3_stage1()
    s1g = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in s1.items()}
    mp = workloads.cfg2_maxpool()
    mpg = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in mp.items()}
    log(f"cfg3/cfg2 inputs ready ({time.time() - t0:.1f}s)")
    # block-table inputs: run the cfg5 pipeline up to top-k once (untimed)
    p5 = workloads.cfg5_pipeline()
    q5, k5 = p5["q"].to(dev), p5["k"].to(dev)
    cu_q5, cu_k5 = p5["cu_seqlens_q"].to(dev), p5["cu_seqlens_k"].to(dev)
    sc = infllmv2_attn_stage1(q5, k5, None, cu_q5, cu_k5, max_seqlen_k=p5["max_seqlen_k"],
                              causal=True)
    kp = sc.shape[-1]
    pooled = max_pooling_1d_varlen(sc, cu_q5, cu_k5, torch.zeros(1, dtype=torch.int32, device=dev),
                                   max_seqlen_q=16 * kp, max_context_len=p5["max_context_len"],
                                   local_blocks=1, init_blocks=1)
    topk = topk_blocks(pooled, 64)
    bt = dict(topk_idx=topk, block_table=p5["block_table"].to(dev),
              token_to_bs=p5["token_to_bs"].to(dev), token_pos_in_bs=p5["token_pos_in_bs"].to(dev),
              seqlen_q=p5["seqlen_q"].to(dev))
    # cfg5's stage 1 and max-pool are timed too (reported as components, not
    # part of the headline step), and key compression on its raw keys.
    raw5 = torch.randn(135168, 2, 128, generator=torch.Generator().manual_seed(5)).to(
        torch.bfloat16).to(dev)
    c5 = dict(raw=raw5, cu_raw=torch.tensor([0, 135168], dtype=torch.int32, device=dev),q=q5, k=k5, cu_q=cu_q5, cu_k=cu_k5, max_seqlen_k=p5["max_seqlen_k"],
              max_context_len=p5["max_context_len"], scores=sc,
              cache=torch.zeros(1, dtype=torch.int32, device=dev),
              cu_q_cpu=p5["cu_seqlens_q"], cu_k_cpu=p5["cu_seqlens_k"])
    c5["pooled"] = pooled
    # cfg4: 64 decode / chunked-prefill sequences (1-16 new tokens after
    # 16K-64K cached ones), stage 1 over their compressed keys.
    p4 = workloads.cfg4_pipeline()
    c4 = dict(q=p4["q"].to(dev), k=p4["k"].to(dev), cu_q=p4["cu_seqlens_q"].to(dev),
              cu_k=p4["cu_seqlens_k"].to(dev), max_seqlen_k=p4["max_seqlen_k"],
              cu_q_cpu=p4["cu_seqlens_q"], cu_k_cpu=p4["cu_seqlens_k"])
    c5["cfg4"] = c4
    # Pure decode (not a BASELINE config; the serving shape the decode kernel
    # is for): 64 sequences of one new token after 32768 cached tokens.
    pd = workloads.pipeline_inputs([1] * 64, [32768] * 64, raw_keys=False)
    c5["decode"] = dict(q=pd["q"].to(dev), k=pd["k"].to(dev), cu_q=pd["cu_seqlens_q"].to(dev),
                        cu_k=pd["cu_seqlens_k"].to(dev), max_seqlen_k=pd["max_seqlen_k"],
                        cu_q_cpu=pd["cu_seqlens_q"], cu_k_cpu=pd["cu_seqlens_k"],
                        max_context_len=pd["max_context_len"],
                        bt={n: pd[n].to(dev) for n in ("block_table", "token_to_bs",
                                                       "token_pos_in_bs", "seqlen_q")})
    cd = c5["decode"]
    cd["bt"]["topk_idx"] = topk_blocks(
        infllmv2_attn_stage1_maxpool(cd["q"], cd["k"], cd["cu_q"], cd["cu_k"],
                                     cd["max_context_len"], max_seqlen_k=cd["max_seqlen_k"]), 64)
    # Eight query heads a kv head: a prefill.
    p8 = workloads.stage1_inputs([2000, 2400], [2000, 2400], Hq=32, Hkv=4, seed=8)
    c5["group8"] = dict(q=p8["q"].to(dev), k=p8["k"].to(dev), cu_q=p8["cu_seqlens_q"].to(dev),
                        cu_k=p8["cu_seqlens_k"].to(dev), max_seqlen_k=p8["max_seqlen_k"],
                        cu_q_cpu=p8["cu_seqlens_q"], cu_k_cpu=p8["cu_seqlens_k"])
    # cfg5's Hq16/Hkv1 variant through the same stages (H = 1 everywhere).
    p6 = workloads.cfg5_pipeline(Hq=16, Hkv=1)
    q6, k6 = p6["q"].to(dev), p6["k"].to(dev)
    sc6 = infllmv2_attn_stage1(q6, k6, None, cu_q5, cu_k5, max_seqlen_k=p6["max_seqlen_k"],
                               causal=True)
    pooled6 = max_pooling_1d_varlen(sc6, cu_q5, cu_k5, torch.zeros(1, dtype=torch.int32, device=dev),
                                    max_seqlen_q=16 * sc6.shape[-1],
                                    max_context_len=p6["max_context_len"], local_blocks=1,
                                    init_blocks=1)
    c5["h16"] = dict(q=q6, k=k6, scores=sc6, max_seqlen_k=p6["max_seqlen_k"],
                     bt=dict(topk_idx=topk_blocks(pooled6, 64), block_table=bt["block_table"],
                             token_to_bs=bt["token_to_bs"], token_pos_in_bs=bt["token_pos_in_bs"],
                             seqlen_q=bt["seqlen_q"]))
    del pooled6
    # cfg4's block-table stage: its stage 1, max-pool and top-64 run once here.
    sc4 = infllmv2_attn_stage1(c4["q"], c4["k"], None, c4["cu_q"], c4["cu_k"],
                               max_seqlen_k=c4["max_seqlen_k"], causal=True)
    pooled4 = max_pooling_1d_varlen(sc4, c4["cu_q"], c4["cu_k"],
                                    torch.zeros(64, dtype=torch.int32, device=dev),
                                    max_seqlen_q=16 * sc4.shape[-1],
                                    max_context_len=p4["max_context_len"], local_blocks=1,
                                    init_blocks=1)
    c4["max_context_len"] = p4["max_context_len"]
    c4["bt"] = dict(topk_idx=topk_blocks(pooled4, 64), block_table=p4["block_table"].to(dev),
                    token_to_bs=p4["token_to_bs"].to(dev),
                    token_pos_in_bs=p4["token_pos_in_bs"].to(dev), seqlen_q=p4["seqlen_q"].to(dev))
    del sc4, pooled4
    # Stage 2 over the selections above: random bf16 paged K/V caches of the
    # configurations' page pools ([pages, 64, Hkv, 128]; cfg5 2112 pages,
    # 138 MB per cache; cfg4 65536 pages, 2.1 GB per cache).
    gen = torch.Generator(device=dev).manual_seed(2)
    c5["kv"] = [torch.randn(2112, 64, 2, 128, generator=gen, device=dev).to(torch.bfloat16)
                for _ in range(2)]
    c4["kv"] = [torch.randn(65536, 64, 2, 128, generator=gen, device=dev).to(torch.bfloat16)
                for _ in range(2)]
    # The reference's published benchmark shapes (largest row of each CSV):
    # stage 1 non-causal 1024 x 1024 (benchmark/test_infllmv2_attn_stage1.py:67-75),
    # the H=8 bf16 max-pool at seqlen 8192 (benchmark/test_max_polling_1d.py:27-56),
    # the block table at B=256, seq 8192, top-k 96 (benchmark/test_sparse_kernel.py:41-100).
    gp = torch.Generator(device=dev).manual_seed(3)
    pub = dict(s1_q=torch.randn(1024, 32, 128, generator=gp, device=dev).to(torch.bfloat16),
               s1_k=torch.randn(1024, 2, 128, generator=gp, device=dev).to(torch.bfloat16),
               s1_cu=torch.tensor([0, 1024], dtype=torch.int32, device=dev),
               mp_x=torch.randn(8, 8192, 16384, generator=gp, device=dev, dtype=torch.bfloat16),
               mp_cu_q=torch.tensor([0, 8192], dtype=torch.int32, device=dev),
               mp_cu_k=torch.tensor([0, 16384], dtype=torch.int32, device=dev),
               mp_cache=torch.zeros(1, dtype=torch.int32, device=dev))
    rb = workloads.reference_test_block_table(256, 8192, 96)
    pub["bt"] = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in rb.items()}
    c5["published"] = pub
    torch.cuda.synchronize()
    log(f"cfg4/cfg5 inputs ready ({time.time() - t0:.1f}s)")
    return s1, s1g, mp, mpg, bt, c5


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (--gpus {args.gpus} requested); "
              "the selection path shards by kv head or by sequence with no exchange, "
              "so multi-GPU throughput is not measured here.", file=sys.stderr)
        sys.exit(2)

    import torch

    from tests import workloads
    from unum_ops_amd.compression import CompressionPlan, compress_keys
    from unum_ops_amd.infllm_v2 import (infllmv2_attn_stage1, infllmv2_attn_stage1_maxpool,
                                        max_pooling_1d_varlen)
    from unum_ops_amd.pipeline import maxpool_topk, select_blocks, topk_blocks
    from unum_ops_amd.sparse_attention import sparse_gather_calibrate, sparse_paged_attention
    from unum_ops_amd.sparse_kernel_extension import get_block_table

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.only == "copy":
        calibration_copy(dev, args)
        return
    s1, s1g, mp, mpg, bt, c5 = build_inputs(dev)
    mp_kw = {k: mp[k] for k in ("max_seqlen_q", "max_context_len", "local_blocks",
                                "init_blocks", "block_size", "stride")}

    def op_stage1():
        return infllmv2_attn_stage1(s1g["q"], s1g["k"], None, s1g["cu_seqlens_q"],
                                    s1g["cu_seqlens_k"], max_seqlen_k=s1g["max_seqlen_k"],
                                    causal=True)

    # cfg3 with its keys times 8 (exact in bf16): peaky scores, as real
    # attention has, against the nearly flat softmax of mean-pooled keys.
    k_peaky = s1g["k"] * 8

    def op_stage1_peaky():
        return infllmv2_attn_stage1(s1g["q"], k_peaky, None, s1g["cu_seqlens_q"],
                                    s1g["cu_seqlens_k"], max_seqlen_k=s1g["max_seqlen_k"],
                                    causal=True)

    def op_maxpool():
        return max_pooling_1d_varlen(mpg["input"], mpg["cu_seqlens_q"], mpg["cu_seqlens_k"],
                                     mpg["cache_lens"], **mp_kw)

    def op_block_table():
        return get_block_table(bt["topk_idx"], bt["block_table"], bt["token_to_bs"],
                               bt["token_pos_in_bs"], bt["seqlen_q"])

    def op_stage1_cfg5():
        return infllmv2_attn_stage1(c5["q"], c5["k"], None, c5["cu_q"], c5["cu_k"],
                                    max_seqlen_k=c5["max_seqlen_k"], causal=True)

    def op_maxpool_cfg5():
        return max_pooling_1d_varlen(c5["scores"], c5["cu_q"], c5["cu_k"], c5["cache"],
                                     max_seqlen_q=16 * c5["scores"].shape[-1],
                                     max_context_len=c5["max_context_len"], local_blocks=1,
                                     init_blocks=1)

    def op_topk():
        return maxpool_topk(mpg["input"], mpg["cu_seqlens_q"], mpg["cu_seqlens_k"],
                            mpg["cache_lens"], topk=64, **mp_kw)

    def op_topk_cfg5():
        return maxpool_topk(c5["scores"], c5["cu_q"], c5["cu_k"], c5["cache"],
                            max_seqlen_q=16 * c5["scores"].shape[-1],
                            max_context_len=c5["max_context_len"], local_blocks=1,
                            init_blocks=1, topk=64)

    plan5 = CompressionPlan(torch.tensor([0, 135168]), 2, 128, dev)

    def op_stage1_maxpool():
        return infllmv2_attn_stage1_maxpool(s1g["q"], s1g["k"], s1g["cu_seqlens_q"],
                                            s1g["cu_seqlens_k"], 8192,
                                            max_seqlen_k=s1g["max_seqlen_k"], causal=True)

    def op_stage1_maxpool_cfg5():
        return infllmv2_attn_stage1_maxpool(c5["q"], c5["k"], c5["cu_q"], c5["cu_k"],
                                            c5["max_context_len"],
                                            max_seqlen_k=c5["max_seqlen_k"], causal=True)

    c4 = c5["cfg4"]

    def op_stage1_cfg4():
        return infllmv2_attn_stage1(c4["q"], c4["k"], None, c4["cu_q"], c4["cu_k"],
                                    max_seqlen_k=c4["max_seqlen_k"], causal=True)

    cd = c5["decode"]

    def op_stage1_decode():
        return infllmv2_attn_stage1(cd["q"], cd["k"], None, cd["cu_q"], cd["cu_k"],
                                    max_seqlen_k=cd["max_seqlen_k"], causal=True)

    def op_stage1_maxpool_decode():
        return infllmv2_attn_stage1_maxpool(cd["q"], cd["k"], cd["cu_q"], cd["cu_k"],
                                            cd["max_context_len"],
                                            max_seqlen_k=cd["max_seqlen_k"], causal=True)

    def op_stage2_decode():
        b = cd["bt"]
        return sparse_paged_attention(cd["q"], c4["kv"][0], c4["kv"][1], 32, 2, 128 ** -0.5,
                                      b["topk_idx"], b["block_table"], b["token_to_bs"],
                                      b["token_pos_in_bs"], b["seqlen_q"])

    c8 = c5["group8"]

    def op_stage1_group8():
        return infllmv2_attn_stage1(c8["q"], c8["k"], None, c8["cu_q"], c8["cu_k"],
                                    max_seqlen_k=c8["max_seqlen_k"], causal=True)

    def op_compress_cfg5():
        return compress_keys(c5["raw"], c5["cu_raw"], plan=plan5)

    h16 = c5["h16"]

    def op_stage1_cfg5_h16():
        return infllmv2_attn_stage1(h16["q"], h16["k"], None, c5["cu_q"], c5["cu_k"],
                                    max_seqlen_k=h16["max_seqlen_k"], causal=True)

    def op_maxpool_cfg5_h16():
        return max_pooling_1d_varlen(h16["scores"], c5["cu_q"], c5["cu_k"], c5["cache"],
                                     max_seqlen_q=16 * h16["scores"].shape[-1],
                                     max_context_len=c5["max_context_len"], local_blocks=1,
                                     init_blocks=1)

    def op_block_table_cfg5_h16():
        b = h16["bt"]
        return get_block_table(b["topk_idx"], b["block_table"], b["token_to_bs"],
                               b["token_pos_in_bs"], b["seqlen_q"])

    def op_block_table_cfg4():
        b = c4["bt"]
        return get_block_table(b["topk_idx"], b["block_table"], b["token_to_bs"],
                               b["token_pos_in_bs"], b["seqlen_q"])

    def op_stage2_cfg5():
        return sparse_paged_attention(c5["q"], c5["kv"][0], c5["kv"][1], 32, 2, 128 ** -0.5,
                                      bt["topk_idx"], bt["block_table"], bt["token_to_bs"],
                                      bt["token_pos_in_bs"], bt["seqlen_q"])

    def op_stage2_cfg4():
        b = c4["bt"]
        return sparse_paged_attention(c4["q"], c4["kv"][0], c4["kv"][1], 32, 2, 128 ** -0.5,
                                      b["topk_idx"], b["block_table"], b["token_to_bs"],
                                      b["token_pos_in_bs"], b["seqlen_q"])

    # The gather time of each stage-2 selection: the same rows read once per
    # (token, kv head), coalesced, with no arithmetic.  Stage 2 can run below
    # it: it moves a block that two neighbouring tokens share once.
    def op_stage2_gather_cfg5():
        return sparse_gather_calibrate(c5["kv"][0], c5["kv"][1], 2, bt["topk_idx"],
                                       bt["block_table"], bt["token_to_bs"],
                                       bt["token_pos_in_bs"], bt["seqlen_q"])

    def op_stage2_gather_cfg4():
        b = c4["bt"]
        return sparse_gather_calibrate(c4["kv"][0], c4["kv"][1], 2, b["topk_idx"],
                                       b["block_table"], b["token_to_bs"],
                                       b["token_pos_in_bs"], b["seqlen_q"])

    # cfg3 with the reference's own storage dtype for the scores (bf16,
    # infllmv2_attn_stage1_triton_v2.py:188-194).
    def op_stage1_bf16():
        return infllmv2_attn_stage1(s1g["q"], s1g["k"], None, s1g["cu_seqlens_q"],
                                    s1g["cu_seqlens_k"], max_seqlen_k=s1g["max_seqlen_k"],
                                    causal=True, out_dtype=torch.bfloat16)

    # The shapes the reference publishes figures for (benchmark/output/
    # Performance_*.csv, largest row of each; inputs as benchmark/*.py build
    # them): context for reading those figures, not a target.
    rp = c5["published"]

    def op_ref_stage1_1024():
        return infllmv2_attn_stage1(rp["s1_q"], rp["s1_k"], rp["s1_k"], rp["s1_cu"], rp["s1_cu"],
                                    cu_seqlens_v=rp["s1_cu"], max_seqlen_q=1024,
                                    max_seqlen_k=1024, causal=False, out_dtype=torch.bfloat16)

    def op_ref_maxpool_8192():
        return max_pooling_1d_varlen(rp["mp_x"], rp["mp_cu_q"], rp["mp_cu_k"], rp["mp_cache"],
                                     8192, max_context_len=8192, local_blocks=32, init_blocks=1,
                                     block_size=64, stride=16)

    def op_ref_block_table_256():
        b = rp["bt"]
        return get_block_table(b["topk_idx"], b["block_table"], b["token_to_bs"],
                               b["token_pos_in_bs"], b["seqlen_q"])

    def op_topk_pooled_cfg5():
        return topk_blocks(c5["pooled"], 64)

    def op_select_cfg5():
        return select_blocks(c5["q"], c5["k"], c5["cu_q"], c5["cu_k"], bt["block_table"],
                             bt["token_to_bs"], bt["token_pos_in_bs"], bt["seqlen_q"],
                             c5["max_context_len"], max_seqlen_k=c5["max_seqlen_k"], topk=64)

    def op_stage1_maxpool_cfg4():
        return infllmv2_attn_stage1_maxpool(c4["q"], c4["k"], c4["cu_q"], c4["cu_k"],
                                            c4["max_context_len"],
                                            max_seqlen_k=c4["max_seqlen_k"], causal=True)

    ops = [("stage1", op_stage1), ("maxpool", op_maxpool), ("block_table", op_block_table)]
    # Timed per kernel only: the long-context configuration's stage 1 and
    # max-pool, the fused pool + top-64 selection on both pool inputs, and key
    # compression of cfg5's raw keys.
    extra = [("stage1_cfg5", op_stage1_cfg5), ("maxpool_cfg5", op_maxpool_cfg5),
             ("maxpool_topk", op_topk), ("maxpool_topk_cfg5", op_topk_cfg5),
             ("compress_keys_cfg5", op_compress_cfg5), ("stage1_maxpool", op_stage1_maxpool),
             ("stage1_maxpool_cfg5", op_stage1_maxpool_cfg5), ("stage1_cfg4", op_stage1_cfg4),
             ("stage1_decode", op_stage1_decode), ("stage1_peaky", op_stage1_peaky),
             ("stage1_maxpool_decode", op_stage1_maxpool_decode),
             ("stage1_group8", op_stage1_group8), ("stage2_decode", op_stage2_decode),
             ("stage1_cfg5_h16", op_stage1_cfg5_h16), ("maxpool_cfg5_h16", op_maxpool_cfg5_h16),
             ("block_table_cfg5_h16", op_block_table_cfg5_h16),
             ("block_table_cfg4", op_block_table_cfg4),
             ("stage1_maxpool_cfg4", op_stage1_maxpool_cfg4),
             ("stage2_cfg5", op_stage2_cfg5), ("stage2_cfg4", op_stage2_cfg4),
             ("stage2_gather_cfg5", op_stage2_gather_cfg5),
             ("stage2_gather_cfg4", op_stage2_gather_cfg4),
             ("topk_cfg5", op_topk_pooled_cfg5), ("select_cfg5", op_select_cfg5),
             ("stage1_bf16", op_stage1_bf16), ("ref_stage1_1024", op_ref_stage1_1024),
             ("ref_maxpool_8192", op_ref_maxpool_8192),
             ("ref_block_table_256", op_ref_block_table_256)]
    if args.only:
        ops = [o for o in ops if o[0] == args.only]
        extra = [o for o in extra if o[0] == args.only]

    for _ in range(args.warmup):
        for _, fn in ops:
            fn()
    torch.cuda.synchronize()
    log(f"warmup done ({args.warmup} steps)")

    # The timed region: K steps of the path (stage 1, max-pool, block table),
    # bracketed by device synchronisation; its wall clock gives ms_per_step.
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        for _, fn in ops:
            fn()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0

    # Per-kernel launch durations: K back-to-back launches of one kernel
    # between two HIP events on torch's current stream (the stream the
    # kernels run on), so per-launch event overhead is amortised; each kernel
    # first runs untimed for KERNEL_WARM_S, so its figure is the settled
    # clock's.
    per_op = {}
    for name, fn in ops + extra:
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        warm(fn, KERNEL_WARM_S)
        e0.record()
        for _ in range(args.steps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        per_op[name] = e0.elapsed_time(e1) / args.steps          # ms
    log("per-kernel: " + ", ".join(f"{k} {v * 1e3:.1f} us" for k, v in per_op.items())
        + f"; step {wall * 1e3 / args.steps:.3f} ms")

    # Kernels shorter than their Python wrapper's ~11 us of host time per call
    # are launch-bound when timed as above: they are timed again as a HIP
    # graph of K captured calls, replayed between two events (the GPU time of
    # K back-to-back launches); the eager figure is kept beside it.
    per_op_eager = {}
    for name, fn in ops + extra:
        if name not in GRAPH_TIMED:
            continue
        per_op_eager[name] = per_op[name]
        per_op[name] = graph_ms(fn, args.steps)
    if per_op_eager:
        log("graph-timed: " + ", ".join(f"{k} {per_op[k] * 1e3:.1f} us (eager {v * 1e3:.1f})"
                                         for k, v in per_op_eager.items()))

    comps = {}
    if "stage1" in per_op:
        flop, nbytes, _ = workloads.stage1_work(s1["cu_seqlens_q"], s1["cu_seqlens_k"], 32, 2,
                                                128, 512)
        t = per_op["stage1"] * 1e-3
        comps["stage1"] = dict(us=per_op["stage1"] * 1e3, tflops=flop / t / 1e12,
                               pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                               gbs=nbytes / t / 1e9, pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                               flop=flop, bytes=nbytes, bound="hbm",
                               config="cfg3 4x8192 causal, Hq32/Hkv2/D128, fp32 out [2,32768,512]")
    if "stage1_peaky" in per_op:
        flop, nbytes, _ = workloads.stage1_work(s1["cu_seqlens_q"], s1["cu_seqlens_k"], 32, 2,
                                                128, 512)
        t = per_op["stage1_peaky"] * 1e-3
        comps["stage1_peaky"] = dict(us=per_op["stage1_peaky"] * 1e3, tflops=flop / t / 1e12,
                                     pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                                     gbs=nbytes / t / 1e9, pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                     flop=flop, bytes=nbytes, bound="hbm",
                                     config="cfg3 with keys x8 (peaky scores), fp32 out [2,32768,512]")
    if "maxpool" in per_op:
        nbytes = workloads.maxpool_bytes(mp["cu_seqlens_q"], mp["cu_seqlens_k"], mp["cache_lens"],
                                         2, 256)
        t = per_op["maxpool"] * 1e-3
        comps["maxpool"] = dict(us=per_op["maxpool"] * 1e3, gbs=nbytes / t / 1e9,
                                pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
                                config="cfg2 q {4096,6144,8192,16384}, fp32 [2,34816,1024]->[2,34816,256]")
    if "block_table" in per_op:
        nbytes = workloads.block_table_bytes(bt["topk_idx"].cpu(), bt["token_to_bs"].cpu(), 2,
                                             4096, 64, 1)
        t = per_op["block_table"] * 1e-3
        comps["block_table"] = dict(us=per_op["block_table"] * 1e3, gbs=nbytes / t / 1e9,
                                    pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                    bytes=nbytes,
                                    config="cfg5 block-table stage: T=4096 H=2 K=64 -> int32 [4096,2,4096]")

    if "stage1_cfg5" in per_op:
        flop, nbytes, _ = workloads.stage1_work(c5["cu_q_cpu"], c5["cu_k_cpu"], 32, 2, 128,
                                                c5["scores"].shape[-1])
        t = per_op["stage1_cfg5"] * 1e-3
        comps["stage1_cfg5"] = dict(us=per_op["stage1_cfg5"] * 1e3, tflops=flop / t / 1e12,
                                    pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                                    gbs=nbytes / t / 1e9,
                                    pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                    flop=flop, bytes=nbytes, bound="mfma",
                                    config="cfg5 4096-token chunk of a 135168-token context, "
                                           "Hq32/Hkv2/D128, fp32 out [2,4096,8448]")
    if "stage1_cfg4" in per_op:
        ncols = -(-c4["max_seqlen_k"] // 128) * 128
        flop, nbytes, _ = workloads.stage1_work(c4["cu_q_cpu"], c4["cu_k_cpu"], 32, 2, 128, ncols)
        t = per_op["stage1_cfg4"] * 1e-3
        comps["stage1_cfg4"] = dict(us=per_op["stage1_cfg4"] * 1e3, tflops=flop / t / 1e12,
                                    pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                                    gbs=nbytes / t / 1e9,
                                    pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                    flop=flop, bytes=nbytes, bound="hbm",
                                    config=f"cfg4 64 sequences, 1-16 new tokens after 16K-64K "
                                           f"cached, Hq32/Hkv2/D128, fp32 out "
                                           f"[2,{int(c4['cu_q_cpu'][-1])},{ncols}]")
    if "stage1_decode" in per_op:
        ncols = -(-cd["max_seqlen_k"] // 128) * 128
        flop, nbytes, _ = workloads.stage1_work(cd["cu_q_cpu"], cd["cu_k_cpu"], 32, 2, 128, ncols)
        t = per_op["stage1_decode"] * 1e-3
        comps["stage1_decode"] = dict(us=per_op["stage1_decode"] * 1e3, tflops=flop / t / 1e12,
                                      gbs=nbytes / t / 1e9,
                                      pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                      flop=flop, bytes=nbytes, bound="hbm",
                                      config=f"decode: 64 sequences of 1 new token after 32768 "
                                             f"cached, Hq32/Hkv2/D128, fp32 out [2,64,{ncols}] "
                                             f"(not a BASELINE config)")
    if "stage1_maxpool_decode" in per_op:
        # the scores not written, the pooled blocks written
        flop, nbytes, _ = workloads.stage1_work(cd["cu_q_cpu"], cd["cu_k_cpu"], 32, 2, 128, 0)
        nblk = -(-cd["max_context_len"] // 64)
        nbytes += 4 * 2 * 64 * nblk
        t = per_op["stage1_maxpool_decode"] * 1e-3
        comps["stage1_maxpool_decode"] = dict(
            us=per_op["stage1_maxpool_decode"] * 1e3, tflops=flop / t / 1e12, gbs=nbytes / t / 1e9,
            pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, flop=flop, bytes=nbytes, bound="hbm",
            config=f"stage1_decode fused with the max-pool: pooled fp32 [2,64,{nblk}] only (scores "
                   f"not stored)")
    if "stage1_group8" in per_op:
        ncols = -(-c8["max_seqlen_k"] // 128) * 128
        flop, nbytes, _ = workloads.stage1_work(c8["cu_q_cpu"], c8["cu_k_cpu"], 32, 4, 128, ncols)
        t = per_op["stage1_group8"] * 1e-3
        comps["stage1_group8"] = dict(
            us=per_op["stage1_group8"] * 1e3, tflops=flop / t / 1e12,
            pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS, gbs=nbytes / t / 1e9,
            pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, flop=flop, bytes=nbytes, bound="hbm",
            config=f"prefill of 2000 and 2400 tokens, causal, Hq32/Hkv4/D128, fp32 out "
                   f"[4,4400,{ncols}]")
    if "maxpool_cfg5" in per_op:
        nbytes = workloads.maxpool_bytes(c5["cu_q_cpu"], c5["cu_k_cpu"], [0], 2,
                                         -(-c5["max_context_len"] // 64))
        t = per_op["maxpool_cfg5"] * 1e-3
        comps["maxpool_cfg5"] = dict(us=per_op["maxpool_cfg5"] * 1e3, gbs=nbytes / t / 1e9,
                                     pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                     bytes=nbytes,
                                     config="cfg5 scores fp32 [2,4096,8448] -> [2,4096,2112]")

    for name, cu_q, cu_k, nbk in (("maxpool_topk", mp["cu_seqlens_q"], mp["cu_seqlens_k"], 256),
                                  ("maxpool_topk_cfg5", c5["cu_q_cpu"], c5["cu_k_cpu"],
                                   -(-c5["max_context_len"] // 64))):
        if name in per_op:
            rows = 2 * (int(cu_q[-1]) if name == "maxpool_topk_cfg5" else mp["input"].shape[1])
            cache = mp["cache_lens"] if name == "maxpool_topk" else [0]
            nbytes = (workloads.maxpool_bytes(cu_q, cu_k, cache, 2, nbk) - 4 * rows * nbk
                      + 4 * rows * 64)                   # pooled scores read, ids written
            t = per_op[name] * 1e-3
            comps[name] = dict(us=per_op[name] * 1e3, gbs=nbytes / t / 1e9,
                               pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
                               config=("cfg2 input" if name == "maxpool_topk" else "cfg5 scores")
                               + " -> top-64 block ids int32 [2, T, 64]")

    if "topk_cfg5" in per_op:
        rows, nbk = 2 * int(c5["cu_q_cpu"][-1]), -(-c5["max_context_len"] // 64)
        nbytes = 4 * rows * nbk + 4 * rows * 64           # pooled rows read, ids written
        t = per_op["topk_cfg5"] * 1e-3
        comps["topk_cfg5"] = dict(us=per_op["topk_cfg5"] * 1e3, gbs=nbytes / t / 1e9,
                                  pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
                                  config="cfg5 pooled fp32 [2,4096,2112] -> top-64 block ids "
                                         "int32 [2,4096,64]")
    if "select_cfg5" in per_op:
        comps["select_cfg5"] = dict(
            us=per_op["select_cfg5"] * 1e3,
            config="select_blocks on cfg5 end to end: stage 1 with the max-pool in its kernel, "
                   "top-64 over the pooled rows, block table int32 [4096,2,4096]")

    if "stage1_cfg5_h16" in per_op:
        flop, nbytes, _ = workloads.stage1_work(c5["cu_q_cpu"], c5["cu_k_cpu"], 16, 1, 128,
                                                h16["scores"].shape[-1])
        t = per_op["stage1_cfg5_h16"] * 1e-3
        comps["stage1_cfg5_h16"] = dict(us=per_op["stage1_cfg5_h16"] * 1e3, tflops=flop / t / 1e12,
                                        pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                                        gbs=nbytes / t / 1e9,
                                        pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                        flop=flop, bytes=nbytes, bound="mfma",
                                        config="cfg5 Hq16/Hkv1 variant, fp32 out [1,4096,8448]")
    if "maxpool_cfg5_h16" in per_op:
        nbytes = workloads.maxpool_bytes(c5["cu_q_cpu"], c5["cu_k_cpu"], [0], 1,
                                         -(-c5["max_context_len"] // 64))
        t = per_op["maxpool_cfg5_h16"] * 1e-3
        comps["maxpool_cfg5_h16"] = dict(us=per_op["maxpool_cfg5_h16"] * 1e3, gbs=nbytes / t / 1e9,
                                         pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                         bytes=nbytes,
                                         config="cfg5 Hq16/Hkv1 scores fp32 [1,4096,8448] -> [1,4096,2112]")
    for name, b, T, B, cfg in (
            ("block_table_cfg5_h16", h16["bt"], 4096, 1,
             "cfg5 Hq16/Hkv1 block-table stage: T=4096 H=1 K=64 -> int32 [4096,1,4096]"),
            ("block_table_cfg4", c4["bt"], int(c4["cu_q_cpu"][-1]), 64,
             f"cfg4 block-table stage: T={int(c4['cu_q_cpu'][-1])} H=2 K=64, 64 sequences "
             f"-> int32 [{int(c4['cu_q_cpu'][-1])},2,4096] (latency-bound)")):
        if name in per_op:
            H = b["topk_idx"].shape[0]
            nbytes = workloads.block_table_bytes(b["topk_idx"].cpu(), b["token_to_bs"].cpu(), H, T,
                                                 64, B)
            t = per_op[name] * 1e-3
            comps[name] = dict(us=per_op[name] * 1e3, gbs=nbytes / t / 1e9,
                               pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
                               config=cfg)

    for name, b, nseq, cfg in (
            ("stage2_cfg5", bt, 1, "cfg5 selection: T=4096, Hq32/Hkv2, top-64 blocks of 64 tokens, "
                                   "paged bf16 K/V [2112,64,2,128], bf16 out [4096,32,128]"),
            ("stage2_cfg4", c4["bt"], 64, "cfg4 selection: 64 sequences, Hq32/Hkv2, top-64, paged "
                                         "bf16 K/V [65536,64,2,128], bf16 out"),
            ("stage2_decode", cd["bt"], 64, "stage1_decode's selection: 64 sequences of 1 token, "
                                            "Hq32/Hkv2, top-64, paged bf16 K/V [65536,64,2,128], "
                                            "bf16 out")):
        if name in per_op:
            nbytes, flop, n_ent = workloads.sparse_attn_work(b["topk_idx"], b["token_to_bs"],
                                                             b["token_pos_in_bs"], b["seqlen_q"],
                                                             nseq)
            t = per_op[name] * 1e-3
            comps[name] = dict(us=per_op[name] * 1e3, tflops=flop / t / 1e12,
                               pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                               gathered_gbs=nbytes / t / 1e9, bytes_gathered=nbytes, flop=flop,
                               entries=n_ent, bound="gather",
                               config=cfg + " (bytes_gathered: every attended K and V row once "
                                            "per token and kv head, q, out; rows gathered by "
                                            "neighbouring tokens hit the L2 / MALL, so "
                                            "gathered_gbs may exceed the HBM peak; beside it "
                                            "the same rows read with no arithmetic, "
                                            "stage2_gather_*)")
            gather = name.replace("stage2_", "stage2_gather_")
            if gather in per_op:
                comps[name].update(gather_us=per_op[gather] * 1e3,
                                   gather_over_time=per_op[gather] / per_op[name])
    for name in ("stage2_gather_cfg5", "stage2_gather_cfg4"):
        if name in per_op:
            comps[name] = dict(us=per_op[name] * 1e3,
                               config="calibration: every row " + name.replace("stage2_gather_", "")
                                      + "'s stage 2 attends, gathered once per token and kv head "
                                        "(coalesced, no arithmetic)")

    if "stage1_bf16" in per_op:
        flop, nbytes, _ = workloads.stage1_work(s1["cu_seqlens_q"], s1["cu_seqlens_k"], 32, 2,
                                                128, 512, out_bytes=2)
        t = per_op["stage1_bf16"] * 1e-3
        comps["stage1_bf16"] = dict(us=per_op["stage1_bf16"] * 1e3, tflops=flop / t / 1e12,
                                    pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                                    gbs=nbytes / t / 1e9,
                                    pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                    flop=flop, bytes=nbytes, bound="hbm",
                                    config="cfg3 with bf16 scores (the reference's storage "
                                           "dtype) [2,32768,512]")
    if "ref_stage1_1024" in per_op:
        flop, nbytes, _ = workloads.stage1_work([0, 1024], [0, 1024], 32, 2, 128, 1024,
                                                causal=False, out_bytes=2)
        t = per_op["ref_stage1_1024"] * 1e-3
        comps["ref_stage1_1024"] = dict(
            us=per_op["ref_stage1_1024"] * 1e3, tflops=flop / t / 1e12,
            pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS, gbs=nbytes / t / 1e9,
            pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, flop=flop, bytes=nbytes,
            reference_published_ms={"CUDA": 0.264032, "Triton": 1.410048, "Triton_v2": 0.95744},
            config="the reference's published stage-1 shape: seqlen_q = seqlen_k = 1024, "
                   "non-causal, Hq32/Hkv2/D128, bf16 scores [2,1024,1024] "
                   "(Performance_infllmv2_attn_stage1.csv:9; its GPU is not named)")
    if "ref_maxpool_8192" in per_op:
        nbytes = workloads.maxpool_bytes([0, 8192], [0, 16384], [0], 8, 128, elem=2)
        t = per_op["ref_maxpool_8192"] * 1e-3
        comps["ref_maxpool_8192"] = dict(
            us=per_op["ref_maxpool_8192"] * 1e3, gbs=nbytes / t / 1e9,
            pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
            reference_published_ms={"CUDA": 0.432128, "Triton": 0.55552},
            config="the reference's published max-pool shape: H=8, seqlen 8192, bf16 scores "
                   "[8,8192,16384] read with row stride 512, local 32, init 1 -> [8,8192,128] "
                   "(Performance_max_pooling_1d.csv:9; its GPU is not named)")
    if "ref_block_table_256" in per_op:
        b = c5["published"]["bt"]
        nbytes = workloads.block_table_bytes(b["topk_idx"].cpu(), b["token_to_bs"].cpu(), 2, 256,
                                             96, 256)
        t = per_op["ref_block_table_256"] * 1e-3
        comps["ref_block_table_256"] = dict(
            us=per_op["ref_block_table_256"] * 1e3, gbs=nbytes / t / 1e9,
            pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS, bytes=nbytes,
            reference_published_ms={"Torch": 0.616416, "CUDA_v3": 0.173056,
                                    "Triton_v3": 0.116736},
            config="the reference's published block-table shape: B=256, seq 8192, top-k 96 "
                   "(inputs regenerated from benchmark/test_sparse_kernel.py:41-100's seeds) "
                   "-> int32 [256,2,6144] (Performance_get_block_table.csv:7; its GPU is not "
                   "named)")

    for name, src in (("stage1_maxpool", "stage1"), ("stage1_maxpool_cfg5", "stage1_cfg5"),
                      ("stage1_maxpool_cfg4", "stage1_cfg4")):
        if name in per_op and src in comps:
            # the unfused kernel's bytes with its score tensor replaced by the
            # pooled tensor (both sizes read off one call's outputs)
            fns = dict(ops + extra)
            scores, pooled = fns[src](), fns[name]()
            flop = comps[src]["flop"]
            nbytes = comps[src]["bytes"] - scores.numel() * scores.element_size() \
                + pooled.numel() * pooled.element_size()
            t = per_op[name] * 1e-3
            comps[name] = dict(us=per_op[name] * 1e3, tflops=flop / t / 1e12,
                               pct_bf16_mfma_peak=100 * flop / t / 1e12 / PEAK_BF16_TFLOPS,
                               gbs=nbytes / t / 1e9,
                               pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                               flop=flop, bytes=nbytes, bound=comps[src]["bound"],
                               config=f"{src} fused with the max-pool: pooled fp32 "
                                      f"{list(pooled.shape)} only (scores not stored)")
    if "compress_keys_cfg5" in per_op:
        nbytes = 2 * 135168 * 2 * 128 + 2 * 8447 * 2 * 128
        t = per_op["compress_keys_cfg5"] * 1e-3
        comps["compress_keys_cfg5"] = dict(us=per_op["compress_keys_cfg5"] * 1e3,
                                           gbs=nbytes / t / 1e9,
                                           pct_hbm_peak=100 * nbytes / t / 1e9 / PEAK_HBM_GBS,
                                           bytes=nbytes,
                                           config="cfg5 raw keys bf16 [135168,2,128] -> "
                                                  "[8447,2,128] (kernel 32, stride 16), "
                                                  "planned (no host sync)")
    for name, eager_ms in per_op_eager.items():
        if name in comps:
            comps[name].update(us_eager=eager_ms * 1e3, timing=f"HIP graph of {args.steps} calls")

    cpu = None
    if not args.no_cpu_baseline and "stage1" in comps:
        cpu = cpu_baseline(s1, mp, bt)

    s1c = comps.get("stage1")
    line = {
        "metric": METRIC,
        "value": round(s1c["tflops"], 3) if s1c else None,
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall * 1e3 / args.steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded torch.Generator('cpu'), BASELINE.json configs)",
        "config": {"workload": "selection path @32K: stage1 cfg3 + maxpool cfg2 + "
                               "block table cfg5 (headline value: stage1 cfg3)",
                   "stage1": "cfg3", "maxpool": "cfg2", "block_table": "cfg5 stage",
                   "parallelism": "single GPU"},
        "components": {k: {kk: (round(vv, 4) if isinstance(vv, float) else vv)
                           for kk, vv in v.items()} for k, v in comps.items()},
    }
    if s1c:
        line["roofline"] = {"bound": "hbm", "achieved": round(s1c["gbs"], 1),
                            "peak": PEAK_HBM_GBS, "unit": "GB/s",
                            "frac": round(s1c["gbs"] / PEAK_HBM_GBS, 4),
                            "traffic": profiled_traffic("stage1_cfg3.txt",
                                                        "unum_ops_amd/csrc/stage1.hip"),
                            "kernel": "stage1 (cfg3)",
                            "mfma_frac": round(s1c["tflops"] / PEAK_BF16_TFLOPS, 4)}
    line["cpu_baseline"] = cpu
    print(json.dumps(line), flush=True)


def calibration_copy(dev, args):
    """A plain 256 MiB device-to-device copy (reads and writes exactly 256 MiB):
    what FETCH_SIZE / WRITE_SIZE report for it scales the kernels' readings."""
    import torch

    n = 256 << 20
    src = torch.ones(n // 4, dtype=torch.float32, device=dev)
    dst = torch.empty_like(src)
    for _ in range(args.warmup + args.steps):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"calibration": "copy", "bytes_read": n, "bytes_written": n}), flush=True)


def source_digest(rel):
    """sha256 (first 16 hex digits) of a repository file."""
    import hashlib

    with open(os.path.join(os.path.dirname(os.path.abspath(__file__)), rel), "rb") as f:
        return hashlib.sha256(f.read()).hexdigest()[:16]


def profiled_traffic(name, source):
    """HBM bytes per launch of a kernel, as measured with the FETCH_SIZE and
    WRITE_SIZE counters (copy-calibrated) and recorded in profiles/<name>.
    The summary records the sha256 of the kernel's source it was measured
    on; when that source has changed since, or the summary is absent, the
    reading no longer describes this build and None is returned."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", name)
    traffic, digest = None, None
    try:
        with open(path) as f:
            for row in f:
                if row.startswith("traffic_bytes_per_launch:"):
                    traffic = int(float(row.split(":", 1)[1].split()[0]))
                elif row.startswith("source_sha256:"):
                    digest = row.split(":", 1)[1].split()[0]
    except OSError:
        return None
    if digest is None or digest != source_digest(source):
        log(f"profiles/{name} was measured on another {source}: traffic not reported")
        return None
    return traffic


def host_cpu():
    """The host's CPU model, physical cores and the CPUs this process may use."""
    model, cores = None, set()
    phys = None
    try:
        with open("/proc/cpuinfo") as f:
            for row in f:
                key, _, val = row.partition(":")
                key, val = key.strip(), val.strip()
                if key == "model name" and model is None:
                    model = val
                elif key == "physical id":
                    phys = val
                elif key == "core id":
                    cores.add((phys, val))
    except OSError:
        pass
    try:
        avail = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        avail = os.cpu_count()
    # When the model name is generic (a VM may report just the vendor line),
    # add lscpu's model name and the family / model / stepping numbers.
    fms = {}
    try:
        with open("/proc/cpuinfo") as f:
            for row in f:
                key, _, val = row.partition(":")
                key = key.strip()
                if key in ("cpu family", "model", "stepping") and key not in fms:
                    fms[key] = val.strip()
                if len(fms) == 3:
                    break
    except OSError:
        pass
    try:
        import subprocess
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for row in out.splitlines():
            if row.startswith("Model name:"):
                name = row.split(":", 1)[1].strip()
                if name and (model is None or len(name) > len(model)):
                    model = name
    except (OSError, ValueError, subprocess.SubprocessError):
        pass
    if fms:
        model = f"{model or 'unknown'} (family {fms.get('cpu family', '?')}, model " \
                f"{fms.get('model', '?')}, stepping {fms.get('stepping', '?')})"
    return {"cpu_model": model, "physical_cores": len(cores) or None, "cpus_available": avail}


def _median_time(fn, budget_s, min_runs=3):
    times = []
    t_end = time.time() + budget_s
    while len(times) < min_runs or time.time() < t_end:
        t0 = time.perf_counter()
        fn()
        times.append(time.perf_counter() - t0)
    return sorted(times)[len(times) // 2], len(times)


def cpu_baseline(s1, mp, bt):
    """The CPU oracle -- the reference algorithm of each op restated in torch
    (oracle/) -- on this host, on every thread the process may use, median of
    bounded repeated runs:

    * stage 1 (the headline unit, TFLOP/s): torch fp32, the whole cfg3
      workload, about 10 s;
    * max-pool (GB/s): the torch restatement of the reference's Triton kernel
      (max_pooling_1d_varlen.py:33-124; the reference has no torch version)
      on the whole cfg2 input, at least 3 runs;
    * block table (GB/s): get_block_table_ref_torch's steps in torch
      (get_table_torch.py:4-44: block_table[bs], gather, where) on the whole
      cfg5 block-table stage, at least 3 runs.
    """
    import torch

    from oracle.block_table import get_block_table_torch
    from oracle.maxpool import max_pooling_1d_varlen_torch
    from oracle.stage1 import infllmv2_attn_stage1 as oracle_stage1
    from tests import workloads

    host = host_cpu()
    threads = host["cpus_available"] or os.cpu_count() or 1
    torch.set_num_threads(threads)
    threads = torch.get_num_threads()
    flop, _, _ = workloads.stage1_work(s1["cu_seqlens_q"], s1["cu_seqlens_k"], 32, 2, 128, 512)
    oracle_stage1(s1["q"][:512], s1["k"][:511], None, torch.tensor([0, 512], dtype=torch.int32),
                  torch.tensor([0, 511], dtype=torch.int32), max_seqlen_k=511,
                  causal=True)                                          # warm-up
    med, n = _median_time(lambda: oracle_stage1(
        s1["q"], s1["k"], None, s1["cu_seqlens_q"], s1["cu_seqlens_k"],
        max_seqlen_k=s1["max_seqlen_k"], causal=True), 10)
    log(f"cpu baseline: stage 1 {med:.2f} s per cfg3 pass ({n} runs, {threads} threads)")
    line = {"value": round(flop / med / 1e12, 5), "unit": "TFLOP/s", "cores": threads,
            "kind": "port",
            "sample": f"oracle stage 1 (torch fp32 CPU) on the whole cfg3 workload (4 x 8192 "
                      f"tokens), median of {n} runs", **host}

    mp_bytes = workloads.maxpool_bytes(mp["cu_seqlens_q"], mp["cu_seqlens_k"], mp["cache_lens"],
                                       2, 256)
    med, n = _median_time(lambda: max_pooling_1d_varlen_torch(
        mp["input"], mp["cu_seqlens_q"], mp["cu_seqlens_k"], mp["cache_lens"],
        mp["max_seqlen_q"], mp["max_context_len"], mp["local_blocks"], mp["init_blocks"]), 5)
    log(f"cpu baseline: max-pool {med:.2f} s per cfg2 pass ({n} runs, {threads} threads)")
    comps = {"maxpool": {"value": round(mp_bytes / med / 1e9, 3), "unit": "GB/s",
                         "cores": threads, "kind": "port",
                         "sample": "torch restatement of the reference's Triton max-pool "
                                   "(the reference ships no torch version) on the whole cfg2 "
                                   f"input, median of {n} runs"}}

    ids, table = bt["topk_idx"].cpu(), bt["block_table"].cpu()
    tok, pos, slen = bt["token_to_bs"].cpu(), bt["token_pos_in_bs"].cpu(), bt["seqlen_q"].cpu()
    bt_bytes = workloads.block_table_bytes(ids, tok, 2, 4096, 64, 1)
    med, n = _median_time(lambda: get_block_table_torch(ids, table, tok, pos, slen), 5)
    log(f"cpu baseline: block table {med:.2f} s per cfg5 stage ({n} runs, {threads} threads)")
    comps["block_table"] = {"value": round(bt_bytes / med / 1e9, 3), "unit": "GB/s",
                            "cores": threads, "kind": "port",
                            "sample": "get_block_table_ref_torch's steps in torch (block_table[bs], "
                                      "gather, where) on the whole cfg5 block-table stage, "
                                      f"median of {n} runs"}
    line["components"] = comps
    return line


if __name__ == "__main__":
    main()
