"""CPU tests of bench.py's contract (no GPU needed):

* ``--gpus N`` with N > 1 exits with status 2 and says that one GPU is what
  this build measures; with no GPU visible the bench exits 1 (it never falls
  back to a CPU path);
* the algorithmic work it reports: valid slots exclude ``-1`` and count
  duplicates, F_alg = 4 h d N_valid, gathered bytes = 2 d N_valid, and the
  compulsory bytes count each (batch, row) once;
* every configuration has a measured traffic figure, and the track-02
  scenarios are the reference's (track-02/workloads.py:19-24).
"""
import os
import subprocess
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, REPO)

import bench  # noqa: E402
import sa_workloads as wl  # noqa: E402


def run_bench(*args):
    env = dict(os.environ, HIP_VISIBLE_DEVICES="", CUDA_VISIBLE_DEVICES="")
    return subprocess.run([sys.executable, os.path.join(REPO, "bench.py"), *args],
                          capture_output=True, text=True, env=env, timeout=300)


def test_more_than_one_gpu_is_refused():
    r = run_bench("--gpus", "2")
    assert r.returncode == 2
    assert "one GPU" in r.stderr


def test_no_gpu_exits_loudly():
    if torch.cuda.is_available():
        return  # only meaningful on a host without a GPU
    r = run_bench("--steps", "1", "--warmup", "0")
    assert r.returncode == 1
    assert "no GPU" in r.stderr
    assert r.stdout.strip() == ""


def test_algorithmic_work():
    idx = torch.tensor([[[3, 3, -1, 7], [-1, -1, -1, -1], [0, 7, 7, 7]]], dtype=torch.int32)
    b, m = 1, 3
    n_valid, flops, gathered, uniq, compulsory = bench.algorithmic(idx, b, m)
    assert n_valid == 7                      # duplicates count, -1 does not
    assert flops == 4.0 * 16 * 512 * 7
    assert gathered == 7 * 512 * 2
    assert uniq == 3                         # rows 0, 3, 7 of batch 0
    io = b * m * 16 * 512 * 2 * 2 + idx.numel() * 4 + 16 * 4
    assert compulsory == 3 * 512 * 2 + io


def test_tables():
    # traffic of every BASELINE config and every track-03 workload comes from
    # a committed profile summary that names the sources it measured
    for name in list(wl.CONFIGS) + [f"moe{i}" for i in range(len(bench.MOE_WORKLOADS))]:
        tr = bench.traffic_of(name)
        assert tr is not None and tr["bytes_per_launch"] > 0, name
        assert os.path.exists(os.path.join(bench.REPO, tr["profile"])), name
    assert len(bench.MOE_WORKLOADS) == 8
    shapes = {(d, p) for _, d, _, p, _ in bench.HC_WORKLOADS}
    assert shapes == {((1, 1), (1, 16384)), ((16, 1), (16, 4096)), ((64, 1), (64, 1024))}
    assert [n for n, *_ in bench.HC_WORKLOADS] == ["16k-1k-1", "4k-1k-16", "1k-1k-64", "1k-1-64"]


def test_source_digest_covers_kernel_sources(tmp_path, monkeypatch):
    """The digest that stamps the profiles changes with any kernel source,
    header or build flag, and with nothing else."""
    import shutil
    for rel in ("include", os.path.join("kernelgen-challenge_amd", "csrc")):
        shutil.copytree(os.path.join(REPO, rel), tmp_path / rel)
    shutil.copy(os.path.join(REPO, "kernelgen-challenge_amd", "build.py"),
                tmp_path / "kernelgen-challenge_amd" / "build.py")
    monkeypatch.setattr(bench, "REPO", str(tmp_path))
    d0 = bench.source_digest()
    assert d0 == bench.source_digest() and len(d0) == 16
    (tmp_path / "README.md").write_text("not a source")
    assert bench.source_digest() == d0
    hip = tmp_path / "kernelgen-challenge_amd" / "csrc" / "sparse_attn_gfx950.hip"
    hip.write_text(hip.read_text() + "\n")
    d1 = bench.source_digest()
    assert d1 != d0
    hdr = tmp_path / "include" / "sparse_attn.h"
    hdr.write_text(hdr.read_text() + " ")
    assert bench.source_digest() not in (d0, d1)


def test_roofline_record_checks_provenance(monkeypatch):
    """frac comes from the live kernel time; the committed profile is quoted
    beside it with its own frac; a traffic figure from other sources is
    dropped with the reason; a kernel time more than 1 % above the call
    time voids frac (less is the spread of two loops timing a one-kernel
    call, noted beside it)."""
    flops = 4.0 * 16 * 512 * 1000
    monkeypatch.setattr(bench, "traffic_of", lambda name: {
        "bytes_per_launch": 123, "sources": "0" * 16, "profile": "p.txt"})
    monkeypatch.setattr(bench, "_profile_rec", lambda path, name: {
        "kernel": "sa_fwd_tile_kernel", "avg_us": 100.0, "calls": 10, "profile": "t.txt",
        "sources": bench.source_digest()})
    r = bench.roofline("causal_prefill", flops, 1.0, {"tile": 0.1, "index": 0.02},
                       {"tile": 1.0}, 130.0)
    assert r["bound"] == "mfma" and r["kernel"] == "sa_fwd_tile_kernel"
    assert abs(r["frac"] - flops / 100e-6 / 1e12 / 2500.0) < 1e-4
    assert r["traffic"] is None and "traffic.json" in r["traffic_note"]
    assert r["profile"]["sources_match"] and r["profile"]["kernel_us"] == 100.0
    assert abs(r["profile"]["live_over_profile"] - 1.0) < 1e-9
    r = bench.roofline("causal_prefill", flops, 1.0, {"tile": 0.2}, {"tile": 1.0}, 150.0)
    assert r["frac"] is None and "exceeds" in r["frac_note"]
    # a one-kernel call whose kernel reads 0.5 % above it (separate loops)
    r = bench.roofline("causal_prefill", flops, 1.0, {"tile": 0.1005}, {"tile": 1.0}, 100.0)
    assert r["frac"] is not None and "above" in r["frac_note"]


def test_gemm_ceiling_shapes_follow_the_moe_workload():
    # the batched library GEMMs are fused_moe's per-expert products at its
    # largest prefill workload: E experts of M * topk / E pairs each
    label, M, K, N, E, topk = bench.MOE_WORKLOADS[7]
    assert (label, M, E, topk) == ("prefill", 4096, 64, 6)
    shapes = {lab: (bt, m, k, n) for lab, bt, m, k, n in bench.GEMM_CEILING_SHAPES}
    assert shapes["moe gate-up per expert"] == (E, M * topk // E, K, 2 * N)
    assert shapes["moe down per expert"] == (E, M * topk // E, N, K)


def test_torch_eager_baseline_is_the_reference_oracle():
    # the contest bench's denominator (the reference's own metric) computes
    # what the oracle computes, in the same order: on CPU tensors the two
    # agree bit for bit
    from oracle.sparse_attn_ref import sparse_attn_ref
    g = torch.Generator().manual_seed(3)
    b, m, h, d, kv_len, topk = 2, 3, 16, 512, 40, 7
    q = torch.randn(b, m, h, d, generator=g).to(torch.bfloat16)
    kv = torch.randn(b, kv_len, d, generator=g).to(torch.bfloat16)
    sink = torch.randn(h, generator=g)
    idx = torch.randint(0, kv_len, (b, m, topk), generator=g, dtype=torch.int32)
    got = bench.torch_eager_attn(q, kv, sink, idx, 0.044)
    want = sparse_attn_ref(q, kv, sink, idx, 0.044)
    assert got.dtype == torch.bfloat16 and got.shape == (b, m, h, d)
    assert torch.equal(got, want)


def test_torch_eager_baseline_masks_padding_like_the_oracle():
    # with -1 slots (causal prefill's padding) the baseline masks them as the
    # oracle does; an all -1 query gives o = 0
    from oracle.sparse_attn_ref import sparse_attn_ref
    g = torch.Generator().manual_seed(4)
    b, m, h, d, kv_len, topk = 1, 4, 16, 512, 30, 9
    q = torch.randn(b, m, h, d, generator=g).to(torch.bfloat16)
    kv = torch.randn(b, kv_len, d, generator=g).to(torch.bfloat16)
    sink = torch.randn(h, generator=g)
    idx = torch.randint(0, kv_len, (b, m, topk), generator=g, dtype=torch.int32)
    idx[0, 1, 5:] = -1
    idx[0, 3, :] = -1
    got = bench.torch_eager_attn(q, kv, sink, idx, 0.044, masked=True)
    want = sparse_attn_ref(q, kv, sink, idx, 0.044)
    assert torch.equal(got, want)
    assert not bool(got[0, 3].any())


def test_torch_eager_moe_is_the_track03_oracle():
    # the MoE denominator runs the oracle's dense form (every expert over every
    # token, weight 0 where not routed); on CPU tensors it matches oracle/,
    # which runs the routed tokens only, bit for bit
    from oracle.fused_moe_ref import fused_moe_ref
    g = torch.Generator().manual_seed(5)
    M, K, N, E, topk = 12, 256, 128, 4, 2
    hidden = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w1 = (torch.randn(E, 2 * N, K, generator=g) * 0.02).to(torch.bfloat16)
    w2 = (torch.randn(E, K, N, generator=g) * 0.02).to(torch.bfloat16)
    score = torch.randn(M, E, generator=g).to(torch.bfloat16)
    for renorm in (False, True):
        got = bench.torch_eager_moe(hidden, w1, w2, score, topk, renorm)
        want = fused_moe_ref(hidden, w1, w2, score, topk, renorm)
        assert got.dtype == torch.bfloat16 and got.shape == (M, K)
        assert torch.equal(got, want)


def test_torch_eager_sinkhorn_is_the_track02_oracle():
    from oracle.hc_sinkhorn_ref import hc_split_sinkhorn_np
    g = torch.Generator().manual_seed(6)
    mixes = torch.randn(3, 5, 24, generator=g)
    sc, bs = torch.randn(3, generator=g), torch.randn(24, generator=g)
    got = bench.torch_eager_sinkhorn(mixes, sc, bs)
    want = hc_split_sinkhorn_np(mixes.numpy(), sc.numpy(), bs.numpy())
    for a, b in zip(got, want):
        assert tuple(a.shape) == b.shape
        assert torch.allclose(a, torch.from_numpy(b), rtol=1e-5, atol=1e-6)


def test_kernel_names_follow_the_launch_plans():
    """bench.py restates which kernel a shape launches; the host-side planners
    (256 CUs) say the same."""
    import ctypes

    import sa_capi
    from sa_testutil import host_lib, moe_plan
    shapes = [w[1:] for w in bench.MOE_WORKLOADS]
    shapes += [(M, 2048, N, E, topk) for M in (1, 7, 30, 64, 100, 200, 700, 3000)
               for N in (512, 1024, 1408) for E, topk in ((8, 2), (16, 4), (64, 6), (128, 8))]
    for M, K, N, E, topk in shapes:
        p = moe_plan(M, K, N, E, topk)
        name = bench.moe_gemm_kernel(M, N, E, topk, True)
        want = "fm_gemm_kernel<true>" if p["gemm"] else \
            f"fm_{'stream' if N % 256 == 0 else 'skinny'}_kernel<true, {p['pb']}>"
        assert name == want, (M, K, N, E, topk)
    for name, c in wl.CONFIGS.items():
        a = sa_capi.SaArgs()
        a.q = a.kv = a.sink = a.idx = a.o = 0x10000
        a.b, a.m, a.h, a.d, a.kv_len, a.topk = c.b, c.m, 16, 512, c.kv_len, c.topk
        a.sq[:] = a.so[:] = (c.m * 16 * 512, 16 * 512, 512, 1)
        a.skv[:] = (c.kv_len * 512, 512, 1)
        a.sidx[:] = (c.m * c.topk, c.topk, 1)
        a.scale = wl.SCALE
        out = (ctypes.c_int64 * 12)()
        assert host_lib().sa_host_plan_full(ctypes.byref(a), 256, out) == sa_capi.SA_OK
        waves = out[0] == 1 and not out[2] and 384 < c.topk <= 2048 and c.kv_len > 16384
        assert (bench.kernel_names(name)["query"] == "sa_fwd_waves_kernel") == waves, name
