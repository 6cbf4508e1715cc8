"""GPU parity of the track-03 ``fused_moe`` HIP path against the CPU oracle.

Inputs follow the reference's own test (track-03/test_correctness.py:15-21:
bf16 ``randn`` on the device from a seeded generator, weights scaled by
0.02) on the eight workloads of track-03/workloads.py:3-12. Bars, against
``oracle.fused_moe_ref`` (torch CPU, the reference's op order and bf16
rounding points, lower-index tie rule) on every token:

* the reference's own: ``assert_close(atol=5e-2, rtol=5e-2)``
  (track-03/test_correctness.py:35);
* an internal gate: relative RMS error <= 5e-3, and no element further than
  2^-5 of the output's largest magnitude (the two sides differ only in the
  order of the fp32 sums inside the GEMMs, which moves a bf16 rounding by one
  step now and then).

The exact-rounding NumPy model ``fused_moe_fp64`` is checked on a sample of
tokens. Edge cases: renormalisation, exact ties in the router scores (the
lower expert index wins), every token on one expert, topk = E, E = 1, M = 0
and 1, strided inputs, both tile kinds forced, the C-ABI and its event hook.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

import sa_capi
from oracle.fused_moe_ref import fused_moe_fp64, fused_moe_ref
from sa_testutil import moe_plan

pytestmark = pytest.mark.gpu

DEV = "cuda"
REL_RMS = 5e-3
MAX_FRAC = 2 ** -5

# track-03/workloads.py:3-12: (label, M, K, N, E, topk)
WORKLOADS = [("decode", 1, 2048, 1024, 8, 2), ("decode", 64, 2048, 1024, 8, 2),
             ("decode", 1, 2048, 1024, 64, 6), ("decode", 64, 2048, 1024, 64, 6),
             ("prefill", 512, 2048, 1024, 8, 2), ("prefill", 4096, 2048, 1024, 8, 2),
             ("prefill", 512, 2048, 1024, 64, 6), ("prefill", 4096, 2048, 1024, 64, 6)]


def say(*a):
    print(*a, flush=True)


def make_inputs(M, K, N, E, seed=0):
    """track-03/test_correctness.py:15-21, on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    hidden = torch.randn(M, K, dtype=torch.bfloat16, generator=g, device=DEV)
    w1 = torch.randn(E, 2 * N, K, dtype=torch.bfloat16, generator=g, device=DEV) * 0.02
    w2 = torch.randn(E, K, N, dtype=torch.bfloat16, generator=g, device=DEV) * 0.02
    score = torch.randn(M, E, dtype=torch.bfloat16, generator=g, device=DEV)
    return hidden, w1, w2, score


def cpu(*ts):
    return [t.cpu() for t in ts]


def check(out, ref, label):
    """out: GPU bf16 [M, K]; ref: CPU bf16 oracle output."""
    o = out.cpu()
    assert o.shape == ref.shape and o.dtype == torch.bfloat16
    torch.testing.assert_close(o, ref, atol=5e-2, rtol=5e-2)
    d = (o.double() - ref.double()).abs()
    scale = ref.double().abs().max().item() or 1.0
    rms = math.sqrt(float((ref.double() ** 2).mean())) or 1.0
    rel = math.sqrt(float((d ** 2).mean())) / rms
    frac = float((d > 0).double().mean())
    say(f"  {label}: max|d|={d.max().item():.3e} (of max {scale:.3e}) rel_rms={rel:.3e} "
        f"differing={frac:.4f}")
    assert rel <= REL_RMS, label
    assert d.max().item() <= MAX_FRAC * scale, label


def op(*a, **k):
    import submission
    return submission.fused_moe(*a, **k)


@pytest.mark.parametrize("w", WORKLOADS, ids=lambda w: f"{w[0]}_M{w[1]}_E{w[4]}_topk{w[5]}")
def test_workload_against_oracle(gpu_sa, w):
    _, M, K, N, E, topk = w
    say(f"fused_moe M={M} K={K} N={N} E={E} topk={topk}")
    hidden, w1, w2, score = make_inputs(M, K, N, E)
    out = op(hidden, w1, w2, score, topk)
    torch.cuda.synchronize()
    hc, w1c, w2c, sc = cpu(hidden, w1, w2, score)
    check(out, fused_moe_ref(hc, w1c, w2c, sc, topk), "vs torch oracle")
    # the exact-rounding model on a sample of tokens
    sel = torch.randperm(M, generator=torch.Generator().manual_seed(M))[:min(M, 48)]
    exp = fused_moe_fp64(hc[sel], w1c, w2c, sc[sel], topk)
    d = np.abs(out.cpu()[sel].double().numpy() - exp)
    say(f"  vs exact-rounding model ({len(sel)} tokens): max|d|={d.max():.3e}")
    assert d.max() <= MAX_FRAC * np.abs(exp).max()


@pytest.mark.parametrize("shape", [(64, 2048, 1024, 8, 2), (300, 512, 256, 64, 6)])
def test_renormalize(gpu_sa, shape):
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=3)
    out = op(hidden, w1, w2, score, topk, renormalize=True)
    hc, w1c, w2c, sc = cpu(hidden, w1, w2, score)
    ref = fused_moe_ref(hc, w1c, w2c, sc, topk, renormalize=True)
    check(out, ref, "renormalize")
    plain = fused_moe_ref(hc, w1c, w2c, sc, topk)
    assert (ref.double() - plain.double()).abs().max() > 1e-2  # the flag matters here


@pytest.mark.parametrize("flags", [1, 2, 4], ids=["large", "small", "big"])
@pytest.mark.parametrize("shape", [(64, 2048, 1024, 8, 2), (512, 1024, 512, 64, 6),
                                   (200, 256, 128, 4, 2), (300, 1280, 384, 4, 3)])
def test_forced_tiles(gpu_sa, shape, flags):
    """Every GEMM kernel on the same inputs, whichever the library would pick
    (the last shape: odd column-tile counts, 3 for gate-up and 5 for down, so
    the two column halves of the XCD work split differ in size)."""
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=4)
    out = op(hidden, w1, w2, score, topk, flags=flags)
    check(out, fused_moe_ref(*cpu(hidden, w1, w2, score), topk), f"flags={flags}")


def test_router_ties_go_to_lower_index(gpu_sa):
    """Integer router scores: exact ties everywhere, also across the top-k
    boundary; the selection must follow the lower-index rule of the oracle."""
    M, K, N, E, topk = 256, 512, 256, 64, 6
    hidden, w1, w2, _ = make_inputs(M, K, N, E, seed=5)
    g = torch.Generator().manual_seed(6)
    score = torch.randint(-2, 3, (M, E), generator=g).to(torch.bfloat16)
    out = op(hidden, w1, w2, score.to(DEV), topk)
    check(out, fused_moe_ref(*cpu(hidden, w1, w2), score, topk), "ties")


def test_every_token_on_one_expert(gpu_sa):
    """Expert 3 first for every token: many tiles of one expert (both kinds)."""
    M, K, N, E, topk = 1000, 512, 256, 8, 2
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=7)
    score[:, 3] = 8.0
    ref = fused_moe_ref(*cpu(hidden, w1, w2, score), topk)
    for flags in (0, 1, 2, 4):
        check(op(hidden, w1, w2, score, topk, flags=flags), ref, f"one expert, flags={flags}")


@pytest.mark.parametrize("shape", [(1500, 512, 256, 8, 2), (700, 1024, 512, 4, 3),
                                   (2048, 2048, 1024, 8, 2), (700, 1280, 384, 4, 3)])
def test_big_tiles_equal_large_tiles(gpu_sa, shape):
    """256-pair and 128-pair tiles run the same MFMA sequence per output element,
    so they agree bit for bit, with full and ragged tiles, row blocks past the
    last pair and wave halves without any."""
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=9)
    big = op(hidden, w1, w2, score, topk, flags=4)
    large = op(hidden, w1, w2, score, topk, flags=1)
    assert torch.equal(big, large)


@pytest.mark.parametrize("narrow,counts,K,N", [
    (256, (1, 32, 33, 64), 256, 128), (256, (65, 128, 129, 0, 255, 256), 256, 128),
    (256, (256, 257, 384, 385, 512, 640), 512, 128),
    (0, (300,) * 20 + (100,) * 44, 256, 2048), (0, (17, 200, 256, 31) * 8, 512, 640),
    (128, (1025, 1056, 1057, 1088, 1152, 1153, 1024, 897), 256, 1024),
    (128, (1025, 1056, 1057, 1281, 1152, 1409, 1024, 0), 256, 1024)])
def test_gemm_tiles_at_their_edges(gpu_sa, narrow, counts, K, N):
    """Wide and narrow tiles of every filling (row blocks of one or both wave
    halves, DMA groups partly past the last pair, every tile narrow, every tile
    wide, and wide tiles with the short last ones of an expert narrow: 1 to 128
    pairs, 129 wide, none after a multiple of 256, an empty expert), as chosen
    and with 256- and 128-pair tiles: the same MFMA sequence per output element,
    so the same bits; and the oracle."""
    E, M = len(counts), sum(counts)
    p = moe_plan(M, K, N, E, 1)
    assert p["gemm"] and p["tile_rows"] == 256 and p["narrow_rows"] == narrow
    hidden, w1, w2, _ = make_inputs(M, K, N, E, seed=11)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(M, generator=torch.Generator().manual_seed(12))].to(DEV)
    score = torch.nn.functional.one_hot(ids, E).to(torch.bfloat16) * 4
    out = op(hidden, w1, w2, score, 1)
    assert torch.equal(out, op(hidden, w1, w2, score, 1, flags=4))
    assert torch.equal(out, op(hidden, w1, w2, score, 1, flags=1))
    check(out, fused_moe_ref(*cpu(hidden, w1, w2, score), 1), f"{counts[:6]}")


@pytest.mark.parametrize("shape", [(16, 256, 128, 256, 32), (17, 256, 128, 65, 3),
                                   (100, 256, 128, 256, 32), (4097, 256, 128, 9, 2),
                                   (50, 256, 128, 1, 1)])
def test_routing_over_work_groups(gpu_sa, shape):
    """Routing and plan in one work-group and over several, the last one ragged
    and with 16 or 32 tokens each, one and four experts per lane; half the
    rows have integer scores (ties)."""
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=14)
    score[::2] = score[::2].round()
    check(op(hidden, w1, w2, score, topk), fused_moe_ref(*cpu(hidden, w1, w2, score), topk),
          f"{shape}")


def test_gemm_silu_over_its_range(gpu_sa):
    """Gate values over about +-100: both tails of silu, where the exponential
    overflows or vanishes, against the oracle's exact one."""
    M, K, N, E, topk = 300, 512, 256, 4, 2
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=15)
    w1, w2 = w1 * 56, w2 * 1e-3
    gate = hidden.float() @ w1[0, :N].float().t()
    assert gate.min() < -90 and gate.max() > 90
    out = op(hidden, w1, w2, score, topk)
    check(out, fused_moe_ref(*cpu(hidden, w1, w2, score), topk), "wide gate range")


@pytest.mark.parametrize("flags", [0, 1, 4], ids=["narrow", "large", "big"])
def test_gemm_silu_of_every_bf16_gate(gpu_sa, flags):
    """Token t of expert 0 has gate value w1[j, t] at feature j, up value 1 and
    w2 = 1, so the output is silu of all finite bf16 values: fm_gemm_kernel's
    has the bits of the streamed kernel's, and lies within half a bf16 step
    (2^-8 of the value at most) and 4 float32 ulp of float64's wherever 1 +
    exp(-x) and the result are normal float32 numbers (below -88.7 the
    exponential overflows: 0)."""
    n = 256
    x = torch.arange(n * n, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(n, n)
    x = torch.where(x.isfinite(), x, torch.zeros_like(x))
    w1 = torch.cat([x, torch.ones_like(x)])[None].to(DEV)
    eye = torch.eye(n, dtype=torch.bfloat16, device=DEV)
    score = torch.zeros(n, 1, dtype=torch.bfloat16, device=DEV)
    p = moe_plan(n, n, n, 1, 1, flags)
    assert (p["gemm"], p["tile_rows"], p["narrow_rows"]) == \
        (1, *{0: (256, 256), 1: (128, 0), 4: (256, 0)}[flags])
    got = op(eye, w1, eye[None].contiguous(), score, 1, flags=flags)
    streamed = op(eye, w1, eye[None].contiguous(), score, 1, flags=2 | 8)
    bad = torch.nonzero(got.t().cpu().view(torch.int16) != streamed.t().cpu().view(torch.int16))
    say("  differing gates:", [(x[i, j].item(), got[j, i].item(), streamed[j, i].item())
                               for i, j in bad.tolist()[:8]])
    assert len(bad) == 0
    xd, y = x.double(), got.t().cpu().double()
    exact = xd / (1 + torch.exp(-xd))
    normal = (xd > -88.7) & (xd.abs() > 2.0 ** -120)
    assert ((y - exact).abs() <= (2 ** -8 + 2 ** -21) * exact.abs())[normal].all()
    assert (y[xd < -88.7].abs() <= 1e-36).all()


@pytest.mark.parametrize("M", [16, 64])
def test_streamed_final_sum_forms(gpu_sa, M):
    """Streamed tiles where fm_gemm_kernel is the default: the atomic and the
    ordered final sum give the same bits."""
    hidden, w1, w2, score = make_inputs(M, 2048, 1024, 8, seed=13)
    out = op(hidden, w1, w2, score, 2, flags=2)
    assert torch.equal(out, op(hidden, w1, w2, score, 2, flags=2 | 8))
    check(out, fused_moe_ref(*cpu(hidden, w1, w2, score), 2), f"streamed M={M}")


@pytest.mark.parametrize("shape", [(37, 256, 128, 4, 4), (5, 256, 128, 1, 1), (1, 256, 128, 256, 32),
                                   (3, 512, 128, 200, 7)])
def test_small_and_extreme_shapes(gpu_sa, shape):
    """topk = E, E = 1, the largest E and topk, ragged E."""
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=8)
    out = op(hidden, w1, w2, score, topk)
    check(out, fused_moe_ref(*cpu(hidden, w1, w2, score), topk), f"{shape}")


def test_empty_and_single_token(gpu_sa):
    hidden, w1, w2, score = make_inputs(0, 256, 128, 8)
    out = op(hidden, w1, w2, score, 2)
    assert out.shape == (0, 256)
    hidden, w1, w2, score = make_inputs(1, 256, 128, 8)
    check(op(hidden, w1, w2, score, 2), fused_moe_ref(*cpu(hidden, w1, w2, score), 2), "M=1")


def test_strided_inputs_and_determinism(gpu_sa):
    M, K, N, E, topk = 96, 512, 256, 16, 4
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=9)
    ref = op(hidden, w1, w2, score, topk)
    assert torch.equal(op(hidden, w1, w2, score, topk), ref)
    ht = hidden.t().contiguous().t()                       # column-major view
    w1t = w1.transpose(1, 2).contiguous().transpose(1, 2)
    st = torch.cat([score, score], dim=1)[:, :E]           # row stride 2E
    assert not (ht.is_contiguous() or w1t.is_contiguous() or st.is_contiguous())
    assert torch.equal(op(ht, w1t, w2, st, topk), ref)


def test_bad_inputs_raise(gpu_sa):
    hidden, w1, w2, score = make_inputs(4, 256, 128, 8)
    with pytest.raises(TypeError):
        op(hidden.float(), w1, w2, score, 2)
    with pytest.raises(ValueError):
        op(hidden.cpu(), w1, w2, score, 2)
    with pytest.raises(AssertionError):
        op(hidden, w1[:, :100], w2, score, 2)
    with pytest.raises(ValueError):  # K % 256 != 0
        h2, a1, a2, s2 = make_inputs(4, 200, 128, 8)
        op(h2, a1, a2, s2, 2)
    with pytest.raises(ValueError):  # topk > E
        op(hidden, w1, w2, score, 9)


@pytest.mark.parametrize("shape,flags", [((64, 2048, 1024, 8, 2), 0),
                                         ((600, 512, 256, 8, 2), 0),
                                         ((5, 512, 256, 64, 6), 0)])
def test_capi_matches_operator_and_times_kernels(gpu_sa, shape, flags):
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=10)
    ref = op(hidden, w1, w2, score, topk, flags=flags)
    lib = sa_capi.fm_load()
    assert lib.fm_abi_version() == 4
    out = torch.full_like(hidden, float("nan"))
    a = sa_capi.fm_make_args(hidden, w1, w2, score, out, topk, flags=flags)
    n = sa_capi.fm_workspace_bytes(lib, a)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    stream = torch.cuda.current_stream()
    evs = [torch.cuda.Event(enable_timing=True) for _ in range(2 * sa_capi.FM_KERNEL_COUNT)]
    for ev in evs:  # torch reads elapsed times only of events it has recorded once
        ev.record(stream)
    torch.cuda.synchronize()
    mask = sa_capi.fm_forward_events(lib, a, stream.cuda_stream, evs)
    torch.cuda.synchronize()
    every = (1 << sa_capi.FM_KERNEL_COUNT) - 1
    # up to 16 tokens, routing and plan are one launch (reported as the plan);
    # with topk <= 2 and streamed tiles (at most 24 pairs per expert) the down
    # GEMM adds into the output and there is no final-sum launch
    route = 1 << sa_capi.FM_KERNELS.index("route")
    reduce = 1 << sa_capi.FM_KERNELS.index("reduce")
    expect = every & ~route if M <= 16 else every
    if topk <= 2 and M * topk / E <= 24 and N % 256 == 0:
        expect &= ~reduce
    assert mask == expect
    assert torch.equal(out, ref)
    for k in range(sa_capi.FM_KERNEL_COUNT):
        if (mask >> k) & 1:
            assert evs[2 * k].elapsed_time(evs[2 * k + 1]) > 0.0
    # a workspace one byte short is refused before any device work
    a.workspace_bytes = n - 1
    out.fill_(float("nan"))
    rc = lib.fm_forward(ctypes.byref(a), ctypes.c_void_p(stream.cuda_stream))
    torch.cuda.synchronize()
    assert rc == sa_capi.FM_EWORKSPACE and torch.isnan(out).all()


def _capi_run(hidden, w1, w2, score, topk, flags):
    """fm_forward_events through the C-ABI: (output, launched-kernel mask)."""
    lib = sa_capi.fm_load()
    out = torch.full_like(hidden, float("nan"))
    a = sa_capi.fm_make_args(hidden, w1, w2, score, out, topk, flags=flags)
    n = sa_capi.fm_workspace_bytes(lib, a)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    stream = torch.cuda.current_stream()
    mask = sa_capi.fm_forward_events(lib, a, stream.cuda_stream,
                                     [None] * (2 * sa_capi.FM_KERNEL_COUNT))
    torch.cuda.synchronize()
    return out, mask


@pytest.mark.parametrize("shape", [(1, 2048, 1024, 8, 2), (64, 2048, 1024, 8, 2),
                                   (64, 2048, 1024, 8, 1), (1, 2048, 1024, 8, 1),
                                   (16, 512, 256, 8, 2)])
@pytest.mark.parametrize("scale", ["normal", "subnormal"])
def test_atomic_final_sum_equals_ordered_sum(shape, scale):
    """With topk <= 2 and streamed tiles the down GEMM adds its bf16 products
    into the output with packed bf16 atomics; FM_FLAG_ORDERED_SUM forces the
    separate ascending-expert running sum instead. The two must agree bit for
    bit: a two-term bf16 sum rounds the same exact value either way if the
    atomic rounds to nearest even and keeps subnormals. Random bf16 addends
    tie at the rounding point often (two values one binade apart leave one
    extra bit, a tie half the time it is set), and the "subnormal" inputs put
    the addends around the smallest normal bf16 (2^-126): hidden scaled by
    2^-62 gives intermediate values near 2^-125 and outputs near 2^-127."""
    M, K, N, E, topk = shape
    hidden, w1, w2, score = make_inputs(M, K, N, E, seed=21)
    if scale == "subnormal":
        hidden = hidden * 2.0 ** -62
    say(f"fused_moe atomic vs ordered sum M={M} K={K} N={N} E={E} topk={topk} {scale}")
    out_a, mask_a = _capi_run(hidden, w1, w2, score, topk, 0)
    out_o, mask_o = _capi_run(hidden, w1, w2, score, topk, sa_capi.FM_FLAG_ORDERED_SUM)
    reduce = 1 << sa_capi.FM_KERNELS.index("reduce")
    assert mask_a & reduce == 0, "the default path should add atomically here"
    assert mask_o & reduce, "FM_FLAG_ORDERED_SUM must launch the final sum"
    assert torch.equal(out_a.view(torch.int16), out_o.view(torch.int16))
    if scale == "subnormal":
        tiny = out_o.float().abs()
        sub = ((tiny > 0) & (tiny < 2.0 ** -126)).sum().item()
        assert sub > 0, "no subnormal outputs: the case does not test them"
    # and both agree with the drop-in (operator path, default flags)
    assert torch.equal(op(hidden, w1, w2, score, topk).view(torch.int16),
                       out_a.view(torch.int16))
