"""Failure handling on the GPU, forced from the host with the FT_FAIL_SCRATCH
test hook (every device-scratch request fails as an allocation failure
would; no kernel faults or waits):
  - the paged decode raises (reference attention.cu:1839-1844: its launcher
    throws when the workspace cannot be allocated) and leaves nothing
    half-written; the library works again once memory is back;
  - the contiguous decode falls back (reference attention.cu:1514-1523 runs
    its single-pass kernel instead): here the split partials go to the
    static per-device array, and the result is the same bit for bit;
  - quantize_int8 above its one-launch size raises; below it needs no
    scratch and still runs."""

import numpy as np
import pytest
import torch

import fusedtok_amd as ft
import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"


def t(a, dtype=None):
    x = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    return x if dtype is None else x.to(dtype)


def paged(rng, b=3, hq=16, hkv=4, d=128, lens=(40, 700, 1), page=16):
    width = max((n + page - 1) // page for n in lens)
    nb = b * width + 2
    q = rng.standard_normal((b, hq, d)).astype(np.float32)
    kp = rng.standard_normal((nb, hkv, page, d)).astype(np.float32)
    vp = rng.standard_normal((nb, hkv, page, d)).astype(np.float32)
    tbl = rng.permutation(nb)[: b * width].reshape(b, width).astype(np.int32)
    return q, kp, vp, tbl, np.asarray(lens, np.int32)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_paged_decode_raises_and_recovers(dt, tuning):
    rng = np.random.default_rng(3)
    q, kp, vp, tbl, ln = paged(rng)
    args = (t(q, dt), t(kp, dt), t(vp, dt), t(tbl), t(ln))
    tuning("FT_FAIL_SCRATCH", 1)
    with pytest.raises(RuntimeError, match="out of memory"):
        ft.attention_decode_paged(*args)
    tuning.clear("FT_FAIL_SCRATCH")
    got = ft.attention_decode_paged(*args).float().cpu().numpy()
    r = lambda a: torch.from_numpy(a).to(dt).float().numpy()  # noqa: E731
    ref = oracle.attention_decode_paged(r(q), r(kp), r(vp), tbl, ln)
    np.testing.assert_allclose(got, ref, rtol=1e-2, atol=2e-3)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("generic", [False, True])
def test_contiguous_decode_falls_back_to_the_static_array(dt, generic, tuning):
    if generic:
        tuning("FT_ATTN_FORCE_GENERIC", 1)
    rng = np.random.default_rng(4)
    b, hq, hkv, tt, d = 2, 16, 4, 3000, 128
    q = t(rng.standard_normal((b, hq, d)).astype(np.float32), dt)
    k = t(rng.standard_normal((b, hkv, tt, d)).astype(np.float32), dt)
    v = t(rng.standard_normal((b, hkv, tt, d)).astype(np.float32), dt)
    lens = t(np.array([3000, 1777], np.int32))
    want = ft.attention_decode(q, k, v, lens)
    tuning("FT_FAIL_SCRATCH", 1)
    got = ft.attention_decode(q, k, v, lens)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_quantize_raises_above_one_launch_and_runs_below(tuning):
    big = torch.randn(1 << 20, device=DEV)
    small = torch.randn(1000, device=DEV)
    q_ref, s_ref = ft.quantize_int8(small)
    tuning("FT_FAIL_SCRATCH", 1)
    with pytest.raises(RuntimeError, match="out of memory"):
        ft.quantize_int8(big)
    q, s = ft.quantize_int8(small)
    assert torch.equal(q, q_ref) and s == s_ref
    tuning.clear("FT_FAIL_SCRATCH")
    _, s2 = ft.quantize_int8(big)
    assert s2 == float(np.float32(big.abs().max().item()) / np.float32(127.0))


def test_an_error_that_is_not_want_of_memory_is_reported(tuning):
    # FT_FAIL_SCRATCH=2: the scratch request fails with another HIP error (an
    # earlier kernel's fault shows so). The steps that answer want of memory
    # with another path must raise it, each of them.
    x = torch.randn(8, 4096, device=DEV)
    x100 = torch.randn(100, 4096, device=DEV)
    w = torch.ones(4096, device=DEV)
    rng = np.random.default_rng(5)
    q, kp, vp, tbl, ln = (t(a) for a in paged(rng, d=64))
    kn = torch.randn(3, 4, 64, device=DEV)
    a = torch.ones(150, 4096, dtype=torch.int8, device=DEV)
    b = torch.ones(1024, 4096, dtype=torch.int8, device=DEV)
    sb = torch.ones(1024, device=DEV)
    half = [y.half() for y in (q, kp, vp)]
    calls = dict(
        rmsnorm_one_launch=lambda: ft.rmsnorm_quant(x, w),
        rmsnorm_two_launches=lambda: ft.rmsnorm_quant(x100, w),
        swiglu=lambda: ft.swiglu_quant(x, x),
        sampling=lambda: ft.sample_topp_batched(torch.randn(2, 32768, device=DEV), 0.9,
                                                seeds=[1, 2]),
        gemm=lambda: ft.qgemm_perchannel(a, 0.1, b, sb),
        decode=lambda: ft.attention_decode_paged(q, kp, vp, tbl, ln),
        contiguous=lambda: ft.attention_decode(q, kp.view(-1, 4, 16, 64)[:3].contiguous(),
                                               vp.view(-1, 4, 16, 64)[:3].contiguous(),
                                               torch.full_like(ln, 9)),
        append=lambda: ft.attention_decode_paged_append(half[0], half[1], half[2], tbl,
                                                        kn.half(), kn.half(), ln))
    for name, call in calls.items():
        call()
        tuning("FT_FAIL_SCRATCH", 2)
        with pytest.raises(RuntimeError, match="a HIP error"):
            call()
            pytest.fail(f"{name} took another path")
        tuning.clear("FT_FAIL_SCRATCH")
        call()


@pytest.mark.parametrize("dt,d", [(torch.float32, 128), (torch.float16, 64), (torch.bfloat16, 128),
                                  (torch.bfloat16, 48)])
@pytest.mark.parametrize("fail", [1, 16 << 0, 16 << 6])
def test_append_decode_without_memory_leaves_the_pools(dt, d, fail, tuning):
    # every request fails; the decode's partials alone; lens + 1 alone (which
    # the one-call form does not need)
    rng = np.random.default_rng(6)
    q, kp, vp, tbl, ln = paged(rng, d=d)
    k1, v1 = t(kp, dt), t(vp, dt)
    kn, vn = (torch.randn(3, 4, d, device=DEV).to(dt) for _ in range(2))
    args = (t(q, dt), k1, v1, t(tbl), kn, vn, t(ln))
    k0, v0 = k1.clone(), v1.clone()
    one_call = dt is not torch.float32 and d in (64, 128)
    tuning("FT_FAIL_SCRATCH", fail)
    if fail == 16 << 6 and one_call:
        ft.attention_decode_paged_append(*args)
    else:
        with pytest.raises(RuntimeError, match="out of memory"):
            ft.attention_decode_paged_append(*args)
        assert torch.equal(k1, k0) and torch.equal(v1, v0)
    tuning.clear("FT_FAIL_SCRATCH")
    got = ft.attention_decode_paged_append(*args)
    ft.kv_append_paged(k0, v0, args[3], kn, vn, args[6])
    assert torch.equal(k1, k0) and torch.equal(v1, v0)
    ref = oracle.attention_decode_paged(args[0].float().cpu().numpy(), k0.float().cpu().numpy(),
                                        v0.float().cpu().numpy(), tbl, ln + 1)
    np.testing.assert_allclose(got.float().cpu().numpy(), ref, rtol=1e-2, atol=2e-3)


# room for the general kernel's partials of the cases below (under 150 KB) but
# not for the stream kernels' (256 or 512 segments more: over 270 KB)
ROOM = 200 << 10


@pytest.mark.parametrize("dt,d", [(torch.float32, 64), (torch.float32, 128), (torch.float16, 64),
                                  (torch.bfloat16, 64)])
def test_decode_with_room_for_the_general_kernel_alone(dt, d, tuning):
    # the stream kernels' workspace cannot be had, in an eager call or under a
    # capture: the general kernel's result bit for bit, and replays of it
    rng = np.random.default_rng(7)
    q, kp, vp, tbl, ln = paged(rng, hq=8, hkv=4, d=d, lens=(40, 400, 1))
    args = (t(q, dt), t(kp, dt), t(vp, dt), t(tbl), t(ln))
    stream = ft.attention_decode_paged(*args)
    tuning("FT_ATTN_FORCE_GENERIC", 1)
    want = ft.attention_decode_paged(*args)
    tuning.clear("FT_ATTN_FORCE_GENERIC")
    # so the two can be told apart (bf16's rounding can hide it)
    assert dt is torch.bfloat16 or not torch.equal(stream, want)
    tuning("FT_FAIL_SCRATCH", ROOM)
    assert torch.equal(ft.attention_decode_paged(*args), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ft.attention_decode_paged(*args)
    tuning.clear("FT_FAIL_SCRATCH")
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(ft.attention_decode_paged(*args), stream)  # eager work between


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_append_decode_with_room_for_the_general_kernel_alone(dt, tuning):
    # the appending form at D = 64 then is the append and the general decode
    rng = np.random.default_rng(8)
    q, kp, vp, tbl, ln = paged(rng, hq=8, hkv=4, d=64, lens=(40, 390, 1))
    kn, vn = (torch.randn(3, 4, 64, device=DEV).to(dt) for _ in range(2))
    qt, tt, lt = t(q, dt), t(tbl), t(ln)
    k1, v1, k2, v2 = t(kp, dt), t(vp, dt), t(kp, dt), t(vp, dt)
    ft.kv_append_paged(k2, v2, tt, kn, vn, lt)
    tuning("FT_ATTN_FORCE_GENERIC", 1)
    want = ft.attention_decode_paged(qt, k2, v2, tt, lt + 1)
    tuning.clear("FT_ATTN_FORCE_GENERIC")
    tuning("FT_FAIL_SCRATCH", ROOM)
    got = ft.attention_decode_paged_append(qt, k1, v1, tt, kn, vn, lt)
    assert torch.equal(got, want) and torch.equal(k1, k2) and torch.equal(v1, v2)
    k3, v3 = t(kp, dt), t(vp, dt)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ft.attention_decode_paged_append(qt, k3, v3, tt, kn, vn, lt)
    tuning.clear("FT_FAIL_SCRATCH")
    for _ in range(3):
        out.zero_()
        k3.copy_(t(kp, dt))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(k3, k2) and torch.equal(v3, v2)


def test_capture_without_warm_up_takes_the_paths_that_need_less(tuning):
    # sampling and a K-split GEMM captured where their workspace cannot be had
    # record one workgroup per row and no split: the same tokens and values
    logits = torch.randn(3, 40000, device=DEV)
    a = torch.randint(-127, 128, (150, 4096), dtype=torch.int8, device=DEV)
    b = torch.randint(-127, 128, (1024, 4096), dtype=torch.int8, device=DEV)
    sb = torch.rand(1024, device=DEV) * 0.01
    sa = torch.full((1,), 0.02, device=DEV)
    seeds = torch.tensor([1, 2, 3], device=DEV)

    def sample():
        out = torch.zeros(3, dtype=torch.int64, device=DEV)
        ft._fusedtok.sample_topp_batched_launch(
            logits.data_ptr(), 3, 40000, 0.9, 1.0, seeds.data_ptr(), out.data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        return out

    gemm = lambda: ft.qgemm_perchannel(a, sa, b, sb)  # noqa: E731
    want_t, want_y = sample(), gemm()
    assert want_t.tolist() == ft.sample_topp_batched(logits, 0.9, seeds=[1, 2, 3]).tolist()
    tuning("FT_FAIL_SCRATCH", 1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        toks, y = sample(), gemm()
    tuning.clear("FT_FAIL_SCRATCH")
    for _ in range(3):
        toks.zero_()
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(toks, want_t) and torch.equal(y, want_y)
        assert torch.equal(gemm(), want_y)  # eager work between
