"""Head dims of whole 16-byte chunks that do not fill a padded tile (D % 8 == 0,
D not 64/128/256): their vector paths against the CPU oracle and against the
element-wise path, which the same values take from a base that is not 16-byte
aligned.  The columns past D add exact zeros in both, so results differ by the
last fp16 rounding at most (one path may fuse the final scaling with the
conversion, a single rounding in place of two), NaN and infinities alike."""
import pytest
import torch

from oracle import attention as A
from tests.helpers import assert_close, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gen(seed):
    return torch.Generator().manual_seed(seed)


def misaligned(t):
    """The same contiguous values at an address 2 bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)
    view = buf[1:1 + t.numel()].view(t.shape)
    view.copy_(t)
    assert view.data_ptr() % 16 != 0 and view.is_contiguous()
    return view


def equal(a, b):
    """Same NaN and infinities, and finite values within one fp16 ulp (2^-10 of
    the value, 2^-24 where it is subnormal)."""
    a, b = a.float(), b.float()
    finite = torch.isfinite(a)
    if not (torch.equal(finite, torch.isfinite(b)) and torch.equal(torch.isnan(a), torch.isnan(b))):
        return False
    if not torch.equal(a[torch.isinf(a)], b[torch.isinf(b)]):
        return False
    a, b = a[finite], b[finite]
    return bool(((a - b).abs() <= 2.0 ** -10 * torch.maximum(a.abs(), b.abs()) + 2.0 ** -24).all())


DIMS = [8, 24, 32, 40, 72, 80, 88, 96, 104, 120, 160, 192, 200, 248]


@pytest.mark.parametrize("d", DIMS)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 2, 1, 45),      # key-split workgroups up to D = 128
                                        (3, 20, 4, 161),    # one round of query tiles
                                        (2, 16, 16, 577)])
def test_prefill_chunk_rows(fa, d, causal, b, hq, hkv, n):
    g = gen(d * 1000 + n)
    q, k, v = randn(g, b, hq, n, d), randn(g, b, hkv, n, d), randn(g, b, hkv, n, d)
    qc, kc, vc = (t.to(DEV) for t in (q, k, v))
    out = fa.forward_prefill_gqa_fp16(qc, kc, vc, causal)
    assert equal(out, fa.forward_prefill_gqa_fp16(misaligned(qc), kc, vc, causal))
    if n < 300:
        assert_close(out, A.prefill(q, k, v, causal), what=f"prefill D={d}")


@pytest.mark.parametrize("d", [40, 72, 80, 96, 200])
def test_prefill_chunk_rows_many_blocks(fa, d):
    """More query tiles than one residency round (32-key tiles at D <= 64)."""
    g = gen(d)
    qc, kc, vc = (randn(g, 8, 32, 600, d).to(DEV) for _ in range(3))
    assert equal(fa.forward_fp16(qc, kc, vc, True), fa.forward_fp16(misaligned(qc), kc, vc, True))


@pytest.mark.parametrize("d", [24, 72, 80, 88, 160])
def test_prefill_chunk_rows_special_values(fa, d):
    """Infinities and NaN reach the same outputs whatever LDS held past D."""
    g = gen(d + 5)
    q, k, v = (randn(g, 2, 8, 200, d).to(DEV) for _ in range(3))
    k[0, 1, 50, d - 1] = float("-inf")
    k[1, 2, 60, 3] = float("inf")
    v[0, 3, 70, 0] = float("inf")
    v[1, 4, 80, d - 2] = float("nan")
    q[0, 5, 90, 1] = float("nan")
    junk = torch.full((64 << 20,), float("nan"), dtype=torch.float16, device=DEV)  # LDS and memory hold NaN before
    fa.forward_fp16(junk[:2 * 8 * 200 * 128].view(2, 8, 200, 128), junk[:2 * 8 * 200 * 128].view(2, 8, 200, 128),
                    junk[:2 * 8 * 200 * 128].view(2, 8, 200, 128), False)
    for causal in (True, False):
        out = fa.forward_fp16(q, k, v, causal)
        assert equal(out, fa.forward_fp16(misaligned(q), k, v, causal))
        assert not torch.isnan(out[0, 0]).any()


@pytest.mark.parametrize("d", [64, 80, 128, 256])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,h,n", [(1, 32, 260), (3, 24, 129), (1, 70, 33), (2, 40, 321), (1, 40, 1057)])
def test_prefill_two_wave_blocks(fa, d, causal, b, h, n):
    """Launches whose query blocks are shared by two waves (65 to 256 blocks of 128
    rows, or 512 of causal walks past 1024 keys) at the edges of their 64-row and 64-key tiles."""
    g = gen(d + n)
    q, k, v = (randn(g, b, h, n, d) for _ in range(3))
    out = fa.forward_fp16(*(t.to(DEV) for t in (q, k, v)), causal)
    assert_close(out, A.prefill(q, k, v, causal), what=f"two-wave blocks {b, h, n, d}")
    if d <= 128:
        out2, lse = fa.forward_fp16_with_lse(*(t.to(DEV) for t in (q, k, v)), causal)
        assert torch.equal(out, out2)
        assert_close(lse, A.prefill_lse(q, k, v, causal)[1], atol=2e-3, rtol=0, what="lse")


@pytest.mark.parametrize("d", [8, 32, 72, 80, 96, 112, 192, 200])
@pytest.mark.parametrize("causal", [True, False])
def test_varlen_chunk_rows(fa, d, causal):
    lens = [5, 0, 200, 37, 1, 129]
    g = gen(d + 17)
    cu = torch.tensor([0] + torch.cumsum(torch.tensor(lens), 0).tolist(), dtype=torch.int32)
    tot = int(cu[-1])
    q, k, v = (randn(g, tot, 3, d) for _ in range(3))
    qc, kc, vc, cuc = (t.to(DEV) for t in (q, k, v, cu))
    out = fa.forward_varlen_prefill_fp16(qc, kc, vc, cuc, 200, causal)
    assert equal(out, fa.forward_varlen_prefill_fp16(misaligned(qc), kc, vc, cuc, 200, causal))
    assert_close(out, A.varlen_prefill(q, k, v, cu, 200, causal), what=f"varlen D={d}")


@pytest.mark.parametrize("d", [40, 80, 120])
def test_prefill_lse_chunk_rows(fa, d):
    g = gen(d + 3)
    qc, kc, vc = (randn(g, 2, 4, 150, d).to(DEV) for _ in range(3))
    out, lse = fa.forward_fp16_with_lse(qc, kc, vc, True)
    out2, lse2 = fa.forward_fp16_with_lse(misaligned(qc), kc, vc, True)
    assert equal(out, out2) and torch.equal(lse, lse2)


# Query heads per KV head 1..16 pick the kernels' head blocks; B = 40 x 4 KV
# heads is past the launch size from which contiguous decode stages K in LDS.
DECODE = [(1, 4, 4, 700), (2, 12, 4, 333), (40, 16, 4, 300), (1, 32, 2, 4100)]


@pytest.mark.parametrize("d", [8, 40, 72, 80, 96, 120, 192, 200])
@pytest.mark.parametrize("b,hq,hkv,n", DECODE)
def test_decode_chunk_rows(fa, d, b, hq, hkv, n):
    """Contiguous and sliding-window decode, continuous batching."""
    g = gen(d * 77 + n)
    q, k, v = randn(g, b, hq, 1, d), randn(g, b, hkv, n, d), randn(g, b, hkv, n, d)
    qc, kc, vc = (t.to(DEV) for t in (q, k, v))
    qm = misaligned(qc)
    out = fa.forward_decode_gqa_fp16(qc, kc, vc, True, n - 2)
    assert equal(out, fa.forward_decode_gqa_fp16(qm, kc, vc, True, n - 2))
    if n < 1000:
        assert_close(out, A.decode(q, k, v, True, n - 2), what=f"decode D={d}")
    out = fa.forward_decode_sliding_window_gqa(qc, kc, vc, True, n - 5, n // 2, 9)
    assert equal(out, fa.forward_decode_sliding_window_gqa(qm, kc, vc, True, n - 5, n // 2, 9))
    lens = torch.randint(0, n, (b,), generator=g, dtype=torch.int32).to(DEV)
    out = fa.forward_continuous_batching_fp16(qc, kc, vc, lens, True)
    assert equal(out, fa.forward_continuous_batching_fp16(qm, kc, vc, lens, True))


@pytest.mark.parametrize("d", [8, 40, 72, 80, 96, 120, 192, 200])
@pytest.mark.parametrize("b,hq,hkv,n", DECODE)
def test_paged_and_int8_decode_chunk_rows(fa, d, b, hq, hkv, n):
    g = gen(d * 79 + n)
    blocks = (n + 15) // 16
    pages = b * blocks + 3
    q = randn(g, b, hq, 1, d).to(DEV)
    qm = misaligned(q)
    kp, vp = randn(g, pages, hkv, 16, d).to(DEV), randn(g, pages, hkv, 16, d).to(DEV)
    table = torch.randperm(pages, generator=g)[:b * blocks].to(torch.int32).view(b, blocks).to(DEV)
    lens = torch.randint(1, n + 1, (b,), generator=g, dtype=torch.int32).to(DEV)
    out = fa.forward_paged_decode_gqa_fp16(q, kp, vp, table, lens, blocks)
    assert equal(out, fa.forward_paged_decode_gqa_fp16(qm, kp, vp, table, lens, blocks))

    k, v = randn(g, b, hkv, n, d).to(DEV), randn(g, b, hkv, n, d).to(DEV)
    qs = q.float().abs().amax((2, 3)) / 127.0
    ks = (k.float().abs().amax((2, 3)) / 127.0)[..., None].expand(b, hkv, n).contiguous()
    out = fa.forward_decode_int8_gqa(q, k, v, qs, ks, n - 1)
    assert equal(out, fa.forward_decode_int8_gqa(qm, k, v, qs, ks, n - 1))

    k8 = torch.randint(-127, 128, (b, hkv, n, d), generator=g, dtype=torch.int8).to(DEV)
    v8 = torch.randint(-127, 128, (b, hkv, n, d), generator=g, dtype=torch.int8).to(DEV)
    s1 = (torch.rand(b, hkv, n, generator=g) * 0.03).half().to(DEV)
    s2 = (torch.rand(b, hkv, n, generator=g) * 0.03).half().to(DEV)
    out = fa.forward_decode_int8_kv_cache_gqa(q, k8, v8, s1, s2, n - 1)
    assert equal(out, fa.forward_decode_int8_kv_cache_gqa(qm, k8, v8, s1, s2, n - 1))


@pytest.mark.parametrize("d", [72, 80, 200])
@pytest.mark.parametrize("b,hq,hkv,n", [(1, 4, 2, 200), (40, 16, 4, 300)])
def test_decode_chunk_rows_special_values(fa, d, b, hq, hkv, n):
    """Infinities and NaN of a cache reach the same outputs on both paths."""
    g = gen(d)
    q, k, v = randn(g, b, hq, 1, d).to(DEV), randn(g, b, hkv, n, d).to(DEV), randn(g, b, hkv, n, d).to(DEV)
    k[0, 0, 40, d - 1] = float("-inf")
    v[0, 1, 70, 0] = float("nan")
    v[0, 1, 71, d - 1] = float("inf")
    lens = torch.full((b,), n - 1, dtype=torch.int32, device=DEV)
    qm = misaligned(q)
    assert equal(fa.forward_decode_gqa_fp16(q, k, v, True, n - 1), fa.forward_decode_gqa_fp16(qm, k, v, True, n - 1))
    assert equal(fa.forward_continuous_batching_fp16(q, k, v, lens, True),
                 fa.forward_continuous_batching_fp16(qm, k, v, lens, True))


def _grads_close(got, ref, fp16):
    """fp16: 3e-2 + 3e-2 |x| and rel-L2 1e-2, fp32: 2e-4 + 2e-4 |x| (the bounds of
    the training tests)."""
    tol = 3e-2 if fp16 else 2e-4
    for name, a, r in zip(("dq", "dk", "dv"), got, ref):
        assert_close(a, r, atol=tol, rtol=tol, what=name)
        if fp16 and r.double().norm() > 1e-3:
            assert (a.double().cpu() - r.double().cpu()).norm() <= 1e-2 * r.double().cpu().norm(), name


def _train(fa, q, k, v, do, causal):
    fwd = fa.forward_fp16_with_lse if q.dtype == torch.float16 else fa.forward_with_lse
    out, lse = fwd(q, k, v, causal)
    return out, lse, fa.backward(do, q, k, v, out, lse, causal)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("b,h,n,d", [
    (1, 9, 1, 80), (1, 9, 63, 72), (2, 4, 64, 96), (2, 5, 65, 40), (1, 8, 127, 120), (3, 3, 193, 24),
    (1, 2, 130, 88), (2, 8, 385, 80),           # rows of whole chunks, split blocks
    (1, 9, 31, 64), (2, 4, 97, 64), (1, 8, 129, 128), (2, 8, 450, 128)])  # edges of split 32-row sub-tiles
def test_training_chunk_rows_and_split_blocks(fa, dtype, causal, b, h, n, d):
    g = gen(n * 31 + d)
    q, k, v, do = (randn(g, b, h, n, d, dtype=dtype) for _ in range(4))
    out, lse, grads = _train(fa, *(t.to(DEV) for t in (q, k, v, do)), causal)
    ro, rl = A.prefill_lse(q, k, v, causal, compute_dtype=torch.float64)
    fp16 = dtype == torch.float16
    assert_close(out, ro, **({} if fp16 else {"atol": 2e-4, "rtol": 2e-4}), what="out")
    assert_close(lse, rl, atol=2e-3 if fp16 else 2e-4, rtol=0 if fp16 else 2e-4, what="lse")
    _grads_close(grads, A.backward(do, q, k, v, out.cpu(), lse.cpu(), causal), fp16)
    again = _train(fa, *(t.to(DEV) for t in (q, k, v, do)), causal)[2]
    assert all(torch.equal(x, y) for x, y in zip(grads, again))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("d", [64, 80, 128])
def test_training_large_grid_matches_its_parts(fa, dtype, d):
    """A call past the grid size up to which blocks are split (512 blocks of 128
    rows) agrees with the same heads in a small, split call."""
    g = gen(d)
    q, k, v, do = (randn(g, 8, 13, 580, d, dtype=dtype).to(DEV) for _ in range(4))  # 520 blocks
    big = _train(fa, q, k, v, do, True)
    part = _train(fa, *(t[3:5].contiguous() for t in (q, k, v, do)), True)
    fp16 = dtype == torch.float16
    tol = {} if fp16 else {"atol": 2e-4, "rtol": 2e-4}
    assert_close(big[0][3:5], part[0], **tol, what="out")
    assert_close(big[1][3:5], part[1], atol=2e-3 if fp16 else 2e-4, rtol=0, what="lse")
    _grads_close([x[3:5] for x in big[2]], part[2], fp16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_training_in_order_calls_capture(fa, dtype):
    """A small backward under graph capture equals the eager one on every replay."""
    g = gen(5)
    q, k, v, do = (randn(g, 1, 8, 200, 80, dtype=dtype).to(DEV) for _ in range(4))
    out, lse, ref = _train(fa, q, k, v, do, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = fa.backward(do, q, k, v, out, lse, True)
    for _ in range(3):
        for x in got:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, ref))
        _train(fa, q, k, v, do, False)
