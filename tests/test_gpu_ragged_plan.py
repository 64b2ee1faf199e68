"""Continuous batching and paged decode with the splits planned from the lengths
on the device: sequences against the CPU oracle, and all of them against calls with
one alone, at batch sizes on both sides of the planner's register blocks (64, 128, 256
and 512 sequences) and past it, with empty and negative lengths, lengths on and next
to chunk boundaries, all equal, and one long sequence among short ones."""
import pytest
import torch

from oracle import attention as A
from tests.helpers import assert_close, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gen(seed):
    return torch.Generator().manual_seed(seed)


def lengths(kind, b, n, g):
    if kind == "uniform":
        return torch.randint(0, n, (b,), generator=g)
    if kind == "equal":
        return torch.full((b,), n - 1)
    if kind == "edges":  # attended keys 0, 1, multiples of 256 and their neighbours
        e = torch.tensor([0, 1, 255, 256, 257, 511, 512, 513, 767, 768, 1024, n, n - 1])
        return torch.minimum(e[torch.randint(0, len(e), (b,), generator=g)], torch.tensor(n)) - 1
    lens = torch.randint(0, 9, (b,), generator=g)  # one long sequence
    lens[b // 2] = n - 1
    return lens


@pytest.mark.parametrize("kind", ["uniform", "equal", "edges", "one_long"])
@pytest.mark.parametrize("b,hq,hkv,n,d", [(64, 16, 4, 1100, 64), (65, 8, 4, 900, 128), (129, 8, 2, 1300, 64),
                                          (16, 32, 8, 2500, 64), (512, 2, 1, 600, 64), (513, 2, 1, 600, 64),
                                          (3, 32, 8, 9000, 64), (256, 4, 2, 700, 64), (257, 4, 2, 700, 64),
                                          (160, 8, 4, 256, 64)])  # the last: one split, not planned
def test_continuous_batching_planned(fa, kind, b, hq, hkv, n, d):
    g = gen(b + n)
    q, k, v = randn(g, b, hq, 1, d), randn(g, b, hkv, n, d), randn(g, b, hkv, n, d)
    lens = lengths(kind, b, n, g).to(torch.int32)
    lens[0] = -1  # no key: NaN
    out = fa.forward_continuous_batching_fp16(*(t.to(DEV) for t in (q, k, v, lens)), True)
    for i in sorted({0, 1, b // 2, b // 3, b - 1}):
        ref = A.continuous_batching(q[i:i + 1], k[i:i + 1], v[i:i + 1], lens[i:i + 1], True)
        assert_close(out[i:i + 1], ref, what=f"{kind} sequence {i} of {b}, {int(lens[i])}")
    again = fa.forward_continuous_batching_fp16(*(t.to(DEV) for t in (q, k, v, lens)), True)
    assert torch.equal(torch.nan_to_num(out), torch.nan_to_num(again))  # counters back at zero, same sums


@pytest.mark.parametrize("kind", ["uniform", "equal", "edges", "one_long", "overrun"])
@pytest.mark.parametrize("b,hq,hkv,n,d", [(64, 16, 4, 1100, 64), (65, 8, 4, 900, 128), (129, 8, 2, 1300, 64),
                                          (16, 32, 8, 2500, 64), (512, 2, 1, 600, 64), (513, 2, 1, 600, 64),
                                          (256, 4, 2, 700, 64), (257, 4, 2, 700, 64),
                                          # enough sequences to fill the CUs: split or not by the lengths
                                          (128, 8, 8, 700, 64), (256, 8, 4, 500, 64), (512, 4, 2, 300, 64),
                                          (800, 1, 1, 300, 64),  # (static: past the planned batches)
                                          (100, 8, 8, 9000, 64)])
def test_paged_planned(fa, kind, b, hq, hkv, n, d):
    g = gen(b + n + 1)
    blocks = (n + 15) // 16
    pages = min(b * blocks, 8192)  # (long tables share pages)
    q = randn(g, b, hq, 1, d)
    k, v = randn(g, pages, hkv, 16, d), randn(g, pages, hkv, 16, d)
    table = torch.randperm(b * blocks, generator=g).remainder(pages).to(torch.int32).view(b, blocks)
    lens = (lengths("uniform" if kind == "overrun" else kind, b, n, g) + 1).to(torch.int32)
    lens[0] = 0
    if kind == "overrun":  # reads on into the next table row, as the flat table does
        lens[1] = 16 * blocks + 1
        lens[b // 2] = 16 * blocks + 300
    out = fa.forward_paged_decode_gqa_fp16(*(t.to(DEV) for t in (q, k, v, table, lens)), blocks)
    flat = table.flatten()
    for i in sorted({0, 1, b // 2, b // 3, b - 1}):
        ln = int(lens[i])
        if ln == 0:
            assert torch.isnan(out[i]).all()
            continue
        ids = flat[i * blocks:i * blocks + (ln + 15) // 16].long()
        ks, vs = (t[ids].transpose(0, 1).reshape(1, hkv, -1, d)[:, :, :ln] for t in (k, v))
        assert_close(out[i:i + 1], A.decode(q[i:i + 1], ks, vs, True, ln - 1), what=f"{kind} sequence {i}, {ln}")
    again = fa.forward_paged_decode_gqa_fp16(*(t.to(DEV) for t in (q, k, v, table, lens)), blocks)
    assert torch.equal(torch.nan_to_num(out), torch.nan_to_num(again))


@pytest.mark.parametrize("kind", ["uniform", "equal", "edges", "one_long"])
@pytest.mark.parametrize("b,hq,hkv,n,d", [(128, 8, 8, 700, 64), (256, 8, 4, 500, 64), (100, 8, 8, 21000, 64)])
def test_paged_planned_equals_single_sequences(fa, kind, b, hq, hkv, n, d):
    """Every sequence of a batch that fills the CUs against a call with that
    sequence alone, whose splits come from its table; the last size has chunks of
    more keys than one staging of page ids holds (8192)."""
    g = gen(b + n + 2)
    blocks = (n + 15) // 16
    pages = min(b * blocks, 8192)
    q, k, v = (t.to(DEV) for t in (randn(g, b, hq, 1, d), randn(g, pages, hkv, 16, d), randn(g, pages, hkv, 16, d)))
    table = torch.randint(0, pages, (b, blocks), generator=g).to(torch.int32).to(DEV)
    lens = (lengths(kind, b, n, g) + 1).to(torch.int32).to(DEV)
    lens[1] = 0
    out = fa.forward_paged_decode_gqa_fp16(q, k, v, table, lens, blocks)
    one = [fa.forward_paged_decode_gqa_fp16(q[i:i + 1], k, v, table[i:i + 1], lens[i:i + 1], blocks) for i in range(b)]
    assert_close(out, torch.cat(one), what=f"{kind} [{b}] to {n}")


@pytest.mark.parametrize("kind", ["uniform", "equal", "edges", "one_long"])
@pytest.mark.parametrize("b,hq,hkv,n,d", [(40, 16, 4, 1100, 64), (128, 8, 4, 900, 64), (200, 8, 4, 900, 64),
                                          (400, 8, 4, 600, 64)])
def test_continuous_batching_planned_equals_single_sequences(fa, kind, b, hq, hkv, n, d):
    """Every sequence of a planned batch against a call with that sequence alone."""
    g = gen(b + n + 3)
    q, k, v = (t.to(DEV) for t in (randn(g, b, hq, 1, d), randn(g, b, hkv, n, d), randn(g, b, hkv, n, d)))
    lens = lengths(kind, b, n, g).to(torch.int32).to(DEV)
    lens[1] = -1
    out = fa.forward_continuous_batching_fp16(q, k, v, lens, True)
    one = [fa.forward_continuous_batching_fp16(q[i:i + 1], k[i:i + 1], v[i:i + 1], lens[i:i + 1], True)
           for i in range(b)]
    assert_close(out, torch.cat(one), what=f"{kind} [{b}] to {n}")


def _call_us(call, n=20):
    call()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    for _ in range(n):
        call()
    end.record()
    end.synchronize()
    return start.elapsed_time(end) / n * 1e3


def test_paged_long_sequence_in_a_full_batch_is_split(fa):
    """One long sequence among short ones must not be left to one workgroup per
    KV head, however many sequences there are: split in the four that the
    workspace has, the call takes an 18th of one whose sequences are all as
    long, unsplit a 5th."""
    b, h, n, d = 128, 8, 32768, 128
    pages = 16384
    g = torch.Generator(device=DEV).manual_seed(8)
    q = torch.randn(b, 4 * h, 1, d, generator=g, device=DEV).half()
    k, v = (torch.randn(pages, h, 16, d, generator=g, device=DEV).half() for _ in range(2))
    table = torch.randint(0, pages, (b, n // 16), generator=g, device=DEV, dtype=torch.int32)
    lens = torch.full((b,), n, dtype=torch.int32, device=DEV)
    call = lambda: fa.forward_paged_decode_gqa_fp16(q, k, v, table, lens, n // 16)
    every = _call_us(call)
    lens.fill_(100)
    lens[b // 2] = n
    assert 8 * _call_us(call) < every


def test_planned_calls_replay_with_other_lengths(fa):
    """A captured call plans from the lengths of each replay."""
    g = gen(3)
    b, n = 32, 2000
    q, k, v = (t.to(DEV) for t in (randn(g, b, 8, 1, 64), randn(g, b, 8, n, 64), randn(g, b, 8, n, 64)))
    lens = torch.randint(0, n, (b,), generator=g).to(torch.int32).to(DEV)
    fa.forward_continuous_batching_fp16(q, k, v, lens, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fa.forward_continuous_batching_fp16(q, k, v, lens, True)
    for kind in ("uniform", "one_long", "equal", "edges"):
        lens.copy_(lengths(kind, b, n, g).clamp(min=0).to(torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, fa.forward_continuous_batching_fp16(q, k, v, lens, True))
