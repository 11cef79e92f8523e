"""mp_hip_paged_attention_decode_noalloc (the allocation-free variant)
against mp_hip_paged_attention_decode, the entry point it shares its kernel
with, and against the oracle.

Two calls in a row on rows long enough that their scores leave LDS for the
static device scratch (a KV head's 3 query heads x round_up(length, 16) >
kAttentionLdsScores = 10,240 floats), the second shorter than the first, so
it runs over what the first left there; then a row of 100 tokens, whose
scores stay in LDS.
Outputs must be bit-identical to the allocating entry point's (and to the
oracle's: the kernel keeps the reference CPU path's order). A row beyond
the scratch is rejected before any launch."""
import math

import numpy as np
import pytest

from oracle import Oracle
from tinyinfer_amd.backend import BackendError, paged_attention_decode, paged_attention_decode_noalloc

pytestmark = pytest.mark.gpu

HEADS, KV_HEADS, DIM, BT, LAYERS, LAYER = 9, 3, 64, 16, 2, 1


def _inputs(o, seed, length):
    pages = math.ceil(length / BT) + 8
    kvw = KV_HEADS * DIM
    keys = o.fill_normal(pages * LAYERS * BT * kvw, seed, 1)
    values = o.fill_normal(pages * LAYERS * BT * kvw, seed, 2)
    q = o.fill_normal(HEADS * DIM, seed, 3)
    table = o.permutation(pages, seed, 4)[: math.ceil(length / BT)].copy()
    return q, keys, values, table


def test_noalloc_matches_allocating_entry_point(torch_cuda):
    torch = torch_cuda
    o = Oracle()
    held = None
    # 3 x round_up(length, 16) > 10240 for 6000 and 4000 (scores in the
    # scratch), not for 100 (scores in LDS).
    for seed, length in ((5, 6000), (6, 4000), (7, 100)):
        q, keys, values, table = _inputs(o, seed, length)
        dq, dk, dv, dt = (torch.from_numpy(a).cuda() for a in (q, keys, values, table))
        base = torch.empty(HEADS * DIM, dtype=torch.float32, device="cuda")
        got = torch.full((HEADS * DIM,), float("nan"), dtype=torch.float32, device="cuda")
        args = (dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dt.data_ptr(), length, LAYER, LAYERS, BT, HEADS,
                KV_HEADS, DIM)
        paged_attention_decode(*args, base.data_ptr(), None)
        torch.cuda.synchronize()
        paged_attention_decode_noalloc(*args, got.data_ptr(), None)
        torch.cuda.synchronize()
        b, g = base.cpu().numpy(), got.cpu().numpy()
        assert np.all(np.isfinite(g))
        assert np.array_equal(g.view(np.uint32), b.view(np.uint32)), f"length {length}: differs from the allocating call"
        want = o.attention(q, keys, values, table, length - 1, 1, LAYER, LAYERS, BT, HEADS, KV_HEADS, DIM)[0]
        assert np.max(np.abs(g - want)) <= 1e-4
        assert np.array_equal(g.view(np.uint32), want.view(np.uint32))
        held = args
    # Beyond the scratch (9 x 30000 > 262144 floats): rejected before any launch.
    long_args = held[:4] + (30000,) + held[5:]
    out = torch.empty(HEADS * DIM, dtype=torch.float32, device="cuda")
    with pytest.raises(BackendError) as error:
        paged_attention_decode_noalloc(*long_args, out.data_ptr(), None)
    assert "exceeds" in str(error.value)


def _check(torch, o, seed, length, heads, kv_heads, scale=1.0, equal_keys=False):
    layers, layer = 2, 1
    pages = math.ceil(length / BT) + 3
    kvw = kv_heads * DIM
    keys = o.fill_normal(pages * layers * BT * kvw, seed, 1)
    if equal_keys:
        keys[:] = 0.25
    values = o.fill_normal(pages * layers * BT * kvw, seed, 2)
    q = o.fill_normal(heads * DIM, seed, 3, scale)
    table = o.permutation(pages, seed, 4)[: math.ceil(length / BT)].copy()
    want = o.attention(q, keys, values, table, length - 1, 1, layer, layers, BT, heads, kv_heads, DIM)[0]
    dq, dk, dv, dt = (torch.from_numpy(a).cuda() for a in (q, keys, values, table))
    for call in (paged_attention_decode, paged_attention_decode_noalloc):
        got = torch.full((heads * DIM,), float("nan"), dtype=torch.float32, device="cuda")
        call(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dt.data_ptr(), length, layer, layers, BT, heads, kv_heads, DIM,
             got.data_ptr(), None)
        torch.cuda.synchronize()
        g = got.cpu().numpy()
        assert np.array_equal(g.view(np.uint32), want.view(np.uint32)), (call.__name__, length, heads, kv_heads)


@pytest.mark.parametrize("length", [1, 15, 17, 64, 224, 225, 256, 257, 511, 640, 641, 896, 897, 1025, 3413, 3414, 18431,
                                    18432, 18433, 20000])
def test_row_kernel_edges(torch_cuda, length):
    """Bits of the oracle at the edges of the row kernel: partial pages,
    phases of 14 pages and turns of four phases, the 256 denominator values
    added one by one, rows whose scores take a launch of their own (from 3,409
    tokens on with 3 query heads per KV head, in the scratch), and rows beyond
    the 18,432-token window."""
    _check(torch_cuda, Oracle(), 100 + length, length, HEADS, KV_HEADS)


@pytest.mark.parametrize("group", [1, 2, 4, 5, 6, 7, 8])
def test_row_kernel_groups(torch_cuda, group):
    """Every number of query heads per KV head, scores in the row kernel and
    in the scratch."""
    for length in (77, 1500, 10300):
        _check(torch_cuda, Oracle(), 200 + group, length, 2 * group, 2)


@pytest.mark.parametrize("heads,kv_heads", [(16, 16), (72, 24), (128, 128)])
def test_many_heads(torch_cuda, heads, kv_heads):
    """Short rows of heads of their own and rows of very many heads take the
    general kernel, longer ones the row kernel: bits of the oracle on both
    sides."""
    for length in (1, 63, 90, 130, 600, 1000):
        _check(torch_cuda, Oracle(), 350, length, heads, kv_heads)


@pytest.mark.parametrize("scale,equal", [(0.0, False), (1.0, True), (8.0, False), (0.05, False)])
def test_row_kernel_denominators(torch_cuda, scale, equal):
    """Denominators that are exact in every step (equal scores: all e_t are
    1, the sum crosses each power of two exactly), that hardly change after
    a few tokens (peaked scores, many e_t far below one unit of the sum) and
    that grow evenly."""
    for length in (500, 5000):
        _check(torch_cuda, Oracle(), 300, length, HEADS, KV_HEADS, scale, equal)


@pytest.mark.parametrize("length", [1, 77, 503, 640, 1500, 5000])
def test_out_in_place_of_q(torch_cuda, length):
    """`out` may be q's own buffer: the work-groups of a head that read its q
    must not find another's output there. Bits of the oracle, with more heads
    (96, four work-groups each in the row kernel) than fit the chip at once,
    so that some start after others have ended."""
    torch, o = torch_cuda, Oracle()
    heads, kv_heads = (96, 32) if length <= 2000 else (HEADS, KV_HEADS)
    pages = math.ceil(length / BT)
    kvw = kv_heads * DIM
    keys, values = o.fill_normal(pages * BT * kvw, 400, 1), o.fill_normal(pages * BT * kvw, 400, 2)
    q = o.fill_normal(heads * DIM, 400, 3)
    table = o.permutation(pages, 400, 4)
    want = o.attention(q, keys, values, table, length - 1, 1, 0, 1, BT, heads, kv_heads, DIM)[0]
    dk, dv, dt = (torch.from_numpy(a).cuda() for a in (keys, values, table))
    for call in (paged_attention_decode, paged_attention_decode_noalloc):
        buffer = torch.from_numpy(q.copy()).cuda()
        call(buffer.data_ptr(), dk.data_ptr(), dv.data_ptr(), dt.data_ptr(), length, 0, 1, BT, heads, kv_heads, DIM,
             buffer.data_ptr(), None)
        torch.cuda.synchronize()
        got = buffer.cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (call.__name__, length)


def test_rows_with_scores_on_the_chip_may_overlap(torch_cuda):
    """Allocation-free calls for rows of up to 10,240 score floats per KV head
    share nothing: eight rows of 700 to 3,408 tokens on eight streams at once,
    ten rounds, each with the oracle's bits."""
    torch, o = torch_cuda, Oracle()
    rows = []
    for i, length in enumerate((700, 1000, 1500, 2000, 2500, 3000, 3400, 3408)):
        q, keys, values, table = _inputs(o, 500 + i, length)
        want = o.attention(q, keys, values, table, length - 1, 1, LAYER, LAYERS, BT, HEADS, KV_HEADS, DIM)[0]
        rows.append((length, [torch.from_numpy(a).cuda() for a in (q, keys, values, table)], want,
                     torch.empty(HEADS * DIM, dtype=torch.float32, device="cuda"), torch.cuda.Stream()))
    for _ in range(10):
        for _, _, _, out, _ in rows:
            out.fill_(float("nan"))
        torch.cuda.synchronize()
        for length, inputs, _, out, stream in rows:
            paged_attention_decode_noalloc(*(t.data_ptr() for t in inputs), length, LAYER, LAYERS, BT, HEADS, KV_HEADS,
                                           DIM, out.data_ptr(), stream.cuda_stream)
        torch.cuda.synchronize()
        for length, _, want, out, _ in rows:
            assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32)), length


@pytest.mark.parametrize("length", [300, 1500, 5000])
def test_row_kernel_infinities_and_nans(torch_cuda, length):
    """Infinite and NaN keys (either sign, in the first 256 tokens and in the
    last ones) and values: the oracle's bits where it is not NaN, NaN exactly
    where it is. One KV head holds the odd values, the others stay finite."""
    torch, o = torch_cuda, Oracle()
    bad = [("keys", np.inf), ("keys", -np.inf), ("keys", np.nan), ("keys", -np.nan), ("values", np.inf),
           ("values", np.nan)]
    for i, (where, value) in enumerate(bad):
        for token in (7, length - 3):
            q, keys, values, table = _inputs(o, 600 + i, length)
            pool = (keys if where == "keys" else values).reshape(-1, LAYERS, BT, KV_HEADS, DIM)
            pool[table[token // BT], LAYER, token % BT, 1, 5] = value
            with np.errstate(all="ignore"):
                want = o.attention(q, keys, values, table, length - 1, 1, LAYER, LAYERS, BT, HEADS, KV_HEADS, DIM)[0]
            dq, dk, dv, dt = (torch.from_numpy(a).cuda() for a in (q, keys, values, table))
            for call in (paged_attention_decode, paged_attention_decode_noalloc):
                out = torch.zeros(HEADS * DIM, dtype=torch.float32, device="cuda")
                call(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dt.data_ptr(), length, LAYER, LAYERS, BT, HEADS,
                     KV_HEADS, DIM, out.data_ptr(), None)
                torch.cuda.synchronize()
                got = out.cpu().numpy()
                assert np.array_equal(np.isnan(got), np.isnan(want)), (where, value, token)
                ok = ~np.isnan(want)
                assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32)), (where, value, token)
                assert np.all(np.isfinite(np.delete(got.reshape(KV_HEADS, -1), 1, axis=0)))


@pytest.mark.parametrize("length", [77, 1500, 5000])
def test_values_at_any_float(torch_cuda, length):
    """V pools that start at any float, not only at 16 bytes: the oracle's
    bits."""
    torch, o = torch_cuda, Oracle()
    q, keys, values, table = _inputs(o, 700, length)
    want = o.attention(q, keys, values, table, length - 1, 1, LAYER, LAYERS, BT, HEADS, KV_HEADS, DIM)[0]
    dq, dk, dt = (torch.from_numpy(a).cuda() for a in (q, keys, table))
    for offset in (1, 2, 3):
        room = torch.empty(values.size + 4, dtype=torch.float32, device="cuda")
        dv = room[offset:offset + values.size]
        dv.copy_(torch.from_numpy(values))
        for call in (paged_attention_decode, paged_attention_decode_noalloc):
            out = torch.zeros(HEADS * DIM, dtype=torch.float32, device="cuda")
            call(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dt.data_ptr(), length, LAYER, LAYERS, BT, HEADS, KV_HEADS,
                 DIM, out.data_ptr(), None)
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32)), (call.__name__, offset)
