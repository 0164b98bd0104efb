"""GPU parity of the split-KV verification attention (libqf_spec_attn.so through its C ABI) against
the fp64 oracle (oracle/attn.py), with the tolerance rule of oracle.attn.check_spec_attn.

The case matrix follows the reference's own test (bench/test_spec_attn.py:7-19): H = 24, H_kv = 4,
D = 256, 800-position pages laid out [page][H_kv][PAGE][2D] with K and V interleaved, shuffled
pages, requests of lengths ctx + Q - 7 b, contexts 0 .. 8000 (and 38000) with (Q, B) in
{(3, 1), (4, 1), (3, 2)}.  Further cases cover the other head sizes, every packed-row count class,
vLLM's separate [page][PAGE][H_kv][D] caches with 16-position pages, the split settings, a split
spanning more pages than one block-table window, rows that see no position, determinism and HIP
graph replay.
"""
import numpy as np
import pytest

from oracle import attn as A

pytestmark = pytest.mark.gpu


def _dev(inp: A.SpecInputs, separate: bool = False):
    import torch
    dev = torch.device("cuda:0")
    kv = torch.from_numpy(inp.kv.view(np.int16)).to(dev).view(torch.bfloat16)
    key_cache, value_cache = kv.transpose(1, 2).split(inp.D, dim=-1)
    if separate:
        key_cache, value_cache = key_cache.contiguous(), value_cache.contiguous()
    q = torch.from_numpy(inp.q.view(np.int16)).to(dev).view(torch.bfloat16)
    bt = torch.from_numpy(inp.block_table).to(dev)
    sl = torch.from_numpy(inp.seq_lens).to(dev)
    return q, key_cache, value_cache, bt, sl


def _run(inp, separate=False, **kw):
    import torch
    import qwen_fastpath as qf
    q, kc, vc, bt, sl = _dev(inp, separate)
    out = torch.full_like(q, float("nan"))
    qf.gqa_packed_spec_attention(q, kc, vc, out, sl, bt, inp.B, inp.Q, inp.HKV, inp.D ** -0.5, **kw)
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


def _check(inp, out, tag):
    ref = A.spec_attention(inp.query(), inp.key_cache(), inp.value_cache(), inp.seq_lens, inp.block_table,
                           inp.B, inp.Q, inp.HKV, inp.D ** -0.5)
    rep = A.check_spec_attn(out, ref, inp.seq_lens, inp.Q)
    print(f"spec_attn {tag}: {rep}", flush=True)
    assert rep.ok, (tag, rep)


@pytest.mark.parametrize("ctx", [0, 1, 2, 50, 1000, 8000])
@pytest.mark.parametrize("Q,B", [(3, 1), (4, 1), (3, 2)])
def test_reference_matrix(ctx, Q, B):
    inp = A.gen_spec_inputs(ctx, Q, B, seed=ctx * 10 + Q + B)
    _check(inp, _run(inp), f"ctx={ctx} Q={Q} B={B}")


def test_long_context_38k():
    inp = A.gen_spec_inputs(38000, 3, 1, seed=38)
    _check(inp, _run(inp), "ctx=38000 Q=3 B=1")


@pytest.mark.parametrize("H,HKV,D,Q", [
    (32, 8, 128, 4),    # G = 4, 16 packed rows
    (16, 2, 64, 8),     # G = 8, 64 packed rows
    (24, 4, 256, 8),    # G = 6, 48 packed rows
    (24, 4, 256, 1),    # a single query token
    (8, 8, 128, 2),     # no grouping
])
def test_head_shapes(H, HKV, D, Q):
    inp = A.gen_spec_inputs(3000, Q, 2, H=H, HKV=HKV, D=D, page=800, seed=H + D + Q)
    _check(inp, _run(inp), f"H={H} HKV={HKV} D={D} Q={Q}")


@pytest.mark.parametrize("D", [64, 128, 256])
def test_separate_caches_small_pages(D):
    inp = A.gen_spec_inputs(2500, 3, 2, H=24, HKV=4, D=D, page=16, seed=D)
    _check(inp, _run(inp, separate=True), f"separate D={D} page=16")


@pytest.mark.parametrize("num_splits,min_chunk", [(1, 128), (7, 1), (64, 32), (256, 32), (1000, 1)])
def test_split_settings(num_splits, min_chunk):
    inp = A.gen_spec_inputs(5000, 3, 2, seed=num_splits)
    _check(inp, _run(inp, num_splits=num_splits, min_chunk=min_chunk), f"splits={num_splits} min_chunk={min_chunk}")


@pytest.mark.parametrize("min_chunk", [1 << 26, 1 << 30, (1 << 31) - 40, (1 << 31) - 1])
@pytest.mark.parametrize("B,num_splits", [(1, None), (3, None), (2, 64), (1, 65535)])
def test_min_chunk_past_every_length(min_chunk, B, num_splits):
    """A min_chunk longer than any request means one split each, whatever split * min_chunk comes to: the unused splits
    take no position and the result is that of num_splits=1, bit for bit."""
    inp = A.gen_spec_inputs(700, 3, B, H=8, HKV=2, D=64, page=16, seed=B)
    out = _run(inp, num_splits=num_splits, min_chunk=min_chunk)
    _check(inp, out, f"min_chunk={min_chunk} B={B} splits={num_splits}")
    assert np.array_equal(out.view(np.uint32), _run(inp, num_splits=1).view(np.uint32))


def test_split_spanning_several_table_windows():
    # one split over 20000 positions of 16-position pages: 1251 pages, more than one 1024-entry window
    inp = A.gen_spec_inputs(20000, 3, 1, H=16, HKV=2, D=128, page=16, seed=77)
    _check(inp, _run(inp, num_splits=1), "windows page=16 splits=1")


@pytest.mark.parametrize("D,HKV,G,Q,page,lens", [
    (128, 4, 8, 5, 16, [9005, 7672, 6339, 5006, 3673, 2340]),  # 3 row tiles; the splits go by length
    (256, 2, 6, 3, 800, [5003, 3, 64 + 3, 65 + 3, 2, 1, 2000]),  # no prefix, one stage, one stage and a position
    (256, 1, 8, 8, 24, [3000, 17, 700]),                       # 4 row tiles, pages that cut key tiles
    (256, 2, 6, 8, 17, [1111, 900]),                           # 3 row tiles
    (128, 8, 8, 8, 16, [4200, 77, 129, 128 + 8]),              # 4 row tiles, 4 wavefronts
    (128, 2, 1, 2, 64, [131, 127, 5000]),                      # 1 row tile
    (64, 4, 8, 4, 17, [3001, 16, 260]),                        # 2 row tiles, every other one a wavefront
    (64, 2, 7, 7, 32, [70, 8000]),                             # 4 row tiles
    (64, 1, 2, 2, 16, [1 + 40 * i for i in range(64)]),            # the most requests
])
def test_balanced_batches(D, HKV, G, Q, page, lens):
    """Ragged batches through the balanced splits; every cache row that no query may see holds NaN, and the later
    positions score higher, so that the exponent references move stage after stage."""
    inp = A.gen_spec_inputs(max(lens), Q, len(lens), H=G * HKV, HKV=HKV, D=D, page=page, seed=D + Q + page, lens=lens)
    nan = np.ones(inp.kv.shape[:1] + inp.kv.shape[2:3], dtype=bool)  # [page id, row]
    for b, n in enumerate(lens):
        pos = np.arange(n)
        nan[inp.block_table[b, pos // page], pos % page] = False
        blk, off = inp.block_table[b, pos // page], pos % page
        grow = (1.0 + 6.0 * pos / max(lens))[:, None, None]
        k = A.bf16_bits_to_f32(inp.kv[blk, :, off, :D]) * grow
        inp.kv[blk, :, off, :D] = A.bf16_bits_from_f32(k.astype(np.float32))
    kv_clean = inp.kv.copy()
    inp.kv.transpose(0, 2, 1, 3)[nan] = 0x7FC0
    out = _run(inp)
    inp.kv[:] = kv_clean
    _check(inp, out, f"balanced D={D} HKV={HKV} G={G} Q={Q} page={page} lens={lens[:7]}")


def _growing_poisoned(lens, Q, D, HKV, G, page, seed):
    """A batch whose later positions score higher, so that the exponent references move in stage after stage, and the same
    cache with NaN in every row that no query may see."""
    inp = A.gen_spec_inputs(max(lens), Q, len(lens), H=G * HKV, HKV=HKV, D=D, page=page, seed=seed, lens=lens)
    unseen = np.ones(inp.kv.shape[:1] + inp.kv.shape[2:3], dtype=bool)  # [page id, row]
    for b, n in enumerate(lens):
        pos = np.arange(n)
        blk, off = inp.block_table[b, pos // page], pos % page
        unseen[blk, off] = False
        k = A.bf16_bits_to_f32(inp.kv[blk, :, off, :D]) * (1.0 + 6.0 * pos / n)[:, None, None]
        inp.kv[blk, :, off, :D] = A.bf16_bits_from_f32(k.astype(np.float32))
    poisoned = inp.kv.copy()
    poisoned.transpose(0, 2, 1, 3)[unseen] = 0x7FC0
    return inp, poisoned


@pytest.mark.parametrize("D,G,Q,page,lens", [
    # 8 wavefronts, 128 positions a stage, wavefronts in two row groups
    (64, 8, 2, 17, [700, 643]), (64, 8, 3, 64, [900, 517]), (64, 8, 3, 24, [900, 517]),
    (64, 8, 5, 64, [1100, 641]), (64, 8, 5, 17, [1100, 641]), (64, 8, 8, 16, [1300, 650]), (64, 7, 8, 24, [1300, 650]),
    # 4 wavefronts, 64 positions a stage
    (128, 4, 3, 17, [600, 449]), (128, 8, 5, 24, [600, 449]), (128, 8, 8, 17, [600, 449]),
    (256, 6, 2, 24, [600, 449]), (256, 6, 3, 17, [600, 449]), (256, 8, 8, 24, [600, 449]),
    # more than 64 stages: the block ids are read again
    (256, 6, 3, 17, [4500]), (128, 2, 4, 24, [4460]), (64, 2, 2, 17, [8600]), (64, 2, 2, 32, [8600]),
])
def test_long_splits(D, G, Q, page, lens):
    """One split a request, several stages long, on pages that hold whole key tiles and pages that cut them."""
    inp, poisoned = _growing_poisoned(lens, Q, D, 2, G, page, seed=D + G + Q + page)
    clean = inp.kv
    for kw in ({"num_splits": 1}, {"min_chunk": 1 << 20}):
        inp.kv = poisoned
        out = _run(inp, **kw)
        inp.kv = clean
        _check(inp, out, f"long splits D={D} G={G} Q={Q} page={page} lens={lens} {kw}")


def test_balanced_where_two_slots_a_request(monkeypatch):
    """The default call shares out a batch's splits by length where a kv head has two or more slots a request, and splits
    evenly otherwise (one request, more requests than that, an explicit split count)."""
    import torch
    from qwen_fastpath import _attn_lib as AL
    lib, calls = AL.load(), []

    class Spy:
        def __getattr__(self, name):
            if name.startswith("qf_spec_attention"):
                calls.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(AL, "load", lambda: Spy())
    slots = torch.cuda.get_device_properties(0).multi_processor_count // 4
    for B, kw, want in ((1, {}, False), (2, {}, True), (slots // 2, {}, True), (slots // 2 + 1, {}, False), (2, {"num_splits": 8}, False)):
        inp = A.gen_spec_inputs(90, 2, B, H=4, HKV=4, D=64, page=16, seed=B, lens=[92 - b % 40 for b in range(B)])
        calls.clear()
        _check(inp, _run(inp, **kw), f"B={B} {kw}")
        assert ("qf_spec_attention_balanced" in calls) is (want and B <= 64), (B, kw, calls)


def test_rows_that_see_nothing_are_zero():
    inp = A.gen_spec_inputs(0, 4, 3, seed=5, lens=[1, 2, 4])
    out = _run(inp)
    _check(inp, out, "short requests")
    assert np.all(out[0:3] == 0) and np.all(out[4:6] == 0)


def test_empty_request_in_a_batch_is_zero():
    inp = A.gen_spec_inputs(300, 3, 2, seed=6, lens=[0, 303])
    assert np.all(_run(inp)[:3] == 0)


def test_deterministic():
    inp = A.gen_spec_inputs(6000, 3, 2, seed=9)
    a, b = _run(inp), _run(inp)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_graph_replay_matches_eager():
    import torch
    import qwen_fastpath as qf
    inp = A.gen_spec_inputs(4000, 3, 2, seed=12)
    q, kc, vc, bt, sl = _dev(inp)
    scale = inp.D ** -0.5
    eager = torch.empty_like(q)
    qf.gqa_packed_spec_attention(q, kc, vc, eager, sl, bt, inp.B, inp.Q, inp.HKV, scale)
    torch.cuda.synchronize()
    out = torch.zeros_like(q)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        qf.gqa_packed_spec_attention(q, kc, vc, out, sl, bt, inp.B, inp.Q, inp.HKV, scale)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        qf.gqa_packed_spec_attention(q, kc, vc, out, sl, bt, inp.B, inp.Q, inp.HKV, scale)
    for i in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), f"replay {i}"
        _ = (q.float() * 2).sum().item()  # unrelated eager work between replays
    _check(inp, eager.float().cpu().numpy(), "graph eager")


def test_unsupported_shapes_raise():
    import torch
    import qwen_fastpath as qf
    from qwen_fastpath._lib import QFError
    inp = A.gen_spec_inputs(100, 3, 1, H=8, HKV=2, D=64, page=16, seed=1)
    q, kc, vc, bt, sl = _dev(inp)
    out = torch.empty_like(q)
    with pytest.raises(QFError):  # 3 * 32 packed rows > 64
        qf.gqa_packed_spec_attention(q.repeat(1, 8, 1), kc, vc, out.repeat(1, 8, 1), sl, bt, 1, 3, 2, 0.125)


def test_default_split_count_is_one_workgroup_per_cu():
    import torch
    from qwen_fastpath import spec_attn as SA
    dev = torch.device("cuda:0")
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert SA.auto_num_splits(dev, 1, 4) == max(1, cus // 4)
    assert SA.auto_num_splits(dev, 2, 4) == max(1, cus // 8)
    assert SA.auto_num_splits(dev, cus, 8) == 1
    inp = A.gen_spec_inputs(7000, 3, 2, seed=31)
    auto = _run(inp)
    explicit = _run(inp, num_splits=max(1, cus // (2 * inp.HKV)))
    assert np.array_equal(auto.view(np.uint32), explicit.view(np.uint32))
    _check(inp, auto, "default splits")
