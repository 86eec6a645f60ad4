"""Extend entries cut over their keys (tf_attn_plan_blocks' pieces and merges,
tf_attn_extend_split): the plan against a direct restatement of its rule, and
steps whose entries are cut against the oracle (the extend tests' tolerance) in
every planning mode, at the edges of pieces, with rows that see no key of a
piece, and with the gate, out_amax, fp8 pools and bsz == 1 -1 entries.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests.helpers import assert_attn_close, restatement
from tests.test_gpu_gate import assert_bits_match, module_gate
from tokenfactory_amd import slot_based_attention, workloads
from tokenfactory_amd.attention import SlotAttentionCall
from tokenfactory_amd.planning import plan_extend

pytestmark = pytest.mark.gpu


def case(gpu, seq, ext, hq=24, hkv=4, seed=0, fp8=False):
    return workloads.build("split", seq, ext, num_q_heads=hq, num_kv_heads=hkv, head_dim=256,
                           pool_slots=2 * sum(seq) + 64, device=gpu, seed=seed, kv_fp8=fp8)


def call_of(wl, **kw):
    return SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                             k_scale=wl.k_scale, v_scale=wl.v_scale, **kw)


def lists(call):
    torch.cuda.synchronize()
    r, got = call.route, call._lists.cpu().numpy()
    p0 = 4 * r.n_blocks
    m0 = p0 + 8 * r.n_pieces
    return got[p0:m0].reshape(-1, 8), got[m0:].reshape(-1, 8)


def expected(wl, cus):
    """The pieces and merges of tf_attn_plan_blocks' rule."""
    group = wl.num_q_heads // wl.num_kv_heads
    work = [w for w in plan_extend(wl.ext_lens, wl.num_q_heads, wl.num_kv_heads, True).tolist()
            if w[4] * group > 64]
    tiles = []
    for b, _, row0, _, ext, *_ in work:
        last = min(row0 + 256, ext * group) - 1
        tiles.append(-(-min(wl.seq_lens[b], wl.seq_lens[b] - ext + last // group + 1) // 32))
    count = lambda n: sum(-(-t // n) for t in tiles)
    mx, length = max(tiles), 0
    if len(work) <= cus and mx >= 24:
        n = next(n for n in range(12, mx + 1) if count(n) <= cus)
        # the decode rows' time in tiles: the split has to win with them after it
        rows = sum(l for l, e in zip(wl.seq_lens, wl.ext_lens) if e * group <= 64)
        rows *= 2 * wl.num_kv_heads * 256 * wl.k_pool.element_size() / 9e6
        if n + 24 + 3 + 0.047 * count(n) + rows < 0.92 * max(mx + 15, rows):
            length = n
    pieces, merges, slot = [], [], 0
    for w, t in zip(work, tiles):
        n = -(-t // length) if length else 1
        if n == 1:
            pieces.append(w)
            continue
        merges.append(w[:5] + [slot, n, 0])
        pieces += [w[:5] + [t * k // n, t * (k + 1) // n, slot + k + 1] for k in range(n)]
        slot += n
    return pieces, merges


@pytest.mark.parametrize("seq,ext", [
    ([3000], [100]), ([6100, 1700, 5300], [211, 37, 100]), ([5000], [2000]),
    ([900, 400], [12, 11]), ([4000, 50, 2000], [700, 50, 1]), ([20000], [11]),
    ([1500] * 20, [200] * 20), ([3000] + [2000] * 80, [260] + [1] * 80),
    ([6000] + [2000] * 20 + [500], [260] + [1] * 20 + [4])])
@pytest.mark.parametrize("device_plan", [False, True])
def test_plan(gpu, seq, ext, device_plan):
    wl = case(gpu, seq, ext, seed=len(seq))
    call = call_of(wl, device_plan=device_plan)
    call.run_plan()
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    pieces, merges = expected(wl, cus)
    print(f"[split] L={seq[:4]} ext={ext[:4]}: {len(pieces)} pieces, {len(merges)} merges",
          flush=True)
    if not call.route.split:
        assert not merges
        return
    got_p, got_m = lists(call)
    np.testing.assert_array_equal(got_p[:len(pieces)], np.array(pieces).reshape(-1, 8))
    assert (got_p[len(pieces):] == 0).all()
    np.testing.assert_array_equal(got_m[:len(merges)], np.array(merges).reshape(-1, 8))
    assert (got_m[len(merges):] == 0).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("seq,ext", [([3000], [100]), ([1537, 4097, 2049], [11, 12, 90]),
                                     ([2500, 700, 3300, 40], [300, 1, 12, 5]),
                                     ([2600], [700])])
def test_split_steps_match_the_oracle(gpu, seq, ext, fp8):
    wl = case(gpu, seq, ext, seed=sum(ext), fp8=fp8)
    host = call_of(wl)
    out = host.run().clone()
    _, merges = lists(host)
    print(f"[split] L={seq} ext={ext} fp8={fp8}: {int((merges[:, 4] > 0).sum())} entries cut",
          flush=True)
    assert (merges[:, 4] > 0).any()
    assert_attn_close(out, restatement(wl), what="split")
    step = slot_based_attention(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                                k_scale=wl.k_scale, v_scale=wl.v_scale)
    dev = call_of(wl, device_plan=True).run()
    torch.cuda.synchronize()
    assert torch.equal(step, out) and torch.equal(dev, out)


@pytest.mark.parametrize("hq,hkv", [(8, 1), (4, 4), (40, 2)])
def test_group_sizes_gate_and_amax(gpu, hq, hkv):
    wl = case(gpu, [2900, 1601], [70, 200], hq, hkv, seed=hq)
    plain = call_of(wl).run().clone()
    assert_attn_close(plain, restatement(wl), what=f"G={hq // hkv}")
    gate = module_gate(wl, 256)
    amax = torch.zeros(1, dtype=torch.int32, device=gpu)
    fused = call_of(wl, gate=gate, out_amax=amax).run()
    torch.cuda.synchronize()
    assert_bits_match(fused, plain * F.silu(gate), "gate")
    assert int(amax) == int(fused.abs().max().view(torch.int16))


def test_negative_slot_entries_bsz1(gpu):
    wl = case(gpu, [3000], [64], seed=5)
    wl.batch.req_to_token[wl.rows[0], [0, 1500, 2950]] = -1
    out = call_of(wl).run()
    torch.cuda.synchronize()
    assert_attn_close(out, restatement(wl), what="-1 entries")


def test_captured_split_step_replays(gpu):
    """Replays over other lengths of the same T and B, cut and whole."""
    mk = lambda seq, seed: workloads.build("split", seq, [90, 40], num_q_heads=24, num_kv_heads=4,
                                           head_dim=256, pool_slots=8192, device=gpu, seed=seed,
                                           max_reqs=8)
    live = mk([3000, 900], 1)
    call = call_of(live, device_plan=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call.run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call.run()
    width = live.batch.req_to_token.shape[1]
    for i, seq in enumerate(([2200, 2990], [400, 100], [3000, 41], [2200, 2990])):
        wl = mk(seq, 20 + i)
        live.batch.req_to_token.fill_(-1)
        w = wl.batch.req_to_token.shape[1]
        live.batch.req_to_token[:, :min(w, width)] = wl.batch.req_to_token[:, :width]
        for x, y in ((live.q, wl.q), (live.k_pool, wl.k_pool), (live.v_pool, wl.v_pool),
                     (live.batch.seq_lens, wl.batch.seq_lens),
                     (live.batch.req_pool_indices, wl.batch.req_pool_indices)):
            x.copy_(y)
        torch.cuda.synchronize()
        print(f"[split] replay {i}: L={seq}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        assert_attn_close(call.out, restatement(wl), what=f"replay {i}")


@pytest.mark.parametrize("phases", [False, True])
@pytest.mark.parametrize("fp8", [False, True])
def test_lengths_that_change_after_planning(gpu, fp8, phases):
    """A plan kept on a batch, or on a call whose phases run one by one, with other
    seq_lens in place: contexts beyond the planned pieces, and contexts that leave
    pieces and whole entries without keys."""
    mk = lambda seq, seed: workloads.build("split", seq, [90, 40], num_q_heads=24, num_kv_heads=4,
                                           head_dim=256, pool_slots=16384, device=gpu, seed=seed,
                                           max_reqs=8, kv_fp8=fp8)
    live = mk([3000, 2000], 1)
    width = 8000
    table = torch.full((8, width), -1, dtype=torch.long, device=gpu)
    table[:, :live.batch.req_to_token.shape[1]] = live.batch.req_to_token
    live.batch.req_to_token = table
    call = call_of(live)
    kw = dict(scaling=live.scale, k_scale=live.k_scale, v_scale=live.v_scale)
    run = lambda: slot_based_attention(live.q, live.k_pool, live.v_pool, live.batch, **kw)
    first = (call.run_extend(), call.out)[1] if phases else run()
    assert_attn_close(first, restatement(live), what="as planned")
    r = (call if phases else live.batch._tf_attn_step_plans.popitem()[1]).route
    assert r.split
    if not phases:
        run()   # (planned again, kept on the batch)
    for i, seq in enumerate(([7000, 5000], [2980, 150], [100, 41], [700, 6000])):
        wl = mk(seq, 20 + i)
        table.fill_(-1)
        w = wl.batch.req_to_token.shape[1]
        table[:, :w] = wl.batch.req_to_token
        for x, y in ((live.q, wl.q), (live.k_pool, wl.k_pool), (live.v_pool, wl.v_pool),
                     (live.batch.seq_lens, wl.batch.seq_lens),
                     (live.batch.req_pool_indices, wl.batch.req_pool_indices)):
            x.copy_(y)
        if fp8:
            live.k_scale.copy_(wl.k_scale)
            live.v_scale.copy_(wl.v_scale)
        # scratch that holds anything but finite numbers
        torch.empty(1 << 26, dtype=torch.float32, device=gpu).fill_(float("nan"))
        torch.cuda.synchronize()
        print(f"[split] lengths {seq} after the plan", flush=True)
        out = (call.run_extend(), call.out)[1] if phases else run()
        torch.cuda.synchronize()
        assert_attn_close(out, restatement(wl), what=f"L={seq}")


def test_plan_without_room_for_merges_stays_whole(gpu):
    """tf_attn_plan_blocks with fewer merge entries than the split needs."""
    from tokenfactory_amd import _native
    wl = case(gpu, [6100, 1700, 5300], [211, 37, 100], seed=3)
    call = call_of(wl)
    call.run_plan()
    call._plan_lists()
    _, merges = lists(call)
    r, need = call.route, int((merges[:, 4] > 0).sum())
    assert need > 1
    for room in (need, need - 1):
        got = torch.full((8 * (r.n_pieces + room),), -1, dtype=torch.int32, device=gpu)
        _native.call("tf_attn_plan_blocks", call._meta.data_ptr(), call.n_work, None, None, 0,
                     24, 4, 1, 0, None, 0, got.data_ptr(), r.n_pieces,
                     got.data_ptr() + 32 * r.n_pieces, room, wl.batch.seq_lens.data_ptr(), 0,
                     wl.batch.req_to_token.shape[1], r.key_bytes,
                     torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = got.cpu().numpy()
        cut = (got[:8 * r.n_pieces].reshape(-1, 8)[:, 7] > 0).sum()
        assert (cut > 0) == (room == need)
        assert (got[8 * r.n_pieces:].reshape(-1, 8)[:, 4] > 0).sum() == (need if cut else 0)
