"""Row blocks of the streaming kernel (tf_attn_rows, tf_attn_plan_blocks).

Requests with few new tokens, and every row at head dims other than 256, run the
streaming kernel in units of 16 or 32 query rows with a causal limit per
row.  Checked against the oracle with the decode and extend tests' tolerance at
the edges of those units, the block lists against a direct restatement, and a
captured step against the eager one over batches whose rows take other routes.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from tests.helpers import assert_attn_close, restatement, small_case
from tests.test_gpu_gate import assert_bits_match, module_gate
from tokenfactory_amd import slot_based_attention, workloads
from tokenfactory_amd.attention import MAX_ROW_ITEMS, SHORT_ROWS, TINY_CONTEXT, SlotAttentionCall

pytestmark = pytest.mark.gpu


def run(wl, **kw):
    return slot_based_attention(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                                k_scale=wl.k_scale, v_scale=wl.v_scale, **kw)


def case(gpu, seq, ext, hq, hkv, d, seed, fp8=False):
    return workloads.build("rows", seq, ext, num_q_heads=hq, num_kv_heads=hkv, head_dim=d,
                           pool_slots=2 * sum(seq) + 64, device=gpu, seed=seed, kv_fp8=fp8)


def check(wl, what):
    print(f"[rows] {what} D={wl.head_dim} ext={wl.ext_lens} L={wl.seq_lens} "
          f"Hq={wl.num_q_heads} Hkv={wl.num_kv_heads}", flush=True)
    out = run(wl)
    torch.cuda.synchronize()
    assert_attn_close(out, restatement(wl), what=what)
    return out


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,exts", [
    (24, 4, [2, 2, 2]),             # 12 rows: one group
    (24, 4, [2, 5, 3, 1]),          # up to 30 rows, a decode row among them
    (24, 4, [6, 10, 2, 1, 11, 40]),  # two blocks (36, 60 rows) beside the extend kernel's
    (4, 4, [16, 17, 32, 33, 64, 65]),
    (16, 1, [2, 4, 3, 1]),
    (40, 2, [3, 2, 1]),             # G = 20: 60, 40 rows and two blocks for a decode row
])
def test_few_new_tokens(gpu, hq, hkv, exts, fp8):
    pre = [0, 700, 13, 2100, 40, 305]
    seq = [e + p for e, p in zip(exts, pre)]
    check(case(gpu, seq, exts, hq, hkv, 256, sum(exts), fp8), f"fp8={fp8}")


@pytest.mark.parametrize("L", [3, 16, 17, 18, 33, 63, 64, 65, 1000])
def test_context_tile_edges(gpu, L):
    """The last tile holds keys that only the last tokens see."""
    check(case(gpu, [L], [3], 24, 4, 256, L), "one request")
    check(case(gpu, [L, 2049], [3, 2], 24, 4, 256, L), "two requests")


@pytest.mark.parametrize("d", [8, 40, 64, 72, 128, 136, 200, 248])
@pytest.mark.parametrize("fp8", [False, True])
def test_other_head_dims(gpu, d, fp8):
    """Prefills of several blocks, extends and decodes; an fp8 pool whose head
    dim is not a multiple of 16 stays on the one-wave-per-row kernel."""
    check(case(gpu, [90, 400, 7, 1900, 64], [90, 1, 3, 1, 20], 8, 2, d, d, fp8), "mixed")
    check(case(gpu, [500, 31], [1, 1], 20, 1, d, d, fp8), "decode, G = 20")


@pytest.mark.parametrize("d,fp8", [(64, False), (128, False), (128, True), (72, False)])
@pytest.mark.parametrize("longest", [1, TINY_CONTEXT, TINY_CONTEXT + 1])
def test_tiny_contexts(gpu, d, fp8, longest):
    """Decodes on either side of TINY_CONTEXT, eager; a step captured on tiny contexts
    replays on long ones."""
    seq = [longest, 1, max(longest - 1, 1)]
    wl = case(gpu, seq, [1] * 3, 8, 2, d, d, fp8)
    check(wl, f"longest {longest}")
    gate = module_gate(wl, d)
    amax = torch.zeros(1, dtype=torch.int32, device=gpu)
    fused = run(wl, gate=gate, out_amax=amax)
    want = (run(wl) * F.silu(gate)).float()
    # one bf16 ulp of silu (at most 2^-7 relative) and the product's two roundings
    # (2^-9 each), as in assert_bits_match, whose count of differing elements
    # (one in a thousand) needs more elements than these few rows have
    assert ((fused.float() - want).abs() <= 3 * 2.0 ** -8 * want.abs()).all()
    assert int(amax) == int(fused.abs().max().view(torch.int16))
    long = workloads.build("rows", [600, 3, 77], [1] * 3, num_q_heads=8, num_kv_heads=2, head_dim=d,
                           pool_slots=wl.k_pool.shape[0] + 2000, device=gpu, seed=d, kv_fp8=fp8)
    table = torch.full_like(long.batch.req_to_token, -1)
    wl.k_pool, wl.v_pool, wl.batch.req_to_token = long.k_pool, long.v_pool, table
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = run(wl)
    wl.q.copy_(long.q)
    table.copy_(long.batch.req_to_token)
    wl.batch.req_pool_indices.copy_(long.batch.req_pool_indices)
    wl.batch.seq_lens.copy_(long.batch.seq_lens)
    if fp8:
        wl.k_scale.copy_(long.k_scale)
        wl.v_scale.copy_(long.v_scale)
    for i in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert_attn_close(out, restatement(long), what=f"replay {i}")


def test_strided_q_out_gate_and_amax(gpu):
    for d in (256, 128):
        wl = case(gpu, [50, 700, 9, 300], [2, 5, 1, 3], 24, 4, d, d)
        want = run(wl)
        wide = torch.zeros(wl.q.shape[0], 2, 24, d, dtype=torch.bfloat16, device=gpu)
        wide[:, 0] = wl.q
        out = torch.zeros_like(wide)
        wl.q = wide[:, 0]
        got = run(wl, out=out[:, 1])
        assert torch.equal(got, want) and (out[:, 0] == 0).all()
        gate = module_gate(wl, d)
        amax = torch.zeros(1, dtype=torch.int32, device=gpu)
        fused = run(wl, gate=gate, out_amax=amax)
        torch.cuda.synchronize()
        assert_bits_match(fused, want * F.silu(gate), f"gate D={d}")
        assert int(amax) == int(fused.abs().max().view(torch.int16))


@pytest.mark.parametrize("d", [256, 128, 200])
@pytest.mark.parametrize("workgroups", [1, 3, 7, 40, 100, 513])
def test_units_cut_anywhere(gpu, d, workgroups):
    """Grids with fewer and with more workgroups than units, whose ranges start and
    end inside units: first, inner and last units of a workgroup."""
    wl = case(gpu, [30, 700, 9, 300, 90, 33], [2, 5, 3, 1, 2, 6], 8, 2, d, d)
    got = run(wl, decode_workgroups=workgroups)
    assert_attn_close(got, restatement(wl), what=f"{workgroups} workgroups")


def expected_lists(ext_lens, group, hkv, unit, max_rows):
    starts = np.concatenate([[0], np.cumsum(ext_lens)[:-1]]).tolist()
    blocks = [(b, starts[b], 1, r) for b, e in enumerate(ext_lens) if e == 1
              for r in range(0, group, unit)]
    order = sorted((b for b, e in enumerate(ext_lens) if e > 1), key=lambda b: -ext_lens[b])
    pieces = []
    for b in order:
        rows = ext_lens[b] * group
        for t in reversed(range(-(-rows // 256))):
            if rows <= max_rows:
                blocks += [(b, starts[b], ext_lens[b], r)
                           for r in range(256 * t, min(256 * t + 256, rows), unit)]
            else:
                pieces += [(b, h, 256 * t, starts[b], ext_lens[b], 0, 0, 0) for h in range(hkv)]
    return blocks, pieces


@pytest.mark.parametrize("device_plan", [False, True])
@pytest.mark.parametrize("d,lens", [(256, [3, 1, 700, 1, 22, 1, 10, 11]), (128, [300, 1, 5, 70]),
                                    (256, [2] * 700 + [1] * 500 + [30])])
def test_block_lists(gpu, d, lens, device_plan):
    hq, hkv = 24, 4
    wl = small_case([e + 3 for e in lens], lens, hq=hq, hkv=hkv, d=d, seed=len(lens), device=gpu,
                    dtype=torch.bfloat16)
    call = SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                             device_plan=device_plan)
    call.run_plan()
    torch.cuda.synchronize()
    r = call.route
    blocks, pieces = expected_lists(lens, hq // hkv, hkv, 16 * r.row_groups, r.max_rows)
    got = call._lists.cpu().numpy()
    gb = got[:4 * r.n_blocks].reshape(-1, 4)
    gp = got[4 * r.n_blocks:].reshape(-1, 8)
    assert len(blocks) <= r.n_blocks and len(pieces) <= max(r.n_pieces, 0)
    np.testing.assert_array_equal(gb[:len(blocks)], np.array(blocks).reshape(-1, 4))
    assert (gb[len(blocks):, 0] == -1).all()
    np.testing.assert_array_equal(gp[:len(pieces)], np.array(pieces).reshape(-1, 8))
    assert (gp[len(pieces):] == 0).all()


@pytest.mark.parametrize("exts,hq,hkv,d", [
    ([1100, 700, 1, 900], 64, 4, 64),            # 1351 blocks: one launch
    ([2500], 64, 1, 32),                         # 5000: three
    ([1] * 2060 + [40, 7] * 4, 8, 2, 64),        # 2084: decodes and extends past the 2048th
])
def test_more_blocks_than_one_launch_takes(gpu, exts, hq, hkv, d):
    """Above 2048 blocks the rows kernel is launched over parts of the list."""
    wl = case(gpu, [e + i % 5 for i, e in enumerate(exts)], exts, hq, hkv, d, len(exts))
    call = SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale)
    out = call.run()
    torch.cuda.synchronize()
    blocks = call._lists.cpu().numpy()[:4 * call.route.n_blocks].reshape(-1, 4)
    real = int((blocks[:, 0] >= 0).sum())
    assert real == call.route.n_blocks == sum(-(-e * (hq // hkv) // 32) for e in exts)
    assert (real > MAX_ROW_ITEMS) == (len(exts) != 4)
    if len(exts) > 4:
        assert (blocks[MAX_ROW_ITEMS:, 2] == 1).any() and (blocks[MAX_ROW_ITEMS:, 2] > 1).any()
    assert torch.equal(check(wl, f"{real} blocks"), out)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("groups,ext,pre", [
    (0, [10] * 66, 30), (1, [4] * 130 + [1] * 3 + [70], 25), (0, [7] * 300 + [1] * 280, 20),
    (1, [2] * 5 + [1] * 40, 200), (2, [5] * 16, 900)])
def test_every_way_of_short_extends(gpu, groups, ext, pre, fp8):
    """The extend kernel, units of 16 and of 32 rows, as the rule chooses them, and
    a device-planned call (whose lists have room for other lengths)."""
    hq, hkv = 24, 4
    seq = [e + pre + i % 7 for i, e in enumerate(ext)]
    wl = case(gpu, seq, ext, hq, hkv, 256, len(ext), fp8)
    calls = [SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                               k_scale=wl.k_scale, v_scale=wl.v_scale, device_plan=dev)
             for dev in (False, True)]
    if not fp8:
        assert calls[0].route.row_groups == groups
    outs = [run(wl)] + [c.run() for c in calls]
    torch.cuda.synchronize()
    ref = restatement(wl)
    for out in outs:
        assert_attn_close(out, ref, what=f"{len(ext)} requests")


def test_captured_step_replays_over_other_routes(gpu):
    """Replays over batches with the same T and B whose requests fall on either
    side of SHORT_ROWS: every replay against the oracle."""
    kw = dict(hq=24, hkv=4, d=256, dtype=torch.bfloat16, pool=8192, device=gpu)
    splits = [([900, 300, 1500, 41], [4, 1, 10, 30]), ([900, 300, 1500, 41], [30, 9, 5, 1]),
              ([900, 300, 1500, 41], [2, 40, 2, 1]), ([900, 300, 1500, 41], [4, 1, 10, 30])]
    assert 10 * 6 <= SHORT_ROWS < 30 * 6
    live = small_case(*splits[0], seed=1, **kw)
    call = SlotAttentionCall(live.q, live.k_pool, live.v_pool, live.batch, scaling=live.scale,
                             device_plan=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call.run()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call.run()
    for i, (seq, ext) in enumerate(splits):
        wl = small_case(seq, ext, seed=10 + i, **kw)
        for x, y in ((live.q, wl.q), (live.k_pool, wl.k_pool), (live.v_pool, wl.v_pool),
                     (live.batch.req_to_token, wl.batch.req_to_token),
                     (live.batch.seq_lens, wl.batch.seq_lens),
                     (live.batch.req_pool_indices, wl.batch.req_pool_indices),
                     (live.batch.extend_lens_tensor, wl.batch.extend_lens_tensor)):
            x.copy_(y)
        torch.cuda.synchronize()
        print(f"[rows] replay {i}: ext={ext}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        assert_attn_close(call.out, restatement(wl), what=f"replay {i}")
