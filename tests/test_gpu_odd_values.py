"""NaN and infinite V values at head dims other than 256: a query row's output
depends on the keys that it sees and on nothing else of the tiles they lie in
(later tokens of the step, repeats past the last key), and an infinite value of
a visible key stays infinite.  Against the float64 loop oracle, which reads
only visible keys.
"""
import math

import pytest
import torch

from tests.helpers import brute, small_case
from tokenfactory_amd import workloads
from tokenfactory_amd.attention import SlotAttentionCall

pytestmark = pytest.mark.gpu

SEQ, EXT = [21, 150, 37, 300], [5, 1, 20, 1]


def case(gpu, d, fp8):
    return workloads.build("odd", SEQ, EXT, num_q_heads=8, num_kv_heads=2, head_dim=d,
                           pool_slots=1024, device=gpu, seed=d, kv_fp8=fp8)


def run(wl, **kw):
    out = SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                            k_scale=wl.k_scale, v_scale=wl.v_scale, **kw).run()
    torch.cuda.synchronize()
    return out.float().cpu()


def check(got, ref, what):
    assert torch.equal(got.isnan(), ref.isnan()), what
    inf = ref.isinf()
    assert torch.equal(got.isinf(), inf) and torch.equal(got[inf], ref[inf]), what
    fin = ref.isfinite()
    # the bounds of tests/helpers.py
    assert ((got - ref).abs()[fin] <= 2e-2 + 1e-2 * ref.abs()[fin]).all(), what


@pytest.mark.parametrize("d,fp8", [(64, False), (128, False), (72, False), (200, False),
                                   (64, True), (128, True), (208, True)])
@pytest.mark.parametrize("where", ["last", "middle", "both"])
def test_rows_depend_on_the_keys_they_see(gpu, d, fp8, where):
    wl = case(gpu, d, fp8)
    values = [math.nan] if fp8 else [math.nan, math.inf, -math.inf]
    for b, (n, e) in enumerate(zip(SEQ, EXT)):
        places = {"last": [n - 1], "middle": [n - e - 9], "both": [3, n - 1]}[where]
        for i, pos in enumerate(places):
            slot = int(wl.batch.req_to_token[wl.rows[b], pos])
            dims = torch.tensor([(7 * b + 3 * i) % d, d - 1 - b], device=gpu)
            odd = torch.full((2,), values[(b + i) % len(values)], device=gpu)
            v = wl.v_pool.view(torch.uint8) if fp8 else wl.v_pool
            v[slot, b % 2, dims] = (odd.to(torch.float8_e4m3fn).view(torch.uint8) if fp8
                                    else odd.to(torch.bfloat16))
    ref = torch.from_numpy(brute(wl)).float()
    assert not ref.isfinite().all() and ref.isfinite().float().mean() > 0.5
    print(f"[odd] D={d} fp8={fp8} {where}", flush=True)
    check(run(wl), ref, "default grid")
    check(run(wl, decode_workgroups=301), ref, "301 workgroups: units cut")
    check(run(wl, decode_workgroups=3), ref, "3 workgroups: whole units")


@pytest.mark.parametrize("workgroups", [0, 2])
@pytest.mark.parametrize("value", [math.inf, math.nan])
def test_gate_and_amax_with_odd_values(gpu, value, workgroups):
    """Of units cut over workgroups and of whole ones: out_amax comes from the outputs
    alone."""
    wl = small_case([40, 100], [4, 1], hq=8, hkv=2, d=128, seed=3, device=gpu,
                    dtype=torch.bfloat16)
    wl.v_pool[int(wl.batch.req_to_token[wl.rows[0], 39]), 0, 5] = value
    gate = torch.randn_like(wl.q)
    amax = torch.zeros(1, dtype=torch.int32, device=gpu)
    plain = run(wl, decode_workgroups=workgroups)
    fused = run(wl, gate=gate, out_amax=amax, decode_workgroups=workgroups)
    g = gate.float().cpu()
    want = plain * torch.nn.functional.silu(g)
    fin = want.isfinite()
    assert not fin.all() and torch.equal(fused.isfinite(), fin)
    # one bf16 ulp of silu and the product's two roundings (tests/test_gpu_gate.py)
    assert ((fused - want).abs()[fin] <= 3 * 2 ** -8 * want.abs()[fin]).all()
    assert int(amax) == 0x7f80 if value == math.inf else int(amax) > 0x7f80


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("seq,ext", [([700, 90], [1, 1]), ([400, 900], [4, 10]),
                                     ([1600, 300], [60, 1]), ([2000], [30])])
def test_visible_values_pass_through_merges(gpu, seq, ext, fp8):
    """At 256 dims: NaN and infinite V values that every row of a request sees, through
    units cut over workgroups, row blocks and split extend entries."""
    wl = workloads.build("odd", seq, ext, num_q_heads=12, num_kv_heads=2, head_dim=256,
                         pool_slots=4096, device=gpu, seed=sum(seq), kv_fp8=fp8)
    values = [math.nan] if fp8 else [math.nan, math.inf, -math.inf]
    for b, n in enumerate(seq):
        for i, v in enumerate(values):
            slot = int(wl.batch.req_to_token[wl.rows[b], 3 + 17 * i])
            pool = wl.v_pool.view(torch.uint8) if fp8 else wl.v_pool
            odd = torch.full((1,), v, device=gpu)
            pool[slot, 0, 5 + 100 * i] = (odd.to(torch.float8_e4m3fn).view(torch.uint8) if fp8
                                          else odd.to(torch.bfloat16))[0]
    ref = torch.from_numpy(brute(wl, dense=True)).float()
    print(f"[odd] D=256 L={seq} ext={ext} fp8={fp8}", flush=True)
    for workgroups in (0, 40):
        check(run(wl, decode_workgroups=workgroups), ref, f"{workgroups} workgroups")
