"""Memory of attention calls across streams and graphs.

A call launched on a stream of its own may be dropped while that stream still
has to run it: everything it allocates must belong to that stream, so that no
other stream's allocation can be given the memory meanwhile.
"""
import pytest
import torch

from tests.helpers import small_case
from tokenfactory_amd import attention, slot_based_attention, workloads
from tokenfactory_amd.attention import SlotAttentionCall

pytestmark = pytest.mark.gpu


def calls(wl, **kw):
    return SlotAttentionCall(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale,
                             k_scale=wl.k_scale, v_scale=wl.v_scale, **kw)


@pytest.mark.parametrize("device_plan", [False, True])
@pytest.mark.parametrize("seq,ext,d", [([900, 300, 1500], [4, 1, 10], 256),   # row blocks
                                       ([3000, 40], [100, 1], 256),           # key split
                                       ([300, 700], [70, 1], 128)])
def test_dropped_call_leaves_no_memory_to_other_streams(gpu, seq, ext, d, device_plan):
    wl = small_case(seq, ext, hq=24, hkv=4, d=d, seed=sum(ext), device=gpu, dtype=torch.bfloat16)
    want = calls(wl, device_plan=device_plan).run().clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    out = torch.empty_like(wl.q)
    call = calls(wl, device_plan=device_plan, stream=s, out=out)
    held = {n: t for n, t in (("lists", call._lists), ("meta", call._meta), ("ws", call._scratch()))
            if t is not None}
    spans = {n: (t.data_ptr(), t.data_ptr() + t.numel() * t.element_size(), t.numel(), t.dtype)
             for n, t in held.items()}
    assert "lists" in spans and "meta" in spans
    call.run()
    del call, held
    other = []   # this stream's allocations of the same sizes, overwritten at once
    for name, (lo, hi, n, dtype) in spans.items():
        for _ in range(4):
            t = torch.empty(n, dtype=dtype, device=gpu).fill_(77)
            other.append(t)
            assert t.data_ptr() >= hi or t.data_ptr() + n * t.element_size() <= lo, name
    s.synchronize()
    assert torch.equal(out, want)


def test_inputs_converted_on_the_launch_stream(gpu):
    """q with strided heads is copied, and scales of another shape are converted,
    by the stream that reads them."""
    wl = workloads.build("conv", [500, 90], [1, 1], num_q_heads=24, num_kv_heads=4, head_dim=256,
                         pool_slots=2048, device=gpu, seed=3, kv_fp8=True)
    want = calls(wl).run().clone()
    s = torch.cuda.Stream()
    strided = torch.zeros((2, 24, 512), dtype=torch.bfloat16, device=gpu)
    strided[:, :, :256] = wl.q
    wl.q = strided[:, :, :256]
    wl.k_scale, wl.v_scale = wl.k_scale.double(), wl.v_scale.double()
    s.wait_stream(torch.cuda.current_stream())
    call = calls(wl, stream=s)
    spans = [(t.data_ptr(), t.numel(), t.dtype) for t in (call.q, call.k_scale, call.v_scale)]
    out = call.run()
    del call
    for ptr, n, dtype in spans:
        for _ in range(4):
            assert torch.empty(n, dtype=dtype, device=gpu).fill_(float("nan")).data_ptr() != ptr
    s.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("planned_by", ["other", "own"])
def test_dropped_batch_leaves_no_memory_to_its_first_stream(gpu, planned_by):
    """The step plan kept on a batch is read by every stream that calls with the
    batch: its memory is not reused before the last of them is done."""
    wl = small_case([900, 300, 3000], [4, 1, 100], hq=24, hkv=4, d=256, seed=7, device=gpu,
                    dtype=torch.bfloat16)
    run = lambda: slot_based_attention(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale)
    want = run().clone()
    plan, = wl.batch._tf_attn_step_plans.values()
    if planned_by == "own":   # made on this stream, first planned and read by the other
        plan._planned_on = plan._event = None
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        torch.cuda._sleep(50_000_000)   # the stream is busy while the batch goes away
        out = run()
    spans = [(t.data_ptr(), t.numel()) for t in (plan.meta, plan.lists)]
    del plan
    wl.batch._tf_attn_step_plans.clear()
    other = [torch.empty(n, dtype=torch.int32, device=gpu).fill_(77) for _, n in spans
             for _ in range(4)]
    assert not {t.data_ptr() for t in other} & {p for p, _ in spans}
    s.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("kept", [False, True])
@pytest.mark.parametrize("seq,ext,d", [([700, 900], [1, 1], 128), ([900, 1500], [4, 10], 256),
                                       ([2000, 900], [1, 1], 256),
                                       ([3000, 2000, 50], [100, 1, 1], 256)])   # overlapped
def test_captured_call_owns_its_scratch(gpu, seq, ext, d, kept):
    """Replays write neither the stream's shared scratch nor what became of it
    after a later call on the same stream needed more."""
    kw = dict(hq=24, hkv=4, d=d, dtype=torch.bfloat16, device=gpu)
    wl = small_case(seq, ext, seed=d, **kw)
    run = lambda: slot_based_attention(wl.q, wl.k_pool, wl.v_pool, wl.batch, scaling=wl.scale)
    want = run().clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        call = calls(wl, device_plan=max(ext) > 1)
        call.run()   # a warm-up on the capturing stream
    s.synchronize()
    with torch.cuda.graph(graph, stream=s):
        out = call.run() if kept else run()
    keep = call.ws if kept else None
    key = (gpu.index, s.cuda_stream)
    shared = attention._workspaces[key]
    if kept:
        assert keep.data_ptr() != shared.data_ptr()
    shared.fill_(0x5a)
    for i in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), f"replay {i}"
        assert (shared == 0x5a).all(), f"replay {i} wrote the shared scratch"
        with torch.cuda.stream(s):   # eager work on the stream, with more scratch
            attention._workspace(gpu, s.cuda_stream, shared.numel() + (1 << 20))
            calls(wl, decode_workgroups=600 + 100 * i).run()
        torch.cuda.synchronize()
        shared = attention._workspaces[key].fill_(0x5a)
        torch.cuda.synchronize()
