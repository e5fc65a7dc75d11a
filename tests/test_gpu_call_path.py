"""GPU: the pieces behind the native call path against the oracle or a plain restatement: bit packing with
offsets worked out on the device, and the tables of a planned batch."""
import numpy as np
import pytest
import torch

import oracle
from helpers import make_ragged_masks, max_abs, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1], [64], [65], [0, 63, 1, 64, 0, 129, 8], [1600000, 77], list(range(1024)),
                                  [3] * 1025])   # 1025 segments: beyond the kernel that scans by itself
@pytest.mark.parametrize("bitorder", ["big", "little"])
@pytest.mark.parametrize("indptr_type", [torch.int32, torch.int64])
@pytest.mark.parametrize("first", [0, 5])           # where the first segment begins: unaligned reads
def test_segment_packbits_offsets_on_the_device(dev, lens, bitorder, indptr_type, first):
    import flashomni_amd as fo
    rng = np.random.default_rng(len(lens) + lens[0])
    indptr = first + np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    x = rng.integers(0, 3, size=int(indptr[-1]) + 2).astype(np.uint8)    # bytes: any non-zero is a 1
    y, p = fo.segment_packbits(torch.from_numpy(x).to(dev), torch.from_numpy(indptr).to(dev, indptr_type), bitorder)
    parts = [oracle.packbits(x[a:b] != 0, bitorder) for a, b in zip(indptr[:-1], indptr[1:])]
    assert p.dtype == torch.int32 and y.dtype == torch.uint8
    np.testing.assert_array_equal(p.cpu().numpy(), np.concatenate([[0], np.cumsum([len(v) for v in parts])]))
    np.testing.assert_array_equal(y.cpu().numpy(), np.concatenate(parts))


@pytest.mark.parametrize("batch", [1, 3, 399, 400, 401])    # 400 requests travel as kernel arguments, more are copied
@pytest.mark.parametrize("packed", [False, True])
def test_plan_tables(dev, batch, packed):
    import flashomni_amd as fo
    rng = np.random.default_rng(batch)
    ql, kl = rng.integers(0, 700, batch), rng.integers(0, 900, batch)
    ql[0] = 130
    qo, kv = (torch.from_numpy(np.concatenate([[0], np.cumsum(v)]).astype(np.int32)) for v in (ql, kl))
    hq, hkv = 6, 2 if packed else 6
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(256 << 20, dtype=torch.uint8, device=dev))
    for _ in range(2):                               # planned twice: the second behind the first in the pinned mirror
        w.plan(qo, kv, hq, hkv, 128, q_data_type=torch.bfloat16)
    nq, nk, rows = -(-ql // 128), -(-kl // 128), -(-ql * (hq // hkv) // 128)
    cum = lambda v: np.concatenate([[0], np.cumsum(v)])
    exp = [qo.numpy(), kv.numpy(), cum(nq), cum(nk), cum(nq * hq), cum(nq * nk * hq), np.repeat(np.arange(batch), rows),
           np.concatenate([np.arange(r) for r in rows])]
    for i, e in enumerate(exp):
        np.testing.assert_array_equal(w._planned.table(i).cpu().numpy(), e, err_msg=str(i))


def _small_problem(dev, lens, heads, seed):
    m = make_ragged_masks(lens, lens, heads, 0.7, 0.6, seed=seed)
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(sum(lens), heads, 128, generator=g).to(torch.bfloat16) for _ in range(3))
    sym = [torch.from_numpy(m[n]) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    exp = oracle.sparse_attention(q, k, v, *sym, m["qo_indptr"], m["kv_indptr"], out=torch.zeros_like(q))
    return m, [t.to(dev) for t in (q, k, v)], [t.to(dev) for t in sym], exp


@pytest.mark.parametrize("lens,heads", [([384, 130], 2), ([4500], 40)])     # rows from the symbols, a decoded list
@pytest.mark.parametrize("plan_on_side,how", [(True, "eager"), (False, "eager"), (True, "captured"), (False, "captured"),
                                              (True, "captured on the planning stream")])
def test_plan_and_run_on_two_streams(dev, lens, heads, plan_on_side, how):
    """The tables of a plan are complete when another stream reads them, although plan() does not wait: the
    planning stream is busy when plan() queues them (the memory they land in held other values).  A captured run
    may be replayed on any stream: the tables are complete before it is recorded."""
    import flashomni_amd as fo
    m, qkv, sym, exp = _small_problem(dev, lens, heads, 8)
    qo, kv = torch.from_numpy(m["qo_indptr"]), torch.from_numpy(m["kv_indptr"])
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(qo, kv, heads, heads, 128, q_data_type=torch.bfloat16)
    w.run(*qkv, *sym)          # (the kernels are loaded before the clock matters)
    side, third = torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)
    planner, runner = (side, torch.cuda.current_stream()) if plan_on_side else (torch.cuda.current_stream(), side)
    out = torch.zeros(qkv[0].shape, dtype=torch.bfloat16, device=dev)
    torch.cuda.synchronize(dev)
    with torch.cuda.stream(planner):
        busy = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        for i in range(20):
            busy.fill_(i)
        w.plan(qo, kv, heads, heads, 128, q_data_type=torch.bfloat16)
    if how == "captured on the planning stream":
        third = side
    if how == "eager":
        with torch.cuda.stream(runner):
            w.run(*qkv, *sym, out=out)
        runner.synchronize()
    else:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(third):
            graph.capture_begin()
            w.run(*qkv, *sym, out=out)
            graph.capture_end()
        with torch.cuda.stream(runner):
            graph.replay()
        runner.synchronize()
    got = out.cpu()
    assert max_abs(got, exp) <= 2e-2 and rel_l2(got, exp) <= 1e-2
    torch.cuda.synchronize(dev)


def test_plan_tables_outlive_the_plan_on_another_stream(dev):
    """Planned on the current stream, run on a busy side stream, planned again: the memory of the first plan's
    tables is not handed out before the side stream's launch has read them."""
    import flashomni_amd as fo
    m, qkv, sym, exp = _small_problem(dev, [384, 130], 2, 9)
    qo, kv = torch.from_numpy(m["qo_indptr"]), torch.from_numpy(m["kv_indptr"])
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(qo, kv, 2, 2, 128, q_data_type=torch.bfloat16)
    side = torch.cuda.Stream(device=dev)
    out = torch.zeros(qkv[0].shape, dtype=torch.bfloat16, device=dev)
    torch.cuda.synchronize(dev)
    with torch.cuda.stream(side):
        busy = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        for i in range(20):
            busy.fill_(i)
        w.run(*qkv, *sym, out=out)
    at, ints = w._planned.tables.data_ptr(), w._planned.tables.numel()
    w._planned = None
    again = [torch.empty(ints, dtype=torch.int32, device=dev) for _ in range(64)]
    assert all(t.data_ptr() != at for t in again)
    del again
    side.synchronize()
    assert max_abs(out.cpu(), exp) <= 2e-2


def test_plan_is_refused_under_capture(dev):
    import flashomni_amd as fo
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    ip = torch.tensor([0, 384], dtype=torch.int32)
    graph, s = torch.cuda.CUDAGraph(), torch.cuda.Stream(device=dev)
    torch.cuda.synchronize(dev)
    with torch.cuda.stream(s):
        graph.capture_begin()
        with pytest.raises(RuntimeError, match="cannot be captured"):
            w.plan(ip, ip, 2, 2, 128, q_data_type=torch.bfloat16)
        torch.zeros(8, device=dev)
        graph.capture_end()
    w.plan(ip, ip, 2, 2, 128, q_data_type=torch.bfloat16)


@pytest.mark.parametrize("stream", ["default", "side"])
@pytest.mark.parametrize("capturing", [False, True])
def test_plans_beyond_the_pinned_mirror(dev, stream, capturing):
    """Plans one behind the other in a small pinned mirror, many laps of it, queued behind a busy stretch: every
    copy arrives as it was planned, no other stream is waited for, and another thread may be capturing."""
    import threading

    import flashomni_amd as fo
    ws = torch.empty(128 << 20, dtype=torch.uint8, device=dev)
    batches = [torch.tensor(v, dtype=torch.int32) for v in ([0, 300, 640], [0, 1, 200, 2000], [0, 5000])]

    def plan(w, ip):
        w.plan(ip, ip, 4, 4, 128, q_data_type=torch.bfloat16)

    def arrays(info, workspace, ip):      # (what lies between the aligned arrays is not defined)
        n, rows = info[0], info[1]
        parts = [(info[4], 4 * n), (info[5], 4 * n), (info[6], 4 * n), (info[8], 4 * ip.numel()), (info[9], 4)]
        if info[14]:
            parts += [(info[7], 4 * rows + 4), (info[12], n)]
        return [workspace[a:a + size].tolist() for a, size in parts]

    exp = []
    for ip in batches:
        w = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
        plan(w, ip)
        exp.append((w._plan_info.tolist(), arrays(w._plan_info.tolist(), w._int_workspace_buffer.cpu(), ip)))
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
    w.reset_workspace_buffer(ws, torch.zeros(40960, dtype=torch.uint8, device=dev))
    other, third = torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)
    planner = torch.cuda.current_stream(dev) if stream == "default" else torch.cuda.Stream(device=dev)
    busy = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
    copies = torch.zeros(200, 40960, dtype=torch.uint8, device=dev)
    with torch.cuda.stream(planner):     # (torch itself cannot take memory from the device while a thread captures)
        plan(w, batches[1])
        plan(w, batches[2])
    torch.cuda.synchronize(dev)
    graph, begun, planned, errors = torch.cuda.CUDAGraph(), threading.Event(), threading.Event(), []

    def capture():
        try:
            with torch.cuda.stream(third):
                graph.capture_begin()
                begun.set()
                planned.wait(60)
                torch.zeros(8, device=dev)
                graph.capture_end()
        except Exception as e:
            errors.append(e)
            begun.set()

    thread = threading.Thread(target=capture) if capturing else None
    if thread:
        thread.start()
        begun.wait(60)
    seen = []
    with torch.cuda.stream(other):
        for i in range(300):                      # ~0.1 s
            busy.fill_(i & 1)
    with torch.cuda.stream(planner):
        for i in range(200):
            w._int_workspace_buffer.zero_()
            plan(w, batches[i % 3])
            copies[i].copy_(w._int_workspace_buffer)
            seen.append(w._plan_info.tolist())
    waited = other.query() if not capturing else False
    planned.set()
    if thread:
        thread.join(60)
    torch.cuda.synchronize(dev)
    assert not errors, errors
    assert not waited, "the other stream was waited for"
    for i, (info, got) in enumerate(zip(seen, copies.cpu())):
        assert info == exp[i % 3][0]
        assert arrays(info, got, batches[i % 3]) == exp[i % 3][1], i


@pytest.mark.parametrize("lens", [[5] * 401, [128 * 3000 - 7, 1], [700]])   # copied; several workgroups; one
@pytest.mark.parametrize("capturing", [False, True])
def test_tables_read_from_another_stream(dev, lens, capturing):
    """The tables of a plan queued on a busy side stream, read from another stream, also while the planning stream
    is being captured (then the host waits for the launch's word)."""
    import flashomni_amd as fo
    qo = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
    kv = torch.arange(len(lens) + 1, dtype=torch.int32) * 64
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(256 << 20, dtype=torch.uint8, device=dev))
    side = torch.cuda.Stream(device=dev)
    torch.cuda.synchronize(dev)
    with torch.cuda.stream(side):
        busy = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        for i in range(20):
            busy.fill_(i)
        w.plan(qo, kv, 2, 2, 128, q_data_type=torch.bfloat16)
    got = [torch.empty_like(w._planned.tables) for _ in range(2)]
    graph = torch.cuda.CUDAGraph()
    if capturing:
        with torch.cuda.stream(side):
            graph.capture_begin(capture_error_mode="relaxed")
    w._planned.table(0)
    got[0].copy_(w._planned.tables)
    if capturing:
        with torch.cuda.stream(side):
            got[1].copy_(w._planned.tables)
            graph.capture_end()
    torch.cuda.synchronize(dev)
    rows = -(-np.asarray(lens) // 128)
    at = w._planned._table_at
    exp = {0: qo.numpy(), 1: kv.numpy(), 2: np.repeat(np.arange(len(lens)), rows),
           3: np.concatenate([np.arange(r) for r in rows])}
    for i, e in exp.items():
        np.testing.assert_array_equal(got[0][at[i]:at[i] + len(e)].cpu().numpy(), e, err_msg=str(i))
