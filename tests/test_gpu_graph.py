"""run() and the GEMMs under HIP graph capture (the reference declares run() capturable,
flashomni/attention.py:140-141): a captured layer pass must give, on every replay, what the same
calls give eagerly on the inputs of that moment, including symbols rewritten in place between
replays."""
import numpy as np
import pytest
import torch

from helpers import make_ragged_masks

pytestmark = pytest.mark.gpu


def test_captured_layer_pass_replays(dev):
    import flashomni_amd as fo
    H, hidden = 4, 512
    ql = [640, 300]
    nnz = sum(ql)
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g)
    x = rnd(1, nnz, hidden).to(torch.bfloat16).to(dev)
    wq = (rnd(hidden, hidden) * 0.05).to(torch.bfloat16).to(dev)
    bq = (rnd(hidden) * 0.05).to(torch.bfloat16).to(dev)
    wo = (rnd(hidden, hidden) * 0.05).to(torch.bfloat16).to(dev)
    k = rnd(nnz, H, 128).to(torch.bfloat16).to(dev)
    v = rnd(nnz, H, 128).to(torch.bfloat16).to(dev)

    def symbols(seed):
        m = make_ragged_masks(ql, ql, H, 0.7, 0.5, seed=seed)
        return [torch.from_numpy(m[n]) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]

    info, kv_info, info_ip, kv_ip = [t.to(dev) for t in symbols(1)]
    # the GEMMs see the two requests as one batch entry of nnz rows: their symbols index the
    # 128-row blocks of that entry, so give them a single-request packing of the same size
    n_blk = sum(-(-l // 128) for l in ql)
    gemm_bits = torch.from_numpy((np.random.default_rng(2).random(n_blk * H) < 0.7))
    gemm_info = fo.packbits(gemm_bits.to(dev), "little")
    gemm_ip = torch.tensor([0, gemm_info.numel()], dtype=torch.int32, device=dev)

    ws = torch.empty(32 << 20, dtype=torch.uint8, device=dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
    indptr = torch.tensor([0, ql[0], nnz], dtype=torch.int32)
    w.plan(indptr, indptr, H, H, 128, q_data_type=torch.bfloat16)

    q_buf = torch.zeros(1, nnz, hidden, dtype=torch.bfloat16, device=dev)
    o_buf = torch.zeros(nnz, H, 128, dtype=torch.bfloat16, device=dev)
    y_buf = torch.zeros(1, nnz, hidden, dtype=torch.bfloat16, device=dev)

    def layer_pass(q_out, o_out):
        fo.flashomni_gemm(x, wq, H, gemm_info, gemm_ip, 0, bq, out=q_out)
        w.run(q_out.view(nnz, H, 128), k, v, info, kv_info, info_ip, kv_ip, out=o_out)
        return fo.flashomni_gemm_reduction(o_out.view(1, nnz, hidden), wo, H, gemm_info, gemm_ip, 0,
                                           bias=None, is_for_cache=False)

    # warm up on a side stream, then capture
    s = torch.cuda.Stream(device=dev)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        layer_pass(q_buf, o_buf)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y_graph = layer_pass(q_buf, o_buf)
    for replay in range(4):
        # new activations and, from the second replay on, new attention symbols, written in place
        x.copy_(rnd(1, nnz, hidden).to(torch.bfloat16))
        if replay >= 1:
            for dst, src in zip((info, kv_info), symbols(10 + replay)[:2]):
                dst.copy_(src)
        q_buf.zero_(); o_buf.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = (q_buf.clone(), o_buf.clone(), y_graph.clone())
        # the same pass eagerly, into fresh buffers, with program work and a sync in between
        q_ref = torch.zeros_like(q_buf); o_ref = torch.zeros_like(o_buf)
        y_ref = layer_pass(q_ref, o_ref)
        torch.cuda.synchronize()
        for name, a, b in zip(("gemm_q", "attention", "gemm_o"), got, (q_ref, o_ref, y_ref)):
            assert torch.equal(a, b), "replay %d: %s differs from the eager pass" % (replay, name)


def test_captured_long_gemm_o_replays(dev):
    """A GEMM-O launch of many strips, whose order the kernel works out from the flags.  Flags and
    activations are rewritten in place between replays; each replay equals the eager call of that moment."""
    import flashomni_amd as fo
    m, n, heads = 22016, 3072, 24
    g = torch.Generator(device=dev).manual_seed(9)
    x = torch.randn(1, m, n, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    rng = np.random.default_rng(3)
    bits = lambda: torch.from_numpy(rng.random((m // 128) * heads) < 0.3)
    info = fo.packbits(bits().to(dev), "little")
    ip = torch.tensor([0, info.numel()], dtype=torch.int32, device=dev)

    def two_passes():
        cache = fo.flashomni_gemm_reduction(x, w, heads, info, ip, 0, bias=b, is_for_cache=True)
        return cache, fo.flashomni_gemm_reduction(x, w, heads, info, ip, 0, bias=cache, is_for_cache=False)

    s = torch.cuda.Stream(device=dev)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        two_passes()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        cache_g, final_g = two_passes()
    for replay in range(3):
        x.copy_(torch.randn(1, m, n, generator=g, device=dev).to(torch.bfloat16))
        if replay >= 1:
            info.copy_(fo.packbits(bits().to(dev), "little"))
        graph.replay()
        torch.cuda.synchronize()
        got = (cache_g.clone(), final_g.clone())
        ref = two_passes()
        torch.cuda.synchronize()
        for name, a, r in zip(("cache pass", "final pass"), got, ref):
            assert torch.equal(a, r), "replay %d: %s differs from the eager call" % (replay, name)


def test_graph_captured_on_a_warm_stream_survives_workspace_growth(dev):
    """GEMM-Q keeps its tile list in a scratch buffer cached per stream.  A graph captured on a stream
    that already ran the GEMM eagerly must not record that cached buffer: a later, larger eager GEMM on
    the same stream replaces it, and a replay would then write its list into memory that may belong to
    someone else.  Capture on the warm stream, grow the scratch eagerly on it, replay, compare."""
    import flashomni_amd as fo
    from flashomni_amd import gemm as gemm_mod
    heads, hidden = 4, 512
    g = torch.Generator(device=dev).manual_seed(17)
    rng = np.random.default_rng(17)

    def problem(m):
        x = torch.randn(1, m, hidden, generator=g, device=dev).to(torch.bfloat16)
        info = fo.packbits(torch.from_numpy(rng.random(-(-m // 128) * heads) < 0.6).to(dev), "little")
        ip = torch.tensor([0, info.numel()], dtype=torch.int32, device=dev)
        return x, info, ip

    w = (torch.randn(hidden, hidden, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    # (large enough that the tile list is built by the list kernel into the scratch buffer)
    x, info, ip = problem(128 * 300)
    out = torch.zeros(1, x.size(1), hidden, dtype=torch.bfloat16, device=dev)
    s = torch.cuda.Stream(device=dev)
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fo.flashomni_gemm(x, w, heads, info, ip, 0, None, out=out)   # eager warm-up on s
    s.synchronize()
    eager_bufs = {b.data_ptr() for b in gemm_mod._workspaces[(dev.index, s.cuda_stream)]}
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        fo.flashomni_gemm(x, w, heads, info, ip, 0, None, out=out)
    # a much larger GEMM on the same stream: the stream's scratch buffer is replaced
    xb, infob, ipb = problem(128 * 3000)
    with torch.cuda.stream(s):
        big = fo.flashomni_gemm(xb, w, heads, infob, ipb, 0, None)
    s.synchronize()
    bufs = gemm_mod._workspaces[(dev.index, s.cuda_stream)]
    assert len(bufs) >= 2 and eager_bufs <= {b.data_ptr() for b in bufs}, "superseded scratch must stay alive"
    del big, xb
    torch.cuda.empty_cache()
    junk = [torch.full((1 << 20,), 0x5a, dtype=torch.uint8, device=dev) for _ in range(8)]  # reuse freed memory
    for replay in range(3):
        x.copy_(torch.randn(1, x.size(1), hidden, generator=g, device=dev).to(torch.bfloat16))
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        ref = torch.zeros_like(out)
        fo.flashomni_gemm(x, w, heads, info, ip, 0, None, out=ref)
        torch.cuda.synchronize()
        assert torch.equal(out, ref), "replay %d differs from the eager call" % replay
        assert all(bool((j == 0x5a).all()) for j in junk), "a replay wrote outside its own scratch"


def test_captured_short_run_keeps_its_symbols_in_place(dev):
    """A run that takes its rows straight from the symbols keeps a copy of them for a later reuse.  A graph writes
    that copy at every replay: eager runs with larger symbol tensors in between must not move it, and what the
    replays write is what a reuse then decodes."""
    import flashomni_amd as fo
    heads, lens = 2, [384, 130]
    n = sum(lens)
    g = torch.Generator(device=dev).manual_seed(21)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    m = make_ragged_masks(lens, lens, heads, 0.7, 0.6, seed=21)
    t = lambda name: torch.from_numpy(m[name]).to(dev)
    sym = [t(s) for s in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    indptr = torch.from_numpy(m["qo_indptr"])
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(indptr, indptr, heads, heads, 128, q_data_type=torch.bfloat16)
    exp = w.run(q, k, v, *sym, out=torch.zeros_like(q))
    out = torch.zeros_like(q)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        w.run(q, k, v, *sym, out=out)
    longer = [torch.cat([s, torch.full((3000,), 0xff, dtype=torch.uint8, device=dev)]) for s in sym[:2]] + sym[2:]
    assert torch.equal(w.run(q, k, v, *longer, out=torch.zeros_like(q)), exp)
    junk = [torch.full((1 << s,), 0x5a, dtype=torch.uint8, device=dev) for s in range(9, 15) for _ in range(32)]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, exp)
        assert all(bool((j == 0x5a).all()) for j in junk), "a replay wrote outside its own buffers"
    listed = w.run(q, k, v, *sym, out=torch.zeros_like(q), reuse_decoded=True)
    assert float((listed.float() - exp.float()).abs().max()) <= 8e-3


class _ShortList:
    """Two short requests, a wrapper, and the result of every symbol set by the oracle."""

    heads = 2

    def __init__(self, dev, seed):
        import flashomni_amd as fo
        import oracle
        self.dev, heads, lens = dev, self.heads, [384, 130]
        g = torch.Generator().manual_seed(seed)
        q, k, v = (torch.randn(sum(lens), heads, 128, generator=g).to(torch.bfloat16) for _ in range(3))
        names = ("packed_info", "packed_keep", "info_indptr", "keep_indptr")
        masks = [make_ragged_masks(lens, lens, heads, 0.7, 0.5, seed=seed + i) for i in range(3)]
        self.sym = [[torch.from_numpy(m[n]).to(dev) for n in names] for m in masks]
        self.exp = [oracle.sparse_attention(q, k, v, *(m[n] for n in names), m["qo_indptr"], m["kv_indptr"],
                                            out=torch.zeros_like(q)) for m in masks]
        self.full = oracle.sparse_attention(q, k, v, None, None, None, None, masks[0]["qo_indptr"], masks[0]["kv_indptr"],
                                            is_full=True, out=torch.zeros_like(q))
        self.qkv = [t.to(dev) for t in (q, k, v)]
        self.buf = [t.clone() for t in self.sym[0]]    # rewritten in place between replays
        indptr = torch.from_numpy(masks[0]["qo_indptr"])
        self.w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
        self.w.plan(indptr, indptr, heads, heads, 128, q_data_type=torch.bfloat16)
        self.out = torch.zeros_like(self.qkv[0])

    def run(self, sym, reuse=False, is_full=False):
        return self.w.run(*self.qkv, *sym, is_full, out=self.out, reuse_decoded=reuse)

    def capture(self, fn):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            fn()
        return graph

    def check(self, exp, fn, *args, **kw):
        self.out.zero_()
        fn(*args, **kw)
        torch.cuda.synchronize()
        got = self.out.cpu().float()
        assert float((got - exp.float()).abs().max()) <= 2e-2
        assert float((got - exp.float()).norm()) <= 1e-2 * float(exp.float().norm()) + 1e-6


def test_captured_reuse_runs_the_list_of_the_moment(dev):
    """A reuse in a graph runs, at every replay, what the last run or decode before it left, whether that was
    decoded or took its rows from the symbols, eagerly or in another graph; recording it leaves the eager state
    as it was."""
    s = _ShortList(dev, 30)
    a, b, c = s.sym
    s.check(s.exp[0], s.run, a)                                   # rows from the symbols: no list yet
    reuse = s.capture(lambda: s.run(a, reuse=True))
    s.check(s.exp[0], s.run, a, reuse=True)                       # eagerly, before any replay
    s.check(s.exp[0], reuse.replay)
    s.run(b)
    s.check(s.exp[1], reuse.replay)
    s.check(s.exp[1], reuse.replay)
    s.w.decode(*c)
    s.check(s.exp[2], reuse.replay)
    s.check(s.exp[2], s.run, c, reuse=True)
    run = s.capture(lambda: s.run(s.buf))                         # a run in a graph, symbols rewritten in place
    s.check(s.exp[2], s.run, c, reuse=True)                       # recording it has run nothing
    for i in (1, 2, 0):
        for dst, src in zip(s.buf, s.sym[i]):
            dst.copy_(src)
        s.check(s.exp[i], run.replay)
        s.check(s.exp[i], s.run, s.buf, reuse=True)
        s.check(s.exp[i], reuse.replay)
        s.w.decode(*s.sym[(i + 1) % 3])
        s.check(s.exp[(i + 1) % 3], reuse.replay)
    s.run([None] * 4, is_full=True)
    s.check(s.full, reuse.replay)
    s.check(s.full, s.run, [None] * 4, reuse=True, is_full=True)


@pytest.mark.parametrize("heads", [206, 408])
def test_captured_lists_of_three_launches(dev, heads, monkeypatch):
    """The same where what a run left behind is decoded by more than one launch, of which the device decides each: 1030
    candidates, and 2040, eight to a thread, whose parts of rows lie in memory of the plan's."""
    monkeypatch.setattr(_ShortList, "heads", heads)
    test_captured_reuse_runs_the_list_of_the_moment(dev)


@pytest.mark.parametrize("why, heads", [("fp8", 2), ("fp8", 206), ("soft cap", 206), ("small workspace", 2),
                                        ("small workspace", 206), ("no sharing", 2), ("no sharing", 206)])
def test_reuse_behind_a_capture_of_lists_that_are_always_decoded(dev, why, heads, monkeypatch):
    """A plan whose rows are never taken straight from the symbols (fp8, a soft cap on more than 1024 pairs, no room for parts
    of rows) has nothing that could be newer than its list: a capture costs later reuses, eager and recorded ones, no launch."""
    import flashomni_amd as fo
    from flashomni_amd import _lib
    n, soft = 514, why == "soft cap"
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    m = make_ragged_masks([384, 130], [384, 130], heads, 0.7, 0.6, seed=5)
    sym = [torch.from_numpy(m[s]).to(dev) for s in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    indptr = torch.from_numpy(m["qo_indptr"])
    kw = {}
    if why == "fp8":
        q, kw["q_scale"] = fo.quant_fp8_block(q, indptr)
        k, kw["k_scale"] = fo.quant_fp8_block(k, indptr)
    room = 128 << 20
    if why == "small workspace":  # (from 1025 pairs on the launch needs twice as much)
        room = (2 if heads > 2 else 1) * _lib.lib().fo_sparse_fa_split_workspace_bytes() - 16
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(room, dtype=torch.uint8, device=dev))
    if why == "no sharing":
        w._share_rows = False
    w.plan(indptr, indptr, heads, heads, 128, q_data_type=q.dtype, logits_soft_cap=30.0 if soft else None)
    kept = []
    monkeypatch.setattr(_lib.lib(), "fo_decode_sparse_kept", lambda *a: kept.append(a) or 0)
    run = lambda **more: w.run(q, k, v, *sym, out=torch.zeros_like(v), **kw, **more)
    exp = run()
    out = torch.zeros_like(v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        w.run(q, k, v, *sym, out=out, **kw)
        w.run(q, k, v, *sym, out=out, reuse_decoded=True, **kw)
    again = torch.cuda.CUDAGraph()
    with torch.cuda.graph(again):
        w.run(q, k, v, *sym, out=out, reuse_decoded=True, **kw)
    assert torch.equal(run(reuse_decoded=True), exp)
    for what in (graph, again):
        out.zero_()
        what.replay()
        assert torch.equal(out, exp)
    assert not kept


@pytest.mark.parametrize("why", ["soft cap", "small workspace"])
@pytest.mark.parametrize("recorded", [False, True])
def test_workspace_and_cap_of_the_moment(dev, why, recorded):
    """Whether rows are taken straight from the symbols goes by the float workspace and the soft cap of the run, which may be
    others than the plan's.  A graph that holds a reuse from before, which runs the list as it is, still runs the list of the
    moment: the plan's runs are decoded then."""
    import flashomni_amd as fo
    from flashomni_amd import _lib
    n, heads, cap = 514, 206, 30.0 if why == "soft cap" else None
    g = torch.Generator(device=dev).manual_seed(6)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    masks = [make_ragged_masks([384, 130], [384, 130], heads, 0.7, 0.6, seed=s) for s in (5, 6)]
    first, other = ([torch.from_numpy(m[s]).to(dev) for s in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
                    for m in masks)
    indptr = torch.from_numpy(masks[0]["qo_indptr"])
    room = lambda size: torch.empty(size, dtype=torch.uint8, device=dev)

    def plain(sym, c):
        w = fo.BatchFlashOmniFAWithRaggedKVWrapper(room(128 << 20))
        w.plan(indptr, indptr, heads, heads, 128, q_data_type=q.dtype, logits_soft_cap=c)
        return w.run(q, k, v, *sym)

    small = room(2 * _lib.lib().fo_sparse_fa_split_workspace_bytes() - 16 if cap is None else 128 << 20)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(small)
    w.plan(indptr, indptr, heads, heads, 128, q_data_type=q.dtype, logits_soft_cap=cap)
    out = torch.zeros_like(v)
    w.run(q, k, v, *first, out=out)
    assert w._planned.native.state == 0
    if recorded:
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            w.run(q, k, v, *first, out=out, reuse_decoded=True)
    if cap is None:
        w.reset_workspace_buffer(room(128 << 20), room(8 << 20))
        got = w.run(q, k, v, *other)
    else:
        got = w.forward(q, k, v, *other)
    assert (w._planned.native.state == 0) == recorded
    exp = plain(other, None)
    assert float((got.float() - exp.float()).abs().max()) <= 2e-2
    if recorded:
        exp = plain(other, cap)
        for _ in range(2):
            out.zero_()
            graph.replay()
            assert float((out.float() - exp.float()).abs().max()) <= 2e-2


def test_reuse_behind_a_capture_before_rows_came_from_the_symbols(dev, monkeypatch):
    """Where they can be taken from them but have not been, eagerly or in a graph, an eager reuse makes no launch either; one
    that a graph holds looks at every replay, since a run may come in between."""
    from flashomni_amd import _lib
    s = _ShortList(dev, 33)
    lib, kept = _lib.lib(), []
    launch = lib.fo_decode_sparse_kept
    monkeypatch.setattr(lib, "fo_decode_sparse_kept", lambda *a: kept.append(a) or launch(*a))
    a, b, c = s.sym
    s.w.decode(*a)
    torch.cuda.synchronize()
    decode = s.capture(lambda: s.w.decode(*s.buf))
    s.check(s.exp[0], s.run, a, reuse=True)
    assert not kept
    reuse = s.capture(lambda: s.run(a, reuse=True))
    assert len(kept) == 1
    s.check(s.exp[0], s.run, a, reuse=True)
    assert len(kept) == 1
    s.run(b)
    s.check(s.exp[1], reuse.replay)
    s.run(c)
    s.check(s.exp[2], s.run, c, reuse=True)
    assert len(kept) == 2
    for dst, src in zip(s.buf, b):
        dst.copy_(src)
    decode.replay()
    s.check(s.exp[1], s.run, b, reuse=True)
    s.check(s.exp[1], reuse.replay)


def test_captured_decode_and_reuse(dev):
    """decode() on a second stream and reuse of its list in one graph (no launch but those two), also on a plan that
    has not run before; a reuse made before the first replay computes nothing."""
    s = _ShortList(dev, 40)
    side = torch.cuda.Stream(device=dev)

    def step():
        cur = torch.cuda.current_stream()
        side.wait_stream(cur)
        with torch.cuda.stream(side):
            s.w.decode(*s.buf)
        cur.wait_stream(side)
        s.run(s.buf, reuse=True)

    graph = s.capture(step)
    s.check(torch.zeros_like(s.exp[0]), s.run, s.buf, reuse=True)
    for i in (0, 1, 2):
        for dst, src in zip(s.buf, s.sym[i]):
            dst.copy_(src)
        s.check(s.exp[i], graph.replay)
        s.run(s.sym[(i + 1) % 3])
        s.check(s.exp[i], graph.replay)
        s.check(s.exp[i], s.run, s.buf, reuse=True)
        with pytest.raises(RuntimeError, match="is_full=False"):
            s.run(s.buf, reuse=True, is_full=True)
