"""GPU: run() without a decode launch (rows taken straight from the packed symbols) against the oracle, at
the edges of its range: one candidate, 1024 and one more, rows in eight parts, even shares, batches, a
fresh output whose skipped q blocks the launch clears itself, and a list reused afterwards."""
import numpy as np
import pytest
import torch

import oracle
from helpers import make_ragged_masks, max_abs, rel_l2

pytestmark = pytest.mark.gpu

def _cus(dev):
    return torch.cuda.get_device_properties(dev).multi_processor_count


def _pairs(ql, heads):
    return sum(-(-n // 128) for n in ql) * heads


CASES = [
    ([1], [1], 1, 1.0),
    ([640], [20000], 1, 1.0),                 # 5 rows of ~80 kept blocks: eight parts each
    ([300, 1, 128, 1000, 129], [77, 513, 128, 1100, 64], 3, 0.6),
    ([2048], [300], 64, 0.7),                 # 1024 candidates, ~720 rows: even shares
    ([2049], [300], 64, 0.7),                 # 1088 candidates
    ([1200, 900], [1300, 2500], 24, 0.95),    # more rows than workgroups, rows cut at share boundaries
    ([512], [512], 2, 0.0),                   # nothing to compute
    # 640 candidates and more: two workgroups per CU
    ([3300, 130], [2000, 777], 24, 0.9),      # 672 of two requests, ~600 rows in shares
    ([640], [9000], 128, 0.4),                # 640, fewer rows than workgroups, keep bits staged in LDS
    ([4992], [100], 17, 0.02),                # 663, a dozen rows of one kv block
    ([2500, 1], [70, 1], 32, 0.5),            # 672, all rows shorter than a part
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("is_full", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_from_the_symbols(dev, case, is_full, dtype):
    import flashomni_amd as fo
    ql, kl, heads, pa = case
    m = make_ragged_masks(ql, kl, heads, pa, 0.5, seed=3)
    g = torch.Generator().manual_seed(3)
    nq, nk = sum(ql), sum(kl)
    q, k, v = (torch.randn(n, heads, 128, generator=g).to(dtype) for n in (nq, nk, nk))
    t = lambda n: torch.from_numpy(m[n]).to(dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(t("qo_indptr"), t("kv_indptr"), heads, heads, 128, q_data_type=dtype)
    sym = [t(n) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    args = (q.to(dev), k.to(dev), v.to(dev), *sym, is_full)
    lse = torch.full((nq, heads), 7.0, device=dev)
    junk = torch.full((64 << 20,), 0x7f, dtype=torch.uint8, device=dev)   # what a fresh allocation may hold
    del junk
    out, lse = w.run(*args, lse=lse, return_lse=True)
    if _cus(dev) == 256:
        assert (w._planned.native.state != 0) == (_pairs(ql, heads) <= 2047)    # (0: decoded)
    again, lse2 = w.run(*args, lse=lse.clone(), return_lse=True)
    assert torch.equal(out, again) and torch.equal(lse, lse2)
    exp_lse = torch.full((nq, heads), 7.0)
    exp = oracle.sparse_attention(q, k, v, m["packed_info"], m["packed_keep"], m["info_indptr"], m["keep_indptr"],
                                  m["qo_indptr"], m["kv_indptr"], is_full=is_full, out=torch.zeros_like(q), lse=exp_lse)
    got = out.cpu()
    cached = torch.zeros(nq, heads, dtype=torch.bool)
    for r, info in enumerate(m["info"]):
        for qb in range(0 if is_full else info.shape[0]):
            rows = slice(int(m["qo_indptr"][r]) + qb * 128, min(int(m["qo_indptr"][r]) + qb * 128 + 128, int(m["qo_indptr"][r + 1])))
            cached[rows] = torch.from_numpy(~info[qb])
    assert not got[cached].any()
    assert max_abs(got, exp) <= 2e-2 and rel_l2(got, exp) <= 1e-2
    # A row of one key has the logit itself as lse: 128 products of a bf16 q that is rounded once more after the scale
    # (relative error 2^-9 / sqrt(3)), together 2^-9 / sqrt(3) * 0.1275 * sqrt(128) = 1.6e-3; six times that.  Over
    # more keys the errors average out.
    atol = 1e-2 if dtype is torch.bfloat16 and min(kl) == 1 and len(kl) > 1 else 2e-3
    assert torch.allclose(lse.cpu(), exp_lse, atol=atol, rtol=1e-3)
    # the list of that run, reused after the symbols were overwritten
    for s in sym[:2]:
        s.fill_(0xff)
    listed = torch.zeros_like(out)
    w.run(*args, out=listed, reuse_decoded=True)
    assert max_abs(listed.cpu(), got) <= 8e-3


@pytest.mark.parametrize("case", [
    ([2048], [300], 32, 0.4),                              # 512 candidates: half of the threads have two each
    ([2048], [300], 33, 0.4),                              # 528
    ([128] + [100] * 40, [26000] + [64] * 40, 2, 0.8),     # a row of 204 keep bits among short ones: read where they are
    ([640], [12200], 3, 0.8),                              # 96 bits: three words of a thread, or four by their alignment
    ([2048], [20000], 8, 0.6),                             # kept symbols copied by two workgroups
    ([1] * 700, [1, 300] * 350, 1, 0.7),                   # offsets of 700 requests, by two workgroups
])
@pytest.mark.parametrize("is_full", [False, True])
def test_schedule_of_short_lists(dev, case, is_full):
    """The lines inside the schedule of a short list: threads with and without candidates, where a row's keep bits are found,
    what a workgroup copies of the symbols that a later decode reads."""
    test_rows_from_the_symbols(dev, case, is_full, torch.bfloat16)


@pytest.mark.parametrize("case", [
    ([2049], [300], 64, 0.7),                  # 1088 candidates, seven to a thread
    ([3584], [300], 64, 0.9),                  # 1792, ~1610 rows
    ([3585], [300], 64, 0.9),                  # 1856: eight to a thread
    ([2816], [300], 64, 0.9),                  # 1408
    ([3000, 1, 2300], [1200, 770, 1000], 40, 0.8),   # 1720 of three requests
    ([5500], [300], 24, 0.5),                  # 1032
    ([8200], [300], 16, 0.0),                  # 1040, nothing to compute
    ([4000], [9000], 33, 0.05),                # 1056 of 71 blocks, fewer rows than workgroups
])
@pytest.mark.parametrize("is_full", [False, True])
def test_longer_lists_from_the_symbols(dev, case, is_full):
    """1025 candidates and more: seven to a thread up to 1792, and only the rows of a workgroup's own share are in its table.
    (Keys enough that no result reaches 2: the list's is compared to one bf16 step of what is smaller.)"""
    test_rows_from_the_symbols(dev, case, is_full, torch.bfloat16)


@pytest.mark.parametrize("case", [
    ([2944], [300], 78, 0.9),                  # 1794 candidates, eight to a thread
    ([2944], [300], 89, 0.7),                  # 2047, the most
    ([2048], [300], 128, 0.7),                 # 2048: decoded
    ([3000, 1, 2300], [1200, 770, 1000], 47, 0.8),   # 2021 of three requests
    ([9000], [300], 28, 0.0),                  # 1988, nothing to compute
    ([4000], [9000], 60, 0.05),                # 1920 of 71 blocks, fewer rows than workgroups
])
@pytest.mark.parametrize("is_full", [False, True])
def test_lists_of_eight_candidates_per_thread(dev, case, is_full):
    """1793 to 2047 candidates, with the bounds of the test above."""
    test_rows_from_the_symbols(dev, case, is_full, torch.bfloat16)


@pytest.mark.parametrize("is_full", [False, True])
def test_packed_tiles_of_eight_candidates_per_thread(dev, is_full):
    """1880 tiles of grouped-query attention in fp16: as the decoded list, whose rows other workgroups compute whole."""
    import flashomni_amd as fo
    n, hkv, group = 6000, 10, 4
    m = make_ragged_masks([n * group], [900], hkv, 0.7, 0.5, seed=12)
    g = torch.Generator(device=dev).manual_seed(12)
    q, k, v = (torch.randn(t, h, 128, generator=g, device=dev).to(torch.float16) for t, h in ((n, hkv * group), (900, hkv), (900, hkv)))
    sym = [torch.from_numpy(m[x]).to(dev) for x in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    ip = lambda t: torch.tensor([0, t], dtype=torch.int32)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(ip(n), ip(900), hkv * group, hkv, 128, q_data_type=torch.float16)
    out, lse = w.run(q, k, v, *sym, is_full, out=torch.zeros_like(q), lse=torch.zeros(n, hkv * group, device=dev), return_lse=True)
    assert w._planned.native.state != 0
    w.decode(*sym, is_full)
    exp, exp_lse = w.run(q, k, v, *sym, is_full, out=torch.zeros_like(q), lse=torch.zeros(n, hkv * group, device=dev),
                         return_lse=True, reuse_decoded=True)
    assert rel_l2(out.cpu(), exp.cpu()) <= 1e-3  # (p and the result in 11 bits)
    assert torch.allclose(lse, exp_lse, atol=2e-3, rtol=1e-3)


def test_fresh_output_of_the_shortest_decoded_lists(dev):
    """2059 pairs: the test of longer lists below, past the line."""
    test_fresh_output_of_longer_lists(dev, ([9000], [300], 29, 1, 0.0), "NHD")
    test_fresh_output_of_longer_lists(dev, ([2000, 1, 130, 1500], [300, 77, 513, 640], 72, 1, 0.5), "HND")


@pytest.mark.parametrize("empty", ["all", "half", "most"])
@pytest.mark.parametrize("tokens, heads", [(3584, 64), (5500, 24), (2048, 64), (2000, 64)])
def test_shares_of_rows_without_blocks(dev, tokens, heads, empty):
    """Rows that keep no kv block, which cost a share least: all of them, half of the heads, all but one: as the decoded list."""
    import flashomni_amd as fo
    kv, rows = 640, -(-tokens // 128)
    keep = torch.zeros(rows, heads, 5, dtype=torch.bool)
    if empty == "half":
        keep[:, heads // 2:] = True
    elif empty == "most":
        keep[rows // 2, heads // 3] = True
    ip = lambda n: torch.tensor([0, n], dtype=torch.int32, device=dev)
    flags = torch.ones(rows * heads, dtype=torch.bool, device=dev)
    info, info_ip = fo.segment_packbits(flags, ip(rows * heads), "little")
    kv_info, kv_ip = fo.segment_packbits(keep.view(-1).to(dev), ip(keep.numel()), "little")
    g = torch.Generator(device=dev).manual_seed(7)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for n in (tokens, kv, kv))
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(ip(tokens).cpu(), ip(kv).cpu(), heads, heads, 128, q_data_type=torch.bfloat16)
    sym = (info, kv_info, info_ip, kv_ip)
    out, lse = w.run(q, k, v, *sym, out=torch.full_like(q, 3.0), lse=torch.full((tokens, heads), 7.0, device=dev), return_lse=True)
    w.decode(*sym)
    exp, exp_lse = w.run(q, k, v, *sym, out=torch.full_like(q, 3.0), lse=torch.full((tokens, heads), 7.0, device=dev),
                         return_lse=True, reuse_decoded=True)
    assert max_abs(out.cpu(), exp.cpu()) <= 8e-3
    assert torch.allclose(lse, exp_lse, atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("group", [2, 7])
def test_fresh_output_of_packed_tiles(dev, group):
    """Skipped tiles of grouped-query attention: the rows of a tile are spread over the group's q heads."""
    import flashomni_amd as fo
    hkv, ql, kl = 2, [300, 1, 640], [77, 513, 640]
    hq = hkv * group
    m = make_ragged_masks([n * group for n in ql], kl, hkv, 0.5, 0.5, seed=4)
    qo = torch.from_numpy(np.concatenate([[0], np.cumsum(ql)]).astype(np.int32))
    g = torch.Generator(device=dev).manual_seed(4)
    q, k, v = (torch.randn(n, h, 128, generator=g, device=dev).to(torch.bfloat16) for n, h in ((941, hq), (1230, hkv), (1230, hkv)))
    t = lambda n: torch.from_numpy(m[n]).to(dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(512 << 20, dtype=torch.uint8, device=dev))
    w.plan(qo, t("kv_indptr"), hq, hkv, 128, q_data_type=torch.bfloat16)
    sym = [t(n) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    exp = w.run(q, k, v, *sym, out=torch.zeros_like(q))
    junk = torch.full((64 << 20,), 0x7f, dtype=torch.uint8, device=dev)
    del junk
    assert torch.equal(w.run(q, k, v, *sym), exp)


@pytest.mark.parametrize("case", [([2000, 1, 130, 1500], [300, 77, 513, 640], 40, 1, 0.5), ([2000, 1, 130, 1500], [300, 77, 513, 640], 64, 1, 0.5),
                                  ([5000, 129, 1], [640, 300, 77], 8, 4, 0.3), ([5000, 129, 1], [640, 300, 77], 12, 4, 0.3),
                                  ([9000], [300], 16, 1, 0.0), ([9000], [300], 26, 1, 0.0)])
@pytest.mark.parametrize("layout", ["NHD", "HND"])
def test_fresh_output_of_longer_lists(dev, case, layout):
    """Lists above 1024 pairs, taken from the symbols, and above 2047, decoded: the launch, or the decoder's launches, clear
    the skipped rows of a fresh output (ragged last tiles, tiles of grouped-query rows, nothing to compute); the same bits as
    over a cleared output."""
    import flashomni_amd as fo
    ql, kl, hkv, group, pa = case
    hq = hkv * group
    pairs = sum(-(-n * group // 128) for n in ql) * hkv
    m = make_ragged_masks([n * group for n in ql], kl, hkv, pa, 0.5, seed=6)
    qo = torch.from_numpy(np.concatenate([[0], np.cumsum(ql)]).astype(np.int32))
    g = torch.Generator(device=dev).manual_seed(6)
    kv_shape = (sum(kl), hkv, 128) if layout == "NHD" else (hkv, sum(kl), 128)
    q, k, v = (torch.randn(*s, generator=g, device=dev).to(torch.bfloat16) for s in ((sum(ql), hq, 128), kv_shape, kv_shape))
    t = lambda n: torch.from_numpy(m[n]).to(dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev), layout)
    w.plan(qo, t("kv_indptr"), hq, hkv, 128, q_data_type=torch.bfloat16)
    sym = [t(n) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    exp = w.run(q, k, v, *sym, out=torch.zeros_like(q))
    if _cus(dev) == 256:
        assert (w._planned.native.state == 0) == (pairs > 2047)
    for _ in range(3):
        junk = torch.full((256 << 20,), 0x7f, dtype=torch.uint8, device=dev)   # what a fresh allocation may hold
        del junk
        assert torch.equal(w.run(q, k, v, *sym), exp)


def test_fresh_output_of_a_decoded_fp8_list(dev):
    """The same for fp8 q and k, whose lists are always decoded; q of other heads than planned is still refused."""
    import flashomni_amd as fo
    ql, kl, heads = [5000, 77], [300, 640], 30
    m = make_ragged_masks(ql, kl, heads, 0.4, 0.5, seed=8)
    g = torch.Generator(device=dev).manual_seed(8)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for n in (sum(ql), sum(kl), sum(kl)))
    t = lambda n: torch.from_numpy(m[n]).to(dev)
    q8, qs = fo.quant_fp8_block(q, torch.from_numpy(m["qo_indptr"]))
    k8, ks = fo.quant_fp8_block(k, torch.from_numpy(m["kv_indptr"]))
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(t("qo_indptr"), t("kv_indptr"), heads, heads, 128, q_data_type=torch.float8_e4m3fn)
    sym = [t(n) for n in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    exp = w.run(q8, k8, v, *sym, out=torch.zeros_like(q), q_scale=qs, k_scale=ks)
    for _ in range(3):
        junk = torch.full((256 << 20,), 0x7f, dtype=torch.uint8, device=dev)   # what a fresh allocation may hold
        del junk
        assert torch.equal(w.run(q8, k8, v, *sym, q_scale=qs, k_scale=ks), exp)
    with pytest.raises(ValueError, match="head count"):
        w.run(q8[:, :20].contiguous(), k8, v, *sym, q_scale=qs, k_scale=ks)


@pytest.mark.parametrize("run_on_default", [True, False])
def test_list_of_a_run_reused_on_another_stream(dev, run_on_default):
    """A run that took its rows from the symbols is still to come on its (busy) stream when another stream
    reuses its list: the reuse waits for that run, and does not decode what an earlier run left."""
    import flashomni_amd as fo
    heads, lens = 2, [384, 130]
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(sum(lens), heads, 128, generator=g).to(torch.bfloat16) for _ in range(3))
    masks = [make_ragged_masks(lens, lens, heads, 0.7, 0.6, seed=s) for s in (50, 51)]
    names = ("packed_info", "packed_keep", "info_indptr", "keep_indptr")
    syms = [[torch.from_numpy(m[n]).to(dev) for n in names] for m in masks]
    m = masks[1]
    exp = oracle.sparse_attention(q, k, v, *(m[n] for n in names), m["qo_indptr"], m["kv_indptr"], out=torch.zeros_like(q))
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(torch.from_numpy(m["qo_indptr"]), torch.from_numpy(m["kv_indptr"]), heads, heads, 128, q_data_type=torch.bfloat16)
    w.run(qd, kd, vd, *syms[0])
    w.run(qd, kd, vd, *syms[0], reuse_decoded=True)    # (the list exists, and is the other symbols')
    default, side = torch.cuda.current_stream(dev), torch.cuda.Stream(device=dev)
    first, second = (default, side) if run_on_default else (side, default)
    out, again = torch.zeros_like(qd), torch.zeros_like(qd)
    torch.cuda.synchronize(dev)
    with torch.cuda.stream(first):
        busy = torch.empty(1 << 30, dtype=torch.uint8, device=dev)
        for i in range(20):
            busy.fill_(i)
        w.run(qd, kd, vd, *syms[1], out=out)
    with torch.cuda.stream(second):
        w.run(qd, kd, vd, *syms[1], out=again, reuse_decoded=True)
    torch.cuda.synchronize(dev)
    for got in (out.cpu(), again.cpu()):
        assert max_abs(got, exp) <= 2e-2 and rel_l2(got, exp) <= 1e-2


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("group", [1, 4])
@pytest.mark.parametrize("ws_mib", [68, 64])
def test_routes_of_a_short_list_agree(dev, layout, group, ws_mib):
    """The forms that the size of the workspace chooses between (two workgroups per CU, one, a decoded list) on
    strided operands, symbols at odd addresses, grouped-query rows and a batch with a request without keys: against
    the decoded list, whose rows are not cut."""
    import flashomni_amd as fo
    hkv, ql, kl = (24, [3500, 1, 300], [1100, 64, 0]) if group == 1 else (4, [5500, 1, 77], [640, 64, 0])
    hq = hkv * group
    m = make_ragged_masks([n * group for n in ql], kl, hkv, 0.8, 0.6, seed=7)
    qo = torch.from_numpy(np.concatenate([[0], np.cumsum(ql)]).astype(np.int32))
    g = torch.Generator(device=dev).manual_seed(7)
    rand = lambda *shape: torch.randn(*shape, generator=g, device=dev).to(torch.bfloat16)
    q = rand(sum(ql), 2 * hq, 128)[:, hq:]                       # a slice of a fused projection
    kv = rand(sum(kl), 2 * hkv, 128)
    k, v = kv[:, :hkv], kv[:, hkv:]
    if layout == "HND":
        k, v = k.transpose(0, 1), v.transpose(0, 1).contiguous()
    t = lambda n: torch.from_numpy(m[n]).to(dev)
    odd = lambda x: torch.cat([x.new_full((3,), 0xff), x, x.new_full((5,), 0xff)])[3:3 + x.numel()]
    sym = [odd(t("packed_info")), odd(t("packed_keep")), t("info_indptr"), t("keep_indptr")]
    outs = []
    for nbytes in (1 << 20, ws_mib << 20):
        w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(nbytes, dtype=torch.uint8, device=dev), layout)
        w.plan(qo, t("kv_indptr"), hq, hkv, 128, q_data_type=torch.bfloat16)
        out = torch.full((sum(ql), hq, 128), 7.0, dtype=torch.bfloat16, device=dev)
        lse = torch.full((sum(ql), hq), 7.0, device=dev)
        w.run(q, k, v, *sym, out=out, lse=lse, return_lse=True)
        outs.append((out.cpu(), lse.cpu()))
    (exp, exp_lse), (got, got_lse) = outs
    assert torch.equal(got == 7.0, exp == 7.0)
    assert max_abs(got, exp) <= 2e-2 and rel_l2(got, exp) <= 6e-3
    assert torch.allclose(got_lse, exp_lse, atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("ql, kl, heads", [
    ([300, 1, 700], [1100, 77, 513], 3),            # whole parts
    ([3000, 1, 700], [1100, 77, 513], 24),          # 720 candidates, shares in the pipelined form
    ([2600, 700, 500], [9000, 300, 4000], 24),      # keep bits of 70 and 31 blocks, read where they are or from LDS
    ([1500, 128, 300], [40000, 40000, 700], 16),    # 313 blocks to a row
])
def test_symbols_in_any_order(dev, ql, kl, heads):
    """Segments that lie in the buffer in another order than their requests, at odd bytes: what is outside of the piece from
    the first segment to the end is read where it is, the rest from LDS.  The same bits as in order."""
    import flashomni_amd as fo
    m = make_ragged_masks(ql, kl, heads, 0.8, 0.4, seed=9)
    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(n, heads, 128, generator=g).to(torch.bfloat16).to(dev) for n in (sum(ql), sum(kl), sum(kl)))
    t = lambda a: torch.from_numpy(a).to(dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(torch.empty(128 << 20, dtype=torch.uint8, device=dev))
    w.plan(t(m["qo_indptr"]), t(m["kv_indptr"]), heads, heads, 128, q_data_type=torch.bfloat16)

    def moved(packed, indptr):
        """The second request's segment in front, three bytes of ones before every segment."""
        parts, at, starts = [], 0, {}
        for r in (1, 0, 2):
            seg = packed[indptr[r]:indptr[r + 1]]
            parts += [np.full(3, 0xff, np.uint8), seg]
            starts[r] = at + 3
            at += 3 + len(seg)
        return np.concatenate(parts), np.array([starts[0], starts[1], starts[2], at], np.int32)

    want = w.run(q, k, v, t(m["packed_info"]), t(m["packed_keep"]), t(m["info_indptr"]), t(m["keep_indptr"]))
    info, info_ip = moved(m["packed_info"], m["info_indptr"])
    keep, keep_ip = moved(m["packed_keep"], m["keep_indptr"])
    got = w.run(q, k, v, t(info), t(keep), t(info_ip), t(keep_ip))
    assert torch.equal(got, want)
    # where the last segment ends is nobody's beginning: whatever stands there, no byte behind the segments is asked for
    for end in (0, len(m["packed_keep"]) + 40000, 2 ** 31 - 1):
        ip = m["keep_indptr"].copy()
        ip[-1] = end
        got = w.run(q, k, v, t(m["packed_info"]), t(m["packed_keep"]), t(m["info_indptr"]), t(ip))
        assert torch.equal(got, want), end


@pytest.mark.parametrize("tokens, heads", [(1627, 32), (1627, 31), (5200, 10), (6600, 8), (10500, 5)])
def test_full_rows_around_the_choice_of_form(dev, tokens, heads):
    """Every row computed, 403 to 416 candidates: the two loops meet there.  (Of the two workgroups per CU of the pipelined one
    the second ones' parts lie in the second half of the float workspace, where rows are long enough to be cut.)"""
    import flashomni_amd as fo
    from flashomni_amd import _lib
    g = torch.Generator().manual_seed(tokens)
    q, k, v = (torch.randn(tokens, heads, 128, generator=g).to(torch.bfloat16).to(dev) for _ in range(3))
    ip = torch.tensor([0, tokens], dtype=torch.int32)
    ws = torch.full((128 << 20,), 0x5a, dtype=torch.uint8, device=dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
    w.plan(ip, ip, heads, heads, 128, q_data_type=torch.bfloat16)
    out, lse = w.run(q, k, v, is_full=True, return_lse=True)
    half = _lib.lib().fo_sparse_fa_split_workspace_bytes()
    if _cus(dev) == 256:
        assert w._planned.native.state != 0
        if tokens >= 40 * 128:
            assert bool((ws[half:2 * half] != 0x5a).any()) == (_pairs([tokens], heads) >= 416)
    rows = torch.cat([torch.arange(0, 130), torch.arange(tokens - 130, tokens)]).to(dev)
    for h in (0, heads // 2, heads - 1):
        s = q[rows, h].float() @ k[:, h].float().t().contiguous() * 128 ** -0.5
        exp = torch.softmax(s, -1) @ v[:, h].float()
        # (p and the result are rounded to 8 bits, q * scale as well: 1e-2 of the result's size at most)
        assert float((out[rows, h].float() - exp).norm() / exp.norm()) <= 1e-2
        assert float((lse[rows, h] - torch.logsumexp(s, -1) * 1.4426950408889634).abs().max()) < 2e-2


def _long_list(dev, pairs, is_full, room=128 << 20):
    """A planned list of `pairs` over 300 keys, as a call without arguments; its wrapper and workspace."""
    import flashomni_amd as fo
    blocks, heads = pairs
    tokens = 128 * blocks
    m = make_ragged_masks([tokens], [300], heads, 0.9, 0.5, seed=14)
    g = torch.Generator(device=dev).manual_seed(14)
    q, k, v = (torch.randn(n, heads, 128, generator=g, device=dev).to(torch.bfloat16) for n in (tokens, 300, 300))
    sym = [torch.from_numpy(m[x]).to(dev) for x in ("packed_info", "packed_keep", "info_indptr", "keep_indptr")]
    ws = torch.full((room,), 0x5a, dtype=torch.uint8, device=dev)
    w = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
    w.plan(*(torch.tensor([0, n], dtype=torch.int32) for n in (tokens, 300)), heads, heads, 128, q_data_type=torch.bfloat16)
    out = torch.zeros_like(q)
    return w, ws, sym, out, lambda **kw: w.run(q, k, v, *sym, is_full, out=out, **kw)


@pytest.mark.parametrize("pairs, is_full, shares", [((28, 64), False, True), ((23, 78), False, False), ((23, 89), False, False),
                                                    ((22, 64), True, True), ((23, 62), True, False), ((23, 89), True, False)])
def test_long_lists_leave_the_float_workspace_alone(dev, pairs, is_full, shares):
    """1792 pairs and fewer (1408 where every row is computed) leave partial results in the float workspace.  Longer lists, which
    were always decoded once, leave it to others that may be using it at the time."""
    w, ws, sym, out, run = _long_list(dev, pairs, is_full)
    run()
    assert w._planned.native.state != 0
    assert bool((ws == 0x5a).all()) != shares
    exp = out.clone()
    out.zero_()
    w.decode(*sym, is_full)
    ws.fill_(0x5a)
    run(reuse_decoded=True)
    assert bool((ws == 0x5a).all())    # (more than two rows per CU: taken whole)
    # (p and the result are rounded to 8 bits on either side, by 2^-9 / sqrt(3) of it each: together 2.3e-3, four times that)
    assert rel_l2(out.cpu(), exp.cpu()) <= 1e-2


def test_long_list_without_room_for_its_parts(dev):
    """The allocator has nothing left for the parts of rows: the list is decoded, and later runs do not ask again."""
    w, ws, sym, out, run = _long_list(dev, (23, 78), False)
    w.decode(*sym)
    run(reuse_decoded=True)
    exp = out.clone()
    torch.cuda.synchronize(dev)
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + (8 << 20)) / total, dev)
    held = []    # (what is left in the allocator's own blocks)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            for _ in range(1000):
                held.append(torch.empty(60 << 20, dtype=torch.uint8, device=dev))
        out.zero_()
        run()
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert w._planned.native.state == 0 and torch.equal(out, exp)
    run()
    assert w._planned.native.state == 0 and torch.equal(out, exp)
