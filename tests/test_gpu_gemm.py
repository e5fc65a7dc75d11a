"""GPU parity: GEMM-Q / GEMM-O vs the fp32 masked-GEMM oracle.

bf16/fp16 outputs: max-abs <= 2e-2 and relative L2 <= 1e-2 of the fp32 reference; tiles whose flag
is 0 keep their bytes (GEMM-Q)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from helpers import max_abs, rel_l2, sentinel_like

pytestmark = pytest.mark.gpu

MAX_ABS, REL_L2 = 2e-2, 1e-2


def _flags(batch, n_qblocks, heads, p, seed):
    rng = np.random.default_rng(seed)
    info = rng.random((batch, n_qblocks, heads)) < p
    segs = [np.packbits(info[b].reshape(-1).astype(np.uint8), bitorder="little") for b in range(batch)]
    indptr = np.zeros(batch + 1, dtype=np.int32)
    indptr[1:] = np.cumsum([len(s) for s in segs])
    return info, np.concatenate(segs), indptr


def _operands(batch, m, n, k, dtype, seed, bias=True):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(batch, m, k, generator=g).to(dtype)
    w = (torch.randn(n, k, generator=g) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g) * 0.02).to(dtype) if bias else None
    return x, w, b


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 512, 384, 256, 3, 0), (2, 256, 256, 96, 2, 0),
                                   (1, 1024, 256, 512, 2, 512), (1, 300, 256, 128, 2, 0)])
def test_gemm_q_matches_oracle_and_skips_tiles(dev, dtype, shape):
    import flashomni_amd as fo
    batch, m, n, k, heads, text = shape
    nqb = (text + m + 127) // 128
    info, packed, indptr = _flags(batch, nqb, heads, 0.6, seed=m + n)
    x, w, b = _operands(batch, m, n, k, dtype, seed=k)
    out0 = sentinel_like((batch, m, n), dtype)
    out = out0.clone().to(dev)
    res = fo.flashomni_gemm(x.to(dev), w.to(dev), heads, torch.from_numpy(packed).to(dev),
                            torch.from_numpy(indptr).to(dev), text, b.to(dev), out=out)
    assert res.data_ptr() == out.data_ptr()
    exp = oracle.gemm_q(x, w, heads, packed, indptr, text, b, out=out0.clone())
    out = out.cpu()
    changed = (exp.view(torch.int16) != out0.view(torch.int16))
    # skipped tiles byte-identical
    hd = n // heads
    for bi in range(batch):
        for iy in range((m + 127) // 128):
            for ix in range(n // 128):
                bit = info[bi, (text + iy * 128) // 128, (ix * 128) // hd]
                tile = (bi, slice(iy * 128, min(m, (iy + 1) * 128)), slice(ix * 128, (ix + 1) * 128))
                if not bit:
                    assert torch.equal(out[tile].view(torch.int16), out0[tile].view(torch.int16))
    assert max_abs(out, exp) <= MAX_ABS
    assert rel_l2(out[changed], exp[changed]) <= REL_L2


@pytest.mark.parametrize("case", [(2, 33077, 2048, 96, 16, 0.8), (2, 66100, 1280, 128, 20, 0.5), (1, 70000, 1024, 64, 8, 0.6),
                                  (2, 40000, 2304, 64, 9, 0.25)])
def test_gemm_q_large_lists_with_column_strips(dev, case):
    """Matrices of more than 256 (window, column pair) cells get their work list from the list kernel:
    full quads for rows flagged in both columns of a cell, column strips (three token blocks x one column
    block) for rows flagged in one.  Whole output against the oracle (small K keeps that cheap), skipped
    tiles byte for byte; flag densities that give mostly quads, a mix, mostly strips; a ragged last
    token block, an odd number of token blocks, K = 96 (the slab that counts for one half), heads of
    64 columns (a column block reads the flag of its first head) and of 256 (two column blocks per flag)."""
    import flashomni_amd as fo
    batch, m, n, k, heads, dens = case
    nqb = (m + 127) // 128
    info, packed, indptr = _flags(batch, nqb, heads, dens, seed=m)
    g = torch.Generator(device=dev).manual_seed(m + k)
    x = torch.randn(batch, m, k, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    b = (torch.randn(n, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    out = torch.full((batch, m, n), -7.0, dtype=torch.bfloat16, device=dev)
    fo.flashomni_gemm(x, w, heads, torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev), 0, b, out=out)
    exp = oracle.gemm_q(x.cpu(), w.cpu(), heads, packed, indptr, 0, b.cpu(),
                        out=torch.full((batch, m, n), -7.0, dtype=torch.bfloat16))
    out = out.cpu()
    hd = n // heads
    tile_head = (np.arange(n // 128) * 128) // hd    # the flag a (128 x 128) tile reads (gemm.cuh:50-58)
    active = torch.from_numpy(info[:, :, tile_head]).repeat_interleave(128, 1)[:, :m].repeat_interleave(128, 2)
    assert bool((out[~active] == -7.0).all()) and bool((exp[~active] == -7.0).all())
    assert max_abs(out[active], exp[active]) <= MAX_ABS
    assert rel_l2(out[active], exp[active]) <= REL_L2


@pytest.mark.parametrize("shape", [(1, 4400, 4352, 34, 64), (1, 4401, 5248, 41, 96), (2, 2200, 4608, 36, 160)])
@pytest.mark.parametrize("p", [0.0, 0.1, 0.45, 0.55, 0.9, 1.0])
def test_flagged_gemm_q_as_quads_or_strips(dev, shape, p):
    """Flagged GEMM-Q of 4.5 units per CU and more, wide: quads if one round holds them and items of two units would be more than
    one, strips if not; the first launch leaves in the scratch's first word whether it ran.  Either way each wanted tile is
    the fp32 product's, rounded once, and the others stay; the word, whatever it held, is written by every call."""
    from flashomni_amd import _lib
    batch, m, n, heads, k = shape
    L, blocks = _lib.lib(), -(-m // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    info, packed, indptr = _flags(batch, blocks, heads, p, seed=m)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, k, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    need = L.fo_gemm_workspace_bytes(batch, m, n)
    exp = (x.float() @ w.float().t())
    on = torch.from_numpy(info).to(dev).bool().repeat_interleave(128, 1)[:, :m].repeat_interleave(128, 2)
    units = int(info.astype(np.int64).sum())
    for before in (0, 1):
        ws = torch.full((need // 4,), before, dtype=torch.int32, device=dev)
        y = torch.full((batch, m, n), -7.0, dtype=torch.bfloat16, device=dev)
        _lib.check(L.fo_gemm_q(x.data_ptr(), w.data_ptr(), None, y.data_ptr(), 0, batch, m, n, k, 128, heads, pk.data_ptr(),
                               ip.data_ptr(), 0, 0, ws.data_ptr(), need, torch.cuda.current_stream(dev).cuda_stream))
        assert bool((y[~on] == -7.0).all())
        err = (y.float() - exp).abs() - 2.0 ** -8 * exp.abs() - k * 2.0 ** -24 * 16 * 0.05
        assert not bool(on.any()) or float(err[on].max()) <= 0
        if cus == 256:
            if units > 4 * cus:   # more than a round of quads
                assert int(ws[0]) == 0
            elif units <= cus:    # items of at most two units fit a round
                assert int(ws[0]) == 0
            elif p == 0.45 and m == 4400:
                assert int(ws[0]) == 1


def test_gemm_q_is_full_equals_linear(dev):
    import flashomni_amd as fo
    x, w, b = _operands(1, 384, 256, 192, torch.bfloat16, seed=9)
    out = fo.flashomni_gemm(x.to(dev), w.to(dev), 2, bias=b.to(dev), is_full=True).cpu()
    exp = F.linear(x.float(), w.float(), b.float())
    assert max_abs(out, exp) <= MAX_ABS and rel_l2(out, exp) <= REL_L2


def test_gemm_q_shape_errors(dev):
    import flashomni_amd as fo
    x, w, b = _operands(1, 128, 192, 64, torch.bfloat16, seed=1)
    with pytest.raises(RuntimeError, match="only support"):
        fo.flashomni_gemm(x.to(dev), w.to(dev), 1, is_full=True)
    x, w, b = _operands(1, 128, 128, 32, torch.bfloat16, seed=1)
    with pytest.raises(RuntimeError, match="below the 64 columns"):
        fo.flashomni_gemm(x.to(dev), w.to(dev), 1, is_full=True)
    x = torch.zeros(1, 128, 65600, dtype=torch.bfloat16, device=dev)
    w = torch.zeros(128, 65600, dtype=torch.bfloat16, device=dev)
    with pytest.raises(RuntimeError, match="above 65536"):
        fo.flashomni_gemm(x, w, 1, is_full=True)


def test_undersized_symbols_raise(dev):
    """Packed flags shorter than the last bit the kernels would read are refused on the host."""
    import flashomni_amd as fo
    x, w, b = _operands(2, 512, 256, 256, torch.bfloat16, seed=2)
    x, w = x.to(dev), w.to(dev)
    # (512 text + 512 tokens) / 128 = 8 blocks x 2 heads = 16 bits = 2 bytes per request
    info = torch.zeros(4, dtype=torch.uint8, device=dev)
    ip = torch.tensor([0, 2, 4], dtype=torch.int32, device=dev)
    fo.flashomni_gemm(x, w, 2, info, ip, 512)
    fo.flashomni_gemm_reduction(x, w, 2, info, ip, 512)
    with pytest.raises(RuntimeError, match="a request needs 2"):
        fo.flashomni_gemm(x, w, 2, info[:1], ip, 512)
    with pytest.raises(RuntimeError, match="a request needs 2"):
        fo.flashomni_gemm_reduction(x, w, 2, info[:1], ip, 512)
    with pytest.raises(RuntimeError, match="batch \\+ 1 = 3 entries"):
        fo.flashomni_gemm(x, w, 2, info, ip[:2], 512)
    with pytest.raises(RuntimeError, match="needs sparse_info_indptr"):
        fo.flashomni_gemm(x, w, 2, info, None, 512)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("use_bias", [False, True])
@pytest.mark.parametrize("shape", [(1, 512, 384, 3, 0), (2, 256, 256, 2, 0), (1, 300, 512, 4, 0),
                                   # head widths that are not multiples of the 64-wide operand slabs: 96, 32, 160
                                   (1, 384, 384, 4, 0), (1, 200, 128, 4, 0), (1, 256, 640, 4, 128),
                                   # more heads than the kernel fetches a work item ahead (160 slices of width 32)
                                   (1, 300, 5120, 160, 0)])
def test_gemm_o_two_pass_protocol(dev, dtype, use_bias, shape):
    """cache pass, then final pass fed with the cached partial: each pass matches its oracle and the
    end result equals the dense linear layer (the identity the reference's own script checks,
    benchmark/test_flashomni_gemm_o.py:72-86)."""
    import flashomni_amd as fo
    batch, m, n, heads, text = shape
    k = n
    nqb = (text + m + 127) // 128
    info, packed, indptr = _flags(batch, nqb, heads, 0.5, seed=m)
    x, w, b = _operands(batch, m, n, k, dtype, seed=n, bias=use_bias)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    xd, wd = x.to(dev), w.to(dev)
    cache = fo.flashomni_gemm_reduction(xd, wd, heads, pk, ip, text, bias=b.to(dev) if use_bias else None,
                                        is_for_cache=True)
    exp_cache = oracle.gemm_o(x, w, heads, packed, indptr, text, bias=b, is_for_cache=True)
    assert cache.dtype == dtype
    assert max_abs(cache.cpu(), exp_cache) <= MAX_ABS
    final = fo.flashomni_gemm_reduction(xd, wd, heads, pk, ip, text, bias=cache, is_for_cache=False)
    exp_final = oracle.gemm_o(x, w, heads, packed, indptr, text, bias=cache.cpu(), is_for_cache=False)
    assert max_abs(final.cpu(), exp_final) <= MAX_ABS
    assert rel_l2(final.cpu(), exp_final) <= REL_L2
    dense = F.linear(x.float(), w.float(), b.float() if use_bias else None)
    assert rel_l2(final.cpu(), dense) <= REL_L2
    # fp32 partial keeps the whole chain within the max-abs budget
    cache32 = fo.flashomni_gemm_reduction(xd, wd, heads, pk, ip, text, bias=b.to(dev) if use_bias else None,
                                          is_for_cache=True, out_dtype=torch.float32)
    assert cache32.dtype == torch.float32
    final32 = fo.flashomni_gemm_reduction(xd, wd, heads, pk, ip, text, bias=cache32, is_for_cache=False)
    assert max_abs(final32.cpu(), dense) <= MAX_ABS


def test_gemm_o_extreme_masks(dev):
    """all-ones flags: the cache pass returns the broadcast bias and the final pass the full linear
    layer; all-zero flags: the reverse."""
    import flashomni_amd as fo
    x, w, b = _operands(1, 256, 256, 256, torch.bfloat16, seed=4)
    heads = 2
    ip = torch.tensor([0, 1], dtype=torch.int32, device=dev)
    dense = F.linear(x.float(), w.float(), b.float())
    for byte, cache_is_bias in ((0xFF, True), (0x00, False)):
        pk = torch.tensor([byte], dtype=torch.uint8, device=dev)
        cache = fo.flashomni_gemm_reduction(x.to(dev), w.to(dev), heads, pk, ip, 0, bias=b.to(dev),
                                            is_for_cache=True).cpu()
        if cache_is_bias:
            assert torch.equal(cache, b[None, None, :].expand_as(cache))
        else:
            assert rel_l2(cache, dense) <= REL_L2
        final = fo.flashomni_gemm_reduction(x.to(dev), w.to(dev), heads, pk, ip, 0,
                                            bias=cache.to(dev), is_for_cache=False).cpu()
        assert rel_l2(final, dense) <= REL_L2


def test_flux_gemm_q_full_config(dev):
    import flashomni_amd as fo
    from flashomni_amd.workloads import make_workload
    wl = make_workload(1)
    x, w, b = wl.tensors["x"], wl.tensors["w"], wl.tensors["bias"]
    out0 = sentinel_like((1, 4608, 3072), torch.bfloat16)
    out = out0.clone().to(dev)
    fo.flashomni_gemm(x.to(dev), w.to(dev), 24, wl.packed_info.to(dev), wl.info_indptr.to(dev), 0,
                      b.to(dev), out=out)
    out = out.cpu()
    exp = oracle.gemm_q(x, w, 24, wl.packed_info, wl.info_indptr, 0, b, out=out0.clone())
    active = wl.sparse_info.repeat_interleave(128, 0).repeat_interleave(128, 1)[None]
    assert torch.equal(out[~active].view(torch.int16), out0[~active].view(torch.int16))
    assert max_abs(out[active], exp[active]) <= MAX_ABS
    assert rel_l2(out[active], exp[active]) <= REL_L2


def test_flux_gemm_o_full_config(dev):
    import flashomni_amd as fo
    from flashomni_amd.workloads import make_workload
    wl = make_workload(2)
    a, w, b = wl.tensors["a"], wl.tensors["w"], wl.tensors["bias"]
    pk, ip = wl.packed_info.to(dev), wl.info_indptr.to(dev)
    cache = fo.flashomni_gemm_reduction(a.to(dev), w.to(dev), 24, pk, ip, 0, bias=b.to(dev),
                                        is_for_cache=True, out_dtype=torch.float32)
    final = fo.flashomni_gemm_reduction(a.to(dev), w.to(dev), 24, pk, ip, 0, bias=cache,
                                        is_for_cache=False).cpu()
    exp_cache = oracle.gemm_o(a, w, 24, wl.packed_info, wl.info_indptr, 0, bias=b, is_for_cache=True,
                              out_dtype=torch.float32)
    assert max_abs(cache.cpu(), exp_cache) <= 1e-3
    dense = F.linear(a.float(), w.float(), b.float())
    assert max_abs(final, dense) <= MAX_ABS and rel_l2(final, dense) <= REL_L2


@pytest.mark.parametrize("shape", [(2, 2500, 384, 256), (1, 4224, 640, 128), (3, 130, 128, 64), (2, 10500, 1408, 576)])
def test_dense_tile_enumeration_geometries(dev, shape):
    """Every unit computed (is_full GEMM-Q, GEMM-O): the kernel enumerates its tiles arithmetically.
    More than one 16-block window, a short last window, an odd number of column tiles, a token
    tail and several batches; every output element must be written and right.  (Up to 256 units one to a CU; the last
    shape as quads, GEMM-O as strips.)"""
    import flashomni_amd as fo
    batch, m, n, k = shape
    heads = n // 128
    x, w, b = _operands(batch, m, n, k, torch.bfloat16, seed=m + k)
    out0 = sentinel_like((batch, m, n), torch.bfloat16)
    out = out0.clone().to(dev)
    fo.flashomni_gemm(x.to(dev), w.to(dev), heads, bias=b.to(dev), out=out, is_full=True)
    exp = F.linear(x.float(), w.float(), b.float())
    assert max_abs(out.cpu(), exp) <= MAX_ABS and rel_l2(out.cpu(), exp) <= REL_L2
    # GEMM-O over the same geometry (K = N there: heads slice the contraction)
    nqb = (m + 127) // 128
    info, packed, indptr = _flags(batch, nqb, heads, 0.5, seed=n)
    a = torch.randn(batch, m, n, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    wo = (torch.randn(n, n, generator=torch.Generator().manual_seed(4)) * 0.05).to(torch.bfloat16)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    cache = fo.flashomni_gemm_reduction(a.to(dev), wo.to(dev), heads, pk, ip, 0, bias=None,
                                        is_for_cache=True, out_dtype=torch.float32)
    final = fo.flashomni_gemm_reduction(a.to(dev), wo.to(dev), heads, pk, ip, 0, bias=cache,
                                        is_for_cache=False)
    exp = torch.matmul(a.float(), wo.float().t())       # cache + final = the full product
    assert max_abs(final.cpu(), exp) <= 4e-2 and rel_l2(final.cpu(), exp) <= REL_L2


@pytest.mark.parametrize("shape", [(1, 512, 384, 256, 0.6), (2, 300, 256, 128, 0.7), (1, 1200, 512, 96, 1.0)])
@pytest.mark.parametrize("write_out", [True, False])
def test_gemm_q_with_fused_fp8_quantisation(dev, shape, write_out):
    """GEMM-Q that also emits fp8 e4m3fn tiles + one absmax scale per (head, 128-token block).
    The reference has no such step (parity unpinned against it); pinned by the closed form
    scale = absmax / 448, the e4m3 rounding bound, untouched skipped tiles, and by the attention
    kernel accepting the pair like the separate quantiser's."""
    import flashomni_amd as fo
    batch, m, n, k, p_active = shape
    heads, dtype = n // 128, torch.bfloat16
    nqb = (m + 127) // 128
    info, packed, indptr = _flags(batch, nqb, heads, p_active, seed=m + k)
    x, w, b = _operands(batch, m, n, k, dtype, seed=k + 1)
    out0 = sentinel_like((batch, m, n), dtype)
    q8_0 = torch.full((batch, m, n), 0x5A, dtype=torch.uint8)
    sc_0 = torch.full((heads, batch * nqb), -7.0)
    args = (x.to(dev), w.to(dev), heads, torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev), 0, b.to(dev))
    plain = fo.flashomni_gemm(*args, out=out0.clone().to(dev)).cpu()
    q8 = q8_0.clone().to(dev).view(torch.float8_e4m3fn)
    sc = sc_0.clone().to(dev)
    res = fo.flashomni_gemm(*args, out=out0.clone().to(dev) if write_out else False, quant_out=(q8, sc))
    assert res[1].data_ptr() == q8.data_ptr() and res[2].data_ptr() == sc.data_ptr()
    if write_out:
        assert torch.equal(res[0].cpu().view(torch.int16), plain.view(torch.int16)), "16-bit result changed"
    else:
        assert res[0] is None
    # fp32 result of the flagged tiles (the oracle leaves the sentinel elsewhere)
    ref = oracle.gemm_q(x, w, heads, packed, indptr, 0, b, out=torch.zeros(batch, m, n, dtype=torch.float32))
    q8c, scc = q8.cpu(), sc.cpu()
    deq_all = q8c.float()
    for bi in range(batch):
        for iy in range(nqb):
            rows = slice(iy * 128, min(m, (iy + 1) * 128))
            for h in range(heads):
                cols = slice(h * 128, (h + 1) * 128)
                blk = bi * nqb + iy
                if not info[bi, iy, h]:
                    assert torch.equal(q8c.view(torch.uint8)[bi, rows, cols], q8_0[bi, rows, cols])
                    assert scc[h, blk] == -7.0
                    continue
                y = ref[bi, rows, cols].float()
                s = float(scc[h, blk])
                amax = float(y.abs().max())
                assert abs(s - amax / 448.0) <= 2e-3 * amax / 448.0 + 1e-12
                deq = deq_all[bi, rows, cols] * s
                # e4m3: 3 mantissa bits -> half a step is 2^-4 relative; subnormal step 2^-9 of the scale
                bound = 0.0625 * y.abs() + s * 2.0 ** -9 + 2e-3 * amax
                assert bool(((deq - y).abs() <= bound).all())
                assert float(deq_all[bi, rows, cols].abs().max()) == 448.0 or amax == 0.0
    # the residual term: same first term and scales, second term = e4m3(result / scale - first term)
    lo = torch.full((batch, m, n), 0x5A, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    q8b = q8_0.clone().to(dev).view(torch.float8_e4m3fn)
    res3 = fo.flashomni_gemm(*args, out=False, quant_out=(q8b, sc_0.clone().to(dev), lo))
    assert len(res3) == 4 and res3[3].data_ptr() == lo.data_ptr()
    assert torch.equal(q8b.cpu().view(torch.uint8), q8c.view(torch.uint8))
    two = deq_all + lo.cpu().float()
    for bi in range(batch):
        for iy in range(nqb):
            rows = slice(iy * 128, min(m, (iy + 1) * 128))
            for h in range(heads):
                cols = slice(h * 128, (h + 1) * 128)
                if not info[bi, iy, h]:
                    assert torch.equal(lo.cpu().view(torch.uint8)[bi, rows, cols], q8_0[bi, rows, cols])
                    continue
                y = ref[bi, rows, cols].float()
                s = float(scc[h, bi * nqb + iy])
                bound = 2.0 ** -8 * y.abs() + s * 2.0 ** -9 + 2e-3 * float(y.abs().max()) * 2.0 ** -4
                assert bool(((two[bi, rows, cols] * s - y).abs() <= bound).all())
    # the pair is what fp8 attention takes: against the separate quantiser on the 16-bit result
    if write_out and batch == 1 and p_active == 1.0:
        ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
        wr = fo.BatchFlashOmniFAWithRaggedKVWrapper(ws)
        ip = torch.tensor([0, m], dtype=torch.int32)
        wr.plan(ip, ip, heads, heads, 128, q_data_type=torch.float8_e4m3fn)
        g = torch.Generator().manual_seed(3)
        kk = torch.randn(m, heads, 128, generator=g).to(dtype).to(dev)
        vv = torch.randn(m, heads, 128, generator=g).to(dtype).to(dev)
        k8, ks = fo.quant_fp8_block(kk, ip)
        q_sep, qs_sep = fo.quant_fp8_block(res[0].view(m, heads, 128), ip)
        o_fused = wr.run(q8.view(m, heads, 128), k8, vv, is_full=True, q_scale=sc, k_scale=ks)
        o_sep = wr.run(q_sep, k8, vv, is_full=True, q_scale=qs_sep, k_scale=ks)
        assert rel_l2(o_fused.cpu(), o_sep.cpu()) <= 3e-2


def test_gemm_q_quant_argument_errors(dev):
    import flashomni_amd as fo
    x = torch.zeros(1, 128, 64, dtype=torch.bfloat16, device=dev)
    w = torch.zeros(256, 64, dtype=torch.bfloat16, device=dev)
    with pytest.raises(RuntimeError, match="out=False needs quant_out"):
        fo.flashomni_gemm(x, w, 2, is_full=True, out=False)
    with pytest.raises(RuntimeError, match="only 128"):
        fo.flashomni_gemm(x, w, 1, is_full=True, quant_out=True)       # one head of width 256
    with pytest.raises(RuntimeError, match=r"quant_out\[1\]"):
        fo.flashomni_gemm(x, w, 2, is_full=True,
                          quant_out=(torch.empty(1, 128, 256, dtype=torch.float8_e4m3fn, device=dev),
                                     torch.empty(2, 3, device=dev)))


def test_video_gemms_sampled_token_blocks(dev):
    """The 14B-video shape at full size (M=76112 with an 80-row last block, K=N=5120, 40 heads):
    GEMM-Q, the GEMM-O cache pass and the final pass run over the whole matrix; the first, the last
    and 10 seeded random token blocks are checked against the oracle, which is run on each block's
    rows alone with the text-token offset that makes it read that block's flags.  Weights ~ N(0, 0.02)
    as the configuration states: outputs have standard deviation 1.4 and a few of the 4 * 10^8 exceed
    8, where half a bf16 unit (2^-5) is above the 2e-2 bound: no bf16 result can be closer to the
    oracle's fp32 value than that, so from |y| = 8 on the bound is half a unit of y plus 2e-3."""
    import flashomni_amd as fo
    from flashomni_amd.workloads import make_workload
    wl = make_workload(4, tensors=False)
    s = wl.shape
    M, C, H = s.seq, s.hidden, s.heads
    g = torch.Generator(device=dev).manual_seed(41)
    rand = lambda *sz, std=1.0: (torch.randn(*sz, generator=g, device=dev) * std).to(torch.bfloat16)
    x, w_q, b_q, w_o, b_o = rand(1, M, C), rand(C, C, std=0.02), rand(C, std=0.02), rand(C, C, std=0.02), rand(C, std=0.02)

    def within_bound(got, exp):
        half_unit = torch.exp2(torch.floor(torch.log2(exp.abs().clamp_min(1.0))) - 8)
        bound = torch.where(exp.abs() < 8, torch.full_like(exp, MAX_ABS), half_unit + 2e-3)
        return bool(((got.float() - exp).abs() <= bound).all())

    pk, ip = wl.packed_info.to(dev), wl.info_indptr.to(dev)
    y = torch.full((1, M, C), -7.0, dtype=torch.bfloat16, device=dev)
    fo.flashomni_gemm(x, w_q, H, pk, ip, 0, b_q, out=y)
    active = wl.sparse_info.to(dev).repeat_interleave(128, 0)[:M].repeat_interleave(128, 1)[None]
    assert bool((y[~active] == -7.0).all())
    assert bool((y.view(-1, 128)[active.view(-1, 128)[:, 0]] != -7.0).any(-1).all())   # every flagged tile row written
    del active
    cache = fo.flashomni_gemm_reduction(x, w_o, H, pk, ip, 0, bias=b_o, is_for_cache=True,
                                        out_dtype=torch.float32)
    final = fo.flashomni_gemm_reduction(x, w_o, H, pk, ip, 0, bias=cache, is_for_cache=False)
    torch.cuda.synchronize()

    rng = np.random.default_rng(4)
    blocks = sorted({0, s.n_blocks - 1, *rng.choice(s.n_blocks, 10, replace=False).tolist()})
    wq_c, bq_c, wo_c, bo_c = w_q.cpu(), b_q.cpu(), w_o.cpu(), b_o.cpu()
    for iy in blocks:
        r0, r1 = iy * 128, min(M, iy * 128 + 128)
        xs = x[:, r0:r1].cpu()
        exp = oracle.gemm_q(xs, wq_c, H, wl.packed_info, wl.info_indptr, r0, bq_c,
                            out=torch.full((1, r1 - r0, C), -7.0, dtype=torch.float32))
        got = y[:, r0:r1].cpu()
        assert within_bound(got, exp), iy
        assert rel_l2(got, exp) <= REL_L2, iy
        exp_cache = oracle.gemm_o(xs, wo_c, H, wl.packed_info, wl.info_indptr, r0, bias=bo_c,
                                  is_for_cache=True, out_dtype=torch.float32)
        got_cache = cache[:, r0:r1].cpu()
        assert max_abs(got_cache, exp_cache) <= 2e-3, iy
        exp_final = oracle.gemm_o(xs, wo_c, H, wl.packed_info, wl.info_indptr, r0, bias=exp_cache,
                                  is_for_cache=False, out_dtype=torch.float32)
        got_final = final[:, r0:r1].cpu()
        assert within_bound(got_final, exp_final), iy
        assert rel_l2(got_final, exp_final) <= REL_L2, iy


def _check_gemm_o_rows(got, x, w, bias, info, text, cache, rows, hd):
    """Rows of a pass over x [batch, m, k] against the fp32 product of the heads that it selects (info: [batch, blocks, heads])."""
    for b in range(x.size(0)):
        on = torch.from_numpy(info[b, (np.array(rows) + text) // 128]).to(x.device).repeat_interleave(hd, 1)
        exp = (x[b, rows].float() * (~on if cache else on)) @ w.float().t()
        if bias is not None:
            exp = exp + (bias.float() if bias.dim() == 1 else bias[b, rows].float())
        scale = max(1.0, float(exp.abs().max()) / 2)
        assert max_abs(got[b, rows].cpu(), exp.cpu()) <= MAX_ABS * scale, b
        assert rel_l2(got[b, rows].cpu(), exp.cpu()) <= REL_L2, b


def _some_rows(m, step):
    return sorted(r for r in {0, 1, 127, 128, m // 2, m - 1} | set(range(5, m, step)) if r < m)


@pytest.mark.parametrize("shape", [(1, 22016, 3072, 24), (2, 43800, 768, 8)])
def test_long_gemm_o_leaves_scratch_alone(dev, shape):
    """Long launches, both passes: rows of every part of the output against the selected heads' fp32 product, and the
    same bits whether the entry point is given scratch memory, which it neither reads nor writes, or none.  (22016 x 3072: 172
    token blocks, 2064 strips; the second shape has two batch entries, a ragged last token block and heads of width 96,
    i.e. slabs that count for one half only.)"""
    import flashomni_amd as fo
    from flashomni_amd import _lib
    batch, m, n, heads = shape
    info, packed, indptr = _flags(batch, (m + 127) // 128, heads, 0.3, seed=77)
    g = torch.Generator(device=dev).manual_seed(78)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    code = _lib.dtype_code(torch.bfloat16)
    rows = _some_rows(m, 997)
    for is_for_cache, bias, kind in ((True, b, _lib.FO_BIAS_VECTOR), (False, None, _lib.FO_BIAS_MATRIX)):
        if bias is None:
            bias = got_cache
        got = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, bias=bias, is_for_cache=is_for_cache)
        for word in (7, 0):
            scratch = torch.full((64,), word, dtype=torch.int32, device=dev)
            bare = torch.full_like(got, -3.0)
            with _lib.device_guard(dev):
                _lib.check(_lib.lib().fo_gemm_o(
                    _lib.ptr(x), _lib.ptr(w), _lib.ptr(bias), _lib.ptr(bare), code, kind, code, code, batch, m, n, n,
                    128, heads, _lib.ptr(pk), _lib.ptr(ip), 0, int(is_for_cache), _lib.ptr(scratch), 256,
                    _lib.current_stream(dev)))
            assert torch.equal(got.view(torch.int16), bare.view(torch.int16))
            assert bool((scratch == word).all())
        _check_gemm_o_rows(got, x, w, bias, info, 0, is_for_cache, rows, n // heads)
        got_cache = got
    # and the end result is the dense layer
    dense = F.linear(x[0, :256].float(), w.float(), b.float()).cpu()
    assert rel_l2(got[0, :256].cpu(), dense) <= REL_L2


@pytest.mark.parametrize("case", [(1, 128, 1), (129, 128, 1), (1100, 64, 4), (1100, 128, 8), (2176, 96, 4), (3000, 256, 8),
                                  (130, 32, 12)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_units_equal_many(dev, case, dtype):
    """Launches of up to two units per CU give a unit or a pair of them a CU of its own, longer ones compute quads, strips or
    (GEMM-O up to 512 columns) packed units: the same inputs alone and as one of many batch entries give the same bits,
    because all add a unit's k steps in the same order.  One and two token rows past a block, heads of 32 to 256 columns (slabs
    that count for one half only), every unit of the chip in use (3000 x 2048: 384 units, 192 pairs)."""
    import flashomni_amd as fo
    m, hd, heads = case
    n = heads * hd
    units = -(-m // 128) * (n // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert units <= 2 * cus
    batch = 2 * cus // units + 1
    info, packed, indptr = _flags(batch, -(-m // 128) + 1, heads, 0.6, seed=m + hd)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)

    def chain(x, ip):
        q = torch.full_like(x, -3.0)
        fo.flashomni_gemm(x, w, heads, pk, ip, 128, b, out=q)
        full = fo.flashomni_gemm(x, w, heads, num_text_tokens=0, bias=b, is_full=True)
        part = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=b, is_for_cache=True)
        part32 = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, is_for_cache=True, out_dtype=torch.float32)
        return [q, full, part, part32, fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=part),
                fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=part32)]

    many = chain(x, ip)
    for i in sorted({0, batch // 2, batch - 1}):
        for k, (one, all_) in enumerate(zip(chain(x[i:i + 1].contiguous(), ip[i:i + 2].contiguous()), many)):
            if k == 0:
                ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
                assert torch.allclose(one[0].float(), all_[i].float(), rtol=ulp, atol=n * 2.0 ** -24), i
            else:
                assert torch.equal(one[0], all_[i]), (i, k)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(1100, 8, 8, 25), (130, 8, 33, 128), (1025, 10, 6, 20)])
def test_packed_units_equal_quads(dev, case, dtype):
    """Dense GEMM-Q whose quads would fill their rounds badly runs four workgroups of one unit each on a CU, a better
    filled one quads: the same inputs as a few batch entries and as one of many give the same bits.  One and two token rows
    past a block, an odd number of row and column blocks."""
    import flashomni_amd as fo
    m, cols, few, many = case
    n = cols * 128
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    rows = -(-m // 128)
    fill = lambda batch: batch * rows * cols / (4 * cus * -(-batch * ((cols + 1) // 2) * ((rows + 1) // 2) // cus))
    if cus == 256:
        assert few * rows * cols > 2 * cus and fill(few) <= 42 / 64 and fill(many) > 49 / 64
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(many, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    full = lambda x: fo.flashomni_gemm(x, w, cols, num_text_tokens=0, bias=b, is_full=True)
    one, everything = full(x[:few].contiguous()), full(x)
    assert torch.equal(one, everything[:few])
    ref = torch.nn.functional.linear(x[:few].float(), w.float(), b.float())
    assert rel_l2(one, ref) <= REL_L2


def _chain_of_passes(x, w, b, heads, pk, ip, text):
    """GEMM-O's cache pass with either output type and the final pass over either."""
    import flashomni_amd as fo
    o = lambda bias, cache, dtype=None: fo.flashomni_gemm_reduction(x, w, heads, pk, ip, text, bias=bias, is_for_cache=cache,
                                                                    out_dtype=dtype)
    part, part32 = o(b, True), o(b, True, torch.float32)
    return [part, part32, o(part, False), o(part32, False, torch.float32)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(8500, 128, 4, 2), (4000, 64, 6, 6), (9001, 128, 2, 4), (1, 128, 4, 140), (2100, 64, 6, 11)])
def test_packed_gemm_o_equals_one_unit_per_cu(dev, case, dtype):
    """GEMM-O up to 512 columns: more units than two per CU run four workgroups of one each on a CU.  A batch entry alone, of
    at most a unit or a pair of them per CU, gives the same bits, in both passes, with either output and partial type; rows against
    the selected heads' fp32 product."""
    import flashomni_amd as fo
    m, hd, heads, batch = case
    n, rows = hd * heads, -(-m // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert n <= 512 and (cus != 256 or (batch * rows * (n // 128) > 2 * cus >= 2 * rows * -(-n // 256)))
    info, packed, indptr = _flags(batch, rows + 1, heads, 0.6, seed=m)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.05).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.05).to(dtype)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    many = _chain_of_passes(x, w, b, heads, pk, ip, 128)
    for i in sorted({0, batch // 2, batch - 1}):
        alone = _chain_of_passes(x[i:i + 1].contiguous(), w, b, heads, pk, ip[i:i + 2].contiguous(), 128)
        for one, all_ in zip(alone, many):
            assert torch.equal(one[0], all_[i]), i
    _check_gemm_o_rows(many[1], x, w, b, info, 128, True, _some_rows(m, 317), hd)
    _check_gemm_o_rows(many[3], x, w, many[1], info, 128, False, _some_rows(m, 317), hd)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(1025, 128, 40), (1407, 160, 32), (1500, 320, 16), (16513, 128, 3), (20001, 96, 4), (33000, 64, 2)])
def test_gemm_o_units_two_to_a_cu(dev, case, dtype):
    """One to two units per CU whose pairs are more than one per CU or whose width is above 4096: a workgroup per unit, two on a
    CU.  Both passes, with either output and partial type, against the selected heads' fp32 product; the same bits as one of two batch
    entries, which strips or packed units compute.  Heads of 160, 320 and 96 columns: slabs of which one half counts."""
    m, hd, heads = case
    n, rows = hd * heads, -(-m // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    units, pairs = rows * (n // 128), rows * -(-n // 256)
    if cus == 256:
        assert cus < units <= 2 * cus < 2 * units and (pairs > cus or n > 4096)
    info, packed, indptr = _flags(2, rows + 1, heads, 0.6, seed=m)
    info[0, 0], info[0, 1] = False, True   # (the text block's flags; a block with every head)
    segs = [np.packbits(f.reshape(-1).astype(np.uint8), bitorder="little") for f in info]
    pk = torch.from_numpy(np.concatenate(segs)).to(dev)
    ip = torch.from_numpy(np.cumsum([0] + [len(f) for f in segs]).astype(np.int32)).to(dev)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(2, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    both = _chain_of_passes(x, w, b, heads, pk, ip, 128)
    for i in range(2):
        xi, ii = x[i:i + 1].contiguous(), info[i:i + 1]
        alone = _chain_of_passes(xi, w, b, heads, pk, ip[i:i + 2].contiguous(), 128)
        for one, all_ in zip(alone, both):
            assert torch.equal(one[0], all_[i]), i
        for out, cache in ((alone[0], True), (alone[1], True), (alone[2], False), (alone[3], False)):
            bias = b if cache else alone[0] if out is alone[2] else alone[1]
            _check_gemm_o_rows(out, xi, w, bias, ii, 128, cache, _some_rows(m, 131), hd)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [64, 96, 352, 384])
@pytest.mark.parametrize("shape", [(1, 18001, 384, 0), (1, 33000, 128, 128), (2, 9100, 384, 0)])
def test_gemm_q_units_two_to_a_cu(dev, shape, k, dtype):
    """The same for GEMM-Q, dense and flagged (half, none, all): an odd number of column blocks, whose pairs are more than the
    CUs.  Against the fp32 product, rounded once; tiles that are not flagged keep their bytes.  K of one slab, of 32 mod 64."""
    import flashomni_amd as fo
    batch, m, n, text = shape
    rows, heads = -(-m // 128), n // 128
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or (cus < batch * rows * heads <= 2 * cus and batch * rows * -(-n // 256) > cus)
    x, w, b = (t.to(dev) for t in _operands(batch, m, n, k, dtype, seed=k))
    ref = torch.nn.functional.linear(x.float(), w.float(), b.float())
    half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -11)
    # (one rounding; sums of k products in another order: k * 2^-24 of the sum of their sizes, below 16 standard deviations of one)
    bound = 2 * half_ulp * ref.abs() + k * 2.0 ** -24 * 16 * 0.02
    full = fo.flashomni_gemm(x, w, heads, num_text_tokens=0, bias=b, is_full=True)
    assert bool(((full.float() - ref).abs() <= bound).all())
    for p in (0.0, 0.5, 1.0):
        info, packed, indptr = _flags(batch, text // 128 + rows, heads, p, seed=m)
        out = torch.full((batch, m, n), -7.0, dtype=dtype, device=dev)
        fo.flashomni_gemm(x, w, heads, torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev), text, b, out=out)
        on = torch.from_numpy(info[:, text // 128:]).to(dev).repeat_interleave(128, 1)[:, :m].repeat_interleave(128, 2)
        assert bool((out[~on] == -7.0).all())
        assert torch.equal(out[on], full[on])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(1025, 128, 5, 14), (130, 96, 8, 48), (257, 64, 70, 5), (384, 32, 132, 6), (1, 32, 256, 9),
                                  (2177, 320, 4, 4), (3, 128, 5, 4100)])
def test_strips_equal_units(dev, case, dtype):
    """GEMM-O of many units computes strips of one token block x two column blocks, few units one at a time: a batch
    entry alone and among many gives the same bits, in both passes, with either output and partial type.  Requests with
    no head selected anywhere, with one head (a list of one slab), with all of them; one, two, three and more token rows
    past a block; an odd number of column blocks; heads of 32 to 320 columns, so slabs of which one half counts, at the
    beginning of the matrix too; 5 to 256 heads (one to four words of flags); more token blocks than are put in order."""
    import flashomni_amd as fo
    m, hd, heads, batch = case
    n, rows = heads * hd, -(-m // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert n > 512 and rows * (n // 128) <= 2 * 256 and (cus != 256 or batch * rows * (n // 128) > 2 * cus)
    rng = np.random.default_rng(m + heads)
    info = rng.random((batch, rows + 1, heads)) < rng.random((batch, rows + 1, 1))
    info[0], info[-1] = True, False
    info[1] = np.arange(heads) == rng.integers(heads, size=(rows + 1, 1))
    segs = [np.packbits(f.reshape(-1).astype(np.uint8), bitorder="little") for f in info]
    pk = torch.from_numpy(np.concatenate(segs)).to(dev)
    ip = torch.from_numpy(np.cumsum([0] + [len(f) for f in segs]).astype(np.int32)).to(dev)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)

    def chain(x, ip):
        part = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=b, is_for_cache=True)
        part32 = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=b, is_for_cache=True, out_dtype=torch.float32)
        return [part, part32, fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=part),
                fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 128, bias=part32, out_dtype=torch.float32)]

    many = chain(x, ip)
    for i in sorted({0, 1, batch // 2, batch - 1}):
        for k, (one, all_) in enumerate(zip(chain(x[i:i + 1].contiguous(), ip[i:i + 2].contiguous()), many)):
            assert torch.equal(one[0], all_[i]), (i, k)
    dense = torch.nn.functional.linear(x.float(), w.float(), b.float())
    assert rel_l2(many[3], dense) <= 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 129, 384, k) for k in (64, 96, 128, 256, 288, 320, 384, 672, 704)] +
                         [(1, 1, 128, 5120), (2, 16384, 128, 64), (1, 2603, 3072, 96), (3, 900, 2304, 128), (3, 900, 2304, 160), (1, 130, 17664, 64), (1, 300, 12672, 352),
                          (1, 33000, 256, 64), (1, 32641, 256, 160)])
def test_dense_gemm_q_of_one_and_two_units_per_cu(dev, shape, dtype):
    """Up to 256 units: one per CU, through a ring of five slabs (one to eleven of them, of which the last may count for one
    half).  Up to 512: strips with a CU each, through a ring of three, odd numbers of column blocks, one strip too many for a round.
    Against the fp32 product."""
    import flashomni_amd as fo
    batch, m, n, k = shape
    g = torch.Generator(device=dev).manual_seed(m + k)
    x = torch.randn(batch, m, k, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, k, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    out = torch.full((batch, m, n), float("nan"), dtype=dtype, device=dev)
    y = fo.flashomni_gemm(x, w, n // 128, num_text_tokens=0, bias=b, is_full=True, out=out)
    ref = torch.nn.functional.linear(x.float(), w.float(), b.float())
    half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -11)
    # (one rounding; sums of k products in another order: k * 2^-24 of the sum of their sizes, below 16 standard deviations of one)
    assert bool(((y.float() - ref).abs() <= 2 * half_ulp * ref.abs() + k * 2.0 ** -24 * 16 * 0.02).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 26003, 512, 512), (3, 10497, 384, 96), (1, 7289, 3072, 3072), (2, 3650, 2944, 2976)])
def test_dense_gemm_q_as_strips(dev, shape, dtype):
    """Full GEMM-Q of narrow matrices and of rounds of quads that end half empty: strips.  Ragged last rows, an odd number
    of column blocks, K of 32 mod 64; against the fp32 product (the result is rounded once: half a unit of its last place)."""
    import flashomni_amd as fo
    batch, m, n, k = shape
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, k, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, k, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    y = fo.flashomni_gemm(x, w, n // 128, num_text_tokens=0, bias=b, is_full=True)
    ref = torch.nn.functional.linear(x.float(), w.float(), b.float())
    half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -11)
    # (sums of k products in another order: k * 2^-24 of the sum of their sizes, below 16 standard deviations of one)
    assert bool(((y.float() - ref).abs() <= 2 * half_ulp * ref.abs() + k * 2.0 ** -24 * 16 * 0.02).all())
    assert rel_l2(y, ref) <= half_ulp


@pytest.mark.parametrize("p_active", [0.0, 0.05, 0.35, 0.65, 0.95, 1.0])
@pytest.mark.parametrize("text", [0, 256])
def test_long_gemm_o_at_every_density(dev, p_active, text):
    """Both passes of a long call of eight heads, none to all of them selected, flags from a text token on: rows of
    every part against the selected heads' fp32 product."""
    import flashomni_amd as fo
    m, n, heads, batch = 16384 - 5, 1024, 8, 3
    info, packed, indptr = _flags(batch, (text + m + 127) // 128, heads, p_active, seed=int(100 * p_active) + text)
    g = torch.Generator(device=dev).manual_seed(text)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    for cache in (True, False):
        y = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, text, is_for_cache=cache)
        _check_gemm_o_rows(y, x, w, None, info, text, cache, _some_rows(m, 501), 128)


@pytest.mark.parametrize("shape,p_active", [
    ((8192, 2560), (0.05, 0.95, 0.95)), ((8192, 2560), (0.95, 0.05, 0.05)), ((8192, 2560), (0.1, 0.3, 0.2)),
    ((8192, 2560), (0.9, 0.7, 0.8)), ((8192, 2560), (0.0, 0.0, 0.0)), ((8192, 2560), (1.0, 1.0, 1.0)),
    ((512, 2560), (0.05,) * 35 + (0.9,) * 35),
    ((9609, 3072), (0.5,)), ((9609, 3072), (0.8,)),
])
def test_gemm_o_of_a_mixed_batch(dev, shape, p_active):
    """Requests of unlike densities in one call, whose token blocks are put in order of their selected heads across the
    batch: each request's rows against the selected heads' fp32 product, and the same bits as the request by itself (512
    tokens: a workgroup per unit there), in either pass."""
    import flashomni_amd as fo
    batch, (m, n), text = len(p_active), shape, 128
    heads, blocks = n // 128, -(-m // 128)
    flags = np.concatenate([_flags(1, blocks + 1, heads, p, seed=7 + i)[0] for i, p in enumerate(p_active)])
    segs = [np.packbits(f.reshape(-1).astype(np.uint8), bitorder="little") for f in flags]
    info, indptr = np.concatenate(segs), np.cumsum([0] + [len(s) for s in segs]).astype(np.int32)
    g = torch.Generator(device=dev).manual_seed(batch)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    pk, ip = torch.from_numpy(info).to(dev), torch.from_numpy(indptr).to(dev)
    for cache in (True, False):
        y = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, text, is_for_cache=cache)
        _check_gemm_o_rows(y, x, w, None, flags, text, cache, _some_rows(m, 701), 128)
        for i in sorted({0, batch // 2, batch - 1}) if batch > 1 else ():
            one = fo.flashomni_gemm_reduction(x[i:i + 1].contiguous(), w, heads, pk, ip[i:i + 2].contiguous(), text,
                                              is_for_cache=cache)
            assert torch.equal(one[0], y[i]), i


@pytest.mark.parametrize("shape", [(1, 6200, 1536), (1, 6300, 1536), (1, 16100, 2048), (1, 8185, 3072), (2, 3300, 2560),
                                   (1, 4090, 5120), (1, 2553, 5120)])
def test_gemm_o_sampled_rows(dev, shape):
    """Shapes of 2.3 to 8 units per CU, narrow and wide, an odd number of token blocks among them: sampled rows of both passes
    against the fp32 product of the selected heads."""
    import flashomni_amd as fo
    batch, m, n = shape
    heads, blocks = n // 128, -(-m // 128)
    info, packed, indptr = _flags(batch, blocks, heads, 0.6, seed=m)
    g = torch.Generator(device=dev).manual_seed(m)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    part = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, is_for_cache=True, out_dtype=torch.float32)
    y = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, bias=part)
    rows = sorted({0, 1, 127, 128, m // 2, m - 1} | set(range(5, m, 977)))
    for b in range(batch):
        a = x[b, rows].float()
        on = torch.from_numpy(info[b, np.array(rows) // 128]).to(dev).repeat_interleave(128, 1)
        for got, exp in ((part, (a * ~on) @ w.float().t()), (y, a @ w.float().t())):
            assert max_abs(got[b, rows], exp) <= MAX_ABS * max(1.0, float(exp.abs().max()) / 2) and rel_l2(got[b, rows], exp) <= REL_L2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch", [1, 2, 5])
def test_fp32_output_rounds_to_the_16_bit_one(dev, batch, dtype):
    """GEMM-O forms the same fp32 value whatever it stores: the fp32 result rounded is the 16-bit result,
    without a bias, with a bias vector and with a cached partial, in launches of few and of many units.
    (The fp32 store once read a data register that the next instruction had already overwritten: runs
    of four rows whose every fourth column held another row's value.)"""
    import flashomni_amd as fo
    m, n, heads = 3000, 2048, 8
    info, packed, indptr = _flags(batch, (m + 127) // 128, heads, 0.6, seed=5)
    g = torch.Generator(device=dev).manual_seed(6)
    x = torch.randn(batch, m, n, generator=g, device=dev).to(dtype)
    w = (torch.randn(n, n, generator=g, device=dev) * 0.02).to(dtype)
    b = (torch.randn(n, generator=g, device=dev) * 0.02).to(dtype)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    part = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, bias=b, is_for_cache=True)
    for bias, cache in ((None, True), (b, True), (part, False), (part.float(), False)):
        short = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, bias=bias, is_for_cache=cache)
        for _ in range(4):
            wide = fo.flashomni_gemm_reduction(x, w, heads, pk, ip, 0, bias=bias, is_for_cache=cache,
                                               out_dtype=torch.float32)
            assert torch.equal(wide.to(dtype), short)


@pytest.mark.parametrize("flagged", [0.0, 0.004, 0.05, 0.2, 0.4, 0.7])
@pytest.mark.parametrize("shape", [(1, 4357, 2048, 160, 0), (2, 2100, 2176, 64, 128), (1, 8192, 2048, 128, 0),
                                   (3, 1000, 3200, 96, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_q_few_flagged_units(dev, shape, flagged, dtype):
    """More units than two per CU but few of them flagged: work items of at most two units, a unit's k
    shared by two wavefronts; with more flagged, quads.  Ragged last rows, an odd number of column blocks, K
    of one slab, of two and of 32 mod 64, none and single units flagged; skipped tiles keep their bytes."""
    import flashomni_amd as fo
    batch, m, n, k, text = shape
    heads = n // 128
    assert batch * -(-m // 128) * heads > 2 * torch.cuda.get_device_properties(dev).multi_processor_count
    info, packed, indptr = _flags(batch, (text + m + 127) // 128, heads, flagged, seed=m + int(1000 * flagged))
    x, w, b = _operands(batch, m, n, k, dtype, seed=k)
    out0 = sentinel_like((batch, m, n), dtype)
    out = out0.clone().to(dev)
    fo.flashomni_gemm(x.to(dev), w.to(dev), heads, torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev),
                      text, b.to(dev), out=out)
    exp = oracle.gemm_q(x, w, heads, packed, indptr, text, b, out=out0.clone())
    out = out.cpu()
    rows = torch.arange(m) // 128 + text // 128
    kept = torch.from_numpy(info)[:, rows].repeat_interleave(128, dim=2)
    assert torch.equal(out.view(torch.int16)[~kept], out0.view(torch.int16)[~kept])
    if kept.any():
        assert max_abs(out[kept], exp[kept]) <= MAX_ABS
        assert rel_l2(out[kept], exp[kept]) <= REL_L2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", [(1, 25000, 768, 64, 6, 0, 0.5), (1, 170000, 768, 96, 6, 0, 0.3), (2, 9050, 2432, 160, 19, 256, 0.6),
                                  (1, 8100, 2560, 128, 40, 128, 0.5), (1, 19200, 1280, 64, 5, 0, 0.4), (3, 1409, 5248, 96, 41, 0, 0.2),
                                  (2, 1500, 8960, 64, 70, 0, 0.05), (1, 20000, 1024, 64, 8, 0, 0.0), (1, 20000, 1024, 64, 8, 0, 1.0)])
def test_gemm_q_flagged_strips(dev, case, dtype):
    """GEMM-Q with flags of 4.5 to 32 units per CU: strips of one token block x two of its flagged column blocks, which need not
    be neighbours.  One token block to six (more than are counted together) per thread that counts; one and two groups of columns, of
    more than 64 columns in all; odd numbers of flagged and of column blocks; heads of 64 columns (a column block reads the
    flag of its first head) and of 256; a batch, text tokens, ragged last rows, K of 32 mod 64; none and all flagged.  Skipped
    tiles keep their bytes."""
    import flashomni_amd as fo
    batch, m, n, k, heads, text, flagged = case
    rows = -(-m // 128)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert cus != 256 or 4.5 * cus < batch * rows * (n // 128) <= (32 if n <= 4096 else 16) * cus
    info, packed, indptr = _flags(batch, (text + m + 127) // 128, heads, flagged, seed=m)
    x, w, b = _operands(batch, m, n, k, dtype, seed=k)
    out = sentinel_like((batch, m, n), dtype).to(dev)
    out0 = out.clone()
    x, w, b = x.to(dev), w.to(dev), b.to(dev)
    fo.flashomni_gemm(x, w, heads, torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev), text, b, out=out)
    tile_head = (np.arange(n // 128) * 128) // (n // heads)
    kept = torch.from_numpy(info[:, text // 128:][:, :rows, tile_head]).to(dev)
    half_ulp = 2.0 ** (-9 if dtype == torch.bfloat16 else -11)
    for i in range(batch):
        mask = kept[i].repeat_interleave(128, 0)[:m].repeat_interleave(128, 1)
        assert torch.equal(out[i].view(torch.int16)[~mask], out0[i].view(torch.int16)[~mask])
        ref = torch.nn.functional.linear(x[i].float(), w.float(), b.float())[mask]
        got = out[i].float()[mask]
        # one rounding; sums of k products in another order: k * 2^-24 of the sum of their sizes, below 16 standard deviations of one
        assert bool(((got - ref).abs() <= 2 * half_ulp * ref.abs() + k * 2.0 ** -24 * 16 * 0.02).all())


@pytest.mark.parametrize("seed", range(24))
def test_random_gemm_shapes(dev, seed):
    """Seeded random shapes through GEMM-Q (flags or is_full) and the two passes of GEMM-O (the cached
    partial in 16 bits or fp32): batches, M with and without a tail, head widths 32 to 256, text-token
    offsets, K = 32 mod 64, all-zero and all-one flags.  Skipped tiles keep their bytes; results within
    max-abs 2e-2 (per unit of output magnitude above 2, where one bf16 ulp is 1.6e-2 and more) and
    relative L2 1e-2 of the fp32 oracle."""
    import flashomni_amd as fo
    rng = np.random.default_rng(1000 + seed)
    batch = int(rng.choice([1, 1, 2, 3]))
    m = int(rng.choice([1, 100, 128, 129, 300, 512, 1000, 2176]))
    hd = int(rng.choice([32, 64, 96, 128, 128, 256]))
    heads = int(rng.choice([1, 2, 3, 5, 8]))
    if (heads * hd) % 128:
        heads *= 128 // int(np.gcd(heads * hd, 128))
    n = heads * hd
    text = int(rng.choice([0, 0, 128, 512]))
    dtype = torch.bfloat16 if rng.random() < 0.6 else torch.float16
    p = float(rng.choice([0.0, 0.25, 0.6, 1.0]))
    kind = ["q", "q_full", "o"][seed % 3]
    k = n if kind == "o" else int(rng.choice([64, 96, 128, 160, 256, 512, 1056]))
    info, packed, indptr = _flags(batch, (text + m + 127) // 128, heads, p, seed=seed)
    x, w, b = _operands(batch, m, n, k, dtype, seed=seed)
    pk, ip = torch.from_numpy(packed).to(dev), torch.from_numpy(indptr).to(dev)
    bound = lambda e: MAX_ABS * max(1.0, float(e.float().abs().max()) / 2)
    if kind != "o":
        full = kind == "q_full"
        out0 = sentinel_like((batch, m, n), dtype)
        out = out0.clone().to(dev)
        fo.flashomni_gemm(x.to(dev), w.to(dev), heads, None if full else pk, None if full else ip, text, b.to(dev),
                          out=out, is_full=full)
        exp = oracle.gemm_q(x, w, heads, packed, indptr, text, b, out=out0.clone(), is_full=full)
        got = out.cpu()
        computed = torch.zeros(batch, m, n, dtype=torch.bool)
        for bi in range(batch):
            for iy in range((m + 127) // 128):
                for ix in range(n // 128):
                    if full or info[bi, (text + iy * 128) // 128, (ix * 128) // hd]:
                        computed[bi, iy * 128:iy * 128 + 128, ix * 128:ix * 128 + 128] = True
        assert torch.equal(got[~computed].view(torch.int16), out0[~computed].view(torch.int16))
        if computed.any():
            assert max_abs(got[computed], exp[computed]) <= bound(exp[computed])
            assert rel_l2(got[computed], exp[computed]) <= REL_L2
    else:
        od = torch.float32 if seed % 2 else None
        cache = fo.flashomni_gemm_reduction(x.to(dev), w.to(dev), heads, pk, ip, text, bias=b.to(dev),
                                            is_for_cache=True, out_dtype=od)
        final = fo.flashomni_gemm_reduction(x.to(dev), w.to(dev), heads, pk, ip, text, bias=cache, is_for_cache=False)
        e_cache = oracle.gemm_o(x, w, heads, packed, indptr, text, bias=b, is_for_cache=True, out_dtype=od)
        e_final = oracle.gemm_o(x, w, heads, packed, indptr, text, bias=e_cache, is_for_cache=False)
        for got, exp in ((cache.cpu(), e_cache), (final.cpu(), e_final)):
            assert max_abs(got, exp) <= bound(exp) and rel_l2(got, exp) <= REL_L2
