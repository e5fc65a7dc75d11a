"""GPU: the pieces behind the native call path against the oracle or a plain restatement: bit packing with
offsets worked out on the device, and the tables of a planned batch."""
import numpy as np
import pytest
import torch

import oracle

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
