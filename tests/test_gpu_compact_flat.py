"""One-launch compaction of one long lane (compact_flat): bit-exact against
oracle.compact at the edges of its range and of its 1024-token workgroups, with
segment bounds everywhere, empty and full masks, mask bytes other than 1, and a
mask that does not start at 16 bytes (which takes the three launches)."""

import numpy as np
import pytest
import torch

from logo_amd import _lib
from logo_amd.ops.common import compact_selection
from oracle import compact

pytestmark = pytest.mark.gpu


def _check(dsel, want, cu, n):
    m = dsel.meta.cpu().numpy()
    ns = len(cu) - 1
    sq = want["Sq"]
    assert [m[0], m[3], m[4]] == [sq, n, ns]
    tq, tk = compact.chunk_prefix(want["cu_seqlens_q"], _lib.BQ), compact.chunk_prefix(cu, _lib.BKV)
    assert np.array_equal(m[8:9 + ns], want["cu_seqlens_q"])
    assert np.array_equal(m[9 + ns:10 + 2 * ns], tq) and np.array_equal(m[10 + 2 * ns:11 + 3 * ns], tk)
    assert m[1] == tq[-1] and m[2] == tk[-1]
    assert np.array_equal(dsel.q_idx[0, :sq].cpu().numpy(), want["q_idx"])
    assert np.array_equal(dsel.pos[0, :sq].cpu().numpy(), want["pos_ids"])
    assert int(dsel.q_idx[0, sq:].count_nonzero()) == 0 and int(dsel.pos[0, sq:].count_nonzero()) == 0


@pytest.mark.parametrize("n", [4097, 5119, 5120, 5121, 32768, 40003, 131071, 131072, 131073])
@pytest.mark.parametrize("ratio", [0.0, 0.3, 1.1])
@pytest.mark.parametrize("offset", [0, 3])
def test_bit_exact(gpu, n, ratio, offset):
    rng = np.random.default_rng(n + offset)
    sel = rng.random(n) < ratio
    cuts = np.sort(rng.integers(0, n + 1, 300 if n % 2 else 2))
    cu = np.concatenate([[0], cuts, [n]]).astype(np.int32)
    buf = torch.zeros(n + 16, dtype=torch.bool, device=gpu)
    view = buf[offset:offset + n]
    view.copy_(torch.from_numpy(sel))
    dsel = compact_selection(view, torch.from_numpy(cu).to(gpu))
    _check(dsel, compact.build_selection(sel, cu)[0], cu, n)


def test_any_nonzero_byte_counts(gpu):
    n = 6000
    rng = np.random.default_rng(0)
    raw = (rng.random(n) < 0.4) * rng.integers(1, 256, n)
    cu = np.array([0, 1, 1, 2050, n], dtype=np.int32)
    from logo_amd import _torch_ops

    q_idx, pos, meta = _torch_ops.ops().compact(torch.from_numpy(raw.astype(np.uint8)).to(gpu),
                                                torch.from_numpy(cu).to(gpu))
    want = compact.build_selection(raw != 0, cu)[0]
    assert int(meta[0]) == want["Sq"]
    assert np.array_equal(q_idx[0, :want["Sq"]].cpu().numpy(), want["q_idx"])
    assert np.array_equal(pos[0, :want["Sq"]].cpu().numpy(), want["pos_ids"])
