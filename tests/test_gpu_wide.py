"""Head dim 256 in 16-bit types (logo_amd/csrc/wide_attn.hip) at the edges of
its tiles: 32-key halves and 64-key tiles, 128-row query tiles, 64-key blocks
and 32-row steps of dk / dv, one to many steps of its four-tile rings, key
ranges cut into pieces, GQA, per-head rows, packed and empty segments, fp16 and
dense rows; against the float64 oracle with the bound the generic kernels of
the same head dim are held to.  The CPU test checks the assembled kernels'
asm-MFMA accumulators with the checker of the tuned ones.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import attn
from tests import test_isa_accumulators as isa
from tests.helpers import assert_within, gen, randn

D = 256


def _check(gpu, lens, hq, h, rows, dtype=torch.bfloat16, per_head=False, seed=0):
    """rows: share of tokens selected, None for dense rows."""
    from logo_amd.ops import dense_causal_attn, sq_full_attn

    n = sum(lens)
    g = gen(1200 + n + hq + seed)
    q, k, v, do = (randn((n, x, D), g, dtype=dtype) for x in (hq, h, h, hq))
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    sel = None if rows is None else torch.rand((n, hq) if per_head else (n,), generator=g) < rows
    qg, kg, vg = (x.to(gpu)[None].requires_grad_() for x in (q, k, v))
    if sel is None:
        o = dense_causal_attn(qg, kg, vg, cu.to(gpu))
    else:
        o = sq_full_attn(qg, kg, vg, sel.to(gpu)[None], cu_seqlens=cu.to(gpu))
    o.backward(do.to(gpu)[None])
    qn, kn, vn, dn = (x.double().numpy() for x in (q, k, v, do))
    s = None if sel is None else sel.numpy()
    ro, _ = attn.sq_attn_fwd(qn, kn, vn, s, cu.numpy())
    rdq, rdk, rdv = attn.sq_attn_bwd(qn, kn, vn, ro, dn, s, cu.numpy())
    for name, x, r in (("o", o, ro), ("dq", qg.grad, rdq), ("dk", kg.grad, rdk), ("dv", vg.grad, rdv)):
        assert_within(f"{name} {lens} hq={hq} h={h} rows={rows}", x[0], r,
                      max_abs=2e-2 * max(1.0, float(np.abs(r).max()) / 2))
    if sel is not None and not per_head:
        assert torch.all(o[0][~sel.to(gpu)] == 0) and torch.all(qg.grad[0][~sel.to(gpu)] == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[1], [31], [32], [33], [63, 65], [64, 1, 0, 127], [128], [129], [160, 97], [257]])
def test_tile_edges_every_row_selected(gpu, lens):
    _check(gpu, lens, 2, 1, 1.1)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[1], [31], [32], [33], [63, 65], [64, 1, 0, 127], [129], [160, 97]])
def test_tile_edges_beside_a_long_segment(gpu, lens):
    """(the forward of segments below 352 tokens on average is the generic one)"""
    _check(gpu, [1900] + lens, 2, 1, 1.1)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,hq,h,rows,per_head,dtype", [
    ([1500], 2, 2, 0.3, False, torch.bfloat16),       # rings and rounds of several steps, split key ranges
    ([700, 1, 650], 4, 1, 0.15, False, torch.bfloat16),
    ([900], 4, 2, 0.5, True, torch.bfloat16),
    ([513, 200], 2, 1, 0.4, False, torch.float16),
    ([300, 301], 2, 1, None, False, torch.bfloat16),  # dense rows
    ([1100], 8, 4, 0.02, False, torch.bfloat16),      # few rows
    ([639], 2, 2, 1.1, False, torch.bfloat16),        # one key fewer than is cut, and the fewest that are
    ([640], 2, 2, 1.1, False, torch.bfloat16),
    ([4500], 16, 16, 0.13, False, torch.bfloat16),    # pieces that take turns on the CUs
])
def test_longer_sequences(gpu, lens, hq, h, rows, per_head, dtype):
    _check(gpu, lens, hq, h, rows, dtype, per_head)


@pytest.mark.skipif(not (os.path.exists(isa.LIB) and shutil.which(f"{isa.LLVM}/llvm-objdump")),
                    reason="needs the built library and ROCm's llvm-objdump")
def test_asm_accumulators_are_drained_before_use(tmp_path):
    listings, name = {}, None
    for j, obj in enumerate(isa._gfx950_objects(isa.LIB, tmp_path)):
        if b"w256_dkv_kernel" not in obj:
            continue
        path = tmp_path / f"wide{j}.o"
        path.write_bytes(obj)
        text = subprocess.run([f"{isa.LLVM}/llvm-objdump", "-d", "--mcpu=gfx950", str(path)], capture_output=True,
                              text=True, check=True).stdout
        for line in text.splitlines():
            m = isa._KERNEL.match(line)
            if m:
                name = m.group(1)
                listings[name] = []
            elif name is not None:
                listings[name].append(line)
    kernels = [k for k in listings if "w256_dq_kernel" in k or "w256_dkv_kernel" in k]
    assert len(kernels) == 6, sorted(listings)  # bf16 sparse and dense, fp16 sparse
    for k in kernels:
        assert any(isa._ACC_DST.search(line) for line in listings[k]), f"{k}: no AGPR-accumulator MFMA found"
        for check in (isa.check_accumulators_drained, isa.check_operand_distance):
            bad = check(listings[k])
            assert not bad, f"{k}: " + "; ".join(f"line {n}: {t[:100]}" for n, t in bad[:5])
