"""Sparse MLA + W_UV + W_o on the GPU (8 rows x 2048 selected of 32768).

Bar: the merged latent output, and the attention term out - h (or out itself when
there is no residual), within rel-L2 1e-2 of the CPU oracle (f64 softmax over the same
gathered, dequantized FP8 rows; the term against the oracle's o W_o^T in f64); the
kernel rounds P' and the stage hand-offs to bf16 where the oracle states the same
points.  The residual rows are drawn ~ N(0, (1/128)^2) so that the bf16 rounding of h +
o W_o^T stays well below the term (refs.bf16_rounding_floor).
"""

import pytest
import torch

from oracle import reference as R
from refs import bf16_rounding_floor, cpu, mla_oracle

pytestmark = pytest.mark.gpu

REL_L2 = 1e-2


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _run(cfg, rows, seed, residual=True, holes=False, unscaled=False):
    from sgl_amd_mono.k2 import synth
    from sgl_amd_mono.k2.ops import SparseMlaOp

    dev = _dev()
    ns = synth.make_mla(cfg, rows, seed, dev, residual=residual, h_std=1.0 / 128)
    if holes:  # unused slots (-1) inside and at the end of the list
        ns.sel[:, 5:70] = -1
        ns.sel[0, -64:] = -1
    if unscaled:  # SGLang's MLA cache: E4M3 rows without per-token scales
        ns.kv_scale = None
    op = SparseMlaOp(cfg, ns, rows, ns.page_table.shape[1], device=dev)
    olat = torch.empty(rows, cfg.heads, cfg.kv_lora, dtype=torch.float32, device=dev)
    out = op(ns.q, ns.kv, ns.kv_scale, ns.page_table, ns.req_ids, ns.sel, h=ns.h, o_latent=olat)
    torch.cuda.synchronize()
    ref_lat, ref_out, ref_y = mla_oracle(ns, parts=True)
    e_lat = R.rel_l2(cpu(olat), ref_lat)
    if ns.h is None:
        e_out = R.rel_l2(cpu(out).float(), ref_out)
    else:
        assert bf16_rounding_floor(cpu(out), ref_y) <= 3e-3
        e_out = R.rel_l2(cpu(out).double() - cpu(ns.h).double(), ref_y)
    return e_lat, e_out


@pytest.mark.parametrize("rows", [1, 8])
def test_mla_config3(rows):
    from sgl_amd_mono.k2 import config as C

    e_lat, e_out = _run(C.C3_MLA, rows, seed=300 + rows)
    assert e_lat <= REL_L2 and e_out <= REL_L2, (e_lat, e_out)


def test_mla_unused_slots_and_no_residual():
    from sgl_amd_mono.k2 import config as C

    cfg = C.MlaConfig(context=8192, topk=512)
    e_lat, e_out = _run(cfg, 3, seed=310, residual=False, holes=True)
    assert e_lat <= REL_L2 and e_out <= REL_L2, (e_lat, e_out)


def test_mla_32_rows():
    from sgl_amd_mono.k2 import config as C

    cfg = C.MlaConfig(context=4096, topk=2048)
    e_lat, e_out = _run(cfg, 32, seed=320)
    assert e_lat <= REL_L2 and e_out <= REL_L2, (e_lat, e_out)


@pytest.mark.parametrize("rows, topk", [(17, 64), (17, 512), (18, 2048), (27, 1984), (31, 4096)])
def test_mla_above_16_rows_matches_narrow_calls(rows, topk):
    """Above 16 rows the splits run two at a time, an equal run of them on each half
    workgroup (none or one on most at the first shapes; runs that cross rows at the last
    ones): the bits of the same rows in calls of at most 16, which run them one by one.
    Some rows have unused slots, one row none in use."""
    from sgl_amd_mono.k2 import config as C
    from sgl_amd_mono.k2 import synth
    from sgl_amd_mono.k2.ops import SparseMlaOp

    dev = _dev()
    cfg = C.MlaConfig(context=4096, topk=topk, hidden=1024)
    ns = synth.make_mla(cfg, rows, rows + topk, dev)
    ns.sel[1::3, topk // 3:] = -1
    ns.sel[2, :] = -1
    op = SparseMlaOp(cfg, ns, rows, ns.page_table.shape[1], device=dev)
    args = (ns.kv, ns.kv_scale, ns.page_table)
    for _ in range(2):  # the second launch on the workspace the first left
        out = cpu(op(ns.q, *args, ns.req_ids, ns.sel, h=ns.h))
        for a in range(0, rows, 9):
            b = min(rows, a + 9)
            part = SparseMlaOp(cfg, ns, b - a, ns.page_table.shape[1], device=dev)(
                ns.q[a:b].contiguous(), *args, ns.req_ids[a:b].contiguous(), ns.sel[a:b].contiguous(), h=ns.h[a:b].contiguous())
            assert torch.equal(cpu(part), out[a:b]), (a, b)
    assert op.status() == 0


def test_mla_unscaled_cache():
    """kv_scale None (SGLang's [slots][576] e4m3 cache) reads every row at scale 1:
    the oracle over unit scales, and bit-identical to passing a tensor of ones."""
    from sgl_amd_mono.k2 import config as C
    from sgl_amd_mono.k2 import synth
    from sgl_amd_mono.k2.ops import SparseMlaOp

    cfg = C.MlaConfig(context=8192, topk=1024)
    e_lat, e_out = _run(cfg, 4, seed=330, unscaled=True)
    assert e_lat <= REL_L2 and e_out <= REL_L2, (e_lat, e_out)
    dev = _dev()
    ns = synth.make_mla(cfg, 4, 331, dev)
    op = SparseMlaOp(cfg, ns, 4, ns.page_table.shape[1], device=dev)
    ones = torch.ones_like(ns.kv_scale)
    a = op(ns.q, ns.kv, None, ns.page_table, ns.req_ids, ns.sel, h=ns.h).clone()
    b = op(ns.q, ns.kv, ones, ns.page_table, ns.req_ids, ns.sel, h=ns.h)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
