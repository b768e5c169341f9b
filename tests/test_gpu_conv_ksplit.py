"""The convolutions of few tiles (csrc/gsvk_conv.hip conv1d_ksplit: the waves of a workgroup split the
(chunk, tap) units) at the edges of their tiles, batches and units, and the larger kernel just past
the line between the two (64 x 32 tiles: 800, or 600 with the exact split), against the oracle with
the tolerance of test_gpu_conv.py. Also the stage entry point: the three ResBlocks' convolutions in
one launch give the bits of the same convolutions launched one by one."""
import numpy as np
import pytest
import torch

import gsvk
import oracle as O
from gpu_util import F16, F32, dev, devf, host
from sovits_util import gpu_stage, make_stage
from test_gpu_conv import assert_conv_close, check_case, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,rx", [(F32, False), (F32, True), (F16, False)])
@pytest.mark.parametrize("cin,cout,T,k,dil,epi", [
    (24, 24, 1, 3, 1, 0),        # one column, one chunk, fewer units than waves
    (8, 25, 63, 11, 5, 1),       # a quarter chunk; the widest ResBlock halo; a row past one fragment
    (40, 48, 64, 7, 3, 2),       # a chunk and a quarter; exactly one tile of columns
    (384, 384, 65, 11, 5, 3),    # two batches of chunks, one column into the second tile
    (200, 96, 129, 33, 2, 0),    # halo 64, the largest; ragged batch
    (96, 96, 300, 3, 1, 3),
    (768, 32, 70, 1, 1, 0),      # no halo, 24 chunks of one tap
])
def test_few_tiles(dt, rx, cin, cout, T, k, dil, epi):
    check_case(dt, cin, cout, T, k, dil, epi=epi, round_x=rx, seed=900 + T, use_bias=T != 129)


def test_rows_apart_and_offset():
    check_case(F16, 48, 48, 77, 7, 5, epi=1, seed=950, ld_pad=3, y_offset=2)
    check_case(F32, 96, 96, 78, 7, 5, epi=3, seed=951, ld_pad=1)


@pytest.mark.parametrize("dt,rx,C,T", [
    (F16, False, 24, 51137), (F16, False, 24, 51201), (F32, True, 96, 17100), (F32, True, 192, 8500),
    (F32, False, 48, 19200), (F32, False, 96, 12801), (F32, False, 192, 6400),
])
def test_either_side_of_the_line(dt, rx, C, T):
    check_case(dt, C, C, T, 3, 5, epi=1, round_x=rx, seed=960 + C)


@pytest.mark.parametrize("dt", [F32, F16])
@pytest.mark.parametrize("cin,cout,T,k,u", [
    (48, 24, 33, 2, 2), (64, 48, 40, 16, 8), (768, 96, 5, 20, 10), (24, 40, 64, 9, 4),
    (96, 32, 1, 8, 2),
])
def test_upsampler_phases(dt, cin, cout, T, k, u):
    r = rng(980 + T)
    x = O.to_storage(dt, r.standard_normal((cin, T)).astype(np.float32))
    w = (r.standard_normal((cin, cout, k)) / np.sqrt(cin * k / u)).astype(np.float16)
    b = (0.05 * r.standard_normal(cout)).astype(np.float32)
    want = O.convt1d(dt, x, w.view(np.uint16), u, b)
    ref = O.convt1d(dt, x, w.view(np.uint16), u, None)
    up = gsvk.ConvT1d(dev(w.view(np.uint16), F16), devf(b), u)
    y = up.forward(dev(x, dt))
    torch.cuda.synchronize()
    assert_conv_close(dt, host(y, dt), want, ref, f"{cin}->{cout} T={T} k={k} u={u}")


@pytest.mark.parametrize("dt,rx", [(F32, False), (F32, True), (F16, False)])
@pytest.mark.parametrize("cin,C,T,k_up,u", [(64, 32, 9, 16, 8), (48, 24, 150, 2, 2),
                                             (20, 20, 30, 4, 2), (16, 24, 25703, 2, 2),
                                             (16, 48, 13001, 2, 2), (8, 96, 8700, 2, 2),
                                             (8, 8, 52000, 1, 1), (8, 40, 26011, 1, 1)])
def test_stage_equals_its_convolutions(dt, rx, cin, C, T, k_up, u):
    """gsvk.GeneratorStage (one call: grouped launches, or pairs of convolutions in one) against the
    same passes one by one. (20 channels: not for the few-tiles kernel.) The sizes are such that both
    forms add in the same order: few tiles (a group and a single convolution take the same tiling), or
    more than the few-tiles line (a pair adds as the large kernel does), so the bits agree."""
    r = rng(990 + C)
    up, rbs = make_stage(r, cin, C, k_up, u)
    st = gpu_stage(up, rbs, u)
    x = torch.from_numpy(r.standard_normal((cin, T + 2)).astype(np.float32)).cuda()
    x = x.half()[:, :T] if dt == F16 else x[:, :T]
    out = torch.empty(C, T * u, dtype=x.dtype, device="cuda")
    st.forward(x, out, slope_next=0.1, round_x=rx)
    y = st.ups.forward(x, round_x=rx)
    curs = []
    for rb in st.resblocks:
        cur, src, res = torch.empty_like(y), y, y
        for c1, c2 in zip(rb.convs1, rb.convs2):
            ta = c1.forward(src, epi=gsvk.CONV_EPI_LRELU | gsvk.CONV_X_LRELU, round_x=rx)
            c2.forward(ta, epi=gsvk.CONV_EPI_RES, cur=cur, res=res, round_x=rx)
            src, res = cur, None
        curs.append(cur)
    want = torch.empty_like(out)
    gsvk.resblock_branch_mean(curs, None, want, True, 0.1)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
