"""gsvk_gemv_f16w / _ln with one to four rows (csrc/gsvk_gemv.hip gemv_rows) at the edges of its
range: part-filled last 512-k blocks, odd column counts, both column counts per wave, strided rows,
absent operands, and that one and four rows of the same input agree with the oracle."""
import numpy as np
import pytest
import torch

import gsvk
import oracle as O
from gpu_util import BF16, F16, F32, dev, devf, host
from test_gpu_gemv import assert_gemv_close, rng, run_case, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("n_out,n_in", [(1, 256), (7, 264), (512, 512), (1025, 520), (1023, 1024),
                                        (1024, 1032), (512, 2048), (2049, 2040)])
def test_few_rows(rows, n_out, n_in):
    for i, (x_dt, rx, y_dt) in enumerate([(F16, True, F16), (F32, True, F32), (F32, False, BF16)]):
        run_case(rows, n_out, n_in, x_dt, rx, y_dt, act=(gsvk.ACT_RELU, gsvk.ACT_NONE,
                                                         gsvk.ACT_GELU_ERF)[i],
                 use_bias=i != 1, use_res=i != 2, seed=700 + i)


@pytest.mark.parametrize("rows", [1, 3, 4])
@pytest.mark.parametrize("n_out,n_in", [(1537, 512), (96, 456), (40, 968), (2048, 1024)])
@pytest.mark.parametrize("x_dt,rx", [(F16, True), (F32, True), (F32, False)])
def test_layernorm_then_product(rows, n_out, n_in, x_dt, rx):
    """h against the oracle's LayerNorm, y with the bits of gsvk_gemv_f16w on that h. Rows apart."""
    r = rng(800 + n_in)
    z = O.to_storage(x_dt, r.standard_normal((rows, n_in)).astype(np.float32))
    w = weights(r, n_out, n_in)
    g = (1 + 0.1 * r.standard_normal(n_in)).astype(np.float32) if rows != 3 else None
    b = (0.1 * r.standard_normal(n_in)).astype(np.float32) if rows != 3 else None
    bias = (0.02 * r.standard_normal(n_out)).astype(np.float32)
    zd = torch.zeros(rows, n_in + 8, dtype=dev(z, x_dt).dtype, device="cuda")
    zd[:, :n_in] = dev(z, x_dt)
    zd = zd[:, :n_in]
    hd, wd = torch.empty_like(zd), dev(w, F16)
    hd = torch.zeros(rows, n_in + 8, dtype=zd.dtype, device="cuda")[:, :n_in]
    y = torch.empty(rows, n_out, dtype=torch.float32, device="cuda")
    gd, bd = (devf(g), devf(b)) if g is not None else (None, None)
    gsvk.gemv_f16w_ln(zd, gd, bd, 1e-5, hd, wd, y, bias=devf(bias), round_x=rx)
    y2 = torch.empty_like(y)
    gsvk.gemv_f16w(hd, wd, y2, bias=devf(bias), round_x=rx)
    torch.cuda.synchronize()
    want = O.add_layernorm(x_dt, z, g, b, 1e-5)
    got = O.to_f32(x_dt, host(hd, x_dt)).astype(np.float64)
    w64 = O.to_f32(x_dt, want).astype(np.float64)
    tol = 1e-6 + 1e-5 * np.abs(w64) + (np.spacing(np.abs(w64).astype(np.float16)).astype(float)
                                       if x_dt == F16 else 0)
    assert np.all(np.abs(got - w64) <= tol)
    assert torch.equal(y.view(torch.int32), y2.view(torch.int32))


def test_nonfinite_inputs_stay_in_their_row():
    r = rng(880)
    x = r.standard_normal((3, 520)).astype(np.float32)
    x[1, 519], x[2, 3] = np.inf, np.nan
    w = weights(r, 40, 520)
    y = torch.empty(3, 40, device="cuda")
    gsvk.gemv_f16w(devf(x), dev(w, F16), y)
    torch.cuda.synchronize()
    want = O.gemv_f16w(F32, x, w, F32)
    got = host(y, F32)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isfinite(got[0]).all()
    assert np.array_equal(got[1][np.isinf(want[1])], want[1][np.isinf(want[1])])
    assert_gemv_close(F32, got[:1], want[:1])
