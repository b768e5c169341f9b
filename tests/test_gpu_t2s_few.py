"""A T2S decode step of few sequences: QKV projection and attention of a layer as one launch
(csrc/gsvk_t2s_attn.hip), against the oracle chain with the slack of test_gpu_t2s_decode.py, at the
edges of its key rounds (128 keys, four rounds in flight) and of the widths it takes."""
import numpy as np
import pytest
import torch

import gsvk
from gpu_util import F16, F32, host
from test_gpu_t2s_decode import build, compare, oracle_step, to_device

pytestmark = pytest.mark.gpu


def run(D, kv_pos, max_len, graph=True, params=True, seed=0, poison=True):
    B = len(kv_pos)
    m, io = build(B=B, D=D, H=D // 32, FF=256, L=2, V=50, max_len=max_len, seed=50 + seed)
    io["kv_pos"] = np.array(kv_pos, dtype=np.int64)
    if not params:
        for ly in m["layers"]:
            ly["n2g"], ly["n2b"], ly["bqkv"] = np.ones(D, "f4"), np.zeros(D, "f4"), np.zeros(3 * D, "f4")
    md, iod = to_device(m, io, 256)
    if not params:
        for ly in md["layers"]:
            ly["n2g"] = ly["n2b"] = ly["bqkv"] = None
    if poison:  # rows at and past the new token may hold anything
        for ly in md["layers"]:
            for c in ("k_cache", "v_cache"):
                for b, p in enumerate(kv_pos):
                    ly[c][b, max(p, 0):] = float("nan")
    x_want, lg_want = oracle_step(m, io)
    step = gsvk.T2SDecode(md, iod, len_bound=max_len, graph=graph)
    step.run()
    torch.cuda.synchronize()
    assert int(iod["err"].item()) == 0
    compare(host(iod["x"], F16), host(iod["logits"], F32), x_want, lg_want, f"D={D} {kv_pos}")
    for ly_d, ly_h in zip(md["layers"], m["layers"]):  # the appended rows; the others untouched
        for c in ("k_cache", "v_cache"):
            for b, p in enumerate(kv_pos):
                got = ly_d[c][b, p].float().cpu().numpy()
                want = ly_h[c].view(np.float16)[b, p].astype(np.float32)
                assert np.all(np.abs(got - want) <= 4 * np.spacing(np.abs(want).astype(np.float16)
                                                                   ).astype("f4") + 4e-3)
                assert torch.isnan(ly_d[c][b, p + 1:].float()).all()


@pytest.mark.parametrize("D", [128, 256, 384, 512])
@pytest.mark.parametrize("params", [True, False])
def test_widths(D, params):
    run(D, [0, 1, 63, 40], 64, params=params, seed=D)


@pytest.mark.parametrize("kv_pos", [[127, 128, 129], [511, 512, 513], [640], [1023, 0, 700, 256]])
def test_key_rounds(kv_pos):
    run(512, kv_pos, 1024, seed=kv_pos[0])


def test_either_side_of_the_line():
    """31 sequences at 580 keys run fused, at 600 the separate launches."""
    rng = np.random.default_rng(5)
    for max_len in (580, 600):
        run(128, rng.integers(0, max_len, 31).tolist(), max_len, seed=max_len)


def test_graph_equals_eager_and_bad_slots():
    """A cache slot out of range leaves the caches as they are, sets err and gives a NaN row; the other
    sequences are not touched by it."""
    outs = []
    for graph in (False, True):
        m, io = build(B=3, D=512, H=16, FF=256, L=1, V=50, max_len=96, seed=77)
        io["kv_pos"] = np.array([50, 96, -1], dtype=np.int64)
        md, iod = to_device(m, io, 256)
        before = md["layers"][0]["k_cache"].clone()
        step = gsvk.T2SDecode(md, iod, len_bound=96, graph=graph)
        step.run()
        torch.cuda.synchronize()
        assert int(iod["err"].item()) == 1
        lg = iod["logits"]
        assert torch.isfinite(lg[0]).all() and torch.isnan(lg[1:]).all()
        after = md["layers"][0]["k_cache"]
        assert torch.equal(after[1:], before[1:])
        outs.append(host(iod["logits"], F32)[0])
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
