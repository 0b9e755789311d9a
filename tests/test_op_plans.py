"""laya_op_plan: the tile and split count that laya_op_linear's and laya_op_qkv's planned launches (tile -1)
take, known before the call (no GPU but for the test that a planned fp32 product writes exactly that many partials)."""
import ctypes as ct
import gzip
import json
from pathlib import Path

import pytest

from laya_cuda import _lib


def plan(kind, M, N, K, biased=False, tile=-1, dtype=None):
    t, s = ct.c_int32(-9), ct.c_int32(-9)
    _lib.check(_lib.load().laya_op_plan(kind, _lib.F16 if dtype is None else dtype, M, N, K, int(biased), tile, ct.byref(t),
                                        ct.byref(s)))
    return t.value, s.value


def test_only_fp32_products_without_bias_split():
    split = 0
    for M in (1, 16, 96, 512, 640, 2048, 15088):
        for N, K in [(768, 768), (1024, 4096), (2304, 768), (192, 192)]:
            for kind in range(7):
                tile, splits = plan(kind, M, N, K)
                assert tile >= 0 and 1 <= splits <= 8
                assert kind == 0 or splits == 1
                split += splits > 1
            assert plan(0, M, N, K, biased=True)[1] == 1
    assert split > 5


def test_bad_plan_requests_are_refused():
    lib, t = _lib.load(), ct.c_int32()
    for args in [(7, _lib.F16, 16, 64, 64, 0, -1), (-1, _lib.F16, 16, 64, 64, 0, -1), (1, _lib.F16, 0, 64, 64, 0, -1),
                 (1, _lib.F16, 16, 64, 64, 0, 3), (1, _lib.F16, 16, 64, 64, 0, -4)]:
        assert lib.laya_op_plan(*args, ct.byref(t), ct.byref(t)) == _lib.EINVAL
    assert lib.laya_op_plan(1, _lib.F16, 16, 64, 64, 0, -1, None, None) == _lib.EINVAL


DATA = Path(__file__).resolve().parents[1] / "laya-cuda_amd" / "csrc" / "gemm_cost_data.json.gz"


@pytest.mark.parametrize("where,tile,mean,most", [("forward", -3, 1.01, 1.11), ("held_out", -1, 1.005, 1.12),
                                                  ("isolated", -1, 1.006, 1.13)])
def test_planned_tiles_are_near_the_best_measured(where, tile, mean, most):
    """The planner's choice for 16-bit products of more than 512 rows against the times that its constants come
    from: inside forwards for a forward's plans, isolated launches for an op-level call's.  The bounds are what
    the constants reach."""
    kinds = {"half": 1, "gelu": 2, "relu": 3, "geglu": 4, "qkv": 5, "rope": 6}
    ratios = []
    for kind, M, N, K, timed in json.loads(gzip.decompress(DATA.read_bytes()))[where]:
        if M > 512 and kind in kinds:
            us = {t: u for t, _, u, _ in timed}
            ratios.append(us[plan(kinds[kind], M, N, K, tile=tile)[0]] / min(us.values()))
    print(where, len(ratios), sum(ratios) / len(ratios), max(ratios))
    assert len(ratios) > 100
    assert sum(ratios) / len(ratios) <= mean and max(ratios) <= most


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(16, 768, 3072), (96, 768, 768), (512, 1024, 4096), (1664, 768, 768), (100, 192, 192)])
def test_planned_fp32_product_writes_the_plans_partials(gpu, M, N, K):
    import torch as t
    splits = plan(0, M, N, K)[1]
    g = t.Generator(device=gpu).manual_seed(M)
    x = t.randn((M, K), generator=g, device=gpu).half()
    w = (t.randn((N, K), generator=g, device=gpu) / K ** 0.5).half()
    out = t.full((splits + 1, M, N), float("nan"), device=gpu)
    _lib.check(_lib.load().laya_op_linear(*(ct.c_void_p(v.data_ptr()) for v in (x, w)), None, ct.c_void_p(out.data_ptr()), 0,
                                          _lib.F16, M, N, K, 1, -1, ct.c_void_p(t.cuda.current_stream().cuda_stream)))
    want = x.double() @ w.double().t()
    assert out[splits].isnan().all()  # not one partial more
    assert (out[:splits].double().sum(0) - want).abs().max().item() <= 1e-6 * K ** 0.5 * max(1.0, want.abs().max().item())
