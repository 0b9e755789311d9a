"""The few-row GEMM (csrc/gemm_burst.hip) and the 16x16x32 ring (csrc/gemm.hip, tile 35): every tile and epilogue at the edges of its tiles, stages
and K splits, and the planner's choice around its row bound, against 64-bit products of the same
16-bit operands.

Tolerances: fp32 partials 1e-6 sqrt(K) (products of unit-variance rows with 1/sqrt(K) weights are O(1),
K fp32 additions); 16-bit outputs one rounding (half a unit: 2^-11 / 2^-8 of the value) plus that.
"""
import ctypes as ct
import math

import pytest

from laya_cuda import _lib

pytestmark = pytest.mark.gpu

TILES = range(27, 35)
HALF_HEAD_TILES = [t for t in TILES if t != 33]  # 96 columns span heads: no head-major epilogue
# Rows: one, tile remainders, a partial last tile; K: one slab, a partial stage, past the stages.
SHAPES = [(1, 192, 64), (17, 384, 192), (96, 768, 768), (130, 192, 1152), (200, 768, 3072)]
ROUNDING = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}


def torch():
    import torch as t
    return t


def p(tensor):
    return ct.c_void_p(tensor.data_ptr()) if tensor is not None else None


def stream():
    return ct.c_void_p(torch().cuda.current_stream().cuda_stream)


def half(kind):
    return torch().float16 if kind == "f16" else torch().bfloat16


def code(kind):
    return _lib.F16 if kind == "f16" else _lib.BF16


def operands(gpu, kind, M, N, K):
    t = torch()
    g = t.Generator(device=gpu).manual_seed(M + N + K)
    x = t.randn((M, K), generator=g, device=gpu).to(half(kind))
    w = (t.randn((N, K), generator=g, device=gpu) / math.sqrt(K)).to(half(kind))
    return x, w, t.randn(N, generator=g, device=gpu), x.double() @ w.double().t()


def close(got, want, kind, K):
    bound = ROUNDING[kind] * want.abs() + 4e-6 * math.sqrt(K) + (2.0 ** -24 if kind == "f16" else 0)
    assert ((got.double() - want).abs() <= 1.01 * bound).all()


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("tile", TILES)
def test_row_major_epilogues(gpu, tile, kind):
    t = torch()
    lib = _lib.load()
    for M, N, K in SHAPES:
        x, w, bias, ref = operands(gpu, kind, M, N, K)
        for splits in (1, 3, 8):
            out = t.full((splits, M, N), float("nan"), device=gpu)
            _lib.check(lib.laya_op_linear(p(x), p(w), None, p(out), 0, code(kind), M, N, K, splits, tile, stream()))
            assert (out.double().sum(0) - ref).abs().max().item() <= 1e-6 * math.sqrt(K) * max(1.0, ref.abs().max().item())
        biased = ref + bias.double()
        groups = ref.view(M, N // 32, 2, 16)
        for epilogue, b, want in ((1, bias, biased), (2, bias, t.nn.functional.gelu(biased)), (3, bias, t.relu(biased)),
                                  (4, None, (t.nn.functional.gelu(groups[:, :, 0]) * groups[:, :, 1]).reshape(M, -1))):
            out = t.full(want.shape, float("nan"), dtype=half(kind), device=gpu)
            _lib.check(lib.laya_op_linear(p(x), p(w), p(b), p(out), epilogue, code(kind), M, N, K, 1, tile, stream()))
            close(out, want, kind, K)


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("tile", HALF_HEAD_TILES + [-1])
def test_head_major_epilogue(gpu, tile, rope):
    """Q and K rotated in pairs 32 dims apart (two 16-dim halves of a tile), V transposed; -1: the
    planner's tile, on both sides of its row bound."""
    t = torch()
    lib = _lib.load()
    for M, width in [(8, 64), (104, 192), (512, 320), (520, 768)]:
        heads = width // 64
        x, w, bias, ref = operands(gpu, "bf16", M, 3 * width, width)
        g = t.Generator(device=gpu).manual_seed(3)
        angle = t.rand((700, 32), generator=g, device=gpu) * 6
        cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
        pos = t.randint(0, 700, (M,), generator=g, device=gpu, dtype=t.int32)
        q, k, vt = (t.full((M * width,), float("nan"), dtype=t.bfloat16, device=gpu) for _ in range(3))
        _lib.check(lib.laya_op_qkv(p(x), p(w), None if rope else p(bias), p(q), p(k), p(vt), p(cos) if rope else None,
                                   p(sin) if rope else None, p(pos) if rope else None, _lib.BF16, M, width, tile,
                                   stream()))
        y = ref if rope else ref + bias.double()
        wq, wk, wv = (y[:, i * width:(i + 1) * width].reshape(M, heads, 64).transpose(0, 1) for i in range(3))
        if rope:
            c, s = cos[pos.long()].double(), sin[pos.long()].double()

            def rotate(v):
                return t.cat([v[..., :32] * c - v[..., 32:] * s, v[..., 32:] * c + v[..., :32] * s], -1)
            wq, wk = rotate(wq), rotate(wk)
        close(q.view(heads, M, 64), wq, "bf16", width)
        close(k.view(heads, M, 64), wk, "bf16", width)
        close(vt.view(heads, 64, M), wv.transpose(1, 2), "bf16", width)


def test_columns_across_heads_are_refused(gpu):
    t = torch()
    x = t.zeros((16, 192), dtype=t.float16, device=gpu)
    w = t.zeros((576, 192), dtype=t.float16, device=gpu)
    q, k, vt = (t.zeros(16 * 192, dtype=t.float16, device=gpu) for _ in range(3))
    assert _lib.load().laya_op_qkv(p(x), p(w), None, p(q), p(k), p(vt), None, None, None, _lib.F16, 16, 192, 33,
                                   stream()) != 0


@pytest.mark.parametrize("M", [1, 33, 96, 192, 257, 512, 513])
def test_planned_tiles_around_the_row_bound(gpu, M):
    t = torch()
    lib = _lib.load()
    for N, K in [(768, 768), (3072, 768), (1024, 4096), (64, 512), (64, 64)]:
        x, w, bias, ref = operands(gpu, "f16", M, N, K)
        out = t.full((M, N), float("nan"), dtype=t.float16, device=gpu)
        _lib.check(lib.laya_op_linear(p(x), p(w), p(bias), p(out), 1, _lib.F16, M, N, K, 1, -1, stream()))
        close(out, ref + bias.double(), "f16", K)
    # N that no 64-wide tile divides stays refused, whatever the few-row tiles' width.
    assert lib.laya_op_linear(p(x), p(w), None, p(out), 1, _lib.F16, M, 32, 64, 1, -1, stream()) != 0


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(1, 256, 192), (300, 768, 576), (16421, 2048, 192), (30000, 768, 320)])
def test_ring_of_sixteen_wide_mfmas(gpu, kind, M, N, K):
    """Tile 35, the persistent 256x256 ring with 16x16x32 MFMAs: one tile, partial row tiles, the
    three-slab minimum, and several tiles per workgroup (520 and 354 on 256 CUs), every 16-bit
    row-major epilogue."""
    t = torch()
    lib = _lib.load()
    x, w, bias, _ = operands(gpu, kind, M, N, K)
    ref = t.mm(x.float(), w.float().t()).double()  # fp32 product of 64-bit-exact terms: within 1e-6 sqrt(K)
    groups = ref.view(M, N // 32, 2, 16)
    for epilogue, b, want in ((1, bias, ref + bias), (2, bias, t.nn.functional.gelu(ref + bias)),
                              (3, bias, t.relu(ref + bias)),
                              (4, None, (t.nn.functional.gelu(groups[:, :, 0]) * groups[:, :, 1]).reshape(M, -1))):
        out = t.full(want.shape, float("nan"), dtype=half(kind), device=gpu)
        _lib.check(lib.laya_op_linear(p(x), p(w), p(b), p(out), epilogue, code(kind), M, N, K, 1, 35, stream()))
        close(out, want, kind, K)
    out32 = t.zeros((M, N), device=gpu)
    assert lib.laya_op_linear(p(x), p(w), None, p(out32), 0, code(kind), M, N, K, 1, 35, stream()) != 0  # 16-bit only
    assert lib.laya_op_linear(p(x), p(w), None, p(out), 1, code(kind), M, N, 128, 1, 35, stream()) != 0  # two slabs


@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("M,width", [(8, 256), (1000, 768), (16424, 1024)])
def test_ring_of_sixteen_wide_mfmas_head_major(gpu, M, width, rope):
    t = torch()
    lib = _lib.load()
    heads = width // 64
    x, w, bias, _ = operands(gpu, "f16", M, 3 * width, width)
    ref = t.mm(x.float(), w.float().t()).double()
    g = t.Generator(device=gpu).manual_seed(3)
    angle = t.rand((700, 32), generator=g, device=gpu) * 6
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
    pos = t.randint(0, 700, (M,), generator=g, device=gpu, dtype=t.int32)
    q, k, vt = (t.full((M * width,), float("nan"), dtype=t.float16, device=gpu) for _ in range(3))
    _lib.check(lib.laya_op_qkv(p(x), p(w), p(bias), p(q), p(k), p(vt), p(cos) if rope else None,
                               p(sin) if rope else None, p(pos) if rope else None, _lib.F16, M, width, 35, stream()))
    wq, wk, wv = ((ref + bias)[:, i * width:(i + 1) * width].reshape(M, heads, 64).transpose(0, 1) for i in range(3))
    if rope:
        c, s = cos[pos.long()].double(), sin[pos.long()].double()

        def rotate(v):
            return t.cat([v[..., :32] * c - v[..., 32:] * s, v[..., 32:] * c + v[..., :32] * s], -1)
        wq, wk = rotate(wq), rotate(wk)
    close(q.view(heads, M, 64), wq, "f16", width)
    close(k.view(heads, M, 64), wk, "f16", width)
    close(vt.view(heads, 64, M), wv.transpose(1, 2), "f16", width)
