"""Eight-wave shared attention tiles: the one-block-ahead kernel of global layers (its reference max stays
the first block's until a block's probabilities grow past 2^8), the shared-key kernel that serves short
sequences, and the per-wave block skipping of local layers, against float64.

Tolerance: the 16-bit rounding of probabilities and output, half a unit each (2^-11 / 2^-8), on rows whose
weights sum to one over |v| <= 5: 2 x 2^-11 x |v| plus the exponential's fp32 error."""
import ctypes as ct

import numpy as np
import pytest

from laya_cuda import _lib

pytestmark = pytest.mark.gpu


def attend(gpu, lengths, growth, window, dtype, ahead=False):
    import torch as t
    lib = _lib.load()
    heads, half = 2, t.float16 if dtype == "f16" else t.bfloat16
    starts = np.cumsum([0] + [-(-n // 16) * 16 for n in lengths]).astype(np.int32)
    m = int(starts[-1]) + 16
    g = t.Generator(device=gpu).manual_seed(m)
    q, k = (t.randn((heads, m, 64), generator=g, device=gpu) for _ in range(2))
    vt = t.randn((heads, 64, m), generator=g, device=gpu).to(half)
    for a, n in zip(starts, lengths):  # later keys score higher (growth > 1) or lower
        k[:, a:a + n] *= growth ** (t.arange(n, device=gpu) / 64).floor().clamp(max=15)[None, :, None]
    q, k = q.to(half), k.to(half)
    block, most = lib.laya_attention_block(0, 8), m // 16
    tiles = np.zeros((most, 4), np.int32)
    ip = ct.POINTER(ct.c_int32)
    lens = np.asarray(lengths, np.int32)
    most = lib.laya_attention_tiles(starts.ctypes.data_as(ip), lens.ctypes.data_as(ip), len(lengths), m, block,
                                    tiles.ctypes.data_as(ip), most)
    assert most > 0 and (window >= 0 or (m >= 168 * most) == ahead)
    work = t.from_numpy(tiles[:most].copy()).to(gpu)
    out = t.full((m, heads * 64), float("nan"), dtype=half, device=gpu)
    _lib.check(lib.laya_op_attention(*(ct.c_void_p(x.data_ptr()) for x in (q, k, vt, out, work)), m, heads, most, 0, 8,
                                     window, _lib.F16 if dtype == "f16" else _lib.BF16,
                                     ct.c_void_p(t.cuda.current_stream().cuda_stream)))
    unit = 2.0 ** -11 if dtype == "f16" else 2.0 ** -8
    real = t.zeros(m, dtype=t.bool, device=gpu)
    for a, n in zip(starts.tolist(), lengths):
        real[a:a + n] = True
        s = t.matmul(q[:, a:a + n].double(), k[:, a:a + n].double().transpose(1, 2).contiguous()) / 8
        if window >= 0:
            at = t.arange(n, device=gpu)
            s = s.masked_fill((at[:, None] - at[None, :]).abs() > window, float("-inf"))
        v = vt[:, :, a:a + n].double().transpose(1, 2).contiguous()
        weights = t.softmax(s, -1)
        want = t.matmul(weights, v).transpose(0, 1).reshape(n, -1)
        bound = (t.matmul(weights, v.abs()).transpose(0, 1).reshape(n, -1) * 2 + 0.05) * unit
        assert ((out[a:a + n].double() - want).abs() <= bound).all(), (a, n)
    assert (out[~real] == 0).all()


# One key, tile edges of 64-key blocks and 128-query halves, a lone second half, several tiles; each among
# longer sequences, whose tiles take the list past the rows per tile from which the ahead kernel serves it.
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("growth", [1.0, 1.6, 0.5])
@pytest.mark.parametrize("lengths", [[1, 1024], [63, 64, 65, 2048], [127, 128, 129, 2, 3072], [257, 1024], [640, 130, 1024]])
def test_reference_max_follows_growing_scores(gpu, lengths, growth, dtype):
    attend(gpu, lengths, growth, -1, dtype, ahead=True)


# Short sequences keep the shared-key kernel.
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("lengths", [[1], [63, 64, 65], [127, 128, 129, 2], [257]])
def test_short_global_sequences(gpu, lengths, dtype):
    attend(gpu, lengths, 1.6, -1, dtype)


@pytest.mark.parametrize("window", [0, 1, 31, 64, 200])
@pytest.mark.parametrize("lengths", [[1, 63, 65], [160, 161, 300], [1024]])
def test_local_blocks_skipped_per_wave(gpu, lengths, window):
    attend(gpu, lengths, 1.0, window, "f16")


def test_keys_past_the_slot_bring_no_other_values(gpu):
    """The last block of the last sequence reaches past the slot: what stands in for its V^T keys there
    stays with the head dim's last keys, so another sequence's infinite values, times probabilities of
    zero, make no NaN of it."""
    import torch as t
    lib = _lib.load()
    lengths, m, heads = [64, 1030], 1104, 2
    starts, lens = np.array([0, 64], np.int32), np.array(lengths, np.int32)
    g = t.Generator(device=gpu).manual_seed(4)
    q, k = (t.randn((heads, m, 64), generator=g, device=gpu).half() for _ in range(2))
    vt = t.randn((heads, 64, m), generator=g, device=gpu).half()
    tiles = np.zeros((10, 4), np.int32)
    ip = ct.POINTER(ct.c_int32)
    used = lib.laya_attention_tiles(starts.ctypes.data_as(ip), lens.ctypes.data_as(ip), 2, m,
                                    lib.laya_attention_block(0, 8), tiles.ctypes.data_as(ip), 10)
    work = t.from_numpy(tiles[:used].copy()).to(gpu)

    def attention(values):
        out = t.empty((m, heads * 64), dtype=t.float16, device=gpu)
        _lib.check(lib.laya_op_attention(*(ct.c_void_p(x.data_ptr()) for x in (q, k, values, out, work)), m, heads, used,
                                         0, 8, -1, _lib.F16, ct.c_void_p(t.cuda.current_stream().cuda_stream)))
        return out
    spoiled = vt.clone()
    spoiled[:, :, :64] = float("inf")
    assert m >= 168 * used  # the ahead kernel
    assert t.equal(attention(spoiled)[64:1094], attention(vt)[64:1094])


def test_slots_past_the_resources_range(gpu):
    """2^25 rows: a head's K plane of 4 GiB no longer fits a buffer resource, so the shared-key kernel with
    64-bit addresses takes it.  One sequence, at the slot's end."""
    import torch as t
    lib = _lib.load()
    m, n = 1 << 25, 200
    start = m - 208
    q, k, vt, out = (t.empty(m * 64, dtype=t.float16, device=gpu) for _ in range(4))
    g = t.Generator(device=gpu).manual_seed(5)
    qs, ks, vs = (t.randn((208, 64), generator=g, device=gpu).half() for _ in range(3))
    q.view(m, 64)[start:], k.view(m, 64)[start:] = qs, ks
    vt.view(64, m)[:, start:] = vs.t()
    work = t.tensor([[start, m, start, n]], dtype=t.int32, device=gpu)
    _lib.check(lib.laya_op_attention(*(ct.c_void_p(x.data_ptr()) for x in (q, k, vt, out, work)), m, 1, 1, 0, 8, -1,
                                     _lib.F16, ct.c_void_p(t.cuda.current_stream().cuda_stream)))
    weights = t.softmax(qs[:n].double() @ ks[:n].double().t().contiguous() / 8, -1)
    want, got = weights @ vs[:n].double(), out.view(m, 64)[start:]
    assert ((got[:n].double() - want).abs() <= (weights @ vs[:n].double().abs() * 2 + 0.05) * 2.0 ** -11).all()
    assert (got[n:] == 0).all()
