"""Products of many rows (``ajqd_product``) against float64, over every tile that the sizes choose and its edges."""

import ctypes

import pytest
import torch

from ajllm_amd import _lib, dense

PLAIN, ACT, PAIRS = "plain", "act", "pairs"
ACTS = {
    "relu": torch.relu, "silu": torch.nn.functional.silu, "squared_relu": lambda z: torch.relu(z).square(),
    "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"),
}


def _args(x, w, y, rows, n, k, ldx, ldy, out=_lib.AJQD_BF16, act=-1, pairs=0):
    return _lib.ProductArgs(x=x, w=w, y=y, rows=rows, n=n, k=k, ldx=ldx, ldy=ldy, out_dtype=out, act=act, pairs=pairs)


# (rows, n, k): the smallest; a row and a tile's rows around 64; tiles of 64 x 128, 192 x 128, 128 x 128, 128 x 256, 192 x 256,
# 256 x 256 with remainders on both sides (asserted below); one, two, an odd and an even number of 64-k steps
SIZES = [(1, 16, 64), (63, 144, 64), (65, 272, 192), (500, 1008, 320), (257, 16000, 192), (1025, 4112, 320), (4097, 4112, 64),
         (1537, 4080, 64), (2040, 4080, 640), (2049, 5008, 128), (3000, 4048, 640), (3080, 8080, 64), (4000, 4016, 192),
         (387, 4624, 192), (2307, 784, 256)]
TILES = {(64, 128), (128, 128), (192, 128), (128, 256), (192, 256), (256, 256)}
FORMS = {"fp32": (_lib.AJQD_F32, 0), "bf16": (_lib.AJQD_BF16, 0), "pairs": (_lib.AJQD_BF16, 1)}


def _tiles(sizes, out, pairs):
    """The tiles that sizes take with several of them and a remainder on both sides, and more steps of 64 k than the tile has buffers."""
    lib, found = _lib.load_dense(), set()
    for rows, n, k, *parts in sizes:
        high, wide = divmod(lib.ajqd_product_tile(rows, n, k, out, pairs, *(parts or (1,))), 1 << 16)
        if rows > high and rows % high and n > wide and n % wide and (parts or k >= 192):
            found.add((high, wide))
    return found


@pytest.mark.parametrize("form", FORMS)
def test_sizes_take_every_tile_in_every_form(form):
    assert _tiles(SIZES, *FORMS[form]) == TILES


@pytest.mark.parametrize("out", [_lib.AJQD_F32, _lib.AJQD_BF16])
def test_sizes_in_parts_take_every_tile(out):
    assert _tiles(PARTS, out, 0) == TILES
    assert _lib.load_dense().ajqd_product_tile(64, 24, 64, out, 0, 1) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("kind,out", [(PLAIN, torch.float32), (PLAIN, torch.bfloat16), (ACT, torch.bfloat16), (PAIRS, torch.bfloat16)])
@pytest.mark.parametrize("rows,n,k", SIZES)
def test_product(cuda, rows, n, k, kind, out):
    lib = _lib.load_dense()
    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    ldx = k + 24
    x = torch.randn((rows, ldx), generator=g, device=cuda).to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device=cuda) * k ** -0.5).to(torch.bfloat16)
    sums = x[:, :k].double() @ w.double().t()
    # fp32 sums of k terms: k roundings of 2^-24 of the terms' absolute sum
    slack = k * 2.0 ** -24 * (x[:, :k].double().abs() @ w.double().t().abs())
    for name in (["relu"] if kind == PLAIN else ACTS):
        want, bound = sums, slack
        if kind == ACT:
            want = ACTS[name](sums)
            # slopes: below 1.2, for the square 2 |z|; the functions themselves within 2^-20 of |z| in fp32
            bound = slack * (2 * sums.abs() + slack if name == "squared_relu" else 1.2) + 2.0 ** -20 * want.abs().maximum(sums.abs())
        if kind == PAIRS:
            gate, up = (t.reshape(rows, -1) for t in sums.view(rows, -1, 2, 8).unbind(2))
            gs, us = (t.reshape(rows, -1) for t in slack.view(rows, -1, 2, 8).unbind(2))
            a = ACTS[name](gate)
            ab = gs * (2 * gate.abs() + gs if name == "squared_relu" else 1.2) + 2.0 ** -20 * a.abs().maximum(gate.abs())
            want, bound = a * up, ab * up.abs() + a.abs() * us + ab * us
        ldy = want.shape[1] + 8
        y = torch.full((rows + 1, ldy), float("nan"), dtype=out, device=cuda)
        act = -1 if kind == PLAIN else _lib.AJQD_ACTIVATIONS[name]
        args = _args(x.data_ptr(), w.data_ptr(), y.data_ptr(), rows, n, k, ldx, ldy,
                     _lib.AJQD_F32 if out == torch.float32 else _lib.AJQD_BF16, act, int(kind == PAIRS))
        _lib.check_dense(lib.ajqd_product(ctypes.byref(args), torch.cuda.current_stream().cuda_stream), "product")
        got = y[:rows, : want.shape[1]].double()
        if out == torch.bfloat16:
            bound = bound + 2.0 ** -8 * (want.abs() + bound)   # to the nearest of 8 significant bits
        assert bool(((got - want).abs() <= bound + 1e-30).all()), (name, float(((got - want).abs() - bound).max()))
        assert bool(y[rows:].isnan().all()) and bool(y[:, want.shape[1]:].isnan().all()), "written outside the result"


# a part of one and of several 64-k steps, a last part that is shorter, more parts than steps, remainders of every tile's sides
PARTS = [(1, 16, 128, 2), (65, 272, 192, 3), (130, 144, 448, 3), (500, 1008, 320, 4), (257, 4112, 640, 4), (1025, 1040, 832, 7), (33, 48, 320, 9),
         (129, 3616, 320, 4), (262, 3632, 320, 3), (770, 3120, 448, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k,parts", PARTS)
def test_product_in_parts(cuda, rows, n, k, parts, out):
    lib = _lib.load_dense()
    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    ldx, ldy = k + 24, n + 8
    x = torch.randn((rows, ldx), generator=g, device=cuda).to(torch.bfloat16)
    w = (torch.randn((n, k), generator=g, device=cuda) * k ** -0.5).to(torch.bfloat16)
    want = x[:, :k].double() @ w.double().t()
    bound = k * 2.0 ** -24 * (x[:, :k].double().abs() @ w.double().t().abs())   # (as above: k roundings, wherever they fall)
    y = torch.full((rows + 1, ldy), float("nan"), dtype=out, device=cuda)
    room = torch.full((lib.ajqd_product_workspace(rows, n, parts) // 4 + 64,), float("nan"), device=cuda)
    assert room.numel() == parts * rows * n + 64
    args = _args(x.data_ptr(), w.data_ptr(), y.data_ptr(), rows, n, k, ldx, ldy, _lib.AJQD_F32 if out == torch.float32 else _lib.AJQD_BF16)
    _lib.check_dense(lib.ajqd_product_in_parts(ctypes.byref(args), parts, room.data_ptr(), torch.cuda.current_stream().cuda_stream), "product")
    if out == torch.bfloat16:
        bound = bound + 2.0 ** -8 * (want.abs() + bound)
    assert bool(((y[:rows, :n].double() - want).abs() <= bound + 1e-30).all())
    assert bool(y[rows:].isnan().all()) and bool(y[:, n:].isnan().all()) and bool(room[-64:].isnan().all()), "written outside the result"


def test_parts_are_for_few_tiles_and_long_sums():
    lib, bf16, f32 = _lib.load_dense(), _lib.AJQD_BF16, _lib.AJQD_F32
    assert lib.ajqd_product_parts(500, 4096, 4096, f32) >= 1 and lib.ajqd_product_parts(1, 16, 64, bf16) == 1
    assert lib.ajqd_product_parts(1500, 288, 8192, bf16) > 1 and lib.ajqd_product_parts(110, 4544, 16960, bf16) > 1
    assert lib.ajqd_product_parts(4096, 4096, 18432, f32) == 1 and lib.ajqd_product_parts(8192, 8192, 512, bf16) == 1
    assert not any(lib.ajqd_product_parts(*s, bf16) for s in ((500, 4096, 96), (500, 24, 64), (0, 16, 64), (500, 4096, 0), (2, 16, (1 << 22) + 64)))
    for rows, n, k in ((3, 64, 320), (700, 288, 8192), (64, 4096, 1088), (9000, 16, 18368)):
        parts = lib.ajqd_product_parts(rows, n, k, f32)   # no part is empty, and the sums fit 128 MiB
        assert (parts - 1) * (-(-(k // 64) // parts)) < k // 64 and (parts == 1 or lib.ajqd_product_workspace(rows, n, parts) <= 1 << 27)


def test_product_refuses_what_it_does_not_make():
    lib = _lib.load_dense()
    buf = ctypes.create_string_buffer(4096 + 16)
    p = (ctypes.addressof(buf) + 15) & ~15   # host memory: only its address is looked at
    assert lib.ajqd_product(None, None) == -1
    for change, status in ((dict(x=None), -1), (dict(rows=0), -2), (dict(n=24), -2), (dict(k=96), -2), (dict(ldx=56), -2), (dict(ldy=8), -2),
                           (dict(ldx=68), -3), (dict(ldy=20), -3), (dict(w=p + 8), -3), (dict(out=2), -4), (dict(act=4), -4),
                           (dict(out=_lib.AJQD_F32, act=0), -4), (dict(pairs=1), -4)):
        args = _args(**{**dict(x=p, w=p, y=p, rows=1, n=16, k=64, ldx=64, ldy=16), **change})
        assert lib.ajqd_product(ctypes.byref(args), None) == status, change
    assert lib.ajqd_product_better(500, 4096, 4096) == 1 and lib.ajqd_product_better(1, 16, 64) == 1
    assert lib.ajqd_product_better(919, 640, 15488) == 0          # few tiles, long sums
    assert not any(lib.ajqd_product_better(*s) for s in ((500, 4096, 96), (500, 24, 64), (0, 16, 64), (500, 4096, 0), (4096, 4096, (1 << 22) + 64)))
    for change, status in ((dict(rows=0), -2), (dict(ldy=20), -3), (dict(act=1), -4), (dict(k=128, ldx=128), -1)):   # (the last: no workspace)
        args = _args(**{**dict(x=p, w=p, y=p, rows=1, n=16, k=64, ldx=64, ldy=16), **change})
        assert lib.ajqd_product_in_parts(ctypes.byref(args), 2, None, None) == status, change


def test_rows_that_the_product_does_not_read_are_left_to_the_vendors():
    """Which answers, or says what does not fit: only the forms that the kernel reads are taken to it."""
    w = torch.zeros((32, 64), dtype=torch.bfloat16)
    x = torch.zeros((4, 88), dtype=torch.bfloat16)
    far = torch.zeros(3 * (1 << 22), dtype=torch.bfloat16)   # (not touched)
    assert dense._product_rows(x[:, :64], w) and dense._product_rows(far.as_strided((3, 64), (1 << 22, 1)), w)
    for rows, weights in ((x[:, :72], w), (x[:, :64].float(), w), (x[:, :64], w.float()), (x[:, 4:68], w), (x[:, :64], torch.zeros((64, 32), dtype=w.dtype).t()),
                          (x[:, :64], torch.zeros((32, 128), dtype=w.dtype)[:, ::2]), (x[:1, :64].expand(4, 64), w), (x.as_strided((4, 64), (8, 1)), w),
                          (far.as_strided((2, 64), ((1 << 22) + 8, 1)), w), (x[:, :64], w.to("meta"))):
        assert not dense._product_rows(rows, weights), (rows.shape, rows.stride(), weights.stride())
    with pytest.raises(RuntimeError):
        dense._product(x[:, :72], w, torch.bfloat16)


def test_more_parts_than_there_is_to_cut():
    """Any number of parts is one: the sums that round it up must not overflow."""
    lib = _lib.load_dense()
    buf = ctypes.create_string_buffer(4096 + 16)
    p = (ctypes.addressof(buf) + 15) & ~15   # host memory: only its address is looked at
    args = _args(x=p, w=p, y=p, rows=1, n=16, k=128, ldx=128, ldy=16)
    assert lib.ajqd_product_in_parts(ctypes.byref(args), 2**31 - 1, None, None) == -1   # (no workspace)
