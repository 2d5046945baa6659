"""The selective scan with time cut into parts against the sequential recurrence in float64: part boundaries on and off the kernel's
tiles, ragged channels, fewer states than the kernel has places for, with and without a state to start from or to leave."""

import ctypes
import math

import pytest
import torch

from ajllm_amd import _lib, dense, hybrid
from tests.test_gpu_hybrid import DTYPES, _rel, _scan_case, _scan_plain

# batch, tokens, channels, states, parts (the last of which may turn out empty and be left out)
SHAPES = [(1, 33, 8, 4, 2), (1, 64, 48, 16, 2), (2, 150, 72, 12, 5), (3, 257, 136, 16, 8), (1, 100, 64, 8, 50), (2, 96, 200, 16, 3)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", SHAPES)
def test_scan_in_parts(cuda, dtype, shape):
    batch, seq, inner, states, parts = shape
    lib, st = _lib.load_dense(), torch.cuda.current_stream().cuda_stream
    c, rank = _scan_case(batch, seq, inner, states, sum(shape))
    d = {k: c[k].to(cuda).to(dtype).contiguous() for k in ("x", "raw", "z", "low")}
    a2 = hybrid.state_planes(-torch.exp(c["a_log"].double()) * math.log2(math.e)).float().to(cuda)
    skip, bias = c["d"].to(cuda), c["bias"].to(cuda)
    nbytes = lib.ajqd_scan_workspace(batch, inner, states, parts)
    assert nbytes == 4 * batch * inner * (parts * states + parts - 1)
    for carried in (False, True):
        state = hybrid.state_planes(c["state"] if carried else torch.full_like(c["state"], float("nan"))).to(cuda)
        want, end = _scan_plain(c, rank, states, carried)
        for kept in (state, None) if not carried else (state,):
            out = torch.full((batch, seq, inner), float("nan"), dtype=dtype, device=cuda)
            room = torch.full((nbytes // 4 + 64,), float("nan"), device=cuda)
            args = _lib.ScanArgs(x=d["x"].data_ptr(), dt=d["raw"].data_ptr(), low=d["low"].data_ptr(), z=d["z"].data_ptr(), a2=a2.data_ptr(),
                                 d=skip.data_ptr(), dt_bias=bias.data_ptr(), state=kept.data_ptr() if kept is not None else None, pos=None,
                                 out=out.data_ptr(), batch=batch, seq=seq, start=7 if carried else 0, inner=inner, states=states, dt_ld=inner,
                                 low_ld=rank + 2 * states, b_col=rank, c_col=rank + states, z_ld=inner, out_ld=inner)
            _lib.check_dense(lib.ajqd_scan_in_parts(ctypes.byref(args), parts, room.data_ptr(), dense._flag(dtype), st), "scan_in_parts")
            # the tolerances of the scan in one piece
            assert _rel(out, want) < (4e-6 if dtype == torch.float32 else 4e-3)
            assert bool(room[nbytes // 4:].isnan().all()), "written behind the workspace"
        assert _rel(state, hybrid.state_planes(end)) < 4e-6


def test_parts_are_for_few_channels_and_long_prompts():
    lib = _lib.load_dense()
    assert lib.ajqd_scan_parts(1, 1500, 8192, 16) > 1 and lib.ajqd_scan_parts(2, 192, 2048, 4) > 1
    assert lib.ajqd_scan_parts(1, 100, 8192, 16) == 1 and lib.ajqd_scan_parts(4, 700, 4096, 16) == 1 and lib.ajqd_scan_parts(1, 1500, 8192, 32) == 1
    assert lib.ajqd_scan_workspace(1, 8192, 16, 1) == 0


def test_more_parts_than_tokens():
    """Any number of parts is one: the sums that round it up must not overflow.  (More parts than a grid has rows: refused, not launched.)"""
    lib = _lib.load_dense()
    buf = ctypes.create_string_buffer(4096 + 16)
    p = (ctypes.addressof(buf) + 15) & ~15   # host memory: only its address is looked at
    args = _lib.ScanArgs(x=p, dt=p, low=p, z=p, a2=p, d=p, dt_bias=p, state=None, pos=None, out=p, batch=1, seq=65540 * 32, start=0, inner=8,
                         states=4, dt_ld=8, low_ld=8, b_col=0, c_col=4, z_ld=8, out_ld=8)
    for parts in (65540, 2**31 - 1):
        assert lib.ajqd_scan_in_parts(ctypes.byref(args), parts, p, _lib.AJQD_BF16, None) == -2
