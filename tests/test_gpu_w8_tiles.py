"""The int8 tile kernels whose waves take turns (``dequant_gemm_turns_kernel``) against float64: every tile shape at sizes with
remainders on both sides, the shortest K, an even and an odd number of 128-k blocks; plain fp32 and bf16, and with the SwiGLU gate."""

import shutil

import pytest
import torch

from ajllm_amd import _lib, asm_check, repack_w8

# (rows, columns, K) by the tile they take
SIZES = {(192, 128): [(3841, 4112, 384), (1007, 10800, 128), (993, 10800, 256), (986, 10784, 384)],
         (128, 256): [(1537, 4112, 256), (600, 12304, 256), (257, 16400, 1024)],
         (192, 256): [(900, 9232, 384), (520, 14352, 512), (2049, 5136, 128)],
         (256, 256): [(3900, 3856, 640), (1000, 15888, 640), (3500, 4560, 512)],
         (256, 128): [(2305, 2064, 384)]}   # (their waves do not take turns: one more size of the int8 form)
GATED = {(192, 128): [(998, 5440, 128), (978, 5440, 384)], (128, 256): [(1537, 2112, 256)], (192, 256): [(2049, 2624, 128), (900, 4672, 384)],
         (256, 256): [(3900, 1984, 640)]}


def test_sizes_take_the_tiles_they_are_listed_under():
    lib = _lib.load()
    for tile, sizes in SIZES.items():
        for m, n, k in sizes:
            assert divmod(lib.ajq_matmul_tile(m, n, k, 0), 1 << 16) == tile, (m, n, k)
    for tile, sizes in GATED.items():
        for m, f, k in sizes:
            assert divmod(lib.ajq_matmul_tile(m, 2 * f, k, 0), 1 << 16) == tile, (m, f, k)


def test_short_k_takes_the_tile_that_measured_faster():
    """Below K = 1024 the 192 x 128 tile was chosen by times extrapolated from longer sums (fp32 out, us there / at the tile below: 17.9 / 15.8,
    18.1 / 15.5, 17.8 / 16.0, 74.7 / 64.2, 169.5 / 147.6)."""
    lib = _lib.load()
    for m, n, k in ((2994, 4544, 128), (765, 17584, 128), (5888, 2336, 128), (1143, 23984, 896), (3109, 29472, 512)):
        assert divmod(lib.ajq_matmul_tile(m, n, k, 0), 1 << 16) == (256, 256), (m, n, k)


def _weights(n, k, cuda):
    g = torch.Generator(device=cuda).manual_seed(n + k)
    q = torch.randint(-127, 128, (n, k), generator=g, device=cuda, dtype=torch.int8)
    scales = (torch.rand(n, generator=g, device=cuda) * 1e-3 + 1e-4).half()
    return repack_w8(q), scales, q.double() * scales.double()[:, None]


def _bound(x, w, k):
    """fp32 sums of k terms and one product with the scale: a rounding of 2^-24 of the absolute sum each."""
    return (k + 1) * 2.0 ** -24 * (x.double().abs() @ w.abs().t())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [s for sizes in SIZES.values() for s in sizes])
def test_w8_tiles(cuda, m, n, k):
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    wq, scales, w = _weights(n, k, cuda)
    x = torch.randn((m, k), generator=torch.Generator(device=cuda).manual_seed(m), device=cuda).to(torch.bfloat16)
    want, bound = x.double() @ w.t(), _bound(x, w, k)
    for dtype, flag in ((torch.float32, _lib.AJQ_OUT_F32), (torch.bfloat16, _lib.AJQ_OUT_BF16)):
        y = torch.full((m + 1, n), float("nan"), dtype=dtype, device=cuda)
        _lib.check(lib.ajq_w8a16_gemm(x.data_ptr(), m, k, wq.data_ptr(), scales.data_ptr(), n, y.data_ptr(), flag, stream), "gemm")
        limit = bound if dtype == torch.float32 else bound + 2.0 ** -8 * (want.abs() + bound)
        assert bool(((y[:m].double() - want).abs() <= limit).all()), float(((y[:m].double() - want).abs() - limit).max())
        assert bool(y[m:].isnan().all()), "written behind the last row"


@pytest.mark.gpu
@pytest.mark.parametrize("m,f,k", [s for sizes in GATED.values() for s in sizes])
def test_w8_tiles_with_the_gate(cuda, m, f, k):
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    wq, scales, w = _weights(2 * f, k, cuda)
    x = torch.randn((m, k), generator=torch.Generator(device=cuda).manual_seed(m), device=cuda).to(torch.bfloat16)
    assert lib.ajq_gemm_gate_supported(m, 2 * f, k, 0) == 1
    y = torch.full((m + 1, f), float("nan"), dtype=torch.bfloat16, device=cuda)
    _lib.check(lib.ajq_w8a16_gemm_gate(x.data_ptr(), m, k, wq.data_ptr(), scales.data_ptr(), 2 * f, y.data_ptr(), stream), "gate")
    sums, bound = x.double() @ w.t(), _bound(x, w, k)
    a, u = sums[:, :f], sums[:, f:]
    silu = torch.nn.functional.silu(a)
    ab = 1.2 * bound[:, :f] + 2.0 ** -20 * a.abs()   # silu's slope is below 1.2; the function itself within 2^-20 of |a| in fp32
    limit = ab * u.abs() + silu.abs() * bound[:, f:] + ab * bound[:, f:]
    want = silu * u
    limit = limit + 2.0 ** -8 * (want.abs() + limit) + 1e-30
    assert bool(((y[:m].double() - want).abs() <= limit).all()), float(((y[:m].double() - want).abs() - limit).max())
    assert bool(y[m:].isnan().all()), "written behind the last row"


SOURCE = """
#include <hip/hip_runtime.h>
#include "ajq_common.h"
#include "gemm_kernels.h"
#include "gemm_turns_kernels.h"
namespace ajq {
#define TILE const uint16_t*, int, int, const u32x4_t*, const uint16_t*, int, void*, int
%s
}
""" % "\n".join(f"template __global__ void dequant_gemm_turns_kernel<{gate}, {qm}, {qn}>(TILE);"
               for gate in ("false", "true") for qm, qn in ((4, 2), (3, 2), (2, 2), (3, 1)))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_registers_of_loads_in_flight_are_left_alone():
    """The packed words' loads stay in flight around the main loop; their wait counts leave no room for spills either."""
    listing = asm_check.compile_device_asm(SOURCE)
    found = asm_check.scan(listing, "dequant_gemm_turns")
    assert len(found) == 8, sorted(found)
    offending = {name: lines[:3] for name, lines in found.items() if lines}
    assert not offending, offending
    assert "scratch_" not in listing
