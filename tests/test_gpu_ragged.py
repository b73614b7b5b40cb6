"""GPU parity of rows off the 16-byte grid: widths that are no whole number of 16-byte vectors and
pointers off a 16-byte boundary, at the edges of their tiles, against the oracle's bars."""
from __future__ import annotations

import pytest
import torch

import capi
import test_gpu_capi as checks
from gpu_calls import cuda, ln_forward, workspace

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
KINDS = ["ln", "rms", "gelu_tanh", "gelu_none", "add_ln", "ln_fp8", "ln_dres", "add_rms",
         "rms_fp8", "add_ln_fp8"]
# One column past / short of a wave's, a tile's or a block's worth of vectors (16-bit and fp32),
# with every remainder of a vector among them; 16383 the widest register rows.
WIDTHS = [257, 263, 511, 513, 1030, 1281, 2049, 2561, 3071, 4097, 6145, 8191, 8193, 12292, 16383]
ROWS = [1, 37, 600]


@pytest.fixture(scope="module")
def lib(gpu_available):
    return capi.load()


def _cases():
    for i, cols in enumerate(WIDTHS):
        for j, kind in enumerate(KINDS):
            yield kind, DTYPES[(i + j) % 3], ROWS[(i + 2 * j) % 3], cols, (i + j) % 4 == 3
    for i, cols in enumerate([288, 4096, 16384]):  # whole vectors and MX blocks, off alignment
        for j, kind in enumerate(KINDS + ["ln_mx", "add_rms_mx"]):
            yield kind, DTYPES[(i + j) % 3], ROWS[(i + j) % 3], cols, True


@pytest.mark.parametrize("kind,dtype,rows,cols,shifted", list(_cases()),
                         ids=lambda v: str(v)[6:] if isinstance(v, torch.dtype) else str(v))
def test_ragged_rows(lib, kind, dtype, rows, cols, shifted):
    """The forward (and backward, where the flavour has one) of ragged rows within the bars of
    the random-shape test."""
    checks.test_random_shapes_against_the_oracle(lib, kind, dtype, rows, cols, shifted)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows,cols", [(5, 1023), (300, 513), (2, 8193), (3, 20001)])
def test_ragged_outputs_stay_inside(lib, dtype, rows, cols):
    """y and dx inside larger buffers: not a byte before or after them changes."""
    gen = torch.Generator().manual_seed(cols)
    pad = 64
    x, dy = (cuda(torch.randn(rows, cols, generator=gen).to(dtype)) for _ in range(2))
    g = cuda(torch.randn(cols, generator=gen).to(dtype))
    y0, mean, rstd = ln_forward(lib, x, g, None, 1e-5)
    n = rows * cols
    p = capi.ptr
    code, st = capi.dtype_code(x), capi.stream()
    ws, nb = workspace(lib, rows, cols, x)

    def fwd(out):
        return lib.fln_layernorm_forward(p(x), p(g), None, p(out), None, None, rows, cols, code,
                                         1e-5, st)

    def bwd(out):  # dx alone
        return lib.fln_layernorm_backward(p(dy), p(x), p(mean), p(rstd), p(g), None, p(out), None,
                                          None, rows, cols, code, capi.F32, p(ws), nb, st)

    dx0 = torch.empty_like(x)
    capi.check(bwd(dx0))
    for lead in (1, pad):  # off and on a 16-byte boundary
        for call, want in ((fwd, y0), (bwd, dx0)):
            buf = torch.full((lead + n + pad,), 7.0, device="cuda", dtype=dtype)
            out = buf[lead:lead + n]
            capi.check(call(out))
            assert (buf[:lead] == 7).all() and (buf[lead + n:] == 7).all()
            assert torch.equal(out.view(rows, cols), want)


# In place, the elements that a row's last vector shares with the one before it matter where the two
# lie in different waves, blocks or steps: within a wave all loads come before any store.
IN_PLACE = [(3, 600), (300, 1023), (7, 8193), (5, 20001), (300, 33001),
            (5, 20481), (40, 20481), (300, 20481),  # starts a wave and a column block
            (5, 32769), (40, 32769)]                # ... and a step of the streamed forward


def test_in_place_widths_part_the_shared_elements():
    """The widths above do what they are there for (in each element size; the quarter vectors of the
    few-row column pass are 2 16-bit elements, or one fp32 one, which share nothing)."""
    for cols, step in ((20481, 64), (32769, 4096)):
        for vec in (2, 4, 8):
            last = -(-cols // vec) - 1  # index of the last vector
            assert (last + 1) * vec - cols == vec - 1  # one element of its own
            assert last % 256 == 0 and (vec == 2 or last % step == 0)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows,cols", IN_PLACE)
def test_ragged_in_place(lib, monkeypatch, dtype, rows, cols):
    """y over x and dx over dy, x or dres, on the routes of separate buffers (without the one-launch
    backward, which takes no such call): the outputs of separate buffers bit for bit."""
    gen = torch.Generator().manual_seed(cols + 1)
    x, dy, r = (cuda(torch.randn(rows, cols, generator=gen).to(dtype)) for _ in range(3))
    g, b = (cuda(torch.randn(cols, generator=gen).to(dtype)) for _ in range(2))
    p = capi.ptr
    code, st = capi.dtype_code(x), capi.stream()
    y0, mean, rstd = ln_forward(lib, x, g, b, 1e-5)
    y = x.clone()
    capi.check(lib.fln_layernorm_forward(p(y), p(g), p(b), p(y), None, None, rows, cols, code,
                                         1e-5, st))
    assert torch.equal(y, y0)
    ws, nb = workspace(lib, rows, cols, x)

    def backward(dres, over):
        t = {"dy": dy.clone(), "x": x.clone(), "dres": r.clone() if dres else None}
        dx = t[over] if over else torch.empty_like(x)
        dg, db = torch.empty(cols, device="cuda"), torch.empty(cols, device="cuda")
        capi.check(lib.fln_layernorm_backward(p(t["dy"]), p(t["x"]), p(mean), p(rstd), p(g),
                                              p(t["dres"]), p(dx), p(dg), p(db), rows, cols, code,
                                              capi.F32, p(ws), nb, st))
        return dx, dg, db

    small = backward(False, None)  # by whatever route
    monkeypatch.setenv("FLN_BWD_SMALL_ROWS", "-1")
    capi.reload_tuning()
    for dres in (False, True):
        want = backward(dres, None)
        for over in ("dy", "x", "dres")[:3 if dres else 2]:
            for a, c in zip(backward(dres, over), want):
                assert torch.equal(a, c), (dres, over)
    # The one launch sums in another order: within a rounding of the largest value.
    ulp = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    for a, c in zip(small, backward(False, None)):
        scale = c.float().abs().max()
        assert (a.float() - c.float()).abs().max() <= (ulp if a.dtype == dtype else 1e-5) * scale


@pytest.mark.parametrize("threads", ["256", "512", "1024"])
@pytest.mark.parametrize("kind,dtype,cols", [("ln", torch.bfloat16, 1401), ("rms", torch.float16, 1030),
                                             ("gelu_tanh", torch.bfloat16, 1401),
                                             ("gelu_none", torch.float32, 1403),
                                             ("ln", torch.float32, 1403)])
def test_forced_blocks_hold_whole_row_groups(lib, monkeypatch, kind, dtype, cols, threads):
    """Ragged rows of three waves in forced block sizes: 256 threads are one row group of 192, fewer
    than the GELU' table has entries and so many blocks per CU that the partial rows of all of them
    would pass the workspace."""
    monkeypatch.setenv("FLN_BWD_THREADS", threads)
    monkeypatch.setenv("FLN_BWD_WPR", "3")
    capi.reload_tuning()
    checks.test_random_shapes_against_the_oracle(lib, kind, dtype, 1500, cols, False)


def test_streamed_grids_do_not_depend_on_the_calls_before(lib, monkeypatch, capfd):
    """The grid of a streamed forward is what its own kernel's occupancy gives, whichever flavour ran
    first: a ragged bf16 LayerNorm fits a CU twice, residual + LayerNorm (over 64 VGPRs) once."""
    cols, p, st = 20001, capi.ptr, capi.stream()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rows = 2 * cus
    x = torch.randn(rows, cols, device="cuda", dtype=torch.bfloat16)
    y, h = torch.empty_like(x), torch.empty_like(x)
    monkeypatch.setenv("FLN_DEBUG_GEOMETRY", "2")
    capi.reload_tuning()
    grids = []
    for _ in range(2):
        for residual in (True, False):
            capfd.readouterr()
            if residual:
                rc = lib.fln_add_layernorm_forward(p(x), p(x), None, None, p(h), p(y), None, None,
                                                   rows, cols, capi.BF16, 1e-5, st)
            else:
                rc = lib.fln_layernorm(p(x), None, None, p(y), rows, cols, capi.BF16, 1e-5, st)
            capi.check(rc)
            torch.cuda.synchronize()
            grids.append(int(capfd.readouterr().err.split("fln wide: blocks=")[1].split()[0]))
    assert grids == [cus, 2 * cus] * 2


def test_mean_sums_each_vector_by_itself(lib):
    """fp32 rows of 4093 columns: 4 waves of 4 vectors per lane, columns 0-3, 1024-1027, ... in lane
    0.  2^24 and then 15 ones there: three of them are lost against 2^24 in its own vector (ties
    to even), the others arrive as sums of four; in one chain all 15 are lost."""
    rows, cols = 3, 4093
    x = torch.zeros(rows, cols, dtype=torch.float64)
    for k in range(4):
        x[:, 1024 * k:1024 * k + 4] = 1
    x[:, 0] = 2.0 ** 24
    want = x.sum(1)
    _, mean, _ = ln_forward(lib, cuda(x.float()), None, None, 1e-5)
    # sum / cols is rounded to within an ulp: 2^-23 of it
    assert ((mean.double().cpu() * cols - want).abs() <= 3 + 2.0 ** -23 * want).all()
