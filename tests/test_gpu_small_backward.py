"""The one-launch backward of few rows: the oracle's bars at the edges of its tiles, every subset of
the outputs, calls without a workspace, and the calls that it leaves to the other kernels."""
from __future__ import annotations

import pytest
import torch

import capi
import test_gpu_capi as checks
from gpu_calls import cuda, ln_forward, workspace

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
KINDS = ["ln", "rms", "gelu_tanh", "gelu_none", "ln_dres"]
# Vectors of a row around a wave's, 16 waves' and 16 waves' times 2, 4 and 8, by the vector width;
# the last is past the kernel's widest row.
VECTORS = [1, 2, 63, 65, 250, 1024, 1025, 2049, 4097, 8192, 8193]
ROWS = [1, 2, 17, 65, 200, 256]


@pytest.fixture(scope="module")
def lib(gpu_available):
    return capi.load()


def _cases():
    for i, nvec in enumerate(VECTORS):
        for j, kind in enumerate(KINDS):
            dtype = DTYPES[(i + j) % 3]
            vec = 4 if dtype == torch.float32 else 8
            off = (0, 1, 3)[(i + 2 * j) % 3] if nvec > 1 else 0
            cols = nvec * vec - off
            rows = min(ROWS[(i + j) % len(ROWS)], 4_000_000 // cols)
            yield kind, dtype, rows, cols, (i + j) % 4 == 0


@pytest.mark.parametrize("kind,dtype,rows,cols,shifted", list(_cases()),
                         ids=lambda v: str(v)[6:] if isinstance(v, torch.dtype) else str(v))
def test_small_backward(lib, monkeypatch, capfd, kind, dtype, rows, cols, shifted):
    monkeypatch.setenv("FLN_DEBUG_GEOMETRY", "1")
    capi.reload_tuning()
    capfd.readouterr()
    checks.test_random_shapes_against_the_oracle(lib, kind, dtype, rows, cols, shifted)
    err = capfd.readouterr().err
    assert err.count("fln backward:") == 1, err
    # 16 waves of 8 vectors per lane at most; of those few rows and 16-bit GELU take the two passes,
    # and 16-bit GELU of 4 vectors per lane too unless every block has a CU of its own.
    vec = 4 if dtype == torch.float32 else 8
    nvec, cus = -(-cols // vec), torch.cuda.get_device_properties(0).multi_processor_count
    gelu16 = kind.startswith("gelu") and vec == 8
    small = cols >= vec and nvec <= 8192 and rows <= cus
    if nvec > 4096:
        small = small and not gelu16 and rows >= (32 if vec == 8 and cols % vec else 16)
    elif nvec > 2048 and gelu16:
        small = small and rows + -(-nvec // 64) <= cus
    assert ("-> small" in err) == small, err


# Around the rows and widths at which the two passes take over from the one launch, and those of
# their column pass over quarters of a vector (1 to 3 elements past its tiles and vectors).
@pytest.mark.parametrize("rows", [1, 7, 8, 9, 15, 16, 17, 31, 33])
@pytest.mark.parametrize("kind,dtype,cols", [
    ("ln", torch.bfloat16, 33281), ("ln_dres", torch.float16, 40960), ("gelu_none", torch.bfloat16,
     32770), ("gelu_tanh", torch.float32, 16643), ("rms", torch.float32, 20481)])
def test_few_wide_rows(lib, kind, dtype, rows, cols):
    checks.test_random_shapes_against_the_oracle(lib, kind, dtype, rows, cols, rows % 2 == 1)


def _backward(lib, dy, x, mean, rstd, g, want, ws=True, dx=None):
    rows, cols = x.shape
    p = capi.ptr
    dx = torch.empty_like(x) if want[0] and dx is None else dx
    dg = torch.empty(cols, device="cuda") if want[1] else None
    db = torch.empty(cols, device="cuda") if want[2] else None
    buf, n = workspace(lib, rows, cols, x) if ws else (None, 0)
    capi.check(lib.fln_layernorm_backward(
        p(dy), p(x), p(mean), p(rstd), p(g), None, p(dx), p(dg), p(db), rows, cols,
        capi.dtype_code(x), capi.F32, p(buf), n, capi.stream()))
    return dx, dg, db


@pytest.mark.parametrize("rows,cols", [(17, 1023), (256, 768), (20, 40000), (300, 768)])
def test_small_backward_outputs_and_routes(lib, monkeypatch, capfd, rows, cols):
    """Each subset of the outputs has the bits of the full call; dx alone needs no workspace; more
    rows than CUs, outputs over inputs and forced tilings take the other kernels."""
    gen = torch.Generator().manual_seed(rows)
    x, dy = (cuda(torch.randn(rows, cols, generator=gen).to(torch.bfloat16)) for _ in range(2))
    g = cuda(torch.randn(cols, generator=gen).to(torch.bfloat16))
    _, mean, rstd = ln_forward(lib, x, g, None, 1e-5)
    args = (dy, x, mean, rstd, g)

    def routed(**kw):
        capfd.readouterr()
        monkeypatch.setenv("FLN_DEBUG_GEOMETRY", "1")
        capi.reload_tuning()
        out = _backward(lib, *args, **kw) if "args" not in kw else _backward(lib, *kw.pop("args"),
                                                                             **kw)
        torch.cuda.synchronize()
        monkeypatch.delenv("FLN_DEBUG_GEOMETRY")
        capi.reload_tuning()
        err = capfd.readouterr().err
        assert err.count("fln backward:") == 1, err
        return "-> small" in err, out

    small, full = routed(want=(1, 1, 1))
    assert small == (rows <= 256)
    for want in ((1, 0, 0), (0, 1, 1), (0, 1, 0), (0, 0, 1)):
        got = _backward(lib, *args, want=want)
        for a, c, w in zip(got, full, want):
            assert (a is not None) == bool(w)
            assert a is None or not small or torch.equal(a, c)
    if small:
        assert torch.equal(_backward(lib, *args, want=(1, 0, 0), ws=False)[0], full[0])
    over, (dx, _, _) = routed(want=(1, 1, 1), args=(d := dy.clone(), *args[1:]), dx=d)
    assert not over
    assert (dx.float() - full[0].float()).abs().max() <= 2.0 ** -7 * full[0].abs().max()
    monkeypatch.setenv("FLN_BWD_SMALL_ROWS", "-1")
    off, _ = routed(want=(1, 1, 1))
    monkeypatch.delenv("FLN_BWD_SMALL_ROWS")
    capi.reload_tuning()
    assert not off


@pytest.mark.parametrize("rows,cols,fits", [(1, 4194000, True), (1, 4194305, False),
                                            (4, 4194305, False)])
def test_one_block_row_keeps_the_scratch_limit(lib, rows, cols, fits):
    """fln_layernorm_backward_noalloc holds 32 MiB: two fp32 rows of 4194304 columns, less the row
    statistics, also where the column pass writes dgamma and dbeta itself."""
    x = torch.randn(rows, cols, device="cuda")
    mean, rstd = torch.zeros(rows, device="cuda"), torch.ones(rows, device="cuda")
    dx, dg, db = torch.empty_like(x), torch.empty(cols, device="cuda"), torch.empty(cols,
                                                                                  device="cuda")
    p = capi.ptr
    rc = lib.fln_layernorm_backward_noalloc(p(x), p(x), p(mean), p(rstd), None, None, p(dx), p(dg),
                                            p(db), rows, cols, capi.F32, capi.F32, capi.stream())
    torch.cuda.synchronize()
    assert rc == (0 if fits else capi.ERR_TOO_LARGE)
