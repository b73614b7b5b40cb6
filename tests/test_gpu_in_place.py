"""Residual sums in place: h over x or over the residual, y over the other one, on every forward
route, the outputs of buffers of their own
(bit for bit but where a comment says otherwise)."""
from __future__ import annotations

import pytest
import torch

import capi
from gpu_calls import cuda

pytestmark = pytest.mark.gpu

BF16, F16, F32, F64 = torch.bfloat16, torch.float16, torch.float32, torch.float64
# route, dtype, rows, cols, knob.  Of the ragged streamed rows 20481 and 32769 columns start a wave
# (32769: a step) with their last vector, so that another wave holds the elements it shares; 20512
# is off alignment only (MX blocks).
ROUTES = [("registers", BF16, 37, 1023, None), ("registers", F32, 40, 8192, None),
          ("registers", F16, 9, 12293, None), ("lds", F32, 6, 24576, "FLN_FWD_NO_SPLIT"),
          ("split", BF16, 3, 131072, None), ("wide", BF16, 5, 131072, "FLN_FWD_NO_SPLIT"),
          ("wide", F32, 1100, 40960, None), ("wide", BF16, 5, 20481, None),
          ("wide", F16, 300, 32769, None), ("wide", F32, 6, 20481, None),
          ("wide", F32, 6, 32769, None), ("wide", F16, 7, 20512, "shifted"),
          ("loop", BF16, 5, 1030, "FLN_FORCE_LOOP"), ("loop", F32, 3, 4128, "FLN_FORCE_LOOP"),
          ("loop", F64, 3, 515, None)]
KINDS = ["add_ln", "add_rms", "add_ln_fp8", "add_rms_fp8", "add_rms_mx"]


@pytest.fixture(scope="module")
def lib(gpu_available):
    return capi.load()


def _call(lib, kind, x, r, g, b, h, y, stats):
    p, st = capi.ptr, capi.stream()
    rows, cols = x.shape
    code = capi.dtype_code(x)
    mean, rstd, scale = stats
    if kind == "add_ln":
        rc = lib.fln_add_layernorm_forward(p(x), p(r), p(g), p(b), p(h), p(y), p(mean), p(rstd),
                                           rows, cols, code, 1e-5, st)
    elif kind == "add_rms":
        rc = lib.fln_add_rmsnorm_forward(p(x), p(r), p(g), p(h), p(y), p(rstd), rows, cols, code,
                                         1e-5, st)
    elif kind == "add_ln_fp8":
        rc = lib.fln_add_layernorm_fp8_forward(p(x), p(r), p(g), p(b), p(h), p(y), p(scale),
                                               p(mean), p(rstd), rows, cols, code, 1e-5, st)
    elif kind == "add_rms_fp8":
        rc = lib.fln_add_rmsnorm_fp8_forward(p(x), p(r), p(g), p(h), p(y), p(scale), p(rstd), rows,
                                             cols, code, 1e-5, st)
    else:
        rc = lib.fln_add_rmsnorm_mxfp8_forward(p(x), p(r), p(g), p(h), p(y), p(scale), p(rstd),
                                               rows, cols, code, 1e-5, st)
    capi.check(rc)


# fp64 has LayerNorm alone, and MX blocks are 32 columns.
CASES = [(*r, kind) for r in ROUTES for kind in KINDS
         if (kind == "add_ln" or r[1] != F64) and not (kind.endswith("mx") and r[3] % 32)]


@pytest.mark.parametrize("route,dtype,rows,cols,knob,kind", CASES,
                         ids=lambda v: str(v).split(".")[-1])
def test_residual_sum_in_place(lib, monkeypatch, capfd, route, dtype, rows, cols, knob, kind):
    gen = torch.Generator().manual_seed(rows + cols)
    xc, rc = (torch.randn(rows, cols, generator=gen).to(dtype) for _ in range(2))
    g, b = (cuda(torch.randn(cols, generator=gen).to(dtype)) for _ in range(2))
    quant = kind.endswith(("fp8", "mx"))
    if knob and knob != "shifted":
        monkeypatch.setenv(knob, "1")
    monkeypatch.setenv("FLN_DEBUG_GEOMETRY", "1")
    capi.reload_tuning()

    def buffer(t):
        t = cuda(t)
        if knob != "shifted":
            return t
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
        buf[1:] = t.flatten()
        return buf[1:].view(t.shape)

    def run(h_over, y_over):
        x, r = buffer(xc), buffer(rc)
        h = {None: buffer(torch.full_like(xc, 7)), "x": x, "r": r}[h_over]
        y = r if y_over and h_over == "x" else x if y_over else None
        if y is None:
            y = torch.zeros(rows, cols, device="cuda", dtype=torch.uint8 if quant else dtype)
        mean, rstd = torch.zeros(2, rows, device="cuda")
        scale = torch.zeros(rows, cols // 32 if kind.endswith("mx") else 1, device="cuda",
                            dtype=torch.uint8 if kind.endswith("mx") else torch.float32)
        capfd.readouterr()
        _call(lib, kind, x, r, g, b, h, y, (mean, rstd, scale))
        torch.cuda.synchronize()
        if dtype != F64:
            err = capfd.readouterr().err
            taken = "wide" if y_over and route == "split" else route  # y over an input: no split
            assert f"-> {taken} " in err, err
        return h, y, mean, rstd, scale

    want = run(None, False)
    assert torch.equal(want[0], cuda(xc + rc))
    for h_over in ("x", "r"):
        for y_over in (False,) if quant else (False, True):
            got = run(h_over, y_over)
            for a, c in zip(got, want):
                if y_over and route == "split":  # one block per row sums in another order
                    ulp = 2.0 ** -7 * c.abs().max() if c.dtype == dtype else 1e-5
                    assert ((a - c).abs() <= ulp).all()
                elif dtype == F16 and route == "wide" and c is want[1] and not quant:
                    # Two kernels, of which one forms y with a mixed FMA that rounds to fp16 at once
                    # and the other rounds to fp32 first: both are within half an ulp (and half an
                    # fp32 ulp) of the same value, so they are equal or neighbours.
                    assert ((a - c).abs().float() <= 2.0 ** -10 * c.abs().float() + 2.0 ** -24).all()
                else:
                    assert torch.equal(a, c), (h_over, y_over)
