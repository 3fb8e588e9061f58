"""The decode-in-registers QMM (tiles of 64, 128 or 256 rows x 256 columns) at the
edges of its tiles, forced on with EXL3_WIDE=1 and its shape with EXL3_WIDE_R /
EXL3_WIDE_SPLITS, against the CPU oracle (tolerances of test_gpu_linear.py) and
against the producer/consumer QMM.

One K-range on both sides multiplies and adds in the same order through the same
epilogue, so the two kernels are bit-identical there."""

import numpy as np
import pytest

import oracle
from mlxl3_amd import synth
from test_gpu_linear import TOL_MODE1_REL, TOL_MODE1_ULP, bf16_bits, check, make_layer, run, ulp_of

pytestmark = pytest.mark.gpu


def force(monkeypatch, r, splits):
    monkeypatch.setenv("EXL3_WIDE", "1")
    monkeypatch.setenv("EXL3_WIDE_R", str(r))
    monkeypatch.setenv("EXL3_WIDE_SPLITS", str(splits))
    monkeypatch.setenv("EXL3_QMM_SPLITS", "1")  # read only where EXL3_WIDE=0


@pytest.mark.parametrize("k", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
@pytest.mark.parametrize("r", [4, 8, 16])
def test_every_k_and_codebook(monkeypatch, k, cb, r):
    # 384 columns: the second pair holds one 128-column block; 33 rows past a tile
    # of 16*r; 5 steps a split, one more in the last
    n_in, n_out, rows = 704, 384, 16 * r + 33
    n_in = n_in // 128 * 128
    print(f"wide k={k} cb={cb} r={r}", flush=True)
    lin, (tr, suh, svh, _) = make_layer(4000 + 10 * k + cb, n_in, n_out, k, cb)
    x = synth.activations(5, k, rows, n_in)
    ref = oracle.forward(x[-34:], tr, suh, svh, k, cb, mode=1)
    force(monkeypatch, r, 2)
    check(run(lin, x).cpu().numpy()[-34:], ref, TOL_MODE1_REL, TOL_MODE1_ULP, "2 splits")
    force(monkeypatch, r, 1)
    y = run(lin, x).cpu().numpy()
    check(y[-34:], ref, TOL_MODE1_REL, TOL_MODE1_ULP, "1 split")
    monkeypatch.setenv("EXL3_WIDE", "0")
    other = run(lin, x).cpu().numpy()
    assert np.array_equal(y.view(np.uint16), other.view(np.uint16))


@pytest.mark.parametrize("rows", [17, 64, 65, 127, 129, 256, 257, 513])
@pytest.mark.parametrize("n_in, n_out, splits", [(128, 128, 1), (256, 256, 1), (1152, 640, 3)])
def test_rows_and_widths(monkeypatch, rows, n_in, n_out, splits):
    for r in (4, 8, 16):
        print(f"wide rows={rows} {n_in}x{n_out} r={r}", flush=True)
        lin, (tr, suh, svh, _) = make_layer(5000 + rows, n_in, n_out, 4, 0)
        x = synth.activations(6, rows, rows, n_in)
        force(monkeypatch, r, splits)
        y = run(lin, x).cpu().numpy()
        pick = sorted({0, 1, 15, 16, rows // 2, rows - 1})
        check(y[pick], oracle.forward(x[pick], tr, suh, svh, 4, 0, mode=1), TOL_MODE1_REL,
              TOL_MODE1_ULP, f"r{r}")


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("splits", [1, 3])
def test_dtypes_bias_and_group(monkeypatch, dtype, bias, splits):
    """Every output form, through a group whose members end in a half pair: equal
    to the members alone bit for bit (the same K-ranges)."""
    import mlxl3_amd
    import torch

    made = [make_layer(6000 + i, 512, n_out, 3, 1, bias=bias) for i, n_out in enumerate((384, 128, 256))]
    x = synth.activations(7, 1, 100, 512)
    t = torch.from_numpy(x).cuda().to({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dtype])
    force(monkeypatch, 8, splits)
    ys = mlxl3_amd.Exl3Group([m[0] for m in made]).forward(t)
    for (lin, (tr, suh, svh, b)), y in zip(made, ys):
        alone = lin.forward(t)
        assert torch.equal(alone.view(torch.int16 if alone.element_size() == 2 else torch.int32),
                           y.view(torch.int16 if y.element_size() == 2 else torch.int32))
        xr = t.to(torch.float16).cpu().numpy()
        want = oracle.forward(xr, tr, suh, svh, 3, 1, mode=1).astype(np.float64)
        got = y.float().cpu().numpy().astype(np.float64)
        if dtype == "bf16":
            want = (bf16_bits(want).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        if bias:
            want = want + b.astype(np.float64)
        # 2 ulp of the f16 result, one more of the last rounded format
        tol = 3 * ulp_of(np.abs(want).max(), dtype == "bf16")
        assert np.abs(got - want).max() <= tol, (dtype, bias, np.abs(got - want).max(), tol)


def test_workspace_between_the_two_needs(monkeypatch):
    """A workspace that holds the producer/consumer QMM but not the wide kernel's
    partials still serves the call, one below is refused as before."""
    import mlxl3_amd
    import torch

    lin, (tr, suh, svh, _) = make_layer(7000, 2048, 256, 4, 0)
    x = synth.activations(8, 1, 200, 2048)
    force(monkeypatch, 8, 8)
    full = lin.workspace_bytes(200)
    monkeypatch.setenv("EXL3_WIDE", "0")
    least = lin.workspace_bytes(200)
    assert least < full
    force(monkeypatch, 8, 8)
    ref = oracle.forward(x, tr, suh, svh, 4, 0, mode=1)
    t = torch.from_numpy(x).cuda()
    for size in (least, full):
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
        y = lin.forward(t, workspace=ws).cpu().numpy()
        check(y, ref, TOL_MODE1_REL, TOL_MODE1_ULP, f"workspace {size}")
    with pytest.raises(mlxl3_amd.Exl3Error, match="workspace too small"):
        lin.forward(t, workspace=torch.zeros(least - 256, dtype=torch.uint8, device="cuda"))
