"""Which launch a QMM call gets, seen from the host: the workspace a call asks for
holds the split-K partials of the launch that it will make (no GPU needed: none of
these calls reaches the device)."""

import ctypes

import pytest

import mlxl3_amd

FAKE = 0x1000  # never dereferenced by create
COUNTERS = 64 * 1024


@pytest.fixture()
def linear():
    lib = mlxl3_amd.load_library()
    made = []

    def make(n_in, n_out, k=4, trellis=FAKE):
        h = ctypes.c_void_p()
        assert lib.exl3_linear_create(trellis, n_in, n_out, k, 0, FAKE, FAKE, None, ctypes.byref(h)) == 0
        made.append(h)
        return lambda rows: int(lib.exl3_linear_workspace_bytes(h, rows))

    yield make
    for h in made:
        lib.exl3_linear_destroy(h)


def xhat_bytes(rows, n_in):
    return COUNTERS + (2 * rows * n_in + 255) // 256 * 256


# ---------------------------------------------------------------------------
# EXL3_QMM_MB and EXL3_QMM_SPLITS fix the producer/consumer launch
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("env", [{"EXL3_QMM_SPLITS": "2"}, {"EXL3_QMM_MB": "1"},
                                 {"EXL3_QMM_MB": "4", "EXL3_QMM_SPLITS": "3"}])
@pytest.mark.parametrize("n_in, n_out, rows", [(14336, 4096, 300), (14336, 4096, 128), (27648, 5120, 200)])
def test_pinned_qmm_shape_keeps_its_kernel(monkeypatch, linear, env, n_in, n_out, rows):
    need = linear(n_in, n_out)
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    got = need(rows)
    monkeypatch.setenv("EXL3_WIDE", "0")
    assert got == need(rows)
    # EXL3_WIDE=1 still forces the QMM in registers
    monkeypatch.setenv("EXL3_WIDE", "1")
    monkeypatch.setenv("EXL3_WIDE_TILE", "1")
    monkeypatch.setenv("EXL3_WIDE_SPLITS", "2")
    assert need(rows) >= xhat_bytes(rows, n_in) + 4 * 2 * rows * n_out
