"""The decode-in-registers QMM (tiles of 64 rows x 128 columns, 128 x 256 or 256 x
256) at the edges of its tiles, forced on with EXL3_WIDE=1 and its shape with
EXL3_WIDE_TILE / EXL3_WIDE_SPLITS, against the CPU oracle (tolerances of test_gpu_linear.py) and
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
    monkeypatch.setenv("EXL3_WIDE_TILE", str({4: 0, 8: 1, 16: 2}[r]))
    monkeypatch.setenv("EXL3_WIDE_SPLITS", str(splits))
    monkeypatch.setenv("EXL3_QMM_SPLITS", "1")  # read only where EXL3_WIDE=0


@pytest.mark.parametrize("k", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
@pytest.mark.parametrize("r", [4, 8, 16])
def test_every_k_and_codebook(monkeypatch, k, cb, r):
    # 384 columns: the second pair holds one 128-column block; 33 rows past a tile
    # of 16*r; 20 steps in splits of 6, 7 and 7
    n_in, n_out, rows = 1280, 384, 16 * r + 33
    print(f"wide k={k} cb={cb} r={r}", flush=True)
    lin, (tr, suh, svh, _) = make_layer(4000 + 10 * k + cb, n_in, n_out, k, cb)
    x = synth.activations(5, k, rows, n_in)
    ref = oracle.forward(x[-34:], tr, suh, svh, k, cb, mode=1)
    force(monkeypatch, r, 3)
    check(run(lin, x).cpu().numpy()[-34:], ref, TOL_MODE1_REL, TOL_MODE1_ULP, "3 splits")
    force(monkeypatch, r, 1)
    y = run(lin, x).cpu().numpy()
    check(y[-34:], ref, TOL_MODE1_REL, TOL_MODE1_ULP, "1 split")
    monkeypatch.setenv("EXL3_WIDE", "0")
    other = run(lin, x).cpu().numpy()
    assert np.array_equal(y.view(np.uint16), other.view(np.uint16))


@pytest.mark.parametrize("rows", [17, 64, 65, 127, 129, 256, 257, 513])
@pytest.mark.parametrize("n_in, n_out, splits", [(128, 128, 1), (256, 256, 1), (1280, 640, 3)])
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
    to the members alone bit for bit (the same K-ranges: 14 steps, 3 splits of 4, 5
    and 5)."""
    import mlxl3_amd
    import torch

    made = [make_layer(6000 + i, 896, n_out, 3, 1, bias=bias) for i, n_out in enumerate((384, 128, 256))]
    x = synth.activations(7, 1, 100, 896)
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


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("r", [4, 8, 16])
@pytest.mark.parametrize("k,cb", [(3, 1), (4, 0), (5, 2), (8, 0)])
def test_repeat_calls_bit_identical(monkeypatch, k, cb, r, splits):
    """The loop keeps the wait states between its inline-assembly decode and the MFMAs,
    and its counted waits for the copies, by hand: an error of that kind shows as
    outputs that change between calls.  30 calls, two inputs in turn on one workspace
    (what a call reads too early is the other input's), each equal to its input's first
    result bit for bit."""
    import torch

    print(f"wide repeat k={k} cb={cb} r={r} splits={splits}", flush=True)
    lin, _ = make_layer(7100 + k, 2816, 1152, k, cb)  # 44 steps: 14, 15, 15
    force(monkeypatch, r, splits)
    rows = 32 * r + 5
    xs = [torch.from_numpy(synth.activations(70 + i, rows, rows, 2816)).cuda() for i in range(2)]
    ws = torch.zeros(lin.workspace_bytes(rows), dtype=torch.uint8, device="cuda")
    want = [lin.forward(x, workspace=ws).clone() for x in xs]
    assert not torch.equal(want[0], want[1])
    outs = [lin.forward(xs[i % 2], workspace=ws) for i in range(30)]
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y.view(torch.int16), want[i % 2].view(torch.int16)), i


def test_unaligned_trellis_takes_the_producer_consumer_kernel(monkeypatch):
    """The copies of the wide loop are 16 bytes wide: a trellis 8 bytes past that
    alignment runs the other kernel, also where the wide one is forced, and gives its
    bits."""
    import mlxl3_amd
    import torch

    lin, (tr, suh, svh, _) = make_layer(7200, 2048, 384, 4, 0)
    buf = torch.empty(lin.trellis.numel() + 4, dtype=torch.int16, device="cuda")[4:]
    off = buf.view(lin.trellis.shape).copy_(lin.trellis)
    assert off.data_ptr() % 16 == 8
    moved = mlxl3_amd.Exl3Linear(off, lin.suh, lin.svh, None, 4, 0)
    x = synth.activations(71, 1, 150, 2048)
    monkeypatch.setenv("EXL3_QMM_SPLITS", "1")  # no partials, as the wide launch would have
    monkeypatch.setenv("EXL3_WIDE", "0")
    want, least = run(lin, x), lin.workspace_bytes(150)
    monkeypatch.setenv("EXL3_WIDE", "1")
    monkeypatch.setenv("EXL3_WIDE_TILE", "0")
    monkeypatch.setenv("EXL3_WIDE_SPLITS", "8")
    assert moved.workspace_bytes(150) == least < lin.workspace_bytes(150)
    y = run(moved, x)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    check(y.cpu().numpy(), oracle.forward(x, tr, suh, svh, 4, 0, mode=1), TOL_MODE1_REL, TOL_MODE1_ULP, "unaligned")


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


# ---------------------------------------------------------------------------
# the input prologue and the SwiGLU edge by MFMA (from 2048 waves of 16 x 128 on)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("rows", [2032, 2033, 2048])
@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("off", [0, 1])
def test_prologue_on_both_sides_of_the_rule(rows, dtype, off):
    """2032 rows x 2048 inputs are 127 * 16 waves (16 lanes per row), 2033 and 2048
    are 128 * 16 (MFMA), the first with one row in its last block; `off`: an input one
    element past its alignment (the scalar loads)."""
    import torch

    print(f"prologue rows={rows} {dtype} off={off}", flush=True)
    lin, (tr, suh, svh, _) = make_layer(8000, 2048, 128, 4, 0)
    x = synth.activations(9, 1, rows, 2048)
    t = torch.from_numpy(x).cuda().to({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dtype])
    buf = torch.empty(rows * 2048 + off, dtype=t.dtype, device="cuda")
    t = buf[off:].view(rows, 2048).copy_(t)
    pick = np.array([0, 1, 15, 16, 1000, rows - 2, rows - 1])
    y = lin.forward(t).float().cpu().numpy().astype(np.float64)[pick]
    want = oracle.forward(t[pick].half().cpu().numpy(), tr, suh, svh, 4, 0, mode=1).astype(np.float64)
    if dtype == "bf16":
        want = (bf16_bits(want).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    # 2 ulp of the f16 result, one more of the last rounded format
    assert np.abs(y - want).max() <= 3 * ulp_of(np.abs(want).max(), dtype == "bf16")


@pytest.mark.parametrize("n_in,hidden,rows", [(1024, 3584, 40), (1024, 3584, 300), (768, 4096, 700)])
def test_mlp_equals_its_parts_at_split_launches(n_in, hidden, rows):
    """Shapes whose launches split K under the default rules: the fused MLP, whose
    workspace leaves its down projection other room than the linear's own, still equals
    the group, the SwiGLU and the linear bit for bit."""
    import mlxl3_amd
    import torch
    import test_gpu_group as g

    _, parts, _ = g.mlp_case(n_in, hidden, 4, 0)
    x = torch.from_numpy(synth.activations(11, rows, rows, n_in)).cuda()
    down = parts[2]
    assert down.workspace_bytes(rows) > 65536 + 2 * rows * hidden + 255  # partials: it splits
    y, other = mlxl3_amd.Exl3Mlp(*parts).forward(x), g.unfused(parts, x)
    assert torch.equal(y.view(torch.int16), other.view(torch.int16))


@pytest.mark.parametrize("rows", [2032, 2033])
@pytest.mark.parametrize("off", [0, 1])
def test_swiglu_edge_on_both_sides_of_the_rule(rows, off):
    """The edge of 2048 hidden columns: the fused MLP against its own parts, with the
    down projection's input scales aligned and not, and against the oracle."""
    import mlxl3_amd
    import torch
    import test_gpu_group as g

    print(f"swiglu edge rows={rows} off={off}", flush=True)
    _, (gate, up, down), host = g.mlp_case(256, 2048, 3, 1)
    suh = torch.empty(2048 + off, dtype=torch.float16, device="cuda")[off:].copy_(down.suh)
    down = mlxl3_amd.Exl3Linear(down.trellis, suh, down.svh, None, 3, 1)
    x_np = synth.activations(10, 1, rows, 256)
    x = torch.from_numpy(x_np).cuda()
    y, other = mlxl3_amd.Exl3Mlp(gate, up, down).forward(x), g.unfused((gate, up, down), x)
    assert torch.equal(y.view(torch.int16), other.view(torch.int16))
    pick = [0, 17, rows - 1]
    g.check_tol(y.cpu().numpy()[pick], oracle.mlp_forward(x_np[pick], *host), "rows of the oracle")


# ---------------------------------------------------------------------------
# the expert QMMs for many rows per expert
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("cb", [0, 1, 2])
def test_moe_wide_every_k_and_codebook(monkeypatch, k, cb):
    """Experts whose rows fill one block, more than one and none, forced on."""
    import test_gpu_moe as m

    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    print(f"moe wide k={k} cb={cb}", flush=True)
    layer, x, _, _ = m.case(256, 128, 5, 2, 260, k, 700 + k)
    sel, sc = synth.moe_routes(701 + k, 530, 260, 3, 2)  # ~173 rows each, experts 3 and 4 idle
    moe = m.make_moe(layer, 2, k, cb)
    pick = np.arange(0, 260, 7)
    ref = oracle.moe_forward(x[pick], sel[pick], sc[pick], *layer, k, cb)
    m.check(m.run(moe, x, sel, sc)[pick], ref, f"moe wide k={k} cb={cb}")


@pytest.mark.parametrize("rows", [1, 8, 17, 80, 81, 161])
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("score", ["float16", "float32"])
def test_moe_wide_rows(monkeypatch, rows, gelu, score):
    """One expert takes every row (its block at and past its row blocks' edges),
    with f16 and f32 scores, SiLU and GELU, and an id outside the bank."""
    import test_gpu_moe as m

    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    monkeypatch.setenv("EXL3_MOE_GROUPED", "1")  # up to 64 slots too
    print(f"moe wide rows={rows} gelu={gelu} {score}", flush=True)
    layer, x, _, sc = m.case(384, 256, 3, 2, rows, 3, 720)
    sel = np.tile(np.array([[1, 2]], np.uint32), (rows, 1))
    sel[rows // 2:, 1] = 0
    sel[0, 1] = 9  # outside: adds nothing
    sc = sc.astype(score)
    import torch
    import mlxl3_amd

    dev = lambda a: torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()
    moe = mlxl3_amd.Exl3SwitchGlu(*(dev(t) for t in layer), top_k=2, k=3, cb=0,
                                  activation="gelu" if gelu else "silu",
                                  logical_hidden=200 if gelu else None)
    y = moe.forward(dev(x), torch.from_numpy(sel.astype(np.int32)).cuda(), dev(sc)).cpu().numpy()
    monkeypatch.setenv("EXL3_MOE_WIDE", "0")
    other = moe.forward(dev(x), torch.from_numpy(sel.astype(np.int32)).cuda(), dev(sc)).cpu().numpy()
    # the grouped kernel is held to the oracle by test_gpu_moe.py; both sum the same
    # products in the same order and differ by the epilogues' f32 sums
    m.check(y, other, "vs the 64-row blocks")
    pick = sorted({min(1, rows - 1), rows // 2, rows - 1} - ({0} if rows > 1 else set()))
    pick = [r for r in pick if (sel[r] < 3).all()]
    if pick:
        ref = oracle.moe_forward(x[pick], sel[pick], sc[pick].astype(score), *layer, 3, 0,
                                 **(dict(activation="gelu", logical_hidden=200) if gelu else {}))
        m.check(y[pick], ref, "rows of the oracle")


@pytest.mark.parametrize("dtype", ["float16", "bfloat16", "float32"])
def test_moe_wide_unaligned_input(monkeypatch, dtype):
    """An input one element past its alignment takes the gather's scalar loads and
    gives the aligned input's bits."""
    import test_gpu_moe as m
    import torch

    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    print(f"moe wide unaligned {dtype}", flush=True)
    layer, x, sel, sc = m.case(256, 128, 5, 2, 260, 3, 740)
    moe = m.make_moe(layer, 2, 3, 0)
    t = torch.from_numpy(x).cuda().to(getattr(torch, dtype))
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view(t.shape).copy_(t)
    sel, sc = torch.from_numpy(sel.astype(np.int32)).cuda(), torch.from_numpy(sc).cuda()
    assert buf.data_ptr() % 16 != 0
    a, b = moe.forward(t, sel, sc), moe.forward(buf, sel, sc)
    assert torch.equal(a.float(), b.float())


@pytest.mark.parametrize("part", [0, 3])
def test_moe_unaligned_trellis_keeps_the_64_row_blocks(monkeypatch, part):
    """A gate/up or down bank 8 bytes past its 16-byte alignment runs the 64-row blocks,
    also where the wide ones are forced, and gives their bits."""
    import test_gpu_moe as m
    import mlxl3_amd
    import torch

    layer, x, sel, sc = m.case(256, 128, 5, 2, 260, 3, 750)
    bank = [m.dev(a) for a in layer]
    args = (m.dev(x), m.dev(sel), m.dev(sc))
    monkeypatch.setenv("EXL3_MOE_WIDE", "0")
    want = mlxl3_amd.Exl3SwitchGlu(*bank, top_k=2, k=3, cb=0).forward(*args)
    buf = torch.empty(bank[part].numel() + 4, dtype=torch.int16, device="cuda")[4:]
    bank[part] = buf.view(bank[part].shape).copy_(bank[part])
    assert bank[part].data_ptr() % 16 == 8
    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    y = mlxl3_amd.Exl3SwitchGlu(*bank, top_k=2, k=3, cb=0).forward(*args)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("k,cb,gelu", [(3, 0, False), (4, 1, True), (6, 2, False), (8, 0, True)])
def test_moe_wide_repeat_calls_bit_identical(monkeypatch, k, cb, gelu):
    """test_repeat_calls_bit_identical for the expert form: 20 calls, two inputs and
    routings in turn on one operator."""
    import test_gpu_moe as m
    import torch

    print(f"moe wide repeat k={k} cb={cb} gelu={gelu}", flush=True)
    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    layer, _, _, _ = m.case(1152, 640, 6, 2, 4, k, 780)
    moe = m.make_moe(layer, 2, k, cb, activation="gelu" if gelu else "silu")
    ins = []
    for i in range(2):
        sel = routes_of([161, 37 + 3 * i, 160, 16, 200 - 3 * i, 2], 2, 781 + i)
        _, sc = synth.moe_routes(783, i, sel.shape[0], 6, 2)
        ins.append((m.dev(synth.activations(782, i, sel.shape[0], 1152)), m.dev(sel), m.dev(sc)))
    want = [moe.forward(*a).clone() for a in ins]
    assert not torch.equal(want[0], want[1])
    outs = [moe.forward(*ins[i % 2]) for i in range(20)]
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y.view(torch.int16), want[i % 2].view(torch.int16)), i


def routes_of(counts, top_k, seed, idle=0):
    """selected [rows, top_k] that gives expert e counts[e] slots, in random order;
    the ids from len(counts) on are `idle` slots outside the bank."""
    ids = np.concatenate([np.repeat(np.arange(len(counts)), counts), np.full(idle, len(counts))])
    assert ids.size % top_k == 0
    np.random.default_rng(seed).shuffle(ids)
    return ids.reshape(-1, top_k).astype(np.uint32)


# 16 experts, hidden 1024 (16 workgroups a block), mean rows per expert above the 64
# (GELU: 112) from which the host lets the device choose; wide: blocks of 160 rows are at
# least 2 (K = 3, 4 with SiLU: 1.9, K = 5, 6: 1.7) times fewer than blocks of 64, and, for K
# <= 4, their workgroups are not 513 to 639
CHOICES = [
    # counts, k, activation, idle slots, wide
    ([80] * 16, 1, "silu", 0, True),                  # 32 against 16 blocks
    ([80] * 16, 4, "silu", 0, True),
    ([80] * 15 + [64], 4, "silu", 0, True),           # 31 against 16: 1.94
    ([80] * 14 + [64, 64], 4, "silu", 0, False),      # 30 against 16: 1.88
    ([80] * 15 + [64], 2, "silu", 0, False),          # 1.94 < 2
    ([160] * 8 + [64] * 8, 3, "silu", 0, True),       # 32 against 16
    ([161] * 8 + [64] * 8, 3, "silu", 8, False),      # 32 against 24
    ([30, 130] * 8, 4, "silu", 0, True),              # 1 + 3 against 1 + 1
    ([30, 120] * 8, 4, "silu", 0, False),             # 1 + 2 against 1 + 1
    ([30, 120] * 8, 5, "silu", 0, False),             # 1.5 < 1.7
    ([1, 0, 1279] + [0] * 13, 3, "silu", 0, True),    # 21 against 9, idle experts
    ([1, 0, 1279] + [0] * 13, 6, "silu", 16, True),   # ids outside the bank
    ([60] * 12 + [200] * 4, 6, "silu", 0, False),     # 28 against 20: 1.4
    ([320] * 16, 4, "silu", 0, True),                 # 80 against 32: 512 workgroups
    ([320] * 15 + [322], 4, "silu", 0, False),        # 81 against 33: 528
    ([322] * 15 + [320], 5, "silu", 0, True),         # 95 against 47
    ([322] * 7 + [320] * 9, 4, "silu", 0, False),     # 87 against 39: 624
    ([322] * 8 + [320] * 8, 4, "silu", 0, True),      # 88 against 40: 640
    ([120] * 16, 4, "gelu", 0, False),                # GELU banks of K <= 4 never
    ([120] * 16, 5, "gelu", 0, True),
    ([128] * 15 + [64], 6, "gelu", 0, False),         # 31 against 16 < 2
    ([30, 130] * 8, 8, "silu", 0, None),              # K = 8: always, nothing to choose
]


@pytest.mark.parametrize("case_id", range(len(CHOICES)))
def test_moe_block_choice_follows_the_routes(monkeypatch, case_id):
    """Whether the experts run in blocks of 160 rows is decided from the blocks that the
    call's routes really cut, on the device: one of the two kernels gets every block,
    the other none.  The output matches the oracle and both forced forms either way."""
    import test_gpu_moe as m
    import torch

    counts, k, act, idle, wide = CHOICES[case_id]
    print(f"moe choice {case_id} k={k} {act}", flush=True)
    layer, _, _, _ = m.case(1024, 1024, 16, 2, 4, k, 760)
    sel = routes_of(counts, 2, 761 + case_id, idle)
    rows = sel.shape[0]
    x = synth.activations(762, case_id, rows, 1024)
    _, sc = synth.moe_routes(763, 1, rows, 16, 2)
    moe = m.make_moe(layer, 2, k, 0, activation=act)
    y = m.run(moe, x, sel, sc)
    narrow_blocks, routed, wide_blocks = moe._ws.buf[65536:65536 + 12].view(torch.int32).tolist()
    b64 = sum(-(-c // 64) for c in counts)
    bw = sum(-(-c // 160) for c in counts)
    assert routed == sum(counts)
    if wide is not None:
        assert (narrow_blocks, wide_blocks) == ((0, bw) if wide else (b64, 0))
    pick = np.arange(rows)[(sel < 16).all(1)][case_id % 5::rows // 6]
    ref = oracle.moe_forward(x[pick], sel[pick], sc[pick], *layer, k, 0, activation=act)
    m.check(y[pick], ref, f"choice {case_id}")
    # two outputs that may each be TOL away from the oracle are at most twice that apart
    rms = np.sqrt(np.mean(y.astype(np.float64) ** 2))
    for forced in "01":
        monkeypatch.setenv("EXL3_MOE_WIDE", forced)
        gap = m.run(moe, x, sel, sc).astype(np.float64) - y
        assert np.sqrt(np.mean(gap ** 2)) <= 2 * m.TOL_REL * rms, (case_id, forced)
        assert np.abs(gap).max() <= 2 * m.TOL_RMS * rms, (case_id, forced)


@pytest.mark.parametrize("k,hidden,may", [(4, 896, False), (4, 1024, True), (6, 512, False), (6, 640, True)])
def test_moe_small_launches_keep_the_64_row_blocks(monkeypatch, k, hidden, may):
    """Less than half a round of gate/up workgroups (16 experts of one block, hidden / 64 a
    block, 512 a round; at K = 5, 6 0.3 of one) stays with 64-row blocks whatever the routes."""
    import test_gpu_moe as m
    import torch

    layer, _, _, _ = m.case(1024, hidden, 16, 2, 4, k, 790)
    sel = routes_of([80] * 16, 2, 791)
    x = synth.activations(792, 1, sel.shape[0], 1024)
    _, sc = synth.moe_routes(793, 1, sel.shape[0], 16, 2)
    moe = m.make_moe(layer, 2, k, 0)
    m.run(moe, x, sel, sc)
    assert moe._ws.buf[65536:65536 + 12].view(torch.int32).tolist() == ([0, 1280, 16] if may else [32, 1280, 0])


def test_moe_choice_alternates_on_one_workspace():
    """Even and uneven routes in turn on one operator (one workspace): each call equals
    its first result bit for bit, so neither kernel reads what the other left."""
    import test_gpu_moe as m
    import torch

    layer, _, _, _ = m.case(1024, 1024, 16, 2, 4, 4, 770)
    moe = m.make_moe(layer, 2, 4, 0)
    ins = []
    for i, counts in enumerate(([80] * 16, [30, 130, 30, 90] * 4, [30, 120] * 8)):
        sel = routes_of(counts, 2, 771 + i)
        x = synth.activations(772, i, sel.shape[0], 1024)
        _, sc = synth.moe_routes(773, i, sel.shape[0], 16, 2)
        ins.append((m.dev(x), m.dev(sel), m.dev(sc)))
    want = [moe.forward(*a).clone() for a in ins]
    outs = [moe.forward(*ins[i % 3]) for i in range(30)]
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y.view(torch.int16), want[i % 3].view(torch.int16)), i


def test_moe_choice_under_capture():
    """The choice is made by each replay: one captured call, its routes rewritten between
    replays so that either kernel has the blocks, equals the eager call every time."""
    import test_gpu_moe as m
    import torch

    layer, _, _, _ = m.case(1024, 1024, 16, 2, 4, 4, 770)
    moe = m.make_moe(layer, 2, 4, 0)
    routes = [m.dev(routes_of(c, 2, 775 + i)).to(torch.int32) for i, c in enumerate(([80] * 16, [30, 130, 60, 100] * 4))]
    rows = routes[0].shape[0]
    x = m.dev(synth.activations(776, 1, rows, 1024))
    sc = m.dev(synth.moe_routes(777, 1, rows, 16, 2)[1])
    want = [moe.forward(x, sel, sc).clone() for sel in routes]
    assert not torch.equal(want[0], want[1])
    sel = routes[0].clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        moe.forward(x, sel, sc)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = moe.forward(x, sel, sc)
    for i in (0, 1, 1, 0, 1, 0):
        sel.copy_(routes[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want[i].view(torch.int16)), i
        wide = int(moe._ws.buf[65536 + 8:65536 + 12].view(torch.int32))
        assert (wide > 0) == (i == 0)


@pytest.mark.parametrize("experts", [3840, 4096])
def test_moe_wide_largest_bank(monkeypatch, experts):
    """The most experts a bank may have: the route launch's histogram next to its gather
    rows is the largest LDS request there is (66 KB)."""
    import test_gpu_moe as m
    import torch

    print(f"moe wide {experts} experts", flush=True)
    g = torch.Generator().manual_seed(experts)
    t = lambda *s: torch.randint(-32768, 32768, s, dtype=torch.int16, generator=g).cuda()
    f = lambda *s: ((torch.rand(*s, generator=g) + 0.5) / 12).half().cuda()
    import mlxl3_amd

    moe = mlxl3_amd.Exl3SwitchGlu(t(8, 2 * experts * 8, 16), f(experts, 2, 128), f(experts, 2, 128),
                                  t(8, experts * 8, 16), f(experts, 128), f(experts, 128), top_k=2, k=1, cb=0)
    x = torch.randn(60, 128, generator=g).half().cuda()
    sel = torch.randint(0, experts, (60, 2), generator=g).int().cuda()
    sc = torch.rand(60, 2, generator=g).half().cuda()
    monkeypatch.setenv("EXL3_MOE_WIDE", "1")
    y = moe.forward(x, sel, sc).cpu().numpy()
    monkeypatch.setenv("EXL3_MOE_WIDE", "0")
    m.check(y, moe.forward(x, sel, sc).cpu().numpy(), "vs the 64-row blocks")
