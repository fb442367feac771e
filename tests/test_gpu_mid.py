"""The barrier-free mid-M kernel (csrc/kernels/mid_kernel.h): every instantiated launch shape against the float64
oracle at the edges of its tiles, the same call on the general kernels, and the rule that picks it."""
import numpy as np
import pytest
import torch

from _util import parity_err, random_problem, run_product

pytestmark = pytest.mark.gpu
TOL = 1e-2  # the repository's bar: the 16-bit output rounding and the weights' own
SHAPES = [(1, 8), (2, 8), (4, 4), (4, 8)]


def _last_launch(pkg):
    return (pkg._lib.lib.woq_last_launch() or b"").decode()


def _instantiated(rt, ns, group):
    return group == 0 or ns < 4 or rt < (3 if group == 64 else 4)


@pytest.mark.parametrize("rt", [1, 2, 3, 4])
@pytest.mark.parametrize("bits,group,dtype", [(4, 128, "bf16"), (4, 64, "fp16"), (4, 0, "bf16"), (8, 0, "fp16"),
                                              (8, 0, "bf16"), (4, 128, "fp16"), (4, 64, "bf16")])
def test_mid_every_shape(pkg, oracle, dev, woq_env, rt, bits, group, dtype):
    """Strips that do not divide by a workgroup's, one row past a row tile / a whole tile / a second tile of rows, tile
    rows of K that leave some wavefronts one more than others (or none), K split with a last slice that is shorter;
    zeros, bias and smoothing on and off; the same bits on every call."""
    if rt == 1 and bits == 8:
        pytest.skip("one row tile is built for int4 only")
    tk = 128 if bits == 4 else 64
    for ns, waves in SHAPES:
        if not _instantiated(rt, ns, group):
            continue
        for M, tiles, N, splits in [(16 * rt - 15, 9, 16 * 9, 1), (16 * rt, 21, 16 * 11, 2), (16 * rt + 1, 13, 16 * 8, 1),
                                    (32 * rt + 7, 37, 16 * 3, 4)]:
            woq_env(WOQ_MID_SHAPE="%d,%d,%d,%d" % (rt, ns, waves, splits))
            full = splits == 2
            p = random_problem(oracle, M, tk * tiles, N, bits, group, dtype, zero=group != 0 and M % 2 == 1, bias=full,
                               pqs=full, seed=M + tiles + ns)
            out = run_product(pkg, oracle, dev, p, 2)  # (the tiled regime smooths in a pass of its own)
            assert "mid rt=%d ns=%d waves=%d splits=%d" % (rt, ns, waves, splits) in _last_launch(pkg), _last_launch(pkg)
            assert parity_err(oracle, out, p) < TOL, (ns, waves, M, tiles, N, splits)
            again = run_product(pkg, oracle, dev, p, 2)
            assert (again.view(np.uint32) == out.view(np.uint32)).all()


@pytest.mark.parametrize("bits,group", [(4, 128), (4, 64), (4, 0), (8, 0)])
def test_mid_against_the_general_path(pkg, oracle, dev, woq_env, bits, group):
    """One-hot activations return single weights times their scale, on this kernel and on the one it replaces; infinities
    and NaN in one row stay in that row."""
    K, N, M = 2048, 1040, 40
    p = random_problem(oracle, M, K, N, bits, group, "bf16", zero=group != 0, seed=group + bits)
    p["act"] = np.zeros((M, K), np.float32)
    for r in range(M):
        p["act"][r, (53 * r + 7) % K] = 1.0
    p["act"][3, 100] = np.inf
    p["act"][5, 200] = np.nan
    outs = []
    for shape in (None, "0"):
        woq_env(WOQ_MID_SHAPE=shape)
        outs.append(run_product(pkg, oracle, dev, p, 0))
        assert ("mid" in _last_launch(pkg)) == (shape is None), _last_launch(pkg)
    w = oracle.dequantize(p["q"], p["scales"], p["zeros"], group, "bf16")
    for out in outs:
        for r in range(M):
            if r in (3, 5):
                assert not np.isfinite(out[r]).any()
                continue
            row = w[(53 * r + 7) % K]
            # one output rounding (2^-8) on top of the weight's own in `w`
            assert (np.abs(out[r] - row) <= np.abs(row) * 2.0 ** -7 + 2.5e-7).all(), r


def _with_infinities(oracle, p):
    """Plants infinities and a NaN in a problem's activations; returns {row: what that row is}, other rows stay finite."""
    K = p["K"]
    rows = {3: {100: np.inf}, 9: {K - 1: -np.inf}, 17: {5: np.inf, K - 70: np.inf}, 30: {64: np.nan}}
    w = oracle.dequantize(p["q"], p["scales"], p["zeros"], p["group"], p["dtype"]).astype(np.float64)
    want = {}
    for r, planted in rows.items():
        for k, v in planted.items():
            p["act"][r, k] = v
        with np.errstate(invalid="ignore"):
            want[r] = sum(v * w[k] for k, v in planted.items())  # a zero weight makes NaN of an infinity
    return want


@pytest.mark.parametrize("bits,group,dtype", [(4, 128, "bf16"), (4, 64, "fp16"), (4, 0, "fp16"), (8, 0, "bf16"), (8, 0, "fp16")])
@pytest.mark.parametrize("env", [dict(WOQ_MID_SHAPE="2,1,8,1"), dict(WOQ_MID_SHAPE="3,2,8,2"), dict(WOQ_MID_SHAPE="2,4,4,1"),
                                 dict(WOQ_MID_SHAPE="0", WOQ_GEMM_KERNEL="skinny"),
                                 dict(WOQ_MID_SHAPE="0", WOQ_GEMM_KERNEL="skinny", WOQ_GEMM_SPLITS="3")])
def test_infinite_activations_keep_their_sign(pkg, oracle, dev, woq_env, bits, group, dtype, env):
    """A row with an infinite activation is an infinity of the weight's sign in every column (NaN where the weight is
    zero or two infinities disagree), as on the kernel that multiplies scaled weights; the other rows keep their bits."""
    M, K, N = 43, 1280, 176
    woq_env(**env)
    p = random_problem(oracle, M, K, N, bits, group, dtype, zero=group == 128, seed=bits + group)
    clean = run_product(pkg, oracle, dev, p, 2)
    want = _with_infinities(oracle, p)
    out = run_product(pkg, oracle, dev, p, 2)
    assert ("mid" if env["WOQ_MID_SHAPE"] != "0" else "skinny") in _last_launch(pkg), _last_launch(pkg)
    for r in range(M):
        if r in want:
            np.testing.assert_array_equal(out[r], want[r].astype(np.float32))
        else:
            assert (out[r].view(np.uint32) == clean[r].view(np.uint32)).all(), r


@pytest.mark.parametrize("bits,group,activation", [(4, 0, "identity"), (8, 0, "swiglu"), (4, 128, "swiglu")])
def test_infinite_activations_of_an_expert(pkg, oracle, dev, woq_env, bits, group, activation):
    """The same for grouped problems on the deferred-scale kernel, gated epilogue included: what the exact-dequantize
    kernel returns for that row."""
    from _util import preprocess, to_dev
    F = pkg.functional
    K, N, counts = 640, 288, [40, 0, 70]
    probs = [random_problem(oracle, 8, K, N, bits, group, "fp16", seed=e) for e in range(3)]
    w = torch.stack([preprocess(pkg, oracle, p["q"], bits, torch.float16) for p in probs]).to(dev)
    sc = torch.stack([to_dev(p["scales"], "fp16", dev) for p in probs])
    act = torch.randn(sum(counts), K, generator=torch.Generator().manual_seed(1)).half()
    act[5, 9], act[60, K - 1], act[108, 300] = float("inf"), float("-inf"), float("nan")
    rows = torch.tensor(np.cumsum(counts), dtype=torch.int64, device=dev)
    outs = {}
    for kernel in ("exact", "skinny"):
        woq_env(WOQ_GEMM_KERNEL=kernel)
        outs[kernel] = F.woq_grouped_matmul_raw(act.to(dev), w, sc, None, None, rows, n=N, k=K, group_size=group,
                                                quant_algo=F.INT8_WEIGHT if bits == 8 else 0, activation=activation, regime=2)
        torch.cuda.synchronize()
        assert kernel in _last_launch(pkg), _last_launch(pkg)
    exact, got = outs["exact"].float().cpu().numpy(), outs["skinny"].float().cpu().numpy()
    for r in (5, 60, 108):
        assert not np.isfinite(exact[r]).any()
        np.testing.assert_array_equal(got[r], exact[r])
    rest = [r for r in range(sum(counts)) if r not in (5, 60, 108)]
    assert np.isfinite(got[rest]).all()
    assert np.abs(got[rest] - exact[rest]).max() < TOL * np.abs(exact[rest]).max()


def test_mid_rule(pkg, oracle, dev, woq_env):
    """Taken on narrow matrices from 17 rows on when nothing is forced; with one row tile where the multi-row kernel
    declines; not for more than 160 rows, flexible groups, int8 with group scales, a K that is no multiple of the weight
    tile, a smoothing vector that the streaming regime would apply itself, or a regime the caller named."""
    woq_env(WOQ_MID_SHAPE=None)
    run = lambda M, K, N, bits, group, regime=0: (run_product(
        pkg, oracle, dev, random_problem(oracle, M, K, N, bits, group, "bf16", seed=M), regime), _last_launch(pkg))[1]
    for M in (17, 33, 48, 64, 65, 160):
        assert "mid" in run(M, 4096, 1024, 4, 128), M
    assert "mid" in run(48, 4096, 1024, 8, 0)
    assert "mid rt=1" in run(16, 2048, 8208, 4, 128) and "mid rt=1" in run(8, 2048, 1024, 4, 0)
    assert "mid rt=1 ns=4 waves=8 splits=4" in run(12, 8192, 272, 4, 64)
    for args in [(16, 4096, 1024, 4, 128), (11, 2048, 8208, 4, 128), (16, 2048, 1024, 8, 0), (161, 4096, 1024, 4, 128), (48, 4096, 1024, 4, 256), (48, 4096, 1024, 8, 128),
                 (48, 2112, 1024, 4, 64)]:
        assert "mid" not in run(*args), args
    for regime in (1, 2):
        assert "mid" not in run(48, 4096, 1024, 4, 128, regime)


def test_mid_needs_aligned_activations(pkg, oracle, dev, woq_env):
    """Activations that start 8 bytes into an allocation run on the kernel that took them before, with the same result."""
    from _util import preprocess, to_dev
    F = pkg.functional
    woq_env(WOQ_MID_SHAPE=None)
    p = random_problem(oracle, 32, 4096, 1024, 4, 128, "bf16", seed=4)
    w, sc = preprocess(pkg, oracle, p["q"], 4).to(dev), to_dev(p["scales"], "bf16", dev)
    room = torch.empty(32 * 4096 + 8, dtype=torch.bfloat16, device=dev)
    for skip, mid in ((8, True), (4, False)):
        act = room[skip:skip + 32 * 4096].view(32, 4096)
        act.copy_(to_dev(p["act"], "bf16", dev))
        out = F.woq_matmul_raw(act, None, w, sc, None, None, n=1024, k=4096, group_size=128, quant_algo=0)
        torch.cuda.synchronize()
        assert ("mid" in _last_launch(pkg)) == mid, _last_launch(pkg)
        assert parity_err(oracle, out.float().cpu().numpy(), p) < TOL


def test_mid_and_the_tuned_table(pkg, oracle, dev, woq_env):
    """A table entry that leaves the choice to the heuristics leaves this kernel in it; one that names another does not."""
    F = pkg.functional
    woq_env(WOQ_MID_SHAPE=None)
    p = random_problem(oracle, 48, 4096, 1024, 4, 128, "bf16", seed=3)
    key = "1024 4096 0 128 %d 48 " % F._WOQ_DT[torch.bfloat16]
    try:
        for entry, mid in (("0 0 0 0 0 0 0 0 0", True), ("2 0 0 0 0 0 0 4 2", False)):
            F.import_tactics("woq-tactics 1\n" + key + entry + "\n")
            out = run_product(pkg, oracle, dev, p, 0)
            assert ("mid" in _last_launch(pkg)) == mid, _last_launch(pkg)
            assert parity_err(oracle, out, p) < TOL
    finally:
        F.clear_tactics()


def test_mid_split_only_with_room(pkg, oracle, dev, woq_env):
    """24 rows that need no workspace: four K slices when it holds their slabs, none when it is a byte too small or not
    there; all three against the oracle, the split one twice on a workspace full of garbage."""
    F = pkg.functional
    from _util import preprocess, to_dev
    M, K, N = 24, 4096, 2048
    p = random_problem(oracle, M, K, N, 4, 128, "bf16", zero=True, bias=True, seed=5)
    woq_env(WOQ_MID_SHAPE=None)
    w = preprocess(pkg, oracle, p["q"], 4).to(dev)
    ops = [to_dev(p[x], "bf16", dev) for x in ("act", "scales", "zeros", "bias")]
    slabs = 4 * M * N * 4
    for given, splits in ((slabs, 4), (slabs, 4), (slabs - 1, 1), (1, 1)):
        ws = torch.full((slabs,), 0x7F, dtype=torch.uint8, device=dev)[:given]
        out = F.woq_matmul_raw(ops[0], None, w, *ops[1:], n=N, k=K, group_size=128, quant_algo=F.ZERO | F.BIAS, workspace=ws)
        torch.cuda.synchronize()
        assert _last_launch(pkg).startswith("mid") and _last_launch(pkg).endswith("splits=%d" % splits), _last_launch(pkg)
        assert parity_err(oracle, out.float().cpu().numpy(), p) < TOL


@pytest.mark.parametrize("bits,group,dtype", [(4, 128, "bf16"), (4, 64, "bf16"), (4, 0, "fp16"), (8, 0, "bf16"), (8, 0, "fp16")])
@pytest.mark.parametrize("M", [161, 257, 512])
def test_mid_above_160_rows(pkg, oracle, dev, woq_env, M, bits, group, dtype):
    """Up to 512 rows on a narrow matrix the built-in rule takes it (several workgroups of rows share the weights; int8 in
    fp16 only where the kernel it replaces sums as long): the oracle's bar, and no larger an error against 64 bits than the
    other kernel's."""
    p = random_problem(oracle, M, 2048, 2048, bits, group, dtype, zero=group != 0, seed=M + group)
    run_product(pkg, oracle, dev, p)
    if (bits, dtype) != (8, "fp16") and group != 64:  # (those two: wherever the estimates put them)
        assert "mid" in _last_launch(pkg), _last_launch(pkg)
    woq_env(WOQ_MID_SHAPE="4,2,8,1")
    out = run_product(pkg, oracle, dev, p)
    assert parity_err(oracle, out, p) < TOL
    woq_env(WOQ_MID_SHAPE="0")
    other = run_product(pkg, oracle, dev, p)
    rows = (lambda t: np.repeat(t.astype(np.float64), 2048 // t.shape[0], 0)) if group else (lambda t: t.astype(np.float64)[None])
    exact = p["act"].astype(np.float64) @ (p["q"] * rows(p["scales"]) + (rows(p["zeros"]) if group else 0.0))
    error = lambda x: np.linalg.norm(x - exact) / np.linalg.norm(exact)
    assert error(out) <= 1.01 * error(other), (error(out), error(other), _last_launch(pkg))  # (330 000 roundings: 0.2 % of chance)
