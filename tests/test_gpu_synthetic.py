"""GPU H*psi on seeded synthetic middle-site problems against the oracle:
every tile configuration of the grouped GEMM (32x32, 64x64, 128x128 forced
through B2G_TILE, and the automatic choice), the scratch split into several
chunks, split-K partial tiles (B2G_KSPLIT), 4 and many right-hand sides, FP32
and split-BF16 three-term (every tile shape).  Blocks range from 1x1 up to
200x200, so edge tiles, K remainders and single-element blocks all occur.
Tolerances: FP64 1e-12 relative (2-norm), FP32 2e-6, split-BF16 1e-4."""
import ctypes as C
import os

import numpy as np
import pytest
import torch

from b2g import _lib as L
from b2g import synth
from b2g.effham import EffectiveHamiltonian
import b2g_oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.fixture(scope="module")
def problem():
    pb = synth.middle_site(n_orb=16, m=500, max_dim=200, seed=3)
    orc = O.Oracle(pb)
    rng = np.random.default_rng(9)
    xs = rng.standard_normal((4, pb.ket_len))
    ys = np.stack([orc.hpsi(x, nthreads=8) for x in xs])
    return pb, xs, ys


def cfg(tile):
    """Tile configuration of "T" or "TMxTN"."""
    t = [int(v) for v in tile.split("x")]
    return 3 * (t[0] // 64) + t[-1] // 64


def run(gpu_ctx, pb, xs, env, precision="f64"):
    # the product as well: the packed split-BF16 plan and the lists for many
    # right-hand sides are tiled by the first of them
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        h = EffectiveHamiltonian(pb, gpu_ctx, fp32=precision == "f32")
        x = torch.tensor(xs, dtype=torch.float64, device="cuda:0")
        y = h.multiply(x, precision=precision).cpu().numpy()
        fl = np.array(h.kernel_flops(precision))
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    h.deallocate()
    for k in (L.K_PHASE1, L.K_PHASE2):  # what was forced is what ran
        used = set(np.flatnonzero(fl[k:k + 9]))
        if "B2G_TILE" in env:
            assert used == {cfg(env["B2G_TILE"])}, (env, used)
        if env.get("B2G_TILE_CAP") == "64":
            assert used <= {0, 4}, (env, used)
        elif "B2G_TILE_CAP" in env:
            assert 8 in used, (env, used)
    return y


TILES = ["32", "64", "128", "32x64", "64x32", "32x128", "128x32", "64x128",
         "128x64", "auto"]


@pytest.mark.parametrize("tile", TILES)
def test_tile_configurations(gpu_ctx, problem, tile):
    pb, xs, ys = problem
    print("tile", tile, flush=True)
    env = {} if tile == "auto" else {"B2G_TILE": tile}
    y = run(gpu_ctx, pb, xs, env)
    for r in range(4):
        assert rel(y[r], ys[r]) < 1e-12, (tile, r)


def test_scratch_chunks(gpu_ctx, problem):
    pb, xs, ys = problem
    # about a tenth of the W scratch per chunk -> many chunks that accumulate
    y = run(gpu_ctx, pb, xs, {"B2G_W_CAP": "200000"})
    for r in range(4):
        assert rel(y[r], ys[r]) < 1e-12, r


@pytest.mark.parametrize("ksplit", ["1", "64", "1000"])
def test_split_k(gpu_ctx, problem, ksplit):
    # deep output blocks cut into partial tiles plus a fixed-order reduction;
    # with several scratch chunks the reductions accumulate into y
    pb, xs, ys = problem
    print("ksplit", ksplit, flush=True)
    for env in ({"B2G_KSPLIT": ksplit},
                {"B2G_KSPLIT": ksplit, "B2G_W_CAP": "200000"}):
        y = run(gpu_ctx, pb, xs, env)
        for r in range(4):
            assert rel(y[r], ys[r]) < 1e-12, (env, r)
    y = run(gpu_ctx, pb, xs, {"B2G_KSPLIT": ksplit}, precision="f32")
    for r in range(4):
        assert rel(y[r], ys[r]) < 2e-6, r


@pytest.mark.parametrize("cap", ["64", "128"])
@pytest.mark.parametrize("ksplit", ["16", "64", "2048"])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_tile_cap(gpu_ctx, problem, cap, ksplit, precision):
    # tiles of 32 and 64 mixed in one launch, and up to 128 with one launch
    # per larger shape, each with shallow and deep partial tasks (1e-12: sums
    # of 1e4 FP64 products; FP32 as below)
    pb, xs, ys = problem
    print("cap", cap, "ksplit", ksplit, precision, flush=True)
    y = run(gpu_ctx, pb, xs, {"B2G_TILE_CAP": cap, "B2G_KSPLIT": ksplit},
            precision=precision)
    for r in range(4):
        assert rel(y[r], ys[r]) < (1e-12 if precision == "f64" else 2e-6), r


@pytest.mark.parametrize("tile", TILES)
def test_bf16x3_tile_configurations(gpu_ctx, problem, tile):
    # split-BF16 three-term kernels, every tile shape; 1e-4 relative
    pb, xs, ys = problem
    print("bf16x3 tile", tile, flush=True)
    env = {} if tile == "auto" else {"B2G_TILE": tile}
    y = run(gpu_ctx, pb, xs, env, precision="bf16x3")
    for r in range(4):
        assert rel(y[r], ys[r]) < 1e-4, (tile, r, rel(y[r], ys[r]))


def test_fp32(gpu_ctx, problem):
    pb, xs, ys = problem
    y = run(gpu_ctx, pb, xs, {}, precision="f32")
    for r in range(4):
        assert rel(y[r], ys[r]) < 2e-6, r


@pytest.fixture(scope="module")
def small_blocks():
    # blocks of 1 to 33: depths on both sides of a k-chunk (16) and of a
    # packed line (32), most tiles partly outside their block
    pb = synth.middle_site(n_orb=12, m=120, max_dim=33, seed=5)
    xs = np.random.default_rng(4).standard_normal((3, pb.ket_len))
    orc = O.Oracle(pb)
    return pb, xs, np.stack([orc.hpsi(x, nthreads=8) for x in xs])


@pytest.mark.parametrize("tile", ["auto", "32", "128"])
@pytest.mark.parametrize("precision", ["f64", "f32", "bf16x3"])
def test_chunk_edges(gpu_ctx, small_blocks, precision, tile):
    # one and three right-hand sides (tasks dealt with their right-hand sides
    # next to one another); a vector's result does not depend on the others.
    # Tolerances as above (split-BF16: 2^-16 dropped per product, and sums)
    pb, xs, ys = small_blocks
    print(precision, "tile", tile, flush=True)
    env = {} if tile == "auto" else {"B2G_TILE": tile}
    y = run(gpu_ctx, pb, xs, env, precision=precision)
    tol = {"f64": 1e-12, "f32": 2e-6, "bf16x3": 1e-4}[precision]
    for r in range(3):
        assert rel(y[r], ys[r]) < tol, r
        one = run(gpu_ctx, pb, xs[r:r + 1], env, precision=precision)
        assert np.array_equal(one[0], y[r]), r


@pytest.mark.parametrize("precision", ["f64", "f32", "bf16x3"])
def test_many_right_hand_sides(gpu_ctx, precision):
    # 20000 vectors on some 900 tasks: more (task, vector) items than a launch
    # may have workgroups.  A vector's result does not depend on the others,
    # tolerances as above
    pb = synth.middle_site(n_orb=6, m=16, max_dim=4, seed=5)
    n = 20000
    xs = np.random.default_rng(3).standard_normal((n, pb.ket_len))
    print(precision, flush=True)
    y = run(gpu_ctx, pb, xs, {"B2G_KSPLIT": "100000"}, precision=precision)
    orc = O.Oracle(pb)
    tol = {"f64": 1e-12, "f32": 2e-6, "bf16x3": 1e-4}[precision]
    for r in (0, 1, 4097, n - 1):
        assert rel(y[r], orc.hpsi(xs[r], nthreads=8)) < tol, r
    part = run(gpu_ctx, pb, xs[n - 500:], {"B2G_KSPLIT": "100000"},
               precision=precision)
    assert np.array_equal(part, y[n - 500:])


@pytest.mark.parametrize("xcd", ["0", "1"])
@pytest.mark.parametrize("precision", ["f64", "f32", "bf16x3"])
def test_right_hand_side_groups(gpu_ctx, small_blocks, precision, xcd):
    # counts around a group of eight, whole and short groups, tasks dealt in
    # turn and by XCD list: every vector as alone
    pb, xs, ys = small_blocks
    x = np.random.default_rng(6).standard_normal((25, pb.ket_len))
    env = {"B2G_XCD": xcd}
    print(precision, "xcd", xcd, flush=True)
    want = np.stack([run(gpu_ctx, pb, v[None], env, precision=precision)[0]
                     for v in x])
    for n in (2, 7, 8, 9, 16, 17, 25):
        y = run(gpu_ctx, pb, x[:n], env, precision=precision)
        assert np.array_equal(y, want[:n]), n


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_lists_for_many_right_hand_sides(gpu_ctx, problem, precision):
    # from 64 right-hand sides on, this plan runs tiles up to 128; fewer after
    # that run its own lists again, on the scratch that is there
    pb, xs, ys = problem
    tol = 1e-12 if precision == "f64" else 2e-6
    h = EffectiveHamiltonian(pb, gpu_ctx, fp32=precision == "f32")
    x = torch.tensor(np.tile(xs, (17, 1)), device="cuda:0")
    own = None
    for n in (3, 63, 64, 65, 68, 3, 63):
        print(precision, n, flush=True)
        h.set_timing(True)
        y = h.multiply(x[:n], precision=precision).cpu().numpy()
        ms, cnt = h.timing()
        h.set_timing(False)
        for k in (L.K_PHASE1, L.K_PHASE2):
            assert (cnt[k + 8] > 0) == (n >= 64), (n, k)
        for r in range(n):
            assert rel(y[r], ys[r % 4]) < tol, (n, r)
        if n < 64:
            own = y[:3] if own is None else own
            assert np.array_equal(y[:3], own), n
    h.deallocate()


def test_many_right_hand_sides_in_chunks(gpu_ctx, problem):
    # the W scratch split into chunks that accumulate: lists for many of each
    pb, xs, ys = problem
    y = run(gpu_ctx, pb, np.tile(xs, (24, 1)), {"B2G_W_CAP": "200000"})
    for r in range(96):
        assert rel(y[r], ys[r % 4]) < 1e-12, r


@pytest.mark.parametrize("precision", ["f64", "f32", "bf16x3"])
@pytest.mark.parametrize("n", [1, 4, 70])
def test_captured_product(gpu_ctx, problem, precision, n):
    # a product on reserved scratch captured into a graph on the context's
    # stream (its output's address first asked for in the capture): every
    # replay as the eager product on the same vectors
    pb, xs, _ = problem
    lib, prec = gpu_ctx.lib, L.PREC[precision]
    h = EffectiveHamiltonian(pb, gpu_ctx, fp32=precision == "f32")
    L.check(lib.b2g_plan_reserve(h.plan, n, prec))
    buf = C.c_void_p()
    L.check(lib.b2g_buf_create(gpu_ctx.h, n * pb.bra_len, L.B2G_F64,
                               C.byref(buf)))
    x = torch.empty((n, pb.ket_len), dtype=torch.float64, device="cuda:0")
    st = torch.cuda.ExternalStream(lib.b2g_ctx_stream(gpu_ctx.h))
    graph = torch.cuda.CUDAGraph()
    print(precision, n, flush=True)
    with torch.cuda.graph(graph, stream=st):
        y = lib.b2g_buf_device_ptr(buf)
        L.check(lib.b2g_hpsi(gpu_ctx.h, h.plan, x.data_ptr(), y, n, 1.0, 0,
                             prec))
    got = np.empty((n, pb.bra_len))
    for k in range(3):
        x.copy_(torch.tensor(np.resize(xs[k:], (n, pb.ket_len))))
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            graph.replay()
        L.check(lib.b2g_buf_read(buf, got.ctypes.data, 0, got.size))
        # (one right-hand side: eager launches overlap, with the same sums)
        want = h.multiply(x, precision=precision).cpu().numpy()
        assert np.array_equal(got, want), k
    del graph
    lib.b2g_buf_destroy(buf)
    h.deallocate()
