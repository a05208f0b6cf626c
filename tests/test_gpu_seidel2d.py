"""GPU parity of the 2-D Gauss-Seidel sweeps (npbx_seidel2d) against the FP64
oracle.

Tiles of 64 rows and 4 sweeps run with the reference's arithmetic, so results
must be bitwise the oracle's.  Sizes cover the smallest grids (one wave up to 10
points a side), row counts around the tiles' bands and sweep counts around their
groups, launches split by the "seidel.blocks" budget, the division operator's
path, zeros of either sign, calls on two streams and under capture, a wait that
gives up, the reference's initialisation at its S, M, L and paper presets, and
the largest accepted N.  Large cases are checked
against the oracle's C restatement (pinned bit for bit to the NumPy oracle on
the CPU).
"""

import numpy as np
import pytest

from oracle import stencils as ref

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def st():
    from npbench_amd import device, stencils
    device.require_device()
    return stencils


def assert_bitwise(x, y, what):
    if not np.array_equal(x, y):
        bad = np.argwhere(x != y)
        first = tuple(bad[0])
        raise AssertionError(f"{what}: {len(bad)} elements differ, first at {first}: "
                             f"{x[first]!r} vs {y[first]!r}")


def check(st, tsteps, A, what, oracle=None):
    from npbench_amd import device
    n = A.shape[0]
    want = A.copy()
    (oracle or ref.seidel_2d_kernel)(tsteps, n, want)
    d = device.to_device(A, torch.float64)
    print(f"seidel2d {what}", flush=True)
    st.seidel2d(d, tsteps)
    torch.cuda.synchronize()
    assert_bitwise(d.cpu().numpy(), want, what)


@pytest.mark.parametrize("n", [3, 4, 5, 17, 64, 65, 66, 130, 257, 258, 259, 600])
@pytest.mark.parametrize("tsteps", [1, 2, 3, 7])
def test_seidel2d_fp64_bitwise(st, n, tsteps):
    rng = np.random.default_rng(n * 100 + tsteps)
    check(st, tsteps, rng.random((n, n)), f"n={n} tsteps={tsteps}")


def test_seidel2d_two_launches(st):
    rng = np.random.default_rng(9)
    check(st, 70, rng.random((20, 20)), "n=20 tsteps=70 (69 sweeps)")


@pytest.mark.parametrize("tsteps,n", [(8, 50), (15, 100), (40, 200)])
def test_seidel2d_reference_presets_bitwise(st, tsteps, n):
    from npbench_amd.benchmarks.polybench.seidel_2d import seidel_2d
    check(st, tsteps, seidel_2d.initialize(n), f"preset n={n} tsteps={tsteps}")


def test_seidel2d_zero_field(st):
    """Zeros take the division-operator path of every row."""
    check(st, 3, np.zeros((9, 9)), "zeros")


def test_seidel2d_dropin_numpy_roundtrip(st):
    from npbench_amd.benchmarks.polybench.seidel_2d import seidel_2d_mi355x
    rng = np.random.default_rng(8)
    A = rng.random((30, 30))
    want = A.copy()
    ref.seidel_2d_kernel(5, 30, want)
    assert seidel_2d_mi355x.kernel(5, 30, A) is None
    assert_bitwise(A, want, "drop-in")


@pytest.fixture
def seidel_blocks():
    """Sets the slot-blocks-per-launch knob for one test and restores it."""
    from npbench_amd import _native
    old = _native.get_tuning("seidel.blocks")
    yield lambda b: _native.set_tuning("seidel.blocks", b)
    _native.set_tuning("seidel.blocks", old)


@pytest.mark.parametrize("tsteps,n", [(100, 400), (66, 300)])
def test_seidel2d_full_slots_bitwise(st, tsteps, n):
    """Slots of all 64 rows (lanes 0..63 of the recurrence wave), at the
    paper preset and at N=300 with 65 sweeps."""
    from npbench_amd.benchmarks.polybench.seidel_2d import seidel_2d
    from oracle import c_oracle
    check(st, tsteps, seidel_2d.initialize(n), f"full slots n={n} tsteps={tsteps}",
          oracle=c_oracle.seidel_2d_kernel)


@pytest.mark.parametrize("blocks", [1, 7, 64])
def test_seidel2d_launches_split_at_any_slot(st, seidel_blocks, blocks):
    """Launches of 1, 7 and 64 slot-blocks (a slot of N=300 has 2 blocks):
    the split never changes a bit."""
    from oracle import c_oracle
    seidel_blocks(blocks)
    rng = np.random.default_rng(blocks)
    check(st, 70, rng.random((300, 300)), f"n=300 tsteps=70 seidel.blocks={blocks}",
          oracle=c_oracle.seidel_2d_kernel)


def test_seidel2d_largest_n(st):
    """N = 16384, the largest accepted, two sweeps."""
    from oracle import c_oracle
    rng = np.random.default_rng(16384)
    check(st, 3, rng.random((16384, 16384)), "n=16384 tsteps=3",
          oracle=c_oracle.seidel_2d_kernel)



@pytest.mark.parametrize("n", [61, 62, 63, 64, 65, 66, 67, 125, 126, 127, 128, 129, 130, 131, 193])
@pytest.mark.parametrize("tsteps", [2, 5, 6, 10])
def test_seidel2d_tile_edges(st, n, tsteps):
    """Row counts around the 64-row bands (which shift up by a row per sweep
    of a group) and sweep counts around the groups of four, the last group
    holding one, two and four sweeps."""
    from oracle import c_oracle
    rng = np.random.default_rng(n * 10 + tsteps)
    check(st, tsteps, rng.random((n, n)), f"edges n={n} tsteps={tsteps}",
          oracle=c_oracle.seidel_2d_kernel)


# the one-wave form's sizes beside the first of the tiles, and two launches of it
@pytest.mark.parametrize("n,tsteps", [(6, 2), (7, 40), (9, 3), (10, 2), (10, 41), (11, 41),
                                      (4, 65539)])
def test_seidel2d_small_grids(st, n, tsteps):
    from oracle import c_oracle
    A = np.random.default_rng(n).random((n, n))
    A[n // 2, 1:3] = 1e300  # past the tiles' short division
    check(st, tsteps, A, f"small n={n} tsteps={tsteps}", oracle=c_oracle.seidel_2d_kernel)


@pytest.mark.parametrize("case", ["tiny", "huge", "zeros and signs"])
def test_seidel2d_division_range(st, case):
    """Values past the short division's range take the operator; zeros of
    either sign stay on it."""
    n = 140
    rng = np.random.default_rng(2)
    A = rng.random((n, n))
    if case == "tiny":
        A *= 1e-300
    elif case == "huge":
        A[70, 70] = 1e300
    else:
        A[20:120, 20:120] = np.where(rng.random((100, 100)) < 0.5, 0.0, -0.0)
    from oracle import c_oracle
    check(st, 6, A, case, oracle=c_oracle.seidel_2d_kernel)


def test_seidel2d_two_streams(st):
    """Calls in flight on two streams do not share state."""
    from npbench_amd import device
    from oracle import c_oracle
    rng = np.random.default_rng(31)
    grids = [rng.random((n, n)) for n in (150, 260, 150, 260)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    dev_grids = [device.to_device(A, torch.float64) for A in grids]
    torch.cuda.synchronize()
    for rep in range(6):
        for k, d in enumerate(dev_grids):
            st.seidel2d(d, 9, stream=streams[k % 2])
    torch.cuda.synchronize()
    for A, d in zip(grids, dev_grids):
        want = A.copy()
        for rep in range(6):
            c_oracle.seidel_2d_kernel(9, A.shape[0], want)
        assert_bitwise(d.cpu().numpy(), want, f"two streams n={A.shape[0]}")


@pytest.mark.parametrize("n,tsteps", [(50, 8), (200, 14)])
def test_seidel2d_captured(st, n, tsteps):
    """Under capture the tiles run slot by slot; every replay continues the
    grid as an eager call does."""
    from npbench_amd import device
    from oracle import c_oracle
    rng = np.random.default_rng(n)
    want = rng.random((n, n))
    d = device.to_device(want, torch.float64)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        st.seidel2d(d, tsteps)
    for rep in range(3):
        graph.replay()
        torch.cuda.synchronize()
        c_oracle.seidel_2d_kernel(tsteps, n, want)
        assert_bitwise(d.cpu().numpy(), want, f"replay {rep}")
        st.seidel2d(d, tsteps)  # an eager call between the replays
        torch.cuda.synchronize()
        c_oracle.seidel_2d_kernel(tsteps, n, want)
        assert_bitwise(d.cpu().numpy(), want, f"eager {rep}")


@pytest.mark.parametrize("n,tsteps", [(5, 2), (140, 10)])
@pytest.mark.parametrize("signs", ["all negative", "half"])
@pytest.mark.parametrize("captured", [False, True])
def test_seidel2d_signed_zeros(st, n, tsteps, signs, captured):
    """Zeros keep the sign that the reference's sums give them, in every bit:
    nine -0.0 sum to -0.0, and any +0.0 among them makes a sum +0.0."""
    from npbench_amd import device
    want = np.full((n, n), -0.0)
    if signs == "half":  # every other block of rows, so that whole stencils are -0.0
        want[(np.arange(n) // 16) % 2 == 1] = 0.0
    d = device.to_device(want, torch.float64)
    torch.cuda.synchronize()
    print(f"seidel2d signed zeros n={n} tsteps={tsteps} {signs} captured={captured}", flush=True)
    if captured:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            st.seidel2d(d, tsteps)
        graph.replay()
    else:
        st.seidel2d(d, tsteps)
    torch.cuda.synchronize()
    ref.seidel_2d_kernel(tsteps, n, want)
    assert np.array_equal(d.cpu().numpy().view(np.uint64), want.view(np.uint64))


def test_seidel2d_wait_that_gives_up_is_reported(st):
    """A wait that may poll once only gives up: the kernel ends, every row of
    the tile that waited is NaN, and the next synchronisation (or call) says
    so, once."""
    from npbench_amd import _native, device
    from oracle import c_oracle
    n = 200
    A = np.random.default_rng(6).random((n, n))
    d = device.to_device(A, torch.float64)
    old = _native.get_tuning("seidel.polls")
    print("seidel2d bounded wait", flush=True)
    _native.set_tuning("seidel.polls", 0)
    try:
        st.seidel2d(d, 2)
    finally:
        _native.set_tuning("seidel.polls", old)
    with pytest.raises(_native.NpbxError, match="gave up"):
        device.sync()
    # the last band of 64 rows waits before its first column
    assert np.isnan(d.cpu().numpy()[193:-1, 1:-1]).all()
    device.sync()
    check(st, 5, A, "after a failed call", oracle=c_oracle.seidel_2d_kernel)
