"""Calls of neighbouring sizes cost alike: no launch shape is chosen where it is
many times slower than one that the call could take.  Each pair does the same
work, and the bounds leave room for several times the spread of such timings."""

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

DT = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}


@pytest.fixture(scope="module")
def st():
    from npbench_amd import device, stencils
    device.require_device()
    return stencils


def fastest(call, reps=20, rounds=5):
    """us a call, the best of several rounds of calls."""
    call()
    torch.cuda.synchronize()
    start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = float("inf")
    for _ in range(rounds):
        start.record()
        for _ in range(reps):
            call()
        stop.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(stop) / reps * 1e3)
    return best


def compare(what, call, like, bound):
    a, b = fastest(call), fastest(like)
    print(f"{what}: {a:.1f} us, like {b:.1f} us", flush=True)
    assert a < bound * b


@pytest.mark.parametrize("dtype,shape,like", [
    ("f64", (489, 489, 1), (122, 122, 16)), ("f64", (1732, 1732, 2), (433, 433, 32)),
    ("f32", (663, 663, 2), (166, 166, 32)), ("bf16", (500, 500, 4), (125, 125, 64))])
def test_hdiff_short_columns_cost_as_long_ones(st, dtype, shape, like):
    def call(I, J, K):
        gen = torch.Generator(device="cuda").manual_seed(I + K)
        f = [torch.rand(s, generator=gen, device="cuda").to(DT[dtype])
             for s in ((I + 4, J + 4, K), (I, J, K), (I, J, K))]
        return lambda: st.hdiff(*f)
    compare(f"hdiff {dtype} {shape} {like}", call(*shape), call(*like), 2)


@pytest.mark.parametrize("dtype,n,like", [("bf16", 264, 256), ("bf16", 513, 512),
                                          ("f64", 385, 384)])
def test_heat3d_side_just_past_a_vectors_multiple(st, dtype, n, like):
    def call(n):
        gen = torch.Generator(device="cuda").manual_seed(n)
        a = torch.rand((n,) * 3, generator=gen, device="cuda").to(DT[dtype])
        b = a.clone()
        return lambda: st.heat3d_sweeps(a, b, 8)
    a, b = fastest(call(n), 2), fastest(call(like), 2)
    print(f"heat3d {dtype} {n}^3 {a:.1f} us, {like}^3 {b:.1f} us", flush=True)
    assert a < 1.3 * (n / like) ** 3 * b


@pytest.mark.parametrize("nx,ny,nit", [(3, 400, 1), (400, 3, 1), (33, 33, 20)])
def test_cavity_flow_small_grids_cost_as_a_square_one(st, nx, ny, nit):
    def call(nx, ny):
        u, v, p = (torch.full((ny, nx), 0.01, dtype=torch.float64, device="cuda")
                   for _ in range(3))
        return lambda: st.cavity_flow(nx, ny, 50, nit, u, v, 1e-6, 2 / (nx - 1), 2 / (ny - 1), p,
                                      1.0, 0.1)
    compare(f"cavity_flow {nx} x {ny}, {nit} iterations", call(nx, ny),
            call(32, 32) if nit > 1 else call(20, 20), 1.15 if nit > 1 else 1.8)


def test_seidel2d_small_grids_cost_less_than_larger_ones(st):
    a, b = (torch.full((n, n), 0.5, dtype=torch.float64, device="cuda") for n in (4, 16))
    compare("seidel_2d 4 x 4, 69 sweeps", lambda: st.seidel2d(a, 70), lambda: st.seidel2d(b, 70),
            0.7)
