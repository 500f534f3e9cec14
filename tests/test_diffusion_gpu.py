"""GPU: the energy diffusion at the edges of its tiling, bit for bit against the oracle (with
the GPU's correctly rounded x**2.5): lines a block of kept rows shorter or longer by one,
column counts around a half group of 32, a group of 64 and an interleaved block of 128, both
solvers, both chunk heights (4 always takes the wave kernel) and the small-grid kernel at each
of its block widths; singular columns in the wave kernel; the fitting extension in both; and
x**2.5 outside the range of its fast form."""
import numpy as np
import pytest

import gemini_amd as ga
import oracle
from gemini_amd.transport import Transport
from helpers import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 1, 1), (5, 7, 3), (7, 8, 4), (8, 31, 1), (9, 32, 1), (10, 33, 1),
                                   (15, 9, 7), (16, 13, 5), (17, 8, 16), (18, 43, 3), (23, 3, 43),
                                   (24, 16, 17), (33, 20, 13), (40, 14, 14),
                                   # more columns than the small-grid kernel takes
                                   (9, 115, 113), (16, 92, 91), (24, 77, 78), (33, 60, 61),
                                   # long lines: two columns a block, the last one the wave kernel
                                   (110, 3, 5), (230, 3, 3), (440, 2, 3), (700, 1, 3), (1100, 1, 2)])
@pytest.mark.parametrize("solver", [2, 1])
def test_diffusion_tiles_match_oracle(shape, solver):
    print(f"case {shape} solver {solver}", flush=True)
    grid = ga.dipole_grid if shape[1] > 1 and shape[2] % 2 else ga.cartesian_grid
    g = grid(*shape)
    st = ga.synthetic_state(g, seed=sum(shape))
    # temperatures that vary from row to row, so that rows interchange in both solves
    st.Ts[...] *= np.random.default_rng(1).uniform(0.5, 2.0, st.Ts.shape)
    np.maximum(st.Ts, 100.0, out=st.Ts)
    ref = st.copy()
    with oracle.pow_mode(1):
        oracle.op(g, ref, "energy_diffusion", dt=0.3, diffsolvetype=solver)
    tr = Transport(g, st.nn, st.Tn, own_context=True, diffsolvetype=solver)
    for chunk in (8, 4):
        tr.set_tuning("diff_chunk", chunk)
        got = st.copy()
        tr.energy_diffusion(got, 0.3)
        compare(got, ref, exact=("Ts", "ns"))
    tr.close()


@pytest.mark.parametrize("shape", [
    # blocks of 8 and 16 columns (512 and 1024 threads), the last one partly filled, up to three
    # blocks a CU and just beyond
    (96, 24, 20), (150, 15, 17), (98, 40, 36), (61, 41, 43),
    # and many more columns, short and long rows
    (9, 135, 135), (16, 108, 107), (24, 91, 91), (33, 71, 70)])
def test_wide_blocks_and_the_wave_kernel_beyond_them(shape):
    g = ga.cartesian_grid(*shape)
    st = ga.synthetic_state(g, seed=sum(shape))
    st.Ts[...] *= np.random.default_rng(1).uniform(0.5, 2.0, st.Ts.shape)
    np.maximum(st.Ts, 100.0, out=st.Ts)
    ref, got = st.copy(), st.copy()
    with oracle.pow_mode(1):
        oracle.op(g, ref, "energy_diffusion", dt=0.3, diffsolvetype=2)
    tr = Transport(g, st.nn, st.Tn, own_context=True, diffsolvetype=2)
    tr.energy_diffusion(got, 0.3)
    compare(got, ref, exact=("Ts", "ns"))
    tr.close()


# columns a block of the small-grid kernel owns there (0: the wave kernel takes the grid)
WIDTHS = [((17, 8, 16), 4), ((150, 15, 17), 8), ((96, 24, 20), 16), ((98, 40, 36), 16),
          # 1024 threads and the shortest rows, four and two columns because more do not fit
          # the LDS, the longest row that fits and one more
          ((4, 23, 21), 16), ((300, 20, 20), 4), ((600, 10, 20), 2), ((1073, 2, 2), 2),
          ((1074, 2, 2), 0),
          # blocks that outnumber the CUs three times
          ((61, 41, 43), 0), ((24, 77, 78), 0)]


def small_columns(lx1, lx2, lx3):
    """The kernel's rule: the fewest columns that leave one block per CU, else the most that
    fit the LDS if that makes at most three."""
    best = 0
    for w in (2, 4, 8, 16):
        if (lx1 + 3) * (9 * w + 1) * 8 + (lx1 + 31) // 32 * w * 4 > 160 * 1024:
            break
        blocks = (lx2 * lx3 + w - 1) // w * 7
        if blocks <= 256:
            return w
        best = w if blocks <= 768 else 0
    return best


@pytest.mark.parametrize("shape,width", WIDTHS)
def test_both_solvers_at_each_block_width(shape, width):
    print(f"case {shape} width {width}", flush=True)
    assert small_columns(*shape) == width
    g = ga.cartesian_grid(*shape)
    st = ga.synthetic_state(g, seed=sum(shape))
    st.Ts[...] *= np.random.default_rng(1).uniform(0.5, 2.0, st.Ts.shape)
    np.maximum(st.Ts, 100.0, out=st.Ts)
    for solver in (2, 1):
        ref, got = st.copy(), st.copy()
        with oracle.pow_mode(1):
            oracle.op(g, ref, "energy_diffusion", dt=0.3, diffsolvetype=solver)
        tr = Transport(g, st.nn, st.Tn, own_context=True, diffsolvetype=solver)
        tr.energy_diffusion(got, 0.3)
        compare(got, ref, exact=("Ts", "ns"))
        tr.close()


@pytest.mark.parametrize("shape,width", [((17, 8, 16), 4), ((40, 14, 14), 8), ((96, 24, 20), 16),
                                         ((24, 77, 78), 0), ((33, 70, 71), 0), ((16, 64, 90), 0)])
def test_fitting_extension_at_each_block_width(shape, width):
    """Also the wave kernel of chunk height 8, its groups with columns in turn and with even and
    odd ones apart; conductivity scale and heat flux together and each alone."""
    print(f"case {shape} width {width}", flush=True)
    assert small_columns(*shape) == width
    g = ga.cartesian_grid(*shape)
    st = ga.synthetic_state(g, seed=6)
    rng = np.random.default_rng(7)
    kappa = rng.uniform(0.5, 1.5, (g.lx2, g.lx3))
    qtop = rng.uniform(0.0, 1e-5, (g.lx2, g.lx3))
    tr = Transport(g, st.nn, st.Tn, own_context=True)
    tr.set_residency(1)
    for k, q in ((kappa, qtop), (kappa, None), (None, qtop)):
        ref, got = st.copy(), st.copy()
        with oracle.pow_mode(1):
            oracle.transport_step(g, ref, 0.2, kappa=k, qtop=q)
        tr.set_conductivity_scale(k)
        tr.set_top_heat_flux(q)
        tr.push(got)
        tr.transport_step(0.2)
        tr.pull(got)
        compare(got, ref, exact=("Ts", "ns"))
    tr.close()


@pytest.mark.parametrize("shape,width", [((21, 24, 20), 16), ((21, 45, 46), 0), ((24, 46, 46), 0)])
@pytest.mark.parametrize("solver", [2, 1])
def test_singular_columns_at_chunk_height_eight(shape, width, solver):
    """Zero pivots (see test_singular_columns_in_both_kernels) in every column group: rows of
    odd length put the groups' row windows at every phase."""
    print(f"case {shape} solver {solver}", flush=True)
    assert small_columns(*shape) == width
    g = ga.cartesian_grid(*shape)
    st = ga.synthetic_state(g, seed=5)
    st.J1[...] = 0.0
    cold = np.random.default_rng(3).random((g.lx2, g.lx3, 7)) < 0.04
    T = st.Ts[8:13, 2:-2, 2:-2, :]
    T[...] = np.where(cold, 0.0, T)
    ref, got = st.copy(), st.copy()
    with oracle.pow_mode(1):
        oracle.op(g, ref, "energy_diffusion", dt=np.inf, diffsolvetype=solver)
    tr = Transport(g, st.nn, st.Tn, own_context=True, diffsolvetype=solver)
    tr.energy_diffusion(got, np.inf)
    compare(got, ref, exact=("Ts",))
    tr.close()


@pytest.mark.parametrize("solver", [2, 1])
def test_singular_columns_in_both_kernels(solver):
    """Zero temperature on five rows and an infinite step make exact zero pivots."""
    g = ga.cartesian_grid(20, 40, 3)
    st = ga.synthetic_state(g, seed=5)
    st.J1[...] = 0.0
    for isp, i2, i3 in ((1, 2, 1), (3, 39, 2), (6, 7, 2)):
        st.Ts[8:13, i2 + 1, i3 + 1, isp] = 0.0
    ref = st.copy()
    with oracle.pow_mode(1):
        oracle.op(g, ref, "energy_diffusion", dt=np.inf, diffsolvetype=solver)
    tr = Transport(g, st.nn, st.Tn, own_context=True, diffsolvetype=solver)
    for chunk in (8, 4):
        tr.set_tuning("diff_chunk", chunk)
        got = st.copy()
        tr.energy_diffusion(got, np.inf)
        compare(got, ref, exact=("Ts",))
    tr.close()


@pytest.mark.parametrize("shape", [(21, 5, 3), (64, 9, 8)])
def test_fitting_extension_in_both_kernels(shape):
    g = ga.cartesian_grid(*shape)
    st = ga.synthetic_state(g, seed=6)
    rng = np.random.default_rng(7)
    kappa = rng.uniform(0.5, 1.5, (g.lx2, g.lx3))
    qtop = rng.uniform(0.0, 1e-5, (g.lx2, g.lx3))
    ref = st.copy()
    with oracle.pow_mode(1):
        oracle.transport_step(g, ref, 0.2, kappa=kappa, qtop=qtop)
    tr = Transport(g, st.nn, st.Tn, own_context=True)
    tr.set_conductivity_scale(kappa)
    tr.set_top_heat_flux(qtop)
    tr.set_residency(1)
    for chunk in (8, 4):
        tr.set_tuning("diff_chunk", chunk)
        got = st.copy()
        tr.push(got)
        tr.transport_step(0.2)
        tr.pull(got)
        compare(got, ref, exact=("Ts", "ns"))
    tr.close()


def test_pow25_outside_its_fast_range():
    g = ga.cartesian_grid(8, 4, 3)
    st = ga.synthetic_state(g)
    tr = Transport(g, st.nn, st.Tn, own_context=True)
    m = np.random.default_rng(2).uniform(1.0, 4.0, 4096)
    core = tr.eval_math(0, m)
    for k in (-280, -205, 201, 202):               # results stay normal numbers
        x = np.ldexp(m, 2 * k)
        x[::3] = m[::3]                            # waves that hold both kinds
        want = np.ldexp(core, 5 * k)
        want[::3] = core[::3]
        fin = np.isfinite(want) & (np.abs(want) >= 2.0 ** -1022)
        assert np.array_equal(tr.eval_math(0, x)[fin], want[fin])
    x = np.array([0.0, -0.0, np.inf, np.nan, -1.0, 1e300, 1e-300, 5e-324, 1.0, 4.0])
    want = np.array([0.0, 0.0, np.inf, np.nan, np.nan, np.inf, 0.0, 0.0, 1.0, 32.0])
    assert np.array_equal(tr.eval_math(0, x), want, equal_nan=True)
    tr.close()
