"""GPU: the x2 and x3 sweeps at the edges of their dispatch, bit for bit against the oracle
(with the GPU's correctly rounded x**2.5): blocks of two, four and seven species waves, lines
of every remainder of their step groups, rows of even and odd length (LDS DMA or registers),
periodic x3, in the fused step and in the transport block."""
import numpy as np
import pytest

import gemini_amd as ga
import oracle
from gemini_amd.transport import Transport
from helpers import compare

pytestmark = pytest.mark.gpu

VARS = ("ns", "vs1", "vs2", "vs3", "Ts", "rhovs1", "rhoes")


@pytest.mark.parametrize("shape", [(20, 2, 1), (20, 3, 2), (65, 4, 3), (66, 5, 4), (24, 6, 5), (24, 7, 9),
                                   (67, 8, 7), (70, 33, 34), (71, 34, 33), (130, 44, 43), (131, 43, 45)])
@pytest.mark.parametrize("periodic", [False, True])
def test_sweep_dispatch_matches_oracle(shape, periodic):
    if periodic and shape[2] < 2:
        pytest.skip("periodic x3 with one cell")
    print(f"case {shape} periodic {periodic}", flush=True)
    g = ga.cartesian_grid(*shape, flagper=periodic)
    st = ga.synthetic_state(g, seed=shape[1], perturb=True)
    dt = ga.cfl_dt(g, st)
    tr = Transport(g, st.nn, st.Tn, own_context=True)
    tr.set_residency(1)
    with oracle.pow_mode(1):
        for name in ("transport_step", "fluid_adv_block"):
            ref, got = st.copy(), st.copy()
            tr.push(got)
            for _ in range(2):
                getattr(oracle, name)(g, ref, dt)
                getattr(tr, name)(dt)
            tr.pull(got)
            compare(got, ref, exact=VARS)
    tr.close()


@pytest.mark.parametrize("size", [(4, 1, 1), (5, 1, 7), (4, 2, 1), (12, 3, 2), (61, 4, 9), (130, 17, 16)])
def test_ghost_fill_in_one_launch(size):
    """Inner columns that end as one, two or all of the ghost columns around them, blocks of
    columns and of cells with remainders."""
    g = ga.cartesian_grid(*size)
    st = ga.synthetic_state(g, seed=9, perturb=g.lx2 > 1 and g.lx3 > 1)
    rng = np.random.default_rng(9)
    oracle.op(g, st, "v12rhov1")
    oracle.op(g, st, "T2rhoe")
    st.fluidvars[...] *= rng.uniform(0.5, 1.5, st.fluidvars.shape)
    st.fluidauxvars[..., :14] *= rng.uniform(0.5, 1.5, st.fluidauxvars[..., :14].shape)
    tr = Transport(g, st.nn, st.Tn)
    tr.set_interface_vels(st)
    a, b = st.copy(), st.copy()
    oracle.op(g, a, "set_global_boundaries_allspec")
    tr.set_global_boundaries_allspec(b)
    assert np.array_equal(a.fluidvars, b.fluidvars)
    assert np.array_equal(a.fluidauxvars[..., :14], b.fluidauxvars[..., :14])
    tr.close()
