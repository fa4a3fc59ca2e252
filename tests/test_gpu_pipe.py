"""Pipelined window passes (fiber_pipe_kernel): shapes with ragged last tiles,
odd column counts and fibers of several sizes, each form of a pass (plain,
transposing, with phases, with a fused diagonal and the column factor it
leaves) against the oracle or against the same gates applied one by one."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import ffsim_amd
from oracle import oracle as O

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU"),
]

# eps times the square root of the rotations per amplitude, on normalized states
TOL = {"complex128": 1e-12, "complex64": 2e-5}
SHAPES = [(14, (7, 5)), (15, (7, 4)), (15, (6, 7)), (16, (5, 5)), (16, (4, 7))]


def _rotated(vec, mat, norb, nocc):
    return O.apply_orbital_rotation(vec, mat, norb, nocc)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("norb,nelec", SHAPES)
def test_rotation_of_product_states(norb, nelec, dtype):
    rng = np.random.default_rng(norb * 100 + nelec[1])
    facs = [O.random_state_vector(ffsim_amd.dim(norb, n), rng) for n in nelec]
    mats = [ffsim_amd.random.random_unitary(norb, seed=rng) for _ in nelec]
    state = torch.from_numpy(np.kron(*facs).astype(dtype)).cuda()
    for pair in ((mats[0], mats[1]), (None, mats[1]), (mats[0], None)):
        got = ffsim_amd.apply_orbital_rotation(state, pair, norb, nelec).cpu().numpy()
        want = np.kron(*[f if m is None else _rotated(f, m, norb, n)
                         for f, m, n in zip(facs, pair, nelec)])
        scale = np.abs(want).max()
        bound = TOL[dtype] if dtype == "complex128" else TOL[dtype] * scale
        assert np.abs(got - want).max() <= bound


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("norb,nelec", [(15, (7, 6)), (16, (5, 6))])
def test_ansatz_equals_its_gates(norb, nelec, dtype):
    """Fused diagonals, their column factors left to the next rotation, an
    identity rotation among them, against separate gate calls."""
    rng = np.random.default_rng(7)
    n_reps = 3
    rots = np.stack([ffsim_amd.random.random_unitary(norb, seed=rng) for _ in range(n_reps)])
    rots[1] = rots[0]  # the merged rotation between them is the identity
    mats = rng.uniform(-3, 3, (n_reps, 2, norb, norb))
    mats = mats + mats.transpose(0, 1, 3, 2)
    op = ffsim_amd.UCJOpSpinBalanced(diag_coulomb_mats=mats, orbital_rotations=rots)
    dim = ffsim_amd.dim(norb, nelec)
    g = torch.Generator(device="cuda").manual_seed(3)
    state = torch.empty(dim, dtype=getattr(torch, dtype), device="cuda")
    torch.view_as_real(state).normal_(generator=g)
    state /= torch.linalg.vector_norm(state)
    got = ffsim_amd.apply_unitary(state, op, norb, nelec)
    want = state.clone()
    for (aa, ab), u in zip(mats, rots):
        want = ffsim_amd.apply_diag_coulomb_evolution(want, (aa, ab, aa), -1.0, norb, nelec,
                                                      orbital_rotation=u)
    err = (got - want).abs().max().item()
    assert err <= (TOL[dtype] if dtype == "complex128"
                   else TOL[dtype] * want.abs().max().item())


# (norb, nelec, states): one workgroup's tile holds every string of a sector.  Each
# tile size (256, 480 and 928 strings of 128 bytes, 960 of 64, 256 and 464 of
# 256) with full and with ragged columns, down to a single one.
SMALL = [(6, (3, 1), 1), (7, (6, 3), 3), (10, (5, 3), 2), (10, (5, 3), 40), (11, (5, 2), 1),
         (11, (4, 6), 12), (11, (4, 6), 20), (12, (6, 1), 1), (12, (6, 4), 1), (12, (4, 6), 6)]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("norb,nelec,n_states", SMALL)
def test_small_sectors_in_place(norb, nelec, n_states, dtype):
    """Whole-sector passes in place, both orientations, on states that lie one
    element apart (8-byte alignment in complex64) with a guard between them."""
    from ffsim_amd.gates.orbital_rotation import orbital_rotations_in_place

    rng = np.random.default_rng(norb * 1000 + n_states)
    dim = ffsim_amd.dim(norb, nelec)
    facs = [O.random_state_vector(ffsim_amd.dim(norb, n), rng) for n in nelec]
    buf = torch.full((n_states * (dim + 1) + 1,), 7.0, dtype=getattr(torch, dtype), device="cuda")
    states = [buf[1 + i * (dim + 1):][:dim] for i in range(n_states)]
    start = torch.from_numpy(np.kron(*facs).astype(dtype)).cuda()
    mats = [tuple(ffsim_amd.random.random_unitary(norb, seed=rng) for _ in nelec)
            for _ in range(n_states)]
    for s in states:
        s.copy_(start)
    orbital_rotations_in_place(states, mats, norb, nelec)
    assert torch.all(buf[:: dim + 1] == 7.0)
    for i in {0, n_states // 2, n_states - 1}:
        want = np.kron(*[_rotated(f, m, norb, n) for f, m, n in zip(facs, mats[i], nelec)])
        bound = TOL[dtype] * (1.0 if dtype == "complex128" else np.abs(want).max())
        assert np.abs(states[i].cpu().numpy() - want).max() <= bound
