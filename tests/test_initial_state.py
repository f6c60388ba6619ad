"""initial_state on the CPU: the values of the oracle's mixture energy, and the mechanism file read anew
on every call (its parsed tables are kept by the file's contents)."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from pelec_amd import mechanism as M  # noqa: E402
from pelec_amd.autograd import initial_state  # noqa: E402


def state(mech, n, seed=3):
    m = M.load(mech)
    rng = np.random.default_rng(seed)
    Y = rng.uniform(size=(m.nsp, n))
    return (torch.tensor(rng.uniform(300, 3000, n)), torch.tensor(Y / Y.sum(0)),
            torch.tensor(rng.uniform(1e-4, 1e-2, n)))


@pytest.mark.parametrize("mech", ["LiDryer", "drm19", "gri30"])
def test_energy_vs_oracle(mech):
    from oracle.kinetics_np import NpMech
    T, Y, rho = state(mech, 5)
    m = M.load(mech)
    W = np.array([s.W for s in m.species])
    p = rho.numpy() * 8.31446261815324e7 * T.numpy() * (Y.numpy() / W[:, None]).sum(0)
    rho_ref, e_ref = NpMech(m).mixture(p, T.numpy(), Y.numpy().T)
    rY, rE = initial_state(mech, T, Y, rho)
    np.testing.assert_allclose(rY.numpy(), rho.numpy() * Y.numpy(), rtol=1e-15)
    # sums of up to 53 terms of both signs: ~53 eps of the largest term
    np.testing.assert_allclose(rE.numpy(), rho_ref * e_ref, rtol=1e-11)


def test_edited_file_is_parsed_again(tmp_path):
    path = str(tmp_path / "m.yaml")
    text = M.source("LiDryer").decode()
    T, Y, rho = state("LiDryer", 2)
    with open(path, "w") as f:
        f.write(text)
    a = initial_state(path, T, Y, rho)[1]
    with open(os.path.join(M.MECH_DIR, "drm19.yaml")) as f:
        other = f.read()
    with open(path, "w") as f:
        f.write(other)
    T, Y, rho = state("drm19", 2)
    b = initial_state(path, T, Y, rho)[1]
    assert torch.equal(b, initial_state("drm19", T, Y, rho)[1]) and a.shape == b.shape
