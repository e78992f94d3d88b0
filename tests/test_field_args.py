"""CPU test of the full-field entry points: a field that is no cube (a half field,
say) is refused before the device reads it by the cube's indices."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import pyspectrum as P


@pytest.mark.parametrize("d", [np.zeros((4, 4, 3), complex), torch.zeros((8, 4, 4), dtype=torch.complex64),
                               np.zeros((4, 4), complex)])
def test_only_cubes(d):
    with pytest.raises(ValueError, match="shape"):
        P._Bk_periodic(d, Nmax=1, Ncut=1, step=1)
    with pytest.raises(ValueError, match="shape"):
        P._B0_survey(d, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, Nmax=1, Ncut=1, step=1)
