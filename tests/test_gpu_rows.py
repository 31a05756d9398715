"""Neighbour rows built by a tile's workgroup (rows of at most 64 entries), by one lane per vertex
(wider rows), and without cells (boxes narrower than three cells): the oracle's rows, ascending."""
import numpy as np
import pytest

from cudaring_amd import packing
from tests.helpers import gpu_from_state, oracle_from_state

pytestmark = pytest.mark.gpu


# ring sizes: tiles of four 16-vertex rings (64 lanes in use), of one 33-vertex ring (31 idle), of one 64;
# skins: rows of a few entries, of about 64, of more than 64; 4 rings: all-pairs search
@pytest.mark.parametrize("nrings,n_small,n_large", [(40, 16, 16), (40, 33, 33), (24, 13, 64), (4, 16, 22)])
@pytest.mark.parametrize("skin", [0.0, 0.5, 4.0, 6.0])
def test_rows_match_oracle(oracle_mod, nrings, n_small, n_large, skin):
    st = packing.lattice_system(nrings, 0.8, 11, n_small=n_small, n_large=n_large, perturb=0.1)
    size = 2 * float(np.mean(st["rad"]))
    g = gpu_from_state(st)
    o = oracle_from_state(oracle_mod, st)
    cut = g.set_displacement_cutoff(skin, size)
    o.set_displacement_cutoff(skin, size)
    g.calc_neighbor_list(cut)
    o.calc_neighbor_list(cut)
    rows, width, cnt = g.neighbors()
    assert cnt.max() <= width
    for a, b in zip(rows, o.neighbors()[0]):
        assert a == sorted(b)
    g.close()
