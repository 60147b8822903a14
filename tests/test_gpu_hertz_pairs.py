"""The sphere pair kernel of the Hertz–Mindlin engine over several tiles of pairs, bit for bit
against the oracle: contacts that open and close, no contact at all, and nearly every pair in
contact."""
import numpy as np
import pytest

from test_gpu_hertz import assert_same, hip_sim, pile_scene
from oracle_binding import oracle_sim


@pytest.mark.gpu
@pytest.mark.parametrize("n,sp,skin", [(343, 0.98, 0.6), (343, 0.90, 0.05), (120, 0.98, 1.2),
                                       (9, 1.4, 2.0), (1, 1.0, 0.3)])
def test_pair_tiles(hip_lib, n, sp, skin):
    h, r = (pile_scene(s, n, 13, sp=sp, row=7) for s in (hip_sim(n), oracle_sim(n)))
    for c in range(4):
        tag = f"n={n} sp={sp} skin={skin} call {c}"
        print(tag, flush=True)
        # (short calls: the list outlives the call, and its contacts with it)
        for s in (h, r):
            s.step_hertz(1e-4, 40, skin)
            if c == 1:  # every body thrown away from its contacts: pairs part and are cleared
                s.set_velocities(20.0 * (s.get_positions() - np.array([4.0, 4.0, 2.0])))
        assert_same(h, r, tag)
