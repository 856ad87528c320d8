"""Every group width against the host build, which plays a match on one lane in sequence: the loops
split over the lanes of a match (2 to 64), the work its halves share and the places where the matches
of a wavefront meet give the same outputs and states, bit for bit. The scenarios have the ball in
flight, touched, carried by a keeper and at rest, and teams of 3 to 11 players."""

import numpy as np
import pytest
import torch

from conftest import PRODUCT, digest_actions
from oracle import ref

pytestmark = pytest.mark.gpu

# Scenario, agents, steps.
PLAYED = [('11_vs_11_stochastic_l11_r0', 11, 30), ('5_vs_5_l4_r0', 4, 60), ('academy_3_vs_1_with_keeper_l3_r0', 3, 60)]


def host(x):
    return x.detach().cpu().numpy()


@pytest.mark.parametrize('assets,agents,steps', PLAYED, ids=[p[0] for p in PLAYED])
@pytest.mark.parametrize('matches,lanes', [(32, 2), (16, 4), (8, 8), (3, 16), (2, 32), (1, 64)])
def test_every_width_plays_as_one_lane(assets, agents, steps, matches, lanes, host_library, monkeypatch):
    import cuju_amd
    environments = 35  # a last wavefront that is not full, at every width but 64 (one match fills one)
    theirs = ref.ReferenceBatch(assets, environment_count=environments, seed=9, threads=0, library_path=host_library)
    monkeypatch.setenv('CUJU_AMD_MATCHES', str(matches))
    monkeypatch.setenv('CUJU_AMD_LANES', str(lanes))
    mine = cuju_amd.BatchEnvironment(assets, library=PRODUCT, device='cuda:0', environment_count=environments, seed=9)
    try:
        assert mine.geometry == (matches, lanes)
        assert host(mine.reset()).tobytes() == theirs.reset().tobytes()
        for step in range(steps):
            actions = digest_actions(step, environments, agents, 19)
            a = mine.step(torch.as_tensor(actions, device='cuda:0'))
            b = theirs.step(actions)
            for x, y in zip(a[:3], b):
                assert host(x).astype(y.dtype).tobytes() == y.tobytes(), f'step {step}'
        for e in range(environments):
            assert mine.get_state(e) == theirs.get_state(e), f'state of environment {e}'
    finally:
        mine.close()
        theirs.close()
