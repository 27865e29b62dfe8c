"""The N-body kernel that spreads any multiple of 1,024 bodies over the compute units
(ktt_amd/kernels/NbodySplit.hip) against the FP64 oracle, at every shape the default picks (8 x 1 to 64 x 4 lanes x
bodies), by itself or named, and at the extremes of BODY_LANES and BODIES_PER_THREAD: one and several source tiles,
one and 64 source groups per wave."""

from __future__ import annotations

import numpy as np
import pytest

from ktt_amd import capi
from test_gpu_nbody import bodies, check, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,config", [(1024, None), (2048, None), (3072, None), (9216, None), (16384, None),
                                      (2048, "BODY_LANES=8,BODIES_PER_THREAD=4"), (3072, "BODY_LANES=16,BODIES_PER_THREAD=4"),
                                      (2048, "BODY_LANES=32,BODIES_PER_THREAD=4"), (3072, "BODY_LANES=8,BODIES_PER_THREAD=2"),
                                      (1024, "BODY_LANES=1,BODIES_PER_THREAD=1"), (2048, "BODY_LANES=4,BODIES_PER_THREAD=4"),
                                      (3072, "BODY_LANES=64,BODIES_PER_THREAD=4"), (2048, "BODY_LANES=16,BODIES_PER_THREAD=2")])
def test_split_against_fp64(n, config):
    pos, vel = bodies(n, seed=n)
    print("nbody split", n, config, flush=True)
    outputs = run(pos, vel, config)
    check(pos, vel, *outputs)
    for first, second in zip(outputs, run(pos, vel, config)):
        np.testing.assert_array_equal(first, second)


def test_split_refuses_what_it_cannot_take():
    pos, vel = bodies(1536)
    with pytest.raises(capi.KttHipError, match="multiple of 1024"):
        run(pos, vel)
    pos, vel = bodies(1024)
    for config in ("BODY_LANES=48", "BODY_LANES=64,BODIES_PER_THREAD=8", "BODY_LANES=8,BODIES_PER_THREAD=3", "BODY_LANES=0"):
        with pytest.raises(capi.KttHipError, match="BODY_LANES"):
            run(pos, vel, config)
