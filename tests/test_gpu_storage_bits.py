"""16-bit storage rounds the step that FP32 storage computes: from the same
populations, one step of either gives the same FP32 values before the rounding, so
that the 16-bit populations are the FP32 ones rounded, bit for bit."""
import numpy as np
import pytest
import torch

from helpers import random_velocity_field, tables
from lb_amd import Lattice, abi, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walls", [False, True], ids=["box", "walls"])
@pytest.mark.parametrize("before", [2, 3])   # the step under test is an even or an odd one
@pytest.mark.parametrize("coll", [abi.COLLISION_SRT, abi.COLLISION_CUM2015, abi.COLLISION_CUM2017,
                                  abi.COLLISION_COMBINED], ids=["srt", "2015", "2017", "combined"])
@pytest.mark.parametrize("storage,kept", [(abi.STORAGE_F16DEV, torch.float16), (abi.STORAGE_BF16DEV, torch.bfloat16)],
                         ids=["f16", "bf16"])
def test_one_step_is_the_rounded_fp32_step(storage, kept, coll, before, walls):
    shape = (8, 16, 33)
    flags = np.ones(shape, np.int32)
    if walls:
        flags[:, :, 0] = flags[:, 0] = 0
        flags[3:5, 6:9, 12:15] = 0
        flags[:, 10:, :] *= 2   # the Combined operator's 2017 branch
    fluid = flags != 0
    u = [np.where(fluid, c, 0.0) for c in random_velocity_field(shape, 0.04, 9)]
    kw = dict(collision=coll, closure=abi.CLOSURE_SMAGORINSKY, arith=abi.ARITH_FAST, tau=0.53, c_les=0.17,
              periodic=(0, 0, 1) if walls else (1, 1, 1))
    a = Lattice(make_desc(flags, [], storage=storage, **kw))
    b = Lattice(make_desc(flags, [], storage=abi.STORAGE_F32, **kw))
    a.init_equilibrium(None, *u)
    b.init_equilibrium(None, *u)
    a.step(before)
    b.set_populations(a.populations())
    a.step(1)
    b.step(1)
    fb = b.populations().astype(np.float32)
    rest = tables(0)[2].astype(np.float32).reshape(-1, 1, 1, 1)   # w rho0
    expect = torch.from_numpy(fb - rest).to(kept).float().numpy() + rest
    assert np.array_equal(a.populations().astype(np.float32)[:, fluid], expect[:, fluid])

