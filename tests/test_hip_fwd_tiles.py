"""The forward over bias tiles (k_fwd_tiles) in every split of its waves, at the edges of its 32-query blocks and steps."""
import pytest
import torch

from oracle import ua_oracle as orc
from tests.util import NAMES, TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,r,L,d", [(1, 1, 1, 31, 24), (2, 2, 1, 33, 64), (1, 3, 3, 129, 72), (1, 2, 2, 255, 128), (2, 1, 4, 97, 100), (1, 2, 1, 640, 128)])
def test_every_split_of_the_waves_matches_the_oracle(b, h, r, L, d):
    from universal_attention_triton_amd import ops
    inp = orc.make_inputs(b, h, r, L, d, L, dtype=torch.bfloat16, seed=81)
    ref = [inp[k].double() for k in NAMES]
    O_ref, lse_ref = orc.dense_forward(ref[0].reshape(b, h, L, d), ref[1].reshape(b, h, L, d), ref[2], ref[3].reshape(b, h, L), ref[4].reshape(b, h, L),
                                       return_lse=True)
    dev = [inp[k].cuda() for k in NAMES]
    for v in range(ops.tune_variants(dev[0], dev[2], "fwd_tiles")):
        ops.tune_set(dev[0], dev[2], v, "fwd_tiles")
        try:
            for prune in (False, True):
                print("case", (b, h, r, L, d), "variant", v, "prune", prune, flush=True)
                O, lse, _ = ops.fused_forward(*dev, prune=prune)
                assert rel_err(O, O_ref) <= TOL[torch.bfloat16] and float((lse.double().cpu() - lse_ref.reshape(lse.shape)).abs().max()) <= 2e-2, (v, prune)
        finally:
            ops.tune_set(dev[0], dev[2], -1, "fwd_tiles")
