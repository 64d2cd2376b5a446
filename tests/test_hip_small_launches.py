"""bf16 backward in the launches that pick its workgroups by their number: 4 waves up to 256 key groups of 128 (in balanced order between one
and two workgroups per CU), pairs of complementary key groups above."""
import pytest
import torch

from oracle import ua_oracle as orc
from tests.util import NAMES, TOL, dense_reference, key_gradient_bar, rel_err

pytestmark = pytest.mark.gpu
GRADS = ("dkc", "dvc", "dxq", "dsrc", "ddest")


# b copies of the same h heads: workgroups of 64 keys 2, 12, 264 (not a multiple of 8 heads), 512 and 512 (two parts of the query groups);
# then 390 and 264 key groups of 128, an odd and an even number per head
@pytest.mark.parametrize("b,h,r,L,d", [(1, 1, 1, 31, 64), (1, 2, 2, 333, 128), (66, 1, 1, 250, 72), (64, 2, 1, 161, 128), (64, 1, 2, 256, 64),
                                       (65, 2, 1, 300, 128), (66, 2, 1, 200, 64)])
@pytest.mark.parametrize("prune", [False, True])
def test_launches_of_every_size_match_the_oracle(b, h, r, L, d, prune):
    from universal_attention_triton_amd.universal_attention import universal_attention
    print("case", (b, h, r, L, d), prune, flush=True)
    inp = orc.make_inputs(1, h, r, L, d, L, dtype=torch.bfloat16, seed=85)
    O_ref, _, grads_ref = dense_reference(inp)
    leaves = [inp[k].repeat(b, *[1] * (inp[k].dim() - 1)).cuda().requires_grad_() for k in NAMES]
    out = universal_attention(*leaves, prune=prune)
    up = inp["dO"].repeat(b, *[1] * (inp["dO"].dim() - 1)).cuda().reshape(out.shape)
    grads = torch.autograd.grad(out, leaves, up)
    assert rel_err(out[:1].reshape(O_ref.shape), O_ref) <= TOL[torch.bfloat16]
    for name, x, y in zip(GRADS, grads, grads_ref):
        assert torch.equal(x, x[:1].expand_as(x)), name          # whatever place of the launch a head has
        bar = key_gradient_bar(inp, torch.bfloat16, y) if name == "dkc" else TOL[torch.bfloat16]
        assert rel_err(x[:1], y) <= bar, name
