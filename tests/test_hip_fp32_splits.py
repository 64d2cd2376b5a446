"""float32: the forward with the keys of a query block divided among waves (two or four ways), and the small workgroups of the
backward, at the edges of their query blocks and steps."""
import pytest
import torch

from oracle import ua_oracle as orc
from tests.util import NAMES, TOL, dense_reference, key_gradient_bar, rel_err

pytestmark = pytest.mark.gpu
GRADS = ("dkc", "dvc", "dxq", "dsrc", "ddest")


# b copies of the same h heads.  Few of them: four splits (launches under one 32-query workgroup per CU); many: two.
@pytest.mark.parametrize("b,h,r,L,d", [(1, 1, 1, 15, 24), (1, 2, 2, 97, 64), (1, 1, 3, 129, 100), (2, 2, 1, 385, 128),
                                       (64, 1, 2, 130, 64), (64, 2, 1, 161, 72), (128, 1, 1, 257, 40)])
@pytest.mark.parametrize("prune", [False, True])
def test_small_workgroups_match_the_oracle(b, h, r, L, d, prune):
    from universal_attention_triton_amd import ops
    from universal_attention_triton_amd.universal_attention import universal_attention
    print("case", (b, h, r, L, d), prune, flush=True)
    inp = orc.make_inputs(1, h, r, L, d, L, dtype=torch.float32, seed=83)
    O_ref, lse_ref, grads_ref = dense_reference(inp)
    dev = [inp[k].repeat(b, *[1] * (inp[k].dim() - 1)).cuda() for k in NAMES]
    O, lse, _ = ops.fused_forward(*dev, prune=prune)
    assert torch.equal(O, O[:1].expand_as(O)) and torch.equal(lse.reshape(b, -1), lse.reshape(b, -1)[:1].expand(b, -1))
    # float32 sums of up to L terms, and exp2 of a bias of up to L rounded terms
    assert rel_err(O[:1].reshape(O_ref.shape), O_ref) <= 2e-5
    assert float((lse.reshape(b, -1)[0].double().cpu() - lse_ref.reshape(-1)).abs().max()) <= 1e-4
    leaves = [x.requires_grad_() for x in dev]
    up = inp["dO"].repeat(b, *[1] * (inp["dO"].dim() - 1)).cuda()
    out = universal_attention(*leaves, prune=prune)
    grads = torch.autograd.grad(out, leaves, up.reshape(out.shape))
    for name, x, y in zip(GRADS, grads, grads_ref):
        assert torch.equal(x, x[:1].expand_as(x)), name
        bar = key_gradient_bar(inp, torch.float32, y) if name == "dkc" else TOL[torch.float32]
        assert rel_err(x[:1], y) <= bar, name
