"""The host module (csrc/ua_host.cpp): every entry point through it against the dense float64 oracle, with the layouts it
hands to the kernels without copies (sequence-major projections, a fused gate tensor, r-major heads, strided upstream)."""
import pytest
import torch

from oracle import ua_oracle as orc
from tests.util import TOL, dense_reference, key_gradient_bar, rel_err

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("entry", ["universal", "universal2d", "decoder", "gen2"])
@pytest.mark.parametrize("b,h,r,L,d,dtype,gates", [(2, 2, 2, 96, 64, BF, BF), (1, 3, 1, 131, 80, BF, F32), (2, 1, 4, 33, 24, BF, F32),
                                                   (1, 2, 2, 160, 64, F32, F32), (1, 2, 1, 1, 16, BF, BF)])
def test_entry_points_through_the_host_module_match_the_oracle(entry, b, h, r, L, d, dtype, gates):
    from universal_attention_triton_amd import _lib, ops
    print("case", entry, b, h, r, L, d, dtype, gates, flush=True)
    inp = orc.make_inputs(b, h, r, L, d, L, dtype=dtype, seed=71)
    for k in ("static_src", "static_dest"):
        inp[k] = inp[k].to(gates)
    O_ref, _, g_ref = dense_reference(inp)
    k4, v4, q5, dO = inp["kc"][:, :, 0], inp["vc"][:, :, 0], inp["xq"], inp["dO"]
    src, dest = inp["static_src"].reshape(b, h, L), inp["static_dest"].reshape(b, h, L)
    host = ops.native()
    assert host is _lib.host()
    leaf = lambda t: t.contiguous().cuda().requires_grad_()
    if entry == "decoder":
        args = [leaf(q5.flatten(1, 2).transpose(1, 2)), leaf(k4.transpose(1, 2)), leaf(v4.transpose(1, 2)),
                leaf(torch.stack([src, dest]).permute(1, 3, 0, 2).reshape(b, L, 2 * h))]
        out = host.decoder(*args, False, False)[0]
        up = dO.flatten(1, 2).transpose(1, 2).cuda()                  # a view: not contiguous
        g = torch.autograd.grad(out, args, up)
        gs = g[3].view(b, L, 2, h).permute(2, 0, 3, 1)
        got = [out.transpose(1, 2), g[1].transpose(1, 2), g[2].transpose(1, 2), g[0].transpose(1, 2), gs[0], gs[1]]
    elif entry == "gen2":
        args = [leaf(q5.transpose(1, 2).flatten(1, 2)), leaf(k4), leaf(v4), leaf(src), leaf(dest)]
        out = host.gen2(*args, True)[0]
        up = dO.transpose(1, 2).flatten(1, 2).cuda()
        g = torch.autograd.grad(out, args, up)
        back = lambda t: t.unflatten(1, (r, h)).transpose(1, 2)
        got = [back(out), g[1], g[2], back(g[0]), g[3], g[4]]
    else:
        q = q5 if entry == "universal" else q5.unflatten(3, (1, L))
        gate = torch.stack([src, dest], -1).cuda()                    # gates as strided views of one tensor
        args = [leaf(inp["kc"]), leaf(inp["vc"]), leaf(q), gate[..., 0].detach().requires_grad_(), gate[..., 1].detach().requires_grad_()]
        out = host.universal(*args, False, False, True)[0]
        g = torch.autograd.grad(out, args, dO.reshape(q.shape).cuda())
        got = [out, g[0], g[1], g[2], g[3], g[4]]
    bar = key_gradient_bar(inp, dtype, g_ref[0]) if L > 1 else 1.0
    assert rel_err(got[0].reshape(O_ref.shape), O_ref) <= TOL[dtype]
    for name, x, y in zip(("kc", "vc", "xq", "src", "dest"), got[1:], g_ref):
        if L == 1 and name != "vc":          # exactly zero in the oracle: rounding noise of dP - delta here
            assert float(x.float().abs().max()) <= 1e-2
            continue
        assert rel_err(x.reshape(y.shape), y) <= (bar if name == "kc" else TOL[dtype]), (name, rel_err(x.reshape(y.shape), y))


def test_host_module_leaves_what_it_does_not_take_to_the_general_path():
    """None for other dtypes, shapes that do not match and tensors off the GPU; a graph recorded through the backward ends in
    a clear error, as in the general path."""
    from universal_attention_triton_amd import ops
    from universal_attention_triton_amd.universal_attention import universal_attention
    dev = [orc.make_inputs(1, 2, 1, 64, 32, 64, dtype=BF, seed=3)[k].cuda() for k in ("kc", "vc", "xq", "static_src", "static_dest")]
    host = ops.native()
    assert host.universal(*[t.cpu() for t in dev], False, False, True) is None
    assert host.universal(*[t.half() for t in dev], False, False, True) is None
    assert host.universal(dev[0], dev[1], dev[2][:, :, :, :32], dev[3], dev[4], False, False, True) is None
    with pytest.raises(ValueError):
        universal_attention(dev[0], dev[1], dev[2][:, :, :, :32], dev[3], dev[4])
    leaves = [t.requires_grad_() for t in dev]
    O = universal_attention(*leaves)
    g = torch.autograd.grad(O.float().sum(), leaves, create_graph=True)
    with pytest.raises(RuntimeError, match="not differentiable"):
        g[2].float().sum().backward()
