"""GPU parity of the GDN recurrent step on both sides of its kernel choice: 256, 512 and 2560 workgroups (sequences x value
heads) of one token, and several tokens, which take the column kernel at every size. Tolerances as test_gpu_gdn.py."""
import pytest
import torch

import test_gpu_gdn
import test_gpu_layer
from axk import configs, gdn, layer
from oracle import gdn as ogdn
from oracle import layer as olayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("bsz,t,nk,nv", [(16, 1, 16, 16), (257, 1, 1, 1), (32, 1, 8, 16), (27, 1, 1, 19),
                                         (18, 2, 16, 32), (80, 1, 16, 32), (2561, 1, 1, 1)])
def test_gdn_workgroup_counts(dev, bsz, t, nk, nv, inplace):
    g = torch.Generator().manual_seed(bsz + t)
    c = configs.gdn_inputs(bsz, t, g, nk=nk, nv=nv, state_std=0.05)
    c["a_log"] = torch.randn(nv, generator=g) * 0.5
    c["dt_bias"] = torch.randn(nv, generator=g) * 0.5
    out, st = test_gpu_gdn._run(c, dev, inplace)
    o32, s32 = ogdn.gdn_fp32(*test_gpu_gdn._args(c))
    torch.testing.assert_close(out.float(), o32.to(torch.bfloat16).float(), **test_gpu_gdn.TOL)
    torch.testing.assert_close(st, s32, rtol=1e-3, atol=1e-4)


@pytest.mark.parametrize("over", ["q", "k", "v"])
@pytest.mark.parametrize("bsz,t", [(3, 1), (3, 5), (20, 1), (40, 1)])
def test_gdn_output_over_an_input(dev, bsz, t, over):
    """As many key heads as value heads: the output in the place of q, k or v is the output in a tensor of its own, bit
    for bit (each kernel of one token, and several tokens)."""
    g = torch.Generator().manual_seed(bsz + t)
    c = {n: x.to(dev) for n, x in configs.gdn_inputs(bsz, t, g, nk=16, nv=16, state_std=0.05).items()}
    print(f"gdn output over {over} b={bsz} t={t}", flush=True)
    want, state = gdn.gdn_recurrent(*test_gpu_gdn._args(c))
    got, st = gdn.gdn_recurrent(*test_gpu_gdn._args(c), output=c[over])
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(st, state)


# With the output norm and gate: 256, 272, 512 and 544 workgroups. The layer rounds to bf16 some ten times between x and
# its output (2^-9 each, about 6e-3 in the 2-norm if all of them fell differently), and an input of the state that
# rounds the other way moves single elements by more than an elementwise bound allows: hence 1e-2 in the 2-norm.
@pytest.mark.parametrize("b,nk,nv", [(16, 2, 16), (17, 2, 16), (16, 4, 32), (17, 4, 32)])
def test_gdn_layer_workgroup_counts(dev, b, nk, nv):
    w, x, st, cv = test_gpu_layer._gdn_case(b + nk + nv, b, nk, nv)
    w_dev = test_gpu_layer._dev(w, dev)
    out, so, _ = layer.gdn_layer_decode(x.to(dev), w_dev, st.to(dev), cv.to(dev), nk, nv)
    ro, rs, _ = olayer.gdn_layer_decode(x, w, st, cv, nk, nv)
    for got, ref in ((out.float().cpu(), ro.float()), (so.cpu(), rs)):
        assert (got - ref).norm() <= 1e-2 * ref.norm()
