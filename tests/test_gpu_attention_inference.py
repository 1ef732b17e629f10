"""gat_attention under no_grad (or on tensors that want no gradients) keeps nothing for a backward pass, also when its inputs are
parameters: the forward operator alone, no second array of the output's size."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["no_grad", "inference_mode", "detached"])
def test_inference_takes_the_forward_operator(monkeypatch, mode):
    import torch
    from featgraph_amd.autograd import Graph
    from featgraph_amd.module import GraphAttentionhip
    adj = sp.random(3000, 2000, density=0.01, format="csr", random_state=np.random.default_rng(2)).astype("float32")
    H, D = 8, 64
    gen = torch.Generator(device="cuda").manual_seed(1)
    er, el, v = (torch.randn(s, generator=gen, device="cuda").requires_grad_() for s in ((3000, H), (2000, H), (2000, H, D)))
    g = Graph(adj)
    with_grad = g.gat_attention(er, el, v)
    assert with_grad.requires_grad
    monkeypatch.setattr(GraphAttentionhip, "train_forward", lambda *a: pytest.fail("inference took the training pass"))
    if mode == "detached":
        out = g.gat_attention(er.detach(), el.detach(), v.detach())
    else:
        with getattr(torch, mode)():
            out = g.gat_attention(er, el, v)
    assert not out.requires_grad
    assert torch.equal(out, with_grad.detach())
