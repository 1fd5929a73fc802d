"""The routers' rounds of arg-max where they can go wrong: equal scores, every expert picked, more than one flush of 64
picks (renormalised after the fact instead of in the flush), expert counts around the 64 lanes."""
import numpy as np
import pytest
import torch

from oracle import moe as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("tokens,experts,topk", [(1, 1, 1), (3, 63, 8), (2, 64, 64), (5, 65, 65), (3, 130, 70), (1, 1024, 8)])
def test_router_edges(dev, softmax, tokens, experts, topk):
    import sglang_amd as sa

    g = torch.Generator().manual_seed(experts + topk)
    logits = torch.randn(tokens, experts, generator=g)
    if experts > 4:
        logits[0] = torch.randint(0, 3, (experts,), generator=g).float()  # many equal scores: the lower expert first
    w = torch.empty(tokens, topk, device=dev)
    ids = torch.empty(tokens, topk, device=dev, dtype=torch.int32)
    if softmax:
        sa.topk_softmax(w, ids, logits.to(dev), True)
        rw, ri = om.topk_softmax(logits, topk, True)
    else:
        sa.topk_sigmoid(w, ids, logits.to(dev), True)
        rw, ri = om.topk_sigmoid(logits, topk, True)
    assert np.array_equal(ids.cpu().numpy(), np.asarray(ri))
    assert torch.allclose(w.cpu(), torch.as_tensor(np.asarray(rw)), rtol=1e-5, atol=1e-7)
