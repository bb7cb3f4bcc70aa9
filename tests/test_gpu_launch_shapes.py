"""Launch shapes that follow the problem size: every rule that picks a split,
a tile count or a kernel from the sizes is checked on both of its sides, at
the edges, against the general path or the oracle."""
import numpy as np
import pytest
import torch

from oracle import t2t_oracle as O

pytestmark = pytest.mark.gpu


def g(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def c(t):
    return t.detach().cpu().numpy()


def structure(rng, H, N, CQ, CK=2048):
    """Random labels with empty and one-row clusters, their counts and
    stable permutations."""
    qlab = rng.integers(0, max(1, CQ - 1), (H, N)).astype(np.int32)
    klab = (rng.integers(0, CK, (H, N)) // 3 * 3 % CK).astype(np.int32)
    qperm, qcounts = O.stable_perm(qlab, CQ)
    kperm, kcounts = O.stable_perm(klab, CK)
    return qlab, klab, qperm, qcounts, kperm, kcounts


# one, two, seven and sixteen row batches per selection work-group, with
# partial last batches and work-groups
@pytest.mark.parametrize("H,N,CQ", [(1, 2049, 5), (4, 2500, 40), (7, 8161, 64), (19, 8161, 33)])
def test_score_select_batches_match_unfused(dev, H, N, CQ):
    from token2tile_amd import ops
    rng = np.random.default_rng(N)
    _, _, qperm, qcounts, _, kcounts = structure(rng, H, N, CQ)
    QU = g(rng.normal(0, 1, (H, N, 32)).astype(np.float16), dev)
    cks = g((rng.normal(0, 1, (H, 2048, 32)) / 5).astype(np.float16), dev)
    tq, tp, tk = g(qcounts, dev), g(qperm, dev), g(kcounts, dev)
    ns = torch.tensor(N // 20, dtype=torch.int32, device=dev)
    u, r = ops.score_select(QU, cks, tk, tp, tq, ns)
    u2, r2 = ops.select_union(ops.score(QU, cks), tk, tp, tq, ns)
    assert torch.equal(u, u2) and torch.equal(r, r2)
