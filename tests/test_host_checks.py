"""Host-side argument checks of the operator surface that run before any
device work (no GPU needed)."""
import threading

import pytest
import torch

from token2tile_amd import deploy_step as DS


def test_online_u_rejects_nonfinite_and_names_heads():
    q = torch.zeros(3, 10, 128)
    q[2, 3, 4] = float("nan")
    q[0, 1, 1] = float("inf")
    with pytest.raises(RuntimeError, match=r"q \(3, 10, 128\) holds 2 non-finite values, in heads \[0, 2\]"):
        DS.online_u(q, torch.zeros_like(q))
    k = torch.zeros(3, 10, 128)
    k[1, 0, 0] = float("-inf")
    with pytest.raises(RuntimeError, match=r"online_u: k .* in heads \[1\]"):
        DS.online_u(torch.zeros_like(k), k)


def test_fused_update_vstats_rejects_unsupported_widths():
    lab = torch.zeros(1, 8, dtype=torch.int32)
    with pytest.raises(ValueError, match="ku must be"):
        DS.fused_update_vstats(torch.zeros(1, 8, 16, dtype=torch.float16), lab,
                               torch.zeros(1, 4, 16, dtype=torch.float16))
    with pytest.raises(ValueError, match="v must be"):
        DS.fused_update_vstats(torch.zeros(1, 8, 32, dtype=torch.float16), lab,
                               torch.zeros(1, 4, 32, dtype=torch.float16),
                               torch.zeros(1, 8, 64, dtype=torch.float16))


def test_eigh_robust_matches_eigh_on_host():
    a = torch.randn(2, 6, 6, dtype=torch.float64)
    m = a @ a.transpose(1, 2)
    e, v = DS._eigh_robust(m)
    assert torch.allclose(v @ torch.diag_embed(e) @ v.transpose(1, 2), m, atol=1e-10)


# a full-rank Gram, and few effective dimensions beside one large channel, every
# Gram eigenvalue far above the floor of 1e-8
@pytest.mark.parametrize("rank,channel,rest", [(128, 0.0, 0.5), (2, 1000.0, 0.01),
                                               (1, 30000.0, 0.01)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_projection_fit_of_graded_inputs(rank, channel, rest, dtype):
    """However the singular values are graded, the Cholesky form's score products
    are as near to the scores as the square-root form's, and fp16 holds its
    projections and the projected rows.  (Both take V from an eigensolution of
    M^T M, which resolves singular values down to sqrt(eps) = 1.5e-8 of the
    largest: that much is allowed beside the truncation.)"""
    gen = torch.Generator().manual_seed(rank)
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    basis = 0.5 * r(rank, 128)
    x = [r(2000, rank) @ basis + rest * r(2000, 128) for _ in range(2)]
    for t in x:
        t[:, 7] += channel
    q, k = (t.to(dtype).half().double().unsqueeze(0) for t in x)
    Mq, Mk = (t.transpose(1, 2) @ t / 2000 for t in (q, k))
    assert min(float(torch.linalg.eigvalsh(M).min()) for M in (Mq, Mk)) > 1e-5
    Uq, Uk = DS._fit_chol(Mq, Mk, torch.linalg.cholesky(Mk), 32)
    for t, U in ((q, Uq), (k, Uk)):
        assert bool(U.half().isfinite().all())
        assert bool((t @ U.half().double()).half().isfinite().all())
    S = q @ k.transpose(1, 2)
    err = lambda a, b: float(((q @ a) @ (k @ b).transpose(1, 2) - S).norm() / S.norm())  # noqa: E731
    assert err(Uq, Uk) <= 1.1 * err(*DS._fit_eigh(Mq, Mk, 32)) + 1.5e-8


def test_a_call_runs_under_its_own_device(monkeypatch):
    """Whatever form a call takes, all of it runs with the object's GPU current."""
    inside = []

    class Guard:
        def __init__(self, device):
            self.device = device

        def __enter__(self):
            inside.append(self.device)

        def __exit__(self, *exc):
            inside.pop()

    monkeypatch.setattr(torch.cuda, "device", Guard)
    op = DS.MaskedStepDeploy.__new__(DS.MaskedStepDeploy)
    op.dev, op._lock = torch.device("cuda", 1), threading.Lock()
    op._step = lambda *a: (list(inside), a)
    seen, args = op.step("q", "k", "v", "state")
    assert seen == [op.dev] and args == ("q", "k", "v", "state", None) and not inside
