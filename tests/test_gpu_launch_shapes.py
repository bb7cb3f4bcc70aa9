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


# one, two, eight and ten row batches per selection work-group, with
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


# row blocks of 1, 2 and 4 per wave; cluster counts around the 32-centroid
# blocks and 512-centroid chunks; rows that end inside a block
@pytest.mark.parametrize("H,N,C", [(1, 33, 1), (2, 1000, 31), (3, 4097, 513), (16, 16450, 100),
                                   (4, 262500, 40), (2, 3000, 2048)])
def test_fast_assign_rank32_equals_general_form(dev, H, N, C):
    """D = 32 has its own kernel; zero dims appended change no sum, so the
    general kernel at D = 64 must give the same labels, bit for bit."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N + C)
    x = torch.randn(H, N, 32, generator=gen, device=dev).half()
    cen = torch.randn(H, C, 32, generator=gen, device=dev).half()
    if C > 30:
        cen[:, 7] = cen[:, 29]               # equal distances: the lowest index wins
        x[:, :20] = cen[:, 10:30]            # distance zero, of either sign
        x[:, 21, 3] = float("inf")
        x[:, 22, 5] = float("nan")
        x[:, 23] = 60000.0
    pad = lambda t: torch.cat([t, torch.zeros_like(t)], 2).contiguous()  # noqa: E731
    want = ops.fast_assign_labels(pad(x), pad(cen))
    assert torch.equal(ops.fast_assign_labels(x, cen), want)


@pytest.mark.parametrize("H,N,C", [(2, 3001, 7), (3, 5000, 2048)])
def test_lloyd_equals_separate_calls(dev, H, N, C):
    """The in-place iterations (labels seeded by the previous ones) against
    assign, update and cast called one by one."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N)
    x = torch.randn(H, N, 32, generator=gen, device=dev).half()
    cen = torch.randn(H, C, 32, generator=gen, device=dev).half()
    cen[:, 3] = 100.0                        # an empty cluster
    want = cen.clone()
    for _ in range(3):
        lab = ops.fast_assign_labels(x, want)
        want = ops.fused_update_vstats(x, lab, want)[0].half()
    assert torch.equal(ops.lloyd(x, cen.clone(), 3), want)
    assert torch.equal(ops.lloyd(x, cen.clone(), 0), cen)


# rows that end inside a staged step and a k-step, several splits, the element
# path (D not 128, unaligned or odd strides), a token-major view
@pytest.mark.parametrize("H,N,D,view", [(1, 3, 128, ""), (2, 257, 128, ""), (3, 5001, 128, "token"),
                                        (2, 700, 128, "odd"), (2, 300, 100, ""), (1, 65, 16, "")])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gram_strided(dev, H, N, D, view, dtype):
    """fp64 Gram of every layout; products of fp16 values are exact, so only
    the order of the fp64 sum differs from the reference's."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N + D)
    x = torch.randn(H, N, D, generator=gen, device=dev).to(dtype)
    if view == "token":
        x = x.transpose(0, 1).contiguous().transpose(0, 1)
    elif view == "odd":
        x = torch.nn.functional.pad(x, (3, 2))[:, :, 3:3 + D]
    flag = torch.full((H,), -1, dtype=torch.int32, device=dev)
    G = ops.gram_strided(x, flag)
    xd = x.half().double().cpu()
    want = xd.transpose(1, 2) @ xd / N
    bound = 2.0 ** -52 * N * (xd.abs().transpose(1, 2) @ xd.abs() / N)
    assert bool(((G.cpu() - want).abs() <= bound).all())
    assert torch.equal(G, G.transpose(1, 2)) and not flag.any()
    x[H - 1, N - 1, D - 1] = float("-inf")
    ops.gram_strided(x, flag)
    assert flag.tolist() == [0] * (H - 1) + [1]


@pytest.mark.parametrize("D", [8, 100, 128])
def test_projection_fit_forms(dev, D):
    """The Cholesky form against the square-root form on the same Grams (fp64,
    up to the sign of a column pair), and its fall-back to the latter."""
    from token2tile_amd import deploy_step as DS, ops
    gen = torch.Generator(device=dev).manual_seed(D)
    q, k = (torch.randn(3, 2000, D, generator=gen, device=dev) / D ** 0.5
            * torch.linspace(0.2, 3.0, D, device=dev) for _ in range(2))
    Mq, Mk = (ops.gram_strided(t.half()) for t in (q, k))
    small = torch.empty(2, 3, dtype=torch.int32, device=dev)
    L = ops.fit_chol(Mq, Mk, 1e-8, small)
    assert not small.any()
    assert float((L @ L.transpose(1, 2) - Mk).abs().max()) <= 1e-13 * float(Mk.abs().max())
    r = min(32, D)
    a, b = DS._fit_chol(Mq, Mk, L, r), DS._fit_eigh(Mq, Mk, r)
    sign = (a[0] * b[0]).sum(1, keepdim=True).sign()
    for x, y in zip(a, b):
        assert float((x * sign - y).abs().max()) <= 1e-7 * float(y.abs().max())
    Mq[1, :, 0] = Mq[1, 0, :] = 0.0            # a zero eigenvalue in one head of q
    Mk[2, -1, :] = Mk[2, :, -1] = 0.0
    Mk[2, -1, -1] = 1e-9                       # and one under the floor in one of k
    ops.fit_chol(Mq, Mk, 1e-8, small)
    assert small.tolist() == [[0, 1, 0], [0, 0, 1]]
    qz = q.half().clone()
    qz[:, :, 0] = 0                            # the operator takes the other form
    Uq, Uk = DS.online_u(qz, k.half(), r)
    Eq, Ek = DS._fit_eigh(*(ops.gram_strided(t) for t in (qz, k.half())), r)
    assert torch.equal(Uq, Eq.float()) and torch.equal(Uk, Ek.float())


def test_projection_fit_of_a_head_ignores_its_neighbours(dev):
    """A head with a dead channel takes the square-root form alone: the heads
    beside it get, bit for bit, what they get without it."""
    from token2tile_amd import deploy_step as DS, ops
    gen = torch.Generator(device=dev).manual_seed(7)
    q, k = (torch.randn(5, 3000, 128, generator=gen, device=dev).half() for _ in range(2))
    qz, kz = q.clone(), k.clone()
    qz[1, :, 9] = 0
    kz[4, :, 100] = 0
    plain, mixed = DS.online_u(q, k), DS.online_u(qz, kz)
    same, low = [0, 2, 3], [1, 4]
    E = DS._fit_eigh(*(ops.gram_strided(t)[low] for t in (qz, kz)), 32)
    for a, b, e in zip(plain, mixed, E):
        assert torch.equal(a[same], b[same]) and torch.equal(b[low], e.float())


# row blocks per wave 4, 2 and 1 (rows in whole, partial and single chunks; a head
# alone and the last shape with two centroid groups), the key pass sharing the first query pass's launches with more and fewer clusters
@pytest.mark.parametrize("H,N,CQ,CK,pin", [(8, 131100, 200, 2048, 0), (16, 16450, 33, 500, 77),
                                           (3, 4097, 4096, 64, 0), (40, 1030, 65, 600, 0),
                                           (2, 255, 7, 31, 255)])
def test_kmeans_of_many_heads_equals_each_head_alone(dev, H, N, CQ, CK, pin):
    """A head's clustering does not depend on how many heads share the launch,
    so the launch shapes that follow H N agree bit for bit with the smallest;
    the sort and the query means are checked against torch on the labels."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).half()  # noqa: E731
    QU, KU, V = r(H, N, 32), r(H, N, 32), r(H, N, 128)
    cq0, ck0 = r(H, CQ, 32), r(H, CK, 32)
    cq0[:, 0] = 50.0                                    # an empty cluster
    lab0 = lambda n: torch.zeros(n, N, dtype=torch.int32, device=dev)  # noqa: E731
    o = ops.kmm_run(QU, KU, V, cq0, ck0, pin_tail=pin, out=dict(qlab=lab0(H), klab=lab0(H)))
    for h in range(0, H, max(1, H // 3)):
        one = ops.kmm_run(*(t[h:h + 1].contiguous() for t in (QU, KU, V, cq0, ck0)), pin_tail=pin,
                          out=dict(qlab=lab0(1), klab=lab0(1)))
        for name, t in one.items():
            assert torch.equal(t[0], o[name][h]), name
        for lab, perm, counts, C in ((o["qlab"], o["qperm"], o["qcounts"], CQ),
                                     (o["klab"], o["kperm"], o["kcounts"], CK)):
            assert torch.equal(perm[h].long(), torch.sort(lab[h], stable=True).indices)
            assert torch.equal(counts[h].long(), torch.bincount(lab[h], minlength=C))
        S = torch.zeros(CQ, 32, dtype=torch.int64, device=dev)
        S.index_add_(0, o["qlab"][h].long(), torch.round(QU[h].float() * 32768.0).long())
        n = o["qcounts"][h].float().unsqueeze(1)
        full = o["qcounts"][h] > 0
        assert torch.equal(o["cq2"][h][full], (S.float() / (32768.0 * n)).half()[full])


# 8, 4, 2 and 1 parts per task at most; unions from empty over one tile and a
# few keys around the least part length to all keys; ragged tasks and tiles
@pytest.mark.parametrize("H,N,CQ", [(1, 2500, 3), (2, 8190, 100), (3, 20011, 201), (5, 32760, 256)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_exact_split_matches_whole_tasks(dev, H, N, CQ, dtype):
    """The split call against the unsplit kernel on the same plan.  Both round
    every weight to the type (a relative u) against a max of their own, so each
    is within u (sum w |v| / sum w + |o|) of the exact result, and rounds the
    output once more.  (fp16 scores stay small: no weight is subnormal.)"""
    from token2tile_amd import ops
    rng = np.random.default_rng(N)
    qlab, klab, qperm, qcounts, kperm, kcounts = structure(rng, H, N, CQ)
    density = rng.choice([0.0, 0.002, 0.05, 0.2, 0.7, 1.0], (H, CQ, 1))
    density[:, 0], density[:, 1 % CQ] = 0.0, 1.0
    sel = (rng.random((H, CQ, 2048)) < density).astype(np.uint8)
    unip = np.packbits(sel, axis=2, bitorder="little").view(np.int32)
    gen = torch.Generator(device=dev).manual_seed(N)
    q, k, v = (torch.randn(H, N, 128, generator=gen, device=dev).to(dtype) for _ in range(3))
    q *= 0.5
    if dtype == torch.bfloat16:
        k[:, N // 2] *= 40                    # a score far above the earlier parts' max
    t = lambda a: g(a, dev)                   # noqa: E731
    tq, tk, tu, tqp, tkp, tql = map(t, (qcounts, kcounts, unip, qperm, kperm, qlab))
    plan = ops.tile_plan(tq, tk, tu, N)
    out = [torch.full_like(q, float("nan")) for _ in range(2)]
    lse = [torch.full((H, N), float("nan"), device=dev) for _ in range(2)]
    ops.tile_attn_exact_orig_gather_kv(q, k, v, tkp, tk, tu, tqp, plan, out[0], lse[0])
    ops.tile_attn_exact_split(q, k, v, tkp, tk, tu, tql, tqp, plan, out[1], lse[1])
    # tokens of an even view, as the backend passes them
    qs, ks, vs, os_ = (x.transpose(0, 1).contiguous().transpose(0, 1) for x in (q, k, v, out[1]))
    lse2 = lse[1].clone()
    ops.tile_attn_exact_split(qs, ks, vs, tkp, tk, tu, tql, tqp, plan, os_, lse2)
    assert torch.equal(os_, out[1]) and torch.equal(lse2, lse[1])
    # and the gathered forms, bit for bit
    kp, vp = ops.fast_gather(k, tkp), ops.fast_gather(v, tkp)
    for kk, vv, gather in ((kp, vp, 0), (k, vp, 1)):
        o2 = torch.full_like(q, float("nan"))
        ops.tile_attn_exact_split(q, kk, vv, tkp, tk, tu, tql, tqp, plan, o2, lse2, gather=gather)
        assert torch.equal(o2, out[1]) and torch.equal(lse2, lse[1])
    a, b = (o.float() for o in out)
    mean, lse3 = torch.empty_like(q), torch.empty_like(lse2)
    ops.tile_attn_exact_orig_gather_kv(q, k, v.abs(), tkp, tk, tu, tqp, plan, mean, lse3)
    u = 2.0 ** (-11 if dtype == torch.float16 else -8)   # unit roundoff of 11 and 8 bits
    bound = 4 * u * 1.01 * mean.float() + 2 * u * a.abs() + 1e-6
    assert not a.isnan().any() and bool(((a - b).abs() <= bound).all())
    fin = lse[0].isfinite()
    assert torch.equal(fin, lse[1].isfinite())
    assert float((lse[0] - lse[1])[fin].abs().max()) <= 2 * u * 1.4427 * 1.01 + 2e-5


def test_step_stages_and_streams(dev):
    """One call's stages in one library call (sharing kernels), launched stage by
    stage (stage_events) and from another stream: same bits."""
    from token2tile_amd.deploy_step import MaskedStepDeploy
    from token2tile_amd.synth import generate
    H, N, CQ = 2, 3000, 40
    q, k, v = generate(H, N, grid=(1, 1, N), seed=3, device=dev, dtype=torch.bfloat16)
    op = MaskedStepDeploy(H, N, CQ, s_frac=0.05, mask_refresh=4, device=dev)
    state = op.init_state(q, k, seed=1)

    def call(step, **kw):
        op.set_cfg_call(0, key=0, step=step)
        st = dict(state)
        out = op.step(q, k, v, st, **kw).clone()
        return out, st["ck"].clone(), st["cq"].clone()

    full, reuse = call(0), call(1)
    assert torch.equal(reuse[1], state["ck"])
    op.stage_events = []
    staged = call(4), call(5)
    names = [n for n, _, _ in op.stage_events]
    assert names == ["project", "kmeans", "score", "select", "plan", "attention_exact",
                     "attention_prep", "attention_residual", "attention_exact",
                     "attention_residual"]
    op.stage_events = None
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = call(8), call(9)
    torch.cuda.current_stream().wait_stream(side)
    for a, b in (staged, other):
        assert all(torch.equal(x, y) for x, y in zip(full + reuse, a + b))


@pytest.mark.parametrize("with_kmeans", [False, True])
def test_step_stages_run_in_order(dev, with_kmeans):
    """The tile image of a call that also finalises the centroids holds those,
    not the ones that were there before."""
    from token2tile_amd import _lib, ops
    from token2tile_amd.deploy_step import MaskedStepDeploy
    gen = torch.Generator(device=dev).manual_seed(2)
    H, N, CQ = 2, 3000, 20
    q, k, v = (torch.randn(H, N, 128, generator=gen, device=dev).half() for _ in range(3))
    op = MaskedStepDeploy(H, N, CQ, device=dev)
    state = op.init_state(q, k, seed=1)
    first = dict(state)
    op._ctiles.zero_()                       # (its rows are padded)
    op.step(q, k, v, state)
    want = op._ctiles.clone()
    a, last = op._own_args(), op._last
    cks, ck16 = torch.zeros_like(last["cks"]), torch.zeros_like(last["cks"])
    cq2 = torch.empty_like(state["cq"])
    kcounts, kperm, qcounts, qperm = (last[n].clone() for n in ("counts", "kperm", "tile_sizes", "qperm"))
    a.v, a.v_head_stride, a.v_row_stride = v.data_ptr(), N * 128, 128
    for name, t in (("kcounts", kcounts), ("kperm", kperm), ("qcounts", qcounts), ("qperm", qperm),
                    ("cks", cks), ("ck16", ck16), ("cq2", cq2), ("cq0", first["cq"]), ("ck0", first["ck"])):
        setattr(a, name, t.data_ptr())
    op._ctiles.zero_()
    stages = _lib.STEP_VSTATS | _lib.STEP_FINALIZE | _lib.STEP_TILES
    assert _lib.lib().t2t_step(a, stages | (_lib.STEP_KMEANS if with_kmeans else 0),
                               _lib.stream_handle()) == 0
    assert torch.equal(cks, last["cks"]) and torch.equal(op._ctiles, want)


# one wave's sort, strides across waves, several keys per thread, more clusters
# than key clusters, and a list past the sort's limit (cluster order)
@pytest.mark.parametrize("H,N,CQ,kind", [(2, 5000, 1, "mix"), (2, 9000, 65, "mix"),
                                         (3, 20000, 513, "mix"), (1, 30000, 2049, "mix"),
                                         (1, 40000, 4096, "mix"), (1, 60000, 4096, "full")])
def test_plan_order(dev, H, N, CQ, kind):
    from token2tile_amd import ops
    rng = np.random.default_rng(CQ)
    lab = np.minimum(rng.integers(0, CQ, (H, N)), rng.integers(0, CQ, (H, N)))
    if kind == "full":                         # every cluster, a few of them long
        lab[:, :CQ] = np.arange(CQ)
        lab[:, CQ:CQ + 3000] = 7
    qcounts = np.stack([np.bincount(x, minlength=CQ) for x in lab]).astype(np.int32)
    kcounts = np.stack([np.bincount(rng.integers(0, 2048, N) // 2 * 2, minlength=2048)
                        for _ in range(H)]).astype(np.int32)
    sel = rng.random((H, CQ, 2048)) < rng.choice([0.0, 0.05, 0.05, 1.0], (H, CQ, 1))
    unip = np.packbits(sel.astype(np.uint8), axis=2, bitorder="little").view(np.int32)
    plan = ops.tile_plan(g(qcounts, dev), g(kcounts, dev), g(unip, dev), N)
    pv = {k: c(v) for k, v in ops.plan_views(plan, H, N, CQ).items()}
    for h in range(H):
        assert np.array_equal(pv["k_off"][h], np.concatenate([[0], np.cumsum(kcounts[h])]))
        kv = np.where(qcounts[h] > 0, sel[h] @ kcounts[h], 0)
        assert np.array_equal(pv["kvlen"][h], kv)
        tasks, start = [], 0
        for t, n in enumerate(qcounts[h]):
            nt, nw = -(-n // 128), -(-n // 32)
            s = start
            for i in range(nt):
                rows = min(32 * (nw // nt + (i < nw % nt)), start + n - s)
                big = 32 * (nw // nt + (nw % nt > 0))
                tasks.append((t, s, rows, big))
                s += rows
            start += n
        if len(tasks) <= 4096:
            tasks.sort(key=lambda x: -min(x[3] * int(kv[x[0]]), 2 ** 32 - 1))  # stable
        else:
            assert kind == "full"
        assert pv["ntask"][h] == len(tasks)
        assert np.array_equal(pv["tasks"][h][:len(tasks)], np.array(tasks))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_residual_groups(dev, dtype):
    """288 work-groups walk all centroid tiles; a head alone has 32, whose two
    wave groups share them.  Both round every weight to fp16 (a relative u)
    against a max of their own, so each is within u (sum w |v| / sum w + |o|)
    of the exact sums, and rounds the output once more."""
    from token2tile_amd import ops
    H, N, CQ = 9, 4000, 50
    rng = np.random.default_rng(5)
    qlab, _, qperm, qcounts, _, kcounts = structure(rng, H, N, CQ)
    density = rng.choice([0.0, 0.1, 0.9, 1.0], (H, CQ, 1))
    sel = (rng.random((H, CQ, 2048)) < density).astype(np.uint8)
    sel[0, :, 1024:] = 1                       # nothing outside the union in the second half
    unip = np.packbits(sel, axis=2, bitorder="little").view(np.int32)
    gen = torch.Generator(device=dev).manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)  # noqa: E731
    QU, cks, sumv = r(H, N, 32).half(), (0.1 * r(H, 2048, 32)).half(), r(H, 2048, 128).half()
    exact, lse = r(H, N, 128).to(dtype), 9.0 + r(H, N)
    lam, tw = torch.linspace(1, 2, H, device=dev), torch.tensor(0.7, device=dev)
    tk, tu, tl, tp = g(kcounts, dev), g(unip, dev), g(qlab, dev), g(qperm, dev)

    def merge(x, s, hs):
        o = x[hs].clone()
        tiles = ops.centroid_tiles(cks[hs].contiguous(), s[hs].contiguous())
        return ops.resid_merge_inplace(o, lse[hs].contiguous(), QU[hs].contiguous(), tiles, tk[hs],
                                       tu[hs], tl[hs], tp[hs], lam[hs], tw)
    every = slice(0, H)
    a, mean = merge(exact, sumv, every), merge(exact.abs(), sumv.abs(), every)
    b = torch.cat([merge(exact, sumv, slice(h, h + 1)) for h in range(H)])
    u = 2.0 ** -11
    bound = 4 * u * 1.01 * mean.float() + 2.0 ** (-10 if dtype == torch.float16 else -7) * a.float().abs() + 1e-6
    assert not a.isnan().any() and bool(((a - b).float().abs() <= bound).all())


# parts added by the combine (fewer than 256 row blocks) and by the residual
# (from 256 on, with two wave groups and with one)
@pytest.mark.parametrize("H,N,CQ", [(1, 4100, 16), (2, 16384, 100), (3, 20011, 201)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_split_call_equals_its_stages(dev, H, N, CQ, dtype):
    """run_planned, which may leave the parts to the residual, against the split
    exact attention (always combined) and the residual one by one: same bits."""
    from token2tile_amd import ops
    rng = np.random.default_rng(N)
    qlab, klab, qperm, qcounts, kperm, kcounts = structure(rng, H, N, CQ)
    density = rng.choice([0.0, 0.01, 0.3, 1.0], (H, CQ, 1))
    sel = (rng.random((H, CQ, 2048)) < density).astype(np.uint8)
    unip = np.packbits(sel, axis=2, bitorder="little").view(np.int32)
    gen = torch.Generator(device=dev).manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)  # noqa: E731
    q, kp, vp = (r(H, N, 128).to(dtype) for _ in range(3))
    QU, cks, sumv = r(H, N, 32).half(), (0.1 * r(H, 2048, 32)).half(), r(H, 2048, 128).half()
    lam, tw = torch.linspace(1, 2, H, device=dev), torch.tensor(1.0, device=dev)
    tq, tk, tu, tqp, tql = (g(a, dev) for a in (qcounts, kcounts, unip, qperm, qlab))
    plan = ops.tile_plan(tq, tk, tu, N)
    a, b = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    lse = torch.empty(H, N, device=dev)
    ops.tile_attn_exact_split(q, kp, vp, None, tk, tu, tql, tqp, plan, a, lse, gather=0)
    ops.resid_merge_inplace(a, lse, QU, ops.centroid_tiles(cks, sumv), tk, tu, tql, tqp, lam, tw)
    ops.tile_attn_run_planned(q, kp, vp, tq, tk, tu, QU, cks, sumv, lam, tql, tqp, tw, b, plan, False)
    assert not a.isnan().any() and torch.equal(a, b)


# parts added by the combine and by the residual
@pytest.mark.parametrize("H,N,CQ", [(1, 4100, 16), (3, 12000, 60)])
def test_split_call_on_a_kept_plan(dev, H, N, CQ):
    """A plan serves the query clusters it was built for whatever the union is
    now (it orders and cuts the queries): lengths that grew, shrank to less than
    a tile per part or to nothing.  Bounds as between split and whole tasks."""
    from token2tile_amd import ops
    rng = np.random.default_rng(N)
    qlab, klab, qperm, qcounts, kperm, kcounts = structure(rng, H, N, CQ)
    dens = rng.choice([0.0, 0.002, 0.3, 1.0], (2, H, CQ, 1))
    dens[0, :, :4], dens[1, :, :4] = [[0.0], [1.0], [1.0], [1.0]], [[1.0], [0.0], [0.001], [0.05]]
    dens[1, :, 2] = 0.0
    sel = (rng.random((2, H, CQ, 2048)) < dens).astype(np.uint8)
    sel[1, :, 2, 0] = 1                        # a single cluster, of at most a few keys
    was, now = (g(np.packbits(x, axis=2, bitorder="little").view(np.int32), dev) for x in sel)
    gen = torch.Generator(device=dev).manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)  # noqa: E731
    q, kp, vp = (r(H, N, 128).half() for _ in range(3))
    q *= 0.5
    QU, cks, sumv = r(H, N, 32).half(), (0.1 * r(H, 2048, 32)).half(), r(H, 2048, 128).half()
    lam, tw = torch.linspace(1, 2, H, device=dev), torch.tensor(1.0, device=dev)
    tq, tk, tqp, tql = (g(a, dev) for a in (qcounts, kcounts, qperm, qlab))
    plan = ops.tile_plan(tq, tk, was, N)
    new = lambda: (torch.full_like(q, float("nan")), torch.full((H, N), float("nan"), device=dev))  # noqa: E731
    (a, la), (b, lb), (m, lm) = new(), new(), new()
    ops.tile_attn_exact_orig(q, kp, vp, tk, now, tqp, plan, a, la)
    ops.tile_attn_exact_orig(q, kp, vp.abs(), tk, now, tqp, plan, m, lm)
    ops.tile_attn_exact_split(q, kp, vp, None, tk, now, tql, tqp, plan, b, lb, gather=0)
    u = 2.0 ** -11
    assert not a.isnan().any() and not b.isnan().any()
    assert bool(((a - b).float().abs() <= 4.04 * u * m.float() + 2 * u * a.float().abs() + 1e-6).all())
    fin = la.isfinite()
    assert not fin.all() and torch.equal(la[~fin], lb[~fin])
    assert float((la - lb)[fin].abs().max()) <= 2 * u * 1.4427 * 1.01 + 2e-5
    ops.resid_merge_inplace(b, lb, QU, ops.centroid_tiles(cks, sumv), tk, now, tql, tqp, lam, tw)
    c2, _ = new()
    ops.tile_attn_run_planned(q, kp, vp, tq, tk, now, QU, cks, sumv, lam, tql, tqp, tw, c2, plan, False)
    assert torch.equal(c2, b)


# parts added by the combine, and by the residual
@pytest.mark.parametrize("H,N,CQ", [(1, 4100, 16), (3, 12000, 60)])
def test_attention_without_room_for_parts(dev, H, N, CQ):
    """A workspace of lse and the tile image alone, as one sized for a longer
    sequence may be, serves a small call unsplit: the bits of the whole-task
    kernel and the residual after it."""
    from token2tile_amd import _lib, ops
    rng = np.random.default_rng(N)
    qlab, klab, qperm, qcounts, kperm, kcounts = structure(rng, H, N, CQ)
    sel = (rng.random((H, CQ, 2048)) < 0.3).astype(np.uint8)
    unip = np.packbits(sel, axis=2, bitorder="little").view(np.int32)
    gen = torch.Generator(device=dev).manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)  # noqa: E731
    q, kp, vp = (r(H, N, 128).half() for _ in range(3))
    QU, cks, sumv = r(H, N, 32).half(), (0.1 * r(H, 2048, 32)).half(), r(H, 2048, 128).half()
    lam, tw = torch.linspace(1, 2, H, device=dev), torch.tensor(1.0, device=dev)
    tq, tk, tu, tqp, tql = (g(a, dev) for a in (qcounts, kcounts, unip, qperm, qlab))
    plan = ops.tile_plan(tq, tk, tu, N)
    a, lse = torch.full_like(q, float("nan")), torch.empty(H, N, device=dev)
    ops.tile_attn_exact_orig(q, kp, vp, tk, tu, tqp, plan, a, lse)
    one = torch.full_like(q, float("nan"))
    lse1 = torch.empty_like(lse)
    assert ops.attn_split_ws_bytes(H, N, CQ) > 0
    hs = N * 128
    for ws, size in ((None, 0), (torch.empty(256, dtype=torch.uint8, device=dev), 256)):
        one.fill_(float("nan"))
        _lib.call("t2t_tile_attn_exact_split", q, hs, 128, kp, hs, 128, vp, hs, 128, None, 0, 0, tk, tu,
                  tql, tqp, plan, one, hs, 128, lse1, H, N, CQ, ws, size, _lib.stream_handle())
        assert torch.equal(one, a) and torch.equal(lse1, lse)
    ops.resid_merge_inplace(a, lse, QU, ops.centroid_tiles(cks, sumv), tk, tu, tql, tqp, lam, tw)
    size = -(-H * N * 4 // 256) * 256 + ops.size_query("t2t_centroid_tiles_bytes", H)
    assert size < ops.attn_ws_bytes(H, N, q.dtype)
    ws = torch.empty(size + 512, dtype=torch.uint8, device=dev)
    ws[size:] = 77
    for rebuild in (True, False):
        b = torch.full_like(q, float("nan"))
        ops.tile_attn_run_planned(q, kp, vp, tq, tk, tu, QU, cks, sumv, lam, tql, tqp, tw, b, plan,
                                  rebuild, ws=ws[:size])
        assert not a.isnan().any() and torch.equal(a, b)
    assert bool((ws[size:] == 77).all())


@pytest.mark.parametrize("H,N,C", [(2, 1000, 33), (1, 300, 2048)])
def test_update_leaves_foreign_labels_out(dev, H, N, C):
    """Rows labelled outside [0, C) belong to no cluster (the checked call raises
    from the counts' sum): means and counts are those of the other rows."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(N)
    x = torch.randn(H, N, 32, generator=gen, device=dev).half()
    v = torch.randn(H, N, 128, generator=gen, device=dev).bfloat16()
    old = torch.randn(H, C, 32, generator=gen, device=dev).half()
    lab = torch.randint(0, C, (H, N), generator=gen, device=dev, dtype=torch.int32)
    bad = lab.clone()
    bad[:, 5::7], bad[:, 6::70], bad[:, 8::90] = -1, C, 2 ** 31 - 1
    for h in range(H):
        ok = ((bad[h] >= 0) & (bad[h] < C)).nonzero().flatten()
        args = (x[h:h + 1], bad[h:h + 1], old[h:h + 1], v[h:h + 1])
        part = (x[h:h + 1, ok], bad[h:h + 1, ok], old[h:h + 1], v[h:h + 1, ok])
        for half in (False, True):
            got = ops.fused_update_vstats(*args, check_labels=False, half=half)
            want = ops.fused_update_vstats(*(t.contiguous() for t in part), half=half)
            assert all(torch.equal(a, b) for a, b in zip(got, want))
        with pytest.raises(ValueError, match="labels"):
            ops.fused_update_vstats(*args)


def test_calls_on_a_stream_allocate_there(dev, monkeypatch):
    """Scratch and outputs of a call on another stream come from that stream's
    memory: the current stream's may still be in use by its earlier work, and
    would go back to it while the call runs."""
    from token2tile_amd import ops
    gen = torch.Generator(device=dev).manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev).half()  # noqa: E731
    H, N, CQ, rng = 2, 4096, 16, np.random.default_rng(1)
    x, q, k, v, old = r(H, N, 32), r(H, N, 128), r(H, N, 128), r(H, N, 128), r(H, 64, 32)
    qlab, _, qperm, qcounts, kperm, kcounts = structure(rng, H, N, CQ)
    tq, tk, tp, tl, tkp = (g(a, dev) for a in (qcounts, kcounts, qperm, qlab, kperm))
    unip = torch.full((H, CQ, 64), -1, dtype=torch.int32, device=dev)
    plan = ops.tile_plan(tq, tk, unip, N)
    M, small = ops.gram_strided(q), torch.empty(2, H, dtype=torch.int32, device=dev)
    want = (ops.lloyd(x, old.clone(), 2), M, ops.fit_chol(M, M, 1e-8, small),
            ops.tile_attn_exact_split(q, k, v, tkp, tk, unip, tl, tp, plan, torch.empty_like(q),
                                      torch.empty(H, N, device=dev)))
    cen, out, lse = old.clone(), torch.empty_like(q), torch.empty(H, N, device=dev)
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream())
    made, empty = [], torch.empty

    def recorded(*a, **kw):
        made.append(torch.cuda.current_stream().cuda_stream)
        return empty(*a, **kw)
    monkeypatch.setattr(torch, "empty", recorded)
    got = (ops.lloyd(x, cen, 2, stream=side), ops.gram_strided(q, stream=side),
           ops.fit_chol(M, M, 1e-8, small, stream=side),
           ops.tile_attn_exact_split(q, k, v, tkp, tk, unip, tl, tp, plan, out, lse, stream=side))
    monkeypatch.undo()
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert len(made) >= 5 and set(made) == {side.cuda_stream}
