"""GPU parity of the cross-tokenizer marginalisation and the fused reverse KL against it."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def D():
    import llm_distillery_amd as d
    d._lib.load()
    return d


def _case(R, Vs, Vt, seed, alphabet=4, drop=0.0):
    from llm_distillery_amd import synthetic as S
    import llm_distillery_amd as d
    student = S.random_byte_vocab(Vs, seed, alphabet=alphabet, max_len=6, all_single_bytes=(alphabet == 256))
    teacher = S.random_byte_vocab(Vt, seed + 1, alphabet=alphabet, max_len=8)
    t2s = d.vocab_utils.longest_prefix_map(student, teacher)
    if drop:
        t2s = t2s.copy()
        t2s[np.random.default_rng(seed).random(Vt) < drop] = -1
    g = torch.Generator().manual_seed(seed)
    probs = torch.softmax(torch.randn(R, Vt, generator=g) * 2, -1)
    return t2s, probs


def _map_in_the_form(D, planned, t2s, Vs):
    """False: the bare map on the GPU (LDS atomics); "full": the plan over the student ids only; "auto": what
    MarginalPlan builds by itself (the compact plan beside the full one where the map's image is small)."""
    if not planned:
        return torch.tensor(t2s, device=DEV)
    return D.vocab_utils.MarginalPlan(t2s, Vs, DEV, compact=False if planned == "full" else None)



@pytest.mark.parametrize("Vs,Vt,alphabet", [(1000, 5000, 4), (32000, 152064, 256), (40000, 50001, 16)])
def test_marginal_map_and_csr_forms(D, Vs, Vt, alphabet):
    t2s, probs = _case(6, Vs, Vt, 1, alphabet, drop=0.02)
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    off, ind = D.vocab_utils.csr_from_map(t2s, Vs)
    np.testing.assert_allclose(ref, O.marginalise_csr(probs.numpy(), off, ind), rtol=1e-12, atol=1e-15)
    m_map = D.vocab_utils.marginalise(probs.to(DEV), t2s=torch.tensor(t2s, device=DEV), n_student=Vs).cpu().numpy()
    m_csr = D.vocab_utils.marginalise(probs.to(DEV), csr=(torch.tensor(off, device=DEV), torch.tensor(ind, device=DEV)),
                                      n_student=Vs).cpu().numpy()
    # marginal sums within fp32 tolerance; exact zeros where no teacher token maps
    np.testing.assert_allclose(m_map, ref, rtol=2e-6, atol=1e-9)
    np.testing.assert_allclose(m_csr, ref, rtol=2e-6, atol=1e-9)
    assert np.array_equal(m_map == 0, ref == 0) and np.array_equal(m_csr == 0, ref == 0)
    np.testing.assert_allclose(m_map.astype(np.float64).sum(-1), probs.double().numpy()[:, t2s >= 0].sum(-1), rtol=1e-5)
    # the CSR form is bit-reproducible
    again = D.vocab_utils.marginalise(probs.to(DEV), csr=(torch.tensor(off, device=DEV), torch.tensor(ind, device=DEV)),
                                      n_student=Vs).cpu().numpy()
    assert np.array_equal(m_csr, again)
    if Vs <= 36000:
        plan = D.vocab_utils.MarginalPlan(t2s, Vs, DEV)
        m_plan = D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy()
        np.testing.assert_allclose(m_plan, ref, rtol=2e-6, atol=1e-9)
        assert np.array_equal(m_plan == 0, ref == 0)
        assert np.array_equal(m_plan, D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy())
    lg = D.vocab_utils.marginalise(probs.to(DEV), t2s=torch.tensor(t2s, device=DEV), n_student=Vs, log=True).cpu().numpy()
    with np.errstate(divide="ignore"):
        np.testing.assert_allclose(lg[ref > 0], np.log(ref[ref > 0]), rtol=1e-5, atol=1e-5)
    assert np.isneginf(lg[ref == 0]).all()


def test_planned_marginal_with_lists_longer_than_one_batch(D):
    """A student vocabulary that leaves the LDS almost no room for replicas, and a few very hot ids:
    the per-thread lists of a tile then run over several batches of the kernel."""
    Vs, Vt, R = 36500, 30000, 5
    rng = np.random.default_rng(11)
    t2s = rng.integers(-1, Vs, Vt).astype(np.int32)
    hot = rng.random(Vt) < 0.9
    t2s[hot] = rng.integers(0, 16, int(hot.sum())) * 977
    probs = torch.softmax(torch.randn(R, Vt, generator=torch.Generator().manual_seed(11)) * 2, -1)
    plan = D.vocab_utils.MarginalPlan(t2s, Vs, DEV)
    assert plan.ent is not None and int(np.diff(plan.row_off.cpu().numpy()).max()) > 8
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    m_plan = D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy()
    np.testing.assert_allclose(m_plan, ref, rtol=4e-6, atol=1e-9)
    assert np.array_equal(m_plan == 0, ref == 0)
    assert np.array_equal(m_plan, D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy())


@pytest.mark.parametrize("case", ["one_hot_id", "all_dropped", "short", "tiny_student", "zipf"])
def test_planned_marginal_on_degenerate_maps(D, case):
    rng = np.random.default_rng(3)
    Vs, Vt, R = 3000, 20000, 4
    if case == "one_hot_id":
        t2s = np.where(rng.random(Vt) < 0.95, 17, rng.integers(0, Vs, Vt))
    elif case == "all_dropped":
        t2s = np.full(Vt, -1)
    elif case == "short":
        Vt = 1000
        t2s = rng.integers(0, Vs, Vt)
    elif case == "tiny_student":
        Vs = 4
        t2s = rng.integers(0, Vs, Vt)
    else:
        t2s = np.minimum(rng.zipf(1.2, Vt) - 1, Vs - 1)
    t2s = t2s.astype(np.int32)
    probs = torch.softmax(torch.randn(R, Vt, generator=torch.Generator().manual_seed(5)) * 2, -1)
    plan = D.vocab_utils.MarginalPlan(t2s, Vs, DEV)
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    m_plan = D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy()
    np.testing.assert_allclose(m_plan, ref, rtol=2e-5, atol=1e-9)
    assert np.array_equal(m_plan == 0, ref == 0)


def test_a_plan_built_for_other_vocabularies_is_refused(D):
    t2s = np.random.default_rng(0).integers(0, 1000, 5000).astype(np.int32)
    plan = D.vocab_utils.MarginalPlan(t2s, 1000, DEV)
    probs = torch.rand(2, 5000, device=DEV)
    with pytest.raises(RuntimeError, match="the plan maps"):
        D.vocab_utils.marginalise(probs, plan=plan, n_student=1008)
    with pytest.raises(RuntimeError, match="the plan maps"):
        D.vocab_utils.marginalise(torch.rand(2, 6000, device=DEV), plan=plan, n_student=1000)
    with pytest.raises(RuntimeError, match="the plan maps"):
        D.vocab_utils.rkl_marginalised(torch.randn(2, 1008, device=DEV), probs, plan)


def test_marginal_of_16bit_probabilities(D):
    t2s, probs = _case(4, 512, 2048, 2)
    got = D.vocab_utils.marginalise(probs.to(torch.bfloat16).to(DEV), t2s=torch.tensor(t2s, device=DEV), n_student=512)
    ref = O.marginalise_map(probs.to(torch.bfloat16).double().numpy(), t2s, 512)
    np.testing.assert_allclose(got.cpu().numpy(), ref, rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("planned", [False, "full", "auto"])
@pytest.mark.parametrize("dtype,Vs,Vt,alphabet,T", [(torch.bfloat16, 32000, 152064, 256, 1.5), (torch.float32, 2048, 9000, 4, 1.0),
                                                    (torch.float16, 8192, 30000, 8, 0.8)])
def test_fused_reverse_kl_against_marginal(D, dtype, Vs, Vt, alphabet, T, planned):
    R = 12
    t2s, probs = _case(R, Vs, Vt, 3, alphabet, drop=0.01)
    g = torch.Generator().manual_seed(9)
    logits = (torch.randn(R + 3, Vs, generator=g) * 2).to(dtype)
    valid = torch.ones(R + 3, dtype=torch.bool)
    valid[[2, 5, 14]] = False
    rm = torch.full((R + 3,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R, dtype=torch.int32)
    tmap = _map_in_the_form(D, planned, t2s, Vs)
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), tmap, row_map=rm.to(DEV), T=T,
                                              grad_scale=1.0 / R)
    if planned:       # fixed summation order: bit-reproducible
        rl2, grad2 = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), tmap, row_map=rm.to(DEV), T=T,
                                                    grad_scale=1.0 / R)
        assert torch.equal(rl, rl2) and torch.equal(grad, grad2)
    marg = torch.tensor(O.marginalise_map(probs.numpy(), t2s, Vs))
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    loss64, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, T, t_logits=t_logits, valid=valid, dtype=torch.float64)
    np.testing.assert_allclose(D.reduce_sum(rl, 1.0 / R).item(), loss64.item(), rtol=1e-5)
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    assert torch.count_nonzero(grad.cpu()[~valid]) == 0 and torch.count_nonzero(rl.cpu()[~valid]) == 0
    err = (grad.cpu().double() - grad64).abs()
    rtol = 1e-4 if dtype == torch.float32 else 2e-3
    bound = O.storage_tolerance(grad64, dtype, rtol)
    sel = torch.nonzero(valid).squeeze(-1)
    bound[sel] = O.marginal_rkl_gradient_tolerance(grad64[sel], logits[sel], t_logits, rows64, T, T, 1.0 / R, dtype, rtol)
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    # the gradient is confined to the marginal's support
    assert torch.count_nonzero(grad.cpu()[valid][:, (marg.sum(0) == 0)]) == 0


@pytest.mark.parametrize("planned", [False, "full", "auto"])
@pytest.mark.parametrize("T", [1.0, 2.0, 0.5])
def test_fused_reverse_kl_on_rows_whose_sums_leave_the_range(D, T, planned):
    """Rows for which a bias of 0 for the teacher and the row's largest logit for the student do not keep
    the sums in range: hardly any teacher mass (down to denormal entries), an unnormalised teacher, a student
    whose mass sits on a column outside the marginal's support, and a teacher row without mass (zero loss,
    zero gradient)."""
    R, Vs, Vt = 6, 2048, 9000
    t2s, probs = _case(R, Vs, Vt, 5, 4, drop=0.01)
    g = torch.Generator().manual_seed(11)
    logits = torch.randn(R, Vs, generator=g) * 2
    probs = probs.clone()
    probs[0] *= 1e-25
    probs[1] *= 1e25
    probs[5] *= 1e-33                                # most of the marginal's entries are denormal: their logarithms still count
    off = int(t2s[t2s >= 0][0])                      # a student column that is taken off the support of row 2
    probs[2, torch.tensor(t2s == off)] = 0.0
    logits[2, off] = 300.0
    probs[3] = 0.0
    tmap = _map_in_the_form(D, planned, t2s, Vs)
    with_mass = torch.tensor([0, 1, 2, 4, 5])
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), tmap, T=T, grad_scale=1.0 / len(with_mass))
    rl, grad = rl.cpu(), grad.cpu()
    assert rl[3] == 0 and torch.count_nonzero(grad[3]) == 0
    marg = torch.tensor(O.marginalise_map(probs.double().numpy(), t2s, Vs))[with_mass]
    assert marg[2, off] == 0
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits[with_mass], T, t_logits=t_logits, dtype=torch.float64)
    np.testing.assert_allclose(rl[with_mass].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    err = (grad[with_mass].double() - grad64).abs()
    bound = 1e-4 * grad64.abs() + 2e-6 * grad64.abs().amax(-1, keepdim=True)
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    assert torch.count_nonzero(grad[with_mass][marg == 0]) == 0
    # without a gradient the loss takes other passes over the row: the same values to rounding
    rl_only, none = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), tmap, T=T, want_grad=False)
    assert none is None
    np.testing.assert_allclose(rl_only.cpu().numpy(), rl.numpy(), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lift", [3.0, 6.0, 12.0, 30.0])
def test_fused_reverse_kl_16bit_student_with_its_largest_logits_off_the_support(D, dtype, lift):
    """The student's largest logits sit on columns without teacher mass, `lift` above the rest: reverse KL
    renormalises the student over the support, so the columns that carry the gradient lie far below the
    row's maximum (what the kernel keeps of 2^logit between its passes must still resolve them)."""
    R, Vs, Vt = 5, 4096, 12000
    t2s, probs = _case(R, Vs, Vt, 7, 16, drop=0.01)
    g = torch.Generator().manual_seed(3)
    logits = torch.randn(R, Vs, generator=g) * 2
    marg0 = torch.tensor(O.marginalise_map(probs.double().numpy(), t2s, Vs))
    on = torch.nonzero(marg0[0] > 0).squeeze(-1)
    off_cols = on[:6]                                # taken off the support of every row
    probs = probs.clone()
    probs[:, torch.isin(torch.tensor(t2s), off_cols)] = 0.0
    logits[:, off_cols] += lift
    logits = logits.to(dtype)
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), torch.tensor(t2s, device=DEV), T=0.7,
                                              teacher_T=1.0, grad_scale=1.0 / R)
    marg = torch.tensor(O.marginalise_map(probs.double().numpy(), t2s, Vs))
    assert (marg[:, off_cols] == 0).all()
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, 0.7, t_logits=t_logits, t_T=1.0, dtype=torch.float64)
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    err = (grad.cpu().double() - grad64).abs()
    bound = O.marginal_rkl_gradient_tolerance(grad64, logits, t_logits, rows64, 0.7, 1.0, 1.0 / R, dtype, 2e-3)
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    assert torch.count_nonzero(grad.cpu()[:, off_cols]) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_reverse_kl_16bit_rows_whose_maximum_is_negative_zero_or_towering(D, dtype):
    """16-bit student rows take a non-negative maximum from the raw bit patterns, else from the values: rows
    of negative logits only, maxima of exactly +0 and -0, and one logit far above the rest at every position
    inside a 16-byte chunk in turn (a maximum that missed it would let the sums overflow)."""
    R, Vs, Vt = 12, 4096, 12000
    t2s, probs = _case(R, Vs, Vt, 9, 16, drop=0.01)
    g = torch.Generator().manual_seed(4)
    logits = torch.randn(R, Vs, generator=g) * 2
    logits[0] = -logits[0].abs() - 0.5
    logits[1] = -logits[1].abs() - 1.0
    logits[1, 77] = 0.0
    logits[2] = -logits[2].abs() - 1.0
    logits[2, 1234] = -0.0
    marg0 = torch.tensor(O.marginalise_map(probs.double().numpy(), t2s, Vs))
    for r in range(4, 12):
        on = torch.nonzero(marg0[r] > 0).squeeze(-1)
        col = int(on[(on % 8) == (r - 4)][5])          # a column of the support at position r - 4 of its chunk
        logits[r, col] = 120.0
    logits = logits.to(dtype)
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), torch.tensor(t2s, device=DEV), T=1.0,
                                              grad_scale=1.0 / R)
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg0)
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, 1.0, t_logits=t_logits, dtype=torch.float64)
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    err = (grad.cpu().double() - grad64).abs()
    bound = O.marginal_rkl_gradient_tolerance(grad64, logits, t_logits, rows64, 1.0, 1.0, 1.0 / R, dtype, 2e-3)
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("planned", [False, "full", "auto"])
def test_fused_reverse_kl_gradient_may_overwrite_the_logits(D, dtype, planned):
    """The gradient written over the logits, also for rows that are put back and redone (their logits are
    read a second time before anything of the row is written): the same bits as into a buffer of its own."""
    R, Vs, Vt = 6, 4096, 12000
    t2s, probs = _case(R, Vs, Vt, 7, 16, drop=0.01)
    g = torch.Generator().manual_seed(6)
    logits = torch.randn(R, Vs, generator=g) * 2
    marg0 = torch.tensor(O.marginalise_map(probs.double().numpy(), t2s, Vs))
    off_cols = torch.nonzero(marg0[0] > 0).squeeze(-1)[:4]
    probs = probs.clone()
    probs[:, torch.isin(torch.tensor(t2s), off_cols)] = 0.0
    logits[1::2, off_cols] += 40.0                   # every other row has its mass off the support
    probs[4] *= 1e-30                                # and one hardly any teacher mass
    x = logits.to(dtype).to(DEV)
    tmap = _map_in_the_form(D, planned, t2s, Vs)
    rl, grad = D.vocab_utils.rkl_marginalised(x, probs.to(DEV), tmap, T=1.3, grad_scale=0.5)
    y = x.clone()
    rl2, g2 = D.vocab_utils.rkl_marginalised(y, probs.to(DEV), tmap, T=1.3, grad_scale=0.5, grad_out=y)
    assert g2.data_ptr() == y.data_ptr()
    if planned:                                      # fixed summation order: the same bits
        assert torch.equal(rl, rl2) and torch.equal(grad, y)
    else:                                            # LDS atomics: the marginal's sums come in any order
        np.testing.assert_allclose(rl2.cpu().numpy(), rl.cpu().numpy(), rtol=1e-5)
        tol = 1e-4 if dtype == torch.float32 else 2.0 ** -7
        diff = (grad.float() - y.float()).abs()
        assert (diff <= tol * grad.float().abs() + 1e-6 * grad.float().abs().max()).all()
    assert torch.isfinite(rl).all() and torch.isfinite(grad.float()).all() and grad.float().abs().max() > 0


def test_fused_path_limits_are_reported(D):
    with pytest.raises(RuntimeError, match="exceeds"):
        D.vocab_utils.rkl_marginalised(torch.zeros(2, 40000, device=DEV), torch.zeros(2, 64, device=DEV),
                                       torch.zeros(64, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_column_gather_and_expansion(D, dtype):
    """dl_gather_columns / dl_expand_columns move raw elements: a subset of the columns out (padding reads -inf)
    and back in (columns outside the subset read 0), every bit as it was."""
    g = torch.Generator().manual_seed(3)
    R, V = 7, 4104
    x = (torch.randn(R, V + 8, generator=g) * 3).to(dtype).to(DEV)[:, :V]           # rows of another pitch
    used = torch.sort(torch.randperm(V, generator=g)[:1001]).values
    cols = torch.full((1008,), -1, dtype=torch.int32)
    cols[:1001] = used.to(torch.int32)
    col_src = torch.full((V,), -1, dtype=torch.int32)
    col_src[used] = torch.arange(1001, dtype=torch.int32)
    xc = D.vocab_utils.gather_columns(x, cols.to(DEV))
    assert torch.equal(xc[:, :1001], x[:, used.to(DEV)]) and torch.isneginf(xc[:, 1001:].float()).all()
    back = D.vocab_utils.expand_columns(xc, col_src.to(DEV), V)
    want = torch.zeros_like(x)
    want[:, used.to(DEV)] = x[:, used.to(DEV)]
    assert torch.equal(back, want)


@pytest.mark.parametrize("dtype,Vs,Vt,alphabet", [(torch.bfloat16, 128256, 152064, 256), (torch.float32, 50000, 60000, 8),
                                                  (torch.float16, 8192, 30000, 16)])
def test_fused_reverse_kl_on_a_student_vocabulary_compacted_to_the_map_s_image(D, dtype, Vs, Vt, alphabet):
    """Student vocabularies wider than the fused kernel's marginal (and, on request, narrower ones): the plan is
    built over the student ids the map reaches, the logits' columns are gathered, the gradient expanded.  Loss
    and gradient against the oracle on the full vocabulary; columns outside the image get exactly 0; masked
    rows; bit-reproducible."""
    R = 9
    t2s, probs = _case(R, Vs, Vt, 5, alphabet, drop=0.01)
    g = torch.Generator().manual_seed(11)
    logits = (torch.randn(R + 2, Vs, generator=g) * 2).to(dtype)
    valid = torch.ones(R + 2, dtype=torch.bool)
    valid[[1, 7]] = False
    rm = torch.full((R + 2,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R, dtype=torch.int32)
    plan = D.vocab_utils.MarginalPlan(t2s, Vs, DEV, compact=True)
    assert plan.cols is not None and plan.n_compact % 8 == 0 and plan.n_compact < Vs
    T = 1.5
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), plan, row_map=rm.to(DEV), T=T, grad_scale=1.0 / R)
    rl2, grad2 = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), plan, row_map=rm.to(DEV), T=T, grad_scale=1.0 / R)
    assert torch.equal(rl, rl2) and torch.equal(grad, grad2) and grad.shape == logits.shape and grad.dtype == dtype
    marg = torch.tensor(O.marginalise_map(probs.numpy(), t2s, Vs))
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    loss64, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, T, t_logits=t_logits, valid=valid, dtype=torch.float64)
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    assert torch.count_nonzero(grad.cpu()[~valid]) == 0 and torch.count_nonzero(rl.cpu()[~valid]) == 0
    rtol = 1e-4 if dtype == torch.float32 else 2e-3
    bound = O.storage_tolerance(grad64, dtype, rtol)
    sel = torch.nonzero(valid).squeeze(-1)
    bound[sel] = O.marginal_rkl_gradient_tolerance(grad64[sel], logits[sel], t_logits, rows64, T, T, 1.0 / R, dtype, rtol)
    err = (grad.cpu().double() - grad64).abs()
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    outside = torch.ones(Vs, dtype=torch.bool)
    outside[torch.as_tensor(np.unique(t2s[t2s >= 0])).long()] = False
    assert torch.count_nonzero(grad.cpu()[:, outside]) == 0
    rl3, _ = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), plan, row_map=rm.to(DEV), T=T, want_grad=False)
    np.testing.assert_allclose(rl3.cpu().numpy(), rl.cpu().numpy(), rtol=2e-5, atol=1e-6)


@pytest.mark.parametrize("Vs,dtype", [(4008, torch.float32), (4000, torch.bfloat16)])
def test_a_plan_that_holds_the_compact_form_only(D, Vs, dtype):
    """No full plan to fall back to: the fused kernel runs on the compact ids, and `marginalise` gives the full-width marginal from the bare map."""
    R, Vt = 5, 9000
    t2s, probs = _case(R, Vs, Vt, 9, 16)
    plan = D.vocab_utils.MarginalPlan(t2s, Vs, DEV, compact=True)
    assert plan.full is None and plan.compact is not None
    g = torch.Generator().manual_seed(4)
    logits = (torch.randn(R, Vs, generator=g) * 2).to(dtype)
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), probs.to(DEV), plan, T=1.2, grad_scale=1.0 / R)
    marg = torch.tensor(O.marginalise_map(probs.numpy(), t2s, Vs))
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, 1.2, t_logits=t_logits, dtype=torch.float64)
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    bound = O.marginal_rkl_gradient_tolerance(grad64, logits, t_logits, rows64, 1.2, 1.2, 1.0 / R, dtype,
                                              1e-4 if dtype == torch.float32 else 2e-3)
    err = (grad.cpu().double() - grad64).abs()
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    m = D.vocab_utils.marginalise(probs.to(DEV), plan=plan, n_student=Vs).cpu().numpy()
    np.testing.assert_allclose(m, marg.numpy(), rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("Vt", [8, 1024, 4100, 8196, 12292, 20484, 24580])
@pytest.mark.parametrize("shift", [1, 3])
def test_planned_forms_on_teacher_rows_off_the_16_byte_grid(D, Vt, shift):
    """Rows of whole 16-byte units that start on any element: rows shorter than a tile and a last tile of one unit.  The rows
    end where the buffer ends."""
    R, Vs = 5, 2048
    rng = np.random.default_rng(Vt)
    t2s = rng.integers(-1, 700, Vt).astype(np.int32)
    t2s[-1] = 13                                     # the last element counts
    probs = torch.softmax(torch.randn(R, Vt, generator=torch.Generator().manual_seed(Vt)) * 2, -1)
    buf = torch.zeros(shift + R * Vt, device=DEV)
    on_gpu = buf[shift:].view(R, Vt)
    on_gpu.copy_(probs)
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    logits = torch.randn(R, Vs, generator=torch.Generator().manual_seed(1)) * 2
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(torch.tensor(ref))
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, 1.3, t_logits=t_logits, dtype=torch.float64)
    for form in ("full", "auto"):
        plan = _map_in_the_form(D, form, t2s, Vs)
        got = D.vocab_utils.marginalise(on_gpu, plan=plan, n_student=Vs).cpu().numpy()
        np.testing.assert_allclose(got, ref, rtol=2e-6, atol=1e-9)
        assert np.array_equal(got == 0, ref == 0)
        rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), on_gpu, plan, T=1.3, grad_scale=1.0 / R)
        rl2, grad2 = D.vocab_utils.rkl_marginalised(logits.to(DEV), on_gpu, plan, T=1.3, grad_scale=1.0 / R)
        assert torch.equal(rl, rl2) and torch.equal(grad, grad2)
        np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
        bound = O.marginal_rkl_gradient_tolerance(grad64, logits, t_logits, rows64, 1.3, 1.3, 1.0 / R, torch.float32, 1e-4)
        err = (grad.cpu().double() - grad64).abs()
        assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("Vt,Vs", [(5, 2048), (1023, 2048), (4097, 2048), (8193, 2048), (12290, 2048), (16387, 8192), (20483, 2048),
                                   (24577, 2048)])
@pytest.mark.parametrize("shift", [0, 3])
def test_a_plan_with_teacher_rows_that_end_inside_a_unit(D, Vt, Vs, shift):
    """Teacher vocabularies that are no multiple of four ids: the last 1-3 probabilities of every row count.  The rows end where
    the buffer ends."""
    R = 5
    rng = np.random.default_rng(Vt)
    t2s = rng.integers(-1, 700, Vt).astype(np.int32)
    t2s[-3:] = (13, 700, Vs - 1)                     # the last two ids of their own
    probs = torch.softmax(torch.randn(R, Vt, generator=torch.Generator().manual_seed(Vt)) * 2, -1)
    buf = torch.zeros(shift + R * Vt, device=DEV)
    on_gpu = buf[shift:].view(R, Vt)
    on_gpu.copy_(probs)
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    logits = torch.randn(R, Vs, generator=torch.Generator().manual_seed(1)) * 2
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(torch.tensor(ref))
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits, 1.3, t_logits=t_logits, dtype=torch.float64)
    for form in ("full", "auto"):
        plan = _map_in_the_form(D, form, t2s, Vs)
        got = D.vocab_utils.marginalise(on_gpu, plan=plan, n_student=Vs).cpu().numpy()
        np.testing.assert_allclose(got, ref, rtol=2e-6, atol=1e-9)
        assert np.array_equal(got == 0, ref == 0)
        rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), on_gpu, plan, T=1.3, grad_scale=1.0 / R)
        np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
        bound = O.marginal_rkl_gradient_tolerance(grad64, logits, t_logits, rows64, 1.3, 1.3, 1.0 / R, torch.float32, 1e-4)
        err = (grad.cpu().double() - grad64).abs()
        assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Vt,Vs,used", [(1027, 1000, 300), (8192, 2048, 2048), (24581, 4096, 700), (40000, 16384, 9000)])
def test_more_rows_than_cus_take_two_workgroups_per_cu(D, Vt, Vs, used, dtype):
    """More than 256 rows: workgroups of 512 threads that walk two lists per wave and tile (one tile, odd numbers of tiles, a
    row that ends inside a unit; the last map is too wide for two workgroups per CU), masked rows, the gradient over the logits."""
    R = 259
    rng = np.random.default_rng(Vt)
    ids = rng.permutation(Vs)[:used]
    t2s = ids[rng.integers(0, used, Vt)].astype(np.int32)
    t2s[rng.random(Vt) < 0.05] = -1
    t2s[-1] = ids[0]
    g = torch.Generator().manual_seed(Vt)
    probs = torch.softmax(torch.randn(R - 2, Vt, generator=g) * 2, -1)
    logits = (torch.randn(R, Vs, generator=g) * 2).to(dtype)
    rm = torch.full((R,), -1, dtype=torch.int32)
    valid = torch.ones(R, dtype=torch.bool)
    valid[[0, 200]] = False
    rm[valid] = torch.arange(R - 2, dtype=torch.int32)
    ref = O.marginalise_map(probs.numpy(), t2s, Vs)
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(torch.tensor(ref))
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits[valid], 1.3, t_logits=t_logits, dtype=torch.float64)
    x = logits.to(DEV)
    plan = _map_in_the_form(D, "auto", t2s, Vs)
    rl, grad = D.vocab_utils.rkl_marginalised(x, probs.to(DEV), plan, row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / (R - 2), grad_out=x)
    rl, grad = rl.cpu(), grad.cpu()
    assert torch.count_nonzero(rl[~valid]) == 0 and torch.count_nonzero(grad[~valid]) == 0
    np.testing.assert_allclose(rl[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    bound = O.marginal_rkl_gradient_tolerance(grad64, logits[valid], t_logits, rows64, 1.3, 1.3, 1.0 / (R - 2), dtype,
                                              1e-4 if dtype == torch.float32 else 2e-3)
    err = (grad[valid].double() - grad64).abs()
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("R,Vt,Vs,used,dtype", [(3, 70001, 2048, 500, torch.bfloat16),      # tiles dealt to several workgroups, a ragged end
                                                (2, 200064, 16384, 16384, torch.float16),    # the full plan, six parts
                                                (128, 70000, 2048, 700, torch.float32), (129, 70000, 2048, 700, torch.float32)])
def test_few_rows_against_a_wide_teacher(D, R, Vt, Vs, used, dtype):
    """Up to 128 rows a row's tiles are shared by several workgroups through a workspace, and the passes take a launch of their
    own; masked rows, the gradient over the logits."""
    rng = np.random.default_rng(Vt + R)
    ids = rng.permutation(Vs)[:used]
    t2s = ids[rng.integers(0, used, Vt)].astype(np.int32)
    t2s[rng.random(Vt) < 0.05] = -1
    t2s[-1] = ids[0]
    plan = _map_in_the_form(D, "auto", t2s, Vs)
    tile = (plan.compact or plan.full).tile
    n = plan.n_compact if plan.compact is not None else Vs
    ws = D._lib.load().dl_rkl_marginalised_workspace_bytes(R, Vt, n, tile)
    assert (ws == 0) == (R > 128 or 256 // R < 2 or -(-Vt // tile) < 8)
    g = torch.Generator().manual_seed(Vt)
    probs = torch.softmax(torch.randn(R, Vt, generator=g) * 2, -1)
    logits = (torch.randn(R, Vs, generator=g) * 2).to(dtype)
    rm = torch.arange(R, dtype=torch.int32)
    valid = torch.ones(R, dtype=torch.bool)
    rm[1], valid[1] = -1, False
    ref = O.marginalise_map(probs[valid].numpy(), t2s, Vs)
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(torch.tensor(ref))
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits[valid], 1.3, t_logits=t_logits, dtype=torch.float64)
    nv = int(valid.sum())
    for in_place in (False, True):
        x = logits.to(DEV)
        rl, grad = D.vocab_utils.rkl_marginalised(x, probs.to(DEV), plan, row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / nv,
                                                  grad_out=x if in_place else None)
        rl, grad = rl.cpu(), grad.cpu()
        assert torch.count_nonzero(rl[~valid]) == 0 and torch.count_nonzero(grad[~valid]) == 0
        np.testing.assert_allclose(rl[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
        bound = O.marginal_rkl_gradient_tolerance(grad64, logits[valid], t_logits, rows64, 1.3, 1.3, 1.0 / nv, dtype,
                                                  1e-4 if dtype == torch.float32 else 2e-3)
        err = (grad[valid].double() - grad64).abs()
        assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


def _map_onto(Vt, Vs, used, dropped=0.05):
    """Teacher ids onto `used` of the student ids, every one of them named; some teacher ids onto none."""
    rng = np.random.default_rng(Vt + used)
    ids = rng.permutation(Vs)[:used]
    t2s = ids[rng.integers(0, used, Vt)].astype(np.int32)
    t2s[rng.random(Vt) < dropped] = -1
    t2s[rng.permutation(Vt)[:used]] = ids
    t2s[-3:] = ids[:3]                               # the last three count
    t2s[:3] = ids[-3:]
    t2s[5] = t2s[6] = -1
    missing = np.setdiff1d(ids, t2s)
    t2s[np.nonzero(t2s < 0)[0][:missing.size]] = missing
    return t2s


def _check_against_marginal(rl, grad, logits, probs, t2s, T, scale, dtype, rows=None):
    """Row losses and gradients of `rows` (all: None) against float64."""
    sel = torch.arange(logits.shape[0]) if rows is None else rows
    marg = torch.tensor(O.marginalise_map(probs[sel].double().numpy(), t2s, logits.shape[1]))
    with np.errstate(divide="ignore"):
        t_logits = O.marginal_to_teacher_logits(marg)
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", logits[sel], T, t_logits=t_logits, dtype=torch.float64)
    grad64 = grad64 * (len(sel) * scale)
    np.testing.assert_allclose(rl[sel].cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    bound = O.marginal_rkl_gradient_tolerance(grad64, logits[sel], t_logits, rows64, T, T, scale, dtype,
                                              1e-4 if dtype == torch.float32 else 2e-3)
    err = (grad[sel].cpu().double() - grad64).abs()
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"
    assert torch.count_nonzero(grad[sel].cpu()[marg == 0]) == 0


@pytest.mark.parametrize("R", [3, 130, 259])         # several workgroups per row; one of 1024 threads; of 512
@pytest.mark.parametrize("Vt,Vs,used,tile", [(61441, 2048, 700, 6144), (61442, 2048, 700, 6144), (86019, 2048, 300, 7168),
                                             (131075, 8192, 8192, 8192)])
def test_a_last_tile_without_a_whole_unit(D, R, Vt, Vs, used, tile):
    """One to three probabilities are all that the last tile of the plan holds: no whole 16-byte unit of it is fetched.  The rows
    end where the buffer ends, and start on any element."""
    t2s = _map_onto(Vt, Vs, used)
    plan = _map_in_the_form(D, "auto", t2s, Vs)
    assert (plan.compact or plan.full).tile == plan.full.tile == tile and Vt % tile in (1, 2, 3) and (t2s[-(Vt % tile):] >= 0).all()
    g = torch.Generator().manual_seed(Vt)
    probs = torch.softmax(torch.randn(R, Vt, generator=g) * 2, -1)
    probs[:, -(Vt % tile):] += 0.05                  # what the last tile brings is no rounding
    logits = torch.randn(R, Vs, generator=g) * 2
    buf = torch.zeros(1 + R * Vt, device=DEV)
    on_gpu = buf[1:].view(R, Vt)
    on_gpu.copy_(probs)
    few = torch.arange(min(R, 40))
    got = D.vocab_utils.marginalise(on_gpu, plan=plan, n_student=Vs).cpu().numpy()[few]
    ref = O.marginalise_map(probs[few].numpy(), t2s, Vs)
    np.testing.assert_allclose(got, ref, rtol=2e-6, atol=1e-9)
    assert np.array_equal(got == 0, ref == 0)
    rl, grad = D.vocab_utils.rkl_marginalised(logits.to(DEV), on_gpu, plan, T=1.3, grad_scale=0.25)
    _check_against_marginal(rl, grad, logits, probs, t2s, 1.3, 0.25, torch.float32, few)


@pytest.mark.parametrize("Vt,Vs,used,dtype,half", [
    (40000, 32000, 6704, torch.bfloat16, True),      # 838 units of 8 ids for 512 threads: two each
    (40000, 32000, 6704, torch.float32, True),
    (40000, 18000, 8192, torch.float32, True),       # as many fp32 ids as two units per thread hold,
    (40000, 18000, 8200, torch.float32, False),      # and a unit more
    (40001, 32000, 12088, torch.float16, True),      # as many as the LDS of two workgroups per CU holds (three units each),
    (40001, 32000, 12096, torch.float16, False)])    # and a unit more
def test_widths_that_two_workgroups_per_cu_hold(D, Vt, Vs, used, dtype, half):
    """The passes behind the marginal with several units per thread of a 512-thread workgroup, and the borders of its rule, among
    them rows whose sums leave the range and are redone on their maxima, a row without mass, a masked row."""
    R = 259
    t2s = _map_onto(Vt, Vs, used)
    plan = _map_in_the_form(D, "auto", t2s, Vs)
    c = plan.compact
    assert plan.n_compact == used and c.tile == 8192 and c.n_extra == 0
    lds = 4 * (used + 64 + c.tile + 4)               # the marginal, the lanes' spare slots, the tile and its zeros
    assert half == (used <= (8192 if dtype == torch.float32 else 16384) and lds <= 80 * 1024 - 512)
    g = torch.Generator().manual_seed(Vt)
    probs = torch.softmax(torch.randn(R, Vt, generator=g) * 2, -1)
    logits = torch.randn(R, Vs, generator=g) * 2
    probs[7] *= 1e-25
    probs[8] *= 1e25
    off = int(t2s[20])
    probs[9, torch.tensor(t2s == off)] = 0.0         # the student's mass on a column that is off row 9's support
    logits[9, off] = 300.0
    probs[10] = 0.0
    logits = logits.to(dtype)
    rm = torch.arange(R, dtype=torch.int32)
    rm[11] = -1
    x = logits.to(DEV)
    rl, grad = D.vocab_utils.rkl_marginalised(x, probs.to(DEV), plan, row_map=rm.to(DEV), T=1.3, grad_scale=0.25, grad_out=x)
    assert torch.count_nonzero(rl[10:12]) == 0 and torch.count_nonzero(grad[10:12]) == 0
    _check_against_marginal(rl, grad, logits, probs, t2s, 1.3, 0.25, dtype, torch.tensor([0, 1, 7, 8, 9, 12, 100, 255, 256, 258]))


@pytest.mark.parametrize("R,Vt,Vs,used,dtype,parts", [
    (2, 270000, 16384, 16384, torch.float16, 8),     # the full plan, 33 tiles of 8192: as many parts as there ever are
    (3, 70001, 2048, 500, torch.bfloat16, 3),        # a ragged end
    (85, 100000, 8192, 8192, torch.float32, 3),      # 256 / 85
    (128, 131075, 8192, 8192, torch.float32, 2)])    # the last of 17 tiles holds three probabilities
def test_partial_marginals_against_one_launch(D, R, Vt, Vs, used, dtype, parts):
    """With a workspace the tiles of few rows are dealt to `parts` workgroups each: the same within rounding as one launch.  A
    workspace that is too small, off the 16-byte grid or absent is one launch, bit for bit."""
    lib = D._lib.load()
    t2s = _map_onto(Vt, Vs, used)
    plan = _map_in_the_form(D, "full", t2s, Vs)
    assert lib.dl_rkl_marginalised_workspace_bytes(R, Vt, Vs, plan.full.tile) == R * parts * Vs * 4
    g = torch.Generator(device=DEV).manual_seed(Vt)
    probs = torch.softmax(torch.randn(R, Vt, generator=g, device=DEV) * 2, -1)
    logits = (torch.randn(R, Vs, generator=g, device=DEV) * 2).to(dtype)
    rm = torch.arange(R, dtype=torch.int32, device=DEV)
    rm[1] = -1
    ws = torch.full((R * parts * Vs + 4,), float("nan"), device=DEV)
    assert ws.data_ptr() % 16 == 0

    def run(workspace):
        rl, grad = torch.empty(R, device=DEV), torch.empty_like(logits)
        args = [logits.data_ptr(), D.ops._DT[dtype], Vs, R, Vs, rm.data_ptr(), probs.data_ptr(), D.ops._DT[torch.float32], Vt, R, Vt,
                plan.t2s.data_ptr(), *plan.full.args(), 1 / 1.3, 1 / 1.3, 0.25, rl.data_ptr(), grad.data_ptr(), Vs]
        stream = torch.cuda.current_stream().cuda_stream
        if workspace is None:
            D._lib.check(lib.dl_rkl_marginalised(*args, stream), "dl_rkl_marginalised")
        else:
            D._lib.check(lib.dl_rkl_marginalised_ws(*args, *workspace, stream), "dl_rkl_marginalised_ws")
        return rl, grad

    n = R * parts * Vs * 4
    one = run(None)
    for short in ((ws.data_ptr(), n - 1), (ws.data_ptr() + 4, n), (0, 0)):
        assert all(torch.equal(a, b) for a, b in zip(one, run(short)))
    assert torch.isnan(ws).all()
    rl, grad = run((ws.data_ptr(), n))
    assert not torch.isnan(ws[:Vs]).any()
    torch.testing.assert_close(rl, one[0], rtol=3e-5, atol=3e-6)
    live = [r for r in range(min(R, 40)) if r != 1]
    for got in (one, (rl, grad)):
        assert got[0][1] == 0 and torch.count_nonzero(got[1][1]) == 0
        _check_against_marginal(*got, logits.cpu(), probs.cpu(), t2s, 1.3, 0.25, dtype, torch.tensor(live))
