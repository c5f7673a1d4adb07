"""GPU parity of the dense-teacher kernels (forward KL, reverse KL, JSD) against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RTOL = {torch.float32: 1e-4, torch.bfloat16: 2e-3, torch.float16: 2e-3}


@pytest.fixture(scope="module")
def D():
    import llm_distillery_amd as d
    d._lib.load()
    return d


def _check(D, kind, logits, t_logits, T, valid=None, teacher_T=None, **hooks):
    R, V = logits.shape
    n_valid = R if valid is None else int(valid.sum())
    loss64, rows64, grad64 = O.mean_loss_and_grad(kind, logits, T, t_logits=t_logits, valid=valid, t_T=teacher_T,
                                                  dtype=torch.float64)
    row_map = None
    if valid is not None:
        rm = torch.full((R,), -1, dtype=torch.int32)
        rm[valid] = torch.arange(n_valid, dtype=torch.int32)
        row_map = rm.to(DEV)
    rl, grad = D.div_dense(kind, logits.to(DEV), t_logits.to(DEV), row_map=row_map, T=T, teacher_T=teacher_T,
                           grad_scale=1.0 / n_valid, **hooks)
    loss = D.reduce_sum(rl, 1.0 / n_valid).item()
    rows = rl.cpu()
    g = grad.cpu()
    if valid is not None:
        assert torch.count_nonzero(rows[~valid]) == 0 and torch.count_nonzero(g[~valid]) == 0
        rows = rows[valid]
    np.testing.assert_allclose(loss, loss64.item(), rtol=1e-5)
    np.testing.assert_allclose(rows.double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    err = (g.double() - grad64).abs()
    sel = torch.arange(R) if valid is None else torch.nonzero(valid).squeeze(-1)
    bound = O.storage_tolerance(grad64, logits.dtype, RTOL[logits.dtype])
    # valid rows: the stated relative tolerance plus 4e-6 of the cancelling terms (see the oracle's helper)
    bound[sel] = O.dense_gradient_tolerance(grad64[sel], logits[sel], t_logits, rows64, T, T if teacher_T is None else teacher_T,
                                            1.0 / n_valid, logits.dtype, RTOL[logits.dtype], kind=kind)
    assert (err <= bound).all(), f"{int((err > bound).sum())} entries off, worst ratio {(err / bound).max():.2f}"


def _pair(R, V, dtype, seed, t_dtype=None, noise=1.0, std=2.0):
    g = torch.Generator().manual_seed(seed)
    s = (torch.randn(R, V, generator=g) * std).to(dtype)
    t = (s.float() * 0.8 + torch.randn(R, V, generator=g) * noise).to(t_dtype or dtype)
    return s, t


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("dtype,t_dtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                           (torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                           (torch.float32, torch.bfloat16), (torch.float32, torch.float16),
                                           (torch.bfloat16, torch.float16)])
def test_dense_small(D, kind, dtype, t_dtype):
    s, t = _pair(21, 2048, dtype, 1, t_dtype)
    _check(D, kind, s, t, T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "jsd"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_16bit_rows_whose_maximum_is_negative_or_zero(D, kind, dtype):
    """16-bit rows take non-negative maxima from the raw bit patterns, else from the values: student or
    teacher rows of negative logits only, and maxima of exactly +0 and -0."""
    s, t = _pair(12, 4096, dtype, 7)
    s, t = s.float(), t.float()
    s[0] = -s[0].abs() - 0.25
    t[1] = -t[1].abs() - 3.0
    s[2] = -s[2].abs() - 1.0
    t[2] = -t[2].abs() - 1.0
    s[3] = torch.minimum(s[3], torch.zeros(()))
    t[4] = -t[4].abs()
    t[4, 17] = -0.0
    _check(D, kind, s.to(dtype), t.to(dtype), T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "jsd"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_16bit_rows_with_one_towering_logit(D, kind, dtype):
    """A logit far above the rest of its row, at every position inside a 16-byte chunk in turn: a maximum
    that missed it would let the sums of exponentials overflow."""
    s, t = _pair(8, 4096, dtype, 9)
    s, t = s.float(), t.float()
    for r in range(8):
        s[r, 8 * (3 + 17 * r) + r] = 150.0
        t[r, 8 * (5 + 11 * r) + (7 - r)] = 140.0
    _check(D, kind, s.to(dtype), t.to(dtype), T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("dtype,V,pitch,offset", [(torch.bfloat16, 5001, 5001, 0),      # contiguous odd rows: every row starts elsewhere on the 16-byte grid
                                                  (torch.float32, 1003, 1003, 0),
                                                  (torch.float16, 7, 7, 0),               # rows shorter than a chunk
                                                  (torch.bfloat16, 4099, 4104, 3),        # a column slice of aligned rows
                                                  (torch.float32, 20001, 20001, 0)])      # 1024 threads
@pytest.mark.parametrize("in_place", [False, True])
def test_dense_rows_off_the_16_byte_grid(D, kind, dtype, V, pitch, offset, in_place):
    """Student and teacher rows of one dtype that do not start on 16-byte boundaries or do not end on one
    stay in the register kernel (units from the student row's first 16-byte boundary on, the columns beside
    them one by one), with masked rows and the gradient written over the logits."""
    R = 6
    s, t = _pair(R, V, dtype, 13)
    valid = torch.ones(R, dtype=torch.bool)
    valid[1] = False
    if kind == "rkl":
        t[:, ::5] = -float("inf")                     # a teacher without mass on a fifth of the columns, the last one among them or not
    loss64, rows64, grad64 = O.mean_loss_and_grad(kind, s, 1.3, t_logits=t[valid], valid=valid, dtype=torch.float64)
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R - 1, dtype=torch.int32)

    def on_gpu(x):
        if pitch == V:
            return x.to(DEV)
        wide = torch.zeros(x.shape[0], pitch + 8, dtype=dtype, device=DEV)
        wide[:, offset:offset + V] = x.to(DEV)
        return wide[:, offset:offset + V]

    xs, xt = on_gpu(s), on_gpu(t[valid])
    rl, grad = D.div_dense(kind, xs, xt, row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / (R - 1), grad_out=xs if in_place else None)
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    assert rl[1].item() == 0 and torch.count_nonzero(grad[1]) == 0
    err = (grad.cpu().double() - grad64).abs()
    sel = torch.nonzero(valid).squeeze(-1)
    bound = O.storage_tolerance(grad64, dtype, RTOL[dtype])
    bound[sel] = O.dense_gradient_tolerance(grad64[sel], s[sel], t[valid], rows64, 1.3, 1.3, 1.0 / (R - 1), dtype, RTOL[dtype], kind=kind)
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
def test_dense_vocab_32000_bf16_temperature_ragged_mask(D, kind):
    s, t = _pair(48, 32000, torch.bfloat16, 2, noise=1.5)
    valid = torch.ones(48, dtype=torch.bool)
    valid[30:41] = False
    _check(D, kind, s, t[valid], T=2.0, valid=valid)


def test_dense_fp32_vocab_32000_config1_shape(D):
    s, t = _pair(32, 32000, torch.float32, 3)
    valid = torch.arange(32) < 29
    _check(D, "fkl", s, t[valid], T=1.0, valid=valid)
    _check(D, "jsd", s, t[valid], T=1.5, valid=valid, teacher_T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
def test_teacher_with_zero_mass_entries(D, kind):
    # -inf teacher logits: zero mass; RKL renormalises the student over the remaining support
    s, t = _pair(10, 4096, torch.float32, 4)
    g = torch.Generator().manual_seed(4)
    drop = torch.rand(10, 4096, generator=g) < 0.6
    t = t.masked_fill(drop, float("-inf"))
    _check(D, kind, s, t, T=1.0)


@pytest.mark.parametrize("V,dtype", [(1001, torch.float32), (70000, torch.bfloat16), (50264, torch.float32),
                                     (128256, torch.bfloat16), (151936, torch.bfloat16), (70000, torch.float32), (70001, torch.bfloat16)])
def test_dense_rows_beyond_the_register_budget(D, V, dtype):
    # in column parts; without a workspace up to 131072 16-bit / 65536 fp32 columns the student row stays on the CU and the
    # teacher row is streamed, beyond both are streamed (multi-pass, 16-byte loads), and odd vocabularies take the scalar kernel
    s, t = _pair(5, V, dtype, 5)
    for kind in ("fkl", "rkl", "jsd"):
        for split in (True, False):
            _check(D, kind, s, t, T=1.3, split=split)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("V", [70000, 151936])
def test_wide_rows_with_zero_mass_teacher_entries(D, kind, V):
    # rows swept from memory take maxima and sums in one sweep with running maxima: stretches without any
    # teacher mass (the first 20000 columns, and 60 % of the rest) must neither poison nor bias the sums,
    # and the largest entries sit late in the row so that the running maxima do move
    s, t = _pair(6, V, torch.bfloat16, 8)
    g = torch.Generator().manual_seed(8)
    drop = torch.rand(6, V, generator=g) < 0.6
    drop[:, :20000] = True
    t = t.float().masked_fill(drop, float("-inf"))
    t[:, V - 5000:] += 6.0
    s = s.float()
    s[:, V // 2:] += 4.0
    _check(D, kind, s.to(torch.bfloat16), t.to(torch.bfloat16), T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
def test_dense_wide_16bit_student_fp32_teacher_with_masked_rows(D, kind):
    s, t = _pair(9, 100000, torch.bfloat16, 6, torch.float32)
    valid = torch.ones(9, dtype=torch.bool)
    valid[[2, 7]] = False
    _check(D, kind, s, t[valid], T=1.7, valid=valid, teacher_T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("V,t_dtype", [(32000, torch.bfloat16), (70000, torch.float16), (151936, torch.bfloat16)])
def test_dense_fp32_student_against_a_16bit_teacher(D, kind, V, t_dtype):
    # the student already cast to fp32 by the caller, the teacher as its model left it: register kernels up to
    # 1024 threads x 4 units, the student row on the CU beyond, both rows streamed beyond that
    s, t = _pair(7, V, torch.float32, 12, t_dtype)
    valid = torch.ones(7, dtype=torch.bool)
    valid[3] = False
    _check(D, kind, s, t[valid], T=1.2, valid=valid, teacher_T=0.9)


def test_dense_identical_distributions_give_zero(D):
    s, _ = _pair(8, 8192, torch.float32, 6)
    for kind in ("fkl", "rkl", "jsd"):
        rl, grad = D.div_dense(kind, s.to(DEV), s.to(DEV))
        assert rl.abs().max().item() < 1e-5 and grad.abs().max().item() < 2e-6


def test_jsd_bounded_by_ln2_on_disjoint_supports(D):
    a = torch.full((2, 1024), float("-inf"))
    b = a.clone()
    a[:, :500] = torch.randn(2, 500)
    b[:, 500:] = torch.randn(2, 524)
    rl, _ = D.div_dense("jsd", a.to(DEV), b.to(DEV))
    np.testing.assert_allclose(rl.cpu().numpy(), np.log(2.0), rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_jsd_with_student_logits_of_minus_infinity(D, dtype):
    """Masked vocabulary entries (-inf) in the student row, some of them where the teacher has no mass
    either: the loss stays finite and equals the oracle's, the gradient is exactly 0 on the masked columns
    and matches central differences of the oracle's float64 loss elsewhere (autograd through the oracle
    yields NaN for such rows: 0 * inf in the branch that `where` drops)."""
    R, V = 3, 2048
    s, t = _pair(R, V, dtype, 21)
    s, t = s.float(), t.float()
    s[:, 40:90] = -float("inf")
    t[:, 70:130] = -float("inf")
    s[1, ::7] = -float("inf")
    s, t = s.to(dtype), t.to(dtype)
    rl, grad = D.div_dense("jsd", s.to(DEV), t.to(DEV), T=1.5, teacher_T=1.0)
    rows64 = O.jsd_dense_rows(s.double() / 1.5, t.double())
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=2e-5)
    g = grad.cpu().double()
    assert torch.isfinite(g).all() and torch.count_nonzero(g[torch.isinf(s.float())]) == 0
    gen = torch.Generator().manual_seed(5)
    eps = 1e-5
    for _ in range(24):
        r = int(torch.randint(0, R, (1,), generator=gen))
        j = int(torch.randint(0, V, (1,), generator=gen))
        if torch.isinf(s[r, j].float()):
            continue
        hi, lo = s[r].double().clone(), s[r].double().clone()
        hi[j] += eps
        lo[j] -= eps
        fd = (O.jsd_dense_rows(hi[None] / 1.5, t[r:r + 1].double()) - O.jsd_dense_rows(lo[None] / 1.5, t[r:r + 1].double())).item() / (2 * eps)
        tol = (1e-4 if dtype == torch.float32 else 2e-3 + 2.0 ** -8) * abs(fd) + 2e-9
        assert abs(g[r, j].item() - fd) <= tol, (r, j, g[r, j].item(), fd)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [2048, 2051])
def test_reverse_kl_with_student_logits_of_minus_infinity(D, dtype, V):
    """Masked vocabulary entries (-inf) in the student row where the teacher has mass carry no student mass
    (0 log 0 = 0): loss and gradient stay finite, the gradient is exactly 0 on the masked columns and on the
    columns without teacher mass, and matches central differences of the oracle's float64 loss elsewhere.
    (The reference's F.kl_div(log_target=True) yields NaN for such a row.)  2051 columns with one fp32 row take
    the scalar kernel."""
    R = 3
    s, t = _pair(R, V, dtype, 22)
    s, t = s.float(), t.float()
    s[:, 40:90] = -float("inf")
    t[:, 70:130] = -float("inf")
    s[1, ::7] = -float("inf")
    t_dtype = torch.float32 if V % 8 else dtype
    s, t = s.to(dtype), t.to(t_dtype)
    rl, grad = D.div_dense("rkl", s.to(DEV), t.to(DEV), T=1.5, teacher_T=1.0)
    rows64 = O.rev_kl_dense_rows(s.double() / 1.5, t.double())
    assert torch.isfinite(rows64).all()
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=2e-5)
    g = grad.cpu().double()
    assert torch.isfinite(g).all() and torch.count_nonzero(g[torch.isinf(s.float()) | torch.isinf(t.float())]) == 0
    gen = torch.Generator().manual_seed(5)
    eps = 1e-5
    for _ in range(24):
        r = int(torch.randint(0, R, (1,), generator=gen))
        j = int(torch.randint(0, V, (1,), generator=gen))
        if torch.isinf(s[r, j].float()) or torch.isinf(t[r, j].float()):
            continue
        hi, lo = s[r].double().clone(), s[r].double().clone()
        hi[j] += eps
        lo[j] -= eps
        fd = (O.rev_kl_dense_rows(hi[None] / 1.5, t[r:r + 1].double()) - O.rev_kl_dense_rows(lo[None] / 1.5, t[r:r + 1].double())).item() / (2 * eps)
        tol = (1e-4 if dtype == torch.float32 else 2e-3 + 2.0 ** -8) * abs(fd) + 2e-9
        assert abs(g[r, j].item() - fd) <= tol, (r, j, g[r, j].item(), fd)


@pytest.mark.parametrize("kind", ["fkl", "rkl"])
@pytest.mark.parametrize("dtype,t_dtype,V,threads", [
    (torch.float32, torch.float32, 32000, 256),      # 4 parts of 256 threads x 4 units of 8 columns, cut evenly: 3 x 1024 + 928 units
    (torch.float32, torch.float32, 32000, 512),      # 2 parts of 512 x 4
    (torch.bfloat16, torch.bfloat16, 32000, 256),    # 2 parts of 256 x 8
    (torch.bfloat16, torch.bfloat16, 128256, 0),     # the library's choice: 4 parts of 512 x 8
    (torch.bfloat16, torch.bfloat16, 128256, 256),   # 8 parts
    (torch.float16, torch.float16, 65536, 256),      # 4 full parts
    (torch.float16, torch.float16, 262144, 0),       # 8 full parts of 512 x 8
    (torch.bfloat16, torch.float32, 50264, 256),     # mixed pair (6 units per thread): 5 parts, the last one shorter
    (torch.bfloat16, torch.float32, 50304, 0),       # the library's choice: 3 parts of 512 x 6
    (torch.float16, torch.float32, 12296, 256),      # one unit more than a part holds: 2 parts of 832 and 705 units
    (torch.float16, torch.float32, 40000, 0),        # mixed pair, 4 parts of 256 x 6
    (torch.bfloat16, torch.float32, 200064, 0),      # too wide for 8 parts of 512 x 6: 5 parts of 1024 threads
    (torch.float32, torch.float32, 151936, 0),       # the same for an fp32 pair: 5 parts of 1024 x 4
    (torch.float32, torch.float32, 40000, 1024),     # 2 parts of 1024 x 4
    (torch.float32, torch.float32, 65536, 0),        # 4 full parts of 512 x 4
    (torch.float32, torch.bfloat16, 50304, 0),       # fp32 student against a 16-bit teacher: 4 parts of 512 x 4
    (torch.float32, torch.float16, 32000, 256),      # 4 parts of 256 x 4
    (torch.float32, torch.bfloat16, 151936, 0)])     # 5 parts of 1024 x 4
def test_rows_cut_into_column_parts(D, kind, dtype, t_dtype, V, threads):
    """dl_div_dense_ws: wide forward / reverse-KL rows cut into parts of 256, 512 or 1024 threads that exchange their
    maxima and sums through the workspace.  Both forms against the oracle, the row losses of the two against each other
    (the same numbers to fp32 rounding), with parts that do
    not wait for their partners (the second launch finishes them: the same bits), twice (the same bits), with
    masked rows, and with the gradient written over the logits."""
    s, t = _pair(13, V, dtype, 31, t_dtype, noise=1.5, std=3.0)
    valid = torch.ones(13, dtype=torch.bool)
    valid[[0, 6]] = False
    _check(D, kind, s, t[valid], 1.3, valid=valid, teacher_T=1.0, part_threads=threads)
    _check(D, kind, s, t[valid], 1.3, valid=valid, teacher_T=1.0, split=False)
    rm = torch.full((13,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(11, dtype=torch.int32)
    xs, xt, rm = s.to(DEV), t[valid].to(DEV), rm.to(DEV)
    kw = dict(row_map=rm, T=1.3, teacher_T=1.0, grad_scale=1.0 / 11, part_threads=threads)
    assert D._lib.load().dl_div_dense_workspace_bytes(D.ops.KINDS[kind], D.ops._DT[dtype], D.ops._DT[t_dtype], 13, V) > 0
    rl, g = D.div_dense(kind, xs, xt, **kw)
    rl2, g2 = D.div_dense(kind, xs, xt, **kw)
    rl3, g3 = D.div_dense(kind, xs, xt, no_wait=True, **kw)
    assert torch.equal(rl, rl2) and torch.equal(g, g2) and torch.equal(rl, rl3) and torch.equal(g, g3)
    rl1, _ = D.div_dense(kind, xs, xt, split=False, row_map=rm, T=1.3, teacher_T=1.0, grad_scale=1.0 / 11)
    np.testing.assert_allclose(rl.cpu().numpy(), rl1.cpu().numpy(), rtol=2e-6, atol=1e-7)
    for no_wait in (False, True):
        y = xs.clone()
        rl4, g4 = D.div_dense(kind, y, xt, grad_out=y, no_wait=no_wait, **kw)
        assert g4.data_ptr() == y.data_ptr() and torch.equal(rl, rl4) and torch.equal(g, y)


@pytest.mark.parametrize("kind", ["fkl", "rkl"])
def test_a_column_part_without_teacher_mass_or_without_student_mass(D, kind):
    """Whole column parts of -inf: a teacher that masks a stretch of the vocabulary as wide as a part (no
    support there for reverse KL, no mass for forward KL), and a student that masks another one where the
    teacher has none either.  The parts' records then carry -inf maxima; the row's statistics come from the
    other parts and the masked columns get zero gradient."""
    R, V = 5, 32768                                          # four parts of 8192 fp32 columns
    s, t = _pair(R, V, torch.float32, 41, noise=1.5, std=3.0)
    t[:, 8192:16384] = -float("inf")                          # part 1: no teacher mass
    t[:, 24576:] = -float("inf")
    s[:, 24576:] = -float("inf")                              # part 3: neither
    _check(D, kind, s, t, 1.1, part_threads=256)
    rl, g = D.div_dense(kind, s.to(DEV), t.to(DEV), T=1.1, part_threads=256)
    rl2, g2 = D.div_dense(kind, s.to(DEV), t.to(DEV), T=1.1, no_wait=True, part_threads=256)
    assert torch.isfinite(rl).all() and torch.isfinite(g).all() and torch.equal(rl, rl2) and torch.equal(g, g2)
    assert torch.count_nonzero(g[:, 24576:]) == 0
    if kind == "rkl":
        assert torch.count_nonzero(g[:, 8192:16384]) == 0


def test_synthetic_configs_1_and_2_at_reduced_rows(D):
    from llm_distillery_amd import synthetic as S
    c = S.config1(DEV, B=1, S=64)
    assert int(c["valid"].sum()) == 57                    # ceil(10 %) of 64 = 7 padded
    _check(D, "fkl", c["logits"].cpu(), c["t_logits"].cpu(), 1.0, valid=c["valid"].cpu())
    c = S.config2(DEV, B=2, S=48)
    assert c["t_logits"].shape[0] == int(c["lengths"].sum())
    _check(D, "jsd", c["logits"].cpu(), c["t_logits"].cpu(), 2.0, valid=c["valid"].cpu())


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("V,dtype", [(32000, torch.bfloat16), (1001, torch.float32), (128256, torch.bfloat16)])
def test_dense_gradient_may_overwrite_the_logits(D, kind, V, dtype):
    g = torch.Generator().manual_seed(17)
    x = (torch.randn(12, V, generator=g) * 2).to(dtype).to(DEV)
    t = (0.7 * x.float() + torch.randn(12, V, generator=g).to(DEV)).to(dtype)
    rl, grad = D.div_dense(kind, x, t, T=1.3)
    y = x.clone()
    rl2, g2 = D.div_dense(kind, y, t, T=1.3, grad_out=y)
    assert g2.data_ptr() == y.data_ptr() and torch.equal(rl, rl2) and torch.equal(grad, y)



@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("dtype,t_dtype,V,pitch", [(torch.float32, torch.bfloat16, 5, 5), (torch.bfloat16, torch.float32, 2047, 2047),
                                                   (torch.float32, torch.float16, 8197, 8204), (torch.float16, torch.float32, 20003, 20003),
                                                   (torch.float32, torch.bfloat16, 20001, 20001)])
def test_dense_rows_off_the_grid_with_a_teacher_of_another_dtype(D, kind, dtype, t_dtype, V, pitch):
    """Mixed dtypes off the 16-byte grid: the register kernels as for equal ones, the V % 8 columns behind the last unit
    in the first threads; with masked rows and rows of a wider pitch."""
    R = 7
    s, t = _pair(R, V, dtype, 21, t_dtype)
    valid = torch.ones(R, dtype=torch.bool)
    valid[3] = False
    wide = torch.full((R, pitch), 1e4, dtype=dtype)          # what lies behind a row must not be read as part of it
    wide[:, :V] = s
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R - 1, dtype=torch.int32)
    loss64, rows64, grad64 = O.mean_loss_and_grad(kind, s, 1.3, t_logits=t[valid], valid=valid, dtype=torch.float64)
    rl, grad = D.div_dense(kind, wide.to(DEV)[:, :V], t[valid].to(DEV), row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / (R - 1))
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    assert rl[3].item() == 0 and torch.count_nonzero(grad[3]) == 0
    sel = torch.nonzero(valid).squeeze(-1)
    bound = O.storage_tolerance(grad64, dtype, RTOL[dtype])
    bound[sel] = O.dense_gradient_tolerance(grad64[sel], s[sel], t[valid], rows64, 1.3, 1.3, 1.0 / (R - 1), dtype, RTOL[dtype], kind=kind)
    err = (grad.cpu().double() - grad64).abs()
    assert (err <= bound).all(), f"worst ratio {(err / bound).max():.2f}"


@pytest.mark.parametrize("kind", ["fkl", "rkl"])
@pytest.mark.parametrize("dtype,t_dtype,V,threads", [(torch.bfloat16, torch.bfloat16, 16385, 256), (torch.bfloat16, torch.bfloat16, 65543, 512),
                                                     (torch.float16, torch.float16, 16391, 256), (torch.float32, torch.float32, 8193, 256),
                                                     (torch.float32, torch.float32, 33001, 0), (torch.bfloat16, torch.float32, 49157, 0),
                                                     (torch.float32, torch.float16, 65537, 512), (torch.float32, torch.bfloat16, 70001, 1024)])
@pytest.mark.parametrize("no_wait", [False, True])
def test_dense_rows_off_the_grid_in_column_parts(D, kind, dtype, t_dtype, V, threads, no_wait):
    """Column parts of rows that are no whole number of 8-column units long and start anywhere: the columns behind the
    last unit belong to the last part; also where every part goes through the retry list."""
    R = 5
    s, t = _pair(R, V, dtype, 23, t_dtype)
    valid = torch.ones(R, dtype=torch.bool)
    valid[2] = False
    s[0, V - 1] = 60.0                                       # a row whose maximum is its last column
    _check(D, kind, s, t[valid], T=1.3, valid=valid, no_wait=no_wait, part_threads=threads)


@pytest.mark.parametrize("dtype,t_dtype,V,threads", [
    (torch.bfloat16, torch.float32, 98922, 0),       # off the grid, 3 columns behind the last unit
    (torch.float32, torch.bfloat16, 40003, 256),
    (torch.float16, torch.float32, 200064, 0),       # parts of 1024 threads
    (torch.float32, torch.float32, 50257, 0),        # fp32 pairs keep the gradient's ingredients in the registers
    (torch.float32, torch.float32, 65536, 512),
    (torch.bfloat16, torch.bfloat16, 70001, 0),
    (torch.float16, torch.float16, 32776, 256)])     # three parts, the last one shorter
def test_jsd_rows_cut_into_column_parts(D, dtype, t_dtype, V, threads):
    """JSD parts meet twice: against the oracle and against one workgroup per row, twice and with parts that wait at neither
    meeting (two further launches finish them) the same bits, with masked rows, a part without any mass, and the gradient
    written over the logits."""
    R = 9
    s, t = _pair(R, V, dtype, 35, t_dtype, noise=1.5, std=3.0)
    s[2, V // 2:] = -float("inf")
    t[2, V // 2:] = -float("inf")
    valid = torch.ones(R, dtype=torch.bool)
    valid[[0, 6]] = False
    _check(D, "jsd", s[valid][:1], t[valid][:1], 1.3, teacher_T=1.0, part_threads=threads)
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R - 2, dtype=torch.int32)
    xs, xt, rm = s.to(DEV), t[valid].to(DEV), rm.to(DEV)
    kw = dict(row_map=rm, T=1.3, teacher_T=1.0, grad_scale=1.0 / (R - 2), part_threads=threads)
    assert D._lib.load().dl_div_dense_workspace_bytes(D.ops.KINDS["jsd"], D.ops._DT[dtype], D.ops._DT[t_dtype], R, V) > 0
    rl, g = D.div_dense("jsd", xs, xt, **kw)
    rl2, g2 = D.div_dense("jsd", xs, xt, **kw)
    rl3, g3 = D.div_dense("jsd", xs, xt, no_wait=True, **kw)
    assert torch.equal(rl, rl2) and torch.equal(g, g2) and torch.equal(rl, rl3) and torch.equal(g, g3)
    assert torch.isfinite(rl).all() and torch.isfinite(g).all() and torch.count_nonzero(g[2, V // 2:]) == 0
    assert torch.count_nonzero(rl[~valid.to(DEV)]) == 0 and torch.count_nonzero(g[~valid.to(DEV)]) == 0
    rl1, g1 = D.div_dense("jsd", xs, xt, split=False, row_map=rm, T=1.3, teacher_T=1.0, grad_scale=1.0 / (R - 2))
    np.testing.assert_allclose(rl.cpu().numpy(), rl1.cpu().numpy(), rtol=2e-6, atol=1e-7)
    assert torch.linalg.norm(g.double() - g1.double()) <= 3e-3 * torch.linalg.norm(g1.double())
    for no_wait in (False, True):
        y = xs.clone()
        rl4, g4 = D.div_dense("jsd", y, xt, grad_out=y, no_wait=no_wait, **kw)
        assert g4.data_ptr() == y.data_ptr() and torch.equal(rl, rl4) and torch.equal(g, y)


@pytest.mark.parametrize("dtype,t_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                           (torch.float32, torch.float16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("V,threads", [(8192, 0), (8195, 0), (12000, 0), (20000, 0), (20005, 0),      # rows held whole, on the grid and off it
                                       (40960, 256), (40963, 256), (40960, 512), (66001, 512)])      # rows in column parts
def test_jsd_without_a_gradient(D, dtype, t_dtype, V, threads):
    """Calls without a gradient run instances of their own, which keep nothing for it: the row losses are those of float64, and of the
    call with a gradient, also where every part is finished by the later launches; masked rows, a masked student column."""
    R = 7
    g = torch.Generator().manual_seed(V + threads)
    s, t = (torch.randn(R, V, generator=g) * 3).to(dtype), (torch.randn(R, V, generator=g) * 3).to(t_dtype)
    s[2, :V // 2] = float("-inf")
    valid = torch.ones(R, dtype=torch.bool)
    valid[4] = False
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R - 1, dtype=torch.int32)
    ref = O.jsd_dense_rows(s[valid].double() / 1.3, t[valid].double())
    xs, xt = s.to(DEV), t[valid].to(DEV)
    for no_wait in (False, True):
        kw = dict(row_map=rm.to(DEV), T=1.3, teacher_T=1.0, part_threads=threads, no_wait=no_wait)
        rl, none = D.div_dense("jsd", xs, xt, want_grad=False, **kw)
        assert none is None and rl[4] == 0
        np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), ref.numpy(), rtol=3e-5, atol=3e-6)      # as _check
        with_grad, _ = D.div_dense("jsd", xs, xt, **kw)
        torch.testing.assert_close(rl, with_grad, rtol=3e-5, atol=3e-6)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("dtype,t_dtype,V,threads", [(torch.bfloat16, torch.bfloat16, 40000, 256), (torch.bfloat16, torch.bfloat16, 40003, 256),
                                                     (torch.float32, torch.float32, 33000, 256), (torch.float32, torch.float32, 33001, 256),
                                                     (torch.float16, torch.float16, 49155, 256), (torch.bfloat16, torch.float32, 49157, 0),
                                                     (torch.float32, torch.bfloat16, 49160, 512)])
@pytest.mark.parametrize("T", [1.0, 2.0])
def test_a_column_part_masked_with_low_finite_values(D, kind, dtype, t_dtype, V, threads, T):
    """A stretch of the vocabulary wider than a column part, masked with the lowest value of the type or other finite ones
    instead of -inf, in both rows, in the teacher's alone (forward KL, JSD) or in the student's alone (JSD): what -inf
    gives there, which is held against the oracle.  (The value times 1 / T overflows at T = 1 and does not at T = 2.)"""
    values = [v for v in (-3.38e38, -1e30, -2e9, -1e9, -6e4) if dtype != torch.float16 or v == -6e4] + [torch.finfo(dtype).min]
    sides = {"fkl": ("both", "teacher"), "rkl": ("both",), "jsd": ("both", "teacher", "student")}[kind]
    rows = [(side, v) for side in sides for v in values]
    R = len(rows)
    s, t = _pair(R, V, dtype, V, t_dtype, noise=1.5, std=3.0)
    s0, t0 = s.clone(), t.clone()
    a, b = int(0.24 * V), int(0.76 * V)
    for r, (side, v) in enumerate(rows):
        if side != "teacher":
            s[r, a:b], s0[r, a:b] = v, -float("inf")
        if side != "student":
            t[r, a:b], t0[r, a:b] = max(v, torch.finfo(t_dtype).min), -float("inf")
    assert D._lib.load().dl_div_dense_workspace_bytes(D.ops.KINDS[kind], D.ops._DT[dtype], D.ops._DT[t_dtype], R, V) > 0
    rl0, g0 = D.div_dense(kind, s0.to(DEV), t0.to(DEV), T=T, part_threads=threads)
    if kind != "jsd":
        _check(D, kind, s0, t0, T, part_threads=threads)
    else:                                                # (autograd's gradient of the oracle is NaN where a probability is 0)
        rows64 = O.DENSE_ROWS[kind](s0.double() / T, t0.double() / T)
        np.testing.assert_allclose(rl0.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
        g1 = D.div_dense(kind, s0.to(DEV), t0.to(DEV), T=T, split=False)[1]
        assert torch.linalg.norm(g0.double() - g1.double()) <= 3e-3 * torch.linalg.norm(g1.double())
    for no_wait in (False, True):
        rl, g = D.div_dense(kind, s.to(DEV), t.to(DEV), T=T, part_threads=threads, no_wait=no_wait)
        # the parts' sums are those of the -inf masks; a part above the line where it counts as masked adds terms of 2^-80000
        np.testing.assert_allclose(rl.cpu().numpy(), rl0.cpu().numpy(), rtol=1e-6, err_msg=str(rows))
        assert torch.isfinite(g).all() and torch.allclose(g.float(), g0.float(), rtol=1e-2 if dtype != torch.float32 else 1e-5, atol=1e-9)


@pytest.mark.parametrize("dtype,t_dtype,V", [(torch.float32, torch.float32, 50257), (torch.float32, torch.float32, 20003),
                                             (torch.float32, torch.bfloat16, 100277), (torch.float32, torch.float16, 1003)])
@pytest.mark.parametrize("T", [1.0, 1.5])
def test_reverse_kl_gradient_rows_off_the_grid_sum_to_nothing(D, dtype, t_dtype, V, T):
    """sum_j r_j (log ratio_j - mean) is 0 about the mean of the ratios as they are rounded: what is left is the rounding of the
    mean itself, a sum of a few units in fp32 (2^-22 of it, taken as the root mean square over the rows); about the row's loss it
    is the rounding of the two normalisers, half a unit in the last place of values of 8 to 32: 2^-20."""
    R = 64
    s, t = _pair(R, V, dtype, V, t_dtype)
    rl, g = D.div_dense("rkl", s.to(DEV), t.to(DEV), T=T)
    assert (g.double().sum(-1) * T).square().mean().sqrt().item() <= 2.0 ** -22
    _, rows64, grad64 = O.mean_loss_and_grad("rkl", s, T, t_logits=t, dtype=torch.float64)
    np.testing.assert_allclose(rl.cpu().double().numpy(), rows64.numpy(), rtol=3e-5, atol=3e-6)
    assert torch.linalg.norm(g.cpu().double() - grad64 * R) <= 1e-6 * torch.linalg.norm(grad64 * R)


@pytest.mark.parametrize("kind", ["fkl", "rkl", "jsd"])
@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 128256), (torch.float32, 150000)])      # the student's row on the CU; both rows streamed
@pytest.mark.parametrize("T", [1.0, 2.0])
def test_streamed_rows_masked_with_low_finite_values(D, kind, dtype, V, T):
    """Rows swept from memory choose a bias per thread from the columns it has met: where those are all masked with low finite
    values (the first two thirds of the row), the row's loss and gradient are those of an -inf mask."""
    values = [torch.finfo(dtype).min, -1e30, -2e9, -1e9, -6e4]
    R = len(values)
    s, t = _pair(R, V, dtype, V, noise=1.5, std=3.0)
    b = 2 * V // 3
    s[:, :b] = t[:, :b] = -float("inf")
    rl0, g0 = D.div_dense(kind, s.to(DEV), t.to(DEV), T=T, split=False)
    if kind != "jsd":
        _check(D, kind, s, t, T, split=False)
    for r, v in enumerate(values):
        s[r, :b] = t[r, :b] = v
    rl, g = D.div_dense(kind, s.to(DEV), t.to(DEV), T=T, split=False)
    np.testing.assert_allclose(rl.cpu().numpy(), rl0.cpu().numpy(), rtol=1e-6)
    assert torch.isfinite(g).all() and torch.allclose(g.float(), g0.float(), rtol=1e-2 if dtype != torch.float32 else 1e-5, atol=1e-9)
