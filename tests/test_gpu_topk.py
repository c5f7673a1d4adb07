"""GPU parity of the sparse-teacher kernels (through the C ABI) against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-3, torch.float16: 2e-3}


@pytest.fixture(scope="module")
def D():
    import llm_distillery_amd as d
    d._lib.load()
    return d


def _case(R, V, K, dtype, seed, std=2.0, idx_dtype=torch.int32, val_dtype=torch.float16):
    g = torch.Generator().manual_seed(seed)
    logits = (torch.randn(R, V, generator=g) * std).to(dtype)
    tl = torch.log_softmax(logits.float() + torch.randn(R, V, generator=g), -1)
    tv, ti = torch.topk(tl, K)
    return logits, tv.to(val_dtype), ti.to(idx_dtype)


def _check(D, kind, logits, tv, ti, T, valid=None, teacher_T=None, hooks=None, **tol_over):
    R, V = logits.shape
    n_valid = R if valid is None else int(valid.sum())
    loss64, rows64, grad64 = O.mean_loss_and_grad(kind, logits, T, t_vals=tv, t_idx=ti, valid=valid, t_T=teacher_T,
                                             dtype=torch.float64)
    row_map = None
    if valid is not None:
        rm = torch.full((R,), -1, dtype=torch.int32)
        rm[valid] = torch.arange(n_valid, dtype=torch.int32)
        row_map = rm.to(DEV)
    rl, grad = D.div_topk(kind, logits.to(DEV), tv.to(DEV), ti.to(DEV), row_map=row_map, T=T, teacher_T=teacher_T,
                          grad_scale=1.0 / n_valid, **(hooks or {}))
    loss = D.reduce_sum(rl, 1.0 / n_valid)
    torch.cuda.synchronize()
    rows_gpu = rl.cpu()
    if valid is not None:
        assert torch.count_nonzero(rows_gpu[~valid]) == 0
        assert torch.count_nonzero(grad.cpu()[~valid]) == 0
        rows_gpu = rows_gpu[valid]
    # loss: 1e-5 relative against the float64 oracle (fp32 accumulation in the kernel)
    np.testing.assert_allclose(loss.item(), loss64.item(), rtol=1e-5)
    np.testing.assert_allclose(rows_gpu.double().numpy(), rows64.numpy(), rtol=2e-5, atol=2e-6)
    # gradients, entry by entry: 1e-4 (fp32 logits) / 2e-3 (16-bit logits) of the entry's own value, the half
    # ulp that storing it in the logits' dtype may add, and fp32 rounding of the entry's own cancelling terms
    rtol = tol_over.get("rtol", TOL[logits.dtype])
    err = (grad.cpu().double() - grad64).abs()
    bound = O.topk_gradient_tolerance(kind, grad64, logits, tv, ti, T, teacher_T, 1.0 / n_valid, logits.dtype, rtol, valid)
    bad = err > bound
    assert not bad.any(), f"{int(bad.sum())} gradient entries off; worst ratio {(err / bound).max().item():.3f}"
    return grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["fkl", "rkl"])
def test_topk_small(D, dtype, kind):
    logits, tv, ti = _case(37, 1024, 24, dtype, 1)
    _check(D, kind, logits, tv, ti, T=1.0)


@pytest.mark.parametrize("V,K", [(32000, 200), (128256, 200), (50264, 64), (8192, 400), (32000, 2048), (128256, 1024),
                                 (65536, 2048), (40968, 200), (49152, 1000), (53248, 400), (53256, 16)])      # 512 x 13 chunks up to 53248 columns
def test_fkl_topk_register_path_sizes(D, V, K):
    logits, tv, ti = _case(24, V, K, torch.bfloat16, 2, std=3.0)
    _check(D, "fkl", logits, tv, ti, T=1.0)


def test_fkl_topk_fp32_vocab_32000_temperature_and_mask(D):
    logits, tv, ti = _case(40, 32000, 100, torch.float32, 3)
    valid = torch.ones(40, dtype=torch.bool)
    valid[[3, 4, 17, 39]] = False
    _check(D, "fkl", logits, tv[:36], ti[:36], T=2.0, valid=valid)
    _check(D, "rkl", logits, tv[:36], ti[:36], T=0.7, valid=valid)


def test_validation_asymmetry_teacher_not_scaled(D):
    # classes/student/model.py:501-502: the student is divided by T, the teacher is not
    logits, tv, ti = _case(16, 4096, 32, torch.float32, 4)
    _check(D, "fkl", logits, tv, ti, T=1.7, teacher_T=1.0)


@pytest.mark.parametrize("V", [1000, 32003, 130001])
def test_streaming_path_odd_vocab_and_int64_fp32_teacher(D, V):
    # V not a multiple of the 16-byte chunk -> streaming kernel; teacher as the reference loads it (fp32/int64)
    logits, tv, ti = _case(9, V, 50, torch.bfloat16, 5, idx_dtype=torch.int64, val_dtype=torch.float32)
    _check(D, "fkl", logits, tv, ti, T=1.3)
    _check(D, "rkl", logits, tv, ti, T=1.3)


@pytest.mark.parametrize("dtype,V,pitch,offset", [(torch.bfloat16, 32003, 32003, 0),      # contiguous odd rows: every row starts elsewhere on the grid
                                                  (torch.float32, 1003, 1003, 0),
                                                  (torch.bfloat16, 5001, 5120, 3),          # a column slice of aligned rows: one phase for all rows
                                                  (torch.float16, 7, 7, 0),                 # rows shorter than a chunk
                                                  (torch.float32, 4099, 4104, 2),
                                                  (torch.bfloat16, 50257, 50257, 0),        # wider than 256 x 16 chunks: 512 threads x 13
                                                  (torch.float16, 151665, 151665, 0),       # five
                                                  (torch.float32, 40003, 40003, 0),         # three, of four-byte chunks
                                                  (torch.float32, 10001, 10001, 0)])        # 512 threads x 8 chunks of fp32
@pytest.mark.parametrize("grad_mode", ["fresh", "in_place", "other_phase"])
@pytest.mark.parametrize("kind", ["fkl", "rkl"])
def test_rows_off_the_16_byte_grid(D, kind, dtype, V, pitch, offset, grad_mode):
    """Rows that do not start on 16-byte boundaries or do not end on one.  Forward KL: the register kernels of rows on the
    grid, their chunks from the row's first boundary on, the columns beside them one by one, whatever the gradient row's
    phase (a fresh gradient of the same pitch, the gradient written over the logits, another pitch).  Reverse KL, which
    only gathers from the logits, goes by the gradient rows alone.  All against the oracle."""
    R, K = 7, min(24, V)
    logits, tv, ti = _case(R, V, K, dtype, 61, std=3.0)
    valid = torch.ones(R, dtype=torch.bool)
    valid[2] = False
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(R - 1, dtype=torch.int32)
    tv, ti = tv[valid], ti[valid]
    ti[:, 0] = 0                                                  # entries in the first and the last column
    ti[:, 1] = V - 1
    if K > 3:
        ti[:, 2] = V - 1                                          # and a repeated id there
    tl = torch.log_softmax(logits[valid].float() * 1.1, -1)       # teacher values that belong to those ids
    tv = torch.gather(tl, 1, ti.long()).to(tv.dtype)
    loss64, rows64, grad64 = O.mean_loss_and_grad(kind, logits, 1.3, t_vals=tv, t_idx=ti, valid=valid, dtype=torch.float64)
    full = torch.zeros(R, pitch + 8, dtype=dtype, device=DEV)
    x = full[:, offset:offset + V] if pitch != V else logits.to(DEV)
    if pitch != V:
        x.copy_(logits.to(DEV))
    assert x.stride(0) == (pitch + 8 if pitch != V else V)
    if grad_mode == "fresh":
        out = None
    elif grad_mode == "in_place":
        out = x
    else:
        out = torch.empty(R, x.stride(0) + 1, dtype=dtype, device=DEV)[:, 1:1 + V]
    rl, grad = D.div_topk(kind, x, tv.to(DEV), ti.to(DEV), row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / (R - 1), grad_out=out)
    assert grad_mode == "fresh" or grad.data_ptr() == out.data_ptr()
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=2e-5, atol=2e-6)
    assert rl[2].item() == 0 and torch.count_nonzero(grad[2]) == 0
    err = (grad.cpu().double() - grad64).abs()
    bound = O.topk_gradient_tolerance(kind, grad64, logits, tv, ti, 1.3, None, 1.0 / (R - 1), dtype, TOL[dtype], valid)
    assert (err <= bound).all(), f"worst {(err / bound).max():.2f}"
    if pitch != V and grad_mode != "in_place":      # nothing outside the slice was touched
        assert torch.count_nonzero(full[:, :offset]) == 0 and torch.count_nonzero(full[:, offset + V:]) == 0


@pytest.mark.parametrize("dtype,V,pitch", [(torch.bfloat16, 50257, 50304),      # GPT-2's vocabulary in its padded rows: 512 x 13, one workgroup per row
                                           (torch.bfloat16, 151665, 151936),    # Qwen's: five column parts, the last one ragged
                                           (torch.float16, 100277, 100352),     # four parts of 13 chunks per thread
                                           (torch.float32, 32003, 32064),       # 512 x 16 of four-byte chunks
                                           (torch.float16, 4099, 4104),         # 256 x 4
                                           (torch.bfloat16, 65537, 65544),      # one column more than two parts hold: the third part is one ragged chunk
                                           (torch.float32, 70001, 70008),       # five parts of four-byte chunks
                                           (torch.bfloat16, 262139, 262144)])   # eight parts in four workgroups of 512 threads
@pytest.mark.parametrize("grad_mode", ["fresh", "in_place", "other_pitch", "other_phase"])
def test_crop_of_a_padded_vocabulary(D, dtype, V, pitch, grad_mode):
    """logits[:, :, :crop] of rows padded to a multiple of 16 bytes (classes/student/model.py:408): rows start on
    the 16-byte grid and end inside a chunk.  The register kernels take them like whole rows, one workgroup per
    row or cut into column parts, and move only the columns behind the last whole chunk one by one; nothing beyond the crop
    is written.  A gradient buffer off the grid (other_phase) is written by the same kernels, unaligned.
    With and without waiting for the partners: the oracle's numbers and the same bits."""
    R, K = 11, 48
    logits, tv, ti = _case(R, V, K, dtype, 71, std=3.0)
    valid = torch.ones(R, dtype=torch.bool)
    valid[[2, 10]] = False
    nv = int(valid.sum())
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(nv, dtype=torch.int32)
    tv, ti = tv[valid], ti[valid]
    ti[:, 0] = 0                                                  # entries in the first and the last column
    ti[:, 1] = V - 1
    ti[:, 2] = V - 1                                              # a repeated id in the ragged chunk
    ti[:, 3] = V - V % (8 if dtype != torch.float32 else 4)       # the ragged chunk's first column
    tl = torch.log_softmax(logits[valid].float() * 1.1, -1)
    tv = torch.gather(tl, 1, ti.long()).to(tv.dtype)
    _, rows64, grad64 = O.mean_loss_and_grad("fkl", logits, 1.3, t_vals=tv, t_idx=ti, valid=valid, dtype=torch.float64)
    bound = O.topk_gradient_tolerance("fkl", grad64, logits, tv, ti, 1.3, None, 1.0 / nv, dtype, TOL[dtype], valid)
    results = []
    for no_wait in (False, True):
        full = torch.full((R, pitch), 7.0, dtype=dtype, device=DEV)
        x = full[:, :V]
        x.copy_(logits.to(DEV))
        assert x.data_ptr() % 16 == 0 and (x.stride(0) * x.element_size()) % 16 == 0
        if grad_mode == "fresh":
            out = None
        elif grad_mode == "in_place":
            out = x
        elif grad_mode == "other_pitch":
            out = torch.full((R, pitch + 64), 5.0, dtype=dtype, device=DEV)[:, :V]
        else:
            out = torch.full((R, pitch + 1), 5.0, dtype=dtype, device=DEV)[:, 1:1 + V]
        rl, grad = D.div_topk("fkl", x, tv.to(DEV), ti.to(DEV), row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / nv, grad_out=out,
                              no_wait=no_wait)
        assert grad_mode == "fresh" or grad.data_ptr() == out.data_ptr()
        np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=2e-5, atol=2e-6)
        assert torch.count_nonzero(rl[~valid.to(DEV)]) == 0 and torch.count_nonzero(grad[~valid.to(DEV)]) == 0
        err = (grad.cpu().double() - grad64).abs()
        assert (err <= bound).all(), f"worst {(err / bound).max():.2f}"
        assert (full[:, V:] == 7.0).all()                         # nothing beyond the crop was touched
        if grad_mode == "other_pitch":
            assert (out.as_strided((R, pitch + 64 - V), (pitch + 64, 1), out.storage_offset() + V) == 5.0).all()
        results.append((rl.clone(), grad.clone()))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


def test_streaming_path_rows_larger_than_register_file(D):
    logits, tv, ti = _case(6, 152064, 200, torch.bfloat16, 6)
    _check(D, "fkl", logits, tv, ti, T=1.0)
    logits, tv, ti = _case(4, 100000, 64, torch.float32, 7)
    _check(D, "fkl", logits, tv, ti, T=1.0)


def test_cropped_view_of_wider_model_vocab(D):
    # classes/student/model.py:408 slices [:, :, :crop] out of the model's vocabulary
    g = torch.Generator().manual_seed(8)
    full = (torch.randn(2, 10, 32064, generator=g) * 2).to(torch.bfloat16)
    crop = full[:, :, :32000]
    flat = crop.reshape(20, 32000)
    tl = torch.log_softmax(flat.float() + torch.randn(20, 32000, generator=g), -1)
    tv, ti = torch.topk(tl, 40)
    loss64, rows64, grad_ref = O.mean_loss_and_grad("fkl", flat, 1.0, t_vals=tv, t_idx=ti, dtype=torch.float32)
    dev_full = full.to(DEV)
    rl, grad = D.div_topk("fkl", dev_full[:, :, :32000], tv.to(DEV), ti.to(torch.int32).to(DEV), grad_scale=1 / 20)
    assert grad.shape == (2, 10, 32000)
    np.testing.assert_allclose(rl.cpu().numpy(), rows64.numpy(), rtol=2e-5, atol=2e-6)
    err = (grad.cpu().float().reshape(20, -1) - grad_ref).abs()
    assert (err <= O.sparse_gradient_tolerance(grad_ref.double(), flat, 1.0, ti, torch.bfloat16, 2e-3)).all()


def test_duplicate_ids_ragged_counts_and_out_of_range_ids(D):
    g = torch.Generator().manual_seed(9)
    R, V, K = 12, 2048, 16
    logits = (torch.randn(R, V, generator=g) * 2)
    ti = torch.randint(0, V, (R, K), generator=g)
    ti[:, 5] = ti[:, 2]                  # duplicates inside a row accumulate
    tv = torch.randn(R, K, generator=g)
    _check(D, "fkl", logits, tv, ti.to(torch.int32), T=1.0)
    _check(D, "rkl", logits, tv, ti.to(torch.int32), T=1.0)
    # ragged: only the first cnt entries count; ids outside [0, V) are ignored; empty rows give 0
    cnt = torch.tensor([16, 1, 0, 7, 16, 3, 0, 9, 2, 16, 5, 11], dtype=torch.int32)
    ti2 = ti.clone()
    ti2[4, 3] = V + 5
    ti2[9, 0] = -3
    rl, grad = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti2.to(torch.int32).to(DEV), t_cnt=cnt.to(DEV))
    rl, grad = rl.cpu(), grad.cpu()
    for r in range(R):
        keep = [k for k in range(int(cnt[r])) if 0 <= int(ti2[r, k]) < V]
        if not keep:
            assert rl[r] == 0 and torch.count_nonzero(grad[r]) == 0
            continue
        z = logits[r:r + 1].double()
        t = O.teacher_logprobs_topk(tv[r:r + 1, keep], 1.0, torch.float64)
        ref = O.fwd_kl_topk_rows(z, t, ti2[r:r + 1, keep])
        np.testing.assert_allclose(rl[r].item(), ref.item(), rtol=2e-5, atol=2e-6)


def test_forward_only_and_bit_reproducible(D):
    logits, tv, ti = _case(64, 32000, 200, torch.bfloat16, 10)
    a = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV), want_grad=False)
    assert a[1] is None
    b = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV))
    c = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV))
    assert torch.equal(a[0], b[0]) and torch.equal(b[0], c[0]) and torch.equal(b[1], c[1])
    assert torch.equal(D.reduce_sum(b[0]), D.reduce_sum(c[0]))


def test_errors_are_python_exceptions(D):
    logits, tv, ti = _case(4, 512, 8, torch.float32, 11)
    with pytest.raises(RuntimeError):
        D.div_topk("fkl", logits, tv, ti)                         # CPU tensors: no fallback
    with pytest.raises(RuntimeError):
        D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV)[:, :4])
    big = torch.zeros(2, 4096, dtype=torch.float16, device=DEV)
    with pytest.raises(RuntimeError, match="exceeds"):
        D.div_topk("fkl", torch.zeros(2, 8192, device=DEV), big, torch.zeros(2, 4096, dtype=torch.int32, device=DEV))
    with pytest.raises(ValueError):
        D.div_topk("jsd", logits.to(DEV), tv.to(DEV), ti.to(DEV))


@pytest.mark.parametrize("parts", [1, 2, 4])
def test_split_row_parts_agree_and_give_up_path(D, parts):
    """A 128256-wide row is cut into column parts that exchange statistics through the workspace.
    Every setting must give the oracle's numbers, also when no part waits for its partners
    (the no-wait flag: every part that finds a record missing leaves and is finished by the second
    launch), and the same bits as with waiting.  The hooks travel with the call: the library keeps
    no state."""
    logits, tv, ti = _case(40, 128256, 200, torch.bfloat16, 12, std=3.0)
    valid = torch.ones(40, dtype=torch.bool)
    valid[[0, 7, 33]] = False
    _check(D, "fkl", logits, tv[:37], ti[:37], T=1.0, valid=valid, hooks={"parts": parts})
    waited = _check(D, "fkl", logits, tv[:37], ti[:37], T=2.0, valid=valid, hooks={"parts": parts})
    retried = _check(D, "fkl", logits, tv[:37], ti[:37], T=2.0, valid=valid, hooks={"parts": parts, "no_wait": True})
    assert torch.equal(waited, retried)
    with pytest.raises(ValueError):
        D.div_topk("fkl", logits[:2].to(DEV), tv[:2].to(DEV), ti[:2].to(DEV), parts=3)


@pytest.mark.parametrize("kind,V,dtype", [("fkl", 128256, torch.bfloat16), ("fkl", 32000, torch.bfloat16), ("fkl", 152064, torch.float16),
                                          ("fkl", 1001, torch.float32), ("rkl", 32000, torch.bfloat16)])
def test_gradient_may_overwrite_the_logits(D, kind, V, dtype):
    """grad == logits (same buffer): every kernel holds, or has consumed, what it still needs of a
    row before it writes there, and a split part that gives up leaves its columns untouched for the
    retry launch; results are the bits of the out-of-place call."""
    logits, tv, ti = _case(24, V, 64, dtype, 31)
    x = logits.to(DEV)
    rl, g = D.div_topk(kind, x, tv.to(DEV), ti.to(DEV), T=1.5)
    for no_wait in (False, True):
        y = x.clone()
        rl2, g2 = D.div_topk(kind, y, tv.to(DEV), ti.to(DEV), T=1.5, grad_out=y, no_wait=no_wait)
        assert g2.data_ptr() == y.data_ptr() and torch.equal(rl, rl2) and torch.equal(g, y)



@pytest.mark.parametrize("V,dtype", [(152064, torch.bfloat16), (128256, torch.float32), (262144, torch.float16),
                                     (100000, torch.float32), (98304, torch.float32), (229376, torch.bfloat16),
                                     (100352, torch.bfloat16), (114688, torch.float16), (200064, torch.bfloat16),
                                     (50304, torch.float32), (57344, torch.float32)])
def test_rows_cut_into_five_to_eight_parts(D, V, dtype):
    """Vocabularies beyond 131072 two-byte (65536 four-byte) entries are cut into 5..8 parts of 4096
    chunks, or (four-byte rows of 6 parts and more, two-byte rows of 8) into 3..4 parts of 8192; two-byte rows that do
    not fill their parts -- and four-byte rows of up to five -- into parts of 13 to 15 chunks per thread (100352
    two-byte columns: 4 x 256 x 13, 114688: 4 x 14, 152064: 5 x 15, 200064: 7 x 14; 50304 four-byte columns: 4 x 13); with and without waiting for the partners the oracle's numbers and the same bits."""
    logits, tv, ti = _case(10, V, 48, dtype, 41, std=3.0)
    valid = torch.ones(10, dtype=torch.bool)
    valid[4] = False
    waited = _check(D, "fkl", logits, tv[:9], ti[:9], T=1.3, valid=valid)
    retried = _check(D, "fkl", logits, tv[:9], ti[:9], T=1.3, valid=valid, hooks={"no_wait": True})
    assert torch.equal(waited, retried)


@pytest.mark.parametrize("V,dtype", [(40000, torch.float32), (70000, torch.bfloat16), (98304, torch.float16), (98312, torch.bfloat16)])
def test_rows_cut_into_three_parts(D, V, dtype):
    """Rows of 8193-12288 chunks fill three parts of 4096 chunks, not four: no part may be left
    without columns."""
    logits, tv, ti = _case(11, V, 48, dtype, 43, std=3.0)
    waited = _check(D, "fkl", logits, tv, ti, T=1.1)
    retried = _check(D, "fkl", logits, tv, ti, T=1.1, hooks={"no_wait": True})
    forced = _check(D, "fkl", logits, tv, ti, T=1.1, hooks={"parts": 4})      # not honoured here: same launch, same bits
    assert torch.equal(waited, retried) and torch.equal(waited, forced)
    _check(D, "fkl", logits, tv, ti, T=1.1, hooks={"parts": 2})
    _check(D, "fkl", logits, tv, ti, T=1.1, hooks={"parts": 1})


@pytest.mark.parametrize("V,dtype,K", [(128256, torch.bfloat16, 200), (32000, torch.bfloat16, 400), (32000, torch.float32, 300),
                                       (8200, torch.float16, 64), (40000, torch.float32, 700), (131072, torch.float16, 32)])
def test_rows_cut_into_parts_of_1024_chunks(D, V, dtype, K):
    """The finer cut (up to 16 parts of 256 threads x 4 chunks per row): the oracle's numbers, with
    repeated ids, masked rows, waiting or not."""
    logits, tv, ti = _case(21, V, K, dtype, 47, std=3.0)
    ti[3, 5] = ti[3, 9]
    ti[6, :] = ti[6, 0]
    valid = torch.ones(21, dtype=torch.bool)
    valid[[2, 20]] = False
    waited = _check(D, "fkl", logits, tv[:19], ti[:19], T=1.2, valid=valid, hooks={"parts": 16})
    retried = _check(D, "fkl", logits, tv[:19], ti[:19], T=1.2, valid=valid, hooks={"parts": 16, "no_wait": True})
    assert torch.equal(waited, retried)


def test_a_column_part_that_holds_only_minus_infinity(D):
    """A masked stretch of the vocabulary (-inf logits) as wide as a whole column part: that part has
    no finite maximum; its columns get zero gradient and the row's statistics come from the others."""
    g = torch.Generator().manual_seed(44)
    R, V, K = 9, 128256, 64
    logits = torch.randn(R, V, generator=g) * 3
    logits[:5, 65536:98304] = float("-inf")                   # part 2 of 4, whole
    logits[5:, 120000:] = float("-inf")                       # the tail of the last part
    logits = logits.to(torch.bfloat16)
    tl = torch.log_softmax(logits.float() + torch.randn(R, V, generator=g), -1)
    tv, ti = torch.topk(tl, K)
    grad = _check(D, "fkl", logits, tv.to(torch.float16), ti.to(torch.int32), T=1.0)
    assert torch.count_nonzero(grad[:5, 65536:98304]) == 0 and torch.isfinite(grad.float()).all()
    _check(D, "fkl", logits, tv.to(torch.float16), ti.to(torch.int32), T=1.0, hooks={"no_wait": True})


@pytest.mark.parametrize("kind", ["fkl", "rkl"])
@pytest.mark.parametrize("V,K", [(4096, 24), (128256, 300), (32000, 900)])
def test_entries_of_zero_mass_are_no_entries(D, kind, V, K):
    """A stored log-prob of -inf (a teacher that masks part of its vocabulary) carries no mass: the
    entry counts neither for the loss nor for the support, exactly as if it were not there."""
    logits, tv, ti = _case(7, V, K, torch.bfloat16, 51)
    tv = tv.float()
    dead = torch.zeros(7, K, dtype=torch.bool)
    dead[:, 3::4] = True
    dead[5, 1:] = True                                        # one live entry
    tv_dead = tv.masked_fill(dead, float("-inf"))
    rl, g = D.div_topk(kind, logits.to(DEV), tv_dead.to(DEV), ti.to(DEV), T=1.2)
    # the same rows with the dead entries pointed outside the vocabulary (ignored by contract)
    ti_out = ti.masked_fill(dead, -1)
    rl2, g2 = D.div_topk(kind, logits.to(DEV), tv.to(DEV), ti_out.to(DEV), T=1.2)
    assert torch.isfinite(rl).all() and torch.equal(rl, rl2) and torch.equal(g, g2)


def test_repeated_ids_on_wide_four_byte_rows(D):
    # 16 chunks of fp32 per thread: the shapes that write their corrections behind the dense stores
    g = torch.Generator().manual_seed(78)
    R, V, K = 5, 32000, 96
    logits = torch.randn(R, V, generator=g) * 2
    ti = torch.randint(0, 40, (R, K), generator=g) * 797 + 5
    tv = torch.randn(R, K, generator=g)
    a = _check(D, "fkl", logits, tv, ti.to(torch.int32), T=0.9)
    b = _check(D, "fkl", logits, tv, ti.to(torch.int32), T=0.9)
    assert torch.equal(a, b)
    wide = torch.randn(3, 60000, generator=g) * 2                  # cut into 4 parts
    ti = torch.randint(0, 30, (3, K), generator=g) * 1999 + 11
    _check(D, "fkl", wide, tv[:3], ti.to(torch.int32), T=1.0)


@pytest.mark.parametrize("kind", ["fkl", "rkl"])
def test_rows_whose_ids_all_repeat(D, kind):
    """Every entry of a row on one id, on two ids of one 16-byte chunk, on a handful of ids: the
    masses add per id (the thread that holds the chunk sums them from its list), the result is the
    oracle's and the same bits on every run."""
    g = torch.Generator().manual_seed(77)
    R, V, K = 6, 4096, 512
    logits = (torch.randn(R, V, generator=g) * 2).to(torch.bfloat16)
    ti = torch.empty(R, K, dtype=torch.int64)
    ti[0] = 1234
    ti[1] = torch.where(torch.arange(K) % 2 == 0, 801, 806)
    ti[2] = torch.randint(0, 5, (K,), generator=g) * 1000 + 3
    ti[3] = torch.randint(0, V, (K,), generator=g)
    ti[4] = torch.arange(K) % 16 + 64
    ti[5] = V - 1
    if kind == "rkl":
        # on a single id the reverse-KL gradient is an exact zero made of 512 cancelling terms: nothing
        # for a relative tolerance to hold on to; two ids instead
        ti[0] = torch.where(torch.arange(K) % 3 == 0, 1234, 77)
        ti[5] = torch.where(torch.arange(K) % 5 == 0, V - 1, 0)
    tv = torch.randn(R, K, generator=g)
    a = _check(D, kind, logits, tv, ti.to(torch.int32), T=1.2)
    b = _check(D, kind, logits, tv, ti.to(torch.int32), T=1.2)
    assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 98305),        # the fourth part of 256 x 16 chunks holds one column
                                     (torch.float16, 53255),         # the 512-thread shape's last chunk, 7 columns behind it
                                     (torch.bfloat16, 204801),       # seven parts of 15 chunks per thread
                                     (torch.float32, 65537),         # three parts of four-byte chunks, one column more
                                     (torch.bfloat16, 16391)])       # 256 x 16 chunks, seven columns more
def test_columns_beside_the_chunks_of_a_part(D, dtype, V):
    """Contiguous rows of odd length: every row starts elsewhere on the 16-byte grid, and every column part has columns
    ahead of its first chunk and behind its last.  Entries (one id twice) on those columns on both sides of the parts'
    borders, a -inf logit among them, masked rows; waiting or not the same bits."""
    R, step = 9, 32768 if dtype != torch.float32 else 16384
    g = torch.Generator().manual_seed(V)
    logits = (torch.randn(R, V, generator=g) * 3).to(dtype)
    logits[3, 1] = -float("inf")
    edges = [c + d for c in range(0, V, step) for d in range(-7, 8) if 0 <= c + d < V and c + d != 1] + [V - 1, V - 2, V - 7]
    ids = torch.tensor(sorted(set(edges)))
    ids = torch.cat([ids, torch.tensor([0, V - 1]), torch.randperm(V - 40, generator=g)[:20] + 20])
    valid = torch.ones(R, dtype=torch.bool)
    valid[[1, 8]] = False
    nv = int(valid.sum())
    ti = ids.expand(nv, -1).contiguous().int()
    tv = torch.log_softmax(torch.randn(nv, ids.numel(), generator=g), -1).half()
    rm = torch.full((R,), -1, dtype=torch.int32)
    rm[valid] = torch.arange(nv, dtype=torch.int32)
    _, rows64, grad64 = O.mean_loss_and_grad("fkl", logits, 1.3, t_vals=tv, t_idx=ti, valid=valid, dtype=torch.float64)
    bound = O.topk_gradient_tolerance("fkl", grad64, logits, tv, ti, 1.3, None, 1.0 / nv, dtype, TOL[dtype], valid)
    got = [D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV), row_map=rm.to(DEV), T=1.3, grad_scale=1.0 / nv, no_wait=w)
           for w in (False, True)]
    rl, grad = got[0]
    np.testing.assert_allclose(rl.cpu()[valid].double().numpy(), rows64.numpy(), rtol=2e-5, atol=2e-6)
    assert torch.count_nonzero(rl.cpu()[~valid]) == 0 and torch.count_nonzero(grad.cpu()[~valid]) == 0
    err = (grad.cpu().double() - grad64).abs()
    assert (err <= bound).all(), f"worst {(err / bound).max():.2f}"
    assert torch.equal(rl, got[1][0]) and torch.equal(grad, got[1][1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V,pitch,offset,teachers", [(50304, 50312, 1, 1), (50304, 50312, 1, 3),      # 512 x 13: whole chunks of columns, off the grid
                                                     (65536, 65537, 0, 1), (65536, 65537, 0, 3),      # 512 x 16
                                                     (80008, 80013, 0, 1), (100277, 100277, 0, 1)])   # 1024 x 16: without a workspace
def test_probabilities_of_wide_rows_off_the_grid_are_rounded_once(D, monkeypatch, dtype, V, pitch, offset, teachers):
    """Gradients of 16-bit rows that lie off the 16-byte grid and that one workgroup of 512 threads or more holds (whole chunks
    of columns; without a workspace also wider rows of any length) are made from the logits, not from 16-bit probabilities: one
    rounding to the gradient's type (half a unit in the last place, and the 1e-5 that exponents of up to 64 leave of an fp32
    exponential), also for probabilities of 2^-50 of the row's largest."""
    R, K = 5, 16
    g = torch.Generator().manual_seed(V + pitch)
    x = torch.zeros(R, pitch + 8, dtype=dtype, device=DEV)[:, offset:offset + V] if pitch != V else torch.zeros(R, V, dtype=dtype, device=DEV)
    logits = (torch.randn(R, V, generator=g) * 2).to(dtype)
    logits[1] = (torch.rand(R, V, generator=g)[1] * -40).to(dtype)
    logits[1, 70] = 1.0
    x.copy_(logits.to(DEV))
    ti = torch.stack([torch.randperm(V, generator=g)[:K] for _ in range(R)]).int()
    tv = torch.log_softmax(torch.randn(R, K, generator=g), -1).half()
    scale = float(V) if dtype == torch.float16 else 1.0      # entries of the first row among fp16's normal numbers
    if teachers == 1:
        monkeypatch.setattr(D._lib.load(), "dl_div_topk_workspace_bytes", lambda *a: 0)
        _, grad = D.div_topk("fkl", x, tv.to(DEV), ti.to(DEV), grad_scale=scale)
    else:
        _, grad = D.fkl_multi_teacher(x, [tv.to(DEV)] * 3, [ti.to(DEV)] * 3, [0.5, 0.25, 0.25], None, grad_scale=scale)
    ref = torch.softmax(logits.double(), -1) * scale
    smallest, bits = (2.0 ** -14, 10) if dtype == torch.float16 else (2.0 ** -126, 7)
    ulp = torch.exp2(torch.floor(torch.log2(ref)) - bits)
    dense = torch.ones(R, V, dtype=torch.bool).scatter_(1, ti.long(), False) & (ref > 2 * smallest)
    assert dense[0].sum() > V // 2 and (dtype == torch.float16 or (dense[1] & (ref[1] < 2.0 ** -50)).any())
    err = (grad.cpu().double() - ref).abs()
    assert (err <= 0.5 * ulp + 1e-5 * ref)[dense].all(), (err / ulp)[dense].max()
    if teachers == 1:                                        # and the same bits written over the logits
        _, over = D.div_topk("fkl", x, tv.to(DEV), ti.to(DEV), grad_scale=scale, grad_out=x)
        assert over.data_ptr() == x.data_ptr() and torch.equal(grad, x)


@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 128256), (torch.bfloat16, 128251), (torch.float32, 65536), (torch.float32, 65533),
                                     (torch.bfloat16, 300000), (torch.float32, 150003)])      # streamed: threads that have met masked columns only
@pytest.mark.parametrize("T", [1.0, 2.0])
@pytest.mark.parametrize("level", [0.0, -300.0])
def test_a_column_part_masked_with_low_finite_values(D, dtype, V, T, level):
    """A stretch of the vocabulary wider than a column part masked with the lowest value of the type or other finite ones
    instead of -inf: the row's loss and gradient are those of the -inf mask, which is held against the oracle; also where the
    row's other logits lie so low that 2^-(their log-sum-exp) is out of fp32's range."""
    g = torch.Generator().manual_seed(V)
    values = [torch.finfo(dtype).min, -3.38e38, -1e30, -2e9, -1.3e9, -1e9, -7e8, -3e8, -1.1e8, -3.3e7, -1.7e7, -6e4]
    R, K = len(values), 64
    logits = (torch.randn(R, V, generator=g) * 3 + level).to(dtype)
    a, b = int(0.24 * V), int(0.76 * V)
    logits[:, a:b] = -float("inf")
    tv, ti = torch.topk(torch.log_softmax(logits.float() + torch.randn(R, V, generator=g), -1), K)
    tv, ti = tv.half(), ti.int()
    if level == 0.0:      # (300 apart, loss and log-sum-exp cancel by more than the oracle's tolerance allows)
        _check(D, "fkl", logits, tv, ti, T=T)
    rl0, g0 = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV), T=T)
    for r, v in enumerate(values):
        logits[r, a:b] = v
    for no_wait in (False, True):
        rl, grad = D.div_topk("fkl", logits.to(DEV), tv.to(DEV), ti.to(DEV), T=T, no_wait=no_wait)
        np.testing.assert_allclose(rl.cpu().numpy(), rl0.cpu().numpy(), rtol=1e-6)
        assert torch.isfinite(grad).all() and torch.equal(grad, g0)


@pytest.mark.parametrize("dtype,V,pitch,K", [(torch.bfloat16, 102400, 102400, 200),      # 25 whole parts of 8 KiB
                                             (torch.bfloat16, 102408, 102408, 256),      # a last part of one chunk
                                             (torch.float16, 102407, 102407, 257),       # off the 16-byte grid: columns beside the chunks
                                             (torch.bfloat16, 106497, 106504, 513),      # a loop over the entries
                                             (torch.float32, 51201, 51201, 40), (torch.float32, 51200, 51204, 1)])
@pytest.mark.parametrize("grad_mode", ["fresh", "in_place", "other_phase"])
def test_rkl_values_and_fill_match_the_one_launch_form(D, dtype, V, pitch, K, grad_mode):
    """Wide rows: the values of all rows in one launch, the rows themselves in a second one, through a workspace;
    dl_div_topk_static, which has none for it, keeps one launch.  The same arithmetic, bit for bit; repeated ids (their values
    are added up), ids outside the row, entries in the first and last columns, masked rows, rows without an entry."""
    assert D._lib.load().dl_rkl_topk_workspace_bytes(D.ops._DT[dtype], 9, V, K) == 9 * K * 8
    R = 9
    g = torch.Generator().manual_seed(V + K)
    x = torch.zeros(R, pitch, dtype=dtype, device=DEV)[:, :V]
    x.copy_((torch.randn(R, V, generator=g) * 3).to(dtype).to(DEV))
    tv = torch.log_softmax(torch.randn(R, K, generator=g) * 2, -1).half().to(DEV)
    ti = torch.randint(0, V, (R, K), generator=g, dtype=torch.int32).to(DEV)
    if K > 8:
        ti[:, 0], ti[:, 1], ti[:, 2], ti[:, 3] = 0, V - 1, V, -1
        ti[1, 4:8] = ti[1, 8]                            # one id five times
        ti[2, K // 2:] = ti[2, :K - K // 2].clone()      # every id twice, the ends of the row among them
        tv[3] = float("-inf")                            # no entry at all
    rm = torch.arange(R, dtype=torch.int32, device=DEV)
    rm[5] = -1
    rl, grad = torch.empty(R, device=DEV), torch.empty_like(x)
    D.div_topk_static("rkl", x, tv, ti, rl, grad, row_map=rm, T=1.4, grad_scale=0.3)
    out = None
    if grad_mode == "in_place":
        out = x
    elif grad_mode == "other_phase":
        out = torch.full((R * (V + 3) + 1,), float("nan"), dtype=dtype, device=DEV)[1:].view(R, V + 3)[:, :V]
    rl2, grad2 = D.div_topk("rkl", x, tv, ti, row_map=rm, T=1.4, grad_scale=0.3, grad_out=out)
    assert torch.equal(rl, rl2) and torch.equal(grad, grad2)


@pytest.mark.parametrize("dtype,V,std", [(torch.bfloat16, 4104, 4.0), (torch.float32, 4104, 15.0), (torch.float16, 102400, 4.0)])
@pytest.mark.parametrize("K", [1, 200, 256, 257, 512])
def test_rkl_entries_in_registers_match_the_general_form(D, dtype, V, std, K):
    """Up to 512 stored entries a row are held in registers, more pass through LDS.  The same rows with 528 stored entries
    of which `t_cnt` leaves K take the second way: the same roundings, bit for bit.  In particular the logits are scaled by
    1 / T (which is not exact here) inside a fused multiply-add in both: a product rounded by itself costs precision where
    logits are large."""
    R, KW = 24, 528
    g = torch.Generator().manual_seed(V + K)
    x = (torch.randn(R, V, generator=g) * std + 15).to(dtype).to(DEV)
    tv = torch.log_softmax(torch.randn(R, KW, generator=g) * 2, -1).half().to(DEV)
    ti = torch.stack([torch.randperm(V, generator=g)[:KW] for _ in range(R)]).int().to(DEV)
    ti[2, 0] = -1                                                    # an entry that does not count
    cnt = torch.full((R,), K, dtype=torch.int32, device=DEV)
    kw = dict(T=1.4, teacher_T=1.3, grad_scale=0.3)
    rl, grad = D.div_topk("rkl", x, tv[:, :K], ti[:, :K], **kw)
    rl2, grad2 = D.div_topk("rkl", x, tv, ti, t_cnt=cnt, **kw)
    assert torch.equal(rl, rl2) and torch.equal(grad, grad2)


@pytest.mark.parametrize("R,K", [(1025, 2048), (2051, 2048), (8200, 257)])      # 2, 3 and 2 turns of at most 16 MiB of pairs
@pytest.mark.parametrize("in_place", [False, True])
def test_rkl_on_many_rows_takes_them_in_turns(D, R, K, in_place):
    """More rows than the workspace of the two launches holds: values and stores of a share of the rows, then of the next one.
    Bit for bit what one launch writes, masked rows and rows mapped onto others' teachers among them."""
    V = 100004                                                       # rows off the 16-byte grid in turn
    per_turn, rest = divmod(D._lib.load().dl_rkl_topk_workspace_bytes(D.ops._DT[torch.bfloat16], R, V, K), 8 * K)
    assert rest == 0 and 0 < per_turn < R
    g = torch.Generator(device=DEV).manual_seed(R)
    x = torch.randn(R, V, generator=g, device=DEV, dtype=torch.bfloat16) * 3
    tv = torch.log_softmax(torch.randn(R, K, generator=g, device=DEV) * 2, -1).half()
    ti = torch.randint(0, V, (R, K), generator=g, device=DEV, dtype=torch.int32)
    rm = torch.arange(R, dtype=torch.int32, device=DEV).flip(0)
    rm[::17] = -1
    rm[per_turn] = -1
    rl, grad = torch.empty(R, device=DEV), torch.empty_like(x)
    D.div_topk_static("rkl", x, tv, ti, rl, grad, row_map=rm, T=1.4, grad_scale=0.3)
    rl2, grad2 = D.div_topk("rkl", x, tv, ti, row_map=rm, T=1.4, grad_scale=0.3, grad_out=x if in_place else None)
    assert torch.equal(rl, rl2) and torch.equal(grad, grad2)
