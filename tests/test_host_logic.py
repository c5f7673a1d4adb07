"""CPU-side checks: the Losses accumulator mirrors classes/losses.py, the C-ABI library loads and
exports every symbol the header declares, and the Python layer refuses to run without a GPU."""
import os
import re

import pytest
import torch

import llm_distillery_amd as D

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class _Log:
    def __init__(self):
        self.rows = []

    def log(self, d, step=None):
        self.rows.append((d, step))


def _dict(v, leaf):
    out = {k: torch.tensor(float(v + i)) for i, k in enumerate(D.LOSS_KEYS)}
    out["train_loss"] = leaf * v
    return out


def test_losses_accumulates_sums_and_backward_divides():
    leaf = torch.tensor(2.0, requires_grad=True)
    L = D.Losses(_Log())
    with pytest.raises(ValueError):
        L.add_losses({})
    L.add_losses(_dict(1.0, leaf))
    L.add_losses(_dict(3.0, leaf))
    assert L.num_steps_accumulated == 2
    assert L.loss_dict["kl_div"].item() == (1 + 3) + (3 + 3) and not L.loss_dict["kl_div"].requires_grad
    L.backward(divisor=4)
    assert "train_loss" not in L.loss_dict
    assert leaf.grad.item() == pytest.approx((1.0 + 3.0) / 4)      # sum over conversations / divisor
    L.log(step=7)
    keys = [list(d)[0] for d, _ in L.logger.rows]
    assert keys == [f"Loss/{k}" for k in D.LOSS_KEYS if k != "train_loss"]
    d0, step = L.logger.rows[0]
    assert step == 7 and d0["Loss/custom loss"].item() == pytest.approx(((1 + 1) + (3 + 1)) / 2)
    L.empty()
    assert L.loss_dict == {} and L.num_steps_accumulated == 0


def test_losses_add_batch_equals_adding_one_by_one():
    leaf_a, leaf_b = torch.tensor(2.0, requires_grad=True), torch.tensor(2.0, requires_grad=True)
    one, many = D.Losses(None), D.Losses(None)
    one.add_losses(_dict(0.5, leaf_a))                         # something accumulated before the batch
    many.add_losses(_dict(0.5, leaf_b))
    for v in (1.0, 3.0, 4.0):
        one.add_losses(_dict(v, leaf_a))
    many.add_batch([_dict(v, leaf_b) for v in (1.0, 3.0, 4.0)])
    assert one.num_steps_accumulated == many.num_steps_accumulated == 4
    assert set(one.loss_dict) == set(many.loss_dict)
    for k in one.loss_dict:
        assert one.loss_dict[k].item() == pytest.approx(many.loss_dict[k].item())
        assert k == "train_loss" or not many.loss_dict[k].requires_grad
    one.backward(divisor=2)
    many.backward(divisor=2)
    assert leaf_a.grad.item() == pytest.approx(leaf_b.grad.item()) == pytest.approx(8.5 / 2)
    with pytest.raises(ValueError):
        many.add_batch([])
    single = D.Losses(None)
    single.add_batch([_dict(1.0, leaf_b)])
    assert single.num_steps_accumulated == 1


def test_losses_validation_prefix_and_scaling_operators():
    L = D.Losses(_Log(), validation=True)
    L.add_losses({"train_loss": torch.tensor(1.0), "kl_div": torch.tensor(4.0)})
    L.log(step=1, average=False)
    assert list(L.logger.rows[0][0]) == ["Val Loss/kl_div"]
    half = L / 2
    assert half.loss_dict["kl_div"].item() == 2.0 and half.validation
    L *= 3
    assert L.loss_dict["kl_div"].item() == 12.0
    assert "Validation Losses" in str(L)


def test_losses_packed_dicts_accumulate_like_plain_ones():
    """`calculate_divergence` hands out dicts whose values are views of one [9] tensor; `Losses` sums
    those with one addition per conversation.  Totals, step count, backward and logging must be what
    the key-by-key form gives, also when packed and plain dicts are mixed."""
    from llm_distillery_amd.losses import LossDict
    keys = D.LOSS_KEYS
    leafs = [torch.tensor(float(i + 1), requires_grad=True) for i in range(3)]

    def make(i, packed):
        row = torch.arange(9, dtype=torch.float32) * (i + 1)
        train = leafs[i] * 2
        d = LossDict(zip(keys, row.unbind(0))) if packed else dict(zip(keys, row.clone().unbind(0)))
        d["train_loss"] = train
        if packed:
            d.packed, d.keys_packed = row, keys
        return d

    for pattern in ((True, True, True), (False, False, False), (True, False, True), (False, True, True)):
        for leaf in leafs:
            leaf.grad = None
        L = D.Losses(_Log())
        for i, packed in enumerate(pattern):
            L.add_losses(make(i, packed))
        assert L.num_steps_accumulated == 3
        got = L.loss_dict
        assert list(got)[0] == "train_loss" and set(got) == set(keys)
        assert got["train_loss"].item() == 2 * (1 + 2 + 3)
        for j, k in enumerate(keys[1:], start=1):
            assert got[k].item() == j * (1 + 2 + 3) and not got[k].requires_grad
        L.backward(divisor=2)
        assert all(leaf.grad.item() == 1.0 for leaf in leafs) and "train_loss" not in L.loss_dict
        L.log(step=3)
        assert L.logger.rows[0][0]["Loss/custom loss"].item() == pytest.approx(1 * 6 / 3)
        L.empty()
        assert L.loss_dict == {} and L.num_steps_accumulated == 0
    # the batch form: stack + sum
    L = D.Losses(None)
    L.add_batch([make(i, True) for i in range(3)])
    assert L.num_steps_accumulated == 3 and L.loss_dict["kl_div"].item() == 3 * 6 and L.loss_dict["train_loss"].item() == 12
    half = L / 2
    assert half.loss_dict["kl_div"].item() == 9.0


def test_losses_loss_dict_is_a_plain_writable_dict_also_after_packed_additions():
    """classes/losses.py:22 keeps a plain dict attribute that callers may write into, delete from or scale in
    place; the packed accumulation must not turn such writes into no-ops, and a second backward finds the key
    gone (KeyError) as in the reference (classes/losses.py:77-79)."""
    from llm_distillery_amd.losses import LossDict
    keys = D.LOSS_KEYS
    leaf = torch.tensor(1.0, requires_grad=True)

    def make(i):
        row = torch.arange(9, dtype=torch.float32) * (i + 1)
        d = LossDict(zip(keys, row.unbind(0)))
        d["train_loss"] = leaf * (i + 1)
        d.packed, d.keys_packed = row, keys
        return d

    L = D.Losses(_Log())
    L.add_losses(make(0))
    L.add_losses(make(1))
    L.loss_dict["kl_div"] = torch.tensor(100.0)
    L.loss_dict["CE loss"] /= 2
    del L.loss_dict["CE diff"]
    assert L.loss_dict["kl_div"].item() == 100.0 and L.loss_dict["CE loss"].item() == 2 * 3 / 2 and "CE diff" not in L.loss_dict
    L.add_losses(make(2))                                     # a packed dict after the write: added key by key
    assert L.loss_dict["kl_div"].item() == 100.0 + 3 * 3 and L.loss_dict["CE diff"].item() == 8 * 3
    assert L.loss_dict["train_loss"].item() == 6.0 and L.num_steps_accumulated == 3
    L.backward(divisor=3)
    assert leaf.grad.item() == pytest.approx(2.0)
    with pytest.raises(KeyError):
        L.backward()
    P = D.Losses(None)                                        # never touched from outside: still packed at the second backward
    P.add_losses(make(0))
    P.backward()
    with pytest.raises(KeyError):
        P.backward()


def test_registered_operators_trace_with_fake_tensors():
    """The V-wide launches are registered torch.library operators with fake (shape-only) implementations, so that
    FakeTensor tracing / torch.compile see through them without touching a GPU."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from llm_distillery_amd import ops
    with FakeTensorMode():
        logits = torch.empty(10, 64, dtype=torch.bfloat16)
        t_val = torch.empty(7, 5, dtype=torch.float16)
        t_idx = torch.empty(7, 5, dtype=torch.int32)
        labels = torch.empty(5, dtype=torch.int64)
        avoid = torch.empty(1, dtype=torch.int64)
        offsets = torch.empty(3, 3, dtype=torch.int32)                  # two conversations
        row_map = torch.empty(10, dtype=torch.int32)
        train, nine, lse, zk, rec, coef = ops.composite_forward_op(logits, t_val, t_idx, labels, avoid, offsets, row_map, 1.0, 1.0, 2.0, 48)
        assert train.shape == (2,) and nine.shape == (2, 9) and lse.shape == (7,) and zk.shape == (7, 5)
        assert rec.shape == (7, 8) and coef.shape == (7, 4) and train.dtype == torch.float32
        grad = ops.composite_backward_op(logits, t_val, t_idx, lse, zk, rec, coef, train, offsets, row_map, 1.0, 1.0, 48)
        assert grad.shape == logits.shape and grad.dtype == logits.dtype
        lse2, zk2 = ops.rowstats_topk(logits, t_idx, row_map, 1.0, 48)
        assert lse2.shape == (7,) and zk2.shape == (7, 5)


def test_library_exports_every_symbol_the_header_declares():
    header = open(os.path.join(ROOT, "include", "distill_hip.h")).read()
    declared = set(re.findall(r"\b(dl_[a-z0-9_]+)\s*\(", header))
    lib = D._lib.load()
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in the header but not exported"
    assert declared == set(D._lib.exported_symbols())
    assert lib.dl_abi_version() >= 1
    assert lib.dl_status_string(0) == b"ok" and b"NULL" in lib.dl_status_string(-1)


def test_argument_errors_are_reported_before_any_gpu_work():
    """Host-side validation of the entry points that take host arrays: every call below returns its
    status before the first HIP call, so the (never dereferenced) device pointers can be anything."""
    import ctypes
    lib = D._lib.load()
    fake = ctypes.c_void_p(4096)
    i32 = lambda *v: (ctypes.c_int32 * len(v))(*v)
    # composite: offsets that travel with the launch are checked on the host
    def fwd(row, lab, av, C, N):
        return lib.dl_composite_forward(fake, fake, fake, 2, 1.0, fake, 0, 8, fake, fake, 1, row, lab, av, 1, C, N, 2.0, fake, fake,
                                        fake, None)
    assert fwd(i32(0, 5, 3), i32(0, 4, 6), i32(0, 0, 0), 2, 3) == -3            # rows not non-decreasing
    assert fwd(i32(0, 5, 9), i32(0, 4, 7), i32(0, 0, 0), 2, 10) == -3           # rows do not end at n_rows
    assert fwd(i32(1, 5), i32(0, 4), i32(0, 0), 1, 5) == -3                     # rows do not start at 0
    many = i32(*range(66))
    assert fwd(many, many, many, 65, 65) == -4                                  # more conversations than a launch carries
    assert lib.dl_composite_forward(fake, fake, fake, 2, 1.0, fake, 0, 8, fake, fake, 7, i32(0, 5), i32(0, 4), i32(0, 0), 1, 1, 5,
                                    2.0, fake, fake, fake, None) == -2          # ignore entries of an unknown integer type
    assert lib.dl_composite_backward(fake, fake, fake, 2, 1.0, fake, 0, 8, i32(0, 4), 1, 1, 5, fake, fake, fake, fake, fake,
                                     None) == -3
    # multi-teacher loss: limits, weights, workspace
    ptrs = (ctypes.c_void_p * 3)(4096, 4096, 4096)
    w = lambda *v: (ctypes.c_float * len(v))(*v)
    def multi(V=128256, n=3, K=200, ws=fake, ws_bytes=1 << 40, weights=w(0.5, 0.3, 0.2), stride=None):
        return lib.dl_fkl_multi_teacher(fake, 1, stride or V, 64, V, None, n, ptrs, ptrs, 2, 0, K, 64, weights, None, 0, 1.0, 1.0,
                                        fake, fake, V, ws, ws_bytes, 0, None)
    assert multi(n=3, K=700) == -4                                              # more than DL_MAX_TOPK entries per row
    assert multi(V=300000) == -4                                                # rows too wide for the register kernels
    assert multi(V=128257, stride=128264) == -6                                 # odd vocabulary
    assert multi(ws=None) == -7 and multi(ws_bytes=1000) == -7                  # no / too small a workspace
    assert multi(weights=w(0.5, -0.1, 0.2)) == -3 and multi(weights=w(0.5, float("nan"), 0.2)) == -3
    need = lib.dl_fkl_multi_teacher_workspace_bytes(1, 64, 128256, 3, 200, 64, 0)
    assert need > 64 * 4 * 256 * 8 and multi(ws_bytes=need - 1) == -7
    assert lib.dl_fkl_multi_teacher_workspace_bytes(1, 64, 300000, 3, 200, 64, 0) == 0


def test_no_cpu_fallback():
    x = torch.randn(4, 64)
    tv, ti = torch.randn(4, 8), torch.randint(0, 64, (4, 8), dtype=torch.int32)
    with pytest.raises(RuntimeError, match="no CPU path"):
        D.div_topk("fkl", x, tv, ti)
    with pytest.raises(RuntimeError, match="no CPU path"):
        D.calculate_divergence(x, tv, ti.long(), torch.zeros(3, dtype=torch.long), 2.0, torch.zeros(0, dtype=torch.long))


def test_product_code_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "llm-distillery_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".cpp", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower() or f == "synthetic.py", f"{f} mentions the oracle"


def test_losses_of_a_whole_batch_are_summed_without_their_views():
    """Dicts that one call made together: the same totals, logged values and gradients as one by one, also where one of them was
    scaled in place; a hook on an entry still runs, a replaced entry still counts, a part of the batch is summed as before."""
    from llm_distillery_amd.losses import LossDict
    keys = tuple(D.finetuning_utils.LOSS_KEYS) if hasattr(D, "finetuning_utils") else ("train_loss", "custom loss", "CE loss")

    def make():
        leaf = torch.arange(1.0, 5.0, requires_grad=True)
        train = leaf * leaf
        nine = torch.arange(4.0 * len(keys)).view(4, len(keys))
        out = []
        for c in range(4):
            row = nine[c]
            d = LossDict(zip(keys, row.unbind(0)))
            d["train_loss"] = train[c]
            d.packed, d.keys_packed, d.batch = row, keys, (train, nine, c, d["train_loss"], row)
            out.append(d)
        return leaf, out

    def plain(mutate=lambda o: None, pick=slice(None)):
        leaf, out = make()
        mutate(out)
        L = D.Losses(None)
        for d in out[pick]:
            L.add_losses(d)
        view = {k: v.clone() for k, v in L._view().items()}
        L.backward(2)
        return leaf.grad, view

    def batch(mutate=lambda o: None, pick=slice(None)):
        leaf, out = make()
        mutate(out)
        L = D.Losses(None)
        L.add_batch(out[pick])
        view = {k: v.clone() for k, v in L._view().items()}
        L.backward(2)
        return leaf.grad, view

    def scale(out):
        out[1]["train_loss"].mul_(3.0)

    def replace(out):
        out[2]["train_loss"] = out[2]["train_loss"] * 5.0

    seen = []
    for mutate, pick in ((lambda o: None, slice(None)), (scale, slice(None)), (replace, slice(None)), (lambda o: None, slice(1, 4)),
                         (lambda o: o[0]["train_loss"].register_hook(lambda g: seen.append(1) or g * 10.0), slice(None))):
        (ga, va), (gb, vb) = plain(mutate, pick), batch(mutate, pick)
        assert torch.equal(ga, gb) and set(va) == set(vb) and all(torch.allclose(va[k], vb[k]) for k in va)
    assert len(seen) == 2


def test_marks_on_the_train_losses_of_a_batch_work_before_and_after_adding_it(monkeypatch):
    """Every conversation's train loss of one call stays in the graph of the batch's sum: a hook or retain_grad() on it works
    whether it came before or after `add_batch`, and the sum can be differentiated with respect to it; scaled in place an
    entry counts as scaled.  The logged values come from the table of which the dicts hold the rows.  (The launch is stood in for.)"""
    from llm_distillery_amd import finetuning_utils as FU
    nine = torch.arange(4.0 * 9).view(4, 9).clone()
    monkeypatch.setattr(FU.ops, "composite_loss", lambda x, *_: (x * x, nine))
    one, none = torch.zeros(1, 2), torch.zeros(0, dtype=torch.long)

    def make(grad=True):
        leaf = torch.arange(1.0, 5.0, requires_grad=grad)
        return leaf, FU._fused_dicts(leaf, None, 1.0, 0, [1] * 4, [one] * 4, [one.int()] * 4, [none] * 4, [none] * 4, 1.0, 2.0)

    for after in (False, True):
        leaf, out = make()
        assert all(d["train_loss"] is d["custom loss"] for d in out)
        L, seen = D.Losses(None), []
        if after:
            L.add_batch(out)
        out[0]["train_loss"].register_hook(lambda g: seen.append(g.item()) or g * 10.0)
        out[1]["train_loss"].retain_grad()
        if not after:
            L.add_batch(out)
        assert torch.equal(L._packed, nine.sum(0))
        L.backward(2)
        assert leaf.grad.tolist() == [10.0, 2.0, 3.0, 4.0] and out[1]["train_loss"].grad.item() == 0.5 and seen == [0.5]
    leaf, out = make()
    out[2]["train_loss"].mul_(3.0)
    L = D.Losses(None)
    L.add_batch(out)
    L.backward()
    assert leaf.grad.tolist() == [2.0, 4.0, 18.0, 8.0]
    _, out = make()
    L = D.Losses(None)
    L.add_batch(out)
    assert torch.autograd.grad(L._train, out[3]["train_loss"])[0].item() == 1.0
    _, plain = make(False)                                                   # a validation call: views of one tensor
    assert [d["train_loss"].item() for d in plain] == [1.0, 4.0, 9.0, 16.0]
    plain[1]["train_loss"].mul_(2.0)
    L = D.Losses(None)
    L.add_batch(plain)
    assert L._train.item() == 34.0 and torch.equal(L._packed, nine.sum(0))
    _, plain = make(False)
    plain[0]["train_loss"].requires_grad_()
    L = D.Losses(None)
    L.add_batch(plain)
    L.backward()
    assert plain[0]["train_loss"].grad.item() == 1.0


def test_packed_rows_of_one_row_slices():
    """One-row slices of a wider tensor count as contiguous whatever their row stride is: the concatenation is torch.cat's, also
    where the slices lie back to back, for 2-D rows (teachers) and 1-D entries (labels, ignore lists), with empty ones between."""
    from llm_distillery_amd.finetuning_utils import _packed_rows
    full = torch.arange(5 * 2 * 4).view(5, 2, 4)
    tok = torch.arange(10).view(5, 2)
    wide = torch.arange(12).view(1, 3, 4)
    row = torch.arange(24).view(6, 4)
    for parts in ([full[0:1, 0], full[0:1, 1]], [full[1:2, 0], full[1:2, 1], full[2:3, 0]], [wide[:, c] for c in range(3)],
                  [tok[2:3, 0], tok[2:3, 1]], [tok[0:1, 1], tok[1:2, 0], tok[3:3, 0]], [tok[0:0, 0], tok[1:2, 0], tok[1:2, 1]],
                  [row[0:2], row[2:3], row[3:6]], [row[0:2], row[3:4]], [full[0:2, 0], full[0:2, 1]]):
        assert torch.equal(_packed_rows(parts), torch.cat(parts))
    assert _packed_rows([row[0:2], row[2:6]]).data_ptr() == row.data_ptr()      # and no copy where none is needed
    with pytest.raises(RuntimeError):
        _packed_rows([row[0:1], row.view(-1)[4:10].view(2, 3)])                 # other widths are no rows of one tensor


def test_rows_that_one_workgroup_holds_need_no_workspace():
    """dl_div_topk_workspace_bytes asks for records where a row is cut into column parts, and only there: not below 8193 chunks of
    16 bytes, whole or not, however many rows (dl_div_topk_static refuses by this size)."""
    lib = D._lib.load()
    size = lambda dtype, rows, V, kind=D.ops.KINDS["fkl"]: lib.dl_div_topk_workspace_bytes(kind, D.ops._DT[dtype], rows, V)
    for rows in (1, 110000, 1 << 30):
        assert all(size(torch.bfloat16, rows, V) == 0 for V in (5, 32768, 32769, 50257, 50304, 65535, 65536))
        assert all(size(torch.float32, rows, V) == 0 for V in (5, 16385, 32767, 32768)) and size(torch.bfloat16, rows, 128256, 1) == 0
        assert all(size(dt, rows, V) > 16 * rows for dt, V in ((torch.bfloat16, 65537), (torch.bfloat16, 262144), (torch.float32, 32769)))
    assert size(torch.bfloat16, 1 << 20, 262145) == 0      # too wide to be cut


@pytest.mark.parametrize("dtype,V,parts", [(0, 65536, 32), (1, 128256, 32), (2, 102408, 26), (1, 6 << 20, 1536)])
@pytest.mark.parametrize("K", [1, 16, 500, 2048])
def test_reverse_kl_in_two_launches_takes_many_rows_in_turns(dtype, V, parts, K):
    """The pairs of ids and values between the two launches take no more than 16 MiB however many rows there are, and neither
    launch reaches 2^32 threads (a workgroup of 256 threads for every 8 KiB of a gradient row), the most that one takes."""
    lib = D._lib.load()
    for rows in (1, 100, 4096, 32768, 524287, 524288, 2 ** 24, 2 ** 31 - 1):
        per_turn, rest = divmod(lib.dl_rkl_topk_workspace_bytes(dtype, rows, V, K), 8 * K)
        assert rest == 0 and 0 < per_turn <= rows and per_turn * K * 8 <= 16 << 20
        assert (per_turn * parts + 7) // 8 * 8 * 256 < 2 ** 32
        assert per_turn == rows or 2 * per_turn * max(K * 8 / 2 ** 24, parts * 256 / 2 ** 32) > 0.99      # no more turns than that asks for


def test_partial_marginals_take_a_workspace_for_fp32_probabilities_only():
    """Probabilities of 16 bits go without a plan, in one launch: no room for partial marginals is taken for them."""
    from llm_distillery_amd.vocab_utils import _parts_workspace
    ws, n = _parts_workspace(16, 152064, torch.float32, 2048, 8192, "cpu")
    assert n == ws.numel() == 16 * 4 * 2048 * 4
    for dtype in (torch.bfloat16, torch.float16):
        assert _parts_workspace(16, 152064, dtype, 2048, 8192, "cpu") == (None, 0)
    assert _parts_workspace(129, 152064, torch.float32, 2048, 8192, "cpu") == (None, 0)


@pytest.mark.parametrize("rows,Vt,columns,tile,parts", [
    (64, 152064, 3752, 8192, 4), (128, 152064, 3752, 8192, 2), (1, 270000, 16384, 8192, 8), (27, 152064, 16384, 8192, 4),      # narrow marginals, many tiles
    (128, 70000, 704, 7168, 2), (128, 70000, 9000, 8192, 1), (64, 70000, 15000, 8192, 1),      # few tiles: up to a width
    (27, 70000, 32000, 8192, 1), (128, 100000, 36000, 4096, 1), (128, 152064, 32000, 8192, 1), (128, 262144, 36000, 4096, 2),
    (129, 262144, 704, 8192, 1), (0, 262144, 704, 8192, 1), (64, 262144, 704, 0, 1)])
def test_partial_marginals_are_taken_where_the_tiles_spared_outweigh_them(rows, Vt, columns, tile, parts):
    """Several workgroups to a row write and read partial marginals as wide as the columns: more than a call gains where a wide
    marginal meets few tiles."""
    n = D._lib.load().dl_rkl_marginalised_workspace_bytes(rows, Vt, columns, tile)
    assert n == (rows * parts * columns * 4 if parts > 1 else 0)
