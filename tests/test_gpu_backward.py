"""Backward of the block-sparse attention (bf16): dq, dk, dv of the HIP kernel, reached through the autograd
function and the C ABI, against the oracle's closed-form float64 gradients on the same bf16 inputs.

Tolerance: the kernel rounds P, dS, O and the results to bf16 and sums in fp32, so every gradient tensor must
be within 2e-2 of its own largest magnitude (max-abs, the same bar as the forward's outputs, scaled because
gradients are not O(1)); the saved log-sum-exp within 2e-3 absolute.  Rows of padded slots must be zero."""
import math

import numpy as np
import pytest
import torch

import blockrank_amd as br
from blockrank_amd import synthetic
from oracle import blockrank_oracle as orc
from tests._util import real_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(lay, Nq, Nkv, D, seed=0, packed=False):
    q, k, v = synthetic.random_qkv(lay, Nq, Nkv, D, torch.bfloat16, DEV, seed=seed)
    scale = D ** -0.5
    gen = torch.Generator().manual_seed(seed + 1000)
    dout = torch.randn((lay.B, lay.S, Nq, D), generator=gen).to(torch.bfloat16).to(DEV)
    want = orc.dense_attention_backward(q.float().cpu().numpy(), k.float().cpu().numpy(), v.float().cpu().numpy(),
                                        dout.float().cpu().numpy(), lay.valid.numpy(), scale)
    rows = real_rows(lay)                                                   # (B, S)
    if packed:
        from tests.test_gpu_packed import _pack
        lengths = torch.as_tensor(lay.lengths, dtype=torch.int32, device=DEV)
        mask = br.BlockMask.from_lengths(lengths, H=lay.H, packed=True, dtype=torch.bfloat16)
        qq, kk, vv = (_pack(t, lay.valid).requires_grad_(True) for t in (q, k, v))
        out = br.blockrank_attention(qq, kk, vv, mask, scale)
        out.backward(dout[rows.to(DEV)][None])
        grads = []
        for t, heads in ((qq, Nq), (kk, Nkv), (vv, Nkv)):
            full = torch.zeros((lay.B, heads, lay.S, D), dtype=torch.float32)
            full.transpose(1, 2)[rows] = t.grad.float().cpu()[0].transpose(0, 1)
            grads.append(full)
    else:
        mask = br.BlockMask(lay.valid.to(DEV), torch.bfloat16)
        qq, kk, vv = (t.clone().requires_grad_(True) for t in (q, k, v))
        out = br.blockrank_attention(qq, kk, vv, mask, scale)
        out.backward(dout)
        grads = [t.grad.float().cpu() for t in (qq, kk, vv)]
    torch.cuda.synchronize()
    for name, got, ref in zip(("dq", "dk", "dv"), grads, want[:3]):
        got = got.numpy().astype(np.float64)
        assert np.isfinite(got).all(), f"{name} has non-finite values"
        real = rows.numpy()[:, None, :, None]
        assert (got * ~real == 0).all(), f"{name}: rows of padded slots must be zero"
        err = np.abs(got - ref).max()
        bound = 2e-2 * max(np.abs(ref).max(), 1e-6)
        assert err <= bound, f"{name}: max abs error {err:.3e} > {bound:.3e} (largest gradient {np.abs(ref).max():.3e})"
    return want[3]


def test_saved_log_sum_exp_matches_oracle():
    lay = synthetic.make_layout([[40, 100, 160, 33, 192, 20], [64, 7, 150, 90, 0, 31]])
    Nq, Nkv, D = 8, 2, 128
    q, k, v = synthetic.random_qkv(lay, Nq, Nkv, D, torch.bfloat16, DEV, seed=3)
    qq = q.clone().requires_grad_(True)
    out = br.blockrank_attention(qq, k, v, br.BlockMask(lay.valid.to(DEV), torch.bfloat16), D ** -0.5)
    lse = out.grad_fn.saved_tensors[4].cpu().double().numpy() * math.log(2.0)
    *_, want = orc.dense_attention_backward(q.float().cpu().numpy(), k.float().cpu().numpy(), v.float().cpu().numpy(),
                                            np.zeros((lay.B, lay.S, Nq, D)), lay.valid.numpy(), D ** -0.5)
    rows = np.broadcast_to(real_rows(lay).numpy()[:, None, :], want.shape)
    assert np.abs(lse[rows] - want[rows]).max() <= 2e-3


def test_log_sum_exp_of_split_rows_is_exact_too():
    # one request with many documents: the query block's key walk is cut into several items and its rows' log-sum-exp
    # comes from the merge of their partials.  Peaked rows (large logits: one key carries the mass, so the sum of the
    # bf16-rounded probabilities that normalises the output is off from the exact one by up to 2^-9) must come out as
    # exact as the rows a single item finishes: 1e-4 in natural-log units.
    lay = synthetic.random_layout(1, 48, 40, 30, 96, 24, seed=8)
    Nq, Nkv, D = 8, 2, 128
    q, k, v = synthetic.random_qkv(lay, Nq, Nkv, D, torch.bfloat16, DEV, seed=5)
    q = (q * 6).contiguous()
    qq = q.clone().requires_grad_(True)
    out = br.blockrank_attention(qq, k, v, br.BlockMask(lay.valid.to(DEV), torch.bfloat16), D ** -0.5)
    lse = out.grad_fn.saved_tensors[4].cpu().double().numpy() * math.log(2.0)
    *_, want = orc.dense_attention_backward(q.float().cpu().numpy(), k.float().cpu().numpy(), v.float().cpu().numpy(),
                                            np.zeros((lay.B, lay.S, Nq, D)), lay.valid.numpy(), D ** -0.5)
    rows = np.broadcast_to(real_rows(lay).numpy()[:, None, :], want.shape)
    err = np.abs(lse - want)
    assert err[rows].max() <= 1e-4
    last = np.zeros_like(rows)
    last[:, :, -lay.H:] = rows[:, :, -lay.H:]                    # the query block's rows: the split ones
    assert last.any() and err[last].max() <= 1e-4


def test_ragged_blocks_four_heads_per_group():
    _check(synthetic.make_layout([[40, 100, 160, 33, 192, 20], [64, 7, 150, 90, 0, 31]]), 8, 2, 128)


@pytest.mark.parametrize("G", [1, 2, 3, 7, 8])
def test_head_group_sizes(G):
    _check(synthetic.make_layout([[20, 70, 45, 130, 37]]), 2 * G, 2, 128, seed=G)


def test_head_dim_64():
    _check(synthetic.make_layout([[5, 17, 0, 64, 33, 9], [40, 1, 65, 31, 2, 70]]), 8, 2, 64, seed=11)


def test_single_block_and_no_documents():
    _check(synthetic.make_layout([[100]]), 4, 2, 128, seed=12)
    _check(synthetic.make_layout([[100, 50]]), 4, 2, 128, seed=13)
    _check(synthetic.make_layout([[0, 30, 0, 40, 5]]), 4, 1, 128, seed=14)


def test_long_document_list_splits_the_query_walk():
    # 30 documents of up to 96 tokens: the query block's key walk is cut into several items whose dq partial
    # sums meet in the accumulation buffer
    lay = synthetic.random_layout(1, 48, 30, 30, 96, 24, seed=4)
    _check(lay, 8, 2, 128, seed=15)


def test_packed_layout():
    _check(synthetic.make_layout([[40, 100, 160, 33, 192, 20], [64, 7, 150, 90, 0, 31]]), 8, 2, 128, seed=16, packed=True)


def test_random_layouts():
    """Seeded random block layouts (empty, one-token, tile-edge and long blocks; every head grouping; both head
    dims), the same generator as the forward's randomised test."""
    from tests.test_gpu_random_layouts import _cases
    for it, lens, G, Nkv, D in _cases(seed=23, n=16):
        lay = synthetic.make_layout(lens)
        if lay.S > 2600:                                   # keep the dense float64 oracle within seconds
            continue
        try:
            _check(lay, G * Nkv, Nkv, D, seed=100 + it)
        except AssertionError as e:
            raise AssertionError(f"case {it}: lengths {lens}, {G} heads per kv head, {Nkv} kv heads, D={D}: {e}") from e


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("prefix,docs,query", [
    (1, [32, 33, 31, 1], 1),                     # one key, row or group more or less than a whole one
    (32, [64, 65, 63, 0, 96], 33),               # an empty block; four groups with the prefix's, and a fifth
    (33, [128, 129, 97], 31),
    (130, [5, 40], 64),                          # five prefix groups: items that hold nothing but prefix keys
])
def test_key_groups_and_row_blocks_at_their_edges(D, prefix, docs, query):
    _check(synthetic.make_layout([[prefix, *docs, query], [prefix, *reversed(docs), query]]), 4, 2, D, seed=D + prefix)


def test_more_sets_than_a_window_of_the_dkv_queue():
    # 8 kv heads x 2 sequences x 50 blocks over eight queues: 100 sets each, two windows of 16 and a last one
    lens = [[9] + [(7 * i + 5 * b) % 33 + 1 for i in range(48)] + [12] for b in range(2)]
    _check(synthetic.make_layout(lens), 8, 8, 64, seed=5)


def _step(lay, seed, Nq=8, Nkv=2, D=128):
    q, k, v = (t.requires_grad_(True) for t in synthetic.random_qkv(lay, Nq, Nkv, D, torch.bfloat16, DEV, seed=seed))
    mask = br.BlockMask(lay.valid.to(DEV), torch.bfloat16)
    out = br.blockrank_attention(q, k, v, mask, D ** -0.5)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(seed)).to(DEV, torch.bfloat16)
    return out, (q, k, v), dout, mask


def _same(got, want):
    # (sums that several workgroups add to come in any order: a rounding of the largest magnitude apart)
    for g, w in zip(got, want):
        assert (g.float() - w.float()).abs().max() <= 2 ** -7 * w.float().abs().max()


def test_backward_passes_on_one_plan_may_overlap():
    lay = synthetic.random_layout(2, 48, 30, 30, 200, 24, seed=4)
    out, qkv, dout, _ = _step(lay, 3)
    grads = lambda: torch.autograd.grad(out, qkv, dout, retain_graph=True)
    want = grads()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(DEV) for _ in range(2)]
    results = []
    for _ in range(8):
        for st in streams:
            with torch.cuda.stream(st):
                results.append(grads())
    torch.cuda.synchronize()
    for got in results:
        _same(got, want)


def test_backward_with_a_workspace_of_just_the_stated_size():
    """Then the ticket counters are the plan's."""
    from blockrank_amd import _lib
    from blockrank_amd.attention import _stream_ptr
    lay = synthetic.random_layout(2, 48, 12, 30, 200, 24, seed=4)
    out, qkv, dout, mask = _step(lay, 5)
    want = torch.autograd.grad(out, qkv, dout, retain_graph=True)
    q, k, v, o, lse = out.grad_fn.saved_tensors
    lib, (B, Nq, S, D), Nkv = _lib.load(), q.shape, k.shape[1]
    n = lib.br_prefill_bwd_workspace_bytes(B, Nq, Nkv, lay.H, D, B * S)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    got = [torch.full((B, S, heads, D), float("nan"), dtype=torch.bfloat16, device=DEV) for heads in (Nq, Nkv, Nkv)]
    dense = lambda heads: _lib._I64x3(S * heads * D, D, heads * D)
    for _ in range(2):
        _lib.check(lib.br_prefill_bwd(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dout.data_ptr(), lse.data_ptr(), mask.plan(Nq, Nkv).data_ptr(),
            B, Nq, Nkv, lay.M, lay.H, D, _lib.strides3(q), _lib.strides3(k), _lib.strides3(v), dense(Nq), dense(Nq), _lib._I64x3(Nq * S, S, 1),
            *(t.data_ptr() for t in got), dense(Nq), dense(Nkv), dense(Nkv), D ** -0.5, B * S, ws.data_ptr(), n, _stream_ptr(q.device)))
        _same([t.transpose(1, 2) for t in got], want)



def _c_backward(out, mask, dout, lay, workspace, max_looks=1 << 20):
    """dq, dk, dv of br_prefill_bwd_ex for what autograd saved of an attention call on the padded layout."""
    from blockrank_amd import _lib
    from blockrank_amd.attention import _stream_ptr
    q, k, v, o, lse = out.grad_fn.saved_tensors
    (B, Nq, S, D), Nkv, g = q.shape, k.shape[1], dout.transpose(1, 2)
    got = [torch.full((B, S, heads, D), float("inf"), dtype=torch.bfloat16, device=DEV) for heads in (Nq, Nkv, Nkv)]
    dense = lambda heads: _lib._I64x3(S * heads * D, D, heads * D)
    _lib.check(_lib.load().br_prefill_bwd_ex(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), g.data_ptr(), lse.data_ptr(), mask.plan(Nq, Nkv).data_ptr(),
        B, Nq, Nkv, lay.M, lay.H, D, _lib.strides3(q), _lib.strides3(k), _lib.strides3(v), dense(Nq), _lib.strides3(g), _lib._I64x3(Nq * S, S, 1),
        *(t.data_ptr() for t in got), dense(Nq), dense(Nkv), dense(Nkv), D ** -0.5, B * S, workspace.data_ptr(), workspace.numel(),
        max_looks, _stream_ptr(q.device)))
    return [t.transpose(1, 2) for t in got]


def _absolute_sums(lay, q, k, v, o, lse, dout, scale):
    """What bounds any split of a gradient's sums: the sums of their terms' magnitudes, in float64, of the tensors that autograd saved
    (o with its heads behind its tokens)."""
    (B, Nq, S, D), o, dev = q.shape, o.transpose(1, 2), q.device
    assert o.shape == dout.shape == q.shape and lse.shape == (B, Nq, S)
    G = Nq // k.shape[1]
    valid = lay.valid.reshape(B, S).to(dev)
    block = torch.arange(S, device=dev) // lay.H
    sums = [torch.zeros((B, heads, S, D), dtype=torch.float64, device=dev) for heads in (Nq, Nq // G, Nq // G)]
    for b in range(B):
        at = valid[b].nonzero().squeeze(1)
        row, key = block[at][:, None], block[at][None]
        seen = torch.where(row == key, at[:, None] >= at[None], (key == 0) | (row == lay.M - 1)) & (row >= key)
        for h in range(Nq):
            Q, K, V, O, g = (t[b, i, at].double() for t, i in ((q, h), (k, h // G), (v, h // G), (o, h), (dout, h)))
            P = torch.where(seen, torch.exp2(scale * math.log2(math.e) * (Q @ K.T) - lse[b, h, at].double()[:, None]), 0.0)
            dS = (P * (g @ V.T - (g * O).sum(1, keepdim=True))).abs()
            sums[0][b, h, at] = scale * (dS @ K.abs())
            sums[1][b, h // G, at] += scale * (dS.T @ Q.abs())
            sums[2][b, h // G, at] += P.T @ g.abs()
    return sums


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq,Nkv,blocks,two_launches_at", [
    (4, 1, [[5]], ()),                                                   # one block, one item: every other queue is empty
    (2, 1, [[33, 1]], ()),                                               # two query tiles per item, no documents
    (4, 4, [[64, 0, 129, 0, 17], [1, 32, 0, 0, 128]], ()),               # one head to a kv head, empty documents
    (8, 2, [[64] + [(97 * i) % 161 for i in range(30)] + [33]] * 3, ()), # ... and 64 in one
    (8, 2, [[31, 96, 33, 160, 65, 1, 40], [64, 100, 7, 0, 128, 31, 9], [2, 3, 150, 32, 32, 64, 33]], ()),
    (11, 1, [[33, 70, 0, 40]], ()),                                      # no divisor up to eight: a head to a workgroup
    (32, 8, [[61] + [33 + 18 * i for i in range(12)] + [45]] * 2, (64,)),        # more items than workgroups; three to a CU
    (14, 2, [[31, 96, 33, 160, 40]], (64, 128)),                         # seven heads, not four waves
])
def test_one_launch_does_what_two_do(Nq, Nkv, blocks, two_launches_at, D):
    """dK, dV in dQ's launch wait for the deltas of their rows, dQ's last tickets go to whoever is free: the same sums of the same
    products.  A (row, key) pair's products do not depend on who computes them; only rows that several items add to (the query
    block's dQ, the prefix's dK and dV, in fp32) may be summed in another order.  n parts are then n - 1 fp32 roundings of at most
    2^-24 of the parts' magnitudes off on either side, and a bf16 rounding of 2^-8 on either side: n is the non-empty blocks of a
    sequence for the prefix, at most the 64-key tiles of the walk for the query block."""
    from blockrank_amd import _lib
    lay = synthetic.make_layout(blocks)
    out, qkv, dout, mask = _step(lay, 11, Nq, Nkv, D)
    lib, sizes = _lib.load(), (lay.B, Nq, Nkv, lay.M, lay.H, D, lay.B * lay.S)
    least = lib.br_prefill_bwd_workspace_bytes(lay.B, Nq, Nkv, lay.H, D, lay.B * lay.S) + _lib.BR_BWD_TICKET_BYTES
    full = lib.br_prefill_bwd_full_workspace_bytes(*sizes)
    assert [lib.br_prefill_bwd_launches(*sizes, n) for n in (full, least)] == [2 if D in two_launches_at else 1, 2]
    two = _c_backward(out, mask, dout, lay, torch.empty(least, dtype=torch.uint8, device=DEV))
    sums = _absolute_sums(lay, *out.grad_fn.saved_tensors, dout.transpose(1, 2), D ** -0.5)
    one = torch.autograd.grad(out, qkv, dout)
    lengths = torch.as_tensor(lay.lengths)
    tiles = int((lengths + 63).div(64, rounding_mode="floor").sum(1).max())
    for name, a, b, s, n in zip(("dq", "dk", "dv"), one, two, sums, (tiles, *[int((lengths > 0).sum(1).max())] * 2)):
        a, b, s = (t.double().reshape(lay.B, -1, lay.M, lay.H, D) for t in (a, b, s))
        own = slice(0, lay.M - 1) if name == "dq" else slice(1, lay.M)
        assert torch.equal(a[:, :, own], b[:, :, own]), name
        assert ((a - b).abs() <= 2 ** -8 * (a.abs() + b.abs()) + 2 * (n - 1) * 2 ** -24 * 1.01 * s).all(), name


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq,Nkv,one_launch", [(8, 2, True), (14, 2, False)])
def test_an_item_that_gives_up_its_wait_stores_nan(Nq, Nkv, one_launch, D):
    """dK and dV of rows whose deltas did not come within the bound (none do within no looks at all) are NaN, not sums of whatever the
    workspace held; dQ waits for nothing, nor does anything in two launches."""
    from blockrank_amd import _lib
    lay = synthetic.make_layout([[31, 96, 33, 0, 65, 1, 40], [64, 100, 7, 0, 128, 31, 9]])
    out, qkv, dout, mask = _step(lay, 21, Nq, Nkv, D)
    n = _lib.load().br_prefill_bwd_full_workspace_bytes(lay.B, Nq, Nkv, lay.M, lay.H, D, lay.B * lay.S)
    waited, gave_up = (_c_backward(out, mask, dout, lay, torch.zeros(n, dtype=torch.uint8, device=DEV), looks) for looks in (1 << 20, 0))
    _same(waited, torch.autograd.grad(out, qkv, dout))
    if not one_launch:
        return _same(gave_up, waited)
    _same(gave_up[:1], waited[:1])
    real = real_rows(lay).to(DEV)[:, None, :, None]
    for name, t in zip(("dk", "dv"), gave_up[1:]):
        assert (t.isnan() == real).all(), f"{name}: NaN in every real row"
        assert (t.masked_select(~real) == 0).all(), f"{name}: rows of padded slots must be zero"


COUNTER_LINE = 128               # bytes; a pass's 17 ticket counters come first, then one per (sequence, block, kv head)


@pytest.mark.parametrize("Nq,Nkv,D,blocks,launches", [
    (4, 1, 64, [[5]], 1),
    (4, 4, 128, [[64, 0, 129, 0, 17], [1, 32, 0, 0, 128]], 1),
    (8, 2, 64, [[31, 96, 33, 160, 65, 1, 40]] * 3, 1),
    (11, 1, 128, [[33, 70, 0, 40]], 1),                                  # no divisor up to eight: a head to a workgroup
    (14, 2, 128, [[31, 96, 33, 160, 40]], 2),
    (8, 1, 64, [[31, 96, 33, 160, 40]], 2),
    (32, 8, 64, [[61] + [33 + 18 * i for i in range(12)] + [45]] * 2, 2),
])
def test_a_pass_uses_the_counters_of_its_form(Nq, Nkv, D, blocks, launches):
    """One launch counts every (32 rows, query head) of a block whose delta is published; two touch nothing behind the tickets, and
    are not given any of it."""
    from blockrank_amd import _lib
    lay = synthetic.make_layout(blocks)
    out, qkv, dout, mask = _step(lay, 31, Nq, Nkv, D)
    lib, sizes = _lib.load(), (lay.B, Nq, Nkv, lay.M, lay.H, D, lay.B * lay.S)
    stated, full = lib.br_prefill_bwd_workspace_bytes(lay.B, Nq, Nkv, lay.H, D, lay.B * lay.S), lib.br_prefill_bwd_full_workspace_bytes(*sizes)
    pairs = lay.B * lay.M * Nkv
    assert full == stated + COUNTER_LINE * (17 + (pairs if launches == 1 else 0))
    assert lib.br_prefill_bwd_launches(*sizes, full) == launches
    assert [lib.br_prefill_bwd_launches(*sizes, n) for n in (full - 1, stated, stated - 1)] == [2, 2, 0]
    ws = torch.full((stated + COUNTER_LINE * (17 + pairs),), 0x5a, dtype=torch.uint8, device=DEV)
    _same(_c_backward(out, mask, dout, lay, ws), torch.autograd.grad(out, qkv, dout))
    counters = ws[stated + COUNTER_LINE * 17:].view(torch.int32).view(lay.B, lay.M, Nkv, COUNTER_LINE // 4)[..., 0].cpu()
    if launches == 1:
        rows = (torch.as_tensor(lay.lengths) + 31) // 32
        assert (counters == (rows * (Nq // Nkv))[..., None]).all()
    else:
        assert (counters == 0x5a5a5a5a).all()


@pytest.mark.parametrize("blocks", [23, 24])
def test_either_side_of_the_third_workgroup(blocks):
    """Head dim 64 on 256 compute units: three workgroups each from 6 x 256 items on, a block of 16 slots being one for each of 32 heads."""
    gen = np.random.default_rng(blocks)
    _check(synthetic.make_layout([[16] + gen.integers(0, 17, blocks - 2).tolist() + [9] for _ in range(2)]), 32, 32, 64, seed=blocks)
