"""Infinities and NaN stay in the rows that see them: a row of Q that is not finite makes that row of that head not finite,
a key's or value's make the rows that attend to it so (the rows of its block, and of the query block), and every other row
is bit for bit what it is without them.  Layouts whose key walks end in tiles that are only partly filled."""
import pytest
import torch

import blockrank_amd as br
from blockrank_amd import synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = [[40, 100, 75, 9, 130, 45], [70, 33, 128, 64, 1, 20]]
HEADS = [(8, 2, 128, torch.bfloat16, False), (14, 2, 128, torch.bfloat16, False), (4, 4, 64, torch.bfloat16, False),
         (10, 2, 64, torch.float16, False), (8, 2, 128, torch.bfloat16, True), (8, 2, 128, torch.float32, False)]


def _differing_rows(q, k, v, lay, bad_q, bad_k, bad_v, fp8):
    """(B, S, Nq) bool: rows of real tokens whose output is not bit for bit the same with the non-finite tensors."""
    mask = br.BlockMask(lay.valid.to(DEV), q.dtype)
    scale = q.shape[-1] ** -0.5
    for _ in range(2):       # (twice: what an earlier launch left behind must not matter either)
        clean = br.blockrank_attention(q, k, v, mask, scale, qk_fp8=fp8)
        dirty = br.blockrank_attention(bad_q, bad_k, bad_v, mask, scale, qk_fp8=fp8)
    real = lay.valid.reshape(lay.B, lay.S).to(DEV)
    assert torch.isfinite(clean[real]).all()
    return ((clean != dirty) | ~torch.isfinite(dirty)).any(-1) & real[:, :, None]


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("Nq,Nkv,D,dtype,fp8", HEADS)
def test_a_row_of_q_that_is_not_finite_stays_in_its_row(Nq, Nkv, D, dtype, fp8, bad):
    lay = synthetic.make_layout(LENGTHS)
    q, k, v = synthetic.random_qkv(lay, Nq, Nkv, D, dtype, DEV, seed=7)
    G = Nq // Nkv
    for which in range(G):   # one head of every group, the last token of every block (rows past it repeat it)
        hit = q.clone()
        want = torch.zeros(lay.B, lay.S, Nq, dtype=torch.bool, device=DEV)
        hit[:, which::G, lay.H - 1::lay.H] = bad
        want[:, lay.H - 1::lay.H, which::G] = True
        got = _differing_rows(q, k, v, lay, hit, k, v, fp8)
        assert not (got & ~want).any(), f"head {which} of a group: rows that do not hold the bad value changed"
        assert fp8 or (got == want).all()


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("Nq,Nkv,D,dtype,fp8", [h for h in HEADS if not h[4]])
def test_keys_and_values_that_are_not_finite_stay_with_the_rows_that_see_them(Nq, Nkv, D, dtype, fp8, which):
    lay = synthetic.make_layout(LENGTHS * 24)      # (workgroups take several items one after the other)
    q, k, v = synthetic.random_qkv(lay, Nq, Nkv, D, dtype, DEV, seed=8)
    bad = {"k": k.clone(), "v": v.clone()}
    bad[which][1::2, :, 2 * lay.H:3 * lay.H] = float("nan")                # a document of every other sequence, whole
    got = _differing_rows(q, k, v, lay, q, bad["k"], bad["v"], fp8)
    want = torch.zeros_like(got)
    want[1::2, 2 * lay.H:3 * lay.H] = True
    want[1::2, (lay.M - 1) * lay.H:] = True
    want &= lay.valid.reshape(lay.B, lay.S, 1).to(DEV)
    assert (got == want).all()


@pytest.mark.parametrize("docs", [4, 100, 300])                  # (the three forms of the reduction over documents)
@pytest.mark.parametrize("where", ["query row", "document key"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_scores_of_a_sequence_that_is_not_finite(dtype, where, docs):
    """NaN for that sequence, as the softmax of the expressions on the logits has it, and nothing of it for the other."""
    lay = synthetic.make_layout([[20] + [5 + (7 * i) % 20 for i in range(docs)] + [16], [9] + [3 + (5 * i) % 20 for i in range(docs)] + [16]])
    q, k, v = synthetic.random_qkv(lay, 4, 2, 64, dtype, DEV, seed=9)
    if where == "query row":
        q[1, 2, -1] = float("nan")
    else:
        k[1, 1, 3 * lay.H - 1] = float("inf")

    class Layer:
        layer_idx, num_key_value_groups, training = 0, 2, False

    mask = br.BlockMask(lay.valid.to(DEV), dtype)
    _, handle = br.blockrank_attention_forward(Layer(), q, k, v, mask, 0.125, layers_to_return_scores=[0])
    call = lambda x: br.compute_auxiliary_attention_loss(x, lay.labels.to(DEV), lay.valid.to(DEV), return_logits=True)
    want = call(handle.dense())
    rows = torch.tensor([[14, 15]] * 2, device=DEV)
    for got in (call(handle), handle.doc_scores(rows + lay.H - 16), handle.doc_scores_window(rows, head_reduce="sum") / 4):
        assert torch.isfinite(got[0]).all() and torch.isnan(got[1]).all() and torch.isnan(want[1]).all()
        torch.testing.assert_close(got[0], want[0], rtol=1e-3, atol=1e-5)

