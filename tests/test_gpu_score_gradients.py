"""The score logits, their gradient and the steps of the ranking loss as kernels, at the sizes where their tiles end:
head groups that do not fill a pair of heads, rows that do not fill sixteen, slot counts that are no multiple of a chunk
or of four, a key axis long enough to be cut.  Against float64 / torch expressions of the same formulas."""
import pytest
import torch
import torch.nn.functional as F

import blockrank_amd as br
from blockrank_amd import losses, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("lengths,H,Nq,Nkv,D,R,dtype", [
    ([[9, 30, 0, 17, 20]], None, 1, 1, 64, 1, torch.bfloat16),
    ([[5, 7, 19]], 19, 6, 2, 128, 5, torch.bfloat16),                       # 57 slots: no aligned pieces of a row
    ([[31, 100, 64, 65, 33], [33, 1, 128, 90, 64]], None, 7, 1, 64, 16, torch.bfloat16),
    ([[64] + [250, 131, 256] * 8 + [40]], None, 8, 1, 128, 12, torch.bfloat16),   # many chunks of the key axis
    ([[20, 33, 12, 16]], None, 16, 1, 64, 9, torch.float16),
    ([[20, 333, 12, 17]], None, 4, 4, 128, 16, torch.float32),
])
def test_logits_and_their_gradient(lengths, H, Nq, Nkv, D, R, dtype):
    lay = synthetic.make_layout(lengths, H=H)
    B, S, H, scale = lay.B, lay.S, lay.H, 0.17
    q0, k0, _ = synthetic.random_qkv(lay, Nq, Nkv, D, dtype, DEV, seed=5)
    valid = lay.valid.to(DEV).reshape(B, S)
    ds = torch.randn(B, Nq, R, S, generator=torch.Generator().manual_seed(2)).to(DEV)
    qr, kr = q0.double().requires_grad_(True), k0.double().requires_grad_(True)
    tok = torch.arange(S - R, S, device=DEV)
    dots = scale * (qr[:, :, tok] @ kr.repeat_interleave(Nq // Nkv, dim=1).transpose(-1, -2).contiguous())
    dots = dots * (valid[:, tok][:, None, :, None] & valid[:, None, None, :])
    (dots * ds.double()).sum().backward()
    q, k = q0.clone().requires_grad_(True), k0.clone().requires_grad_(True)
    got = br.LastBlockScores(q, k, br.BlockMask(lay.valid.to(DEV), dtype), scale, R).dense()
    see = valid[:, None, None, :] & (torch.arange(S, device=DEV)[None, :] <= tok[:, None])[None, None] & valid[:, tok][:, None, :, None]
    want = dots.detach() + torch.where(see, 0.0, 0.7 * torch.finfo(dtype).min)
    torch.testing.assert_close(got.detach().double(), want, rtol=1e-5, atol=2e-4)
    (got * ds).sum().backward()
    for t, w in ((q, qr), (k, kr)):
        err = (t.grad.double() - w.grad).abs().max() / w.grad.abs().max()
        assert err <= (2e-5 if dtype == torch.float32 else 6e-3), err.item()


@pytest.mark.parametrize("docs,H,N,B", [(1, 16, 1, 1), (3, 70, 5, 2), (66, 16, 4, 5), (300, 32, 2, 17)])
def test_loss_on_dense_logits(docs, H, N, B):
    g = torch.Generator().manual_seed(docs)
    M, h1 = docs + 2, 16
    x0 = (4 * torch.randn(B, N, h1, M * H, generator=g)).to(DEV)
    x0[:, :, :, H:H + 5] = -1e38
    rows = torch.randint(0, h1, (B, 2), generator=g)
    rows[0] = 3                                                             # the same row twice
    answers = torch.randint(0, docs, (B, 2), generator=g)
    answers[0, 1] = -1
    labels = torch.full((B, M * H), -100)
    at = torch.randint(1, h1, (B,), generator=g)
    labels[torch.arange(B), M * H - h1 + at] = 5
    rows, answers, labels = rows.to(DEV), answers.to(DEV), labels.to(DEV)
    mask = torch.ones(B, M, H, dtype=torch.bool, device=DEV)
    for rr in (rows, None):
        x = x0.clone().requires_grad_(True)
        loss, acc, scores = br.compute_auxiliary_attention_loss(x, labels, mask, answer_ids=answers, return_logits=True, rows=rr)
        (loss + (scores * 0.01).sum()).backward()
        y = x0.double().requires_grad_(True)
        r = rows if rr is not None else torch.stack([at - 1, at], dim=1).to(DEV)
        p = F.softmax(y.take_along_dim(r[:, None, :, None], dim=2)[..., H:-H], dim=-1).reshape(B, N, -1, docs, H)
        want = p.mean(dim=(1, 2)).sum(dim=-1) / 0.05
        pos = torch.zeros(B, docs + 1, dtype=torch.bool, device=DEV).scatter_(1, torch.where(answers >= 0, answers, docs), True)[:, :-1]
        wloss = -(torch.logsumexp(want.masked_fill(~pos, float("-inf")), 1) - torch.logsumexp(want, 1)).mean()
        (wloss + (want * 0.01).sum()).backward()
        torch.testing.assert_close(scores.double(), want, rtol=2e-5, atol=1e-6)
        # (scores of up to 20 carry roundings of 1e-6 into the loss and its exponentials)
        torch.testing.assert_close(loss.double(), wloss, rtol=2e-6, atol=4e-6)
        assert acc.item() == pytest.approx(pos.gather(1, want.argmax(1, keepdim=True)).double().mean().item())
        torch.testing.assert_close(x.grad.double(), y.grad, rtol=1e-3, atol=1e-6)
        # (one document: the gradient is p (g - p g) / temperature = 0 but for p's rounding, 2^-22 of 0.01 / 0.05)
        assert (x.grad.double() - y.grad).norm() <= 1e-5 * y.grad.norm() + 2 ** -22 * 0.01 / 0.05


def test_bracket_rows_kernel():
    labels = torch.full((70, 40), -100, device=DEV)
    at = torch.randint(1, 16, (70,), generator=torch.Generator().manual_seed(1)).to(DEV)
    labels[torch.arange(70, device=DEV), 24 + at] = 9
    want = torch.stack([at - 1, at], dim=1)
    assert torch.equal(losses.bracket_rows(labels, 16), want)
    assert losses.bracket_rows(labels, 16, want.to(torch.int32), return_match=True)[1]
    assert not losses.bracket_rows(labels, 16, (want + 1).to(torch.int32), return_match=True)[1]
    labels[3] = -100
    with pytest.raises(AssertionError, match="Bracket token"):
        losses.bracket_rows(labels, 16)
    labels[3, -16] = 1                                                      # nothing in front of the bracket
    with pytest.raises(AssertionError, match="Bracket token"):
        losses.bracket_rows(labels, 16)
