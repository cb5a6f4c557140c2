"""compute_auxiliary_attention_loss on dense logits: what its kernels take is what the torch expressions take, with their
results - the same call on CPU tensors, which runs the expressions, is the reference."""
import pytest
import torch

import blockrank_amd as br
from blockrank_amd import attention, losses, synthetic

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
B, N, H1, DOCS, H = 3, 4, 16, 5, 24
M = DOCS + 2


def _inputs(seed=0, dtype=torch.float32, batch=B):
    g = torch.Generator().manual_seed(seed)
    x = (3 * torch.randn(batch, N, H1, M * H, generator=g)).to(dtype)
    labels = torch.full((B, M * H), -100)
    labels[torch.arange(B), M * H - H1 + torch.tensor([3, 15, 1])] = 7
    return x, labels, torch.ones(B, M, H, dtype=torch.bool), torch.tensor([[1, -1], [0, 4], [2, 2]])


def _call(device, x, labels, mask, answers=None, rows=None, **kw):
    to = lambda t: t.to(device) if torch.is_tensor(t) else t
    return br.compute_auxiliary_attention_loss(to(x), to(labels), to(mask), answer_ids=to(answers), return_logits=True, rows=to(rows), **kw)


def _close(got, want, **tol):
    torch.testing.assert_close(got.detach().cpu(), want.detach(), equal_nan=True, **(tol or dict(rtol=2e-5, atol=2e-6)))


def _loss_and_grad(device, x, labels, mask, answers, rows, **kw):
    x = x.detach().to(device).requires_grad_(True)
    loss, acc, scores = _call(device, x, labels, mask, answers, rows, **kw)
    (loss + (scores * torch.arange(1, DOCS + 1, device=device)).sum()).backward()
    return loss, acc, scores, x.grad


# ---- which rows ---------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("rows", [torch.tensor([[3, 9]]), torch.tensor([[5]])])
def test_rows_of_one_sequence_serve_a_batch(rows):
    x, labels, mask, answers = _inputs()
    for got, want in zip(_loss_and_grad(DEV, x, labels, mask, answers, rows), _loss_and_grad("cpu", x, labels, mask, answers, rows)):
        _close(got, want)
    # labels of one sequence, and logits of one: what the expressions broadcast
    one = labels[:1]
    for got, want in zip(_loss_and_grad(DEV, x, one, mask, answers, None), _loss_and_grad("cpu", x, one, mask, answers, None)):
        _close(got, want)
    x1 = _inputs(batch=1)[0]
    many = torch.tensor([[0, 1], [2, 3], [4, 5]])
    for got, want in zip(_loss_and_grad(DEV, x1, labels, mask, answers, many), _loss_and_grad("cpu", x1, labels, mask, answers, many)):
        _close(got, want)


def test_rows_that_do_not_fit_the_batch_are_refused():
    x, labels, mask, _ = _inputs()
    for device in ("cpu", DEV):
        with pytest.raises(RuntimeError):
            _call(device, x, labels, mask, rows=torch.tensor([[0, 1], [2, 3]]))
        with pytest.raises(RuntimeError, match="Long"):
            _call(device, x, labels, mask, rows=torch.zeros(B, 2, dtype=torch.int32))


def test_rows_outside_the_last_rows_wrap_around_as_take_along_dim_has_it():
    x, labels, mask, answers = _inputs(1)
    rows = torch.tensor([[-1, 2], [16, -16], [37, -35]])
    for got, want in zip(_loss_and_grad(DEV, x, labels, mask, answers, rows), _loss_and_grad("cpu", x, labels, mask, answers, rows)):
        _close(got, want)


def test_answers_beyond_the_documents_are_refused():
    x, labels, mask, answers = _inputs(2)
    answers[0, 1] = DOCS                                        # the padding column of the expressions: ignored
    for rows in (None, torch.tensor([[1, 2], [3, 4], [5, 6]])):
        for got, want in zip(_call(DEV, x, labels, mask, answers, rows), _call("cpu", x, labels, mask, answers, rows)):
            _close(got, want)
    answers[1, 0] = DOCS + 1
    for device in ("cpu", DEV):
        for rows in (None, torch.tensor([[1, 2], [3, 4], [5, 6]])):
            for dtype in (torch.float32, torch.float64):        # (float64 is left to the expressions on the GPU too)
                with pytest.raises(RuntimeError, match="out of bounds"):
                    _call(device, x.to(dtype), labels, mask, answers, rows)


# ---- what is differentiated, and how ------------------------------------------------------------------------------

def test_gradient_of_the_gradient():
    x, labels, mask, answers = _inputs(3)
    out = []
    for device in ("cpu", DEV):
        y = x.detach().to(device).requires_grad_(True)
        loss, _, scores = _call(device, y, labels, mask, answers, temperature=1.5)
        w = torch.linspace(-1, 1, DOCS, device=device)
        g, = torch.autograd.grad(loss + (scores * scores * w).sum(), y, create_graph=True)
        (g * torch.cos(torch.arange(g.numel(), device=device)).view_as(g)).sum().backward()
        out.append((g.detach().cpu(), y.grad.cpu()))
    for got, want in zip(out[1], out[0]):
        torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-6)


def test_function_transforms_and_forward_mode():
    x, labels, mask, answers = _inputs(4)
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]])
    t = torch.randn(x.shape, generator=torch.Generator().manual_seed(1))
    xs = torch.stack([x, 0.5 * x])
    res = []
    for device in ("cpu", DEV):
        scores = lambda y: _call(device, y, labels, mask, rows=rows)
        jvp = torch.func.jvp(scores, (x.to(device),), (t.to(device),))
        with torch.autograd.forward_ad.dual_level():
            dual = scores(torch.autograd.forward_ad.make_dual(x.to(device), t.to(device)))
            tangent = torch.autograd.forward_ad.unpack_dual(dual).tangent
        res.append([*jvp, tangent, torch.func.vmap(scores)(xs.to(device)),
                    torch.func.grad(lambda y: _call(device, y, labels, mask, answers, rows)[0])(x.to(device))])
    for got, want in zip(res[1], res[0]):
        _close(got, want)


def test_in_a_compiled_function():
    x, labels, mask, answers = _inputs(10)
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]])
    step = torch.compile(lambda y: _call(DEV, y, labels, mask, answers, rows), backend="eager")
    y = x.to(DEV).requires_grad_(True)
    got = step(y)
    got[0].backward()
    want = _loss_and_grad("cpu", x, labels, mask, answers, rows)
    for a, b in zip(got, want):
        _close(a, b)
    assert torch.isfinite(y.grad).all() and y.grad.abs().max() > 0


def test_a_temperature_that_is_a_tensor_has_a_gradient():
    x, labels, mask, answers = _inputs(5)
    grads = []
    for device in ("cpu", DEV):
        t = torch.tensor(0.3, device=device, requires_grad=True)
        _call(device, x, labels, mask, answers, temperature=t)[0].backward()
        grads.append(t.grad.cpu())
    _close(grads[1], grads[0])


# ---- values that are not finite, and how exact the others are -------------------------------------------------------

@pytest.mark.parametrize("what", ["nan document", "nan slot", "inf slot", "-inf document", "-inf everywhere", "nan everywhere"])
def test_logits_that_are_not_finite(what):
    x, labels, mask, answers = _inputs(6)
    nan, inf = float("nan"), float("inf")
    if what == "nan document":
        x[0, :, :, 2 * H:3 * H] = nan
    elif what == "nan slot":
        x[0, 1, :, 2 * H + 3] = nan
    elif what == "inf slot":
        x[0, 1, :, 2 * H + 3] = inf
    elif what == "-inf document":
        x[:, :, :, 2 * H:3 * H] = -inf
    else:
        x[0] = -inf if what[0] == "-" else nan
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]])
    for got, want in zip(_loss_and_grad(DEV, x, labels, mask, answers, rows), _loss_and_grad("cpu", x, labels, mask, answers, rows)):
        _close(got, want)


@pytest.mark.parametrize("scores", [[0.1, float("nan"), 3.0], [float("-inf")] * 3, [1.0, float("-inf"), 0.0], [float("nan")] * 3])
def test_infonce_of_scores_that_are_not_finite(scores):
    answers = torch.tensor([[1]])
    out = []
    for device in ("cpu", DEV):
        s = torch.tensor([scores], device=device, requires_grad=True)
        loss, acc = losses._infonce(s, answers.to(device), False)
        loss.backward()
        out.append((loss, acc, s.grad.cpu()))
    for got, want in zip(out[1], out[0]):
        _close(got, want)


@pytest.mark.parametrize("spread", [0.5, 8.0, 60.0])
def test_scores_loss_and_gradient_are_as_exact_as_the_expressions(spread):
    """Against float64, no further off than the fp32 expressions are on the same inputs (half as far again allowed, for the
    order of the sums)."""
    x, labels, mask, answers = _inputs(7)
    x = x * (spread / 3)
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]])
    temperature = 0.05 if spread < 60 else 1.0
    exact = _loss_and_grad("cpu", x.double(), labels, mask, answers, rows, temperature=temperature)
    plain = _loss_and_grad("cpu", x, labels, mask, answers, rows, temperature=temperature)
    got = _loss_and_grad(DEV, x, labels, mask, answers, rows, temperature=temperature)
    for name, e, p, w in zip(("loss", "accuracy", "scores", "gradient"), exact, plain, got):
        off = lambda t: ((t.detach().cpu().double() - e).norm() / e.norm().clamp_min(1e-30)).item()
        assert off(w) <= 1.5 * off(p) + 6e-8, f"{name}: {off(w):.2e} against {off(p):.2e} of the fp32 expressions"


@pytest.mark.parametrize("batch,docs,slots", [(1, 3, 24), (3, 2, 7), (2, 17, 520), (16, 64, 16), (17, 64, 16), (5, 193, 16)])
@pytest.mark.parametrize("of", ["loss", "scores", "both", "loss without scores"])
def test_loss_and_scores_of_one_call(batch, docs, slots, of):
    """Fewer documents than waves and more, slots beyond a wave's registers, an odd row length (zeros by the element), the sums
    in the loss's own workgroup and in a launch of theirs (up to, beyond sixteen times 64 documents); the gradient of either
    output alone, and of a loss that comes without the scores.  The bound is that of the test above."""
    g = torch.Generator().manual_seed(docs)
    blocks, h1 = docs + 2, 5
    x = 2 * torch.randn(batch, 3, h1, blocks * slots, generator=g)
    labels = torch.full((batch, blocks * slots), -100)
    labels[torch.arange(batch), blocks * slots - 1 - torch.arange(batch) % 4] = 7
    answers = torch.randint(-1, docs, (batch, 2), generator=g)
    answers[:, 0] = torch.randint(0, docs, (batch,), generator=g)
    weight = torch.randn(batch, docs, generator=g)

    def both(device, dtype=torch.float32):
        z = x.to(device, dtype, copy=True).requires_grad_(True)
        call = lambda z, **kw: br.compute_auxiliary_attention_loss(z, labels.to(device), torch.ones(batch, blocks, slots, dtype=torch.bool, device=device),
                                                                   answer_ids=answers.to(device), **kw)
        if of == "loss without scores":
            loss, acc = call(z)
            loss.backward()
            return loss.detach(), acc, z.grad
        loss, acc, scores = call(z, return_logits=True)
        y = (scores * weight.to(device, dtype)).sum()
        {"loss": loss, "scores": y, "both": loss + y}[of].backward()
        return loss.detach(), acc, z.grad, scores.detach()

    exact, plain, got = both("cpu", torch.float64), both("cpu"), both(DEV)
    for name, e, p, w in zip(("loss", "accuracy", "gradient", "scores"), exact, plain, got):
        off = lambda t: ((t.cpu().double() - e).norm() / e.norm().clamp_min(1e-30)).item()
        assert off(w) <= 1.5 * off(p) + 6e-8, f"{name}: {off(w):.2e} against {off(p):.2e} of the fp32 expressions"


@pytest.mark.parametrize("rows", [None, torch.tensor([[1, 2], [3, 4], [5, 6]])])
def test_the_loss_is_a_function_of_the_scores_it_is_returned_with(rows):
    """Differentiated with respect to them, their gradient retained, hooks on them that change it or keep it, and with a graph
    of its own; the bound of _close: a few fp32 roundings of an exponential each."""
    x, labels, mask, answers = _inputs(11)
    res = []
    for device in ("cpu", DEV):
        y = x.detach().to(device).requires_grad_(True)
        loss, _, scores = _call(device, y, labels, mask, answers, rows, temperature=0.5)
        of_scores, = torch.autograd.grad(loss, scores, retain_graph=True)
        curved, = torch.autograd.grad(loss, scores, create_graph=True)
        (curved * torch.arange(DOCS, device=device)).sum().backward(inputs=[y], retain_graph=True)
        out, y.grad = [of_scores, y.grad], None
        scores.retain_grad()
        seen = []
        scores.register_hook(seen.append)
        loss.backward(inputs=[y], retain_graph=True)
        out, y.grad = [*out, y.grad, scores.grad, *seen], None
        scores.register_hook(lambda g: 0.25 * g.clamp(min=-0.1))
        loss.backward(inputs=[y])
        res.append([*out, y.grad])
    assert len(res[0]) == len(res[1])
    for got, want in zip(res[1], res[0]):
        _close(got, want)
        assert want.abs().max() > 0


def test_scores_of_documents_of_little_mass_are_as_exact_as_the_expressions():
    """Logits on a grid of 1/8, so that differences are exact and what is left is the exponential's own error: per document
    at most 1e-6 off (24 slots, 4 heads, 2 rows: sums of fp32 roundings of 6e-8 each, with an exponential good to an ulp); an
    exponential of the product with log2 e rounded to fp32 is off by |x| * 6e-8, 3e-6 here."""
    x, labels, mask, _ = _inputs(9)
    x = (x * 8).round() / 8
    x[..., H:2 * H] += 48                                       # the first document has all the mass but e^-48
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]])
    exact = _call("cpu", x.double(), labels, mask, rows=rows)
    for device in ("cpu", DEV):
        off = ((_call(device, x, labels, mask, rows=rows).cpu().double() - exact) / exact).abs().max().item()
        assert off <= 1e-6, f"{device}: {off:.2e}"


def test_loss_under_graph_capture():
    """Rows known beforehand: nothing waits, so the loss can be captured; answers beyond the documents are NaN there."""
    x, labels, mask, answers = (t.to(DEV) for t in _inputs(8))
    rows = torch.tensor([[1, 2], [3, 4], [5, 6]], device=DEV)
    call = lambda: br.compute_auxiliary_attention_loss(x, labels, mask, answer_ids=answers, return_logits=True, rows=rows)
    with torch.no_grad():
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        for seed in (1, 2, 3):
            x.copy_(_inputs(seed)[0])
            answers[0, 0] = seed
            graph.replay()
            torch.cuda.synchronize()
            for got, want in zip(out, call()):
                assert torch.equal(got, want)
        answers[0, 0] = DOCS + 1
        graph.replay()
        torch.cuda.synchronize()
        assert torch.isnan(out[0]) and torch.isnan(out[1])


# ---- state that outlives a call -----------------------------------------------------------------------------------

def test_rows_made_in_inference_mode_serve_training():
    lay = synthetic.make_layout([[9, 30, 17, 20]])
    q, k, _ = synthetic.random_qkv(lay, 4, 2, 64, torch.float32, DEV, seed=1)
    bm = br.BlockMask(lay.valid.to(DEV), torch.float32)
    R = 11                                                       # (a size that no other test has made the rows of)
    with torch.inference_mode():
        br.LastBlockScores(q, k, bm, 0.2, R).dense()
    q.requires_grad_(True)
    br.LastBlockScores(q, k, bm, 0.2, R).dense().sum().backward()
    assert torch.isfinite(q.grad).all()


def test_rows_of_the_last_positions_are_kept_within_bounds(monkeypatch):
    monkeypatch.setattr(attention, "_LAST_ROWS", {})
    first = attention._last_rows(1, 40, 1, torch.device(DEV))
    for R in range(2, 40):
        for n in (1, 2):
            want = torch.arange(40 - R, 40, dtype=torch.int32).expand(n, R)
            for _ in range(2):
                assert torch.equal(attention._last_rows(n, 40, R, torch.device(DEV)).cpu(), want)
    assert len(attention._LAST_ROWS) == 64
    assert attention._last_rows(1, 40, 1, torch.device(DEV)) is first


def test_rows_of_the_callers_made_in_inference_mode():
    """The handle compares them with its guess; such a tensor has no version to remember the comparison by."""
    lay = synthetic.make_layout([[9, 30, 17, 20]])
    q, k, v = synthetic.random_qkv(lay, 4, 2, 64, torch.bfloat16, DEV, seed=1)

    class Layer:
        layer_idx, num_key_value_groups, training = 0, 2, False

    with torch.inference_mode():
        _, handle = br.blockrank_attention_forward(Layer(), q, k, v, br.BlockMask(lay.valid.to(DEV), q.dtype), 0.125, layers_to_return_scores=[0])
        rows = torch.tensor([[14, 15]], device=DEV)
        for _ in range(2):
            assert torch.equal(handle.doc_scores_window(rows), handle.ranked[2])
        rows -= 1
        assert not torch.equal(handle.doc_scores_window(rows), handle.ranked[2])
