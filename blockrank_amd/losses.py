"""Per-document relevance scores from the query block's attention (the reference's layer-score API).

Drop-in for src/blockrank/losses.py::compute_auxiliary_attention_loss: same name, arguments and
return values.  When ``attention_scores`` is the LastBlockScores handle this package's attention hook
returns, the scores come from the fused HIP kernel; a plain (B, N, h1, M*H) tensor (for instance from
``LastBlockScores.dense()`` or from the reference's own attention) is reduced with the same formula in
torch.
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F
from torch._C import _are_functorch_transforms_active as _transforms_active
from torch._C import _get_tracing_state as _tracing_state
from torch.autograd import forward_ad
from torch.compiler import is_compiling

from . import _lib
from .attention import LastBlockScores, _stream_ptr


_NEVER_FREED: list = []
_BEYOND = "answer_ids: index out of bounds for the number of documents"
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _eager(*tensors: torch.Tensor) -> bool:
    """Whether the tensors have memory that a kernel can be given: not under a function transform (vmap, torch.func.grad), in
    forward-mode differentiation, in a trace or a compilation, or as a subclass; the torch expressions serve those."""
    if is_compiling():
        return False
    for t in tensors:
        if type(t) not in _PLAIN:
            return False
    return not (_transforms_active() or forward_ad._current_level >= 0 or _tracing_state())


class _HostFlags:
    """What the host has to know of the device's work, as int32 in pinned memory that kernels write and ``read()``, which
    waits for them, returns: work that does not depend on it can be enqueued in between.  BRACKET: every sequence has
    its bracket; MATCH: the rows equal the guess; ANSWERS (where ``answers`` is set): no answer is beyond the documents."""

    BRACKET, MATCH, ANSWERS = range(3)
    SPIN = 300                                   # microseconds
    answers = pending = False
    first, end = 3, 0                            # the flags that a kernel was given

    def __init__(self, device: torch.device):
        self.device = device
        self._make()

    def _make(self) -> int:
        self.flags = torch.empty(3, dtype=torch.int32, pin_memory=True)
        at = self.flags.data_ptr()
        ctypes.memset(at, 0xff, 12)              # -1: not written yet
        return at

    def ptr(self, i: int = 0) -> int:
        self.pending, self.first, self.end = True, min(i, self.first), max(i + 1, self.end)
        return self.flags.data_ptr() + 4 * i

    def read(self) -> list[int]:
        # Waiting for the stream costs a marker behind the kernel and its way back, five microseconds of a pass that takes the
        # device forty; the flags themselves are seen as they are written.  Not for ever, and not in a long wait's place.
        if not _lib.load().br_wait_written(self.flags.data_ptr() + 4 * self.first, self.end - self.first, self.SPIN):
            torch.cuda.current_stream(self.device).synchronize()
        self.pending = False
        flags = self.flags.tolist()
        if self.answers and not flags[self.ANSWERS]:
            raise RuntimeError(_BEYOND)
        return flags

    def __del__(self):
        # The host allocator does not know that a kernel writes the flags: where an exception came before read(), they must
        # not go back to it while one may still be running.
        if self.pending:
            try:
                torch.cuda.synchronize(self.device)
            except Exception:                    # (nothing can be waited for, as in a capture that failed)
                _NEVER_FREED.append(self.flags)


class _BracketRows(_HostFlags):
    """losses.py:43-48 on the device in one launch: ``rows`` (B, 2) are the first label > -100 (the "[" token) and the
    position before it, as indices into the last h1 positions, or, with ``pos_offset``, ``pos`` the same as positions 0..H-1
    of a block of that many more slots.  ``check()``: every sequence has its bracket, or an AssertionError; whether the rows
    equal ``guess``."""

    rows = pos = None

    def __init__(self, labels: torch.Tensor, h1: int, guess: torch.Tensor | None, pos_offset: int | None = None):
        B, S = labels.shape
        dev = labels.device
        self.device = dev
        with _lib.on_device(dev):
            if pos_offset is None:
                self.rows = out = torch.empty((B, 2), dtype=torch.int64, device=dev)
                where = out.data_ptr(), None, 0
            else:
                self.pos = out = torch.empty((B, 2), dtype=torch.int32, device=dev)
                where = None, out.data_ptr(), pos_offset
            at = self._make()
            self.pending, self.first, self.end = True, 0, 2
            _lib.check(_lib.load().br_bracket_rows(labels.data_ptr(), labels.stride(0), B, S, h1, guess.data_ptr() if guess is not None else None,
                                                   *where, at, _stream_ptr(dev)))

    @staticmethod
    def takes(labels: torch.Tensor, h1: int, guess: torch.Tensor | None) -> bool:
        return (labels.is_cuda and _eager(labels) and labels.dtype == torch.int64 and labels.dim() == 2 and labels.stride(1) == 1 and labels.shape[0] > 0
                and labels.stride(0) >= labels.shape[1] and 0 < h1 <= labels.shape[1]
                and (guess is None or (guess.device == labels.device and guess.dtype == torch.int32 and guess.is_contiguous()
                                       and guess.shape == (labels.shape[0], 2))))

    def check(self) -> bool:
        bracket, match, _ = self.read()
        assert bracket, "Bracket token not found in last h1 positions."
        return bool(match)


def bracket_rows(labels: torch.Tensor, h1: int, guess: torch.Tensor | None = None, return_match: bool = False):
    """(B, S) labels -> (B, 2) indices into the last h1 positions: the first label > -100 (the "["
    token) and the position before it (losses.py:43-48).  With ``guess`` (B, 2) and ``return_match`` also whether the
    rows equal it, found out in the same host synchronisation as the reference's bracket check."""
    if guess is not None and (not return_match or guess.shape != (labels.shape[0], 2)):
        guess = None
    if _BracketRows.takes(labels, h1, guess):
        found = _BracketRows(labels, h1, guess)
        match = found.check()
        return (found.rows, match) if return_match else found.rows
    last = labels[:, -h1:] > -100
    br = last.int().argmax(dim=-1)[:, None]
    rows = torch.hstack([br - 1, br])
    if guess is None:
        assert torch.all(rows >= 0), "Bracket token not found in last h1 positions."
        return (rows, False) if return_match else rows
    same = (rows == guess.to(rows.device)).all()
    ok, match = torch.stack([torch.all(rows >= 0), same]).tolist()
    assert ok, "Bracket token not found in last h1 positions."
    return rows, bool(match)


class _LossWithScores:
    """The loss on scores that are being made, from the launches that make them: ``results`` are then _InfoNCE's."""

    results = None

    def __init__(self, answer_ids: torch.Tensor, host: _HostFlags):
        self.answer_ids, self.host = answer_ids, host

    def make(self, x, rows, sizes, probs_at: int, stat_at: int, scores: torch.Tensor):
        B, dev = scores.shape[0], x.device
        loss, accuracy = torch.empty((), dtype=torch.float32, device=dev), torch.empty((), dtype=torch.float32, device=dev)
        lse = torch.empty((B, 2), dtype=torch.float32, device=dev)
        _lib.check(_lib.load().br_ranking_loss(x.data_ptr(), rows.data_ptr(), *sizes, self.answer_ids.data_ptr(), self.answer_ids.shape[1],
                                               probs_at, stat_at, scores.data_ptr(), loss.data_ptr(), accuracy.data_ptr(), lse.data_ptr(),
                                               self.host.ptr(_HostFlags.ANSWERS), _stream_ptr(dev)))
        self.host.answers = True
        self.results = loss, accuracy, lse


class _DenseDocScores(torch.autograd.Function):
    """Per-document scores of a dense (B, N, h1, M*H) fp32 logits tensor: softmax of the chosen rows over all document
    slots, summed per document, averaged over heads and rows, divided by the temperature (losses.py:53-74).  The gradient
    of the gradient is that of the torch expressions.  ``with_loss``: made by the same launches, for an _InfoNCE that follows."""

    @staticmethod
    def forward(ctx, x, rows, M, H, temperature, with_loss=None):
        B, N, h1, _ = x.shape
        R = rows.shape[1]
        dev = x.device
        ctx.temperature, ctx.sizes = temperature, (R, B, N, h1, M, H, 1.0 / (temperature * N * R))
        with _lib.on_device(dev):
            probs = torch.empty((B, N, R, M - 2), dtype=torch.float32, device=dev)
            stat = torch.empty((B, N, R, 2), dtype=torch.float32, device=dev)
            scores = torch.empty((B, M - 2), dtype=torch.float32, device=dev)
            if with_loss is not None:
                with_loss.make(x, rows, ctx.sizes, probs.data_ptr(), stat.data_ptr(), scores)
            else:
                _lib.check(_lib.load().br_dense_doc_scores(x.data_ptr(), rows.data_ptr(), *ctx.sizes, probs.data_ptr(), stat.data_ptr(),
                                                           scores.data_ptr(), _stream_ptr(dev)))
        ctx.save_for_backward(x, rows, probs, stat)
        return scores

    @staticmethod
    def backward(ctx, g):
        x, rows, probs, stat = ctx.saved_tensors
        if torch.is_grad_enabled():              # create_graph
            B, M, H = x.shape[0], *ctx.sizes[4:6]
            dx, = torch.autograd.grad(_doc_scores_expression(x, rows, B, M, H, ctx.temperature), x, g, create_graph=True)
            return dx, None, None, None, None, None
        g = g.contiguous()
        with _lib.on_device(x.device):
            dx = torch.empty_like(x)
            _lib.check(_lib.load().br_dense_doc_scores_bwd(g.data_ptr(), x.data_ptr(), rows.data_ptr(), *ctx.sizes, probs.data_ptr(),
                                                           stat.data_ptr(), dx.data_ptr(), _stream_ptr(x.device)))
        return dx, None, None, None, None, None


class _InfoNCE(torch.autograd.Function):
    """Loss and accuracy of losses.py:80-93 on (B, docs) fp32 logits; ``host``: flags that are told of the answers; ``made``:
    what the launches that made the logits left (_LossWithScores)."""

    @staticmethod
    def forward(ctx, logits, answer_ids, host, made=None):
        dev = logits.device
        ctx.set_materialize_grads(False)         # (a launch for the accuracy's zeros)
        ctx.sizes = (*logits.shape, answer_ids.shape[1])
        if made is not None:
            loss, accuracy, lse = made
        else:
            with _lib.on_device(dev):
                loss, accuracy = torch.empty((), dtype=torch.float32, device=dev), torch.empty((), dtype=torch.float32, device=dev)
                lse = torch.empty((logits.shape[0], 2), dtype=torch.float32, device=dev)
                _lib.check(_lib.load().br_infonce_checked(logits.data_ptr(), answer_ids.data_ptr(), *ctx.sizes, loss.data_ptr(),
                                                          accuracy.data_ptr(), lse.data_ptr(),
                                                          host.ptr(_HostFlags.ANSWERS) if host is not None else None, _stream_ptr(dev)))
            if host is not None:
                host.answers = True
        ctx.mark_non_differentiable(accuracy)
        ctx.save_for_backward(logits, answer_ids, lse)
        return loss, accuracy

    @staticmethod
    def backward(ctx, g, _):
        if g is None:
            return None, None, None, None
        logits, answer_ids, lse = ctx.saved_tensors
        if torch.is_grad_enabled():
            loss, _ = _infonce_expression(logits, answer_ids.clamp(max=logits.shape[1]))
            dlogits, = torch.autograd.grad(loss, logits, g, create_graph=True)
            return dlogits, None, None, None
        with _lib.on_device(logits.device):
            dlogits = torch.empty_like(logits)
            _lib.check(_lib.load().br_infonce_bwd(g.data_ptr(), logits.data_ptr(), answer_ids.data_ptr(), lse.data_ptr(), *ctx.sizes,
                                                  dlogits.data_ptr(), _stream_ptr(logits.device)))
        return dlogits, None, None, None


class _RankingLoss(torch.autograd.Function):
    """_DenseDocScores and _InfoNCE as one node: (loss, accuracy), for calls that do not return the scores - where they are
    returned, the loss has to be a function of them: they may be hooked, retained or differentiated with respect to.  A training
    step's loss is mostly what its nodes cost the host: 350 us a step of two requests of 12 documents of 33 to 250 tokens with
    this one, 361 with the two."""

    @staticmethod
    def forward(ctx, x, rows, answer_ids, host, M, H, temperature):
        B, N, h1, _ = x.shape
        R, dev = rows.shape[1], x.device
        ctx.set_materialize_grads(False)
        ctx.temperature, ctx.sizes = temperature, (R, B, N, h1, M, H, 1.0 / (temperature * N * R))
        with _lib.on_device(dev):
            probs = torch.empty((B, N, R, M), dtype=torch.float32, device=dev)       # (N R probabilities and their two numbers, apart)
            scores = torch.empty((B, M - 2), dtype=torch.float32, device=dev)
            at = probs.data_ptr()
            joint = _LossWithScores(answer_ids, host)
            joint.make(x, rows, ctx.sizes, at, at + 4 * B * N * R * (M - 2), scores)
        loss, accuracy, lse = joint.results
        ctx.mark_non_differentiable(accuracy)
        ctx.save_for_backward(x, rows, answer_ids, probs, lse, scores)
        return loss, accuracy

    @staticmethod
    def backward(ctx, g, _):
        nothing = (None,) * 6
        if g is None:
            return None, *nothing
        x, rows, answer_ids, probs, lse, scores = ctx.saved_tensors
        R, B, N, _, M, H, _ = ctx.sizes
        if torch.is_grad_enabled():              # create_graph
            logits = _doc_scores_expression(x, rows, B, M, H, ctx.temperature)
            loss, _ = _infonce_expression(logits, answer_ids.clamp(max=M - 2))
            dx, = torch.autograd.grad(loss, x, g, create_graph=True)
            return dx, *nothing
        with _lib.on_device(x.device):
            dx = torch.empty_like(x)
            at = probs.data_ptr()
            _lib.check(_lib.load().br_ranking_loss_bwd(g.data_ptr(), None, x.data_ptr(), rows.data_ptr(), *ctx.sizes, answer_ids.data_ptr(),
                                                       answer_ids.shape[1], at, at + 4 * B * N * R * (M - 2), scores.data_ptr(), lse.data_ptr(),
                                                       dx.data_ptr(), _stream_ptr(x.device)))
        return dx, *nothing


def _doc_scores_expression(x: torch.Tensor, rows: torch.Tensor, B: int, M: int, H: int, temperature) -> torch.Tensor:
    # losses.py:53-74
    N = x.shape[1]
    x = x.take_along_dim(rows[:, None, :, None], dim=2)[..., H:-H]
    p = F.softmax(x, dim=-1).reshape(B, N, -1, M - 2, H)
    return p.mean(dim=(1, 2)).sum(dim=-1) / temperature


def _kernels_take_scores(x: torch.Tensor, rows: torch.Tensor, B: int, M: int, temperature) -> bool:
    # (the kernels' grids: a workgroup of 256 threads per head and row, a sequence per second index)
    return (x.is_cuda and _eager(x, rows) and x.dtype == torch.float32 and x.is_contiguous() and x.shape[0] == B and rows.device == x.device
            and rows.dtype == torch.int64 and rows.dim() == 2 and rows.shape[0] in (1, B) and rows.shape[1] > 0 and 3 <= M <= 4098
            and B < 1 << 16 and x.shape[1] * max(x.shape[2], rows.shape[1]) < 1 << 24 and x.numel() > 0
            and isinstance(temperature, (int, float)) and temperature != 0)


def _of_every_sequence(rows: torch.Tensor, B: int) -> torch.Tensor:
    return (rows if rows.shape[0] == B else rows.expand(B, -1)).contiguous()


def _kernels_take_answers(answer_ids: torch.Tensor, device: torch.device, B: int, docs: int) -> bool:
    return (answer_ids.device == device and answer_ids.dtype == torch.int64 and answer_ids.dim() == 2
            and answer_ids.shape[0] == B and answer_ids.is_contiguous() and 0 < B * docs < 1 << 30)


def _doc_scores_of_rows(x: torch.Tensor, rows: torch.Tensor, B: int, M: int, H: int, temperature) -> torch.Tensor:
    if _kernels_take_scores(x, rows, B, M, temperature):
        return _DenseDocScores.apply(x, _of_every_sequence(rows, B), M, H, float(temperature))
    return _doc_scores_expression(x, rows, B, M, H, temperature)


def _infonce_expression(logits: torch.Tensor, answer_ids: torch.Tensor):
    # losses.py:80-93
    B, num_docs = logits.shape
    pos_mask = torch.zeros(B, num_docs + 1, dtype=torch.bool, device=logits.device)
    pos_mask.scatter_(1, torch.where(answer_ids >= 0, answer_ids, num_docs), True)
    pos_mask = pos_mask[:, :-1]
    pos_lse = torch.logsumexp(logits.masked_fill(~pos_mask, float("-inf")), dim=1)
    all_lse = torch.logsumexp(logits, dim=1)
    loss = -(pos_lse - all_lse).mean()
    accuracy = pos_mask.gather(1, logits.argmax(dim=1, keepdim=True)).float().mean()
    return loss, accuracy


def _infonce(logits: torch.Tensor, answer_ids: torch.Tensor, return_logits: bool, host: _HostFlags | None = None):
    # An answer beyond the documents is refused: by the caller's reading of ``host``, or here (but not in a graph's capture,
    # which cannot wait: its loss and accuracy are then NaN).
    B, num_docs = logits.shape
    # (with host the call has asked _eager of its labels: what is left are these tensors' types)
    plain = type(logits) in _PLAIN and type(answer_ids) in _PLAIN and (host is not None or _eager())
    if (logits.is_cuda and plain and logits.dtype == torch.float32 and logits.is_contiguous()
            and _kernels_take_answers(answer_ids, logits.device, B, num_docs)):
        flags = host
        if host is None and not torch.cuda.is_current_stream_capturing():
            flags = _HostFlags(logits.device)
        loss, accuracy = _InfoNCE.apply(logits, answer_ids, flags)
        if host is None and flags is not None:
            flags.read()
    elif answer_ids.is_cuda:                     # (there scatter_ checks nothing and writes out of range)
        beyond = (answer_ids > num_docs).any()
        if plain and not torch.cuda.is_current_stream_capturing() and beyond:
            raise RuntimeError(_BEYOND)
        loss, accuracy = (x.masked_fill(beyond, float("nan")) for x in _infonce_expression(logits, answer_ids.clamp(max=num_docs)))
    else:
        loss, accuracy = _infonce_expression(logits, answer_ids)
    return (loss, accuracy, logits) if return_logits else (loss, accuracy)


def compute_auxiliary_attention_loss(
    attention_scores,
    labels: torch.Tensor,
    attention_mask: torch.Tensor,
    answer_ids: torch.Tensor | None = None,
    temperature: float = 0.05,
    return_logits=False,
    rows: torch.Tensor | None = None,
):
    """(B, M-2) per-document logits (and, with ``answer_ids``, the InfoNCE loss and accuracy).

    attention_scores: LastBlockScores handle or (B, N, h1, M*H) tensor; labels (B, M*H) with -100 on
    everything but the completion; attention_mask (B, M, H).  Follows losses.py:37-78: rows =
    {bracket-1, bracket}; softmax over all document tokens jointly; sum per document; mean over heads
    and the two rows; divide by temperature.  ``rows``: the result of ``bracket_rows(labels, h1)`` if the caller
    already has it (the tensor given to the model call as ``score_rows_hint``: the handle then holds the scores).
    """
    B, M, H = attention_mask.shape
    _, N, h1, MH = attention_scores.shape
    assert MH == M * H, "Attention scores last dimension must match M*H"
    handle = attention_scores if isinstance(attention_scores, LastBlockScores) else None
    found = pos = None
    if rows is None:
        guess = handle.speculated_rows() if handle is not None else None
        if guess is not None and guess.shape != (B, 2):
            guess = None
        if _BracketRows.takes(labels, h1, guess):
            # (the stand-alone score kernels take positions in the block, everything else the rows)
            stand_alone = handle is not None and handle.partials is None and not handle.needs_grad()
            found = _BracketRows(labels, h1, guess, H - h1 if stand_alone else None)
            rows, pos = found.rows, found.pos
        else:
            rows, match = bracket_rows(labels, h1, guess, return_match=True)     # (B, 2) in [0, h1)
            if match:
                rows = guess
    if handle is not None and handle.needs_grad():
        attention_scores, handle = handle.dense(), None      # training: the differentiable logits tensor
    if pos is not None:
        logits = handle.doc_scores_window(rows, temperature=temperature, pos=pos)
        found.check()                                        # (a row that is not there reads nothing: everything is enqueued first)
    elif handle is not None:
        if found is not None and found.check():
            rows = guess                                     # the attention call's own guess holds: its scores are these rows'
        logits = handle.doc_scores_window(rows, temperature=temperature)
    elif (found is not None and answer_ids is not None and type(answer_ids) in _PLAIN and _kernels_take_scores(attention_scores, rows, B, M, temperature)
          and _kernels_take_answers(answer_ids, attention_scores.device, B, M - 2)):
        rows = _of_every_sequence(rows, B)
        if return_logits:
            joint = _LossWithScores(answer_ids, found)
            logits = _DenseDocScores.apply(attention_scores, rows, M, H, float(temperature), joint)
            result = (*_InfoNCE.apply(logits, answer_ids, None, joint.results), logits)
        else:
            result = _RankingLoss.apply(attention_scores, rows, answer_ids, found, M, H, float(temperature))
        found.check()
        return result
    else:
        logits = _doc_scores_of_rows(attention_scores, rows, B, M, H, temperature)
        if found is not None:
            result = logits if answer_ids is None else _infonce(logits, answer_ids, return_logits, found)
            found.check()                                    # (everything that takes the rows is enqueued by now)
            assert answer_ids is not None or return_logits, "If answer_ids is None, return_logits must be True."
            return result
    if answer_ids is None:
        assert return_logits, "If answer_ids is None, return_logits must be True."
        return logits
    return _infonce(logits, answer_ids, return_logits)


def rank_documents(logits: torch.Tensor, k: int = 10) -> torch.Tensor:
    """Top-k document indices per sequence, as scripts/eval_attn.py:150-151 takes them."""
    return torch.topk(logits, k=min(k, logits.shape[-1]), dim=-1).indices
