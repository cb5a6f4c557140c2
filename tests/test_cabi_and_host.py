"""CPU-side checks: the C-ABI library loads and exports every symbol the header declares, pure host
entry points behave, the Python hooks keep the reference's error conventions, and the synthetic layout
follows the reference's collate rules.  No kernel is launched here."""
import ctypes
import os
import re
import threading

import numpy as np
import pytest
import torch

import blockrank_amd as br
from blockrank_amd import _lib, attention, synthetic

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "blockrank_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(br_[a-z_0-9]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = declared_symbols()
    assert len(names) >= 10
    for n in names:
        assert hasattr(lib, n), f"{n} declared in include/blockrank_hip.h but not exported"
    assert sorted(_lib.SIGNATURES) == names, "ctypes signatures and header are out of step"
    assert lib.br_version() >= 100
    assert lib.br_last_error() == b""


def test_pure_host_entry_points():
    lib = _lib.load()
    assert lib.br_tile_tokens(32, 8) == 32        # 4 heads x 32 tokens per workgroup
    assert lib.br_tile_tokens(28, 4) == 32        # 7 heads x 32 tokens
    assert lib.br_tile_tokens(8, 8) == 128        # 1 head x 128 tokens
    assert lib.br_tile_tokens(6, 2) == 64
    assert lib.br_tile_tokens(7, 2) == 0          # not a whole number of query heads per kv head
    assert lib.br_plan_ints(4, 22, 160, 32, 8) > 4 * 22 * 5 * 8
    assert lib.br_plan_ints(0, 22, 160, 32, 8) == 0
    # the split partials' pool follows the head layout and the device's compute units, not the batch (0: no device here)
    ws = lib.br_prefill_workspace_bytes(4, 32, 8, 128)
    assert ws == lib.br_prefill_workspace_bytes(64, 32, 8, 128)
    assert ws == 0 or 4 << 20 < ws < 32 << 20
    assert lib.br_doc_scores_workspace_bytes(4, 32, 22, 2) == 4 * 32 * 2 * 20 * 2 * 4
    assert ws == 0 or lib.br_prefill_fp8qk_workspace_bytes(4, 32, 8, 128, 22, 4 * 3520) > ws
    # backward: fp32 sums of the query block's dQ rows and of the prefix keys' dK / dV, rounded up to 256 bytes, then one
    # float per token slot and query head (delta)
    assert lib.br_prefill_bwd_workspace_bytes(4, 32, 8, 160, 128, 4 * 3520) == 4 * (32 + 16) * 160 * 128 * 4 + 4 * 3520 * 32 * 4
    assert lib.br_prefill_bwd_workspace_bytes(0, 32, 8, 160, 128, 10) == 0
    # ... with its counters where there is a device whose compute units decide their form
    full = lib.br_prefill_bwd_full_workspace_bytes(4, 32, 8, 22, 160, 128, 4 * 3520)
    assert full == 0 or full == 4 * (32 + 16) * 160 * 128 * 4 + 4 * 3520 * 32 * 4 + (17 + 4 * 22 * 8) * 128
    assert lib.br_prefill_bwd_full_workspace_bytes(4, 32, 8, 22, 160, 96, 4 * 3520) == 0
    assert lib.br_prefill_bwd_launches(4, 32, 8, 22, 160, 128, 4 * 3520, 1000) == 0
    rc = lib.br_prefill_bwd(None, None, None, None, None, None, None, 1, 4, 2, 3, 8, 96, None, None, None, None, None, None,
                            None, None, None, None, None, None, 1.0, 24, None, 0, None)
    assert rc == _lib.BR_ERR_ARG and b"head dim" in lib.br_last_error()
    # the entry point that allocates nothing refuses a request beyond its built-in scratch, before any device call
    # (without a device the size of the request cannot be worked out: that is refused as well)
    assert lib.br_prefill_noalloc_max_workspace_bytes() == 32 << 20
    rc = lib.br_prefill_fwd_noalloc(None, None, None, None, None, 1, 1024, 1024, 3, 64, 128, None, None, None, None, 1.0, 1, None)
    assert (rc == _lib.BR_ERR_SPACE and b"built-in scratch" in lib.br_last_error()) or (rc == _lib.BR_ERR_HIP and b"device" in lib.br_last_error())
    # argument errors come back as codes with a message, before anything touches a device
    rc = lib.br_prefill_fwd(None, None, None, None, None, 1, 4, 2, 3, 8, 96, None, None, None, None, 1.0, 1, None, 0, None)
    assert rc == _lib.BR_ERR_ARG and b"head dim" in lib.br_last_error()
    rc = lib.br_plan_build(None, 1, 3, 8, 4, 2, None, 0, None)
    assert rc == _lib.BR_ERR_ARG and b"mask" in lib.br_last_error()
    with pytest.raises(AssertionError):
        _lib.check(rc)


@pytest.mark.parametrize("H", [8, 1])
def test_token_strides_beyond_a_tile_offset_are_refused(H):
    """The 16-bit kernels' 32-bit byte offsets hold 64 rows of 2^24 elements, whatever a block has of them; decided before
    anything touches a device."""
    lib = _lib.load()
    some = ctypes.c_void_p(4096)                  # (never dereferenced)
    dense, far = _lib._I64x3(0, 64, 512), _lib._I64x3(0, 64, (1 << 24) + 8)
    for at in range(4):
        strides = [far if i == at else dense for i in range(4)]
        rc = lib.br_prefill_fwd(some, some, some, some, some, 1, 4, 2, 3, H, 64, *strides, 1.0, _lib.BR_DTYPE_BF16, some, 1 << 40, None)
        assert rc == _lib.BR_ERR_ARG and b"token strides" in lib.br_last_error()
    for at in range(5):
        strides = [far if i == at else dense for i in range(5)]
        rc = lib.br_prefill_bwd(*[some] * 7, 1, 4, 2, 3, H, 64, *strides, _lib._I64x3(12 * H, 3 * H, 1), some, some, some, dense, dense, dense, 1.0,
                                3 * H, some, 1 << 40, None)
        assert rc == _lib.BR_ERR_ARG and b"token strides" in lib.br_last_error()


def test_switches_are_read_from_the_environment_as_it_is_now(monkeypatch):
    name = "BLOCKRANK_AMD_DENSE_SCORES"
    monkeypatch.delenv(name, raising=False)
    assert not attention._env_flag(name)
    for value, on in (("1", True), ("0", False), ("", False), ("False", False), ("yes", True)):
        monkeypatch.setenv(name, value)
        assert attention._env_flag(name) is on
    monkeypatch.setattr(os, "environ", {})               # a mapping in its place
    assert not attention._env_flag(name)
    monkeypatch.setattr(os, "environ", {name: "1"})
    assert attention._env_flag(name)
    monkeypatch.undo()
    monkeypatch.delenv(name, raising=False)
    assert not attention._env_flag(name)
    monkeypatch.setattr(os, "environ", {name: "1"})      # (the variable itself is not set)
    assert attention._env_flag(name)


def test_hooks_fail_loudly_without_gpu_tensors():
    valid = torch.ones(1, 3, 8, dtype=torch.bool)
    with pytest.raises(RuntimeError, match="GPU"):
        br.blockrank_attention_mask(batch_size=1, attention_mask=valid)
    with pytest.raises(AssertionError):
        br.blockrank_attention_mask(batch_size=1, attention_mask=None)
    with pytest.raises(AssertionError):
        br.blockrank_attention_forward(None, torch.zeros(1, 2, 24, 64), torch.zeros(1, 2, 24, 64), torch.zeros(1, 2, 24, 64), None, 0.1)


def test_no_fallback_when_library_is_missing(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "libblockrank_hip.so")
    with pytest.raises(_lib.BlockRankLibraryError, match="no CPU or PyTorch fallback"):
        _lib.load()


def test_registration_uses_reference_names():
    from transformers import AttentionInterface, AttentionMaskInterface
    br.register_blockrank_attention()
    br.register_triton_blockrank_attention()
    for name in br.attention.STD_IMPL_NAMES + br.attention.TRITON_IMPL_NAMES:
        assert AttentionInterface()[name] is br.blockrank_attention_forward
        assert AttentionMaskInterface()[name] is br.blockrank_attention_mask
    # a model config accepts the name
    from transformers import MistralConfig, MistralForCausalLM
    cfg = MistralConfig(vocab_size=64, hidden_size=64, intermediate_size=64, num_hidden_layers=1, num_attention_heads=2,
                        num_key_value_heads=1, head_dim=64)
    model = MistralForCausalLM(cfg)
    model.set_attn_implementation("triton_blockrank")
    assert model.config._attn_implementation == "triton_blockrank"


def test_layout_follows_collate_rules():
    lay = synthetic.make_layout([[3, 5, 2, 4]])
    assert lay.H == 16 and lay.S == 64                       # padded to a multiple of 16
    v = lay.valid[0]
    assert v[0].tolist() == [False] * 13 + [True] * 3         # left padding
    pos = lay.position_ids.view(1, 4, 16)[0]
    assert pos[0, -3:].tolist() == [0, 1, 2]                  # prefix 0..p-1
    assert pos[1, -5:].tolist() == [3, 4, 5, 6, 7]            # every document restarts at p
    assert pos[2, -2:].tolist() == [3, 4]
    assert pos[3, -4:].tolist() == [16384, 16385, 16386, 16387]
    assert (pos[~v] == 0).all()
    assert (lay.labels[0, :-1] == -100).all() and lay.labels[0, -1] != -100
    assert lay.unmasked_pairs() == 6 + (5 * 3 + 15) + (2 * 3 + 3) + 4 * 10 + 10


def test_baseline_pair_counts():
    assert synthetic.uniform_layout(1, 32, 8, 64, 16).unmasked_pairs() == 42392
    assert synthetic.uniform_layout(1, 64, 20, 160, 32).unmasked_pairs() == 569456


def test_bracket_rows_match_reference_rule():
    labels = torch.full((2, 48), -100)
    labels[0, -1] = 5
    labels[1, -4:] = 5
    rows = br.losses.bracket_rows(labels, 16)
    assert rows.tolist() == [[14, 15], [11, 12]]
    labels[1, -16:] = 5
    with pytest.raises(AssertionError):
        br.losses.bracket_rows(labels, 16)


def test_tensor_path_of_loss_matches_oracle_on_cpu():
    from oracle import blockrank_oracle as orc
    rng = np.random.default_rng(0)
    B, N, h1, M, H = 2, 3, 8, 4, 8
    s = torch.as_tensor(rng.normal(size=(B, N, h1, M * H)))
    valid = torch.ones(B, M, H, dtype=torch.bool)
    labels = torch.full((B, M * H), -100)
    labels[:, -1] = 1
    got = br.compute_auxiliary_attention_loss(s, labels, valid, answer_ids=None, return_logits=True)
    want = orc.doc_scores_from_logits(s.numpy(), labels.numpy(), valid.numpy(), 0.05)
    np.testing.assert_allclose(got.numpy(), want, rtol=1e-10)


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=300)
    assert r.returncode != 0 and "one GPU" in (r.stderr + r.stdout)


def test_scores_handle_is_a_tensor_to_strangers(monkeypatch):
    """LastBlockScores in place of the reference's s_last tensor: torch functions, methods and indexing reach the
    logits (here a stub of the logits kernel, so that the protocol itself is checked without a GPU)."""
    import types
    from blockrank_amd import attention as att
    B, Nq, R, M, H, D = 2, 4, 16, 5, 32, 64
    g = torch.Generator().manual_seed(0)
    full = torch.randn(B, Nq, H, M * H, generator=g)                       # logits of every query-block position

    def fake_logits(query, key, bm, rows, scaling, neg=None):
        return full.take_along_dim(rows.long()[:, None, :, None], dim=2)

    monkeypatch.setattr(att, "last_block_logits", fake_logits)
    bm = types.SimpleNamespace(B=B, M=M, H=H)
    h = att.LastBlockScores(torch.zeros(B, Nq, M * H, D), torch.zeros(B, 2, M * H, D), bm, 0.125, R)
    want = full[:, :, H - R:]
    idx = torch.tensor([[14, 15], [3, 4]])[:, None, :, None]
    got = h.take_along_dim(idx, dim=2)
    assert h._dense is None and torch.equal(got, want.take_along_dim(idx, dim=2))
    assert torch.equal(h.take_along_dim(torch.tensor([[-1, -2], [0, 1]])[:, None, :, None], dim=2),
                       want.take_along_dim(torch.tensor([[15, 14], [0, 1]])[:, None, :, None], dim=2))
    outside = torch.tensor([[16, 33], [-17, 5]])[:, None, :, None]
    assert torch.equal(h.take_along_dim(outside, dim=2), want.take_along_dim(outside, dim=2))
    assert tuple(h.shape) == (B, Nq, R, M * H) and h.dim() == 4 and h.size(-1) == M * H and len(h) == B
    assert torch.equal(h[..., H:-H], want[..., H:-H])
    assert torch.equal(torch.softmax(h, dim=-1), torch.softmax(want, dim=-1))
    assert torch.equal(torch.nn.functional.softmax(h[..., H:-H], dim=-1), torch.softmax(want[..., H:-H], dim=-1))
    assert torch.equal(h * 2, want * 2) and torch.equal(h.double(), want.double()) and torch.allclose(h.mean(dim=(1, 2)), want.mean(dim=(1, 2)), atol=1e-6)
    with pytest.raises(AttributeError):
        h.no_such_attribute


@pytest.mark.parametrize("waits", [True, False])
def test_flags_a_kernel_may_still_write_are_not_freed(monkeypatch, waits):
    """An exception between the launch that is given the pinned flags and the read that waits for it: they stay until the
    device is idle, or for good where that cannot be waited for."""
    from blockrank_amd import losses
    waited, empty = [], torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))

    def synchronize(device):
        waited.append(device)
        if not waits:
            raise RuntimeError("operation not permitted when stream is capturing")

    monkeypatch.setattr(torch.cuda, "synchronize", synchronize)
    host = losses._HostFlags("cuda:0")
    del host
    assert waited == []                          # nothing was launched with them
    host = losses._HostFlags("cuda:0")
    at = host.ptr()
    del host
    assert waited == ["cuda:0"]
    kept = [f.data_ptr() for f in losses._NEVER_FREED]
    assert (at in kept) == (not waits)


def test_wait_for_written_flags_is_bounded():
    lib = _lib.load()
    flags = (ctypes.c_int32 * 3)(-1, 0, 1)
    at = ctypes.addressof(flags)
    assert lib.br_wait_written(at + 4, 2, 0) == 1 and lib.br_wait_written(at, 0, 0) == 1
    assert lib.br_wait_written(at, 3, 200) == 0 and lib.br_wait_written(None, 1, 0) == 0
    late = threading.Timer(0.02, lambda: flags.__setitem__(0, 0))
    late.start()
    assert lib.br_wait_written(at, 3, 10_000_000) == 1 and list(flags) == [0, 0, 1]
    late.join()
