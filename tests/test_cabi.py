"""CPU-side checks of the boundary: the shared library loads, exports every symbol that
include/verl_amd.h declares, answers its size queries, and the host wrappers refuse to run
without a GPU instead of falling back."""
import ctypes
import os
import pathlib
import re

import numpy as np
import pytest
import torch

from verl_amd import _cabi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "verl_amd.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vamd_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_cabi.lib_path()):
        from verl_amd.csrc.build import build
        build(verbose=False)
    return _cabi.load_library()


def test_every_declared_symbol_is_exported_and_bound(lib):
    declared = _declared_symbols()
    assert len(declared) >= 20
    for name in declared:
        assert hasattr(lib, name), f"{name} declared in include/verl_amd.h but not exported"
    assert sorted(_cabi.SIGNATURES) == declared, "ctypes prototypes and header disagree"
    assert lib.vamd_abi_version() == _cabi.ABI_VERSION
    header = open(os.path.join(os.path.dirname(__file__), "..", "include", "verl_amd.h")).read()
    assert f"#define VAMD_ABI_VERSION {_cabi.ABI_VERSION}\n" in header


def test_documents_state_the_version_of_the_header():
    """A binding is written from them: the version, and that each names the two calls that add to a gradient."""
    root = pathlib.Path(ROOT)
    stated = [(p.name, int(n)) for p in root.glob("*.md")
              for n in re.findall(r"`VAMD_ABI_VERSION` (?:=|is) (\d+)", p.read_text())]
    assert stated and all(n == _cabi.ABI_VERSION for _, n in stated), stated
    for name in {doc for doc, _ in stated}:
        text = (root / name).read_text()
        assert "vamd_row_softmax_backward_add" in text and "vamd_scale_rows_add" in text, name


def test_stale_binaries_are_told_to_be_rebuilt(monkeypatch):
    """A library from before an entry point was added, and a host module linked with such a library."""
    import types
    older = lambda: _cabi.ABI_VERSION - 1
    with monkeypatch.context() as m:
        m.setattr(ctypes, "CDLL", lambda path: types.SimpleNamespace(vamd_abi_version=older))
        with pytest.raises(RuntimeError, match="rebuild"):
            _cabi.load_library()
    current = lambda: _cabi.ABI_VERSION
    for compiled, linked in ((older, current), (current, older)):
        module = types.SimpleNamespace(abi_version=compiled, library_abi_version=linked)
        monkeypatch.setattr(_cabi, "_ops", None)
        monkeypatch.setattr(_cabi.importlib.util, "module_from_spec", lambda spec: module)
        monkeypatch.setattr(_cabi.importlib.util, "spec_from_file_location",
                            lambda *a: types.SimpleNamespace(loader=types.SimpleNamespace(exec_module=lambda m: None)))
        with pytest.raises(RuntimeError, match="rebuild"):
            _cabi.ops()


def test_workspace_queries(lib):
    assert lib.vamd_lce_forward_workspace_bytes(16384, 3584, 152064) > 0
    assert lib.vamd_lce_forward_workspace_bytes(0, 3584, 152064) == 0
    n, h, v = 16384, 3584, 152064
    full = lib.vamd_lce_backward_workspace_bytes(n, h, v, 0)
    assert full < 1 << 30                                         # d_logits panel + fp32 d_hidden accumulator
    one = lib.vamd_lce_backward_workspace_bytes(256, 128, 1024, 0)
    assert one == 256 * (1024 + 128) * 2                          # a single padded panel, no accumulator
    # single-launch reductions: arrival counters (VAMD_TICKET_BYTES) + one record of doubles per 4096-column chunk
    # + 64 records for the share totals of the two-level sum
    ticket = 16640
    assert lib.vamd_masked_moments_workspace_bytes(512, 4096) == ticket + (512 + 64) * 4 * 8
    assert lib.vamd_policy_loss_workspace_bytes(512, 4097) == ticket + (512 * 2 + 64) * 5 * 8
    assert lib.vamd_gae_workspace_bytes(512, 4096) >= ticket + 512 * 4 * 8


def test_pieces_of_a_call_over_some_of_the_tokens(lib):
    """As the workspace query shows them: cut like the whole call where that has one vocabulary chunk, on their own where
    it has several; a planned count below the token count (which the call refuses) is answered too."""
    subset, whole = lib.vamd_lce_backward_subset_workspace_bytes, lib.vamd_lce_backward_workspace_bytes

    def pieces(n, planned, h, v=152064):
        panel = -(-n // 256) * 256 * (v + 128) * 2
        return (subset(n, planned, h, v, 0) - panel) // (n * h * 4)

    assert pieces(200, 1500, 3584) == pieces(1500, 1500, 3584) != pieces(200, 200, 3584)
    for n, planned, h in ((1000, 11290, 3584), (1300, 8000, 896), (200, 2000, 3584)):
        assert subset(n, planned, h, 152064, 0) == whole(n, h, 152064, 0) and pieces(n, planned, h) > 1
    for planned in (0, -5, 1, 99):
        assert subset(100, planned, 3584, 152064, 0) == whole(100, 3584, 152064, 0)


def test_a_call_over_more_tokens_than_planned_is_refused(lib):
    at = 4096                                                # never read: the call is refused on the host
    for planned in (99, 0, -1):
        rc = lib.vamd_lce_backward_subset(at, at, at, 100, planned, 128, 256, 1.0, at, at, None, None, 0.0, None, at, at,
                                          _cabi.DW_STORE, None, 0, None, 0, None)
        assert rc == -1 and b"tokens are no part of" in lib.vamd_last_error()


def test_unaligned_16_bit_row_gradients_are_refused(lib):
    at = 4096                                                # never read: the call is refused on the host
    for d_logprobs, d_entropy in ((at + 1, None), (at, at + 1)):
        rc = lib.vamd_row_softmax_backward_as(at, 1, 4, 256, 256, at, at, at, d_logprobs, d_entropy, 1, at, 128, None)
        assert rc == -1 and b"2-byte aligned" in lib.vamd_last_error()


def test_head_size_queries_are_asked_on_the_tensors_device(monkeypatch):
    """The head's workspaces depend on the compute units of the current device, so the query belongs inside the guard that
    makes the tensors' device current for the call itself (devices need not be alike)."""
    import contextlib

    from verl_amd.utils.kernel import linear_cross_entropy as K
    current, asked = ["another"], []

    @contextlib.contextmanager
    def guard(device):
        current.append(device)
        yield
        current.pop()

    class Library:
        def __getattr__(self, name):
            def call(*args):
                asked.append((name, current[-1]))
                return 4096 if name.endswith("_workspace_bytes") else 0
            return call

    monkeypatch.setattr(_cabi, "lib", Library)
    monkeypatch.setattr(_cabi, "device_guard", guard)
    monkeypatch.setattr(_cabi, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(K, "_check_inputs", lambda *tensors: None)
    hidden, weight = torch.zeros(5, 128, dtype=torch.bfloat16), torch.zeros(16, 128, dtype=torch.bfloat16)
    labels = torch.zeros(5, dtype=torch.int64)
    _, _, lse, mean_z = K.efficient_entropy_forward(hidden, weight, labels)
    K.efficient_entropy_backward(None, None, hidden, weight, labels, lse, mean_z)
    assert len(asked) == 4 and all(device == hidden.device for _, device in asked), asked


def test_a_long_backward_pass_looks_at_its_own_gradients_whatever_ran_before(monkeypatch):
    """Only short calls are spared the look after one that found every token active, and only with the same head."""
    from verl_amd.utils.kernel import linear_cross_entropy as K
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.delenv("VAMD_LCE_SKIP_ZERO_GRAD_TOKENS", raising=False)
    monkeypatch.setattr(K, "_ACTIVE_PROBE", {"rest": 0, "head": None})
    small, other, large = (1024, 128), (1024, 256), (152064, 3584)
    dense, masked = torch.ones(2000), torch.cat((torch.zeros(1600), torch.ones(400)))
    look = lambda g, head: K.active_token_index(g, None, 2000, head)
    for _ in range(2):                                       # the second time round starts with the first one's state
        assert look(dense, small) is None
        for _ in range(3):
            assert look(masked, large).tolist() == list(range(1600, 2000))
            assert look(masked, other).numel() == 400
        assert look(dense, large) is None
        assert look(masked, other).numel() == 400
        for _ in range(K._ACTIVE_PROBE_REST):
            assert look(masked, small) is None
        assert look(masked, small).numel() == 400


def test_argument_errors_are_reported_without_touching_the_gpu(lib):
    rc = lib.vamd_lce_forward(None, None, None, 16, 100, 128, 1.0, None, None, None, None, None, None, None, 0, None)
    assert rc == -1 and b"multiple of 128" in lib.vamd_last_error()
    rc = lib.vamd_policy_loss_forward(None, None, None, None, 0, None, 4, 4, 0.2, 0.2, 3.0, 0, 1.0, -1.0, -1.0, -1.0,
                                      None, None, None, None, 0, None)
    assert rc == -1 and b"null pointer" in lib.vamd_last_error()


@pytest.mark.skipif(torch.cuda.is_available(), reason="needs a machine without a GPU")
def test_no_cpu_fallback():
    from verl_amd.trainer.ppo import core_algos as CA
    from verl_amd.utils import torch_functional as F
    x = torch.ones(2, 4)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        F.masked_mean(x, x)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        CA.compute_gae_advantage_return(x, x, x, 1.0, 1.0)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        CA.agg_loss(x, x, "token-mean")


def test_missing_library_fails_loudly(tmp_path):
    with pytest.raises(RuntimeError, match="is missing"):
        _cabi.load_library(str(tmp_path / "libverl_amd.so"))


def test_registries_and_host_logic_without_gpu():
    from verl_amd.trainer.ppo import core_algos as CA
    from verl_amd.utils.groupwise import as_torch_index, contiguous_group_ids
    from verl_amd.utils.kernel.linear_cross_entropy import get_entropy_reduction_enum_number
    assert CA.get_adv_estimator_fn("gae") is CA.compute_gae_advantage_return
    assert CA.get_adv_estimator_fn(CA.AdvantageEstimator.GRPO) is CA.compute_grpo_outcome_advantage
    assert CA.get_policy_loss_fn("vanilla") is CA.compute_policy_loss_vanilla
    with pytest.raises(ValueError, match="Unsupported loss mode"):
        CA.get_policy_loss_fn("gspo-not-here")
    with pytest.raises(ValueError, match="Unknown advantage estimator"):
        CA.get_adv_estimator_fn("nope")
    with pytest.raises(ValueError, match="already been registered"):
        CA.register_adv_est("grpo")(lambda: None)
    with pytest.raises(ValueError, match="Invalid loss_agg_mode"):
        CA.agg_loss(torch.ones(1, 1), torch.ones(1, 1), "bad-mode")
    assert [get_entropy_reduction_enum_number(r) for r in ("none", "sum", "mean")] == [0, 1, 2]
    with pytest.raises(ValueError, match="Invalid reduction"):
        get_entropy_reduction_enum_number("max")
    g = as_torch_index(["a", "b", "a", "c", "0042", 42])
    assert g.tolist()[4] != g.tolist()[5] and len(torch.unique(g)) == 5
    assert as_torch_index(["5", "6", "5"]).tolist() == [5, 6, 5]
    assert as_torch_index(torch.tensor([1.0, 2.0, 1.0])).tolist() == [1, 2, 1]
    assert as_torch_index(np.array([3, 3, 7])).tolist() == [3, 3, 7]
    assert as_torch_index(np.array([True, False])).tolist() == [1, 0]
    assert as_torch_index(np.array([1.5, 2.5, 1.5])).tolist() == [1, 2, 1]          # numpy floats: integer cast
    t = as_torch_index(torch.tensor([1.5, 2.5, 1.5]))                               # tensor floats: opaque labels
    assert t.tolist() == [0, 1, 0]
    ids, G = contiguous_group_ids([10, 10, 7, 99])                                  # a list: ids by first appearance
    assert G == 3 and ids.tolist() == [0, 0, 1, 2]
    ids, G = contiguous_group_ids(np.array([10, 10, 7, 99]))                        # integers: ids by sorted label
    assert G == 3 and ids.tolist() == [1, 1, 0, 2]
    ids, G = contiguous_group_ids(torch.tensor([[3, 3], [1, 3]]))
    assert G == 2 and ids.tolist() == [1, 1, 0, 1]
    ids, G = contiguous_group_ids(np.array(["u-1", "u-2", "u-1", 5, 5.0], dtype=object))
    assert G == 3 and ids.tolist() == [0, 1, 0, 2, 2]                               # Python equality: 5 == 5.0
    ids, G = contiguous_group_ids(["0042", 42, "x"])
    assert G == 3
    ids, G = contiguous_group_ids(["0042", "42", "7"], vectorized=True)             # numeric strings coincide there
    assert G == 2 and ids.tolist() == [1, 1, 0]                                     # integers again: by sorted label


def test_backward_rejects_operands_beyond_32_bit_offsets(lib):
    """The check runs before any GPU call: dummy non-null pointers are never dereferenced."""
    p = ctypes.c_void_p(256)
    rc = lib.vamd_lce_backward(p, p, p, 700000, 3584, 1024, 1.0, p, p, None, None, 0.0, None, p, p, 0, None, 0, p, 1 << 40, None)
    assert rc == -1 and b"4 GiB" in lib.vamd_last_error()
    # fp32 accumulation of the weight gradient needs its buffer; an unknown mode is refused
    rc = lib.vamd_lce_backward(p, p, p, 256, 128, 1024, 1.0, p, p, None, None, 0.0, None, p, None, 3, None, 0, p, 1 << 40, None)
    assert rc == -1 and b"d_weight_acc32" in lib.vamd_last_error()
    rc = lib.vamd_lce_backward(p, p, p, 256, 128, 1024, 1.0, p, p, None, None, 0.0, None, p, p, 7, None, 0, p, 1 << 40, None)
    assert rc == -1 and b"d_weight_mode" in lib.vamd_last_error()
    # a vocabulary that is not a multiple of 8 is served, but not together with a logits cache
    rc = lib.vamd_lce_forward(p, p, p, 256, 128, 1001, 1.0, p, p, p, p, p, None, p, 1 << 30, None)
    assert rc == -1 and b"multiple of 8" in lib.vamd_last_error()


def test_bench_refuses_more_than_one_gpu():
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert res.returncode != 0 and "one GPU" in res.stderr and res.stdout.strip() == ""


def test_static_forward_refuses_sizes_beyond_its_buffer_before_any_gpu_call(lib):
    # the pointers are never dereferenced: the size check precedes every HIP call
    rc = lib.vamd_lce_forward_static(1, 1, 1, 65536 + 1, 128, 256, 1.0, 1, 1, 1, 1, None, None)
    assert rc == -1 and b"at most 65536 tokens" in lib.vamd_last_error()


def test_as_torch_index_agrees_with_the_oracle_restatement():
    """The product's label handling is written differently from the oracle's line-by-line restatement of
    verl/utils/groupwise.py:91-160; both must give the same ids on every kind of label."""
    import uuid

    from oracle import advantages as A
    from verl_amd.utils.groupwise import as_torch_index
    rng = np.random.default_rng(0)
    uuids = [str(uuid.UUID(int=int(x))) for x in rng.integers(0, 2**62, 9)]
    cases = [
        torch.tensor([3, 1, 3, 2]), torch.tensor([3, 1, 3], dtype=torch.int32), torch.tensor([True, False, True]),
        torch.tensor([1.0, 2.0, 1.0]), torch.tensor([1.0, 2.0000001, 1.0]), torch.tensor([0.5, 1.5, 0.5]),
        torch.tensor([1.0, 2.0], dtype=torch.bfloat16), torch.tensor([[1, 2], [2, 1]]),
        np.array([3, 3, 7]), np.array([1.0, 2.0, 1.0]), np.array([1.5, 2.5, 1.5]), np.array([True, False]),
        np.array(["5", "6", "5"]), np.array(uuids * 2, dtype=object), ["a", "b", "a", "c", "0042", 42],
        ["5", "6", "5"], [3, 1, 3], (1.0, 2.0), np.array([[1, 2], [2, 1]]), [("a", 1), ("b", 2), ("a", 1)],
    ]
    for case in cases:
        want = A.as_torch_index(case)
        got = as_torch_index(case)
        assert got.dtype == torch.long and got.dim() == 1
        assert torch.equal(got, want.cpu()), f"{case!r}: {got.tolist()} vs {want.tolist()}"


def test_free_memory_that_may_hold_the_logits(monkeypatch):
    """What the device has free plus what torch's allocator holds for no tensor, within the process's memory fraction;
    nothing where another allocator does not say."""
    from verl_amd.utils.kernel import linear_cross_entropy as K
    stats = {"reserved_bytes": {"all": {"current": 50}}, "allocated_bytes": {"all": {"current": 30}}}
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (100, 1000))
    monkeypatch.setattr(torch.cuda, "memory_stats_as_nested_dict", lambda device: stats)
    monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda device: 1.0)
    assert K._free_device_bytes("cuda:0") == 120
    monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda device: 0.1)
    assert K._free_device_bytes("cuda:0") == 70
    monkeypatch.setattr(torch.cuda, "memory_stats_as_nested_dict", lambda device: {})
    assert K._free_device_bytes("cuda:0") == 0

    def refuse(device):
        raise RuntimeError("no such query")
    monkeypatch.setattr(torch.cuda, "mem_get_info", refuse)
    assert K._free_device_bytes("cuda:0") == 0


@pytest.mark.parametrize("name,at", [(name, at) for name, count in (("policy", 4), ("value", 4), ("kl", 3), ("agg", 2))
                                     for at in range(count)])
def test_losses_refuse_a_tangent_on_any_input(name, at):
    """A dual tensor needs no ``requires_grad`` and carries its tangent under ``no_grad`` too; a loss returned without one
    would read as a derivative of zero.  (Refused before a device is looked for.)"""
    import torch.autograd.forward_ad as fwAD
    from verl_amd.trainer.ppo import core_algos as CA
    count, fn = {"policy": (4, lambda x, old, adv, mask: CA.compute_policy_loss(old, x, adv, mask, 0.2)),
                 "value": (4, lambda v, ret, val, mask: CA.compute_value_loss(v, ret, val, mask, 0.5)),
                 "kl": (3, CA.compute_kl_loss), "agg": (2, lambda x, mask: CA.agg_loss(x, mask, "token-mean"))}[name]
    for grad_mode in (True, False):
        with fwAD.dual_level(), torch.set_grad_enabled(grad_mode):
            inputs = [torch.ones(2, 8) for _ in range(count)]
            inputs[at] = fwAD.make_dual(inputs[at], torch.ones(2, 8))
            with pytest.raises(NotImplementedError, match="forward mode"):
                fn(*inputs)


def test_group_ids_of_an_object_array_that_is_refilled():
    """The kept results are found by the addresses of the label objects.  Refilling a two-entry array comes back to the
    same three addresses every third time, here with equal labels where there were different ones."""
    from verl_amd.trainer.ppo.core_algos import _group_ids_on_device
    index = np.empty(2, dtype=object)
    for i in range(60):
        for k in range(2):
            index[k] = f"prompt-{(i if i % 2 else 2 * i + k) + 1000}".ljust(300)   # a size nothing else here has
        ids, groups = _group_ids_on_device(index, False, torch.device("cpu"))
        assert groups == (1 if i % 2 else 2) and ids.tolist() == [0, groups - 1], (i, ids, groups)


def test_group_ids_from_several_threads():
    """Threads that push each other's results out of the kept ones."""
    import sys
    import threading
    from verl_amd.trainer.ppo.core_algos import _group_ids_on_device
    wrong, interval = [], sys.getswitchinterval()

    def work(k):
        try:
            for i in range(400):
                ids, groups = _group_ids_on_device(np.array([0, (k + i) % 12, 0]), False, torch.device("cpu"))
                if groups != (1 if (k + i) % 12 == 0 else 2):
                    wrong.append((k, i))
        except Exception as e:   # noqa: BLE001 (a thread's exception is not the test's)
            wrong.append(e)
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not wrong, wrong[0]


@pytest.mark.parametrize("capturing,kept", [(0, True), (1, False)])
def test_logits_are_not_kept_while_their_device_captures(monkeypatch, capturing, kept):
    """The stream that is asked is that of the tensors' device (1), not of the current one (0)."""
    import contextlib
    from verl_amd.utils.kernel import linear_cross_entropy as K
    current = [0]

    @contextlib.contextmanager
    def device(d):
        current.append(d.index)
        yield
        current.pop()
    monkeypatch.delenv("VAMD_LCE_LOGITS_CACHE_GB", raising=False)
    monkeypatch.setattr(K, "_free_device_bytes", lambda d: 1 << 40)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current[-1])
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: current[-1] == capturing)
    assert K.keeps_logits(64, 1024, torch.device("cuda", 1)) == kept and current == [0]
