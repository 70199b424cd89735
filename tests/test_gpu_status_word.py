"""The device status word between operations: what kernels of a token-local execution raise is reported
by that execution, and never by an operation that starts after it was given up."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_backend import MoeCase, TokenLocal, backend, run_greedy, run_matvec, sweep_image_decision  # noqa: F401
from yvex_amd import abi

pytestmark = pytest.mark.gpu


def opened(case, bad=True):
    """An execution behind its routing wait, with an expert whose route weight is not finite queued."""
    t = TokenLocal(case)
    assert t.begin() == 0, t.err.message
    if bad:
        assert t.add(t.expert_views(0)[0], float("inf"), False) == 0, t.err.message
    return t


def deferred(case):
    case.job.eager_execution, case.job.device_completion = 1, C.pointer(abi.DeviceCompletion(1, None))
    rc = case.execute()
    case.job.device_completion = None
    return rc


def complete(case):
    done = abi.RowBatchResult()
    return case.ops.complete_rows(case.b.handle, 0, C.byref(done), C.byref(case.err))


def next_operation(b, case, kind):
    width = case.hidden
    if kind == "rows":
        return case.execute()
    if kind == "deferred rows":
        return deferred(case) or complete(case)
    if kind == "greedy":
        return run_greedy(b, b.f32(np.arange(3 * width)), 3, width)[0]
    out = b.empty_f32(2 * case.intermediate)
    if kind == "matvec":
        rc, _, _ = run_matvec(b, case.host + case.offsets["sgate"], case.parts["sgate"], case.qt, case.intermediate, width,
                              b.f32(np.ones((2, width))), out, 2, 1)
        return rc
    facts, err, at = abi.OperationFacts(), abi.Error(), (C.c_uint * 1)(1)
    return b.lib.yvex_rocm_encoded_gather(b.handle, case.host + case.offsets["sdown"], case.parts["sdown"].nbytes, case.qt,
                                          width, case.intermediate, case.parts["sdown"].nbytes // width, at, 1, out,
                                          C.byref(facts), C.byref(err))


@pytest.mark.parametrize("ended", ["closed", "finish fails"])
@pytest.mark.parametrize("kind", ["matvec", "gather", "greedy", "rows", "deferred rows"])
def test_an_abandoned_execution_is_nobody_elses_failure(backend, oracle, monkeypatch, kind, ended):  # noqa: F811
    case = MoeCase(backend, oracle, rows=3, streams=4, act=abi.ACT_DEVICE_F32)
    backend.workspace(max(case.workspace_bytes, 8 << 20))
    for _ in range(2):
        t = opened(case)
        if ended == "finish fails":
            monkeypatch.setenv("YVEX_TEST_ROCM_SYNC_FAILURE", "1")
            assert t.finish() == abi.BACKEND
            monkeypatch.delenv("YVEX_TEST_ROCM_SYNC_FAILURE")
        assert t.close() == 0
        assert next_operation(backend, case, kind) == 0
        assert next_operation(backend, case, kind) == 0


@pytest.mark.parametrize("between", ["nothing", "image build", "another execution", "barrier"])
def test_an_execution_reports_what_its_kernels_raised(backend, oracle, between):  # noqa: F811
    case = MoeCase(backend, oracle, rows=3, streams=4, act=abi.ACT_DEVICE_F32)
    if between == "barrier":
        backend.workspace(max(case.workspace_bytes, 8 << 20))
        assert deferred(case) == 0, case.err.message
    t = opened(case, bad=between != "another execution")
    if between == "image build":
        decision = sweep_image_decision(case.experts, case.experts * case.intermediate, case.hidden,
                                        abi.CONSUMER_ROUTED_GATE_UP)
        storage, err = abi.ULL(), abi.Error()
        assert backend.lib.yvex_rocm_moe_derived_layout_plan(C.byref(decision), C.byref(storage), C.byref(err)) == 0
        rc, image = backend.tensor(storage.value, abi.DTYPE_I8)
        assert rc == 0
        assert backend.lib.yvex_rocm_moe_sweep_image_build_resident(
            backend.handle, C.byref(decision), case.arena_tensor.contents.data + case.offsets["gate"],
            image.contents.data, storage.value, C.byref(err)) == 0, err.message
    elif between == "another execution":
        other = opened(case, bad=False)
        assert t.add(t.expert_views(0)[0], float("inf"), False) == 0, t.err.message
        assert other.finish() == abi.BACKEND and other.close() == 0     # the word is the backend's: both report it
    elif between == "barrier":
        assert complete(case) != 0
    assert t.finish() == abi.BACKEND
    assert t.close() == 0
    backend.workspace(8 << 20)
    assert next_operation(backend, case, "matvec") == 0


def test_a_phase_counts_the_launches_it_makes(backend, oracle):  # noqa: F811
    """The batches of a phase launch the same kernels; the word is cleared before the first only where somebody
    else may have raised it, and published once at the barrier."""
    case = MoeCase(backend, oracle, rows=3, streams=4, act=abi.ACT_DEVICE_F32)
    backend.workspace(max(case.workspace_bytes, 8 << 20))

    def phase(batches):
        counts = []
        for _ in range(batches):
            assert deferred(case) == 0, case.err.message
            counts.append(case.result.kernel_launches)
        done = abi.RowBatchResult()
        assert case.ops.complete_rows(backend.handle, 0, C.byref(done), C.byref(case.err)) == 0
        return counts, done.kernel_launches
    (first, second, third), published = phase(3)
    assert first == second == third and published == 1
    out, case.out = case.out, abi.RowBatchOutput()      # (no host copies, whose rows would come from other kernels)
    assert case.execute() == 0 and case.result.kernel_launches == first + published
    case.out = out
    assert opened(case).close() == 0
    (first, second), published = phase(2)
    assert first == second + 1 and published == 1
