"""tfqx_plan_set_seed: a plan given a seed draws what a plan built with that seed draws,
without a new upload, for sampling and noisy plans on every path; a captured graph keeps
the seed that its plan had then.  Equal draws, so equal bytes."""

import numpy as np
import pytest

from quantum_amd import _lib, noise
from quantum_amd import circuits as C
from quantum_amd import serialize as S
from quantum_amd._lib import Plan, np_ptr
from quantum_amd.tfq_simulate_ops import _common, _plan_args

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _batch(n, channels):
    q = C.LineQubit.range(n)
    ops = [C.YPowGate(exponent=0.1 + 0.05 * i).on(x) for i, x in enumerate(q)]
    ops += [C.CNOT(a, b) for a, b in zip(q, q[1:])]
    if channels:
        ops += [C.amplitude_damp(0.3).on(x) for x in q]
    sums = [[C.PauliSum([C.PauliString({q[0]: "Z", q[1]: "X"}, 0.6), C.PauliString({q[1]: "Z"})])]]
    return S.convert_to_tensor([C.Circuit(ops)] * 2), S.convert_to_tensor(sums * 2)


def _sampling_plan(kind, n, seed):
    progs, psums = _batch(n, False)
    p, names, values = _common(progs, [], np.zeros((2, 0), np.float32))
    P, N, args = _plan_args(p, names, values)
    if kind == "samples":
        plan = Plan(_lib.lib().tfqx_plan_simulate_samples, *args, 40, seed)
        return plan, (2, 40, n), np.int8
    sums = _lib.StringTensor(psums)
    counts = np.full((2, 1), 60, np.int32)
    plan = Plan(_lib.lib().tfqx_plan_simulate_sampled_expectation, *args, sums.ptr, sums.off, 1,
                np_ptr(counts), seed)
    return plan, (2, 1), np.float32


def _noisy_plan(kind, n, seed):
    progs, psums = _batch(n, True)
    values = np.zeros((2, 0), np.float32)
    if kind == "noisy samples":
        p, names, values = _common(progs, [], values)
        P, N, args = _plan_args(p, names, values)
        return Plan(_lib.lib().tfqx_plan_noisy_samples, *args, 40, seed), (2, 40, n), np.int8
    plan, shape = noise.plan_expectation(progs, [], values, psums, np.full((2, 1), 60, np.int32),
                                         seed, sampled=kind == "noisy sampled")
    return plan, shape, np.float32


KINDS = [("samples", 6), ("sampled", 6), ("samples", 12), ("samples", 15), ("sampled", 15),
         ("noisy", 5), ("noisy sampled", 5), ("noisy samples", 5), ("noisy samples", 11)]


@pytest.mark.parametrize("kind,n", KINDS)
def test_set_seed_equals_a_plan_built_with_it(kind, n):
    import torch
    build = _noisy_plan if kind.startswith("noisy") else _sampling_plan
    print(f"[gpu-case] set_seed, {kind}, {n} qubits", flush=True)
    plan, shape, dtype = build(kind, n, 5)
    if not kind.startswith("noisy"):
        assert plan.stats()["streaming"] == (n > 14)
    dev, stream = torch.device("cuda", 0), torch.cuda.current_stream().cuda_stream

    def launch(p):
        out = torch.empty(shape, dtype=torch.int8 if dtype == np.int8 else torch.float32, device=dev)
        p.launch(out, stream)
        return out.cpu().numpy()

    def fresh(seed):
        p = build(kind, n, seed)[0]
        p.upload(dev, stream)
        return launch(p)

    plan.upload(dev, stream)
    first = launch(plan)
    plan.set_seed(77)
    second = launch(plan)
    np.testing.assert_array_equal(first, fresh(5))
    np.testing.assert_array_equal(second, fresh(77))
    assert (first != second).any()


@pytest.mark.parametrize("kind,n", [("samples", 6), ("samples", 15), ("noisy samples", 5)])
def test_a_graph_keeps_its_seed(kind, n):
    import torch
    build = _noisy_plan if kind.startswith("noisy") else _sampling_plan
    print(f"[gpu-case] set_seed and a captured graph, {kind}, {n} qubits", flush=True)
    plan, shape, _ = build(kind, n, 5)
    dev, side = torch.device("cuda", 0), torch.cuda.Stream()
    with torch.cuda.stream(side):
        out = torch.empty(shape, dtype=torch.int8, device=dev)
        plan.upload(dev, side.cuda_stream)
        plan.launch(out, side.cuda_stream)
        first = out.cpu().numpy()
        graph = plan.capture_graph(out, side.cuda_stream)
        plan.set_seed(77)
        for _ in range(3):
            out.zero_()
            graph.launch(side.cuda_stream)
            side.synchronize()
            np.testing.assert_array_equal(out.cpu().numpy(), first)
        plan.launch(out, side.cuda_stream)
        assert (out.cpu().numpy() != first).any()
