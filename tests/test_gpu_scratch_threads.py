"""Calls that use the library's scratch between their launches, from two host
threads on one stream and on two streams at once: each call's bits are those it
gives alone."""
import threading

import pytest
import torch

from credit_amd import hip_lib
from credit_amd.workloads import WORKLOADS, make_ffn_inputs

pytestmark = pytest.mark.gpu


def ffn_train(gpu, seed):
    """A training forward whose second product is split over K."""
    rows, d, f = 128, 256, 8192
    x, w1, w2 = (t.to(gpu) for t in make_ffn_inputs(
        rows, d, torch.Generator().manual_seed(seed), ffn_dim=f))
    w1, w2 = w1.t().contiguous(), w2.t().contiguous()
    outs = (torch.empty_like(x), torch.empty(rows, device=gpu),
            torch.empty(rows, f, device=gpu, dtype=torch.bfloat16),
            torch.empty(rows, f, device=gpu, dtype=torch.bfloat16))
    return outs, lambda: hip_lib.ffn_train_forward(x, w1, w2, *outs, hip_lib.FFN_EPS,
                                                   hip_lib.make_cfg())


def wide(name, rows, cols):
    """A few wide rows in two launches of chunks."""
    def case(gpu, seed):
        ins = tuple(t.to(gpu) for t in WORKLOADS[name].make_inputs(rows, cols, seed=seed))
        outs = hip_lib.allocate_outputs(name, ins)
        return outs, lambda: hip_lib.HIP_LAUNCHERS[name](ins, outs)
    return case


CASES = {"ffn_train": ffn_train, "softmax_fwd": wide("softmax_fwd", 5, 40003),
         "layernorm_fwd": wide("layernorm_fwd", 16, 131072),
         "rowwise_quant": wide("rowwise_quant", 3, 65539)}


@pytest.mark.parametrize("streams", [1, 2])
@pytest.mark.parametrize("name", CASES)
def test_two_threads(gpu, name, streams):
    print(f"two threads {name} on {streams} stream(s)", flush=True)
    cases = [CASES[name](gpu, seed) for seed in (1, 2)]
    alone = []
    for outs, call in cases:
        call()
        torch.cuda.synchronize()
        alone.append([t.clone() for t in outs])
    shared = [torch.cuda.Stream() for _ in range(streams)]
    torch.cuda.synchronize()
    start, errors = threading.Barrier(2), []

    def work(i):
        outs, call = cases[i]
        wrong = torch.zeros((), dtype=torch.int64, device=gpu)
        try:
            with torch.cuda.stream(shared[i % streams]):
                start.wait(timeout=30)
                for _ in range(50):
                    for t in outs:
                        t.zero_()
                    call()
                    for t, e in zip(outs, alone[i]):
                        wrong += (t != e).sum()
            shared[i % streams].synchronize()
            if int(wrong):
                errors.append((i, int(wrong)))
        except Exception as e:  # noqa: BLE001 (reported by the test's thread)
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not errors and not any(t.is_alive() for t in threads), errors
