"""AdaPNM's keep count from the clip-sum pass against the oracle, bit for bit, where the
count of u * g > 0 may differ from that of d * g > 0 (d = u / clip * lr) and the keep-count
pass has to take over: updates or products that underflow once scaled, learning rates above
1/2, zero and non-finite gradients; and cases that keep the early count.  Which of the two
counted a tensor is read back from its scalar words (word 3: 1 where the keep-count pass did)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import cases  # noqa: E402
from gpu_cases import assert_same_as_oracle, oracle_case_run, run_gpu  # noqa: E402
from test_gpu_nonfinite import _check  # noqa: E402

SHAPES = [[40, 640], [9, 2560], [30, 33], [200, 16], [77], [12, 72]]

CASES = {
    "plain": dict(lr=1e-3),
    "clipped": dict(lr=1e-3, clip_threshold=0.01),
    "tiny_lr": dict(lr=1e-39),
    "denormal_product": dict(lr=1e-33),
    "zero_lr": dict(lr=0.0),
    "lr_above_half": dict(lr=0.9),
    "noclip": dict(lr=1e-3, clip_threshold=0.0),
}


@pytest.fixture(autouse=True, scope="module")
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")


# the tensors whose count the keep-count pass has to take, for bf16 gradients of 1e-3
# (None: not fixed by the case); a NaN clip sum leaves the divisor at 1, and the early count
# holds
LATE = {"plain": set(), "noclip": set(), "tiny_lr": set(range(6)), "zero_lr": set(range(6)),
        "lr_above_half": set(range(6)), "clipped": set(), "denormal_product": None}


def _late(opt, n):
    """Scalar word 3 of each of the n tensors after the last step."""
    from kaon_amd import _lib as L

    (_ptrs, plan), = opt._plans.values()
    descs = (L.KaonTensor * n).from_buffer_copy(plan.table[:n * ctypes.sizeof(L.KaonTensor)].cpu().numpy().tobytes())
    words = plan.workspace.view(torch.int32).cpu().numpy()
    return {int(d.tensor_id) for d in descs if words[d.ws_scal + 3] == 1}


@pytest.mark.parametrize("mom", ["int8", "bfloat16", "4bit", "float32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_keep_count_bit_exact(name, mom):
    for p, sig in (("bf16", None), ("f32", [1e-3, 1e-22, 1e-36, 1e-3, 1e-38, 1e-20])):
        case = dict(steps=2, seed=14, p_dtype=p, g_dtype=p, opt="adapnm", shapes=SHAPES,
                    kwargs=dict(momentum_dtype=mom, momentum_4bit_block=16, **CASES[name]))
        if sig:
            case["grad_sigma"] = sig
        if name == "clipped":
            case["poison"] = {1: [(0, "zero_row", 3)], 2: [(1, "nan", 5), (3, "inf", 40)]}
        print(f"[gpu] pnm keep {name} {mom} {p}", flush=True)
        oparams, _, _ = oracle_case_run(case)
        params, gopt, _ = run_gpu(case)
        if name == "clipped":  # NaN payloads are not compared
            _check(case, oparams, params, gopt, f"{name} {mom} {p}")
        else:
            assert_same_as_oracle(case, oparams, params, gopt, label=name)
        if p == "bf16" and LATE[name] is not None:
            assert _late(gopt, len(SHAPES)) == LATE[name], (name, mom)


@pytest.mark.parametrize("mom,p", [("int8", "bf16"), ("bfloat16", "bf16"), ("4bit", "bf16"), ("float32", "f32")])
def test_keep_count_with_nonfinite_gradients(mom, p):
    """NaN and +-inf in gradients of every row kernel of the clip-sum pass, stepped on (their
    clip sums are NaN)."""
    case = dict(steps=3, seed=15, p_dtype=p, g_dtype=p, opt="adapnm", shapes=SHAPES,
                kwargs=dict(lr=1e-3, momentum_dtype=mom, momentum_4bit_block=16),
                poison={1: [(0, "nan", 5), (1, "inf", 17), (3, "-inf", 3), (5, "zero_row", 2)],
                        2: [(2, "inf", 100), (4, "nan", 50), (0, "-inf", 700)]})
    print(f"[gpu] pnm keep non-finite {mom} {p}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    _check(case, oparams, params, gopt, f"{mom} {p}")
    assert _late(gopt, len(SHAPES)) == set()


@pytest.mark.parametrize("mom,p", [("int8", "bf16"), ("bfloat16", "bf16"), ("4bit", "bf16"), ("float32", "f32")])
def test_keep_count_with_an_infinite_clip_divisor(mom, p, monkeypatch):
    """A row whose second moment (beta2 = 0) falls to 1e-42 under a momentum of 0.1 has u^2 that
    sum to inf: every d is 0 and none is kept, though u * g > 0 for about half of them."""
    import gpu_cases

    def grads(case, i, step):
        g = np.array(cases.grad_values(case, i, step))
        if g.ndim == 2:
            g[3] *= 1e-21 if step == 2 else 1.0
        return g

    monkeypatch.setattr(gpu_cases, "grad_values", grads)
    case = dict(steps=2, seed=16, p_dtype=p, g_dtype=p, opt="adapnm", shapes=SHAPES, grad_sigma=[1.0] * len(SHAPES),
                kwargs=dict(lr=1e-3, betas=(0.8, 0.0), eps=0.0, momentum_dtype=mom, momentum_4bit_block=16,
                            gradient_centralization=False))
    print(f"[gpu] pnm keep infinite divisor {mom} {p}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    _check(case, oparams, params, gopt, f"{mom} {p}")
    assert _late(gopt, len(SHAPES)) == {0, 1, 2, 3, 5}


def test_the_early_count_of_short_rows_costs_little():
    """Matrices of one wave group each: the count beside the clip sum, and the keep-count
    pass's early exit, against the same step without either (equal as measured; 1.74 times
    with the waves that have no rows held at a barrier)."""
    from cases import grad_values, param_values
    from golden_compare import group_for
    from gpu_cases import DEV, make_opt

    print("[gpu] pnm keep short rows", flush=True)
    opts = []
    for cautious in (True, False):
        case = dict(steps=1, seed=18, p_dtype="bf16", g_dtype="bf16", opt="adapnm", shapes=[[16, 64]] * 2048,
                    kwargs=dict(lr=1e-3, momentum_dtype="int8", cautious=cautious))
        params = []
        for i in range(len(case["shapes"])):
            params.append(torch.nn.Parameter(torch.from_numpy(param_values(case, i)).to(DEV, torch.bfloat16)))
            params[-1].grad = torch.from_numpy(grad_values(case, i, 1)).to(DEV, torch.bfloat16)
        opts.append(make_opt(case, params, group_for(case)))
        opts[-1].step()
    best = [float("inf")] * 2
    for _ in range(5):
        for k, o in enumerate(opts):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            e0.record()
            for _ in range(10):
                o.step()
            e1.record()
            torch.cuda.synchronize()
            best[k] = min(best[k], e0.elapsed_time(e1))
    print("cautious / not, ms per 10 steps:", best, flush=True)
    assert best[0] <= 1.35 * best[1], best
