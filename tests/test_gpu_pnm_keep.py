"""AdaPNM's keep count from the clip-sum pass against the oracle, bit for bit, where the
count of u * g > 0 may differ from that of d * g > 0 (d = u / clip * lr) and the keep-count
pass has to take over: updates or products that underflow once scaled, learning rates above
1/2, zero and non-finite gradients; and cases that keep the early count."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from gpu_cases import assert_same_as_oracle, oracle_case_run, run_gpu  # noqa: E402

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


@pytest.mark.parametrize("mom", ["int8", "bfloat16", "4bit"])
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
        if name == "clipped":  # NaN payloads are not compared: the finite tensors are
            for i in (0, 2, 4, 5):
                got = params[i].detach().float().cpu().numpy().reshape(-1)
                import oracle as O
                want = oparams[i].p.reshape(-1)
                want = O.bf16_to_f32(want) if p == "bf16" else want
                assert (got == want).all(), (name, mom, p, i)
        else:
            assert_same_as_oracle(case, oparams, params, gopt, label=name)
