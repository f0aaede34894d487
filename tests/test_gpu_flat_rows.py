"""The flat-chunk keep-count / apply kernels against the oracle, bit for bit, at the row
lengths where a chunk's place in its row matters: rows shorter than a chunk, rows around
multiples of 8 and of a window (512), slices that begin inside a chunk, tensors whose last
chunk is partial, and params whose storage is not 16-byte aligned."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from gpu_cases import assert_same_as_oracle, oracle_case_run, run_gpu, state_of, to_bits  # noqa: E402

# rows of 1 to 4 slices; 85 rows of 7 and 200 of 17 span slices that start inside a chunk
SHAPES = [[5, 1], [40, 3], [85, 7], [30, 8], [50, 9], [41, 15], [200, 17], [24, 16], [3, 511], [5, 512], [7, 513],
          [43, 771], [2, 4097], [33, 20], [1, 1], [1, 70], [13]]

CASES = {
    "ada_int8_sr": ("adakaon", dict(momentum_dtype="int8", weight_decay=0.02), "bf16", "bf16"),
    "ada_4bit_b64": ("adakaon", dict(momentum_dtype="4bit", momentum_4bit_block=64), "bf16", "bf16"),
    "ada_4bit_b24": ("adakaon", dict(momentum_dtype="4bit", momentum_4bit_block=24), "f32", "f32"),
    "ada_4bit_b5": ("adakaon", dict(momentum_dtype="4bit", momentum_4bit_block=5), "bf16", "bf16"),
    "ada_bf16_kahan": ("adakaon", dict(momentum_dtype="bfloat16", bf16_method="kahan", weight_decay=0.02), "bf16",
                       "bf16"),
    "ada_f32_rn_f32g": ("adakaon", dict(momentum_dtype="float32", bf16_method="none"), "bf16", "f32"),
    "ada_none_f16": ("adakaon", dict(betas=(0.0, 0.999)), "f16", "f16"),
    "lion_int8_sr": ("lion", dict(momentum_dtype="int8", weight_decay=0.1), "bf16", "bf16"),
    "lion_f32": ("lion", dict(momentum_dtype="float32", cautious=False), "f32", "f32"),
    "nekaon_4bit": ("nekaon", dict(momentum_dtype="4bit", momentum_4bit_block=32), "bf16", "bf16"),
    "nekaon_int8_f32": ("nekaon", dict(momentum_dtype="int8"), "f32", "f32"),
    "pnm_int8": ("adapnm", dict(momentum_dtype="int8", weight_decay=0.02), "bf16", "bf16"),
    "pnm_4bit_kahan": ("adapnm", dict(momentum_dtype="4bit", momentum_4bit_block=16, bf16_method="kahan"), "bf16",
                       "bf16"),
    "pnm_f32": ("adapnm", dict(momentum_dtype="float32"), "f32", "f32"),
}


@pytest.fixture(autouse=True, scope="module")
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")


@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_of_any_length_bit_exact(name):
    opt, kw, p, g = CASES[name]
    case = dict(steps=3, seed=11, p_dtype=p, g_dtype=g, opt=opt, shapes=SHAPES, kwargs=dict(lr=1e-3, **kw))
    print(f"[gpu] flat rows {name}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    assert_same_as_oracle(case, oparams, params, gopt, label=name)


@pytest.mark.parametrize("name", ["ada_int8_sr", "lion_f32", "pnm_f32"])
def test_unaligned_storage_gives_the_same_bits(name):
    """Params and gradients that start one element into their storage (no vector accesses)
    against the same values aligned."""
    from cases import grad_values, param_values
    from golden_compare import group_for
    from gpu_cases import DEV, make_opt, tdtype

    opt, kw, p, g = CASES[name]
    case = dict(steps=2, seed=12, p_dtype=p, g_dtype=g, opt=opt, shapes=[[9, 64], [43, 771], [24, 16], [40, 3], [77]],
                kwargs=dict(lr=1e-3, **kw))
    print(f"[gpu] unaligned {name}", flush=True)
    runs = []
    for off in (0, 1):
        params = []
        for i, s in enumerate(case["shapes"]):
            n = int(np.prod(s))
            buf = torch.zeros(n + 8, device=DEV, dtype=tdtype(p))
            v = buf[off:off + n].view(s)
            v.copy_(torch.from_numpy(param_values(case, i)).to(DEV, tdtype(p)))
            params.append(torch.nn.Parameter(v))
        o = make_opt(case, params, group_for(case))
        for step in (1, 2):
            for i, prm in enumerate(params):
                buf = torch.zeros(prm.numel() + 8, device=DEV, dtype=tdtype(g))
                gv = buf[off:off + prm.numel()].view(case["shapes"][i])
                gv.copy_(torch.from_numpy(grad_values(case, i, step)).to(DEV, tdtype(g)))
                prm.grad = gv
            o.step()
        torch.cuda.synchronize()
        runs.append((params, o))
    (pa, oa), (pb, ob) = runs
    for a, b in zip(pa, pb):
        assert np.array_equal(to_bits(a), to_bits(b))
        sa, sb = state_of(oa, a), state_of(ob, b)
        for k in sa:
            if torch.is_tensor(sa[k]):
                assert np.array_equal(to_bits(sa[k]).reshape(-1), to_bits(sb[k]).reshape(-1)), k


# rows whose chunks start at every offset, with partial last chunks, for the kernels that
# walk rows with unaligned 16-byte accesses (KProdigy's passes, AdaMuon's momentum, MSAM's
# norm); AdaMuon's orthogonalized update is compared between the two storages instead
ROWS = [[5, 3], [41, 15], [9, 513], [43, 771], [6, 1029], [3, 520], [70], [2, 9, 5]]


@pytest.mark.parametrize("mom,p,method,kw", [
    ("bfloat16", "bf16", "stochastic_rounding", {}),
    ("int8", "bf16", "stochastic_rounding", dict(second_moment="factored", weight_decay=0.01)),
    ("4bit", "bf16", "kahan", dict(momentum_4bit_block=24)),
    ("float32", "f32", "none", dict(second_moment="factored", cautious=True)),
    ("int8", "f16", "none", {}),
    ("bfloat16", "bf16", "none", dict(weight_decay=0.01, decouple=False)),
])
def test_kprodigy_rows_of_any_length_bit_exact(mom, p, method, kw):
    case = dict(steps=3, seed=16, p_dtype=p, g_dtype=p, opt="kprodigy", shapes=ROWS,
                kwargs=dict(lr=1.0, momentum_dtype=mom, bf16_method=method, **kw))
    print(f"[gpu] kprodigy rows {mom} {p} {method}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    assert_same_as_oracle(case, oparams, params, gopt, label=f"pd_{mom}")


@pytest.mark.parametrize("mom", ["int8", "bfloat16"])
def test_msam_and_adamuon_unaligned_rows(mom):
    """MSAM's momentum norm against the oracle, and AdaMuon's momentum (codes, scales)."""
    case = dict(steps=2, seed=17, p_dtype="bf16", g_dtype="bf16", opt="msam", shapes=ROWS,
                kwargs=dict(lr=1e-3, momentum_dtype=mom))
    print(f"[gpu] msam rows {mom}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    assert_same_as_oracle(case, oparams, params, gopt, label=f"msam_{mom}")
    case = dict(steps=1, seed=18, p_dtype="bf16", g_dtype="bf16", opt="adamuon", shapes=[[9, 513], [43, 71], [16, 33]],
                kwargs=dict(lr=1e-3, momentum_dtype=mom))
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    for op, prm in zip(oparams, params):
        for k in ("m", "m_scale"):
            if k in op.state:
                got = to_bits(state_of(gopt, prm)[k]).reshape(-1)
                want = np.asarray(op.state[k]).reshape(-1)
                want = want.view(got.dtype) if want.itemsize == got.itemsize else want
                assert np.array_equal(got, want), k
