"""The flat-chunk keep-count / apply kernels against the oracle, bit for bit, at the row
lengths where a chunk's place in its row matters: rows shorter than a chunk, rows around
multiples of 8 and of a window (512), slices that begin inside a chunk, tensors whose last
chunk is partial, and params whose storage is not 16-byte aligned."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from gpu_cases import assert_same_as_oracle, oracle_case_run, run_gpu, state_of, to_bits  # noqa: E402

# tensors of 1 to 4 slices; the slices of 20 rows of 1601, 12 of 2601 and 4 of 5001 elements
# (4 more than a multiple of 8) begin inside a chunk
SHAPES = [[5, 1], [40, 3], [85, 7], [30, 8], [50, 9], [41, 15], [200, 17], [24, 16], [3, 511], [5, 512], [7, 513],
          [43, 771], [2, 4097], [33, 20], [1, 1], [1, 70], [13], [45, 1601], [26, 2601], [11, 5001]]

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


# the unaligned storage's other optimizers (steps of their own, or passes beside these kernels)
STORAGE = {
    **CASES,
    "pd_bf16": ("kprodigy", dict(momentum_dtype="bfloat16"), "bf16", "bf16"),
    "pd_int8_factored": ("kprodigy", dict(momentum_dtype="int8", second_moment="factored", cautious=True), "bf16",
                         "bf16"),
    "msam_int8": ("msam", dict(momentum_dtype="int8"), "bf16", "bf16"),
    "muon_int8": ("adamuon", dict(momentum_dtype="int8"), "bf16", "bf16"),
    "muon_4bit": ("adamuon", dict(momentum_dtype="4bit", momentum_4bit_block=24), "bf16", "bf16"),
}


def storage_run(case, off_p, off_g):
    """A case stepped with params and gradients that start off_p / off_g elements into
    their storage; (params, optimizer)."""
    from cases import grad_values, param_values
    from golden_compare import group_for
    from gpu_cases import DEV, make_opt, tdtype

    p, g, shapes = case["p_dtype"], case["g_dtype"], case["shapes"]

    def stored(v, dt, off):
        buf = torch.zeros(v.size + 8, device=DEV, dtype=dt)
        t = buf[off:off + v.size].view(v.shape)
        t.copy_(torch.from_numpy(v).to(DEV, dt))
        return t

    params = []
    for i in range(len(shapes)):
        prm = torch.nn.Parameter(stored(param_values(case, i), tdtype(p), off_p))
        if p != g:
            prm.grad_dtype = tdtype(g)
        params.append(prm)
    o = make_opt(case, params, group_for(case))
    for step in range(1, case["steps"] + 1):
        for i, prm in enumerate(params):
            prm.grad = stored(grad_values(case, i, step), tdtype(g), off_g)
        o.step()
    torch.cuda.synchronize()
    return params, o


@pytest.mark.parametrize("off_p,off_g", [(1, 1), (0, 3)])
@pytest.mark.parametrize("name", sorted(STORAGE))
def test_unaligned_storage_gives_the_same_bits(name, off_p, off_g):
    """Params and gradients that start inside a 16-byte line of their storage against the
    same values aligned: weights, every state tensor and the gradients the step leaves."""
    opt, kw, p, g = STORAGE[name]
    case = dict(steps=2, seed=12, p_dtype=p, g_dtype=g, opt=opt, kwargs=dict(lr=1e-3, **kw),
                shapes=[[9, 64], [43, 771], [24, 16], [40, 3], [77], [45, 1601], [6, 2049]])
    print(f"[gpu] unaligned {name} {off_p} {off_g}", flush=True)
    pa, oa = storage_run(case, 0, 0)
    pb, ob = storage_run(case, off_p, off_g)
    for a, b in zip(pa, pb):
        assert np.array_equal(to_bits(a), to_bits(b)), (name, tuple(a.shape))
        assert np.array_equal(to_bits(a.grad), to_bits(b.grad)), (name, tuple(a.shape), "grad")
        sa, sb = state_of(oa, a), state_of(ob, b)
        assert sa.keys() == sb.keys()
        for k in sa:
            if torch.is_tensor(sa[k]):
                assert np.array_equal(to_bits(sa[k]).reshape(-1), to_bits(sb[k]).reshape(-1)), k


@pytest.mark.parametrize("name", ["lion_f32", "ada_bf16_kahan", "ada_int8_sr"])
def test_unaligned_storage_steps_at_the_aligned_rate(name):
    """The same bytes in the same 16-byte accesses: at most 1.5 times the aligned step (1.0 to
    1.1 measured; reading them byte by byte took 1.9 to 3.3)."""
    opt, kw, p, g = STORAGE[name]
    case = dict(steps=1, seed=12, p_dtype=p, g_dtype=g, opt=opt, kwargs=dict(lr=1e-3, **kw),
                shapes=[[2048, 3073], [2048, 2057], [1025, 4097]])
    print(f"[gpu] unaligned rate {name}", flush=True)
    runs = [storage_run(case, off, off)[1] for off in (0, 1)]
    best = [float("inf")] * 2
    for _ in range(5):
        for k, o in enumerate(runs):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(5):
                o.step()
            e1.record()
            torch.cuda.synchronize()
            best[k] = min(best[k], e0.elapsed_time(e1))
    assert best[1] <= 1.5 * best[0], best


# rows whose chunks start at every offset, with partial last chunks, for the kernels that
# walk rows with unaligned 16-byte accesses (KProdigy's passes, AdaMuon's momentum, MSAM's
# norm); AdaMuon's whole step is compared between aligned and unaligned storage above
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
