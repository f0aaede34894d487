"""Phase 1 against the oracle, bit for bit, at the edges of its row kernels: rows of up to
16 chunks (side by side over the workgroup), the first length past them, rows around the
register classes' limits (2048, 5120 and 12288 columns), a partial last chunk, tensors of
fewer than 8 elements, and row counts around the wave group, slice and run of a row length."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from gpu_cases import assert_same_as_oracle, oracle_case_run, run_gpu  # noqa: E402

SHORT = [[7, 1], [321, 2], [400, 16], [81, 33], [161, 64], [85, 65], [325, 32], [20, 120], [21, 121], [83, 127],
         [1, 128], [5, 5], [2, 3]]
LONG = [[3, 129], [85, 137], [21, 511], [41, 513], [13, 1025], [5, 2047], [6, 2049], [33, 2056], [3, 5119], [2, 5121]]

# many runs per column (the finalize step's batches of partials, 1 to 8 columns per thread)
# and many rounds of rows for the row factors' mean
TALL = [[5001, 70], [9000, 9], [4097, 300], [40000, 3], [700, 520], [333, 1100], [50, 2049], [40, 5000], [4100, 16]]
# the same among many short tensors: the finalize step's narrow workgroups
MANY = TALL + [[3, 5]] * 200
# whole 16-byte rows of fewer than 8 chunks: 1 to 7 chunks, several rows side by side
THIN = [[300, 16], [77, 8], [90, 24], [50, 40], [33, 64], [641, 32], [25, 56], [96, 48]]

CASES = {
    "bf16_tall": ("adakaon", TALL, dict(momentum_dtype="int8", clip_threshold=0.05), "bf16", "bf16"),
    "bf16_tall_many": ("adakaon", MANY, dict(momentum_dtype="int8", clip_threshold=0.05), "bf16", "bf16"),
    "f32_tall": ("adakaon", TALL, dict(), "f32", "f32"),
    "pnm_tall": ("adapnm", TALL[:4], dict(momentum_dtype="int8"), "bf16", "bf16"),
    "thin_int8": ("adakaon", THIN, dict(momentum_dtype="int8", weight_decay=0.02), "bf16", "bf16"),
    "thin_4bit_b8": ("adakaon", THIN, dict(momentum_dtype="4bit", momentum_4bit_block=8), "bf16", "bf16"),
    "thin_4bit_b32": ("nekaon", THIN, dict(momentum_dtype="4bit", momentum_4bit_block=32), "bf16", "bf16"),
    "thin_lion": ("lion", THIN, dict(momentum_dtype="int8"), "bf16", "bf16"),
    "bf16_short": ("adakaon", SHORT, dict(momentum_dtype="int8", clip_threshold=0.05), "bf16", "bf16"),
    "bf16_short_nogc": ("adakaon", SHORT, dict(gradient_centralization=False), "bf16", "bf16"),
    "f32_short": ("adakaon", SHORT, dict(momentum_dtype="int8", clip_threshold=0.05), "f32", "f32"),
    "f16_short": ("adakaon", SHORT, dict(bf16_method="none"), "f16", "f16"),
    "lion_short": ("lion", SHORT, dict(momentum_dtype="int8"), "bf16", "bf16"),
    "bf16_long": ("adakaon", LONG + [[3, 12287]], dict(momentum_dtype="int8", clip_threshold=0.05), "bf16", "bf16"),
    "bf16_long_eps0": ("adakaon", LONG, dict(eps=(0.0, 1e-3)), "bf16", "bf16"),
    "bf16_long_tiny_eps": ("adakaon", LONG, dict(eps=(1e-35, 1e-3)), "bf16", "bf16"),
    "f32_long": ("adakaon", LONG, dict(clip_threshold=0.05), "f32", "f32"),
    "f16_long": ("adakaon", LONG, dict(bf16_method="kahan"), "f16", "f16"),
    "lion_f32_long": ("lion", LONG, dict(), "f32", "f32"),
    "pnm_long": ("adapnm", LONG, dict(), "bf16", "f32"),
}


@pytest.fixture(autouse=True, scope="module")
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a ROCm GPU")


@pytest.mark.parametrize("name", sorted(CASES))
def test_row_statistics_bit_exact(name):
    opt, shapes, kw, p, g = CASES[name]
    case = dict(steps=2, seed=13, p_dtype=p, g_dtype=g, opt=opt, shapes=shapes, kwargs=dict(lr=1e-3, **kw))
    print(f"[gpu] row statistics {name}", flush=True)
    oparams, _, _ = oracle_case_run(case)
    params, gopt, _ = run_gpu(case)
    assert_same_as_oracle(case, oparams, params, gopt, label=name)
