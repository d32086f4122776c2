"""fast_logits and eval of one to four tokens at widths without a two-column
GEMV (multiples of 256 other than 512, 1536, 2560, 4096 and 9728), against the
oracle and against themselves: what such a call returns is decided by its inputs,
not by which copies of the weights earlier calls have built."""

import shutil

import numpy as np
import pytest

import gguf_util
from conftest import make_prompt
from oracle import oracle as O
from s2hip import synth

pytestmark = pytest.mark.gpu

SHAPE = synth.TINY.with_(name="w1024", slow_layers=2, dim=1024, ffn=2048, heads=16, kv_heads=4, fast_ffn=2048,
                         fast_heads=16, fast_kv_heads=4, vocab=2304, semantic_begin=1024, semantic_end=2047,
                         im_end_id=1000)
TYPES = {"f16": synth.GGML_F16, "q8_0": synth.GGML_Q8_0, "q4_0": synth.GGML_Q4_0}
PREFIXES = (0, 1, 2, 3, 8, 9)


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / max(1e-30, float(np.max(np.abs(b)))))


def _inputs(seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(SHAPE.dim).astype(np.float32), rng.integers(0, SHAPE.codebook_size, 9).astype(np.uint32)


def _outlier_gguf(model_dir, tmp_path, prefix, layers):
    path = str(tmp_path / "outlier.gguf")
    shutil.copyfile(synth.ensure_gguf(SHAPE, model_dir), path)
    for l in range(layers):
        for w in ("w1", "w3"):
            gguf_util.scale_rows(path, f"{prefix}.{l}.feed_forward.{w}.weight", [300], 1000.0)
    return path


def test_fast_logits_with_an_outlier_channel_after_a_generation(model_dir, tmp_path):
    """Channel 300 of the Fast-AR FFN lies past the headroom of the batched
    product, whose copies the generation before has built."""
    from s2hip import Engine

    path = _outlier_gguf(model_dir, tmp_path, "fast_layers", SHAPE.fast_layers)
    o = O.OracleModel(path, 64, SHAPE.im_end_id)
    hidden, codes = _inputs(1)
    with Engine(path, 64, SHAPE.im_end_id) as e:
        e.generate_codes(make_prompt(SHAPE, 7, seed=1), 2, min_tokens_before_end=100)
        for n in PREFIXES:
            got, want = e.fast_logits(hidden, codes[:n]), o.fast_logits(hidden, codes[:n])
            assert np.all(np.isfinite(got)) and _rel(got, want) < 1e-4, n


@pytest.mark.parametrize("weights", sorted(TYPES))
def test_fast_logits_do_not_depend_on_earlier_calls(model_dir, weights):
    from s2hip import Engine

    path = synth.ensure_gguf(SHAPE.with_(linear_type=TYPES[weights]), model_dir)
    o = O.OracleModel(path, 64, SHAPE.im_end_id)
    hidden, codes = _inputs(2)
    with Engine(path, 64, SHAPE.im_end_id) as e:
        cold = [e.fast_logits(hidden, codes[:n]) for n in PREFIXES]
        e.eval(make_prompt(SHAPE, 5, seed=2))
        e.generate_codes(make_prompt(SHAPE, 7, seed=3), 2, min_tokens_before_end=100)
        for n, want in zip(PREFIXES, cold):
            assert np.array_equal(e.fast_logits(hidden, codes[:n]), want), n
            assert _rel(want, o.fast_logits(hidden, codes[:n])) < 1e-4, n


@pytest.mark.parametrize("weights", sorted(TYPES))
def test_short_evals_do_not_depend_on_earlier_calls(model_dir, weights):
    from s2hip import Engine

    path = synth.ensure_gguf(SHAPE.with_(linear_type=TYPES[weights]), model_dir)
    with Engine(path, 64, SHAPE.im_end_id) as warm:
        warm.eval(make_prompt(SHAPE, 5, seed=2))
        warm.generate_codes(make_prompt(SHAPE, 7, seed=3), 2, min_tokens_before_end=100)
        for n in (1, 2, 3, 4):
            prompt = make_prompt(SHAPE, n, seed=n)
            with Engine(path, 64, SHAPE.im_end_id) as cold:
                want = cold.eval(prompt)
            warm.reset()
            got = warm.eval(prompt)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), n


# an input row wider than the decode GEMV stages in LDS (38400 floats), and more
# heads than the decode attention takes (255)
WIDE = {"ffn": dict(ffn=40960), "heads": dict(heads=256, kv_heads=64)}


@pytest.mark.parametrize("what", sorted(WIDE))
def test_short_evals_of_shapes_past_the_decode_kernels(model_dir, what):
    """Such a model's prompts of any length go through the prompt products."""
    from s2hip import Engine

    shape = synth.TINY.with_(name="wide_" + what, slow_layers=1, fast_layers=1, vocab=2304, semantic_begin=1024,
                             semantic_end=2047, im_end_id=1000, **WIDE[what])
    path = synth.ensure_gguf(shape, model_dir)
    o = O.OracleModel(path, 64, shape.im_end_id)
    with Engine(path, 64, shape.im_end_id) as e:
        for n in (5, 1, 2, 3, 4):
            prompt = make_prompt(shape, n, seed=n)
            (hg, lg), (ho, lo) = e.eval(prompt), o.eval(prompt)
            assert _rel(hg, ho) < 1e-4 and _rel(lg, lo) < 1e-4, n
        assert e.n_past == 15


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
def test_non_finite_activations_are_answered_alike_at_every_length(model_dir, tmp_path, n):
    """A NaN that the last layer's FFN makes reaches nothing but the outputs, which
    are returned; one that a later layer's attention reads is an error."""
    from s2hip import Engine, S2HipError

    for layer in (SHAPE.slow_layers - 1, 0):
        path = str(tmp_path / f"nan{layer}.gguf")
        shutil.copyfile(synth.ensure_gguf(SHAPE, model_dir), path)
        gguf_util.scale_rows(path, f"layers.{layer}.feed_forward.w2.weight", [17], np.inf)
        with Engine(path, 64, SHAPE.im_end_id) as e:
            if layer:
                hidden, _ = e.eval(make_prompt(SHAPE, n, seed=n))
                assert not np.all(np.isfinite(hidden)) and e.n_past == n
            else:
                with pytest.raises(S2HipError, match="not finite"):
                    e.eval(make_prompt(SHAPE, n, seed=n))


def test_a_failed_call_on_another_slot_leaves_range_errors_where_they_are_read(model_dir, tmp_path, monkeypatch):
    """More heads than the decode attention takes, and prompts forced through it:
    eval on slot 3 fails while it launches.  fast_codebooks then still sees that its
    outlier channel is beyond the batched product's range, and runs again."""
    from s2hip import Engine, S2HipError

    shape = SHAPE.with_(name="w1024h256", heads=256, kv_heads=64)
    path = str(tmp_path / "outlier.gguf")
    shutil.copyfile(synth.ensure_gguf(shape, model_dir), path)
    for l in range(shape.fast_layers):
        for w in ("w1", "w3"):
            gguf_util.scale_rows(path, f"fast_layers.{l}.feed_forward.{w}.weight", [300], 1000.0)
    o = O.OracleModel(path, 64, shape.im_end_id)
    hidden, _ = _inputs(3)
    monkeypatch.setenv("S2HIP_PREFILL_GEMV", "1")
    with Engine(path, 64, shape.im_end_id) as e:
        with pytest.raises(S2HipError, match="launch_attention"):
            e.eval_slot(3, make_prompt(shape, 5, seed=3))
        got = e.fast_codebooks(hidden, 7)
        want = o.fast_codebooks(hidden, 7, 0.0, 1.0, 0, 0)
        assert np.array_equal(got[0], want[0])


def test_engines_on_two_devices_of_one_process(model_dir):
    """Prompts, decoding and sampling on a second device after a first: what a kernel
    was granted on one device (its dynamic LDS) is asked for on the other too."""
    import ctypes

    from s2hip import Engine

    count = ctypes.c_int(0)
    ctypes.CDLL("libamdhip64.so").hipGetDeviceCount(ctypes.byref(count))
    if count.value < 2:
        pytest.skip("one device")
    path = synth.ensure_gguf(SHAPE, model_dir)
    prompt = make_prompt(SHAPE, 70, seed=4)
    out = []
    for device in (0, 1):
        with Engine(path, 128, SHAPE.im_end_id, device=device) as e:
            out.append((e.eval(prompt)[0], e.generate_codes(prompt, 3, min_tokens_before_end=100)["codes"]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("weights", sorted(TYPES))
def test_fast_codebooks_of_a_new_engine_equal_those_of_a_used_one(model_dir, weights):
    """And both the oracle's: the first call builds what a generation would have."""
    from s2hip import Engine

    path = synth.ensure_gguf(SHAPE.with_(linear_type=TYPES[weights]), model_dir)
    o = O.OracleModel(path, 64, SHAPE.im_end_id)
    inputs = [(_inputs(s)[0], s) for s in range(10, 18)]
    with Engine(path, 64, SHAPE.im_end_id) as e:
        cold = [e.fast_codebooks(h, s)[0] for h, s in inputs]
        e.generate_codes(make_prompt(SHAPE, 7, seed=3), 2, min_tokens_before_end=100)
        for (h, s), want in zip(inputs, cold):
            assert np.array_equal(e.fast_codebooks(h, s)[0], want), s
            assert np.array_equal(want, o.fast_codebooks(h, s, 0.0, 1.0, 0, 0)[0]), s
