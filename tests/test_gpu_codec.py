"""The back part of the 12 Hz decoder on the GPU (TQwenCodecVulkan.Back,
codec.vulkan.pas:568-652) through the C ABI, against the oracle (pinned to a
float64 PyTorch composition, tests/test_oracle_codec.py). Bars from the
reference's own GPU codec test (tests/test.tts.qwen.codec.vulkan.pas:46-49,
143-165): the wav within 2e-5 absolute, and chunks of 1, 4 and all frames
giving the same samples, bit for bit."""
import numpy as np
import pytest

import codec_torch
import q3h
import q3o
import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def weights():
    return synth.codec_weights(1)


def _gpu(device, w, x, chunks, max_frames=16):
    c = q3h.Codec(device, w, max_frames=max_frames)
    out, f = [], 0
    try:
        for n in chunks:
            print(f"codec back: {n} frame(s)", flush=True)
            out.append(c.back(x[f:f + n]))
            f += n
    finally:
        c.destroy()
    return np.concatenate(out)


def test_codec_matches_oracle(device, weights):
    x = synth.prompt(3, 6)
    gpu = _gpu(device, weights, x, [1, 2, 3])
    oc = q3o.Codec(weights)
    ref = np.concatenate([oc.back(x[:3]), oc.back(x[3:])])
    oc.destroy()
    d = np.abs(gpu - ref).max()
    print(f"max |gpu - oracle| = {d:.3g}, peak {np.abs(ref).max():.3g}")
    assert d <= 2e-5, d


def test_codec_chunks_give_the_same_samples(device, weights):
    x = synth.prompt(4, 8)
    one = _gpu(device, weights, x, [1] * 8)
    four = _gpu(device, weights, x, [4, 4])
    all_ = _gpu(device, weights, x, [8])
    passes = _gpu(device, weights, x, [8], max_frames=3)  # passes of 3, 3, 2 inside
    assert np.array_equal(one, four) and np.array_equal(one, all_)
    assert np.array_equal(one, passes)


@pytest.mark.parametrize("chunks, max_frames", [([17], 64), ([16, 1], 16), ([9, 8], 16),
                                                ([5, 12], 16)])
def test_codec_kernel_choice_keeps_the_samples(device, weights, chunks, max_frames):
    """The products change their kernels with the rows of a call (one to a few
    frames: slices in parallel; many: walked in one workgroup, 32- or 64-row
    tiles; 64 frames: the widest of the front layers): 17 frames in calls on
    both sides of those lines give the samples of 17 calls."""
    x = synth.prompt(6, 17)
    one = _gpu(device, weights, x, [1] * 17)
    assert np.array_equal(one, _gpu(device, weights, x, chunks, max_frames))


def test_codec_many_frames_in_one_pass(device, weights):
    x = synth.prompt(7, 64)
    assert np.array_equal(_gpu(device, weights, x, [64], 64), _gpu(device, weights, x, [64], 7))


def _one_term_weights(rng):
    """The decoder with one weight per output of every product of the main
    branch, near 1, the residual units and ConvNeXt's branch zero and SnakeBeta's
    term below the last bit (e^80): a sample is seven one-term products."""
    w = synth.codec_weights(1)

    def near_one(n):
        return rng.uniform(0.97, 1.03, n).astype(np.float32)

    def tconv(a, stride):  # [in][out][K]: one input channel per output and phase
        o = np.zeros_like(a)
        cin, out, _ = a.shape
        for j in range(stride):
            o[rng.integers(0, cin, out), np.arange(out), j] = near_one(out)
        return o

    for i in range(2):
        w["up_w"][i] = tconv(w["up_w"][i], 2)
        w["up_b"][i] = np.zeros_like(w["up_b"][i])
        w["gamma"][i] = np.zeros_like(w["gamma"][i])
    D, L, _ = w["conv0_w"].shape
    w["conv0_w"] = np.zeros_like(w["conv0_w"])
    w["conv0_w"][np.arange(D), rng.integers(0, L, D), 6] = near_one(D)
    w["conv0_b"] = np.zeros_like(w["conv0_b"])
    for b, rate in zip(w["block"], synth.CODEC_RATES):
        b["up_w"], b["up_b"] = tconv(b["up_w"], rate), np.zeros_like(b["up_b"])
        b["act_beta"] = np.full_like(b["act_beta"], 80)
        for r in b["res"]:
            for k in ("c1_w", "c1_b", "c2_w", "c2_b"):
                r[k] = np.zeros_like(r[k])
            for k in ("a1_beta", "a2_beta"):
                r[k] = np.full_like(r[k], 80)
    w["out_beta"] = np.full_like(w["out_beta"], 80)
    w["out_w"], w["out_b"] = np.zeros_like(w["out_w"]), np.zeros_like(w["out_b"])
    w["out_w"][0, 3, 6] = 1
    return w


@pytest.mark.parametrize("frames", [1, 16])
def test_codec_one_term_products(device, frames):
    """Seven products of one term each against float64, in the kernels of short
    and of long calls: at most 2 x 2^-24 each (rounding; the part products left
    out), 6.6e-8 together (RMS, seven roundings of 2.5e-8) with a mean of 0; 1e-7
    and 5e-8 leave the dropped parts theirs (parts cut off instead of rounded:
    4.3e-7, mean -4e-7)."""
    rng = np.random.default_rng(3)
    w = _one_term_weights(rng)
    x = rng.uniform(0.3, 0.7, (frames, 1024)).astype(np.float32)
    y = _gpu(device, w, x, [frames])
    ref = codec_torch.back(w, x)
    e = (y - ref) / ref
    mean, rms, top = abs(e.mean()), np.sqrt((e ** 2).mean()), abs(e).max()
    print(f"mean {mean:.2e} rms {rms:.2e} max {top:.2e}", flush=True)
    assert top <= 14 * 2.0 ** -24 and rms < 1e-7 and mean < 5e-8, (mean, rms, top)


def test_codec_large_snake_arguments(device):
    """SnakeBeta of arguments up to 1e6, on both sides of the change to sinf
    (4e5) and next to multiples of pi: the second SnakeBeta of block 0's first
    residual unit sees a bias V alone, z = V + ib sin(V)^2 with ib = 3.3e8, and
    its product takes 1e-9 z of one channel on, which reaches the samples through
    products by 1. The samples 1e-9 V + 0.33 sin(V)^2 within 1e-6 (about 12
    roundings of 2^-24 each)."""
    rng = np.random.default_rng(4)
    w = _one_term_weights(rng)
    for i, b in enumerate(w["block"]):
        b["up_w"] = np.zeros_like(b["up_w"])
        if i == 0:
            continue
        cin, out, k = b["up_w"].shape  # output channel o, phase j: input channel k o / 2 + j
        for j in range(k // 2):
            b["up_w"][(np.arange(out) * (k // 2) + j) % cin, np.arange(out), j] = 1
    r = w["block"][0]["res"][0]
    C = r["c1_b"].size
    v = np.exp(rng.uniform(0, np.log(1e6), C))
    v[::3] = np.arange(1, v[::3].size + 1) * 313 * np.pi  # to 2.5e5
    v = np.where(rng.random(C) < 0.5, -v, v).astype(np.float32)
    r["c1_b"] = v
    r["a2_alpha"], r["a2_beta"] = np.zeros_like(r["a2_alpha"]), np.full_like(r["a2_beta"], -20)
    r["c2_w"] = np.zeros_like(r["c2_w"])
    r["c2_w"][np.arange(C), np.arange(C), 0] = 1e-9
    y = _gpu(device, w, np.zeros((1, 1024), np.float32), [1])
    ref = codec_torch.back(w, np.zeros((1, 1024), np.float32))
    ib = 1 / (np.exp(-20) + 1e-9)
    seen = np.unique(ref.round(9)).size
    print(f"{seen} values, peak {ref.max():.3f}, max error {abs(y - ref).max():.2e}")
    assert seen >= 50 and 0.1 < ref.max() <= 1.1e-9 * ib
    assert abs(y - ref).max() <= 1e-6 * ref.max()


def test_codec_reset_and_errors(device, weights):
    x = synth.prompt(5, 2)
    c = q3h.Codec(device, weights, max_frames=4)
    try:
        a = c.back(x)
        b = c.back(x)
        assert not np.array_equal(a, b)  # the histories carry the first call
        c.reset()
        assert np.array_equal(c.back(x), a)
        assert c.back(np.zeros((0, 1024), np.float32)).shape == (0,)
        assert c.bytes > 100 * 1024 * 1024
    finally:
        c.destroy()
    bad = dict(weights)
    bad["conv0_w"] = None
    with pytest.raises(q3h.Q3HError) as e:
        q3h.Codec(device, bad)
    assert e.value.code == q3h.E_ARG and "NULL" in str(e.value)
    with pytest.raises(q3h.Q3HError) as e:
        q3h.Codec(device, weights, max_frames=0)
    assert e.value.code == q3h.E_ARG
