"""The codecs' wave kernels (16-byte aligned buffers) against the oracle, byte
for byte: one block, a wave's 64 blocks and a work-group's 256 with one block
less and more, values on and beside every rounding boundary of their block,
and blocks of zeros, subnormals, infinities and NaN; and the same values at an
unaligned address, which the thread-per-block kernels take."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(nb, top, seed):
    rng = np.random.default_rng(seed)
    v = (rng.standard_normal((nb, 32)) * 0.02).astype(np.float32)
    for b in range(0, nb, 3):  # largest value top * s: half steps of s and their neighbours
        s = np.float32(rng.choice([1.0, 0.25, 0.013, 3e-5, 7.7e4, 1e-39]))
        k = (rng.integers(-2 * top, 2 * top + 1, 32) * 0.5).astype(np.float32) * s
        step = rng.integers(-1, 2, 32)
        k = np.where(step > 0, np.nextafter(k, np.float32(np.inf)),
                     np.where(step < 0, np.nextafter(k, np.float32(-np.inf)), k))
        k[rng.integers(32)] = np.float32(top) * s
        v[b] = k
    special = [np.float32(0), np.float32(-0.0), np.float32(np.nan), np.float32(np.inf),
               np.float32(-np.inf), np.float32(1e-45), np.float32(3e38)]
    for b in range(1, nb, 5):
        for at in rng.integers(0, 32, 2):
            v[b, at] = special[rng.integers(len(special))]
    if nb > 2:
        v[2] = 0.0
    return v.ravel()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("nb", [1, 63, 64, 65, 255, 256, 257, 2111])
@pytest.mark.parametrize("dt", ["q4_0", "q8_0"])
def test_codec_wave(orc, dt, nb, shift):
    import torch

    import hypno_amd as hk
    print(f"{dt} blocks={nb} shift={shift}", flush=True)
    v = _values(nb, 7 if dt == "q4_0" else 127, nb)
    buf = torch.empty(v.size + shift, dtype=torch.float32, device="cuda")
    x = buf[shift:]
    x.copy_(torch.from_numpy(v))
    quant, dequant, oq, od = {
        "q4_0": (hk.quantize_f32_to_q4_0, hk.dequantize_q4_0, orc.quantize_q4_0,
                 orc.dequantize_q4_0),
        "q8_0": (hk.quantize_f32_to_q8_0, hk.dequantize_q8_0, orc.quantize_q8_0,
                 orc.dequantize_q8_0)}[dt]
    q = quant(x).cpu().numpy()
    ref = oq(v)
    assert np.array_equal(q, ref), np.flatnonzero(q != ref)[:8]
    packed = torch.empty(ref.size + 2 * shift, dtype=torch.uint8, device="cuda")
    packed[2 * shift:] = torch.from_numpy(ref).cuda()
    back = dequant(packed[2 * shift:]).cpu().numpy()
    assert np.array_equal(back.view(np.uint32), od(ref).view(np.uint32))
