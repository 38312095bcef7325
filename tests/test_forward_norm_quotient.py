"""The f32 form of the int8 RMSNorm's quotient (rmsnorm_lane in forward.hip) equals the truncating
integer division for every input, with 1 / rms also one ulp off."""
import numpy as np


def test_quotient_exact():
    x = np.arange(-128, 129, dtype=np.int64)
    for rms in range(1, 129):
        want = np.sign(x) * (np.abs(x) * 48 // rms)
        inv0 = np.float32(1) / np.float32(rms)
        for inv in (inv0, np.nextafter(inv0, np.float32(0)), np.nextafter(inv0, np.float32(2))):
            m48 = np.float32(48) * inv
            half = np.copysign(np.float64(np.float32(0.5) * inv), np.where(x == 0, 1.0, x))
            f = (x.astype(np.float64) * np.float64(m48) + half).astype(np.float32)  # the fma's one rounding
            assert np.array_equal(np.trunc(f).astype(np.int64), want), rms
