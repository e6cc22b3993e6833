"""quantizeFeaturesInt8 of widths that are not a multiple of 4: tiles of rows through LDS, or one wave per row
where there are few rows."""
import numpy as np
import pytest

from gpu_cases import features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (1, 5), (3, 6), (4, 7), (5, 50), (1030, 50), (4099, 17), (1025, 277),  # one wave per row
    (7168, 5), (10240, 33), (12288, 95), (14336, 255), (10239, 319), (2049, 321), (8192, 543),  # the most (fewest) such rows
    (7169, 31), (10241, 47), (12289, 49), (14337, 97), (10241, 319), (2048, 321), (8193, 543),  # and tiles beyond them
    (20003, 17), (70001, 50), (20011, 50), (66003, 5),        # tiles of 64, 64, 32 and 256 rows
    (1025, 601), (9, 1023), (7, 1025), (5, 2047), (1, 602),   # up to the largest width
    (6, 2049), (9, 3),                                        # past either end: one wave per row
])
def test_quantize_any_width_bit_exact(oracle, gpu, shape):
    """Scales and bytes are the oracle's, rows that end inside a four-byte store included, and nothing
    is written past the last row."""
    import torch
    from tcc_spmm_amd.device import quantize_features_int8
    s, f = shape
    x = features(s, f, seed=s * 13 + f, stddev=2.0, outlier_fraction=0.1, outlier_scale=50.0)
    x[s // 2] = 0.0
    q = torch.full((s * f + 64,), 0x5A, dtype=torch.int8, device=gpu)
    scale = torch.full((s + 16,), -7.0, device=gpu)
    quantize_features_int8(torch.from_numpy(x).to(gpu), q[:s * f].view(s, f), scale[:s])
    q_ref, s_ref = oracle.quantize(x)
    assert np.array_equal(scale[:s].cpu().numpy().view(np.uint32), s_ref.view(np.uint32))
    assert np.array_equal(q[:s * f].cpu().numpy().reshape(s, f), q_ref)
    assert bool((q[s * f:] == 0x5A).all()) and bool((scale[s:] == -7.0).all())
