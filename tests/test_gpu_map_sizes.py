"""AdaptiveMap kernels at the edges of their tiles, scans and LDS plans,
against the FP64 oracle (the bars of test_gpu_map.py: histograms bit for bit,
exact adapts 1e-13 relative)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def va():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import vegas_amd
    return vegas_amd


@pytest.mark.parametrize("old,new", [(1, 5), (2, 3), (3, 64), (63, 65), (64, 64), (65, 63), (1000, 1),
                                     (1000, 1000), (129, 3072), (3072, 129), (3073, 70)])
@pytest.mark.parametrize("alpha", [0.0, 0.7])
def test_adapt_exact_sizes(va, orc, old, new, alpha):
    rng = np.random.default_rng(old + new)
    m, o = va.AdaptiveMap([[0, 1], [-2, 3]], ninc=old), orc.OracleMap([[0, 1], [-2, 3]], ninc=[old, old])
    y = rng.uniform(0, 1, (4000, 2))
    f = np.exp(rng.normal(0, 3, 4000)) * (y[:, 0] > 0.3)  # empty bins among them
    for q in (m, o):
        q.add_training_data(y, f)
        q.adapt(alpha=alpha, ninc=np.array([new, new]))
    np.testing.assert_allclose(m.grid[:, :new + 1], o.grid[:, :new + 1], rtol=1e-13, atol=1e-13)
