"""The matrix-core router (router_mfma_kernel): logits bit-equal to the oracle's fixed-order sums
for every row length it takes, ragged token and expert tiles, values whose products are
subnormal, infinities and NaN, and the calls just below its size.  Rows of more than 4096 values take
the LDS-tiled kernel (router_gemm_kernel) at these sizes: J = 9 and 10, ragged in tokens and experts."""

import numpy as np
import pytest

import oracle
from gpu_helpers import log

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _logits(x, w, b):
    from pgmoe import ops
    dev = torch.device("cuda", 0)
    bt = None if b is None else torch.from_numpy(b).to(dev)
    return ops.router_topk(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), bt, 2, True)[0].cpu().numpy()


# 24576 logits is the smallest call that takes it: M = 191 / 192 at 128 experts, 1445 / 1446 at 17; from
# J = 5 on 32768: M = 511 / 512 at 64 experts, 63 / 64 at 512
@pytest.mark.parametrize("J,E,M,bias", [(1, 128, 192, True), (2, 40, 1000, False), (3, 17, 1446, True),
                                        (3, 17, 1445, True), (4, 128, 191, False), (4, 128, 301, True),
                                        (5, 64, 385, False), (6, 512, 49, True), (7, 64, 500, False),
                                        (8, 16, 1537, True), (4, 128, 4111, False), (5, 64, 511, True),
                                        (5, 64, 512, True), (6, 512, 63, False), (6, 512, 64, True),
                                        (7, 100, 331, False), (8, 16, 2049, True), (9, 128, 2060, True),
                                        (10, 100, 2600, False)])
def test_bit_exact(J, E, M, bias):
    log(f"router mfma J={J} E={E} M={M}")
    rng = np.random.default_rng(1000 * J + E + M)
    x = rng.standard_normal((M, 512 * J)).astype(np.float16)
    w = (rng.standard_normal((E, 512 * J)) * 0.02).astype(np.float32)
    b = rng.standard_normal(E).astype(np.float32) if bias else None
    assert np.array_equal(_logits(x, w, b), oracle.router_logits(x, w, b))


def test_subnormal_and_non_finite():
    rng = np.random.default_rng(7)
    x = (rng.standard_normal((200, 2048)) * 1e-6).astype(np.float16)  # fp16 subnormals
    w = (rng.standard_normal((128, 2048)) * 1e-34).astype(np.float32)  # every product subnormal (below 2^-126)
    ref = oracle.router_logits(x, w, None)
    assert np.abs(x).max().astype(np.float64) * np.abs(w).max() < 2.0 ** -126 and np.count_nonzero(ref)
    assert np.array_equal(_logits(x, w, None), ref)
    x[3, 5], x[17, 700], w[9, 33] = np.inf, -np.inf, np.nan
    assert np.array_equal(_logits(x, w, None), oracle.router_logits(x, w, None), equal_nan=True)
