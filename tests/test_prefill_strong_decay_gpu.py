"""Prefill with a very large decay at the first token of every chunk: the pairs
behind it keep their own decays to float32 accuracy."""

import numpy as np
import pytest

from deltanet_tpu_amd import chunk_gdn2
from tests.gpu_common import as_np, oracle_prefill, to_dev
from tests._util import rel_frob, rel_l2, sig

pytestmark = pytest.mark.gpu


# the 64-token scan and the 128-token form, one decay per token or per channel.
# Lambda is kept to about 2^-47 of its size (two float32 words), 2e-8 in a decay
# of 2e6; float32 prefill is within 1e-6 of the oracle otherwise, 4e-6 the bound
# of both.  A decay that took 2e6 in one float32 word would be off by 2^-3.
@pytest.mark.parametrize("scalar", [True, False])
@pytest.mark.parametrize("L,chunk", [(200, 64), (4200, 128)])
def test_large_decay_at_chunk_starts(scalar, L, chunk):
    rng = np.random.default_rng(L)
    rn = rng.standard_normal
    Hk, Hv = 1, 2
    q, k, v = rn((1, L, Hk, 128)), rn((1, L, Hk, 128)), rn((1, L, Hv, 128))
    c = () if scalar else (128,)
    g = -0.05 * np.exp(rn((1, L, Hk) + c))
    g[:, ::chunk] = -1.5e6
    b, w = sig(rn((1, L, Hk) + c)), sig(rn((1, L, Hv) + c))
    q, k, v, g, b, w = (x.astype(np.float32) for x in (q, k, v, g, b, w))
    out, st = chunk_gdn2(*(to_dev(x) for x in (q, k, v, g, b, w)), output_final_state=True, qk_l2norm=True,
                         is_inference=True, precision="fp32")
    ro, rs = oracle_prefill(q, k, v, g, b, w, use_c=True, qk_l2norm=True)
    assert rel_l2(as_np(out), ro) < 4e-6 and rel_frob(as_np(st), rs) < 4e-6
