"""DN_PREPASS_SCALAR=0 forces the general phases in every prefill form."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# one decay and one b per token, and the same spread over the channels: the
# general phases repeat a one-channel gate, so their results are the same bits,
# while the scalar phases round elsewhere
CODE = """
import sys
sys.path.insert(0, "deltanet-tpu_amd")
import torch
from deltanet_tpu_amd import chunk_gdn2
gen = torch.Generator(device="cuda").manual_seed(0)
rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")
L, H, chans = int(sys.argv[1]), 2, int(sys.argv[2])
q, k, v = (rn(1, L, H, 128).bfloat16() for _ in range(3))
g, b, w = -torch.exp(rn(1, L, H, 1) - 1), torch.sigmoid(rn(1, L, H, 1)), torch.sigmoid(rn(1, L, H, chans))
spread = lambda t: t.expand(1, L, H, 128)
run = lambda g, b: chunk_gdn2(q, k, v, g, b, w, output_final_state=True, qk_l2norm=True, is_inference=True)
one, full = run(g, b), run(spread(g), spread(b))
print("same" if all(torch.equal(x, y) for x, y in zip(one, full)) else "different", flush=True)
"""


# the scan, and the long form with one or 128 write gates per token
@pytest.mark.parametrize("L,chans", [(200, 1), (6144, 1), (6144, 128)])
def test_switch(L, chans):
    said = {}
    for value in ("0", None):
        env = {k: x for k, x in os.environ.items() if k != "DN_PREPASS_SCALAR"}
        if value is not None:
            env["DN_PREPASS_SCALAR"] = value
        r = subprocess.run([sys.executable, "-c", CODE, str(L), str(chans)], cwd=ROOT, env=env, capture_output=True,
                           text=True, timeout=100)
        assert r.returncode == 0, r.stderr
        said[value] = r.stdout.split()[-1]
    assert said == {"0": "same", None: "different"}
