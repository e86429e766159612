"""GPU parity of batches of many sequences around the wide consumer's range (half
a work-group per (run or short sequence, v-head)): 32 and 33 sequences (the
planner weighs it from 33 on), chunk and 16-token tile boundaries, empty sequences, warm-up and M-run segments beside
short sequences, no initial state, an output that is only 8-byte aligned, and
the plan launch's batches.  Bar: the oracle tolerances of gpu_util (fixed
there; the bounds on outputs and states of every prefill test)."""

import pytest
import torch

from gpu_util import assert_parity
from kachua_mlsys_amd import prefill
from kachua_mlsys_amd.inputs import prefill_inputs_from_lengths
from oracle.gdn_oracle import prefill_ref

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 127, 128, 129, 192, 193]


def _tile(n, extra=()):
    return ([EDGES[i % len(EDGES)] for i in range(n - len(extra))] + list(extra))[:n]


CASES = {
    "33 sequences": (_tile(33), {}),
    "32 sequences (split consumer)": (_tile(32), {}),
    "33 x 256 tokens": ([256] * 33, {}),
    "33 x 257 tokens": ([257] * 33, {}),
    "64 sequences, one long": (_tile(64, [1500]), {}),
    "63 sequences, one long": (_tile(63, [900]), {}),
    "70 sequences, near-1 decay": (_tile(70, [700, 1100]), {"weak": True}),
    "66 sequences, mixed decay": (_tile(66, [640, 900]), {"mixed": True}),
    "40 sequences, no state, int64": (_tile(40), {"state_none": True, "cu64": True}),
    "64 empty and one token": ([0] * 63 + [1], {}),
    "600 sequences (plan launch)": (_tile(600, [400]), {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prefill_wide(gpu, name):
    lengths, kw = CASES[name]
    p = prefill_inputs_from_lengths(lengths, seed=len(lengths) * 13 + sum(lengths) % 97,
                                    cu_dtype=torch.int64 if kw.get("cu64") else torch.int32)
    if kw.get("weak"):
        p.A_log = torch.linspace(-8.0, -5.0, 8)
    if kw.get("mixed"):
        p.A_log = torch.linspace(-7.0, 1.0, 8)
    if kw.get("state_none"):
        p.state = None
    print(f"[case] wide {name}: T={sum(lengths)}", flush=True)
    _, s_ref, o32 = prefill_ref(*p.args(), return_fp32_out=True)
    g = p.to(gpu)
    T, N = sum(lengths), len(lengths)
    # outputs inside larger buffers: 8-byte aligned rows (16-byte stores must
    # not assume more), and the elements around them stay as they were
    buf = torch.full((T * 1024 + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
    out = buf[4:4 + T * 1024].view(T, 8, 128)
    ns = torch.full((N, 8, 128, 128), float("nan"), device=gpu)
    prefill.launch_gdn(*g.args(), out, ns)
    torch.cuda.synchronize()
    assert_parity(out, ns, o32, s_ref, f"wide {name}")
    assert (buf[:4] == 7.0).all() and (buf[-4:] == 7.0).all()
