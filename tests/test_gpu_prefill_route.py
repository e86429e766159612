"""GPU parity of the planner's choice between the split and the wide consumer in
batches of more than 32 sequences: batches that each takes, with warm-up and
M-run segments, whole runs, single-chunk and empty sequences, and the plan
launch's batch sizes.  The plan header in the workspace (word 2: segment length,
word 11: most segments, word 12: 1 for the wide consumer) shows what was run.
Bar: the oracle tolerances of gpu_util."""

import pytest
import torch

from gpu_util import assert_parity
from kachua_mlsys_amd import prefill
from kachua_mlsys_amd.inputs import prefill_inputs_from_lengths
from oracle.gdn_oracle import prefill_ref

pytestmark = pytest.mark.gpu

SPLIT, WIDE = 0, 1
# lengths, decay, consumer, segmented
CASES = {
    "33 x 70": ([70] * 33, "near-1", WIDE, False),
    "65 single chunks": ([30] * 65, "fast", WIDE, False),
    "50 tokens over 100": ([1, 0] * 50, "fast", WIDE, False),
    "one token among 90": ([0] * 40 + [1] + [0] * 49, "near-1", SPLIT, False),
    "90 single chunks": ([30] * 89 + [0], "fast", SPLIT, False),
    "one of 640 among 48": ([20] * 20 + [640] + [20] * 27, "near-1", SPLIT, False),
    "16 of 500 among 34": ([9] * 18 + [500] * 16, "near-1", SPLIT, False),
    "two of 1,500 among 40": ([30] * 19 + [1500, 0, 1477] + [30] * 18, "near-1", SPLIT, True),
    "one of 2,000 among 120 x 100": ([100] * 60 + [2000] + [100] * 59, "near-1", WIDE, True),
    "two of 1,500 among 40, fast": ([30] * 19 + [1500, 0, 1477] + [30] * 18, "fast", WIDE, True),
    "540 sequences, one of 3,000": ([33] * 200 + [3000] + [65, 0, 17] * 113, "near-1", WIDE, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_consumer_route(gpu, name):
    lengths, decay, consumer, segmented = CASES[name]
    p = prefill_inputs_from_lengths(lengths, seed=41 + sum(lengths) % 83)
    if decay == "near-1":
        p.A_log = torch.linspace(-8.0, -5.0, 8)
    print(f"[case] route {name}", flush=True)
    _, s_ref, o32 = prefill_ref(*p.args(), return_fp32_out=True)
    N, T = len(lengths), sum(lengths)
    ws = torch.empty(prefill.workspace_bytes(N, T), dtype=torch.uint8, device=gpu)
    out, ns = prefill.launch_gdn(*p.to(gpu).args(), workspace=ws)
    torch.cuda.synchronize()

    def a256(x):
        return (x + 255) // 256 * 256
    R = (T + 63) // 64 + N
    off = a256(R * 8 * 6 * 512 * 2)
    off = a256(off + R * 8 * 256 * 4)
    off = a256(off + (N + 1) * 4)
    h = ws[off:off + 64].view(torch.int32).tolist()
    print(f"[route] {name}: {'wide' if h[12] else 'split'}, {h[11]} segments of {h[2]} chunks", flush=True)
    assert_parity(out, ns, o32, s_ref, f"route {name}")
    assert h[12] == consumer
    assert (h[11] > 1) == segmented
