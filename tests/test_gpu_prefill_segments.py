"""GPU parity of M-run segments at every length of the finish's scan: one to eight
segments per sequence, sequences of different segment counts in one call, and
heads that stop early beside heads that never do.  The plan header in the
workspace (word 2: segment length, word 11: most segments) shows what was run.
Bar: the oracle tolerances of gpu_util."""

import pytest
import torch

from gpu_util import assert_parity
from kachua_mlsys_amd import prefill
from kachua_mlsys_amd.inputs import prefill_inputs_from_lengths
from oracle.gdn_oracle import prefill_ref

pytestmark = pytest.mark.gpu

CASES = {
    "700, whole": ([700], "near-1", {1}),
    "2 x 600": ([600, 580, 720], "near-1", {1, 2}),
    "1 x 1000": ([1000], "near-1", {2, 3}),
    "2000 and shorter": ([2000, 640, 70, 0, 1300], "near-1", {2, 3, 4}),
    "1 x 2000": ([2000], "near-1", {3, 4}),
    "1 x 2000, mixed": ([2000], "mixed", {3, 4}),
    "1 x 4100, mixed": ([4100], "mixed", {4, 5, 6}),
    "1 x 7000": ([7000], "near-1", {5, 6, 7, 8}),
}


def planned(ws, N, T):
    """(segment length, most segments) of the call that used the workspace ws."""
    def a256(x):
        return (x + 255) // 256 * 256
    R = (T + 63) // 64 + N
    off = a256(R * 8 * 6 * 512 * 2)
    off = a256(off + R * 8 * 256 * 4)
    off = a256(off + (N + 1) * 4)
    h = ws[off:off + 64].view(torch.int32)
    return int(h[2]), int(h[11])


@pytest.mark.parametrize("name", list(CASES))
def test_mrun_segments(gpu, name):
    lengths, decay, expect = CASES[name]
    p = prefill_inputs_from_lengths(lengths, seed=77 + sum(lengths) % 89)
    p.A_log = torch.linspace(-8.0, -5.0, 8) if decay == "near-1" else torch.linspace(-7.0, 1.0, 8)
    print(f"[case] segments {name}", flush=True)
    _, s_ref, o32 = prefill_ref(*p.args(), return_fp32_out=True)
    N, T = len(lengths), sum(lengths)
    ws = torch.empty(prefill.workspace_bytes(N, T), dtype=torch.uint8, device=gpu)
    out, ns = prefill.launch_gdn(*p.to(gpu).args(), workspace=ws)
    torch.cuda.synchronize()
    L, nseg = planned(ws, N, T)
    print(f"[segments] {name}: {nseg} of {L} chunks", flush=True)
    assert_parity(out, ns, o32, s_ref, f"segments {name}")
    assert nseg in expect, f"{name}: {nseg} segments of {L} chunks"
