"""GPU parity of the direct path and of the mixed launch at the edges of their
rules.  Direct: calls of at most 256 tokens and 64 sequences.  Mixed: longer
calls of at most 32 sequences and 64 tokens per sequence on average, whose
sequences of at most four chunks (256 tokens) run directly while the planner and
the prepass take the longer ones: three- and four-chunk sequences beside five-
and eight-chunk ones, together and among short ones.  Beside them calls just past
either rule, which go through the planner.  Empty sequences, no state, int64
cu_seqlens, near-1 decay, and outputs and states that are views into larger
buffers.  Bar: the oracle tolerances of gpu_util."""

import pytest
import torch

from gpu_util import assert_parity
from kachua_mlsys_amd import prefill
from kachua_mlsys_amd.inputs import prefill_inputs_from_lengths
from oracle.gdn_oracle import prefill_ref

pytestmark = pytest.mark.gpu

CASES = {
    "256 tokens": ([256], {}),
    "257 tokens (planned)": ([257], {}),
    "255 and 1": ([255, 1], {"weak": True}),
    "three chunks, partial last": ([129], {"state_none": True}),
    "192, 0, 64": ([192, 0, 64], {"cu64": True}),
    "500 among twelve (mixed: planned beside short ones)": ([1] * 6 + [500] + [1] * 6, {}),
    "500 among twelve, near-1 (mixed)": ([1] * 6 + [500] + [1] * 6, {"weak": True}),
    "505 among seven ones (mixed)": ([505] + [1] * 7, {"state_none": True, "cu64": True}),
    "448, one and six empty (mixed)": ([448] + [0] * 6 + [1], {}),
    "449 tokens, seven empty (mixed)": ([449] + [0] * 7, {"weak": True}),
    "8 x 64 (mixed, all direct)": ([64] * 8, {}),
    "513 over eight (planned)": ([64] * 7 + [65], {}),
    "64 sequences of 8 (planned)": ([8] * 64, {}),
    "16-token tiles": ([15, 16, 17, 31, 33, 47, 49, 63, 65, 80], {}),
    "64 sequences of 4": ([4] * 64, {}),
    "192 to 320 (mixed, two planned)": ([192, 193, 256, 257, 320] + [3] * 20, {}),
    "192 to 320, near-1, no state": ([320, 257, 256, 193, 192] + [2] * 20, {"weak": True, "state_none": True}),
    "256 among short ones, near-1": ([60] * 4 + [256] + [50, 0, 70, 1] * 3, {"weak": True}),
    "257 among short ones": ([60] * 4 + [257] + [50, 0, 70, 1] * 3, {"cu64": True}),
    "193 alone among empty ones (mixed)": ([0, 0, 193, 0, 0, 128], {"state_none": True}),
    "32 sequences, one of 256": ([9] * 16 + [256] + [64] * 15, {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prefill_direct_rule(gpu, name):
    lengths, kw = CASES[name]
    p = prefill_inputs_from_lengths(lengths, seed=len(lengths) * 17 + sum(lengths) % 101,
                                    cu_dtype=torch.int64 if kw.get("cu64") else torch.int32)
    if kw.get("weak"):
        p.A_log = torch.linspace(-8.0, -5.0, 8)
    if kw.get("state_none"):
        p.state = None
    print(f"[case] direct {name}: {lengths[:10]}", flush=True)
    _, s_ref, o32 = prefill_ref(*p.args(), return_fp32_out=True)
    g = p.to(gpu)
    T, N = sum(lengths), len(lengths)
    buf = torch.full((T * 1024 + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
    out = buf[4:4 + T * 1024].view(T, 8, 128)
    ns_buf = torch.full(((N + 1) * 8 * 128 * 128,), 7.0, device=gpu)
    ns = ns_buf[4:4 + N * 8 * 128 * 128].view(N, 8, 128, 128)
    prefill.launch_gdn(*g.args(), out, ns)
    torch.cuda.synchronize()
    assert_parity(out, ns, o32, s_ref, f"direct {name}")
    assert (buf[:4] == 7.0).all() and (buf[-4:] == 7.0).all()
    assert (ns_buf[:4] == 7.0).all() and (ns_buf[4 + N * 8 * 128 * 128:] == 7.0).all()
