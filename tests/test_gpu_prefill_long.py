"""GPU checks of single sequences too long for the oracle's token loop, against the
same tokens run another way.

* An unsplit run of more than 4,096 chunks re-forms its copy resources on the
  way.  The same tokens as three calls of fewer chunks, the state carried between
  them, take the same steps: outputs and state are equal bit for bit.
* More than 64 segments in one sequence: the finish's scan reads the maps' flags
  in blocks of 63.  The planner only cuts so many where a segment's longest length
  (1,024 chunks) leaves it no choice, so the sequence has 4.3 million tokens.
  Against the unsegmented run to the tolerances of gpu_util.
"""

import pytest
import torch

from gpu_util import OUT_ATOL, OUT_RTOL, STATE_REL
from kachua_mlsys_amd import prefill

pytestmark = pytest.mark.gpu


def _inputs(T, gpu, seed, A_log):
    """Inputs of one sequence of T tokens, made on the GPU in slices."""
    g = torch.Generator(gpu).manual_seed(seed)
    t = {n: torch.empty((T, h) + d, dtype=torch.bfloat16, device=gpu)
         for n, h, d in (("q", 4, (128,)), ("k", 4, (128,)), ("v", 8, (128,)), ("a", 8, ()), ("b", 8, ()))}
    for i in range(0, T, 1 << 18):
        for n, x in t.items():
            r = torch.randn(x[i:i + (1 << 18)].shape, generator=g, device=gpu)
            x[i:i + (1 << 18)] = torch.nn.functional.normalize(r, dim=-1) if n in "qk" else r
    t["state"] = 0.02 * torch.randn((1, 8, 128, 128), generator=g, device=gpu)
    t["A_log"] = A_log.to(gpu)
    t["dt_bias"] = 0.1 * torch.randn(8, generator=g, device=gpu)
    return t


def _run(t, lo, hi, state, out, ws):
    cu = torch.tensor([0, hi - lo], dtype=torch.int32, device=out.device)
    ns = torch.empty_like(t["state"])
    prefill.launch_gdn(t["q"][lo:hi], t["k"][lo:hi], t["v"][lo:hi], state, t["A_log"], t["a"][lo:hi], t["dt_bias"],
                       t["b"][lo:hi], cu, None, out[lo:hi], ns, workspace=ws)
    torch.cuda.synchronize()
    return ns


def test_unsplit_run_past_the_copy_resources(gpu):
    T = 2 * 4096 * 64 + 2 * 64 + 17   # re-formed twice, a partial last chunk
    print(f"[case] unsplit {T}", flush=True)
    t = _inputs(T, gpu, 3, torch.linspace(-7.0, 1.0, 8))
    ws = torch.empty(prefill.workspace_min_bytes(1, T), dtype=torch.uint8, device=gpu)   # no segments
    whole, parts = torch.empty_like(t["v"]), torch.empty_like(t["v"])
    ns = _run(t, 0, T, t["state"], whole, ws)
    s = t["state"]
    cuts = [0, 3000 * 64, 6500 * 64, T]
    for lo, hi in zip(cuts, cuts[1:]):
        s = _run(t, lo, hi, s, parts, ws[:prefill.workspace_min_bytes(1, hi - lo)])
    assert torch.isfinite(whole).all() and torch.equal(whole, parts)
    assert torch.equal(ns, s)


def test_more_than_64_segments(gpu):
    T = 65 * 1024 * 64 + 70 * 64 + 5
    print(f"[case] 66 segments, {T} tokens", flush=True)
    t = _inputs(T, gpu, 4, torch.linspace(-9.0, -6.0, 8))
    ws = torch.empty(prefill.workspace_bytes(1, T) + (24 << 20), dtype=torch.uint8, device=gpu)   # some slots more
    cut, whole = torch.empty_like(t["v"]), torch.empty_like(t["v"])
    ns = _run(t, 0, T, t["state"], cut, ws)
    R = (T + 63) // 64 + 1

    def a256(x):
        return (x + 255) // 256 * 256
    off = a256(R * 8 * 6 * 512 * 2)
    off = a256(off + R * 8 * 256 * 4)
    off = a256(off + 8)
    h = ws[off:off + 64].view(torch.int32).tolist()
    print(f"[segments] {h[11]} of {h[2]} chunks", flush=True)
    ns_whole = _run(t, 0, T, t["state"], whole, ws[:prefill.workspace_min_bytes(1, T)])
    rel = float((ns - ns_whole).abs().max() / ns_whole.abs().max())
    print(f"[parity] state_rel={rel:.3e}", flush=True)
    assert rel <= STATE_REL
    for i in range(0, T, 1 << 18):
        x, y = cut[i:i + (1 << 18)].float(), whole[i:i + (1 << 18)].float()
        assert torch.isfinite(x).all()
        assert torch.allclose(x, y, atol=OUT_ATOL, rtol=OUT_RTOL), f"tokens from {i}"
    assert h[2] == 1024 and h[11] == 66
