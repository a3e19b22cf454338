"""kairos_gdn_chunk_fwd_noalloc: the forward entry point that allocates nothing.

It takes its scratch memory from the library's static device array instead of
a caller workspace.  The GPU test calls it through the C ABI twice in a row,
the second time on a smaller problem (so the array still holds the first
call's contents), and checks each result bit-for-bit against
kairos_gdn_chunk_fwd with a freshly allocated workspace on the same inputs.  The cases cover each way the
forward carves the array: the segment scan (bf16, K = V <= 128), the staged
kernels at the model head dims (bf16, K = 256, V = 512, one part: no library
streams) and the staged in-op L2 norm (fp32, K = V = 64), whose normalised q
and k sit at the front of the array.
The CPU test checks that a problem larger than the array is refused before
any GPU work.
"""
import numpy as np
import pytest
import torch

from kairos_gdn import _lib
from gdn_inputs import make_inputs


def _problem(B, T, H, K, V, seed, cu=None, dtype="bf16", l2=0):
    n_states = len(cu) - 1 if cu else B
    x = make_inputs(B, T, H, K, V, seed=seed, dtype=dtype, n_states=n_states)
    if l2:                                   # unnormalised q, k: the op normalises them
        rng = np.random.default_rng(seed + 1)
        for n in ("q", "k"):
            x[n] = x[n] * rng.uniform(0.5, 3.0, x[n].shape[:-1] + (1,)).astype(np.float32)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    dev = lambda a, dt: torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt)  # noqa: E731
    d = dict(q=dev(x["q"], tdt), k=dev(x["k"], tdt), v=dev(x["v"], tdt), g=dev(x["g"], torch.float32),
             beta=dev(x["beta"], tdt), h0=dev(x["h0"], torch.float32))
    d["cu"] = torch.tensor(cu, dtype=torch.int64, device="cuda") if cu else None
    d["shape"] = (B, T, H, K, V, n_states)
    d["dt"] = _lib.BF16 if dtype == "bf16" else _lib.F32
    d["l2"] = l2
    return d


def _run(d, noalloc):
    B, T, H, K, V, N = d["shape"]
    n_seqs = N if d["cu"] is not None else 0
    o = torch.full_like(d["v"], float("nan"))
    ht = torch.full((N, H, K, V), float("nan"), dtype=torch.float32, device="cuda")
    P = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    sp = torch.cuda.current_stream().cuda_stream
    dt = d["dt"]
    args = (P(d["q"]), P(d["k"]), P(d["v"]), P(d["g"]), P(d["beta"]), None, None, P(d["h0"]), P(o), P(ht),
            P(d["cu"]), n_seqs, B, T, H, K, V, dt, dt, _lib.F32, dt, _lib.F32, K ** -0.5, d["l2"])
    if noalloc:
        _lib.call("kairos_gdn_chunk_fwd_noalloc", *args, sp)
    else:
        lib = _lib.load()
        wsb = lib.kairos_gdn_chunk_fwd_workspace_size(B, T, H, K, V, n_seqs, dt, dt, d["l2"])
        ws = torch.empty(max(wsb, 1), dtype=torch.uint8, device="cuda")
        _lib.call("kairos_gdn_chunk_fwd", *args, P(ws), wsb, sp)
    torch.cuda.synchronize()
    return o, ht


@pytest.mark.gpu
def test_noalloc_matches_chunk_fwd_on_two_calls(monkeypatch):
    monkeypatch.setenv("KAIROS_GDN_WIDE_PIPE", "4")      # chunk_fwd in parts at K = 256, noalloc always in one
    cases = [
        ("B=2 T=3000 H=4 K=V=128 (several segments per sequence)", _problem(2, 3000, 4, 128, 128, seed=71)),
        ("varlen T=700 H=2 K=V=64, cu=[0, 1, 300, 700] (smaller)",
         _problem(1, 700, 2, 64, 64, seed=72, cu=[0, 1, 300, 700])),
        ("model head dims B=1 T=1100 H=2 K=256 V=512 (staged, fused recurrence)",
         _problem(1, 1100, 2, 256, 512, seed=73)),
        ("fp32 K=V=64 with the in-op L2 norm, varlen T=400 (staged, normalised q/k at the array's front)",
         _problem(1, 400, 2, 64, 64, seed=74, cu=[0, 150, 151, 400], dtype="fp32", l2=1)),
        ("bf16 K=V=128 with the in-op L2 norm T=500 (segment scan, smaller)", _problem(1, 500, 2, 128, 128, seed=75,
                                                                                      l2=1)),
    ]
    for name, d in cases:
        print(f"noalloc vs chunk_fwd: {name}", flush=True)
        o_n, h_n = _run(d, noalloc=True)
        o_w, h_w = _run(d, noalloc=False)
        assert torch.isfinite(o_n.float()).all() and torch.isfinite(h_n).all()
        assert torch.equal(o_n, o_w), name
        assert torch.equal(h_n, h_w), name


def test_noalloc_refuses_problems_beyond_the_static_array():
    lib = _lib.load()
    cap = lib.kairos_gdn_chunk_fwd_noalloc_max_bytes()
    assert cap == 256 << 20
    B, T, H, K, V = 1, 8 * 32760, 20, 128, 128
    assert lib.kairos_gdn_chunk_fwd_workspace_size(B, T, H, K, V, 0, _lib.BF16, _lib.BF16, 1) > cap
    x = 16  # any 16-byte aligned non-null address: the size check fails before anything is dereferenced
    rc = lib.kairos_gdn_chunk_fwd_noalloc(x, x, x, x, x, None, None, None, x, None, None, 0, B, T, H, K, V,
                                          _lib.BF16, _lib.BF16, _lib.F32, _lib.BF16, _lib.F32, K ** -0.5, 1, None)
    assert rc == _lib.EWORKSPACE
    assert b"static" in lib.kairos_gdn_last_error()


def test_noalloc_refuses_packed_batches_beyond_the_static_array():
    """Four packed sequences that fit the array with neither plan of segments."""
    lib = _lib.load()
    x, H, K = 16, 20, 128
    rc = lib.kairos_gdn_chunk_fwd_noalloc(x, x, x, x, x, None, None, None, x, None, x, 4, 1, 90000, H, K, K, _lib.BF16,
                                          _lib.BF16, _lib.F32, _lib.BF16, _lib.F32, K ** -0.5, 0, None)
    assert rc == _lib.EWORKSPACE
    assert b"static" in lib.kairos_gdn_last_error()


@pytest.mark.gpu
def test_noalloc_packed_batch_that_fits_with_fewer_segments(monkeypatch):
    """A packed batch whose workspace exceeds the array runs with the longer segments that fit: the bits of
    chunk_fwd cut that way."""
    monkeypatch.delenv("KAIROS_GDN_SEG_CHUNKS", raising=False)
    lib = _lib.load()
    H, K = 20, 128
    cu = [0, 3000, 21000, 26500, 66000]
    T, N = cu[-1], len(cu) - 1
    cap = lib.kairos_gdn_chunk_fwd_noalloc_max_bytes()
    assert lib.kairos_gdn_chunk_fwd_workspace_size(1, T, H, K, K, N, _lib.BF16, _lib.BF16, 0) > cap
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    bound = T // 64 + N                                  # all segments of the longer plan fit the CUs at once
    longer = -(-bound * H // max(cus - N * H, cus // 2))
    assert longer > lib.kairos_gdn_segment_chunks(1, T, H, N)
    print(f"noalloc packed batch T={T} H={H} K=V={K}, segments of {longer}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *sh: torch.randn(*sh, device="cuda", generator=gen)  # noqa: E731
    unit = lambda t: (t / t.norm(dim=-1, keepdim=True)).to(torch.bfloat16)  # noqa: E731
    d = dict(q=unit(r(1, T, H, K)), k=unit(r(1, T, H, K)), v=r(1, T, H, K).to(torch.bfloat16), g=-0.02 * r(1, T, H).abs(),
             beta=torch.sigmoid(r(1, T, H)).to(torch.bfloat16), h0=0.02 * r(N, H, K, K),
             cu=torch.tensor(cu, device="cuda"), shape=(1, T, H, K, K, N), dt=_lib.BF16, l2=0)
    o, ht = _run(d, noalloc=True)
    short, _ = _run(d, noalloc=False)
    monkeypatch.setenv("KAIROS_GDN_SEG_CHUNKS", str(longer))
    want, ht_want = _run(d, noalloc=False)
    assert torch.isfinite(o.float()).all() and torch.isfinite(ht).all()
    assert torch.equal(o, want) and torch.equal(ht, ht_want)
    assert not torch.equal(o, short)                     # the packed plan's segments give other roundings
