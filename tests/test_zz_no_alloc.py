"""rppt_logmel_fused_noalloc_gpu through the C-ABI against rppt_logmel_fused_gpu.

The no-allocation entry point runs the same kernels with its tables and workspace in the library's
own device array, so its output must equal the allocating entry point's bit for bit.  Each case
makes two calls in a row, the second with a smaller batch (the array keeps the first call's plan
and records, which the second must not read), and the parameter sets alternate so the tables are
rebuilt in place between cases.
"""
import numpy as np
import pytest
import torch

from rpp_amd import synth

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def params_for(gpu, feat, **kw):
    return gpu.logmel_params(nfft=feat["nfft"], window_length=feat["W"], window_step=feat["H"],
                             sample_rate=feat["sample_rate"], min_freq=feat["fmin"], max_freq=feat["fmax"],
                             num_filter=feat["nmel"], **kw)


def both(gpu, h, bt, n, precision, **kw):
    x, L = bt.x[:n], bt.lengths[:n]
    feat = bt.params
    frames = L // feat["H"] + 1
    hs = int(frames.max())
    p = params_for(gpu, feat, **kw)
    xs, Ls = dev(x), dev(L)
    ref = torch.full((n, feat["nmel"], hs), float("nan"), device="cuda")
    out = torch.full((n, feat["nmel"], hs), float("nan"), device="cuda")
    gpu.logmel_fused(h, xs, ref, Ls, p, precision)
    gpu.logmel_fused_noalloc(h, xs, out, Ls, p, precision)
    torch.cuda.synchronize()
    return ref.cpu().numpy(), out.cpu().numpy(), frames


@pytest.mark.parametrize("precision", ["fp16x3", "fp32"])
@pytest.mark.parametrize("ref_mag", [1.0, 0.0])
def test_noalloc_equals_fused(gpu, handle, precision, ref_mag):
    w1 = synth.workload1(batch=96)
    w2 = synth.workload2(batch=12)
    for bt, sizes in ((w1, (96, 24)), (w2, (12, 5))):
        for n in sizes:
            print(f"noalloc: precision={precision} ref={ref_mag} nfft={bt.params['nfft']} clips={n}", flush=True)
            ref, out, frames = both(gpu, handle, bt, n, precision, reference_magnitude=ref_mag)
            for b, F in enumerate(frames):
                assert np.array_equal(out[b, :, :F], ref[b, :, :F]), (n, b)
                # nothing is written past a clip's frames
                assert np.isnan(out[b, :, F:]).all(), (n, b)


def test_noalloc_rejects_oversized_plan(gpu, handle):
    # 3M clips need a 24 MB tile plan, more than the 16 MiB array: refused before any launch
    bt = synth.workload0(batch=2)
    feat = bt.params
    p = params_for(gpu, feat)
    x, L = dev(bt.x), dev(bt.lengths)
    out = torch.zeros((2, feat["nmel"], 8), device="cuda")
    st = gpu.logmel_fused_noalloc(handle, x, out, L, p, "fp16x3", check_status=False, batch=3_000_000)
    assert st == -22  # RPP_ERROR_OUT_OF_BOUND_SCRATCH_MEMORY_SIZE
    torch.cuda.synchronize()


def test_noalloc_clip_reference_needs_no_more_room(gpu):
    """The most filters whose tables leave room for a batch's plan with a fixed reference leave room for its
    clip maxima too: a word per clip where a line per XCD does not fit."""
    rng = np.random.default_rng(3)
    B = 200
    L = rng.integers(200, 600, B).astype(np.int32)
    x = dev(rng.normal(0, 0.2, (B, 600)).astype(np.float32))
    h = gpu.Handle(B)

    def call(M, ref_mag, out):
        p = gpu.logmel_params(num_filter=M, reference_magnitude=ref_mag)
        return gpu.logmel_fused_noalloc(h, x, out, dev(L), p, "fp32", check_status=False)

    lo, hi = 1000, 16000                       # accepted, refused
    buf = torch.zeros((B, hi, 4), device="cuda")
    assert call(hi, 1.0, buf) == -22
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if call(mid, 1.0, buf) == 0 else (lo, mid)
    out, ref = torch.zeros((B, lo, 4), device="cuda"), torch.zeros((B, lo, 4), device="cuda")
    assert call(lo, 0.0, out) == 0, lo
    gpu.logmel_fused(h, x, ref, dev(L), gpu.logmel_params(num_filter=lo, reference_magnitude=0.0), "fp32")
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    h.close()
