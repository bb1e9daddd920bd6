"""The mel filter bank's split of the filters into groups: banks with fewer filters than groups, with
empty filters (narrower than a bin), ending below and at half the rate, and frame counts around a wave.
Exact against the same FP32 products added in ascending order of the bins."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("bins,M,rate,fmin,fmax,formula,normalize,frames,clips", [
    (257, 80, 16000.0, 0.0, 8000.0, "slaney", True, (1, 63, 64, 65, 300), 1),
    (257, 3, 16000.0, 300.0, 3000.0, "htk", True, (2, 64), 1),
    (129, 1, 8000.0, 0.0, 4000.0, "slaney", False, (5, 129), 1),
    (33, 100, 16000.0, 0.0, 8000.0, "slaney", True, (7, 64), 1),        # more filters than bins: empty ones
    (1025, 128, 44100.0, 20.0, 16000.0, "htk", False, (66,), 1),
    (513, 128, 44100.0, 0.0, 22050.0, "slaney", True, (700, 129), 40)])   # enough waves for 8 groups
def test_mel_groups(gpu, handle, bins, M, rate, fmin, fmax, formula, normalize, frames, clips):
    rng = np.random.default_rng(bins + M)
    F = np.array(list(frames) * clips, np.int32)
    B, S = len(F), int(F.max()) + 3
    x = (rng.uniform(0, 1, (B, bins, S)) ** 4).astype(np.float32)
    out = torch.full((B, M, S), -7.0, device="cuda")
    dims = np.stack([np.full(B, bins), F], 1).reshape(-1).astype(np.int32)
    gpu.mel_filter_bank(handle, dev(x), out, dev(dims), max_freq=fmax, min_freq=fmin, formula=formula, num_filter=M,
                        sample_rate=rate, normalize=normalize)
    o = out.cpu().numpy()
    wd, iv, nf, rg = (np.zeros(bins, np.float32), np.zeros(bins, np.int32), np.zeros(M, np.float32), np.zeros(2, np.int32))
    assert gpu.lib().rppa_debug_mel_tables(handle.h, bins, rate, fmax, fmin, gpu.MEL[formula], M, int(normalize),
                                           *[C.c_void_p(a.ctypes.data) for a in (wd, iv, nf, rg)]) == 0
    ref = np.zeros((B, M, S), np.float32)
    for k in range(rg[0], rg[1]):
        for m, w in ((iv[k] - 1, wd[k]), (iv[k], np.float32(1) - wd[k])):
            if iv[k] >= 0 and 0 <= m < M:
                ref[:, m] = ref[:, m] + x[:, k] * (w * nf[m] if normalize else w)
    for b in range(B):
        assert np.array_equal(o[b, :, :F[b]], ref[b, :, :F[b]]), b
        assert np.all(o[b, :, F[b]:] == -7.0), b


@pytest.mark.parametrize("width", [1, 60, 100, 256])
def test_frames_past_the_descriptors_width(gpu, handle, width):
    """Clips with more frames than the destination's descriptor is wide, in rows that hold them: the mel bank stores the
    frames up to a multiple of 256, the spectrogram up to one of 32, none beyond the rows."""
    rng = np.random.default_rng(width)
    B, bins, M, F, S = 3, 257, 40, 250, 256
    x = rng.uniform(0, 1, (B, bins, S)).astype(np.float32)
    out, full = torch.full((B, M, S), -7.0, device="cuda"), torch.full((B, M, S), -7.0, device="cuda")
    dims = dev(np.tile(np.array([bins, F], np.int32), B))
    for dst, w in ((out, width), (full, S)):
        gpu.mel_filter_bank(handle, dev(x), dst, dims, num_filter=M, dst_desc=gpu.desc_2d(B, M, w, S))
    n = min(F, (width + 255) // 256 * 256)
    assert torch.equal(out[:, :, :n], full[:, :, :n]) and bool(out[:, :, n:].eq(-7.0).all())
    sig = dev(rng.normal(0, 0.2, (B, 160 * F)).astype(np.float32))
    L = dev(np.full(B, 160 * F - 1, np.int32))      # F frames
    for layout in (gpu.NFT, gpu.NTF):
        shape = (B, bins, S) if layout == gpu.NFT else (B, S, bins)
        out, full = torch.full(shape, -7.0, device="cuda"), torch.full(shape, -7.0, device="cuda")
        for dst, w in ((out, width), (full, S)):
            d = gpu.desc_2d(B, bins, w, S) if layout == gpu.NFT else gpu.desc_2d(B, w, bins, bins, layout)
            d.strides.nStride = bins * S
            gpu.spectrogram(handle, sig, dst, L, layout=layout, dst_desc=d)
        if layout == gpu.NTF:
            out, full = out.transpose(1, 2), full.transpose(1, 2)
        n = min(F, (width + 31) // 32 * 32)
        assert torch.equal(out[:, :, :n], full[:, :, :n]) and bool(out[:, :, n:].eq(-7.0).all())


@pytest.mark.parametrize("frames,clips,M", [(64, 1, 256), (65, 60, 80), (640, 7, 80), (640, 13, 80), (640, 26, 80), (640, 52, 80), (300, 3, 5)])
def test_mel_group_counts(gpu, handle, frames, clips, M):
    """Batches for every number of groups from 64 down to 8, banks with fewer filters than groups among them."""
    test_mel_groups(gpu, handle, 257, M, 16000.0, 0.0, 8000.0, "slaney", True, (frames,), clips)
