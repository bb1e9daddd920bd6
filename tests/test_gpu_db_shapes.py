"""to_decibels over shapes where its split into 256-column units can go wrong: rows of one value up to
past several units, unaligned rows, one-column (1-D) clips inside a 2-D batch, many rows, and the clip
maximum with infinities, zeros and NaN in the clip.  Against FP64 log2 rounded once to FP32, the HOST
path's value: equal but for arguments whose logarithm lies within 2^-26 ulp of a rounding tie (one of
10^5 values is allowed to differ by one ulp)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def expected(x, ref, cutoff, mult):
    ratio = np.float32(10.0 ** float(np.float32(cutoff) / np.float32(mult)))
    inv = np.float32(1) / np.float32(ref) if ref != 0 else np.float32(1)
    with np.errstate(all="ignore"):
        v = x * inv
        m = np.where(v > ratio, v, ratio).astype(np.float32)
        lg = np.log2(m.astype(np.longdouble)).astype(np.float32)
    return (np.float32(mult) * np.float32(0.3010299956639812)) * lg


@pytest.mark.parametrize("rows,stride,ref", [(1, 5, 1.0), (3, 257, 0.0), (80, 1027, 0.0), (1025, 70, 0.0), (7, 2600, 2.5),
                                             (600, 512, 0.0)])
def test_db_units(gpu, handle, rows, stride, ref):
    rng = np.random.default_rng(rows + stride)
    widths = np.array([stride, 1, max(stride - 1, 2), min(stride, 256), min(stride, 255), 2], np.uint32)
    heights = np.array([rows, rows, max(rows - 1, 1), rows, rows, 1], np.uint32)
    x = np.exp(rng.uniform(-30, 12, (6, rows, stride))).astype(np.float32)
    x[0, 0, 0], x[2, -1, 0] = 0.0, np.nan
    x[3].reshape(-1)[:4] = [1e-42, 3e-39, 1.0, 0.0]
    x[5] = 0.0                                  # a silent clip: reference 0 counts as 1
    out = torch.full(x.shape, -7.0, device="cuda")
    dims = np.stack([widths, heights], 1).reshape(-1).astype(np.uint32)
    gpu.to_decibels(handle, dev(x), out, dev(dims.view(np.int32)), reference_magnitude=ref,
                    src_desc=gpu.desc_2d(6, rows, stride), dst_desc=gpu.desc_2d(6, rows, stride))
    o = out.cpu().numpy()
    for b in range(6):
        if widths[b] == 1:
            got, val, rest = o[b].reshape(-1)[:rows], x[b].reshape(-1)[:rows], o[b].reshape(-1)[rows:]
        else:
            got, val = o[b, :heights[b], :widths[b]], x[b, :heights[b], :widths[b]]
            rest = np.concatenate([o[b, heights[b]:].reshape(-1), o[b, :, widths[b]:].reshape(-1)])
        r = np.float32(np.nanmax(val)) if ref == 0.0 else np.float32(ref)
        e = expected(val, r, -80.0, 10.0)
        ulp = np.abs(got.reshape(-1).view(np.int32).astype(np.int64) - e.reshape(-1).view(np.int32).astype(np.int64))
        assert ulp.max() <= 1 and np.sum(ulp != 0) <= 1 + got.size // 100000, b
        assert np.all(rest == -7.0), b


def test_db_infinite_maximum(gpu, handle):
    """x / inf is 0 for finite values (the cut-off) and NaN, which the comparison also sends to the cut-off."""
    x = np.ones((1, 2, 300), np.float32)
    x[0, 1, 7] = np.inf
    out = torch.zeros((1, 2, 300), device="cuda")
    gpu.to_decibels(handle, dev(x), out, dev(np.array([300, 2], np.int32)), reference_magnitude=0.0)
    assert np.all(out.cpu().numpy() == np.float32(10.0) * np.float32(0.3010299956639812) *
                  np.log2(np.float64(np.float32(1e-8))).astype(np.float32))
    gpu.to_decibels(handle, dev(x), out, dev(np.array([300, 2], np.int32)), reference_magnitude=1.0)
    assert out[0, 1, 7].item() == float("inf") and out[0, 0, 0].item() == 0.0


def test_db_capture_after_a_smaller_shape(gpu):
    """A clip-maximum call is captured after a call of a smaller shape, and every replay has the eager bits."""
    st = torch.cuda.Stream()
    h = gpu.Handle(4, st)
    rng = np.random.default_rng(5)
    small, x = (dev(np.exp(rng.uniform(-20, 5, (4, r, c))).astype(np.float32)) for r, c in ((2, 30), (600, 2000)))
    dims = [dev(np.array([c, r] * 4, np.int32)) for r, c in ((2, 30), (600, 2000))]
    outs, out, eager = torch.zeros_like(small), torch.zeros_like(x), torch.zeros_like(x)
    torch.cuda.synchronize()
    gpu.to_decibels(h, small, outs, dims[0], reference_magnitude=0.0)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        gpu.to_decibels(h, x, out, dims[1], reference_magnitude=0.0)
    for _ in range(3):
        x.mul_(3.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        gpu.to_decibels(h, x, eager, dims[1], reference_magnitude=0.0)
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and bool(out.ne(0).any())
    del g
    h.close()


@pytest.mark.parametrize("B", [5000, 65535])
def test_db_capture_after_another_call(gpu, B):
    """A clip-maximum call is captured after a call of another kind of the same batch, larger than the batch the handle
    was made for, and every replay has the eager bits."""
    st = torch.cuda.Stream()
    h = gpu.Handle(4, st)
    x = dev(np.exp(np.random.default_rng(B).uniform(-20, 5, (B, 3, 4))).astype(np.float32))
    dims, lens = dev(np.array([4, 3] * B, np.int32)), dev(np.full(B, 12, np.int32))
    begin, count = torch.zeros(B, dtype=torch.int32, device="cuda"), torch.zeros(B, dtype=torch.int32, device="cuda")
    out, eager = torch.zeros_like(x), torch.zeros_like(x)
    torch.cuda.synchronize()
    gpu.non_silent_region_detection(h, x.view(B, 12), lens, begin, count)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        gpu.to_decibels(h, x, out, dims, reference_magnitude=0.0)
    for _ in range(3):
        x.mul_(3.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        gpu.to_decibels(h, x, eager, dims, reference_magnitude=0.0)
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and bool(out.ne(0).any())
    del g
    h.close()
