"""The FFT frames of the FP32 entry points (nfft a power of two up to 2048; 4096 and others run dense) at the
edges of their tiles.

Bound: an FFT of N points in FP32 has an error of at most u (3 log2 N + 4) times the 2-norm of the
spectrum on each bin (u = 2^-24: per level one rounded addition and one rounded twiddle product of
two terms; 4 for the window, the twiddle tables, the split and the square), so a bin's power is off
by at most 2 |X| d + d^2 with that d."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# nfft, window, hop, power, layout: full and short windows, odd windows and hops, every size
CASES = [(64, 64, 16, 2, "NFT"), (64, 33, 7, 1, "NTF"), (128, 128, 100, 2, "NTF"), (128, 101, 64, 2, "NFT"),
         (256, 200, 80, 2, "NFT"), (512, 400, 160, 2, "NFT"), (512, 511, 97, 1, "NTF"), (1024, 1024, 256, 2, "NFT"),
         (1024, 3, 501, 2, "NFT"), (2048, 2048, 512, 1, "NFT"), (2048, 1025, 333, 2, "NTF"), (4096, 4096, 1024, 2, "NFT"),
         (4096, 2500, 999, 2, "NTF")]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_spectrogram_fft_edges(gpu, handle, orc, case):
    N, W, H, power, layout = case
    rng = np.random.default_rng(N + W)
    # around a window, and one, one less and one more frame than tiles of 8, 16, 32 and 64 frames
    L = np.array([1, 2, W - 1, W, W + 1, 7 * H, 8 * H, 15 * H + 1, 16 * H, 31 * H, 32 * H + 3, 63 * H, 64 * H + H - 1,
                  70 * H + 5], np.int32)
    L = np.maximum(L, 1)
    S = int(L.max()) + 3
    x = rng.normal(0, 0.3, (len(L), S)).astype(np.float32)
    ref = orc.spectrogram_f64(x.astype(np.float64), L, N, W, H, True, True, 2, layout, nthreads=8)
    for b, n in enumerate(L):
        x[b, n:] = np.nan                       # samples past the clip never count
    out = torch.full(ref.shape, -1.0, device="cuda")
    gpu.spectrogram(handle, dev(x), out, dev(L), nfft=N, window_length=W, window_step=H, power=power,
                    layout=gpu.NFT if layout == "NFT" else gpu.NTF)
    o = out.cpu().numpy()
    u = 2.0 ** -24 * (3 * np.log2(N) + 4)
    for b, n in enumerate(L):
        F = int(n) // H + 1
        a, r = (o[b, :, :F], ref[b, :, :F]) if layout == "NFT" else (o[b, :F].T, ref[b, :F].T)
        tail = o[b, :, F:] if layout == "NFT" else o[b, F:]
        assert np.all(tail == -1.0), b
        d = u * np.sqrt(2 * r.sum(axis=0, keepdims=True))
        got = a.astype(np.float64) ** 2 if power == 1 else a.astype(np.float64)
        assert np.all(np.abs(got - r) <= 2 * np.sqrt(r) * d + d * d + 1e-30), (b, n)


@pytest.mark.parametrize("N,W,H,M,ref", [(64, 64, 24, 10, 1.0), (128, 100, 33, 20, 0.0), (256, 200, 80, 40, 1.0),
                                         (512, 400, 160, 80, 1.0), (512, 511, 201, 64, 0.0)])
def test_fused_fp32_fft_equals_chain(gpu, N, W, H, M, ref):
    """The fused FP32 launch gives the four calls' bits, also at tile ends and odd hops."""
    rng = np.random.default_rng(N + H)
    L = np.array([1, W - 1, W + 1, 31 * H, 32 * H, 33 * H + 1, 64 * H - 1, 9000], np.int32)
    frames = L // H + 1
    x = rng.normal(0, 0.2, (len(L), int(L.max()) + 5)).astype(np.float32)
    p = gpu.logmel_params(nfft=N, window_length=W, window_step=H, num_filter=M, reference_magnitude=ref)
    fused = torch.full((len(L), M, int(frames.max())), float("nan"), device="cuda")
    h = gpu.Handle(len(L))
    gpu.logmel_fused(h, dev(x), fused, dev(L), p, "fp32")
    chain = torch.full_like(fused, float("nan"))
    gpu.logmel_chain_gpu(h, dev(x), chain, torch.from_numpy(L), p)
    torch.cuda.synchronize()
    h.close()
    a, c = fused.cpu().numpy(), chain.cpu().numpy()
    for b, F in enumerate(frames):
        if F == 1:
            continue    # one column: the to_decibels call reads such a clip as 1-D data of M values
        assert np.array_equal(a[b, :, :F], c[b, :, :F]), (b, int(L[b]))
        assert np.all(np.isnan(a[b, :, F:])), b


@pytest.mark.parametrize("B,longest", [(300, 6000), (2100, 1500)])
def test_tiles_of_large_ragged_batches(gpu, B, longest):
    """More tiles than resident workgroups: planned per workgroup (300 clips) and, past what a plan holds
    (2,100 clips), taken pair by pair / from the planner kernel.  Every clip has the bits it has alone."""
    rng = np.random.default_rng(B)
    N, W, H, M = 256, 200, 16, 20
    L = rng.integers(1, longest, B).astype(np.int32)
    L[:3] = [longest, 1, longest - 1]
    frames = L // H + 1
    F = int(frames.max())
    x = dev(rng.normal(0, 0.2, (B, longest + 3)).astype(np.float32))
    p = gpu.logmel_params(nfft=N, window_length=W, window_step=H, num_filter=M, sample_rate=8000.0, max_freq=4000.0)
    h = gpu.Handle(B)
    spec = torch.full((B, N // 2 + 1, F), -1.0, device="cuda")
    gpu.spectrogram(h, x, spec, dev(L), nfft=N, window_length=W, window_step=H)
    db = torch.full((B, M, F), -1.0, device="cuda")
    gpu.logmel_fused(h, x, db, dev(L), p, "fp32")
    sizes = frames.astype(np.int64) * M
    flat = torch.cat([x[b, :int(n)] for b, n in enumerate(L)])
    src_off = np.concatenate([[0], np.cumsum(L.astype(np.int64))[:-1]])
    dst_off = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    packed = torch.full((int(sizes.sum()),), -1.0, device="cuda")
    gpu.logmel_fused_packed(h, flat, dev(src_off), dev(L), packed, dev(dst_off), p, "fp32")
    pk = packed.cpu().numpy()
    spec, dbs = spec.cpu().numpy(), db.cpu().numpy()
    some = list(range(40)) + list(range(B - 20, B))
    for b in some:
        f = int(frames[b])
        one = torch.full((1, N // 2 + 1, f), -1.0, device="cuda")
        gpu.spectrogram(h, x[b:b + 1], one, dev(L[b:b + 1]), nfft=N, window_length=W, window_step=H)
        alone = torch.full((1, M, f), -1.0, device="cuda")
        gpu.logmel_fused(h, x[b:b + 1], alone, dev(L[b:b + 1]), p, "fp32")
        assert np.array_equal(spec[b, :, :f], one[0].cpu().numpy()), b
        assert np.array_equal(dbs[b, :, :f], alone[0].cpu().numpy()), b
        assert np.array_equal(pk[dst_off[b]:dst_off[b] + sizes[b]].reshape(M, f), alone[0].cpu().numpy()), b
    for b in range(B):
        assert np.all(spec[b, :, frames[b]:] == -1.0) and np.all(dbs[b, :, frames[b]:] == -1.0), b
        assert np.all(spec[b, :, :frames[b]] >= 0.0) and np.all(dbs[b, :, :frames[b]] != -1.0), b
    h.close()


@pytest.mark.parametrize("H", [160, 829, 830, 845, 2600])
def test_fused_fp32_log_table_places(gpu, H):
    """More tiles than resident workgroups, with room for the log2 table in LDS (hops 160 and 845: the latter with
    one workgroup fewer per CU) and without (829, 830): the chain's bits.  A hop of 2,600 is refused, as its
    32-frame segment exceeds LDS."""
    rng = np.random.default_rng(H)
    B, longest = 64, 220 * H
    L = rng.integers(200 * H, longest, B).astype(np.int32)
    x = torch.randn((B, longest), generator=torch.Generator("cuda").manual_seed(H), device="cuda").mul_(0.2)
    F = int((L // H + 1).max())
    p = gpu.logmel_params(nfft=512, window_length=400, window_step=H, num_filter=40)
    h = gpu.Handle(B)
    fused = torch.full((B, 40, F), float("nan"), device="cuda")
    if H == 2600:
        with pytest.raises(gpu.RppError):
            gpu.logmel_fused(h, x, fused, dev(L), p, "fp32")
        h.close()
        return
    gpu.logmel_fused(h, x, fused, dev(L), p, "fp32")
    chain = torch.full_like(fused, float("nan"))
    gpu.logmel_chain_gpu(h, x, chain, torch.from_numpy(L), p)
    torch.cuda.synchronize()
    h.close()
    a, c = fused.cpu().numpy(), chain.cpu().numpy()
    for b in range(B):
        n = int(L[b]) // H + 1
        assert np.array_equal(a[b, :, :n], c[b, :, :n]), b
        assert np.all(np.isnan(a[b, :, n:])), b


def contraction_classes(x, L, N, W, H, win, center, reflect):
    """The frames' power by contraction with FP32 cosine and sine columns ([frames][bins], FP64): where it is infinite
    or NaN is what counts of it."""
    F = (L if center else L - W) // H + 1
    t = np.arange(W)
    i = np.arange(F)[:, None] * H - (W // 2 if center else 0) + t
    if reflect and L > 1:
        i = i % (2 * (L - 1))
        i = np.where(i < L, i, 2 * (L - 1) - i)
    a = np.where((i >= 0) & (i < L), x[np.clip(i, 0, L - 1)], 0).astype(np.float64)
    kt = t[:, None] * np.arange(N // 2 + 1) % N
    c = (win[:, None] * np.cos(2 * np.pi * kt / N)).astype(np.float32).astype(np.float64)
    s = (-win[:, None] * np.sin(2 * np.pi * kt / N)).astype(np.float32).astype(np.float64)
    s[:, [0, -1]] = 0.0
    with np.errstate(all="ignore"):
        re = np.einsum("ft,tk->fk", a, c)
        b = np.einsum("ft,tk->fk", a, s)
        b[:, [0, -1]] = 0.0
        return re * re + b * b


@pytest.mark.parametrize("N,W,H,layout,power,center,reflect", [
    (64, 64, 16, "NFT", 2, True, True), (128, 101, 60, "NTF", 1, True, False), (256, 200, 80, "NFT", 2, False, True),
    (512, 400, 160, "NFT", 2, True, True), (1024, 1024, 256, "NTF", 2, True, True), (2048, 2000, 512, "NFT", 1, True, True),
    (300, 300, 100, "NFT", 2, True, True)])
def test_infinite_samples(gpu, handle, N, W, H, layout, power, center, reflect):
    """A frame with infinite samples has infinite power where the contraction with the bin's columns is infinite and NaN
    where that mixes signs or meets a zero; other frames are as without them."""
    rng = np.random.default_rng(N)
    S = 6 * W + 3 * H
    L = np.array([S, S, S, S, S, W // 3 + 2, S], np.int32)
    x = rng.normal(0, 0.3, (len(L), S)).astype(np.float32)
    plain = x.copy()
    x[0, S // 2] = np.inf
    x[1, S // 2 + 1] = -np.inf
    x[2, [S // 3, S // 3 + 5]] = [np.inf, -np.inf]
    x[3, [0, S - 1, W + H]] = np.inf
    x[4, [S // 2, S // 2 + 2]] = [np.nan, np.inf]
    x[5, W // 5] = np.inf
    F = L // H + 1 if center else np.maximum((L - W) // H + 1, 0)
    K, most = N // 2 + 1, int(F.max())
    win = rng.uniform(0.1, 1.0, W).astype(np.float32) * np.where(rng.random(W) < 0.2, -1, 1).astype(np.float32)
    win[W // 2] = 0.0
    for window in (None, win):
        out, ref = (torch.full((len(L), K, most) if layout == "NFT" else (len(L), most, K), -1.0, device="cuda") for _ in range(2))
        for src, dst in ((x, out), (plain, ref)):
            gpu.spectrogram(handle, dev(src), dst, dev(L), nfft=N, window_length=W, window_step=H, power=power, window=window,
                            center=center, reflect=reflect, layout=gpu.NFT if layout == "NFT" else gpu.NTF)
        o, r = out.cpu().numpy(), ref.cpu().numpy()
        if layout == "NTF":
            o, r = o.transpose(0, 2, 1), r.transpose(0, 2, 1)
        w = 0.5 * (1 - np.cos(2 * np.pi / W * (np.arange(W) + 0.5))) if window is None else win.astype(np.float64)
        w = w.astype(np.float32).astype(np.float64)
        for b, n in enumerate(L):
            e = contraction_classes(x[b], int(n), N, W, H, w, center, reflect).T
            got = o[b, :, :F[b]]
            assert np.array_equal(np.isnan(got), np.isnan(e)) and np.array_equal(np.isposinf(got), np.isposinf(e)), (b, window is None)
            clean = np.isfinite(e).all(axis=0)
            assert np.array_equal(got[:, clean], r[b, :, :F[b]][:, clean]), b


@pytest.mark.parametrize("ref", [1.0, 0.0])
@pytest.mark.parametrize("N,W,H,M", [(128, 100, 33, 20), (512, 400, 160, 80), (1024, 1024, 256, 128), (1024, 700, 301, 40)])
def test_fused_fp32_infinite_samples_equal_chain(gpu, N, W, H, M, ref):
    """The fused FP32 launch gives the four calls' bits on clips with infinite samples too.  Clip 0 ends in one, so that
    no second infinity follows it from the pre-emphasis: the bands of its last frame are infinite."""
    rng = np.random.default_rng(N + W)
    L = np.array([9000, 8000, W + 5 * H, 9000], np.int32)
    frames = L // H + 1
    x = rng.normal(0, 0.2, (len(L), 9003)).astype(np.float32)
    x[0, 8999], x[1, 0], x[2, W + 7], x[3, 8999] = np.inf, np.inf, -np.inf, np.nan
    p = gpu.logmel_params(nfft=N, window_length=W, window_step=H, num_filter=M, reference_magnitude=ref, reflect=False)
    fused, chain = (torch.full((len(L), M, int(frames.max())), -1.0, device="cuda") for _ in range(2))
    h = gpu.Handle(len(L))
    gpu.logmel_fused(h, dev(x), fused, dev(L), p, "fp32")
    gpu.logmel_chain_gpu(h, dev(x), chain, torch.from_numpy(L), p)
    torch.cuda.synchronize()
    h.close()
    a, c = fused.cpu().numpy(), chain.cpu().numpy()
    for b, F in enumerate(frames):
        assert np.array_equal(a[b, :, :F], c[b, :, :F], equal_nan=True), (b, int(L[b]))
    assert np.isposinf(a[0, :, frames[0] - 1]).any() == (ref != 0.0)


@pytest.mark.parametrize("N,B", [(64, 3), (64, 400), (512, 3)])
def test_fused_fp32_more_filters_than_lds(gpu, N, B):
    """45,000 filters, whose intervals do not fit LDS: the chain's bits (nearly all of the filters are empty)."""
    rng = np.random.default_rng(N)
    L = rng.integers(N, 3 * N, B).astype(np.int32)
    H, M = N // 2, 45000
    frames = L // H + 1
    x = dev(rng.normal(0, 0.2, (B, 3 * N)).astype(np.float32))
    p = gpu.logmel_params(nfft=N, window_length=N, window_step=H, num_filter=M)
    h = gpu.Handle(B)
    fused, chain = (torch.full((B, M, int(frames.max())), float("nan"), device="cuda") for _ in range(2))
    gpu.logmel_fused(h, x, fused, dev(L), p, "fp32")
    gpu.logmel_chain_gpu(h, x, chain, torch.from_numpy(L), p)
    torch.cuda.synchronize()
    h.close()
    for b, F in enumerate(frames):
        assert torch.equal(fused[b, :, :F], chain[b, :, :F]) and bool(torch.isnan(fused[b, :, F:]).all()), b


def test_fft_tables_hold_no_basis(gpu):
    """The tables of an FFT size take some 4 nfft floats, not a contraction basis of window length x nfft."""
    h = gpu.Handle(1)
    x, L, out = torch.zeros((1, 4096), device="cuda"), dev(np.array([4096], np.int32)), torch.zeros((1, 1025, 9), device="cuda")

    def call(W):
        gpu.spectrogram(h, x, out, L, nfft=2048, window_length=W, window_step=512)
        torch.cuda.synchronize()

    call(2048)
    before = torch.cuda.mem_get_info()[0]
    for W in range(2040, 2048):
        call(W)
    taken = before - torch.cuda.mem_get_info()[0]
    h.close()
    assert taken <= 32 << 20, taken       # (8 tables of 32 KB, each in pages of its own; 8 bases take 128 MB)


@pytest.mark.parametrize("N,W,H", [(64, 64, 40), (128, 101, 64), (256, 256, 100), (512, 400, 160), (1024, 1024, 256), (2048, 2048, 512)])
def test_spectrogram_fft_is_fp64(gpu, handle, N, W, H):
    """Quiet bins beside a loud tone: every power is the FP64 transform of the FP32-windowed frame rounded once.  Bound:
    2^-24 of the power for the rounding, and an FP64 transform's error d = 2^-53 (6 log2 N + 10) of the frame's norm on
    X (per level one rounded addition and a rounded product with a twiddle off by an ulp; the window
    products are exact), which is 2 |X| d + d^2 on the power."""
    rng = np.random.default_rng(N)
    L = 40 * H + W
    t = np.arange(L)
    x = (np.sin(2 * np.pi * t * 3.7 / N) + 1e-6 * rng.normal(size=L)).astype(np.float32)
    F, K = (L - W) // H + 1, N // 2 + 1
    out = torch.zeros((1, K, F), device="cuda")
    gpu.spectrogram(handle, dev(x[None]), out, dev(np.array([L], np.int32)), nfft=N, window_length=W, window_step=H, center=False)
    w = (0.5 * (1 - np.cos(2 * np.pi / W * (np.arange(W) + 0.5)))).astype(np.float32).astype(np.float64)
    X = np.stack([np.fft.rfft(x[f * H:f * H + W].astype(np.float64) * w, N) for f in range(F)], 1)
    p = np.abs(X) ** 2
    d = 2.0 ** -53 * (6 * np.log2(N) + 10) * np.sqrt(2 * p.sum(axis=0, keepdims=True))
    err = np.abs(out[0].cpu().numpy().astype(np.float64) - p)
    assert np.all(err <= 2.0 ** -24 * p + 2 * np.sqrt(p) * d + d * d), float((err / p).max())
    assert p.min() < 1e-8 * p.max()


@pytest.mark.parametrize("W,H,M", [(1024, 256, 128), (1000, 256, 80), (333, 301, 20)])
@pytest.mark.parametrize("ref", [1.0, 0.0])
def test_fused_fp32_fft_1024_equals_chain(gpu, W, H, M, ref):
    """The nfft-1024 instance, full, short and odd windows."""
    test_fused_fp32_fft_equals_chain(gpu, 1024, W, H, M, ref)


@pytest.mark.parametrize("N,W,H,M", [(300, 300, 100, 40), (100, 99, 33, 20), (600, 500, 40, 40)])
@pytest.mark.parametrize("ref", [1.0, 0.0])
def test_fused_fp32_dense_equals_chain(gpu, N, W, H, M, ref):
    """The contraction of the other sizes, in one pass over the columns and in two, gives the four calls' bits."""
    test_fused_fp32_fft_equals_chain(gpu, N, W, H, M, ref)
