"""GPU parity of the STFT family (stft.hip) against the oracle and the reference's golden vectors.

Bound (north star): SNR >= 110 dB for spectra (the oracle's double spectrum is the reference)
and for STFT -> iSTFT reconstructions, SNR = 10 log10(sum ref^2 / sum err^2)
(tools/stems-parity.cpp:36). Layout changes are exact (bit-identical values).
"""
import glob
import os

import numpy as np
import pytest

import oracle_lib
import stx
import synth
from metrics import snr_db

pytestmark = pytest.mark.gpu

SNR_DB = 110.0
GOLDEN = sorted(glob.glob(os.path.join(os.path.dirname(__file__), "golden", "stft_*.npz")))
SPEC_GOLDEN = [p for p in GOLDEN if "torch" in p or "htdemucs" in p]


@pytest.fixture(scope="module")
def orc():
    return oracle_lib.oracle()


_plans = {}


def plan(n):
    if n not in _plans:
        _plans[n] = stx.FFT(n)
    return _plans[n]


def to_dev(a, device):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def frame_weight(n, hop, T):
    """sqrt(sum(w^2)) over the frames that cover each sample of an iSTFT of T frames. A sample is sum(w x) / sum(w^2), so
    errors of one size in the frames leave that size over this weight: multiplied by it, the bar holds at every hop."""
    span = -(-n // hop)
    w2 = np.zeros(span * hop)
    w2[:n] = (0.5 - 0.5 * np.cos(2.0 * np.pi * np.arange(n) / n)) ** 2
    env = np.zeros((T + span, hop))
    for q in range(span):
        env[q:q + T] += w2[q * hop:(q + 1) * hop]
    return np.sqrt(env.reshape(-1)[n // 2:n // 2 + hop * (T - 1)])


def ws_for(fft, channels, frames, device, use):
    return stx.workspace(stx.istft_workspace_size(fft, channels, frames), device) if use else None


@pytest.mark.parametrize("path", SPEC_GOLDEN, ids=[os.path.basename(p)[5:-4] for p in SPEC_GOLDEN])
@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("use_ws", [False, True], ids=["plain", "workspace"])
def test_golden_spectrum_and_inverse(device, path, layout, use_ws):
    d = np.load(path)
    n = int(d["n_fft"])
    x = to_dev(d["x"][None, :], device)
    spec_ref = d["spec"]
    if "torch" in path:
        hop, nm = int(d["hop"]), bool(int(d["normalized"]))
        spec = stx.torch_stft(plan(n), x, hop, nm, layout=layout)
    else:
        spec = stx.htdemucs_spec(plan(n), x, layout=layout)
    got = host(spec)[0]
    if layout == stx.T_MAJOR:
        got = got.T
    assert got.shape == spec_ref.shape
    assert snr_db(got, spec_ref) >= SNR_DB
    # Inverse of the reference spectrum rounded to complex64.
    s = spec_ref.astype(np.complex64)[None]
    sdev = to_dev(s if layout == stx.F_MAJOR else np.ascontiguousarray(s.transpose(0, 2, 1)), device)
    ws = ws_for(plan(n), 1, spec_ref.shape[1], device, use_ws)
    if "torch" in path:
        y = stx.torch_istft(plan(n), sdev, hop, nm, layout=layout, workspace=ws)
    else:
        y = stx.htdemucs_ispec(plan(n), sdev, d["x"].size, layout=layout, workspace=ws)
    y = host(y)[0]
    assert y.shape == d["y"].shape
    assert snr_db(y, d["y"]) >= SNR_DB


def _stereo(seed, length, sigma=0.1):
    return synth.normal(seed, (2, length), sigma)


@pytest.mark.parametrize("use_ws", [False, True], ids=["plain", "workspace"])
def test_htdemucs_spec_c1_full_size(device, orc, use_ws):
    # HTDemucs spec: stereo 343,980 samples, n_fft 4096, hop 1024 -> [2][2048][336].
    length = 343980
    x = _stereo(2024, length)
    f = plan(4096)
    spec = stx.htdemucs_spec(f, to_dev(x, device))
    y = stx.htdemucs_ispec(f, spec, length, workspace=ws_for(f, 2, 336, device, use_ws))
    spec_h, y_h = host(spec), host(y)
    assert spec_h.shape == (2, 2048, 336)
    for c in range(2):
        ref = orc.htdemucs_spec(x[c], 4096)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        yref = orc.htdemucs_ispec(ref, 4096, length)
        assert snr_db(y_h[c], yref) >= SNR_DB


def test_torch_stft_c1_plain_call(device, orc):
    length = 343980
    x = _stereo(2025, length)
    f = plan(4096)
    spec = stx.torch_stft(f, to_dev(x, device), 1024)
    y = stx.torch_istft(f, spec, 1024)
    spec_h, y_h = host(spec), host(y)
    assert spec_h.shape == (2, 2049, 336)
    for c in range(2):
        ref = orc.torch_stft(x[c], 4096, 1024)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y_h[c], orc.torch_istft(ref, 4096, 1024)) >= SNR_DB
        assert snr_db(y_h[c], x[c][: y_h.shape[1]]) >= SNR_DB


@pytest.mark.parametrize("normalized", [False, True])
@pytest.mark.parametrize("use_ws", [False, True], ids=["plain", "workspace"])
def test_roformer_stft_c3_full_size(device, orc, normalized, use_ws):
    # RoFormer chunk: stereo 352,800 samples, n_fft 2048, hop 441 -> [2][1025][801] (odd T).
    length = 352800
    x = _stereo(2026, length)
    f = plan(2048)
    spec = stx.torch_stft(f, to_dev(x, device), 441, normalized)
    spec_t = stx.torch_stft(f, to_dev(x, device), 441, normalized, layout=stx.T_MAJOR)
    ws = ws_for(f, 2, 801, device, use_ws)
    y = stx.torch_istft(f, spec, 441, normalized, workspace=ws)
    y_t = stx.torch_istft(f, spec_t, 441, normalized, layout=stx.T_MAJOR, workspace=ws)
    spec_h, spec_th, y_h, y_th = host(spec), host(spec_t), host(y), host(y_t)
    assert spec_h.shape == (2, 1025, 801)
    assert np.array_equal(spec_h, spec_th.transpose(0, 2, 1))
    assert np.array_equal(y_h, y_th)
    for c in range(2):
        ref = orc.torch_stft(x[c], 2048, 441, normalized)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y_h[c], orc.torch_istft(ref, 2048, 441, normalized)) >= SNR_DB
        assert snr_db(y_h[c], x[c]) >= SNR_DB


@pytest.mark.parametrize("n", [16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("use_ws", [False, True], ids=["plain", "workspace"])
def test_every_fft_size_stft_round_trip(device, orc, n, use_ws):
    hop = max(1, n // 4 - 1)
    length = 3 * n + 5
    x = _stereo(300 + n, length, 0.5)
    f = plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop)
    y = stx.torch_istft(f, spec, hop, workspace=ws_for(f, 2, length // hop + 1, device, use_ws))
    spec_h, y_h = host(spec), host(y)
    for c in range(2):
        ref = orc.torch_stft(x[c], n, hop)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y_h[c], orc.torch_istft(ref, n, hop)) >= SNR_DB
    if length > 3 * n // 8 * 2:
        s2 = stx.htdemucs_spec(f, to_dev(x, device))
        y2 = stx.htdemucs_ispec(f, s2, length, workspace=ws_for(f, 2, s2.shape[2], device, use_ws))
        s2h, y2h = host(s2), host(y2)
        for c in range(2):
            ref = orc.htdemucs_spec(x[c], n)
            assert snr_db(s2h[c], ref) >= SNR_DB
            assert snr_db(y2h[c], orc.htdemucs_ispec(ref, n, length)) >= SNR_DB


# Every power of two st::FFT accepts (src/stft.h:21-22): 2, 4, 8 as register transforms, 16 to
# 8192 as LDS kernels, and above 8192 in four steps (n1 x n2 transforms around transposes).
@pytest.mark.parametrize("n", [2, 4, 8, 16, 256, 2048, 4096, 8192, 16384, 32768, 1 << 20])
def test_fft_run_against_oracle(device, orc, n):
    import torch
    v = synth.normal(n, (3, 2 * n), 1.0).astype(np.float64)
    a = v[:, 0::2] + 1j * v[:, 1::2]
    d = to_dev(a.astype(np.complex64), device)
    plan(n).run(d)
    fw = host(d)
    plan(n).run(d, inverse=True)
    back = host(d) / n
    for b in range(3):
        assert snr_db(fw[b], orc.fft(a[b].astype(np.complex64).astype(np.complex128))) >= SNR_DB
        assert snr_db(back[b], a[b].astype(np.complex64)) >= SNR_DB
    del torch


def test_fft_run_only_sizes_have_no_stft(device):
    """Sizes with only a complex transform (2, 4, 8 and above 8192) report UNSUPPORTED for the
    STFT/iSTFT; the reference never frames at those sizes."""
    import torch
    x = torch.zeros((1, 100000), dtype=torch.float32, device=device)
    for n in (8, 16384):
        f = plan(n)
        assert f.size() == n
        with pytest.raises(stx.StxError) as e:
            stx.torch_stft(f, x, n // 4)
        assert e.value.status == stx.STATUS_UNSUPPORTED


def test_fft_impulse_known_answer(device):
    n = 2048
    a = np.zeros((1, n), np.complex64)
    a[0, 7] = 1.0
    d = to_dev(a, device)
    plan(n).run(d)
    k = np.arange(n)
    assert np.max(np.abs(host(d)[0] - np.exp(-2j * np.pi * 7 * k / n))) < 1e-6


def test_stft_errors(device):
    import torch
    x = torch.zeros((1, 1024), dtype=torch.float32, device=device)
    with pytest.raises(stx.StxError) as e:
        stx.torch_stft(plan(2048), x, 441)
    assert e.value.status == stx.STATUS_RUNTIME_ERROR
    with pytest.raises(stx.StxError) as e:
        stx.htdemucs_spec(plan(4096), x)
    assert e.value.status == stx.STATUS_RUNTIME_ERROR


def test_small_hop_needs_several_rounds(device, orc):
    # hop n/64 makes every output tile overlap 64 frames, twice the 32 one workgroup transforms
    # at once at n_fft 1024, so the fused path loops over rounds.
    n, hop, length = 1024, 16, 4000
    x = _stereo(55, length, 0.3)
    f = plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop)
    y = host(stx.torch_istft(f, spec, hop))
    spec_h = host(spec)
    for c in range(2):
        ref = orc.torch_stft(x[c], n, hop)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y[c], orc.torch_istft(ref, n, hop)) >= SNR_DB


@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("n,hop,length,channels,sub", [
    (2048, 441, 352800, 48, 3),     # 48 RoFormer chunks: 3,216 tiles; 3 chunks: 201 tiles
    (1024, 8, 2000, 8, 1),          # 4 rounds of 32 frames per tile: 2,000 tiles; 1 channel: 250
])
def test_istft_more_tiles_than_resident_workgroups(device, orc, layout, n, hop, length, channels, sub):
    # A batch whose tiles outnumber the workgroups the GPU holds at once: each workgroup takes a
    # run of hops (and prefetches the next round's frames). Every channel must equal, bit for
    # bit, the same channels inverted in a call small enough to give each tile its own workgroup.
    x = synth.normal(4100 + n, (channels, length), 0.2)
    f = plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop, layout=layout)
    y = host(stx.torch_istft(f, spec, hop, layout=layout))
    for i in range(0, channels, sub):
        part = host(stx.torch_istft(f, spec[i:i + sub].contiguous(), hop, layout=layout))
        assert np.array_equal(part, y[i:i + sub]), f"channels {i}..{i + sub - 1}"
    spec_h = host(spec)
    for c in (0, channels - 1):
        s = spec_h[c] if layout == stx.F_MAJOR else spec_h[c].T
        ref = orc.torch_stft(x[c], n, hop)
        assert snr_db(s, ref) >= SNR_DB
        assert snr_db(y[c], orc.torch_istft(ref, n, hop)) >= SNR_DB


@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
def test_htdemucs_ispec_many_segments_same_bits_as_pairs(device, orc, layout):
    # 16 HTDemucs segments (n_fft 4096) in one call: 1,088 tiles of 5 hops, t-major runs of rounds of
    # 7 frames; a call of two segments takes 6-frame tiles of 3 hops, one per
    # workgroup. Each sample adds the same frames in the same order either way, so every
    # channel must come out bit for bit the same.
    length, channels = 343980, 16
    x = synth.normal(4242, (channels, length), 0.1)
    f = plan(4096)
    spec = stx.htdemucs_spec(f, to_dev(x, device), layout=layout)
    y = host(stx.htdemucs_ispec(f, spec, length, layout=layout))
    for i in range(0, channels, 2):
        part = host(stx.htdemucs_ispec(f, spec[i:i + 2].contiguous(), length, layout=layout))
        assert np.array_equal(part, y[i:i + 2]), f"channels {i}, {i + 1}"
    spec_h = host(spec)
    for c in (0, channels - 1):
        s = spec_h[c] if layout == stx.F_MAJOR else spec_h[c].T
        ref = orc.htdemucs_spec(x[c], 4096)
        assert snr_db(s, ref) >= SNR_DB
        assert snr_db(y[c], orc.htdemucs_ispec(ref, 4096, length)) >= SNR_DB


# The switch to several frames a workgroup (2,048 frames; 512 f-major 3,328, 2048 f-major 2,560, 1024 t-major 8,192, 4096
# f-major by how full its last round of workgroups is), the last workgroup partly past the end and workgroups that cross
# channels, for every group size (8, 4 and 1).
@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("n,hop,length,channels", [(2048, 441, 441 * 1025, 2), (2048, 441, 441 * 682 + 3, 3), (1024, 256, 256 * 410 + 9, 5),
                                                   (512, 128, 128 * 1026, 2), (128, 64, 64 * 2049 + 1, 1), (16, 4, 4 * 1030, 2),
                                                   (8192, 2048, 2048 * 420, 5), (4096, 1024, 1024 * 684, 3),
                                                   (2048, 441, 441 * 870 + 5, 3), (512, 128, 128 * 1110 + 3, 3), (1024, 256, 256 * 1640, 5),
                                                   (4096, 1024, 1024 * 861 + 1, 3), (4096, 1024, 1024 * 1023, 2)])
def test_stft_many_frames(device, orc, layout, n, hop, length, channels):
    """STFT calls of 2,048 frames and more: every channel has the bits of a call of its own (fewer frames, one or two a
    workgroup), and the oracle's values."""
    x = synth.normal(4500 + n + hop, (channels, length), 0.2)
    f, xd = plan(n), to_dev(x, device)
    assert channels * (length // hop + 1) >= 2048
    spec = host(stx.torch_stft(f, xd, hop, layout=layout))
    for c in range(channels):
        if length // hop + 1 < 2048:
            one = host(stx.torch_stft(f, xd[c:c + 1].contiguous(), hop, layout=layout))
            assert np.array_equal(one[0], spec[c])
        s = spec[c] if layout == stx.F_MAJOR else spec[c].T
        assert snr_db(s, orc.torch_stft(x[c], n, hop)) >= SNR_DB


# Runs of istft_run_kernel at its edges: n_fft 8192 (two frames a round, the carry longer than a round finishes), hop n
# (no carry), hops that leave one sample uncovered (n - 1) or divide nothing, one sample past a run's end, and every
# power of two from 16 (many frames a round); 4096 f-major where runs save rounds (1,300 frames) and where tiles stay.
RUN_CASES = [(8192, 1024, 1024 * 400 + 5, 3), (8192, 333, 333 * 500, 2), (4096, 1023, 1023 * 700 + 1, 2), (4096, 1024, 1024 * 1299, 2),
             (4096, 1024, 1024 * 1570 + 3, 3), (2048, 2048, 2048 * 500, 9),
             (2048, 2047, 2047 * 700, 5), (1024, 300, 300 * 9001, 2), (512, 128, 128 * 17000 + 3, 2), (256, 64, 64 * 20001, 2),
             (128, 50, 50 * 30001, 2), (64, 16, 16 * 70001, 1), (32, 8, 8 * 400001, 1), (16, 4, 4 * 400001, 1)]


@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("n,hop,length,channels", RUN_CASES)
def test_istft_runs(device, orc, layout, n, hop, length, channels):
    """Calls with more tiles than the device holds workgroups. Every sample of every channel has the bits of a call on some
    200 tiles' worth of that channel's frames alone (one workgroup a tile), and channel 0 the oracle's values."""
    x = synth.normal(4400 + n + hop, (channels, length), 0.2)
    f = plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop, layout=layout)
    yd = stx.torch_istft(f, spec, hop, layout=layout)
    y, T, span = host(yd), length // hop + 1, -(-n // hop)
    m = 200 * max(1, min(32768 // n - span + 1, 6144 // hop)) + span
    for c in range(channels):
        for t0 in range(0, T, m - 2 * span):
            t1 = min(t0 + m, T)
            if t1 - t0 < 2:
                break
            part = spec[c:c + 1, :, t0:t1] if layout == stx.F_MAJOR else spec[c:c + 1, t0:t1]
            p = host(stx.torch_istft(f, part.contiguous(), hop, layout=layout))[0]
            # Sample i of the part is sample t0 hop + i; all its frames are in the part but near cut ends.
            lo = 0 if t0 == 0 else n // 2
            hi = p.size if t1 == T else p.size - n // 2
            assert np.array_equal(p[lo:hi], y[c, t0 * hop + lo:t0 * hop + hi]), f"channel {c}, frames {t0} .. {t1}"
            if t1 == T:
                break
    s = host(spec[0])
    ref = orc.torch_istft((s if layout == stx.F_MAJOR else s.T).astype(np.complex128), n, hop)
    weight = frame_weight(n, hop, T)
    assert snr_db(y[0] * weight, ref * weight) >= SNR_DB


# Hops above n_fft: samples between the frames that no frame covers. Calls of a few tiles and of more than the device holds
# workgroups; an odd number of channels, one sample uncovered (n + 1) and most of them.
GAP_CASES = [(2048, 2049, 6, 2), (2048, 3000, 5, 1), (2048, 5001, 400, 3), (1024, 1500, 900, 2), (512, 20000, 100, 3), (16, 40, 30, 2),
             (16, 41, 300001, 1), (64, 1000, 4001, 1), (8192, 10000, 300, 2), (4096, 4097, 500, 3),
             # Hops whose product with the frames of a workgroup (512 at n_fft 16) passes 2^31.
             (16, 5000000, 2, 2), (16, 4194305, 4, 1), (32, 10000000, 3, 1)]


@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("n,hop,frames,channels", GAP_CASES)
def test_istft_hop_above_n(device, layout, n, hop, frames, channels):
    """Frames that do not meet: a covered sample is its frame's own inverse (over the window, as w^2 / w^2), so the frames of
    one call laid n apart (hop n, whose oracle comparisons are test_istft_runs') have the same bits; an uncovered one is 0."""
    x = synth.normal(4600 + n + hop, (channels, frames * n), 0.2)
    f = plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), n, layout=layout)
    T = frames + 1                                           # length // n + 1
    y = host(stx.torch_istft(f, spec, hop, layout=layout))
    close = host(stx.torch_istft(f, spec, n, layout=layout))
    assert y.shape == (channels, hop * (T - 1))
    # Signal index J of sample i is i + n / 2; frame t covers [t hop, t hop + n).
    J = np.arange(y.shape[1]) + n // 2
    R = J % hop
    assert np.all(y[:, R >= n] == 0.0)
    covered = (J // hop) * n + R - n // 2
    sel = (R < n) & (covered < close.shape[1]) & (covered >= 0)
    assert np.array_equal(y[:, sel], close[:, covered[sel]])


def test_istft_output_near_2_31(device):
    """An output whose last tile starts less than a whole tile below 2^31 (8.6 GB): the frames' samples have the bits of the
    same frames 3,000 apart, and nothing else is written but zeros."""
    import torch
    n, hop, near, T = 16, 2147483, 3000, 1001
    f = plan(n)
    g = torch.Generator(device=device)
    g.manual_seed(31)
    spec = torch.randn((1, n // 2 + 1, T), generator=g, device=device, dtype=torch.complex64)
    out = torch.full((hop * (T - 1) + 64,), 5.5, device=device)
    stx.torch_istft(f, spec, hop, out=out[:hop * (T - 1)].view(1, -1))
    small = stx.torch_istft(f, spec, near)[0]
    k = torch.arange(n, device=device) - n // 2
    t = torch.arange(T, device=device)[:, None]
    ok = (t * near + k >= 0) & (t * near + k < small.numel())
    assert torch.equal(out[(t * hop + k)[ok]], small[(t * near + k)[ok]])
    assert bool((out[hop * (T - 1):] == 5.5).all())
    assert int(torch.count_nonzero(out[:hop * (T - 1)])) == int(torch.count_nonzero(small))


def test_istft_many_tiles_graph_replays(device):
    """A captured torch_istft call whose tiles outnumber the resident workgroups, replayed on new
    spectra with eager work between the replays: every replay equals the eager call's bits."""
    import torch
    n, hop, length, channels = 2048, 441, 352800, 24
    f = plan(n)
    x = to_dev(synth.normal(4300, (channels, length), 0.2), device)
    spec = stx.torch_stft(f, x, hop)
    y = torch.empty((channels, length), device=device)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        stx.torch_istft(f, spec, hop, out=y, stream=s)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            stx.torch_istft(f, spec, hop, out=y, stream=s)
    torch.cuda.synchronize()
    for rep in range(3):
        xn = to_dev(synth.normal(4310 + rep, (channels, length), 0.1 + 0.2 * rep), device)
        spec.copy_(stx.torch_stft(f, xn, hop))
        want = host(stx.torch_istft(f, spec, hop))
        g.replay()
        assert np.array_equal(host(y), want), f"replay {rep}"


@pytest.mark.parametrize("trim", [0, 4999])
def test_htdemucs_ispec_many_segments_trimmed(device, orc, trim):
    # The batched call with an output shorter than the segment (the tiles' last one cut short)
    # against one segment at a time.
    length, channels = 343980, 12
    x = synth.normal(4400 + trim, (channels, length), 0.1)
    f = plan(4096)
    spec = stx.htdemucs_spec(f, to_dev(x, device))
    y = host(stx.htdemucs_ispec(f, spec, length - trim))
    for i in range(channels):
        one = host(stx.htdemucs_ispec(f, spec[i:i + 1].contiguous(), length - trim))
        assert np.array_equal(one, y[i:i + 1]), f"channel {i}"
    ref = orc.htdemucs_spec(x[channels - 1], 4096)
    assert snr_db(y[channels - 1], orc.htdemucs_ispec(ref, 4096, length - trim)) >= SNR_DB


def test_workspace_too_small(device):
    f = plan(2048)
    x = to_dev(_stereo(56, 20000), device)
    spec = stx.torch_stft(f, x, 441)
    ws = stx.workspace(stx.istft_workspace_size(f, 2, spec.shape[2]) - 4096, device)
    with pytest.raises(stx.StxError) as e:
        stx.torch_istft(f, spec, 441, workspace=ws)
    assert e.value.status == stx.STATUS_INVALID_ARGUMENT


# ----------------------------------------- st::VRFFT sizes (mixed-radix kernels on the device)
_any_plans = {}


def any_plan(n):
    if n not in _any_plans:
        _any_plans[n] = stx.FFT(n, any_size=True)
    return _any_plans[n]


@pytest.mark.parametrize("n", [7680, 3840, 960, 640, 320, 480, 6000])
def test_fft_run_any_size(device, orc, n):
    """Complex transforms of VRFFT's sizes against the oracle's Bluestein (src/vr_dsp.h:11-37)."""
    v = synth.normal(n + 1, (3, 2 * n), 1.0).astype(np.float64)
    a = (v[:, 0::2] + 1j * v[:, 1::2]).astype(np.complex64)
    d = to_dev(a, device)
    any_plan(n).run(d)
    fw = host(d)
    any_plan(n).run(d, inverse=True)
    back = host(d) / n
    for b in range(3):
        assert snr_db(fw[b], orc.vrfft(a[b].astype(np.complex128))) >= SNR_DB
        assert snr_db(back[b], a[b]) >= SNR_DB


@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
@pytest.mark.parametrize("normalized", [False, True])
def test_torch_stft_7680_kim_chunk(device, orc, layout, normalized):
    """Kim_Vocal_2's transform (src/tfc_tdf.cpp:355-359): n_fft 7680, hop 1024, one chunk of
    1024 x 255 = 261,120 stereo samples -> [2][3841][256]; STFT and the workspace iSTFT."""
    length, n, hop = 261120, 7680, 1024
    x = _stereo(7680, length)
    f = any_plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop, normalized, layout=layout)
    ws = stx.workspace(stx.istft_workspace_size(f, 2, length // hop + 1), device)
    y = stx.torch_istft(f, spec, hop, normalized, layout=layout, workspace=ws)
    spec_h, y_h = host(spec), host(y)
    if layout == stx.T_MAJOR:
        spec_h = spec_h.transpose(0, 2, 1)
    assert spec_h.shape == (2, 3841, 256)
    for c in range(2):
        ref = orc.torch_stft(x[c], n, hop, normalized)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y_h[c], orc.torch_istft(ref, n, hop, normalized)) >= SNR_DB
    # A workspace only 4-byte aligned (the frames are then stored a float at a time): same bits.
    ws_odd = stx.workspace(stx.istft_workspace_size(f, 2, length // hop + 1) + 4, device)[1:]
    y_odd = host(stx.torch_istft(f, spec, hop, normalized, layout=layout, workspace=ws_odd))
    assert np.array_equal(y_odd, y_h)


@pytest.mark.parametrize("n,hop", [(320, 80), (640, 160), (960, 240), (1536, 256)])
@pytest.mark.parametrize("extra", [3, "hop"])
def test_torch_stft_vr_sizes_round_trip(device, orc, n, hop, extra):
    """An odd frame count (length 20 n + 3) and an even one (20 n + hop): the f-major iSTFT
    transforms two frames per block when the count is even."""
    length = 20 * n + (hop if extra == "hop" else extra)
    x = _stereo(n, length, 0.5)
    f = any_plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), hop)
    ws = stx.workspace(stx.istft_workspace_size(f, 2, length // hop + 1), device)
    y = stx.torch_istft(f, spec, hop, workspace=ws)
    spec_h, y_h = host(spec), host(y)
    for c in range(2):
        ref = orc.torch_stft(x[c], n, hop)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y_h[c], orc.torch_istft(ref, n, hop)) >= SNR_DB


@pytest.mark.parametrize("n,hop,frames", [(960, 240, 82), (7680, 1024, 32)])
def test_mixed_pairs_unaligned_spectrum(device, n, hop, frames):
    """The mixed-radix STFT and iSTFT transform two f-major frames per block when the frame count
    is even and the spectrum 16-byte aligned; a spectrum 8 bytes off that takes one frame per
    block. Both give the same bits (the run-time plan at 960 and the compiled one at 7680)."""
    import torch
    length = (frames - 1) * hop
    x = to_dev(_stereo(n, length, 0.5), device)
    f = any_plan(n)
    F, T = n // 2 + 1, length // hop + 1
    assert T == frames
    a = stx.torch_stft(f, x, hop)
    assert a.data_ptr() % 16 == 0
    buf = torch.empty(2 * 2 * F * T + 2, dtype=torch.float32, device=x.device)
    b = buf[2:].view(torch.complex64).view(2, F, T)
    assert b.data_ptr() % 16 == 8
    stx.torch_stft(f, x, hop, out=b)
    assert np.array_equal(host(a), host(b))
    ws = stx.workspace(stx.istft_workspace_size(f, 2, T), device)
    ya = host(stx.torch_istft(f, a, hop, workspace=ws))
    yb = host(stx.torch_istft(f, b, hop, workspace=ws))
    assert np.array_equal(ya, yb)


# n_fft with 9 .. 1,000 points in the half transform (16, 32 and 64 threads a frame, plans that start with radix 16
# and not, the limits 240 | 250, 480 | 486, 960 | 1,000), hops from n / 8 to n, ends inside a tile of 16 frames,
# tiles and workgroups that cross channels, and frames just below and above the switch to them (1,024 where the plan
# starts with radix 16).
FRAME_CASES = [(960, 480, 3, 1023 * 160 + 7), (320, 80, 2, 80 * 600 + 3), (320, 106, 1, 106 * 1024), (480, 60, 2, 60 * 700 + 59),
               (500, 125, 2, 125 * 530), (972, 243, 2, 243 * 520 + 1), (18, 9, 2, 9 * 900 + 4), (48, 48, 1, 48 * 1100),
               (640, 640, 2, 640 * 520), (1536, 512, 3, 512 * 400 + 100), (1920, 480, 2, 480 * 515), (2000, 500, 2, 500 * 512),
               (2000, 250, 4, 250 * 256), (960, 240, 1, 240 * 1022), (960, 240, 1, 240 * 1023), (960, 100, 2, 100 * 520),
               # Even hops whose output begins at an odd sample of the frames' grid (n / 2 odd).
               (18, 6, 2, 6 * 1100 + 5), (50, 10, 3, 10 * 700), (810, 202, 2, 202 * 600 + 1),
               # 128 and 256 threads a frame (above 512 frames): the compiled plan, plans that start with radix 15 and 8,
               # 1,920 | 2,025 and 3,840 points, odd frame counts, a size that stays with one frame a workgroup (8100).
               (7680, 1024, 3, 1024 * 255 + 9), (7680, 1920, 2, 1920 * 256), (7680, 1024, 2, 1024 * 255), (3840, 960, 2, 960 * 272),
               (4050, 1350, 4, 1350 * 130 + 1), (6000, 1500, 3, 1500 * 200), (2160, 540, 3, 540 * 200 + 2), (8192 - 192, 1000, 3, 1000 * 180),
               (6144, 6144, 3, 6144 * 180), (8100, 2025, 3, 2025 * 180),
               # Plans that do not start with radix 16 on both sides of their own switch: 1,536 frames up to 64 threads a frame,
               # 640 (f-major) and 1,280 (t-major) with 256; n_fft 7680 where its t-major iSTFT takes one frame a workgroup.
               (500, 125, 2, 125 * 766), (500, 125, 2, 125 * 767), (972, 243, 2, 243 * 780 + 1), (18, 9, 2, 9 * 1500 + 4),
               (18, 6, 2, 6 * 1600 + 5), (810, 202, 2, 202 * 800 + 1), (2000, 500, 2, 500 * 800), (2000, 250, 4, 250 * 400),
               (1350, 450, 2, 450 * 790), (4050, 1350, 2, 1350 * 319), (4050, 1350, 3, 1350 * 256), (4050, 1350, 4, 1350 * 330 + 1),
               (6000, 1500, 4, 1500 * 330), (7290, 2430, 5, 2430 * 257), (7680, 1024, 4, 1024 * 270), (7680, 1920, 4, 1920 * 330)]


# Hops of 4 n and less (fused tiles) and above (two kernels), for calls of many frames.
@pytest.mark.parametrize("n,hop,frames", [(320, 1280, 1100), (320, 1284, 1100), (960, 1500, 1030), (96, 9600, 1025), (2000, 9001, 1600)])
@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
def test_mixed_istft_hop_above_n(device, n, hop, frames, layout):
    """Frames that do not meet: the samples that a frame covers against the same frames laid n apart, the others 0. Both
    sum one windowed frame and divide by the window's square; the transforms' plan is the same at both hops."""
    x = synth.normal(4700 + n + hop, (1, frames * n), 0.2)
    f = any_plan(n)
    spec = stx.torch_stft(f, to_dev(x, device), n, layout=layout)
    ws = stx.workspace(stx.istft_workspace_size(f, 1, frames + 1), device)
    y = host(stx.torch_istft(f, spec, hop, layout=layout, workspace=ws))
    close = host(stx.torch_istft(f, spec, n, layout=layout, workspace=ws))
    J = np.arange(y.shape[1]) + n // 2
    R = J % hop
    assert np.all(y[:, R >= n] == 0.0)
    covered = (J // hop) * n + R - n // 2
    sel = (R < n) & (covered < close.shape[1]) & (covered >= 0)
    w = 0.5 - 0.5 * np.cos(2.0 * np.pi * R[sel] / n)         # a sample is w x / w^2: compare w y, the frame
    assert snr_db(y[:, sel] * w, close[:, covered[sel]] * w) >= SNR_DB


@pytest.mark.parametrize("n,hop,channels,length", FRAME_CASES)
@pytest.mark.parametrize("layout", [stx.F_MAJOR, stx.T_MAJOR])
def test_mixed_many_frames(device, orc, n, hop, channels, length, layout):
    """Mixed-radix STFT and iSTFT of calls with many frames (16 frames a workgroup) against the oracle."""
    x = synth.normal(n + hop, (channels, length), 0.3)
    f = any_plan(n)
    T = length // hop + 1
    spec = stx.torch_stft(f, to_dev(x, device), hop, layout=layout)
    ws = stx.workspace(stx.istft_workspace_size(f, channels, T) + 4, device)
    y = host(stx.torch_istft(f, spec, hop, layout=layout, workspace=ws))
    assert np.array_equal(y, host(stx.torch_istft(f, spec, hop, layout=layout, workspace=ws[1:])))   # 4-byte aligned
    spec_h = host(spec)
    if layout == stx.T_MAJOR:
        spec_h = spec_h.transpose(0, 2, 1)
    weight = frame_weight(n, hop, T)
    for c in {0, channels - 1}:
        ref = orc.torch_stft(x[c], n, hop)
        assert snr_db(spec_h[c], ref) >= SNR_DB
        assert snr_db(y[c] * weight, orc.torch_istft(ref, n, hop) * weight) >= SNR_DB


def test_any_size_errors(device):
    import torch
    for n in (7, 14, 22, 20000):
        with pytest.raises(stx.StxError) as e:
            stx.FFT(n, any_size=True)
        assert e.value.status == stx.STATUS_UNSUPPORTED
    with pytest.raises(stx.StxError) as e:
        stx.FFT(7680)                                              # st::FFT: powers of two only
    assert e.value.status == stx.STATUS_INVALID_ARGUMENT
    assert any_plan(2048).n == 2048                                 # a power of two: the radix-16 plan
    f = any_plan(7680)
    x = torch.zeros((1, 20000), dtype=torch.float32, device=device)
    spec = stx.torch_stft(f, x, 1024)
    with pytest.raises(stx.StxError) as e:
        stx.torch_istft(f, spec, 1024)                             # needs the workspace variant
    assert e.value.status == stx.STATUS_UNSUPPORTED
    with pytest.raises(stx.StxError) as e:
        stx.htdemucs_spec(f, x)
    assert e.value.status == stx.STATUS_UNSUPPORTED
