"""The wavefront kernel's step-by-step hand-off between layers, at the sizes where its ring and its
unrolled blocks of steps can go wrong: sequences shorter than the pipeline, one step around a block (8) and
around a lap of the ring (32), several laps; 8- and 16-row tiles; ragged rows; NaN and large frozen h0.

Bound against the oracle's restatement of the device rounding (fp16 h, fp32 sums): a flipped fp16
rounding of one h moves the final state by a few fp16 ulps of 1 (2^-11 each), so 2e-3."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_regressor, make_x, oracle_layers
from oracle import oracle
from persistent_lstm_hip_amd import PersistentLSTM, PersistentLSTMRegressor

pytestmark = pytest.mark.gpu
BOUND = 2e-3


def _lstm(native):
    return PersistentLSTM.from_native_module(native.lstm).to("cuda").half().eval()


def _oracle(native, x, **kw):
    return oracle.lstm_forward(x.half().float().numpy(), oracle_layers(native.lstm, half=True), want_seq=True,
                               numerics="ref_fp16", **kw)


@pytest.mark.parametrize("T", [1, 2, 3, 4, 7, 8, 9, 11, 12, 13, 31, 32, 33, 40, 63, 65, 100])
@pytest.mark.parametrize("H,L,B", [(20, 3, 9), (64, 2, 17), (128, 4, 5)])
def test_lengths_around_the_ring(gpu, H, L, B, T):
    print(f"[gpu-case] hand-off H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(6, H, L, 3)
    x = make_x(B, T, 6, seed=T)
    out, (h, c) = _lstm(native)(x.to("cuda", torch.float16))
    gpu.check_status(torch.device("cuda"))
    want = _oracle(native, x)
    assert np.abs(out.float().cpu().numpy() - want["out_seq"]).max() <= BOUND
    assert np.abs(h.float().cpu().numpy() - want["h_n"]).max() <= BOUND
    assert np.abs(c.float().cpu().numpy() - want["c_n"]).max() <= 2 * BOUND


@pytest.mark.parametrize("H,L,B,T", [(128, 2, 1100, 41), (60, 4, 40, 70), (128, 5, 400, 70)])
def test_ragged_rows_and_tiles(gpu, H, L, B, T):
    """16-row tiles (1100 rows) and 8-row tiles, of five layers on different XCDs too (50 tiles, which the grid
    has no room to round up); lengths 0 .. T, rows of length 0 with |h0| up to 3."""
    print(f"[gpu-case] hand-off ragged H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(5, H, L, 3)
    x = make_x(B, T, 5, seed=3)
    g = torch.Generator().manual_seed(4)
    lengths = torch.randint(0, T + 1, (B,), generator=g)
    lengths[::7] = 0
    h0 = (torch.rand(L, B, H, generator=g) * 2 - 1).half()
    h0[:, lengths == 0] *= 3
    c0 = torch.randn(L, B, H, generator=g).half()
    model = _lstm(native)
    blob = model.packed_blob(torch.device("cuda", torch.cuda.current_device()))
    res = gpu.forward(blob, (5, H, L, 0), x.to("cuda", torch.float16), lengths=lengths, h0=h0.cuda(), c0=c0.cuda(),
                      want_out=False, want_seq=True, want_state=True, check_status=True)
    rows = np.unique(np.r_[0:16, B - 16:B, np.arange(0, B, 7)[:12]])
    want = _oracle(native, x[rows], lengths=lengths.numpy()[rows], h0=h0.float().numpy()[:, rows],
                   c0=c0.float().numpy()[:, rows])
    assert np.abs(res["out_seq"].float().cpu().numpy()[rows] - want["out_seq"]).max() <= BOUND
    assert np.abs(res["h_n"].float().cpu().numpy()[:, rows] - want["h_n"]).max() <= BOUND


@pytest.mark.parametrize("B", [12, 1100])
def test_nan_stays_in_its_row(gpu, B):
    """A NaN input: NaN in that row of every layer from that step on, every other row unchanged."""
    H, L, T, bad, at = 128, 2, 45, 3, 20
    print(f"[gpu-case] hand-off NaN B={B}", flush=True)
    model = _lstm(make_regressor(5, H, L, 3))
    x = make_x(B, T, 5, seed=9).to("cuda", torch.float16)
    ref = model(x)[0]
    xn = x.clone()
    xn[bad, at] = float("nan")
    got, (h, _) = model(xn)
    gpu.check_status(torch.device("cuda"))
    keep = torch.arange(B) != bad
    assert torch.equal(got[keep], ref[keep])
    assert torch.equal(got[bad, :at], ref[bad, :at])
    assert torch.isnan(got[bad, at:]).all() and torch.isnan(h[:, bad]).all()


@pytest.mark.parametrize("I,H,L,B,T", [
    (129, 128, 1, 3, 1),      # one layer, one step, half a 16-row block
    (300, 60, 3, 17, 33),     # three 8-row tiles: T * rows not a multiple of 16
    (200, 100, 2, 1100, 4),   # 16-row tiles
    (150, 128, 4, 9, 47),     # four layers: rings larger than the layer sequences' place, layer by layer
    (150, 128, 4, 9, 48),     # ... and just fitting it
    (140, 120, 2, 2100, 3),   # more rows than one launch holds
])
def test_wide_inputs(gpu, I, H, L, B, T):
    """Inputs wider than the padded hidden size: layer 0's projections are rounded to fp16 (half an ulp of
    a pre-activation below 4 is 2^-10, and a gate moves by at most that), on top of BOUND."""
    print(f"[gpu-case] wide I={I} H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(I, H, L, 3)
    x = make_x(B, T, I, seed=7)
    lengths = torch.randint(0, T + 1, (B,), generator=torch.Generator().manual_seed(5))
    model = _lstm(native)
    blob = model.packed_blob(torch.device("cuda", torch.cuda.current_device()))
    rows = np.unique(np.r_[0:min(B, 9), max(0, B - 9):B])
    for lens in (None, lengths):
        res = gpu.forward(blob, (I, H, L, 0), x.to("cuda", torch.float16), lengths=lens, want_out=False, want_seq=True,
                          want_state=True, check_status=True)
        want = _oracle(native, x[rows], lengths=None if lens is None else lens.numpy()[rows])
        assert np.abs(res["out_seq"].float().cpu().numpy()[rows] - want["out_seq"]).max() <= 2 * BOUND
        assert np.abs(res["h_n"].float().cpu().numpy()[:, rows] - want["h_n"]).max() <= 2 * BOUND


def _verdict_end(L, B):
    """End of the status and counter words of a wavefront forward in 8-row tiles: 256 bytes, then a word per
    (layer, tile), rounded up to 256 bytes."""
    return 256 + (4 * L * ((B + 7) // 8) + 255) // 256 * 256


@pytest.mark.parametrize("I,H,L,B,T", [(5, 128, 4, 512, 60), (1, 20, 1, 2, 1), (9, 64, 2, 33, 17), (128, 128, 2, 9, 40)])
def test_equal_rows_found_on_the_device(gpu, monkeypatch, I, H, L, B, T):
    """Equal rows, and equal but for one element (the last one, the first one of row 1, the middle of a row):
    the outputs are bit for bit those of a forward without detection, and the verdict words (behind the status
    word, one per block of the prologue) are all zero for equal rows and only for them."""
    print(f"[gpu-case] uniform I={I} H={H} L={L} B={B} T={T}", flush=True)
    model = PersistentLSTMRegressor.from_native_module(make_regressor(I, H, L, 11)).to("cuda").half().eval()
    assert gpu.detects_uniform((I, H, L, 11), B, T, torch.device("cuda"))
    row = make_x(1, T, I, seed=2).to("cuda", torch.float16)
    for where in (None, (B - 1, T - 1, I - 1), (1, 0, 0), (B // 2, T // 2, I // 2)):
        x = row.expand(B, T, I).contiguous()
        if where is not None and where[0] > 0:
            x[where] += 1
        monkeypatch.setenv("PERSISTENT_LSTM_HIP_UNIFORM_BATCH", "auto")
        model(x)  # (a workspace large enough exists from here on)
        words = gpu.workspace(x.device, 256)[:_verdict_end(L, B)].view(torch.int32)[1:]
        words.fill_(-1)  # nothing reads them before the prologue has written its own
        got = model(x)
        gpu.check_status(torch.device("cuda"))
        written = words[words != -1]
        assert written.numel() > 0 and torch.equal(words[:written.numel()], written)
        assert bool((written != 0).any()) == (where is not None and where[0] > 0), where
        monkeypatch.setenv("PERSISTENT_LSTM_HIP_UNIFORM_BATCH", "0")
        assert torch.equal(got, model(x)), where


@pytest.mark.parametrize("I,H,L,B,T,edge", [
    (5, 128, 4, 1060, 40, 1024),    # 1024 rows in 16-row tiles, 36 in 8-row tiles
    (5, 200, 4, 530, 12, 512),      # two tiles per workgroup, then one
    (5, 400, 4, 540, 12, 512),      # layer by layer, then all layers at once
    (300, 256, 2, 1030, 5, 1024),   # layer by layer twice
    (5, 600, 2, 140, 6, 128),       # padded H 1024: 128 rows, then 12
])
def test_rows_after_the_last_full_launch(gpu, I, H, L, B, T, edge):
    """A forward in several launches whose last one takes another plan: rows on both sides of the `edge` between
    them against the oracle (layer-sequential rows also round their projections, as above), states and sequence
    included."""
    print(f"[gpu-case] remainder I={I} H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(I, H, L, 3)
    x = make_x(B, T, I, seed=8)
    out, (h, c) = _lstm(native)(x.to("cuda", torch.float16))
    gpu.check_status(torch.device("cuda"))
    rows = np.unique(np.r_[0:4, edge - 6:min(edge + 8, B), B - 4:B])
    want = _oracle(native, x[rows])
    assert np.abs(out.float().cpu().numpy()[rows] - want["out_seq"]).max() <= 2 * BOUND
    assert np.abs(h.float().cpu().numpy()[:, rows] - want["h_n"]).max() <= 2 * BOUND


@pytest.mark.parametrize("I,H,L,B,T,lengths", [
    (300, 128, 3, 1500, 8, False),    # 1280 rows and 220 in the workspace of all
    (300, 60, 8, 800, 100, True),     # 512 and 288
    (150, 128, 6, 2100, 8, False),    # four launches on a short sequence: layer by layer
    (150, 128, 6, 2100, 40, True),    # ... and all layers at once
    (129, 128, 8, 4300, 9, False),    # more rows than a layer-by-layer launch holds
])
def test_wide_inputs_in_several_launches(gpu, I, H, L, B, T, lengths):
    """Wide inputs whose batch takes several launches: every row is computed by the same kernels (their projections
    are rounded alike), so equal rows are equal bit for bit on both sides of every launch boundary; the first ones
    against the oracle (bound as in test_wide_inputs)."""
    print(f"[gpu-case] wide launches I={I} H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(I, H, L, 3)
    few = make_x(3, T, I, seed=7)
    lens = torch.tensor([T, T // 2, T - 1])
    which = torch.arange(B) % 3
    model = _lstm(native)
    blob = model.packed_blob(torch.device("cuda", torch.cuda.current_device()))
    res = gpu.forward(blob, (I, H, L, 0), few.to("cuda", torch.float16)[which.cuda()],
                      lengths=lens[which] if lengths else None, want_out=False, want_seq=True, want_state=True,
                      check_status=True)
    for key, dim in (("out_seq", 0), ("h_n", 1), ("c_n", 1)):
        same = torch.equal(res[key], res[key].index_select(dim, which.cuda()))
        assert same, key
    want = _oracle(native, few, lengths=lens.numpy() if lengths else None)
    assert np.abs(res["out_seq"][:3].float().cpu().numpy() - want["out_seq"]).max() <= 2 * BOUND
    assert np.abs(res["h_n"][:, :3].float().cpu().numpy() - want["h_n"]).max() <= 2 * BOUND


@pytest.mark.parametrize("I,H,L,B,T,same", [
    (5, 400, 4, 740, 12, True),    # 512 rows and 228, which four launches would take: layer by layer too
    (5, 512, 2, 700, 9, True),     # ... two launches of the sliced kernel
    (5, 300, 3, 740, 20, True),
    (100, 512, 4, 560, 12, False),  # one launch: all layers at once (projections of layers >= 1 in fp32)
])
def test_path_of_the_rows_after_a_layer_sequential_launch(gpu, I, H, L, B, T, same):
    """Padded H 512: the rows after the last full launch change to the sliced kernel only where that is faster.
    Elsewhere all rows are computed alike, so equal rows are equal bit for bit; the oracle's bound holds for both."""
    print(f"[gpu-case] H512 remainder I={I} H={H} L={L} B={B} T={T}", flush=True)
    native = make_regressor(I, H, L, 3)
    few = make_x(3, T, I, seed=7)
    which = torch.arange(B) % 3
    out, (h, c) = _lstm(native)(few.to("cuda", torch.float16)[which.cuda()])
    gpu.check_status(torch.device("cuda"))
    alike = torch.equal(out, out[:3][which.cuda()]) and torch.equal(c, c[:, :3][:, which.cuda()])
    assert alike == same
    want = _oracle(native, few)
    ends = np.r_[0:3, B - 3:B]
    assert np.abs(out[ends].float().cpu().numpy() - want["out_seq"][ends % 3]).max() <= 2 * BOUND
    assert np.abs(h[:, ends].float().cpu().numpy() - want["h_n"][:, ends % 3]).max() <= 2 * BOUND
