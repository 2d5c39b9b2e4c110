"""The mel front end on the MI355X against the oracle
(oracle_mel_spectrogram, pinned in tests/test_mel_oracle.py), as
Tests/Mel/MelSpectrogramTests.cpp checks it: the reduced shape cell by cell
within 1e-4, and Whisper's own shape (30 s, 80 bands, 3000 frames) with a
silent first second, whose output spans exactly two, plus the oracle's cells.
Then the chain into the encoder: the GPU mel fed to the GPU encoder against
the oracle's mel fed to the oracle's encoder."""

import numpy as np
import pytest
import torch

from whispereacp_amd import synthetic as S

pytestmark = pytest.mark.gpu


def gpu_mel(shape, samples, filters):
    from whispereacp_amd.mel import MelSpectrogram
    front = MelSpectrogram(shape)
    out = torch.empty((shape.mel_count, shape.frame_count), dtype=torch.float32, device="cuda")
    front.encode(torch.from_numpy(samples).cuda(), torch.from_numpy(filters).cuda(), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def test_reduced_shape_matches_oracle(oracle):
    s = S.reduced_mel_shape()
    x = S.tone_and_noise(s.sample_count)
    f = S.triangular_filters(s.mel_count, s.bin_count)
    got = gpu_mel(s, x, f)
    expected = oracle.mel_spectrogram(x, f, s.fft_length, s.hop_length, s.frame_count)
    err = float(np.max(np.abs(got - expected)))
    print(f"reduced mel: worst absolute error {err:.2e}")
    assert err <= 1e-4


@pytest.mark.parametrize("samples,fft,hop,frames,mels", [
    (4000, 400, 160, 17, 81),    # one frame past a block of sixteen, one band past a tile
    (3000, 33, 7, 31, 5),        # an odd transform: no middle term
    (40000, 2048, 512, 40, 24),  # too long for one block's memory: the product launches
])
def test_other_shapes_match_oracle(oracle, samples, fft, hop, frames, mels):
    s = S.MelShape(samples, fft, hop, frames, mels)
    x = S.tone_and_noise(s.sample_count)
    f = S.triangular_filters(s.mel_count, s.bin_count)
    got = gpu_mel(s, x, f)
    expected = oracle.mel_spectrogram(x, f, s.fft_length, s.hop_length, s.frame_count)
    assert float(np.max(np.abs(got - expected))) <= 1e-4


@pytest.mark.parametrize("samples,fft,hop,frames,mels", [
    (8000, 600, 160, 33, 20),    # more values of a folded row than one pass of a block folds
    (8000, 602, 160, 33, 20),    # the same folded once
    (20000, 1024, 160, 40, 80),  # and a filterbank too large to go through the block's memory
    (4000, 400, 160, 17, 200)])  # as is one of many bands
def test_longer_transforms_and_filterbanks_match_oracle(oracle, samples, fft, hop, frames, mels):
    s = S.MelShape(samples, fft, hop, frames, mels)
    x = S.tone_and_noise(s.sample_count)
    f = S.triangular_filters(s.mel_count, s.bin_count)
    got = gpu_mel(s, x, f)
    expected = oracle.mel_spectrogram(x, f, s.fft_length, s.hop_length, s.frame_count)
    assert float(np.max(np.abs(got - expected))) <= 1e-4


def test_a_filterbank_may_start_at_any_float(oracle):
    # One float past a 16-byte boundary it is read from memory: the same sums.
    from whispereacp_amd.mel import MelSpectrogram
    s = S.reduced_mel_shape()
    x, f = S.tone_and_noise(s.sample_count), S.triangular_filters(s.mel_count, s.bin_count)
    moved = torch.empty(f.size + 1, dtype=torch.float32, device="cuda")[1:].reshape(f.shape)
    moved.copy_(torch.from_numpy(f))
    assert moved.data_ptr() % 16 == 4
    out = torch.empty((s.mel_count, s.frame_count), dtype=torch.float32, device="cuda")
    MelSpectrogram(s).encode(torch.from_numpy(x).cuda(), moved, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), gpu_mel(s, x, f))


def test_whisper_shape_spans_two_and_matches_oracle(oracle):
    s = S.MelShape()
    x = S.tone_and_noise(s.sample_count)
    x[:16000] = 0.0   # a silent first second reaches the floor
    f = S.triangular_filters(s.mel_count, s.bin_count)
    got = gpu_mel(s, x, f)
    assert got.shape == (80, 3000)
    assert abs((got.max() - got.min()) - 2.0) <= 1e-5
    expected = oracle.mel_spectrogram(x, f, s.fft_length, s.hop_length, s.frame_count)
    err = float(np.max(np.abs(got - expected)))
    print(f"whisper-shape mel: worst absolute error {err:.2e}")
    assert err <= 1e-4


def test_mel_into_encoder_matches_the_oracle_chain(oracle):
    from whispereacp_amd.encoder import Encoder, EncoderWeights
    from whispereacp_amd.mel import MelSpectrogram
    s = S.MelShape()
    x = S.tone_and_noise(s.sample_count)
    f = S.triangular_filters(s.mel_count, s.bin_count)
    shape = S.encoder_workload_shape("tiny.en")
    encoder_file = S.workload_encoder_file(shape, "F16", 3000)
    front = MelSpectrogram(s)
    mel = torch.empty((80, 3000), dtype=torch.float32, device="cuda")
    front.encode(torch.from_numpy(x).cuda(), torch.from_numpy(f).cuda(), mel)
    rows = torch.empty((shape.positions(), shape.width), dtype=torch.float32, device="cuda")
    Encoder(shape).encode(mel, EncoderWeights(shape, encoder_file), rows)
    torch.cuda.synchronize()
    mel_expected = oracle.mel_spectrogram(x, f, s.fft_length, s.hop_length, s.frame_count)
    tensors = [encoder_file[n].floats() for n in S.encoder_canonical_names(shape.layers)]
    expected = oracle.encode(shape, tensors, mel_expected.astype(np.float32))
    got = rows.cpu().numpy()
    err = float(np.max(np.abs(got - expected) / (1 + np.abs(expected))))
    print(f"mel -> tiny.en encoder: worst error {err:.2e}")
    assert err <= 1e-4
