"""AudioVAE V2's streaming decoder (vx_vae) on the GPU against the CPU
oracle's whole-sequence decode (vae.cpp:415-481; the reference's
vae_test compares streamed and at-once decoding, vae_test.cpp:114-138):
chunks of latents decoded in turn equal the whole sequence decoded at
once; a reset starts a new stream; graph replays with the same buffers
match. Tolerance: float32 products in another summation order through
the decoder's 25 layers and Snake on the hardware sine, max |gpu -
oracle| <= 2e-3 on samples in [-1, 1] (measured 5.1e-6 small, 7.7e-4 at
the VoxCPM2 shape)."""
import numpy as np
import pytest
import torch

from voxcpm_amd import _lib, synth

pytestmark = pytest.mark.gpu

BOUND = 2e-3

# "small" and "odd" take channel counts that are not multiples of 16 (8;
# 24 and 12): their products go to the LDS-tiled float32 kernel
# (F32TileKernel), whose epilogue makes the next inputs (unit windows, a
# block's input, the output window) as the 16-column kernel's does. Units
# of at most 256 channels (and the latents' input convolutions) make their
# depthwise convolution in the pointwise product's operand loads; chunks
# of 1, 5 and 2 frames at the VoxCPM2 shape take one- and two-tile row
# blocks and latents' histories that mix the previous chunk's rows with
# this chunk's (fewer than 6 frames).
# "split": a transposed convolution of k = 2080 over 1560 columns at a
# few rows splits k over 32 x 32 tiles (the last column tile partial) and a
# second launch adds the splits; its 520-channel units take depthwise
# launches and the LDS-tiled kernel (520 is not a multiple of 16).
CONFIGS = {
    "small": synth.VaeConfig(latent=16, decoder_dim=64, rates=(3, 2, 2)),
    "odd": synth.VaeConfig(latent=16, decoder_dim=48, rates=(2, 2)),
    "split": synth.VaeConfig(latent=16, decoder_dim=1040, rates=(3,)),
    "voxcpm2": synth.VOXCPM2_VAE,
}


@pytest.mark.parametrize("name,chunks", [("small", (4, 4, 1)), ("small", (9,)),
                                         ("odd", (3, 2, 5)), ("split", (4, 3, 1)),
                                         ("voxcpm2", (4, 4)), ("voxcpm2", (1, 5, 2))])
def test_vae_streaming_decode_against_oracle(vx, oracle, cuda, stream, name, chunks):
    config = CONFIGS[name]
    weights = synth.vae_weights(config, 91)
    frames = sum(chunks)
    rng = synth.Rng(92, frames)
    latents = rng.normal(frames * config.latent).astype(np.float32).reshape(frames, config.latent)
    ref = oracle.OracleVae(weights).decode(latents)
    vae = vx.Vae(weights)
    assert vae.hop == config.hop
    device_latents = torch.from_numpy(latents).to(cuda)
    for attempt in range(2):  # the second stream after a reset
        pieces, at = [], 0
        for n in chunks:
            pieces.append(vae.decode(device_latents[at:at + n]).cpu().numpy())
            at += n
        got = np.concatenate(pieces)
        error = float(np.max(np.abs(got - ref)))
        print(f"{name} {chunks} stream {attempt}: max |d| {error:.2e}, "
              f"signal std {np.std(ref):.3f}", flush=True)
        assert error <= BOUND
        vae.reset()


def test_vae_graph_replays(vx, oracle, cuda, stream):
    """One chunk buffer decoded again and again (the patch loop): the first
    call runs eagerly, later ones replay one graph; every chunk matches the
    oracle's decode of the whole sequence so far."""
    config = CONFIGS["small"]
    weights = synth.vae_weights(config, 93)
    rng = synth.Rng(94, 1)
    latents = rng.normal(5 * 4 * config.latent).astype(np.float32).reshape(20, config.latent)
    ref = oracle.OracleVae(weights).decode(latents)
    vae = vx.Vae(weights)
    chunk = torch.empty((4, config.latent), dtype=torch.float32, device=cuda)
    samples = torch.empty(4 * config.hop, dtype=torch.float32, device=cuda)
    for i in range(5):
        chunk.copy_(torch.from_numpy(latents[4 * i:4 * i + 4]))
        vae.decode(chunk, samples)
        got = samples.cpu().numpy()
        want = ref[4 * i * config.hop:4 * (i + 1) * config.hop]
        assert float(np.max(np.abs(got - want))) <= BOUND, i


def test_vae_chunk_limit(vx, cuda):
    """A chunk of more frames than vx_vae_max_frames is refused before any
    launch (a product's 32-row blocks are grid rows, at most 65535)."""
    config = CONFIGS["small"]
    vae = vx.Vae(synth.vae_weights(config, 95))
    assert vae.max_frames == 65535 * 32 // config.hop
    latents = torch.zeros((vae.max_frames + 1, config.latent), dtype=torch.float32, device=cuda)
    with pytest.raises(_lib.VxError) as info:
        vae.decode(latents)
    assert info.value.status == _lib.VX_BAD_ARG


def test_vae_longest_chunk(vx, cuda):
    """A chunk of vx_vae_max_frames frames at the VoxCPM2 shape (1092: its
    32-row blocks fill the grid's 65535 rows at the output rate) decodes,
    and equals the same latents decoded in chunks of 16 frames (vae.cpp
    streams chunk by chunk; the two take different tilings, so the bound is
    the oracle tolerance)."""
    config = CONFIGS["voxcpm2"]
    weights = synth.vae_weights(config, 97)
    whole = vx.Vae(weights)
    frames = whole.max_frames
    assert frames == 65535 * 32 // config.hop
    rng = synth.Rng(98, frames)
    latents = torch.from_numpy(
        rng.normal(frames * config.latent).astype(np.float32).reshape(frames, config.latent)
    ).to(cuda)
    print(f"longest chunk: {frames} frames", flush=True)
    at_once = whole.decode(latents).cpu().numpy()
    chunked = vx.Vae(weights)
    pieces = [chunked.decode(latents[at:at + 16]).cpu().numpy() for at in range(0, frames, 16)]
    error = float(np.max(np.abs(at_once - np.concatenate(pieces))))
    print(f"longest chunk against 16-frame chunks: max |d| {error:.2e}", flush=True)
    assert np.all(np.isfinite(at_once))
    assert error <= BOUND


def test_vae_decode_argument_checks(vx, cuda):
    """The C ABI takes bare pointers: Vae.decode refuses tensors whose bytes
    are not float32 [frames][latent] rows (bf16, strided, wrong width) and
    sample buffers too small for the chunk, before any launch."""
    config = CONFIGS["small"]
    vae = vx.Vae(synth.vae_weights(config, 96))
    good = torch.zeros((4, config.latent), dtype=torch.float32, device=cuda)
    bad = [good.to(torch.bfloat16),
           torch.zeros((config.latent, 8), dtype=torch.float32, device=cuda).t()[:4],
           torch.zeros((4, config.latent + 1), dtype=torch.float32, device=cuda),
           good.reshape(-1)]
    for latents in bad:
        with pytest.raises(ValueError):
            vae.decode(latents)
    with pytest.raises(ValueError):
        vae.decode(good, torch.empty(4 * config.hop - 1, dtype=torch.float32, device=cuda))
    vae.decode(good, torch.empty(4 * config.hop, dtype=torch.float32, device=cuda))
    torch.cuda.synchronize()


# The wide path (float32 products as float16 pairs, units of 32 and 64 channels
# in one launch) takes chunks of 9 frames and more where it is the faster one,
# and here wherever it can: WIDE has a product per kind of block (128 channels
# by depthwise launch and product, 64 and 32 fused), row counts that fill no tile
# at every dilation, and shorter chunks between wide ones, whose histories
# the two paths share.
WIDE = synth.VaeConfig(latent=16, decoder_dim=256, rates=(8, 3, 2))


def wide_vae(vx, weights, frames):
    vae = vx.Vae(weights)
    vae.set_path(_lib.VAE_PATH_WIDE)
    assert vae.path(frames) == _lib.VAE_PATH_WIDE
    return vae


def test_vae_takes_the_faster_path(vx, cuda):
    """Sizes on which the two paths' measured times leave no doubt."""
    vae = vx.Vae(synth.vae_weights(WIDE, 100))
    assert vae.path(20) == _lib.VAE_PATH_FEW_ROWS and vae.path(96) == _lib.VAE_PATH_FEW_ROWS
    assert vae.path(500) == _lib.VAE_PATH_WIDE
    vae = vx.Vae(synth.vae_weights(CONFIGS["voxcpm2"], 100))
    assert vae.path(8) == _lib.VAE_PATH_FEW_ROWS
    assert all(vae.path(frames) == _lib.VAE_PATH_WIDE for frames in range(9, 127))
    vae.set_path(_lib.VAE_PATH_FEW_ROWS)
    assert vae.path(125) == _lib.VAE_PATH_FEW_ROWS


@pytest.mark.parametrize("chunks", [(20, 4, 31), (9, 9), (3, 50, 1, 10)])
def test_vae_wide_chunks_against_oracle(vx, oracle, cuda, stream, chunks):
    weights = synth.vae_weights(WIDE, 101)
    frames = sum(chunks)
    latents = synth.Rng(102, frames).normal(frames * WIDE.latent).astype(np.float32)
    latents = latents.reshape(frames, WIDE.latent)
    ref = oracle.OracleVae(weights).decode(latents)
    vae = wide_vae(vx, weights, max(chunks))
    device_latents = torch.from_numpy(latents).to(cuda)
    for attempt in range(3):  # the same buffers again: eager, captured, replayed
        pieces, at = [], 0
        for n in chunks:
            pieces.append(vae.decode(device_latents[at:at + n]).cpu().numpy())
            at += n
        error = float(np.max(np.abs(np.concatenate(pieces) - ref)))
        print(f"wide {chunks} stream {attempt}: max |d| {error:.2e}", flush=True)
        assert error <= BOUND
        vae.reset()


def test_vae_wide_past_float16(vx, oracle, cuda):
    """Activations of 1e6 (the input convolution scaled up, the output one
    scaled down): past float16's range the wide path's workgroups start over
    from bfloat16 triples."""
    weights = synth.vae_weights(WIDE, 103)
    weights.tensors["in_pointwise"] = weights.tensors["in_pointwise"] * np.float32(1e6)
    weights.tensors["out_conv"] = weights.tensors["out_conv"] * np.float32(1e-6)
    frames = 25
    latents = synth.Rng(104, frames).normal(frames * WIDE.latent).astype(np.float32)
    latents = latents.reshape(frames, WIDE.latent)
    ref = oracle.OracleVae(weights).decode(latents)
    got = wide_vae(vx, weights, frames).decode(torch.from_numpy(latents).to(cuda)).cpu().numpy()
    error = float(np.max(np.abs(got - ref)))
    print(f"past float16: max |d| {error:.2e}, signal std {np.std(ref):.3f}", flush=True)
    assert np.std(ref) > 0.1
    assert error <= BOUND


def test_vae_wide_against_short_chunks(vx, cuda):
    """61 frames at the VoxCPM2 shape at once (every product tile shape of
    the wide path) against the same latents in chunks of 8 frames, which
    take the float32 kernels."""
    config = CONFIGS["voxcpm2"]
    weights = synth.vae_weights(config, 105)
    frames = 61
    latents = torch.from_numpy(synth.Rng(106, frames).normal(frames * config.latent).astype(
        np.float32).reshape(frames, config.latent)).to(cuda)
    at_once = vx.Vae(weights).decode(latents).cpu().numpy()
    chunked = vx.Vae(weights)
    pieces = [chunked.decode(latents[at:at + 8]).cpu().numpy() for at in range(0, frames, 8)]
    error = float(np.max(np.abs(at_once - np.concatenate(pieces))))
    print(f"wide against 8-frame chunks: max |d| {error:.2e}", flush=True)
    assert error <= BOUND


def scaled_blocks(weights, scale):
    """Every decoder block's residual stream times `scale` (a power of two):
    its transposed convolution and its units' biases scaled, the next block's
    input (of the last block the output convolution) scaled back."""
    blocks = weights.tensors["blocks"]
    for b, block in enumerate(blocks):
        for name in ("up", "up_bias"):
            block[name] = block[name] * np.float32(scale)
        for unit in block["units"]:
            for name in ("depthwise_bias", "pointwise_bias"):
                unit[name] = unit[name] * np.float32(scale)
        if b + 1 < len(blocks):
            blocks[b + 1]["scale"] = blocks[b + 1]["scale"] * np.float32(1 / scale)
    weights.tensors["out_conv"] = weights.tensors["out_conv"] * np.float32(1 / scale)


@pytest.mark.parametrize("scale", [2.0**-18, 2.0**-30, 2.0**-45])
def test_vae_wide_below_float16(vx, oracle, cuda, scale):
    """Weights and activations below the float16 pairs' range, scaled back
    where a block hands its rows on: the wide path's workgroups start over
    from bfloat16 triples. The bound: the float32 products' measured 5.1e-6
    (module docstring), with a factor of four for these weights."""
    weights = synth.vae_weights(WIDE, 107)
    scaled_blocks(weights, scale)
    frames = 25
    latents = synth.Rng(108, frames).normal(frames * WIDE.latent).astype(np.float32)
    latents = latents.reshape(frames, WIDE.latent)
    ref = oracle.OracleVae(weights).decode(latents)
    got = wide_vae(vx, weights, frames).decode(torch.from_numpy(latents).to(cuda)).cpu().numpy()
    error = float(np.max(np.abs(got - ref)))
    print(f"blocks scaled by {scale:.1e}: max |d| {error:.2e}, signal std {np.std(ref):.3f}",
          flush=True)
    assert np.std(ref) > 0.1
    assert error <= 2e-5


@pytest.mark.parametrize("direction", ["past", "below"])
def test_vae_wide_out_of_range_tiles(vx, cuda, direction):
    """Operands outside the float16 pairs' range in every product tile shape
    of the wide path (61 frames at the VoxCPM2 shape: 64 x 64 tiles in four
    groups of k, 128 x 128 in two and in one), against the same latents in
    chunks of 8 frames, which take the float32 kernels."""
    config = CONFIGS["voxcpm2"]
    weights = synth.vae_weights(config, 109)
    if direction == "past":
        weights.tensors["in_pointwise"] = weights.tensors["in_pointwise"] * np.float32(1e6)
        weights.tensors["out_conv"] = weights.tensors["out_conv"] * np.float32(1e-6)
    else:
        scaled_blocks(weights, 2.0**-30)
    frames = 61
    latents = torch.from_numpy(synth.Rng(110, frames).normal(frames * config.latent).astype(
        np.float32).reshape(frames, config.latent)).to(cuda)
    at_once = vx.Vae(weights).decode(latents).cpu().numpy()
    chunked = vx.Vae(weights)
    pieces = [chunked.decode(latents[at:at + 8]).cpu().numpy() for at in range(0, frames, 8)]
    want = np.concatenate(pieces)
    error = float(np.max(np.abs(at_once - want)))
    print(f"{direction} float16's range: max |d| {error:.2e}, signal std {np.std(want):.3f}",
          flush=True)
    assert np.std(want) > 0.1
    assert error <= BOUND
