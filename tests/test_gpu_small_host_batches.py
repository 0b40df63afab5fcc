"""Small host batches, whose faces and embeddings stay in the pinned host
buffer that the kernels address in place: the largest of them and the first
past them, alternating, against the single-face path."""
import numpy as np
import pytest

import fastface_amd as fa
from fastface_amd import synth

pytestmark = pytest.mark.gpu


def test_in_place_host_batches(gpu_lib, synth_ffw4):
    u8 = np.random.default_rng(7).integers(0, 256, (7, 112, 112, 3), dtype=np.uint8)
    sdk = (u8.astype(np.float32) - np.float32(127.5)) / np.float32(127.5)
    f32 = synth.faces_uniform(2, 31)
    with fa.FastFace(synth_ffw4, cwd=fa.REPO_ROOT) as f:
        one = np.stack([f.embed(x) for x in sdk])
        exp2 = np.stack([f.embed(x) for x in f32])
        for n in (6, 7, 1, 7, 6):
            assert np.array_equal(f.embed_batch_rgb8(u8[:n]), one[:n]), n
        for n in (2, 1, 2, 1):
            assert np.array_equal(f.embed_batch(f32[:n]), exp2[:n]), n
        assert not np.array_equal(one[0], one[1])
