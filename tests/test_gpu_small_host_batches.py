"""Small host batches, whose faces and embeddings stay in the pinned host
buffer that the kernels address in place: the largest of them and the first
past them, alternating, against the device entry points and the oracle."""
import numpy as np
import pytest

import fastface_amd as fa
import gpu_util
from fastface_amd import synth

pytestmark = pytest.mark.gpu


def _device(lib, f, call, faces):
    """Embeddings of device-resident faces, one face a call (no pinned buffer)."""
    out = gpu_util.Dev(lib, nbytes=512 * 4)
    rows = []
    for x in faces:
        d = gpu_util.Dev(lib, host=x)
        assert call(f.ff, d.ptr, 1, out.ptr, None) == 0
        gpu_util.check(lib, lib.ffk_stream_sync(lib.fastface_stream(f.ff)))
        rows.append(out.get(np.float32, (512,)))
    return np.stack(rows)


def test_in_place_host_batches(gpu_lib, synth_ffw4, oracle, oracle_model):
    u8 = np.random.default_rng(7).integers(0, 256, (7, 112, 112, 3), dtype=np.uint8)
    sdk = (u8.astype(np.float32) - np.float32(127.5)) / np.float32(127.5)
    f32 = synth.faces_uniform(9, 31)
    with fa.FastFace(synth_ffw4, cwd=fa.REPO_ROOT) as f:
        one = _device(gpu_lib, f, gpu_lib.fastface_embed_batch_rgb8_device, u8)
        exp = _device(gpu_lib, f, gpu_lib.fastface_embed_batch_device, f32)
        for faces, rows in ((sdk, one), (f32, exp)):
            emb, _ = oracle.forward(oracle_model, faces[:1])
            assert np.array_equal(rows[0], emb[0])
        for n in (6, 7, 1, 7, 6):
            assert np.array_equal(f.embed_batch_rgb8(u8[:n]), one[:n]), n
        for n in (2, 1, 8, 1, 9, 2, 1):
            assert np.array_equal(f.embed_batch(f32[:n]), exp[:n]), n
        assert np.array_equal(f.embed(sdk[3]), one[3])
        assert not np.array_equal(one[0], one[1])
