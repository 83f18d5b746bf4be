"""Search shapes known at run time, bit for bit against the oracle where
their launches differ: grey clips, one to four wavefronts per workgroup in
the unpaired form, clips of tied distances (the exact selection), and
batches whose clips differ in form or group size in one launch."""
import numpy as np
import pytest

from vbm3d_amd import synth

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _run(V, noisy, sigma, p1, p2, ctx):
    nz, b, f = noisy.copy(), np.zeros_like(noisy), np.zeros_like(noisy)
    V.run_vbm3d(sigma, nz, None, None, b, f, p1, p2, True, 1, ctx=ctx)
    return b, f


# (channels, shape): unpaired RGB at k 7 takes one wavefront per workgroup,
# unpaired grey one to four; the last two are the paired form
CASES = [(3, dict(Npr=7)), (1, dict(Npr=7)), (3, dict(Ns=8, Npr=8, Nb=4, Nf=2)), (1, dict(Ns=8, Npr=8, Nb=4, Nf=2)),
         (1, dict(Npr=3)), (1, dict(Npr=7, Nb=1, k=5))]


@pytest.mark.parametrize("ties", [False, True], ids=["noise", "ties"])
@pytest.mark.parametrize("C,shape", CASES, ids=lambda v: str(v) if isinstance(v, int) else "-".join(f"{k}{x}" for k, x in v.items()))
def test_shapes(oracle, gpu_ctx, C, shape, ties):
    import vbm3d_amd as V
    W, H, F = 41, 35, 4
    if ties:
        noisy = np.random.default_rng(6).integers(0, 3, (F, C, H, W)).astype(np.float32)
    else:
        _, noisy = synth.noisy_clip(W, H, F, C, 20.0, 71)
    p1, p2 = V.initialize_parameters_1(20.0, **shape), V.initialize_parameters_2(20.0, **shape)
    b, f = _run(V, noisy, 20.0, p1, p2, gpu_ctx)
    ob, of, _ = oracle.run_vbm3d(20.0, noisy, p1, p2, True, 1)
    np.testing.assert_array_equal(_bits(b), _bits(ob))
    np.testing.assert_array_equal(_bits(f), _bits(of))


@pytest.mark.parametrize("persistent", [0, 1])
def test_batch_of_paired_and_unpaired(oracle, persistent):
    import torch
    import vbm3d_amd as V
    items, ref = [], []
    for i, shape in enumerate((dict(), dict(Npr=7), dict(Nb=3))):
        _, noisy = synth.noisy_clip(43 + i, 37, 4, 3, 20.0, 72 + i)
        p1, p2 = V.initialize_parameters_1(20.0, **shape), V.initialize_parameters_2(20.0, **shape)
        items.append(V.BatchItem(20.0, torch.from_numpy(noisy).to("cuda:0"), p1, p2))
        ref.append(oracle.run_vbm3d(20.0, noisy, p1, p2, True, 1))
    V.run_batch(items, 1, dict(chunk_frames=0, waves_per_group=0, grab=1, groups_per_cu=8, use_graph=0,
                               persistent=persistent))
    for it, (ob, of, _) in zip(items, ref):
        # run_vbm3d's outputs after the colour round trip, as the batch's
        np.testing.assert_array_equal(_bits(it.basic.cpu().numpy()), _bits(ob))
        np.testing.assert_array_equal(_bits(it.denoised.cpu().numpy()), _bits(of))


@pytest.mark.parametrize("nb", [1, 4])
def test_batch_groups_of_16(oracle, nb):
    """A batch whose largest group is 16, beside clips of groups of 4 and 8."""
    import torch
    import vbm3d_amd as V
    items, ref = [], []
    for i, (C, N) in enumerate(((3, 16), (3, 4), (1, 16), (1, 8))):
        _, noisy = synth.noisy_clip(90 + i, 70, 3, C, 20.0, 75 + i)
        p1, p2 = V.initialize_parameters_1(20.0, N=N), V.initialize_parameters_2(20.0, N=N)
        items.append(V.BatchItem(20.0, torch.from_numpy(noisy).to("cuda:0"), p1, p2))
        ref.append(oracle.run_vbm3d(20.0, noisy, p1, p2, True, nb))
    V.run_batch(items, nb)
    for it, (ob, of, _) in zip(items, ref):
        np.testing.assert_array_equal(_bits(it.basic.cpu().numpy()), _bits(ob))
        np.testing.assert_array_equal(_bits(it.denoised.cpu().numpy()), _bits(of))
