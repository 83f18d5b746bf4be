"""The aggregation's tiles and the group filter's staged members, bit for
bit against the oracle at the sizes where they can go wrong: frames of one
pixel more and less than the 32 x 16 tiles, tiles that meet several crops
of a tiled reference grid or none, three-channel members whose planes are
not whole cache lines (k = 5, 6, 7) in one lane batch or several, and the
unpadded members of the no-allocation scratch."""
import ctypes as C

import numpy as np
import pytest

from vbm3d_amd import synth

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _check(V, oracle, ctx, W, H, F, ch, k2, N, nb, sigma=20.0):
    _, noisy = synth.noisy_clip(W, H, F, ch, sigma, 41)
    p1, p2 = V.initialize_parameters_1(sigma, N=N), V.initialize_parameters_2(sigma, k=k2, N=N)
    basic, final = V.denoise(noisy, sigma, True, nb, p1, p2, ctx)
    ob, of, _ = oracle.run_vbm3d(sigma, noisy, p1, p2, True, nb)
    np.testing.assert_array_equal(_bits(basic), _bits(ob))
    np.testing.assert_array_equal(_bits(final), _bits(of))


@pytest.mark.parametrize("W,H", [(32, 16), (33, 17), (31, 15), (65, 47)])
@pytest.mark.parametrize("ch", [1, 3])
def test_tile_edges(oracle, gpu_ctx, W, H, ch):
    import vbm3d_amd as V
    _check(V, oracle, gpu_ctx, W, H, 3, ch, 7, 8, 1)


@pytest.mark.parametrize("k2,N", [(4, 8), (5, 8), (6, 16), (7, 1), (7, 16), (8, 16)])
def test_staged_members(oracle, gpu_ctx, k2, N):
    import vbm3d_amd as V
    _check(V, oracle, gpu_ctx, 50, 38, 5, 3, k2, N, 1)


@pytest.mark.parametrize("nb", [2, 16, 32])
def test_crops_of_a_tile(oracle, gpu_ctx, nb):
    import vbm3d_amd as V
    _check(V, oracle, gpu_ctx, 330, 190, 2, 3 if nb == 16 else 1, 7, 8, nb)


def test_unpadded_members(oracle):
    import torch
    import vbm3d_amd as V
    sigma = 20.0
    _, noisy = synth.noisy_clip(45, 37, 5, 3, sigma, 42)
    p1, p2 = V.initialize_parameters_1(sigma), V.initialize_parameters_2(sigma)
    z = torch.from_numpy(noisy).to("cuda:0")
    b, f = torch.empty_like(z), torch.empty_like(z)
    F, ch, H, W = noisy.shape
    fn = V.lib().vbm3d_run_device_noalloc
    fn.argtypes = [C.c_float, C.c_void_p, C.c_void_p, C.c_void_p] + [C.c_uint] * 4 + [
        C.POINTER(V.Parameters), C.POINTER(V.Parameters), C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
    torch.cuda.synchronize()
    assert fn(sigma, z.data_ptr(), None, None, W, H, F, ch, C.byref(p1), C.byref(p2), 1, 1, b.data_ptr(),
              f.data_ptr(), None) == 0
    ob, of, _ = oracle.run_vbm3d(sigma, noisy, p1, p2, True, 1)
    np.testing.assert_array_equal(_bits(b.cpu().numpy()), _bits(ob))
    np.testing.assert_array_equal(_bits(f.cpu().numpy()), _bits(of))


def test_unpadded_rings_under_a_small_budget(oracle, monkeypatch):
    """A ring budget below the smallest padded ring: members unpadded, in the
    per-clip form and in a batch."""
    import torch
    import vbm3d_amd as V
    sigma = 20.0
    _, noisy = synth.noisy_clip(45, 37, 6, 3, sigma, 43)
    p1, p2 = V.initialize_parameters_1(sigma), V.initialize_parameters_2(sigma)
    ob, of, _ = oracle.run_vbm3d(sigma, noisy, p1, p2, True, 1)
    monkeypatch.setenv("VBM3D_EST_BUDGET_MB", "1")
    with V.Context(0) as ctx:
        basic, final = V.denoise(noisy, sigma, True, 1, p1, p2, ctx)
        it = V.BatchItem(sigma, torch.from_numpy(noisy).to("cuda:0"), p1, p2)
        V.run_batch([it], ctx=ctx)
    for b, f in ((basic, final), (it.basic.cpu().numpy(), it.denoised.cpu().numpy())):
        np.testing.assert_array_equal(_bits(b), _bits(ob))
        np.testing.assert_array_equal(_bits(f), _bits(of))


# a reference patch at every pixel (p = 1): a tile meets more members than its
# list holds (512 patches' worth), so the list fills, is summed and filled
# again.  (channels, group size, matches per frame, crops, slices; the crops
# of these frames overlap over most of them)
FULL = [(1, 8, 2, 1, 1), (3, 8, 2, 1, 1), (1, 16, 4, 1, 1), (1, 4, 2, 4, 1), (3, 8, 2, 1, 2), (1, 4, 2, 2, 2)]


@pytest.mark.parametrize("C,N,Nb,nb,kt", FULL)
def test_list_fills(oracle, gpu_ctx, C, N, Nb, nb, kt):
    import vbm3d_amd as V
    sigma, W, H, F = 20.0, 70, 50, 4
    _, noisy = synth.noisy_clip(W, H, F, C, sigma, 44)
    opt = dict(p=1, N=N, Nb=Nb, kt=kt)
    p1, p2 = V.initialize_parameters_1(sigma, **opt), V.initialize_parameters_2(sigma, **opt)
    # the members of step 1 that overlap the tile at (32, 16) in frame 2
    vid = oracle.color(noisy, True) if C == 3 else noisy
    xs, ys, _ = V.grid(W, H, p1.k, 1, 16, 1)
    refs = np.concatenate([t * W * H * C + ys.astype(np.int64) * W + xs for t in range(F - kt + 1)]).astype(np.uint32)
    idx, _, _, nsx = V.block_match(vid, p1, refs, ctx=gpu_ctx)
    m = idx[np.arange(idx.shape[1])[None, :] < nsx[:, None]].astype(np.int64)
    t, r = m // (W * H * C), m % (W * H * C)
    y, x = r // W, r % W
    hit = (t <= 2) & (t > 2 - kt) & (x > 32 - p1.k) & (x < 64) & (y > 16 - p1.k) & (y < 32)
    assert hit.sum() > 512 * N
    basic, final = V.denoise(noisy, sigma, True, nb, p1, p2, gpu_ctx)
    ob, of, _ = oracle.run_vbm3d(sigma, noisy, p1, p2, True, nb)
    np.testing.assert_array_equal(_bits(basic), _bits(ob))
    np.testing.assert_array_equal(_bits(final), _bits(of))


def test_list_fills_in_a_batch_and_the_adjoint(oracle, gpu_ctx, monkeypatch):
    """The batched kernel's and the raw sums' list: against the per-clip run,
    and rings holding the clip against one-frame chunks."""
    import torch
    import vbm3d_amd as V
    sigma = 20.0
    _, noisy = synth.noisy_clip(70, 50, 4, 1, sigma, 45)
    p1, p2 = V.initialize_parameters_1(sigma, p=1), V.initialize_parameters_2(sigma, p=1)
    basic, final = V.denoise(noisy, sigma, True, 1, p1, p2, gpu_ctx)
    it = V.BatchItem(sigma, torch.from_numpy(noisy).to("cuda:0"), p1, p2)
    V.run_batch([it], ctx=gpu_ctx)
    np.testing.assert_array_equal(_bits(it.basic.cpu().numpy()), _bits(basic))
    np.testing.assert_array_equal(_bits(it.denoised.cpu().numpy()), _bits(final))
    z, b = torch.from_numpy(noisy).to("cuda:0"), torch.from_numpy(basic).to("cuda:0")
    g = torch.from_numpy(np.random.default_rng(7).standard_normal(noisy.shape).astype(np.float32)).to("cuda:0")
    whole = V.step2_adjoint(sigma, z, b, g, p2, ctx=gpu_ctx)
    with V.Context(0) as ctx:
        ctx.set_chunk_frames(1)
        assert torch.equal(whole, V.step2_adjoint(sigma, z, b, g, p2, ctx=ctx))
    # J^T g against the 64-bit model of the transposed step
    ref, _ = oracle.step2_adjoint_fp64(sigma, noisy, basic, oracle.params_2(sigma, p=1), g.double().cpu().numpy(), True, 1)
    err = np.abs(whole.double().cpu().numpy() - ref).max()
    assert err <= 1e-4 * np.abs(ref).max(), err
