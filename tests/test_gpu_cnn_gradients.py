"""Gradients of the learned cut proposal at the edges of their kernels' tiles (bricks of 16 x 4 x 4
voxels, rows of 16 in pairs) and with more bricks than workgroups, and the forward layers' split along
z, against the numpy oracle with the same bfloat16 rounding points and float64 sums. The GPU sums in
float32, so a stored bfloat16 may differ by one unit in the last place (2^-8 of its value); a whole
tensor then differs by less than that, relative to its norm."""
import numpy as np
import pytest

import cugip_amd
from oracle import cnn as ocnn
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

BOUNDS = np.cumsum([0, ocnn.N_W1, 16] + [ocnn.N_W, 16] * 3 + [16, 1])


@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (16, 4, 4), (17, 5, 5), (15, 3, 9), (33, 4, 2), (130, 33, 33)])
def test_gradients_at_tile_edges(nx, ny, nz):
    say(f"cnn gradients {nx}x{ny}x{nz}")
    vol, cs, ct, cn = cugip_amd.make_instance(nx, ny, nz, nx + ny)
    p = cugip_amd.Cnn.init_params(nx)
    with cugip_amd.GridGraph() as g, cugip_amd.Cnn() as net:
        g.set_grid(cs, ct, cn)
        g.max_flow()
        label = g.source_set()
        net.set_params(p)
        loss, grad = net.gradients(g, vol)
        again = net.gradients(g, vol)  # (buffers reused; every sum has a fixed order)
    ref_loss, ref = ocnn.loss_and_grad(p, vol, cs, ct, label.reshape(nz, ny, nx), bf=True)
    assert abs(loss - ref_loss) <= 2.0 ** -8 * abs(ref_loss)
    for lo, hi in zip(BOUNDS[:-1], BOUNDS[1:]):
        a, b = grad[lo:hi].astype(np.float64), ref[lo:hi]
        assert np.linalg.norm(a - b) <= 2.0 ** -8 * np.linalg.norm(b), (lo, hi)
    assert again[0] == loss and np.array_equal(again[1], grad)


@pytest.mark.parametrize("nx,ny,nz", [(32, 8, 70), (250, 120, 20), (170, 300, 66)])
def test_forward_split_along_z(nx, ny, nz):
    """1, 4 and (for (170, 300, 66), wide in x and y) 4 bricks a workgroup: a crop whose receptive field
    lies inside the volume predicts what the whole does, bit for bit."""
    say(f"cnn forward {nx}x{ny}x{nz}")
    vol, cs, ct, cn = cugip_amd.make_instance(nx, ny, nz, 3)
    p = cugip_amd.Cnn.init_params(5)
    z0 = nz // 2 - 9
    crop = (slice(z0, z0 + 18), slice(0, min(ny, 24)), slice(0, min(nx, 40)))
    with cugip_amd.GridGraph() as g, cugip_amd.Cnn() as net:
        net.set_params(p)
        g.set_grid(cs, ct, cn)
        whole = net.predict(g, vol)[1].reshape(vol.shape)
        c = [np.ascontiguousarray(a[crop]) for a in (cs, ct)]
        g.set_grid(c[0], c[1], np.zeros((3,) + c[0].shape, np.int32))
        part = net.predict(g, np.ascontiguousarray(vol[crop]))[1].reshape(c[0].shape)
    # the receptive field is 4 voxels; the crop's low y and x faces are the volume's own
    hy, hx = part.shape[1] - (4 if ny > 24 else 0), part.shape[2] - (4 if nx > 40 else 0)
    assert np.array_equal(part[4:-4, :hy, :hx], whole[crop][4:-4, :hy, :hx])
