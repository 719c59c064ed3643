"""The staged march over the kinds of boxes its launches choose between: the
fixed box, chunks that are split, boxes of any extents (with a grown LDS
budget) and the gather where no box fits, against the FP64 oracle and, bit for
bit, against the march without staging."""
import numpy as np
import pytest

import ct_forward_projection_amd as P
from ct_forward_projection_amd import synthetic as S
from oracle import oracle as O

from test_gpu_parity import MIXED_TOL, TOL, rel_err, to_np

pytestmark = pytest.mark.gpu

# pixel pitch (mm) of a 1-mm phantom: pixels 0.4, 0.7, 0.85, 1.4 and 3.3
# voxels apart at its centre (magnification 1.5)
PITCHES = (0.6, 1.05, 1.3, 2.1, 5.0)


@pytest.mark.parametrize("pitch", PITCHES)
@pytest.mark.parametrize("n_mat,dtype", [(1, P.CTFP_F32), (3, P.CTFP_F32), (4, P.CTFP_F16), (2, P.CTFP_BF16)])
def test_boxes_of_every_kind(require_gpu, pitch, n_mat, dtype):
    import torch
    n = 44
    s = S.config2()
    s.n_vox, s.length_mm, s.views = (n, n - 3, n + 5), (n * 1.0, (n - 3) * 1.1, (n + 5) * 0.9), 5
    s.det, s.d_size = (37, 35), pitch
    s.materials = (S.WATER, S.BONE, S.IODINE, S.ALUMINIUM)[:n_mat]
    rng = np.random.default_rng(int(pitch * 100) + n_mat)
    shape = (n + 5, n - 3, n)
    vols = []
    for m in range(n_mat):
        v = np.zeros(shape, np.float32)
        v[4:-5, 3:-4, 6:-2] = rng.uniform(0.0, 0.6, (n - 4, n - 10, n - 8))
        v[:, :, n // 2] = 0.0  # and an empty plane between two halves
        vols.append(v)
    kw = P.spectral_inputs(s, *s.det)
    with P.Projector(P.scan_params(**s.scan_kwargs())) as proj:
        proj.set_volumes(vols, storage_dtype=dtype)
        proj.set_spectral(**kw)
        proj.set_tuning(march="global")
        ref = proj.forward(want_L=True)
        for chunk, lds, wave_u, block_u in ((16, 40960, 8, 2), (48, 40960, 8, 2), (32, 16384, 4, 4), (16, 2048, 16, 1),
                                            (16, 65536, 32, 2)):
            proj.set_tuning(march="lds", chunk=chunk, lds_bytes=lds, wave_u=wave_u, block_u=block_u)
            got = proj.forward(want_L=True)
            for a, b in zip(got, ref):
                assert torch.equal(a, b), (chunk, lds, wave_u, block_u)
        L = to_np(ref[2])
    g = O.geom_from_setup(s)
    L64 = O.march_f64(g, O.paras(g), vols, 0, s.views)
    assert float(np.abs(L64).max()) > 0.0
    # FP32: the suite's parity bound; 16 bit: its bound for line integrals of
    # the storage (one rounding of densities and of weights)
    tol = {P.CTFP_F32: TOL, P.CTFP_F16: MIXED_TOL["f16"], P.CTFP_BF16: 1e-2}[dtype]
    assert rel_err(L, L64) < tol


@pytest.mark.parametrize("pitch", (0.6, 1.3, 5.0))
def test_batch_of_several_kinds(require_gpu, pitch):
    """Scans that take different march kernels in one batch equal their own
    launches bit for bit."""
    import torch
    items, refs, projs = [], [], []
    for k, (p, m) in enumerate(((0.6, 3), (pitch, 1), (2.1, 2))):
        s = S.config2()
        n = 40
        s.n_vox, s.length_mm, s.views, s.det, s.d_size = (n, n, n), (n * 1.0,) * 3, 9, (40, 33), p
        s.materials = s.materials[:m]
        proj = P.Projector(P.scan_params(**s.scan_kwargs()))
        proj.set_volumes(list(S.three_material_phantom(n, seed=5 + k))[:m], storage_dtype=P.CTFP_F16)
        proj.set_spectral(**P.spectral_inputs(s, *s.det))
        refs.append(proj.forward())
        I = torch.zeros((s.views, s.det[1], s.det[0]), device="cuda")
        items.append((proj, 0, s.views, I, torch.zeros_like(I)))
        projs.append(proj)
    with P.Batch(items) as b:
        for _ in range(3):
            b.run()
            torch.cuda.synchronize()
            for it, ref in zip(items, refs):
                assert torch.equal(it[3], ref[0]) and torch.equal(it[4], ref[1])
                it[3].zero_(), it[4].zero_()
    for p in projs:
        p.close()
