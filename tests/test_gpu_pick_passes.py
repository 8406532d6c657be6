"""The search's passes at every side class they are chosen for, against the FP64 oracle (max-CC 1e-4
normwise, identical argmax where the oracle's top-2 margin exceeds 1e-4 * max|top1|, the search's own
bar), and bit for bit against themselves: results must not depend on the batch (one orientation per
pass runs ungrouped, three in one group or three, a full batch in orientation groups that are merged) nor on how many images share
a launch."""
import numpy as np
import pytest

from tests._util import argmax_agreement, rel_linf, to_np

pytestmark = pytest.mark.gpu

TOL = 1e-4


def _inputs(gx, cuda, n, box, nvol, nd, seed):
    import torch
    from gtom_amd import synth
    rng = np.random.default_rng(seed)
    template = synth.blob_template(box, rng, sigma=(1.0, 2.0), radius=box / 5)
    p = 2 * box
    projft = gx.prepare_projector(torch.from_numpy(template).to(cuda), p)
    data = rng.standard_normal((nvol,) + (n,) * nd).astype(np.float32)
    exp_ft = gx.d_FFTR2C(torch.from_numpy(data).to(cuda), ndims=nd)
    ctf = torch.from_numpy(rng.uniform(-1, 1, (nvol,) + (n,) * (nd - 1) + (n // 2 + 1,)).astype(np.float32)).to(cuda)
    return p, projft, exp_ft, ctf


# k_pick_plane_max: 16 .. 128 (several planes per workgroup up to 48); 8, 12, 192: the passes above and
# below it; chirp-z lines: the edges of the convolution lengths 48 .. 1024, odd and even; 37, 67, 131, 191: chirp-z
# lines whose threads hold whole rows of points past the side
@pytest.mark.parametrize("n", [8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 21, 25, 49, 50, 97, 129, 150, 258, 37, 67, 131,
                               191])
def test_passes_match_oracle_and_each_other(gx, orc, cuda, n):
    import torch
    box = 2 * max(2, min(8, n // 4))
    p, projft, exp_ft, ctf = _inputs(gx, cuda, n, box, 1, 3, n)
    angles = gx.fibonacci_angles(5, 3)[:13]
    norc = 13 if n <= 64 else (4 if n <= 130 else 2)
    res = []
    for batch, ang in ((0, angles[:norc]), (0, angles), (1, angles), (3, angles), (5, angles)):
        plan = gx.PickPlan(p, n, batch)
        best, idx = gx.d_PickSubTomograms(plan, projft, p / n, exp_ft, ctf, ang, n / 8)
        torch.cuda.synchronize()
        res.append((to_np(best), to_np(idx)))
        plan.close()
    for b, i in res[2:]:
        assert np.array_equal(b, res[1][0]) and np.array_equal(i, res[1][1])
    ref = orc.pick(to_np(projft).astype(np.complex128), p, p / n, to_np(exp_ft).astype(np.complex128),
                   to_np(ctf)[0].astype(np.float64), n, angles[:norc].astype(np.float64), n / 8)
    assert rel_linf(res[0][0], ref["best"]) <= TOL
    agree, cnt = argmax_agreement(res[0][1], ref["idx"], ref["top1"], ref["top2"], TOL)
    assert cnt > 0 and agree == 1.0


@pytest.mark.parametrize("n,batch", [(8, 0), (24, 3), (32, 0), (96, 7), (128, 0), (256, 0), (48, 6), (64, 11)])
def test_images_in_one_call_equal_images_alone(gx, cuda, n, batch):
    import torch
    box = 2 * max(2, min(8, n // 4))
    nvol = 6  # more than one launch shares, and not a multiple of it
    p, projft, exp_ft, ctf = _inputs(gx, cuda, n, box, nvol, 2, n)
    angles = gx.fibonacci_angles(9, 3)
    stride = ctf[0].numel()
    for shared in (False, True):
        plan = gx.PickPlan(p, n, batch, ndims=2)
        best, idx = gx.d_PickSubTomograms(plan, projft, p / n, exp_ft, ctf, angles, n / 8,
                                          ctf_volume_stride=0 if shared else stride)
        for v in range(nvol):
            b, i = gx.d_PickSubTomograms(plan, projft, p / n, exp_ft[v:v + 1], ctf[0 if shared else v], angles, n / 8)
            torch.cuda.synchronize()
            assert torch.equal(b[0], best[v]) and torch.equal(i[0], idx[v]), (shared, v)
        plan.close()


def test_plan_holds_what_its_passes_use(gx, cuda):
    """One orientation a pass of 300^3: the batch's spectrum, three spectra and three volumes of the local deviation,
    and tables; no volume (108 MB) that only another form reads."""
    n = 300
    plan = gx.PickPlan(32, n, 1)
    h, v = (n // 2 + 1) * n * n, n ** 3
    assert 0 <= plan.device_bytes - (4 * 8 * h + 3 * 4 * v) <= 4 << 20
    plan.close()
