"""The loss of several views in one launch against each view in a launch of its
own. The band height follows from the whole launch, so these have other bands:
dL/dimage does not depend on them (the steps' parameters are equal bits, the
gradient sums having no order at this size), and the f64 sums differ only by
their grouping."""

import numpy as np
import pytest

from conftest import announce
from test_gpu_train import _params, _render_targets

pytestmark = pytest.mark.gpu

# One view of 640 x 480 has nine strips of 74 columns and bands of a few rows;
# with two more it shares the CUs with 27 strips and gets longer ones. Heights
# that leave part of a band.
SIZES = [(640, 480), (635, 473), (601, 359)]


def test_one_launch_equals_a_launch_per_view(gpu):
    import splattar_amd as sa
    from splattar_amd import scenes
    deg = 1
    sc = scenes.make_scene(3000, deg, -3.4, 0.4, 23)
    specs = scenes.sphere_views(3, 29, SIZES)
    targets = _render_targets(gpu, scenes.jittered(sc, 0.01, 24), specs, deg)
    cfg = sa.TrainConfig(lam=0.2, dssim_scale=0.5, lr_pos=1e-3, lr_scales=1e-3, lr_quat=1e-3, lr_opacity=1e-3,
                         lr_sh=1e-3, max_views_per_step=3)
    views = [(sa.Camera(sp.center, sp.quat, sp.focal, deg), t) for sp, t in zip(specs, targets)]
    params, losses = {}, {}
    for mode in (sa.Trainer.PLAIN, sa.Trainer.BATCHED, sa.Trainer.GRAPH):
        announce(f"loss launches: mode {mode}")
        t = sa.Trainer(gpu, cfg, sc.as_init(), views)
        t.step([0, 1, 2], mode=mode)
        params[mode], losses[mode] = _params(t), t.last_losses(3)
        t.close()
    ref = sa.Trainer.PLAIN
    for mode in (sa.Trainer.BATCHED, sa.Trainer.GRAPH):
        for k in params[ref]:
            np.testing.assert_array_equal(params[mode][k], params[ref][k], err_msg=f"mode {mode}: {k}")
        # Both group at most 640 * 480 * 3 f32 terms in chains of fewer than
        # 4096 f64 additions: 4096 * 2^-53 = 4.5e-13 of the sum.
        np.testing.assert_allclose(losses[mode], losses[ref], rtol=0, atol=1e-12)
    assert losses[ref].min() > 1e-4
