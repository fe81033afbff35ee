"""Plain, batched, graph and overlapped steps of one scene. Up to 32768
view-surfels the gradient slots are doubles, whose sums rounded to f32 do not
depend on the order in which the tiles add, and a pass over one view rounds
like a pass over all: the forms give the same bits, step after step. (With f32
slots a last bit parts them, and some steps later a pixel's decision.)"""

import numpy as np
import pytest

from conftest import announce
from test_gpu_train import _params, _render_targets, _small_training_problem

pytestmark = pytest.mark.gpu


# Ten steps, as far as a last bit needs to grow into another decision. 10922
# surfels in three views: the largest with double slots. 1283 x 20: more tiles
# than lists that are long.
@pytest.mark.parametrize("n,size,seed", [(3000, (96, 64), 3), (3000, (96, 64), 4), (3000, (96, 64), 5),
                                         (10_922, (150, 90), 3), (500, (1283, 20), 6)])
def test_step_forms_give_the_same_bits(gpu, n, size, seed):
    import splattar_amd as sa
    deg = 2
    sc, tgt, specs = _small_training_problem(n=n, size=size, deg=deg, seed=seed)
    targets = _render_targets(gpu, tgt, specs, deg)
    cfg = sa.TrainConfig(lam=0.2, dssim_scale=0.5, lr_pos=4e-3, lr_scales=1e-3, lr_quat=1e-3, lr_opacity=1e-3,
                         lr_sh=1e-3, max_views_per_step=3)
    views = [(sa.Camera(sp.center, sp.quat, sp.focal, deg), t) for sp, t in zip(specs, targets)]
    forms = {"plain": (sa.Trainer.PLAIN, (8, 8), False), "plain, whole lists": (sa.Trainer.PLAIN, (8, 0), False),
             "batched": (sa.Trainer.BATCHED, (8, 8), False), "graph": (sa.Trainer.GRAPH, (8, 8), False),
             "graph, 4-bit digits, whole lists": (sa.Trainer.GRAPH, (4, 0), False),
             "overlapped": (sa.Trainer.BATCHED, (8, 4), True)}
    ref = None
    for name, (mode, schedule, overlap) in forms.items():
        t = sa.Trainer(gpu, cfg, sc.as_init(), views)
        t.set_schedule(*schedule)
        t.set_overlap(overlap)
        announce(f"step forms n={n} {size} seed={seed}: {name}")
        for _ in range(10):
            t.step([0, 1, 2], mode=mode)
        got = _params(t)
        t.close()
        if ref is None:
            ref = {k: np.array(v) for k, v in got.items()}
        for k in ref:
            np.testing.assert_array_equal(np.asarray(got[k]), ref[k], err_msg=f"{name}: {k}")
