"""Model preparation's back-face compaction and triangle sort at the edges of their paths, against the oracle:
triangle counts around the wave, the block, its 2 and 4 elements a thread and the global sort, equal depths, and
vertex counts on both sides of the positions kept on chip."""
import numpy as np
import pytest

import sw_model_scenes as S
from test_gpu_models import _compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("subdiv", [3, 5])  # 642 and 10,242 vertices
@pytest.mark.parametrize("triangles", [1, 2, 63, 65, 128, 1023, 1025, 2047, 2050, 4095, 4096, 4097, 9000])
def test_triangle_counts(gpu_ctx, triangles, subdiv):
    print(f"case models triangles={triangles} subdiv={subdiv}", flush=True)
    rng = np.random.default_rng([triangles, subdiv])
    m = S.non_animated_mesh(rng, subdiv=subdiv)
    nv = m.num_vertices
    t = rng.integers(0, nv, size=(triangles, 3)).astype(m.triangles.dtype)
    t[triangles // 2:, 0] = t[0, 0]  # many triangles share a vertex, and with it their depth
    m.triangles = t
    both = S.non_animated_mesh(rng, subdiv=subdiv)
    half = t[: (triangles + 1) // 2]
    both.triangles = np.ascontiguousarray(np.concatenate([half, half[:, [0, 2, 1]]]))  # a front face for every back face
    _compare(gpu_ctx, [m, both], S.instances(rng, [m, both], 6))
