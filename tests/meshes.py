"""Closed triangle meshes for the mesh -> SDF tests (outward-facing triangles) and
their exact signed distances."""
import numpy as np

from atac.workloads import box_mesh as box, icosphere, torus  # noqa: F401


def box_exact_sdf(p, a=1.0):
    """Signed distance to the cube [-a, a]^3 (negative inside)."""
    q = np.abs(p) - a
    out = np.linalg.norm(np.maximum(q, 0.0), axis=-1)
    inn = np.minimum(np.max(q, axis=-1), 0.0)
    return out + inn


def torus_exact_sdf(p, R=1.0, r=0.35):
    xy = np.linalg.norm(p[..., :2], axis=-1)
    return np.sqrt((xy - R) ** 2 + p[..., 2] ** 2) - r


def split_box(half, n):
    """The box [-half, half] (per axis) with n x n quads a face, two triangles each, vertices shared."""
    half = np.broadcast_to(np.asarray(half, dtype=np.float64), 3)
    step = np.arange(n + 1)
    index, V, F = {}, [], []

    def vertex(i):
        if i not in index:
            index[i] = len(V)
            V.append(-half + 2.0 * half * np.array(i) / n)
        return index[i]

    for ax in range(3):
        u, v = (ax + 1) % 3, (ax + 2) % 3
        for side in (0, n):
            for a in step[:-1]:
                for b in step[:-1]:
                    q = []
                    for da, db in ((0, 0), (1, 0), (1, 1), (0, 1)):
                        i = [0, 0, 0]
                        i[ax], i[u], i[v] = side, int(a + da), int(b + db)
                        q.append(vertex(tuple(i)))
                    if side == 0:
                        q.reverse()
                    F += [(q[0], q[1], q[2]), (q[0], q[2], q[3])]
    return np.array(V), np.array(F, dtype=np.int64)
