"""Meshes between the sizes that the library's own refinement reaches."""
import numpy as np


def sphere(frequency, radius):
    """A geodesic sphere: every edge of an icosahedron in `frequency` parts, 10 frequency^2 + 2 vertices."""
    p = (1 + 5 ** 0.5) / 2
    corner = np.array([(-1, p, 0), (1, p, 0), (-1, -p, 0), (1, -p, 0), (0, -1, p), (0, 1, p), (0, -1, -p), (0, 1, -p),
                       (p, 0, -1), (p, 0, 1), (-p, 0, -1), (-p, 0, 1)])
    faces = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2), (10, 7, 6),
             (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10),
             (8, 6, 7), (9, 8, 1)]
    index, verts, tris = {}, [], []

    def at(f, i, j):
        w = sorted((c, n) for c, n in zip(f, (frequency - i - j, i, j)) if n)
        if tuple(w) not in index:
            index[tuple(w)] = len(verts)
            verts.append(sum(n * corner[c] for c, n in w))
        return index[tuple(w)]
    for f in faces:
        for i in range(frequency):
            for j in range(frequency - i):
                tris.append((at(f, i, j), at(f, i + 1, j), at(f, i, j + 1)))
                if i + j < frequency - 1:
                    tris.append((at(f, i + 1, j), at(f, i + 1, j + 1), at(f, i, j + 1)))
    v = np.array(verts)
    return radius * v / np.linalg.norm(v, axis=1)[:, None], np.array(tris, dtype=np.int32)
