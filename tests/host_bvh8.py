"""A small BVH8 of the device's node format (lumen_amd/csrc/bvh_layout.h) made
on the host by median splits, for tests of the traversal rules through
oracle.bvh8_trace that need no GPU."""
import numpy as np

NODE = np.dtype([("p", "<f4", 3), ("e", "i1", 3), ("imask", "u1"), ("child_base", "<u4"), ("tri_base", "<u4"),
                 ("meta", "u1", 8), ("qlo", "<u2", (3, 8)), ("qhi", "<u2", (3, 8))])
TRI = np.dtype([("v", "<f4", (3, 3)), ("gid", "<u4"), ("prim", "<u4"), ("inst", "<u4")])
assert NODE.itemsize == 128 and TRI.itemsize == 48
MAX_PLANE = 65504.0  # the largest fp16


def _outward(x, up):
    """fp16 bits of x >= 0 rounded up or down."""
    h = np.float16(min(max(x, 0.0), MAX_PLANE))
    if up and float(h) < x and float(h) < MAX_PLANE:
        h = np.nextafter(h, np.float16(np.inf))
    if not up and float(h) > x:
        h = np.nextafter(h, np.float16(0))
    return h.view(np.uint16)


def build(tri):
    """(nodes, tris) of triangles [n, 3, 3]; leaves of one triangle."""
    tri = np.asarray(tri, np.float32)
    cen = tri.mean(1)
    nodes, out = [None], []
    todo = [(0, np.arange(len(tri)))]
    while todo:
        slot, idx = todo.pop()
        groups = [idx]
        while len(groups) < 8 and max(map(len, groups)) > 1:
            g = groups.pop(int(np.argmax([len(x) for x in groups])))
            ax = np.ptp(cen[g], axis=0).argmax()
            g = g[np.argsort(cen[g, ax], kind="stable")]
            groups += [g[:len(g) // 2], g[len(g) // 2:]]
        lo = [tri[g].min((0, 1)).astype(np.float64) for g in groups]
        hi = [tri[g].max((0, 1)).astype(np.float64) for g in groups]
        p, ext = np.min(lo, 0), np.max(hi, 0) - np.min(lo, 0)
        e = np.where(ext > 0, np.ceil(np.log2(np.maximum(ext, 1e-60) / MAX_PLANE)), -100).clip(-100, 127).astype(int)
        e += np.ldexp(MAX_PLANE, e) < ext
        axis = 2 if e[2] > max(e[0], e[1]) else (1 if e[1] > e[0] else 0)
        inner = sorted((k for k, g in enumerate(groups) if len(g) > 1), key=lambda k: lo[k][axis] + hi[k][axis])
        order = inner + [k for k, g in enumerate(groups) if len(g) == 1]
        nd = np.zeros((), NODE)
        nd["p"], nd["e"] = p, e
        nd["qlo"] = np.float16(MAX_PLANE).view(np.uint16)  # empty slots
        nd["child_base"], nd["tri_base"] = (len(nodes) if inner else 0), len(out)
        for c, k in enumerate(order):
            for a in range(3):
                nd["qlo"][a, c] = _outward(np.ldexp(lo[k][a] - p[a], -e[a]), False)
                nd["qhi"][a, c] = _outward(np.ldexp(hi[k][a] - p[a], -e[a]), True)
            if c < len(inner):
                nd["imask"] |= 1 << c
                nd["meta"][c] = c
                todo.append((len(nodes), groups[k]))
                nodes.append(None)
            else:
                nd["meta"][c] = ((len(out) - int(nd["tri_base"])) << 3) | 1
                out.append(groups[k][0])
        nodes[slot] = nd
    t = np.zeros(len(tri), TRI)
    t["v"], t["gid"], t["prim"] = tri[out], out, out
    return np.array(nodes, NODE), t
