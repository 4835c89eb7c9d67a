"""Context.cast_rays in two orders of the rays.  One ray that run_walk does not
take (vrt_device.h: start_walk) sends the 64 of its wave to walk_generic, so rays
drawn at random from a range that holds such rays would hardly reach run_walk."""
import numpy as np


def run_walk_takes(start, d):
    with np.errstate(invalid="ignore"):
        return ((start >= 2.0 ** -20) & (start <= 2.0 ** 22) & (abs(d) >= 2.0 ** -19) & (abs(d) <= 2.0 ** 6)).all(1)


def cast_rays(ctx, start, d, dist, budget, steps=True):
    """The outputs of the rays as given, required to be the same, bit for bit,
    with the rays that run_walk takes first, in waves of their own."""
    start, d = np.asarray(start, np.float32).reshape(-1, 3), np.asarray(d, np.float32).reshape(-1, 3)
    dist = np.asarray(dist, np.int32)
    out = ctx.cast_rays(start, d, dist, budget, steps=steps)
    order = np.argsort(~run_walk_takes(start, d), kind="stable")
    again = ctx.cast_rays(start[order], d[order], dist[order], budget, steps=steps)
    for k, v in out.items():
        a, b = v[order], again[k]
        same = a == b
        if k == "hit_pos":  # any NaN equal to any NaN
            same = ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all(1)
        bad = np.nonzero(~same)[0]
        assert bad.size == 0, "%s differs between two orders for %d rays, first start %s dir %s: %s, %s" % (
            k, bad.size, start[order][bad[0]].tolist(), d[order][bad[0]].tolist(), a[bad[0]], b[bad[0]])
    return out
