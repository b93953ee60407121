"""The partition of the joined colour passes (k_gs_rect) restated in Python:
how a level's planes are cut into workgroups, which nodes of each colour a
workgroup updates, the region it stages and the nodes it writes.  Used by the
CPU tests of that partition; the kernel's results are tested on the GPU
against the restatement's 8-colour sweep."""

SHAPES = {"narrow": (21, 2, 10), "wide": (64, 4, 23)}   # nodes of a colour, lines, region's half length


def part(shape, nz, nx, ny):
    """a level's partition for one workgroup shape (None: not for it)"""
    nodes, W, HZ = SHAPES[shape]
    most = nodes // (W // 2 + 1)
    for ns in range(1, (nz + 1) // 2 + 1):
        wz = max(2, ((nz - 1 + ns - 1) // ns + 1) // 2 * 2)
        if max(1, -(-(nz - 1) // wz)) != ns:
            continue
        nk = (nz + 1) // 2 if ns == 1 else min((nz + 1) // 2, wz // 2 + 3)
        if nk > most or min(wz + 7, nz + 2) + 1 > 2 * HZ:
            continue
        return {"nodes": nodes, "W": W, "HZ": HZ, "Wz": wz, "ns": ns, "nstrip": max(1, -(-(nx - 1) // W))}
    return None


def launches(p, ny):
    """(jpar, number of workgroups) of a sweep's two launches"""
    return [(jpar, (ny - jpar + 1) // 2 * p["nstrip"] * p["ns"]) for jpar in range(2)]


def workgroup(p, nz, nx, ny, jpar, b):
    """one workgroup: (j, colours [(k parity, i parity, nodes)], staged region, owned k and i)"""
    seg, b = b % p["ns"], b // p["ns"]
    strip, j = b % p["nstrip"], 2 * (b // p["nstrip"]) + jpar
    i0, k0 = strip * p["W"], seg * p["Wz"]
    k1 = k0 + p["Wz"]
    colours = []
    for ph in range(4):
        kp, ip, grow = ph & 1, ph >> 1, 2 - ph
        klo, khi = max(kp, k0 - grow), min(nz - 1, k1 + grow)
        ilo, ihi = i0 + ip, min(nx - 1, i0 + p["W"] - ip)
        nk = ((khi - klo) >> 1) + 1 if khi >= klo else 0
        ni = ((ihi - ilo) >> 1) + 1 if ihi >= ilo else 0
        colours.append((kp, ip, [(klo + 2 * (t % nk), ilo + 2 * (t // nk)) for t in range(nk * ni)]))
    kr0 = max(k0 - 4, -2)
    region = (kr0, kr0 + 2 * p["HZ"] - 1, i0 - 1, i0 + p["W"] + 1)
    ke = nz if seg == p["ns"] - 1 else k1
    ie = nx if strip == p["nstrip"] - 1 else i0 + p["W"]
    return j, colours, region, list(range(k0, ke)), list(range(i0, ie))
