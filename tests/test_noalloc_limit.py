"""The sizes that tpsph_kick_noalloc takes: the bytes it counts against its 64 MiB, at the smallest
size that it refuses in a box of many cells (refused before the device is touched)."""
import ctypes as C
import math

LIMIT = 64 << 20


def scratch_bytes(nf, nw, cells, nd):
    def region(n):
        return (max(n, 1) + 255) // 256 * 256
    sizes = [4, 4 * ((cells + 1 + 2047) // 2048 + 1)]
    sizes += 4 * [4 * nf] + 2 * [4 * (cells + 1)] + 3 * [8 * (nf + 4)] + [8 * nd * nf, 64 * nf, 16 * nf]
    sizes += 2 * [4 * nw] + 2 * [4 * (cells + 1)] + [4 * nw] + 3 * [8 * (nw + 4)]
    sizes += [32 * nw, 16 * nw, 8 * nw, 8 * nw, cells]
    return sum(region(s) for s in sizes)


def test_smallest_refused_size(tp):
    lib = tp.native.load()
    p = tp.native.TpsphParams()
    p.ndims = 3
    p.memory = tp.native.TPSPH_MEM_DEVICE
    p.smoothing_length = 0.012
    p.reference_density = 1000.0
    p.sound_speed = 48.5
    p.exponent = 7.0
    p.skin = 0.0
    R = 2 * p.smoothing_length
    cells = 1
    for d in range(3):
        p.domain_min[d], p.domain_max[d] = 0.0, 1.0
        cs = (R * 1.00001 + 2e-9 * R) * (1.0 + 1e-9) / (4 if d == 0 else 2)
        cells *= math.ceil((1.0 + 2.0 * cs) / cs) + 1
    nf = LIMIT // 100
    while scratch_bytes(nf, 1000, cells, 3) > LIMIT:
        nf -= 1
    nf += 1
    size = scratch_bytes(nf, 1000, cells, 3)
    assert LIMIT < size < LIMIT + 4096
    dummy = C.c_void_p(8)  # never dereferenced: the size check comes first
    rc = lib.tpsph_kick_noalloc(C.byref(p), nf, 1000, dummy, dummy, dummy, dummy, dummy, dummy, 0.0, None)
    msg = lib.tpsph_last_error(None).decode()
    assert rc == tp.native.TPSPH_ERR_ARGUMENT, (rc, msg)
    assert f"needs {size} bytes" in msg and f"{cells} cells" in msg, (size, cells, msg)
