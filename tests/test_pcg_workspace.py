"""Size of the PCG workspace (host only): a workspace made for one system holds every smaller one's state."""
import ctypes


def test_workspace_size_never_falls():
    """Every row count around the ends of the 64- and 256-row groups up to 2^20 rows, and around the size rules
    of the block count and of the wide product."""
    from ngspsr import _lib
    size = _lib.lib().ngs_pcg_workspace_bytes
    rows = sorted({m + d for step in (64, 256) for m in range(0, 1 << 20, 16 * step) for d in (1, 2, step, step + 1)}
                  | {e + d for e in (2048, 65536, 655360, 2790144) for d in range(-260, 261)})
    sizes = [size(m) for m in rows]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
    # the three vectors, the state, three partials per block and the table entry
    assert all(s >= 12 * m + 256 + 24 * min((m + 255) // 256, 2560) + 512 for m, s in zip(rows, sizes))


def test_noalloc_limit_fits_its_array():
    """The row limit of the solve without allocation keeps its value, and its layout fits the 32 MiB array."""
    from ngspsr import _lib
    assert _lib.lib().ngs_pcg_workspace_bytes(2790144) <= 32 << 20
    fake, it, rr = ctypes.c_void_p(256), ctypes.c_int32(), ctypes.c_double()
    assert _lib.lib().ngs_pcg_solve_runs_noalloc(fake, fake, fake, fake, fake, 2790145, 1e-6, 10, 32, None,
                                                 ctypes.byref(it), ctypes.byref(rr)) == 6
