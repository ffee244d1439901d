"""The autotuner's cache file on the host: a plan's flags are kept, files without
them are read as before."""
import ctypes as C


def test_flags_kept(bws, tmp_path):
    L = bws.lib()
    L.bws_autotune_clear()
    f, g = tmp_path / "in.txt", tmp_path / "out.txt"
    f.write_text("0 12 12 12 -4 1 256 16 64 0 1\n0 11 11 11 -3 1 128 16 64 0\n1 10 10 10 -3 2 0 0 0\n")
    assert L.bws_autotune_load(str(f).encode()) == bws.BWS_OK
    assert L.bws_autotune_save(str(g).encode()) == bws.BWS_OK
    L.bws_autotune_clear()
    assert L.bws_autotune_load(str(g).encode()) == bws.BWS_OK
    p = bws._Plan()
    for size, nnz, prec, want in ((4096, 838861, 0, (1, 256, 1)), (2048, 524288, 0, (1, 128, 0)),
                                  (1000, 100000, 1, (2, 0, 0))):
        assert L.bws_autotune_lookup(size, size, size, nnz, prec, C.byref(p)) == bws.BWS_OK
        assert (p.kernel, p.rows_per_wg, p.flags) == want
    L.bws_autotune_clear()
