"""The radix sort's scratch sizes (no GPU): enough for the count's own tiles, and for every smaller count, so that a
buffer sized for a capacity holds any sort up to it."""
import ctypes as C

from luisacomputesimulator_amd import load_library


def test_histogram_words_never_shrink():
    lib = load_library()
    hist, scan = lib._ZN4lcsx15sort_hist_wordsEj, lib._ZN4lcsx14scan_tmp_wordsEj
    for f in (hist, scan):
        f.restype, f.argtypes = C.c_uint32, [C.c_uint32]
    edges = [1, 2, 1023, 1024, 1025, 65535, 65536, 65537, 131072, 294911, 294912, 294913, 500000, 589824, 1 << 20, 1 << 27]
    most = 0
    for n in edges:
        tile = 256 * (4 if n <= 65536 else 8 if n <= 294912 else 16)
        own = 256 * -(-n // tile) + 1
        assert hist(n) >= max(own, most), n
        most = max(most, own)
    assert all(scan(hist(a)) <= scan(hist(b)) for a, b in zip(edges, edges[1:]))
