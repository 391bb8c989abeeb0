"""Products of few outputs for the tests: at least one for each form of gemm_tn_slices, at the edges of its tiles and of K."""
from tests import abi_ctypes as ac

# (M, N, K, input type): rows and columns at and around whole tiles of 16, 32 and 64; fewer k-steps than waves; a ragged last k-step
PLAIN = [(m, n, k, dt)
         for dt in (ac.BF16, ac.F16, ac.E4M3)
         for m, n, k in [(1, 128, 4096), (15, 132, 4112), (16, 1284, 2560), (17, 68, 4096), (1, 4, 16), (33, 20, 48), (3, 452, 176),
                         (64, 1024, 1024), (65, 1028, 1040), (32, 4100, 256), (8, 2052, 3200), (236, 640, 1536), (237, 644, 1552),
                         (512, 512, 512), (513, 516, 528), (1024, 1024, 1024), (467, 1920, 1024), (1618, 256, 2240), (5, 3204, 64), (1100, 512, 512), (1090, 516, 400)]]
MX = [(1, 128, 8192), (15, 132, 4096), (16, 1280, 5760), (17, 68, 4096), (33, 20, 128), (3, 452, 384), (65, 1028, 1024), (32, 4100, 256),
      (237, 644, 1536), (368, 224, 2816), (513, 516, 512), (1025, 1028, 1024), (993, 240, 4096), (129, 4, 256), (1, 18944, 384)]

# Rows of any alignment (M, N, K, input type, elements before the first row of A and of B, elements between rows)
ANY_ROWS = [(m, n, k, dt, off, gap)
            for dt in (ac.BF16, ac.F16)
            for m, n, k, off, gap in [(1, 129, 8191, 0, 0), (15, 131, 130, 1, 0), (33, 21, 9, 0, 1), (64, 1001, 1023, 0, 0), (65, 40, 71, 3, 2),
                                      (236, 641, 1537, 0, 3), (515, 2050, 4100, 0, 0), (512, 511, 513, 1, 1), (3, 452, 12, 0, 0), (16, 300, 64, 1, 0),
                                      (10, 4099, 2050, 0, 0), (1100, 515, 130, 0, 0), (17, 68, 4103, 5, 0)]]
ANY_ROWS += [(m, n, k, ac.E4M3, off, gap) for m, n, k, off, gap in
             [(234, 1568, 1326, 0, 0), (300, 2048, 1025, 1, 0), (100, 5001, 2047, 0, 3), (16, 4100, 2050, 0, 0), (65, 1027, 4097, 7, 9)]]
