"""Products of few outputs for the tests: at least one for each form of gemm_tn_slices, at the edges of its tiles and of K."""
from tests import abi_ctypes as ac

# (M, N, K, input type): rows and columns at and around whole tiles of 16, 32 and 64; fewer k-steps than waves; a ragged last k-step
PLAIN = [(m, n, k, dt)
         for dt in (ac.BF16, ac.F16, ac.E4M3)
         for m, n, k in [(1, 128, 8192), (15, 132, 8208), (16, 1280, 5760), (17, 68, 4096), (1, 4, 16), (33, 20, 48), (3, 452, 176),
                         (64, 1024, 1024), (65, 1028, 1040), (32, 4100, 256), (8, 2052, 3200), (236, 640, 1536), (237, 644, 1552),
                         (512, 512, 512), (513, 516, 528), (1024, 1024, 1024), (467, 1920, 1024), (1618, 256, 2240), (5, 12804, 64), (1100, 512, 512), (1090, 516, 400)]]
MX = [(1, 128, 8192), (15, 132, 4096), (16, 1280, 5760), (17, 68, 4096), (33, 20, 128), (3, 452, 384), (65, 1028, 1024), (32, 4100, 256),
      (237, 644, 1536), (368, 224, 2816), (513, 516, 512), (1025, 1028, 1024), (993, 240, 4096), (129, 4, 256), (1, 18944, 384)]
