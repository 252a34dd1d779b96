"""Sizes at the edges of the GEMM kernels' tiles, with the kernel that the planner has to send each of
them to and how it sums K: "whole" (one block), "sum" (split, added up by a tile's last block) or
"reduce" (split, added up by a second launch).  tests/test_plan.py holds the planner to them on the
CPU, tests/test_ops_gpu.py runs them."""

PATCH = "conv3_patch_kernel"
DENSE = "gemm_dense_kernel"

# 3x3 convs of stride 1: B, H, W, Ci, Co, time projection, residual, kernel, K sum
CONV = [
    (1, 8, 8, 64, 8, False, False, "conv3_narrow_kernel<8,8>", "whole"),
    # one 8x8 sub-tile x 32 columns, all nine taps' weights in the ring
    (3, 8, 8, 128, 72, True, True, PATCH + "<8,1,32,2,1,9,9>", "whole"),
    (1, 9, 17, 64, 168, False, True, PATCH + "<8,1,32,2,1,9,9>", "whole"),      # a pixel past a sub-tile both ways
    (2, 7, 15, 192, 88, True, False, PATCH + "<8,1,32,2,1,9,9>", "whole"),      # a pixel short
    (1, 48, 47, 128, 128, False, True, PATCH + "<8,1,32,2,1,9,9>", "whole"),
    (1, 33, 39, 64, 72, False, True, PATCH + "<8,1,32,2,1,9,9>", "whole"),      # one chunk
    (1, 128, 120, 64, 64, True, True, PATCH + "<8,1,32,2,1,9,9>", "whole"),
    (1, 16, 16, 704, 320, True, False, PATCH + "<8,1,32,2,1,9,9>", "sum"),      # 11 chunks over 6 splits
    (2, 8, 8, 1280, 1280, False, True, PATCH + "<8,1,32,2,1,9,9>", "sum"),
    (1, 16, 16, 1280, 1280, True, True, PATCH + "<8,1,32,2,1,9,9>", "sum"),
    (1, 39, 6, 640, 72, True, False, PATCH + "<8,1,32,2,1,9,9>", "sum"),
    (1, 9, 35, 1920, 8, False, True, PATCH + "<8,1,32,2,1,9,9>", "reduce"),     # one column chunk
    # one sub-tile x 64 columns
    (1, 34, 38, 1920, 640, True, False, PATCH + "<8,1,64,2,2,9,9>", "whole"),
    (1, 5, 60, 1280, 80, False, True, PATCH + "<8,1,64,2,2,9,9>", "sum"),
    (3, 12, 7, 1920, 72, True, True, PATCH + "<8,1,64,2,2,9,9>", "sum"),
    # two sub-tiles x 64 columns, with the ring of all taps and without
    (2, 36, 28, 640, 640, True, True, PATCH + "<8,2,64,4,1,9,9>", "whole"),     # 10 chunks
    (4, 17, 119, 320, 80, False, True, PATCH + "<8,2,64,4,1,9,9>", "whole"),
    (3, 54, 9, 1280, 168, True, False, PATCH + "<8,2,64,4,1,9,9>", "sum"),      # an odd number of sub-tiles
    (2, 9, 89, 64, 328, True, False, PATCH + "<8,2,64,4,1,9>", "whole"),
    (5, 5, 17, 640, 1280, False, True, PATCH + "<8,2,64,4,1,9>", "sum"),        # sub-tiles of two images
    (4, 19, 9, 1280, 168, True, True, PATCH + "<8,2,64,4,1,9>", "reduce"),
    # two sub-tiles x 80 columns
    (5, 39, 5, 64, 1280, True, False, PATCH + "<8,2,80,4,1,9>", "whole"),
    (3, 203, 190, 64, 72, False, False, PATCH + "<8,2,80,4,1,9>", "whole"),
    (1, 84, 121, 640, 72, False, True, PATCH + "<8,2,80,4,1,9>", "sum"),
    (1, 18, 76, 1920, 72, True, False, PATCH + "<8,2,80,4,1,9>", "reduce"),
    (2, 16, 16, 1280, 1280, True, True, PATCH + "<8,2,80,4,1,9>", "reduce"),    # whole tiles
    # 16x16 pixels x 128 and 160 columns
    (5, 64, 64, 320, 320, True, True, PATCH + "<16,1,128,4,2,9>", "whole"),
    (1, 250, 243, 128, 128, True, False, PATCH + "<16,1,128,4,2,9>", "whole"),
    (2, 9, 118, 1920, 168, False, True, PATCH + "<16,1,128,4,2,9>", "reduce"),
    (1, 256, 256, 64, 136, False, False, PATCH + "<16,1,160,4,2,9>", "whole"),
    (5, 83, 86, 64, 136, True, True, PATCH + "<16,1,160,4,2,9>", "whole"),
    (4, 10, 123, 1920, 136, False, True, PATCH + "<16,1,160,4,2,9>", "reduce"),
    # one chunk: two 16x16 tiles x 64 columns per CU
    (1, 256, 250, 64, 64, True, True, PATCH + "<16,1,64,4,2,9,3,1>", "whole"),
    (5, 101, 28, 64, 72, True, False, PATCH + "<16,1,64,4,2,9,3,1>", "whole"),  # both directions, columns ragged
    (3, 203, 187, 64, 40, False, True, PATCH + "<16,1,64,4,2,9,3,1>", "whole"),
]

# dense products: M, N, K, K2, bias, residual, GEGLU, fp32 output, kernel, K sum
DENSE_TILES = [
    (1, 8, 64, 0, True, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "whole"),     # one row, chunk, K step
    (63, 72, 128, 0, True, False, False, True, DENSE + "<64,64,4,1,3,0,5>", "whole"),  # a row short of a tile
    (65, 64, 192, 64, False, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "whole"),  # a row past; two sources
    (129, 136, 64, 0, True, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "whole"),
    (257, 192, 320, 0, True, False, True, False, DENSE + "<64,64,4,1,3,0,3>", "whole"),
    (1594, 5128, 64, 0, True, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "whole"),  # several tiles a block
    (70, 72, 2048, 0, True, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "sum"),
    (300, 200, 4096, 1024, True, True, False, False, DENSE + "<64,64,4,1,3,0,0>", "sum"),  # splits in source 2
    (65, 136, 4096, 0, True, True, False, True, "gemm_kernel", None),                  # fp32 with a residual
    (65, 136, 4096, 0, True, False, False, False, DENSE + "<64,64,4,1,3,0,0>", "reduce"),
    (33, 128, 4096, 0, True, False, True, False, DENSE + "<64,64,4,1,3,0,3>", "reduce"),
    (33569, 136, 64, 0, False, True, False, False, DENSE + "<128,64,4,1,3,0,0>", "whole"),
    (40000, 136, 64, 0, True, True, False, False, DENSE + "<128,64,4,1,3,0,0>", "whole"),  # several tiles a block
    (33000, 320, 128, 64, True, False, False, False, DENSE + "<128,64,4,1,3,0,0>", "whole"),  # and two sources
    (16604, 8, 1920, 0, True, True, False, False, DENSE + "<128,64,4,1,3,0,0>", "sum"),
    (20000, 640, 192, 0, True, False, True, False, DENSE + "<128,128,2,2,2,0,3>", "whole"),
    (23422, 328, 64, 0, True, False, False, True, DENSE + "<128,128,2,2,2,0,5>", "whole"),
    (16409, 72, 1920, 0, True, True, False, False, DENSE + "<128,128,2,2,2,0,0>", "sum"),
    (33124, 328, 640, 0, True, True, False, False, DENSE + "<256,128,4,2,3,0,0>", "whole"),  # 390 tiles, 256 blocks
    (33124, 328, 640, 320, True, False, False, True, DENSE + "<256,128,4,2,3,0,5>", "whole"),
    (33124, 384, 640, 0, True, False, True, False, DENSE + "<256,128,4,2,3,0,3>", "whole"),
    (16902, 72, 3200, 1280, True, True, False, False, DENSE + "<256,128,4,2,3,0,0>", "sum"),
]
