"""Shapes of the int8 mode's GPU tests, with the kernel each is there for
(on 256 CUs): "small" (64 x 64 blocks) or 160 rows x 128 / 256 tokens."""
Q4_K, Q6_K = 12, 14

# (dtype, rows, k, n, kernel)
INT8_KERNELS = [
    # one unit and several, one block and several, each with a ragged last
    # row tile, token tile and unit
    (Q6_K, 1, 256, 1, "small"), (Q6_K, 63, 130, 64, "small"), (Q6_K, 130, 256, 200, "small"),
    (Q6_K, 65, 512, 65, "small"), (Q6_K, 300, 721, 129, "small"), (Q6_K, 2405, 768, 701, "small"),
]
