"""Shapes of the batched product's GPU tests that are there for one kernel, on
256 CUs."""
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14

# Batches of up to 128 tokens on the 160 x 256 bf16 kernel: one unit a row, one
# and several row tiles with and without a ragged last one, ragged units.
BF16_SHORT_DIRECT = [
    (Q4_K, 480, 256, 97), (Q5_K, 30001, 250, 128), (Q6_K, 14335, 256, 113), (Q8_0, 4800, 224, 128),
    (Q4_K, 37888, 131, 33), (Q8_0, 37889, 512, 128),
]

# The int8 mode: (dtype, rows, k, n, kernel), the kernel "small" (64 x 64 blocks)
# or the tokens of its 160-row blocks.
INT8_KERNELS = [
    # one unit and several, one block and several, each with a ragged last
    # row tile, token tile and unit
    (Q6_K, 1, 256, 1, "small"), (Q6_K, 63, 130, 64, "small"), (Q6_K, 130, 256, 200, "small"),
    (Q6_K, 65, 512, 65, "small"), (Q6_K, 300, 721, 129, "small"), (Q6_K, 2405, 768, 701, "small"),
    # one unit (the kernel without a unit's running sum), several, and K splits
    (Q4_K, 161, 250, 129, 128), (Q4_K, 159, 721, 127, 128), (Q4_K, 161, 1500, 129, 128),
    (Q6_K, 9001, 250, 509, 128), (Q6_K, 600, 1000, 9, 128), (Q6_K, 161, 1500, 129, 128),
    (Q4_K, 18945, 250, 257, 256), (Q4_K, 9003, 721, 600, 256), (Q4_K, 2405, 2500, 129, 256),
    (Q6_K, 18945, 250, 257, 256), (Q6_K, 9003, 721, 600, 256), (Q6_K, 2405, 2500, 129, 256),
]
