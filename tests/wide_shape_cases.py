"""Launches of the wide chain kernel with one destination and the shape that each takes on a GPU of 256 compute units: run on the GPU
by test_gpu_wide_shapes.py, asked of the rule on the CPU by test_host_wide_shapes.py."""
MIB = 1 << 20
CUS = 256
SIZE = {"int8": 1, "int16": 2, "int32": 4, "int64": 8, "fp16": 2, "bf16": 2, "fp32": 4, "fp64": 8}


def segment_lengths(esz, total, straddle):
    """Elements of four segments of `total` bytes in all: around the largest tile (64 KiB).  Straddling: lengths that leave the
    segments at any element; otherwise every segment begins at a multiple of 16 bytes."""
    edge = 65536 // esz
    whole = total // esz
    if straddle:
        return [edge - 1, whole - 3 * edge - 3, 1, 2 * edge + 3]
    return [edge, whole - 3 * edge, 16 // esz, 2 * edge - 16 // esz]


# type, operation, sources, bytes of the result, straddling, shape.  "sum" of the 16-bit floats: fp32 inside, narrowed once.
SMALL = [(d, op, 5, total, straddle, shape)
         for d, op in (("fp32", "prod"), ("fp32", "min"), ("bf16", "max"), ("fp16", "sum"), ("fp16", "prod"), ("fp64", "sum"), ("fp64", "min"),
                       ("int8", "sum"), ("int8", "prod"), ("int8", "max"), ("int16", "min"), ("int32", "prod"), ("int64", "sum"))
         for total, straddle, shape in ((2 * MIB, False, "many"), (4 * MIB, True, "small"), (11 * MIB, False, "three"),
                                        (15 * MIB, False, "four"))]
# both sides of every limit
EDGES = [("fp32", "sum", 5, 4 * MIB - 16, True, "many"), ("fp32", "sum", 5, 4 * MIB, True, "small"),
         ("fp32", "sum", 5, 8 * MIB - 16, False, "many"), ("fp32", "sum", 5, 8 * MIB, False, "three"),
         ("bf16", "sum", 9, 32 * MIB - 16, True, "small"), ("bf16", "sum", 9, 32 * MIB, True, "three")]
LARGE = ([(d, op, 9, 144 * MIB, False, "large") for d, op in (("fp32", "sum"), ("bf16", "sum"), ("fp16", "prod"), ("int8", "sum"), ("int16", "min"),
                                                              ("int64", "sum"))] +
         [("fp32", "min", 9, 144 * MIB, True, "large"), ("fp64", "sum", 9, 144 * MIB, True, "large"), ("int32", "max", 5, 144 * MIB, False, "large"),
          ("fp32", "sum", 5, 144 * MIB - 16, False, "three"), ("bf16", "sum", 9, 144 * MIB, True, "three"),
          ("bf16", "max", 7, 144 * MIB, False, "three")])
CASES = SMALL + EDGES + LARGE
