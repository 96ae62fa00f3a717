"""Shapes at which the operator plans take every chunk capacity, and those of the
paired gradients, shared by the GPU parity tests and by the host test that
checks which plans they give."""

# (line, capacity of the plan, every chunk holds it): y / z lines in wide launches
WIDE_LINES = [(22, 12, False), (24, 12, True), (44, 12, False), (48, 12, True), (60, 16, False), (64, 16, True),
              (130, 24, False), (190, 24, False), (192, 24, True), (200, 32, False), (250, 32, False), (256, 32, True),
              (384, 24, True)]
# as WIDE_LINES, in launches of few lines
FEW_LINES = [(60, 8, False), (64, 8, True), (100, 8, False)]
# x lines beside those of test_wave_local_x: 64 chunks of nine to twelve points
X_LINES = [(520, 12, False), (640, 12, False), (700, 12, False), (768, 12, True)]


def wide(line, dim, lanes=49, outer=86):
    return (lanes, line, outer) if dim == 2 else (lanes, outer, line)


# (shape, periodic in y, species, the y and z gradients share a launch)
PAIRS = [((24, 20, 20), True, 1, True), ((24, 33, 20), True, 1, False), ((64, 17, 19), True, 1, True),
         ((50, 40, 36), True, 2, True), ((12, 9, 24), True, 1, False), ((64, 64, 64), True, 1, True),
         ((64, 66, 64), True, 1, False), ((64, 62, 64), True, 1, True), ((64, 64, 62), False, 1, True),
         ((20, 30, 28), False, 1, True)]
