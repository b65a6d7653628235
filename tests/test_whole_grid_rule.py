"""The fused engine's choice between the sweep and whole-grid steps at grids where both forms
were measured."""
import pytest

from fdtd_accelerate_amd import autotune

# arguments of whole_grid_faster without the measured us per step: (cells, box, segments, tile,
# face cells, bytes of CE, CE triples, Drude box, plane wave); whole grid, sweep
_MEASURED = [
    ((23040000, (299, 299, 224), 1, (13, 28), 1800000, 12, False, False, False), 400, 351),  # 300x300x250, CPML 10, CE float, z faces, periodic x and y
    ((16777216, (255, 255, 224), 1, (8, 32), 1310720, 3, True, False, False), 270, 246),  # 256x256x256, CPML 10, CE index, z faces, periodic x and y
    ((89915392, (447, 447, 416), 2, (13, 64), 4014080, 12, False, False, False), 1472, 1345),  # 448x448x448, CPML 10, CE float, z faces, periodic x and y
    ((29376000, (359, 299, 224), 1, (13, 33), 2160000, 3, True, False, False), 497, 436),  # 360x300x270, CPML 10, CE index, z faces, periodic x and y
    ((27948288, (302, 241, 384), 2, (13, 24), 0, 12, False, False, False), 422, 352),  # 302x241x369, CPML 0, CE float
    ((27855168, (327, 242, 352), 2, (13, 26), 0, 0, False, False, False), 356, 331),  # 327x242x339, CPML 0, CE none
    ((35687872, (311, 326, 352), 2, (11, 39), 0, 12, False, False, False), 534, 495),  # 311x326x340, CPML 0, CE float
    ((22791040, (239, 298, 320), 2, (13, 22), 0, 3, True, False, False), 315, 285),  # 239x298x318, CPML 0, CE index
    ((15586560, (205, 198, 384), 2, (11, 15), 0, 12, False, False, False), 248, 232),  # 205x198x384, CPML 0, CE float
    ((35060736, (404, 226, 384), 2, (13, 29), 0, 12, False, False, False), 559, 494),  # 404x226x384, CPML 0, CE float
    ((86687744, (511, 406, 384), 2, (13, 32), 4167680, 3, True, False, False), 1291, 1160),  # 512x407x416, CPML 10, CE index, z faces, periodic x and y
    ((21852160, (352, 388, 160), 1, (13, 44), 0, 0, False, False, False), 302, 268),  # 352x388x160, CPML 0, CE none
    ((10422496, (143, 220, 224), 1, (7, 8), 2304848, 3, True, True, False), 205, 286),  # 161x238x265, CPML 8, CE index, Drude box
    ((56623104, (362, 362, 352), 2, (13, 16), 8847360, 12, False, False, True), 982, 1176),  # 384x384x384, CPML 10, CE float, plane wave
    ((89915392, (426, 426, 384), 2, (7, 16), 12042240, 3, True, True, False), 1557, 1923),  # 448x448x448, CPML 10, CE index, Drude box
    ((56623104, (362, 362, 352), 2, (13, 16), 8847360, 3, True, False, True), 948, 1077),  # 384x384x384, CPML 10, CE index, plane wave
    ((79027200, (482, 328, 384), 2, (7, 16), 11179840, 0, False, True, False), 1317, 1721),  # 504x350x448, CPML 10, CE none, Drude box
    ((306240, (36, 44, 32), 1, (1, 8), 274960, 3, True, False, False), 15, 41),  # 58x66x80, CPML 10, CE index
    ((456320, (0, 0, 0), 0, (1, 1), 426000, 0, False, False, False), 16, 19),  # 62x115x60, CPML 12, CE none
    ((12161664, (206, 152, 352), 2, (13, 10), 506736, 12, False, False, False), 211, 236),  # 207x153x384, CPML 8, CE float, z faces, periodic x and y
    ((4239872, (156, 78, 192), 1, (5, 10), 1991808, 0, False, False, False), 64, 86),  # 182x104x224, CPML 12, CE none
    ((16839040, (306, 291, 128), 1, (13, 28), 5018016, 0, False, False, False), 279, 318),  # 332x317x160, CPML 12, CE none
    ((10394208, (167, 280, 96), 1, (9, 21), 3369480, 0, False, False, False), 170, 245),  # 193x306x163, CPML 12, CE none
    ((3038208, (74, 111, 224), 1, (4, 9), 1095104, 0, False, False, False), 46, 66),  # 92x129x256, CPML 8, CE none
    ((6899200, (196, 110, 320), 2, (11, 8), 0, 12, False, False, False), 91, 120),  # 196x110x320, CPML 0, CE float
    ((7862400, (175, 234, 192), 1, (13, 13), 0, 0, False, False, False), 85, 97),  # 175x234x178, CPML 0, CE none
    ((664000, (99, 82, 32), 1, (4, 9), 132800, 12, False, False, False), 26, 58),  # 100x83x77, CPML 8, CE float, z faces, periodic x and y
    ((5628480, (163, 194, 96), 1, (13, 10), 767520, 12, False, False, False), 92, 152),  # 164x195x170, CPML 12, CE float, z faces, periodic x and y
    ((307200, (79, 59, 32), 1, (3, 8), 76800, 12, False, False, False), 22, 49),  # 80x60x60, CPML 8, CE float, z faces, periodic x and y
]


@pytest.mark.parametrize("args,whole,sweep", _MEASURED)
def test_the_faster_form_is_picked(args, whole, sweep):
    assert autotune.whole_grid_faster(*args) == (whole < sweep)


@pytest.mark.gpu
def test_a_tuned_tile_does_not_force_the_sweep():
    """A tile that tune_fused measured is the sweep's; whether a step sweeps is the rule's."""
    from fdtd_accelerate_amd.sim import YeeSim
    key = (40, 44, 48, 6)
    assert key not in autotune._load()
    autotune._load()[key] = (3, 8)
    try:
        s = YeeSim(40, 44, 48, npml=6, coeff_use="", engine="fused")
        s.run(1)
        assert (s._fused.T, s._fused.CX) == (3, 8) and s._fused.whole_grid
    finally:
        del autotune._load()[key]
