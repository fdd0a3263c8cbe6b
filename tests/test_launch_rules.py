"""The rules that choose a kernel by block count, against times of both kernels on an
MI355X (256 compute units; us of one step, tiles and the other kernel): where a rule
leaves the tiles, the other kernel is not slower than them by more than such times
differ from run to run."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")
NOISE = 1.03

# (dimension, flux, mode): blocks -> (tiles, marching in 3D or pairs of blocks in 2D);
# flux 0 HLLC, 1 Roe; mode 0 exact, 1 FP64 with FMA.
TIMES = {
    (3, 0, 0): {
        64: (212, 438), 96: (300, 446), 97: (378, 441), 100: (379, 447), 112: (383, 451),
        128: (388, 457), 192: (574, 726), 225: (733, 743), 256: (778, 768), 257: (824, 1067),
        320: (982, 1099), 353: (1124, 1108), 384: (1188, 1155), 385: (1220, 1384),
        449: (1417, 1423), 512: (1567, 1524), 513: (1598, 1729), 600: (1845, 1825),
        640: (1957, 1894), 768: (2339, 2249), 1024: (3103, 2967), 1536: (4670, 4448),
        2047: (6242, 5896), 2048: (6220, 5886), 2560: (7816, 7394),
    },
    (3, 0, 1): {
        64: (115, 231), 96: (164, 235), 97: (194, 235), 100: (196, 236), 112: (200, 239),
        128: (212, 245), 192: (317, 406), 225: (398, 430), 256: (440, 462), 257: (448, 609),
        320: (547, 645), 353: (638, 664), 384: (682, 697), 385: (695, 820), 449: (800, 863),
        512: (913, 925), 513: (921, 1032), 600: (1060, 1106), 640: (1134, 1142),
        768: (1349, 1364), 1024: (1793, 1794), 1536: (2666, 2679), 2047: (3555, 3539),
        2048: (3567, 3525), 2560: (4480, 4413),
    },
    (3, 1, 0): {
        64: (248, 506), 96: (361, 522), 97: (448, 520), 100: (447, 525), 112: (451, 533),
        128: (466, 549), 192: (698, 873), 225: (878, 896), 256: (946, 936), 257: (991, 1301),
        320: (1175, 1329), 353: (1355, 1345), 384: (1418, 1392), 385: (1465, 1703),
        449: (1709, 1737), 512: (1877, 1848), 513: (1935, 2127), 600: (2228, 2220),
        640: (2353, 2295), 768: (2817, 2736), 1024: (3748, 3614), 1536: (5629, 5420),
        2047: (7541, 7221), 2048: (7570, 7189), 2560: (9448, 8981),
    },
    (3, 1, 1): {
        64: (135, 257), 96: (192, 269), 97: (230, 270), 100: (232, 271), 112: (238, 276),
        128: (251, 285), 192: (376, 462), 225: (478, 497), 256: (528, 537), 257: (548, 714),
        320: (675, 754), 353: (776, 781), 384: (828, 811), 385: (844, 955), 449: (985, 1008),
        512: (1101, 1085), 513: (1126, 1209), 600: (1299, 1308), 640: (1370, 1351),
        768: (1637, 1608), 1024: (2172, 2126), 1536: (3250, 3143), 2047: (4335, 4205),
        2048: (4335, 4187), 2560: (5423, 5214),
    },
    (2, 0, 0): {
        1152: (176, 207), 1535: (181, 211), 1536: (180, 212), 1600: (224, 214), 2025: (276, 228),
        2500: (308, 277), 2560: (322, 280), 3249: (370, 388), 4096: (458, 446), 4900: (510, 512),
        8192: (853, 814), 9025: (946, 908), 16384: (1666, 1644),
    },
    (2, 0, 1): {
        1152: (99, 114), 1535: (124, 118), 1536: (123, 118), 1600: (124, 121), 2025: (129, 130),
        2500: (173, 156), 2560: (174, 156), 3249: (199, 210), 4096: (246, 246), 4900: (283, 280),
        8192: (491, 470), 9025: (519, 531), 16384: (998, 978),
    },
    (2, 1, 0): {
        1152: (197, 233), 1535: (204, 239), 1536: (202, 239), 1600: (253, 240), 2025: (310, 252),
        2500: (357, 312), 2560: (361, 324), 3249: (422, 440), 4096: (523, 513), 4900: (591, 591),
        8192: (993, 960), 9025: (1082, 1057), 16384: (1967, 1889),
    },
    (2, 1, 1): {
        1152: (106, 122), 1535: (112, 126), 1536: (112, 126), 1600: (136, 129), 2025: (163, 142),
        2500: (188, 167), 2560: (191, 172), 3249: (220, 231), 4096: (270, 269), 4900: (312, 308),
        8192: (549, 531), 9025: (596, 579), 16384: (1101, 1056),
    },
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """rule(dim, flux, mode, blocks): whether the tiles are left."""
    if CXX is None:
        pytest.skip("no host compiler")
    work = tmp_path_factory.mktemp("rules")
    src, exe = work / "rules.cpp", work / "rules"
    src.write_text('#include <cstdio>\n#include "launch_rules.h"\n'
                   "int main() {\n  int dim, flux, mode;\n  long long n;\n"
                   '  while (std::scanf("%d %d %d %lld", &dim, &flux, &mode, &n) == 4)\n'
                   '    std::printf("%d\\n", int(dim == 3 ? alpaca::rule_marches(flux, mode, n, 256)\n'
                   "                                      : alpaca::rule_pairs(flux, mode, n, 256)));\n}\n")
    subprocess.run([CXX, "-std=c++17", "-I", os.path.join(ROOT, "alpaca_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True)

    def ask(*args):
        out = subprocess.run([str(exe)], input=" ".join(map(str, args)), capture_output=True,
                             text=True, check=True)
        return out.stdout.strip() == "1"
    return ask


@pytest.mark.parametrize("form", sorted(TIMES))
def test_tiles_are_left_for_a_kernel_that_is_not_slower(rule, form):
    left = [n for n in TIMES[form] if rule(*form, n)]
    slower = {n: TIMES[form][n] for n in left if TIMES[form][n][1] > NOISE * TIMES[form][n][0]}
    assert left and not slower


@pytest.mark.parametrize("flux", [0, 1])
@pytest.mark.parametrize("blocks", [1, 255, 256, 2048, 16384, 1 << 24])
def test_mixed_forms_never_march(rule, flux, blocks):
    assert not rule(3, flux, 2, blocks)
