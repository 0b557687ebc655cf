"""Static checks on the gfx950 assembly hipcc generates for the kernel on bf16 planes (no GPU needed): the registers of as many wavefronts as a SIMD is to
hold, nothing spilled in the loop over the slices, and the order of instructions that the source gives."""
import os
import re
from concurrent.futures import ThreadPoolExecutor

import pytest

import test_kernel_asm as K

pytestmark = pytest.mark.skipif(not os.path.exists(K.HIPCC), reason="hipcc not installed")

MFMA = "v_mfma_f32_16x16x32_bf16"
#        tile: wavefronts per SIMD (work-group of eight, of twelve), MFMAs of a wavefront's slice
TILES = {0: (2, 96), 1: (2, 48), 2: (2, 48), 3: (3, 24)}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    outdir = str(tmp_path_factory.mktemp("asm"))
    with ThreadPoolExecutor(max_workers=4) as ex:
        return dict(zip(TILES, ex.map(lambda t: K._compile(("inst_planes.hip", [f"-DMMBO_TILE={t}"]), outdir), TILES)))


def _main_loop(body):
    """The instructions of the loop with the most of these MFMAs: from a label to the last branch back to it."""
    at = {t[:-1]: i for i, t in enumerate(body) if t.endswith(":")}
    loops = []
    for i, t in enumerate(body):
        m = re.match(r"s_c?branch\S*\s+(\.LBB\w+)", t)
        if m and m[1] in at and at[m[1]] < i:
            loops.append((sum(x.startswith(MFMA) for x in body[at[m[1]]:i]), at[m[1]], i))
    return loops


@pytest.mark.parametrize("tile", TILES)
def test_registers_and_the_main_loop(assembly, tile):
    per_simd, mfmas = TILES[tile]
    text, kernels = open(assembly[tile]).read(), K._kernels(assembly[tile])
    assert len(kernels) == 4                                    # the transposes
    for name, body in kernels.items():
        m = re.search(r"\.amdhsa_kernel " + re.escape(name) + r"\b.*?\.amdhsa_next_free_vgpr (\d+)", text, re.S)
        assert int(m[1]) <= 512 // per_simd // 8 * 8, (name, m[1])
        loops = _main_loop(body)
        most = max(n for n, _, _ in loops)
        assert most == 2 * mfmas, (name, most)                  # a turn: two slices
        first, last = min(a for n, a, _ in loops if n == most), max(b for n, _, b in loops if n == most)
        inside = body[first:last + 1]
        assert sum(t.startswith(MFMA) for t in inside) == 2 * mfmas
        assert not [t for t in inside if t.startswith(("scratch_", "v_readlane", "v_writelane"))], name
        # every MFMA is followed by its share of the rest: never more than two of them in a row but where a slice has next to nothing else
        row = longest = 0
        for t in inside:
            row = row + 1 if t.startswith(MFMA) else 0
            longest = max(longest, row)
        assert longest <= 3, (name, longest)
