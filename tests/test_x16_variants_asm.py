"""The 16x16-block ring kernel's variants by what of C they are sent, on the gfx950 assembly hipcc generates (no GPU needed): each holds
only its own code, and the odd-column one passes the checks of the others."""
import os
import re
from concurrent.futures import ThreadPoolExecutor

import pytest

import test_kernel_asm as K

pytestmark = pytest.mark.skipif(not os.path.exists(K.HIPCC), reason="hipcc not installed")

TILES = (0, 2, 5)                          # 256x256, 128x128, 192x192


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    outdir = str(tmp_path_factory.mktemp("asm"))
    units = [("inst_x16.hip", ["-DMMBO_DTYPE=1", f"-DMMBO_TILE={t}"] + odd) for t in TILES for odd in ([], ["-DMMBO_ODD_C"])]
    units += [("inst_x16.hip", ["-DMMBO_DTYPE=1", f"-DMMBO_TILE={t}", "-DMMBO_ODD_C"]) for t in range(8) if t not in TILES]
    with ThreadPoolExecutor(max_workers=8) as ex:
        return list(zip(units, ex.map(lambda u: K._compile(u, outdir), units)))


def _code_bytes(path):
    return {m[1]: int(m[2]) for m in re.finditer(r"^(_Z\w+):.*?; codeLenInByte = (\d+)", open(path).read(), re.S | re.M)}


def _key(name):
    """A kernel's name without its role (the last enumerator of the mangled template arguments)."""
    return re.sub(r"CRoleE\d", "CRole", name)


def test_variants_hold_less_code_than_the_general_kernel(assembly):
    size = {}
    for _, path in assembly:
        for name, code in _code_bytes(path).items():
            size.setdefault(_key(name), {})[re.search(r"CRoleE(\d)", name)[1]] = code
    compared = 0
    for name, by_role in size.items():
        if "0" not in by_role:
            continue
        assert len(by_role) == 3, (name, by_role)
        # (general, old C ahead, odd columns: 130, 85 and 63 KB for 256 x 256 TN)
        assert by_role["1"] < 0.8 * by_role["0"] and by_role["2"] < 0.8 * by_role["0"], (name, by_role)
        compared += 1
    assert compared == 5 + 5 + 4             # four transposes, TN once more on five buffers with both operands on the even slices


def test_odd_column_kernels_pass_the_checks_of_the_others(assembly):
    seen = 0
    for (_, defs), path in assembly:
        if "-DMMBO_ODD_C" not in defs:
            continue
        text = open(path).read()
        own = K._compiler_generated(path)
        for name, body in K._kernels(path).items():
            assert "CRoleE2" in name
            assert not K._inflight_violations(body), name
            assert not K._unpadded_wide_stores(body), name
            assert all(re.search(r"s\[\d+:\d+\], 0 offen", t) for t in body if t.startswith("buffer_store_dwordx")), name
            assert not [t for t in own[name] if re.search(r"\ba\[?\d|\bm0\b", t)], name
            used = set()
            for t in body:
                for a, b in re.findall(r"\ba\[(\w+):(\w+)\]", t):
                    used.update(range(int(a, 0), int(b, 0) + 1))
                used.update(int(a, 0) for a in re.findall(r"\ba\[(\w+)\]", t))
            m = re.search(r"\.amdhsa_kernel " + re.escape(name) + r"\b.*?\.amdhsa_next_free_vgpr (\d+).*?\.amdhsa_accum_offset (\d+)", text, re.S)
            assert used == set(range(len(used))) and int(m[1]) - int(m[2]) == len(used), name
            seen += 1
    assert seen == 8 * 4 + 5
