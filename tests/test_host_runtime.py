"""The library's host side on a HIP runtime of host memory (host_runtime.cpp):
what calls keep, free and rebuild when allocations fail, without a GPU."""
import os
import subprocess

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(ROOT, "cugridder_amd", "libcurafft.so")


@pytest.fixture(scope="module")
def scenario(tmp_path_factory):
    """scenario(name, **environment) -> {name: value} of one run of the program"""
    import cugridder_amd
    cugridder_amd.lib()  # built
    exe = str(tmp_path_factory.mktemp("host_runtime") / "host_runtime")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                           "-rdynamic", os.path.join(HERE, "host_runtime.cpp"), "-o", exe, "-ldl", "-lpthread"])

    def run(name, **env):
        p = subprocess.run([exe, LIB, name], capture_output=True, text=True, timeout=60,
                           env={**os.environ, **env})
        assert p.returncode == 0, (p.returncode, p.stdout, p.stderr)
        out = {k: int(v) for k, v in (line.split() for line in p.stdout.splitlines())}
        assert out["bad_frees"] == 0 and out["bad_copies"] == 0, out
        return out

    return run


@pytest.mark.parametrize("where", ["twiddle_tags", "context_tags"])
def test_twiddle_tables_do_not_outlive_their_memory(scenario, where):
    """A call whose table cannot be allocated, or which ends between the two
    tables of a new precision, must not leave a later call a table that is
    gone or of the other precision."""
    r = scenario(where)
    assert r["first_tables"] == 2 and r["again_tables"] == 0
    assert r["failed_ier"] == 5
    assert r["after_row_ier"] == 0 and r["after_row_tables"] >= 1
    assert r["single_tables"] == 2
    assert r["failed_column_ier"] == 5
    assert r["single_again_ier"] == 0 and r["single_again_tables"] == 2
    assert r.get("left", 0) == 0


def test_release_without_host_memory(scenario):
    """cg_host_release is a C function: no exception may leave it, and with no
    host memory at hand it still gives everything back."""
    r = scenario("release_without_heap")
    assert r["ier"] == 0 and r["kept"] == 1
    assert r["release_ier"] == 0 and r["left"] == 0 and r["allocations_left"] == 0


def test_kept_memory_makes_room(scenario):
    """Memory kept from one call is given up when the next one needs the room,
    also by the call that leased it: neither is a call refused nor a grid cut
    into slabs that would run whole without the earlier call."""
    r = scenario("surplus")
    assert r["alone_ier"] == 0 and r["before_ier"] == 0 and r["kept"] == 1
    assert r["after_ier"] == 0
    assert r["many_ier"] == 0 and r["many_kept"] == 1
    assert r["whole_ier"] == 0 and r["slabs"] == 1


def test_device_reset_between_host_calls(scenario):
    """After hipDeviceReset a host call works as the first one did, and what the
    earlier calls kept is neither used nor freed, whoever has the addresses
    now."""
    r = scenario("device_reset")
    assert r["before_ier"] == 0 and r["kept"] == 1
    assert r["after_ier"] == 0
    assert r["release_ier"] == 0 and r["left"] == 0
    assert r["again_ier"] == 0 and r["moved_ier"] == 0 and r["others_freed"] == 0


def test_kept_memory_is_bounded(scenario):
    """CG_HOST_KEEP_MB bounds what host calls keep, down to nothing."""
    whole = scenario("kept_bytes")
    assert whole["ier"] == 0 and whole["second_ier"] == 0
    assert 3 << 20 < whole["kept"] <= whole["second_kept"]
    for mb in (0, 2, 1000):
        r = scenario("kept_bytes", CG_HOST_KEEP_MB=str(mb))
        assert r["ier"] == 0 and r["second_ier"] == 0
        for k in ("kept", "second_kept"):
            assert r[k] == (whole[k] if whole[k] <= mb << 20 else 0)


def test_release_from_python():
    import cugridder_amd
    cugridder_amd.release_host_memory()
    assert "release_host_memory" in cugridder_amd.__all__


def test_tile_edges_stay_accepted(scenario):
    """Gridding tiles of one cell, asked for or left after halving (3 and 12 on
    80 x 72 cells), are accepted up to kernel width 9, where the bins around a
    tile are at most 81, and refused by size above."""
    r = scenario("tile_edges")
    for tile in (0, 1, 2, 3, 5, 8, 12):
        for kw in (4, 9, 10, 13):
            assert r[f"tile{tile}_kw{kw}"] == (3 if tile < 2 and kw > 9 else 0)


def test_crowded_rule(scenario):
    """k_grid takes crowded regions where it is the faster one and nothing else
    does: narrow kernels or small tiles, enough rows for a region to be crowded,
    no dense path below that, tiles and blocks that cover the same cells."""
    r = scenario("crowded_rule")
    for name in ("narrow", "width8_tile2", "no_dense", "late_dense"):
        assert r[name] == 1, name
    for name in ("few_rows", "few_rows_wide", "width8_tile8", "width13", "odd_tile", "dense"):
        assert r[name] == 0, name
    # several windows of planes: narrower kernels only, complex64's narrower still
    for prec, windows, widest in ((1, 2, 6), (1, 4, 5), (0, 2, 5), (0, 4, 4)):
        for kw in (3, 4, 5, 6, 7):
            assert r[f"p{prec}_windows{windows}_kw{kw}"] == (kw <= widest), (prec, windows, kw)


def test_degrid_rule(scenario):
    """Tiles are read straight from the planes up to the mean number of points per
    tile from which staging them is the faster: fewer the smaller the tile and the
    wider the kernel, as the halo read for them grows; more the more planes there
    are, which staging reads whole; more from width 12 on, where the staged kernel
    spills."""
    r = scenario("degrid_rule")
    until = {(2, 4, 10): 40, (2, 6, 10): 40, (2, 9, 10): 25, (4, 4, 10): 40, (4, 6, 10): 40, (4, 9, 10): 40,
             (8, 4, 10): 90, (8, 6, 10): 90, (8, 9, 10): 70,
             (2, 4, 620): 70, (2, 6, 620): 40, (2, 9, 620): 25, (4, 4, 620): 90, (4, 6, 620): 90,
             (4, 9, 620): 40, (8, 9, 620): 90}
    for w in (10, 620, 4000):
        for tile in (2, 4, 8, 16):
            for kw in (4, 6, 9, 13):
                for per in (10, 25, 40, 70, 90, 120, 130):
                    most = until.get((tile, kw, w), 120)
                    assert r[f"tile{tile}_kw{kw}_w{w}_{per}"] == (per <= most), (tile, kw, w, per)


def test_column_rule(scenario):
    """complex128 column steps of powers of two take the prefetching kernel
    below a gibibyte and at lengths whose mixed-radix blocks are narrow."""
    r = scenario("column_rule")
    for name in ("p1_1x1024x1024", "p1_16x2048x1024"):
        assert r[name] == 2, name
    assert r["p1_16x8192x2048"] == 1  # of its steps of 64 and 128 points
    for name in ("p1_16x2048x2048", "p1_17x4096x2048", "p1_1x1000x1024", "p0_1x1024x1024"):
        assert r[name] == 0, name


def test_plans_without_heap(scenario):
    """A transform whose plan cannot be kept runs all the same: no exception
    leaves a C entry."""
    r = scenario("plans_without_heap")
    for prec in (0, 1):
        assert r[f"none{prec}_ier"] == 0
        for what in ("rows", "cols"):
            assert r[f"none{prec}_{what}"] == r[f"some{prec}_{what}"] > 0


def test_list_rule(scenario):
    """2-D gridding takes the tiles that are read from a list, which loses their
    order, on tiles of 32 cells and, where few are reached, on tiles whose rows fill
    cache lines: 3000^2 and 5400^2 cells have tiles of 8."""
    r = scenario("list_rule")
    for prec in (0, 1):
        for m in (30000, 1000000):
            assert r[f"p{prec}_256_{m}"] == 0        # 256 tiles
            for n in (1024, 2048):
                assert r[f"p{prec}_{n}_{m}"] == 1
            for n in (1500, 2700):
                assert r[f"p{prec}_{n}_{m}"] == (prec == 1 and m == 30000)
