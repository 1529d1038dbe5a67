"""Loads that go from global memory to LDS directly take their LDS address from M0, which a scalar instruction writes.  That write needs
one wait state before such a load reads it; between instructions of its own the compiler sees to it, inside one asm statement nobody
does.  The assembly of every unit that holds such a load is looked over, compiled as the library is.  No GPU is needed."""
import functools
import os
import re
import subprocess

import pytest

from polarquant_amd import build

UNITS = [u for us in [build.UNITS] + list(build.LAYER_UNITS.values()) for u in us]


def _includes(name, seen):
    if name not in seen and os.path.exists(os.path.join(build.CSRC, name)):
        text = seen[name] = open(os.path.join(build.CSRC, name)).read()
        for inner in re.findall(r'#include "([^"]+)"', text):
            _includes(inner, seen)
    return seen


WITH_LOADS = [u for u in UNITS if any("global_load_lds" in t for t in _includes(u[0], {}).values())]


def _early_loads(listing):
    """(loads to LDS, those that directly follow a write of M0)"""
    loads, early, previous = 0, [], ""
    for line in listing.splitlines():
        line = line.split(";")[0].strip()
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        if re.match(r"(global_load_lds|buffer_load\S* .*\blds\b)", line):
            loads += 1
            if re.match(r"s_\S+ m0\b", previous):
                early.append(previous + " / " + line)
        previous = line
    return loads, early


def test_the_check_itself():
    bad = "\ts_mov_b32 m0, s4\n\t;;#note\n\tglobal_load_lds_dwordx4 v[0:1], off\n"
    assert _early_loads(bad) == (1, ["s_mov_b32 m0, s4 / global_load_lds_dwordx4 v[0:1], off"])
    assert _early_loads(bad.replace(";;#note", "s_nop 0")) == (1, [])


@functools.lru_cache(maxsize=None)
def _listing(src, defines):
    cmd = [build._hipcc()] + build.FLAGS + ["-D" + d for d in defines] + ["--cuda-device-only", "-S", os.path.join(build.CSRC, src), "-o", "-"]
    run = subprocess.run(cmd, capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    return run.stdout


@pytest.mark.parametrize("src,defines", [u[:2] for u in WITH_LOADS], ids=[u[0] + u[2] for u in WITH_LOADS])
def test_a_wait_state_before_every_load_to_lds(src, defines):
    loads, early = _early_loads(_listing(src, defines))
    assert loads > 0 and not early, "%d of %d loads: %s" % (len(early), loads, early[:3])


def test_latent_prompts_of_any_width_stay_in_registers():
    """The kernels with a row of values per channel, heads up to 64, 128, 192 and 256 wide in both dtypes.  Spilled sums go through memory
    in every tile (256 wide: 1.6 times the time)."""
    spilled = {name: int(n) for name, n in re.findall(r"\.name: +(\S*prompt_attn_kernel\S*)\n(?:.*\n)*? +\.vgpr_spill_count: (\d+)", _listing("pq_latent_attn.hip", ()))}
    assert len(spilled) == 8 and not any(spilled.values()), spilled


@pytest.mark.parametrize("src,defines", [u[:2] for u in WITH_LOADS], ids=[u[0] + u[2] for u in WITH_LOADS])
def test_the_first_tile_waits_for_no_load(src, defines):
    """The queries are asked for first, but the first tile must not wait for them, nor one of them for another: a prompt of a tile or two
    is little else than its start."""
    kernels = re.findall(r"^(\S*prompt_attn_kernel\S*):.*\n((?:.*\n)*?).*\bglobal_load_lds", _listing(src, defines), re.M)
    assert kernels
    for name, start in kernels:
        loads, waits = len(re.findall(r"^\s+global_load_dwordx4", start, re.M)), re.findall(r"s_waitcnt .*vmcnt", start)
        assert loads >= 4 and not waits, (name, loads, len(waits))
