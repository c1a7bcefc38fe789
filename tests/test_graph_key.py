"""Keys of the kept CG/FCG graphs (CPU): every value and buffer that the launches
of the operators hold changes the key.

A small program is compiled against the library's internal header; it changes
one field of a context at a time and compares the keys (mf_key: the FP32
matrix-free operator, tiled and element by element; kf_key: the FP64 element
products).  The fields are those that the launch code reads.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

TILED = ["mf_tile", "mt_nt[0]", "mt_nt[1]", "mt_nt[2]", "mt_fn[0]", "mt_fn[1]", "mt_fn[2]", "mf_box_inv[0]",
         "mf_box_inv[1]", "mf_box_inv[2]", "mf_box_det", "mt_nh", "kf_nface", "nu", "d_mt_tmap.p", "d_mt_coef.p",
         "d_mt_part.p", "d_mt_hfine.p", "d_mt_hblk.p", "d_kf_pidx.p", "d_kf_pptr.p", "d_kf_psrc.p", "d_kf_bblk.p",
         "d_mf_bm.p", "d_mf_pt.p", "d_mf_dis.p"]
ELEMENTS = ["mf_tile", "dim", "nstate", "nvol", "nb", "neq", "nu", "tvol.nq", "tvol.nsh", "tbc.nsh", "mf_nbcd",
            "mf_nout", "d_mf_tab.p", "d_mf_blk.p", "d_mf_xe.p", "d_mf_coef.p", "d_mf_geo.p", "d_mf_pt.p",
            "d_mf_pos.p", "d_mf_ye.p", "d_mf_mfma.p", "d_mf_bblk.p", "d_mf_bm.p", "d_mf_bpos.p", "d_mf_ptr.p",
            "d_mf_dis.p"]
FP64 = ["bs", "neq", "nvol", "kf_nface", "E", "d_vcoef.p", "d_kf_tab.p", "d_kf_blk.p", "d_kf_ye.p",
        "d_blk_iptr.p", "d_blk_inc.p", "d_kf_pidx.p", "d_kf_pptr.p", "d_kf_psrc.p", "d_kf_bblk.p", "d_kf_bm.p"]


def _source():
    def checks(fields, fn, start):
        out = []
        for f in fields:
            change = f"*(char **)&c.{f} += 4096" if f.endswith(".p") else \
                f"c.{f} = !c.{f}" if f == "mf_tile" else f"c.{f} += 1"
            out.append(f'  {{ Ctx c; {start} auto a = key({fn}, c); {change}; '
                       f'if (key({fn}, c) == a) {{ std::puts("{fn}: {f}"); bad = 1; }} }}')
        return "\n".join(out)
    return f"""#include <cstdio>
#include "pzg_internal.h"
using namespace pzg;
typedef std::vector<uint64_t> Key;
static Key key(void (*fn)(const Ctx &, Key &), const Ctx &c) {{ Key k; fn(c, k); return k; }}
int main() {{
  int bad = 0;
{checks(TILED, "mf_key", "c.mf_tile = true;")}
{checks(ELEMENTS, "mf_key", "")}
{checks(FP64, "kf_key", "c.material = PZG_MAT_ELAST3D;")}
  {{ Ctx c; auto a = key(kf_key, c); c.vol_coef.assign(1, 1.); if (key(kf_key, c) == a) {{ std::puts("vol_coef"); bad = 1; }} }}
  return bad;
}}
"""


def test_every_field_is_in_the_key(tmp_path):
    lib = os.path.join(ROOT, "neopz_amd")
    if not os.path.exists(os.path.join(lib, "libpzg.so")):
        pytest.skip("library not built")
    src, exe = tmp_path / "key.cpp", tmp_path / "key"
    src.write_text(_source())
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(lib, "csrc"), str(src), "-o", str(exe), "-L" + lib, "-lpzg",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib + ":/opt/rocm/lib"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, "not in the key:\n" + r.stdout + r.stderr
