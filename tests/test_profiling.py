"""Short kernel names of the profile summaries against the launches in the sources (CPU)."""
import glob
import os
import re

from large_model_amd.profiling import counters, short_name

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "large_model_amd", "csrc")


def test_short_names_match_launch_names():
    src = "".join(open(p).read() for p in glob.glob(os.path.join(CSRC, "*.hip")))
    launches = re.findall(r'QLAUNCH\("(\w+)",\s*\(?(\w+_kernel)\b', src)
    assert len(launches) > 30
    for name, kernel in launches:
        if kernel not in ("tile_rows_kernel", "mx_kernel"):          # named by a template argument
            assert short_name(f"void qmsg::{kernel}<14, 1, 8>(qmsg::Args)") == name, kernel


def test_short_names_by_template_argument():
    for full, name in (("void qmsg::mx_kernel<2, 1, 1, 8, 4, 3, 2>(qmsg::MxArgs)", "gateup"),
                       ("void qmsg::mx_kernel<14, 1, 0, 4, 4, 2, 1>(qmsg::MxArgs)", "down"),
                       ("void qmsg::mx_kernel<14, 1, 3, 4, 4, 2, 1>(qmsg::MxArgs)", "down"),
                       ("void qmsg::mx_kernel<2, 2, 2, 4, 8, 2, 1>(qmsg::MxArgs)", "dense"),
                       ("void qmsg::tile_rows_kernel<14, 4, 32, 1>(qmsg::TileArgs)", "gateup"),
                       ("void qmsg::tile_rows_kernel<14, 4, 32, 0>(qmsg::TileArgs)", "down"),
                       ("void qmsg::(anonymous namespace)::chain_rows_kernel<8, 2, true, false>(qmsg::ChainArgs)", "gateup"),
                       ("void qmsg::(anonymous namespace)::chain_rows_kernel<8, 2, false, false>(qmsg::ChainArgs)", "rows_f32"),
                       ("__amd_rocclr_copyBuffer", "__amd_rocclr_copyBuffer")):
        assert short_name(full) == name, full


def test_counters_keep_kernels_of_an_anonymous_namespace_apart(tmp_path):
    rows = ["Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value"]
    for i, arg in enumerate(("true", "false", "true")):
        rows.append(f'{i},"void qmsg::(anonymous namespace)::chain_rows_kernel<8, 2, {arg}, false>(qmsg::ChainArgs)",SQ_WAVES,{i + 1}')
    (tmp_path / "p_counter_collection.csv").write_text("\n".join(rows) + "\n")
    out = counters([str(tmp_path)])
    assert out[0].startswith("void qmsg::chain_rows_kernel<8, 2, false, false>  [1 ") and out[1].split() == ["SQ_WAVES", "2"]
    assert out[2].startswith("void qmsg::chain_rows_kernel<8, 2, true, false>  [2 ") and out[3].split() == ["SQ_WAVES", "2"]
