"""Host-side parts of the library compiled with g++ against a runtime that the test itself stands in for: no GPU, no
HIP runtime."""
import os
import re
import struct
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture
def run_native(tmp_path):
    def run(source, *more):
        exe = str(tmp_path / source.rsplit(".", 1)[0])
        subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                               "-x", "c++", os.path.join(HERE, "native", source)] + list(more) + ["-o", exe])
        out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stdout + out.stderr
        return out.stdout
    return run


def test_lds_limit_of_a_kernel_is_set_once_and_to_the_most(run_native):
    """A limit that follows the launches' sizes can be lowered by one thread between another's call and its launch."""
    run_native("lds_opt_in.cpp")
    csrc = os.path.join(os.path.dirname(HERE), "thundergbm_amd", "csrc")
    setters = [f for f in sorted(os.listdir(csrc)) if os.path.isfile(os.path.join(csrc, f)) and
               "hipFuncSetAttribute" in open(os.path.join(csrc, f)).read()]
    assert setters == ["device_api.h"]


def test_sums_lie_in_the_range_of_their_codes(run_native):
    """The filter of the rare features may exclude a run only by a true bound on its candidates' sums: an end that is
    scaled up moves inwards where the whole range is on one side of zero."""
    run_native("rare_range.cpp")


def test_kept_device_blocks(run_native):
    """Reuse, the limit, the order in which blocks go, an allocation that fails, and who pays: requests that follow a
    training call free nothing that it has left, and no thread waits for another one's driver call."""
    run_native("device_pool.cpp")


def test_slices_of_a_scoring_call(run_native):
    """A slice of fewer rows than the kernel of the whole call is for would go to the other one, which is slower there."""
    run_native("score_slices.cpp")


def test_runs_of_features_for_bins(run_native):
    """Bins looked for by runs of features: rows with few values in a run take the other way."""
    run_native("bin_groups.cpp")


def test_query_groups_of_a_workgroup(run_native):
    """Short query groups share a workgroup: one each makes a million workgroups of a million groups of one or two rows."""
    run_native("rank_packs.cpp")


def test_places_of_frequent_features(run_native):
    """Sparse data with close to 2^31 values has more places than an int counts; what counts them must not overflow."""
    run_native("table_places.cpp")


@pytest.fixture(scope="module")
def transfers(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "transfer")
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-std=c++17", "-O1", "-w", "-c",
                           os.path.join(HERE, "native", "transfer.hip"), "-o", exe + ".o"])
    subprocess.check_call(["g++", exe + ".o", "-pthread", "-ldl", "-Wl,--unresolved-symbols=ignore-in-object-files", "-no-pie", "-o", exe])
    return exe


def test_a_download_keeps_off_the_copy_streams(transfers):
    """The copy streams are the process's: a download that has them wait for its own call's kernels holds up every other call's
    copies. And a small upload pays for one round of waits."""
    out = subprocess.run([transfers], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr


def test_transfers_without_threads(transfers):
    """A process may have no thread left to start: the copies are the caller's work then, and nothing ends the program."""
    out = subprocess.run([transfers, "no threads"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr


def test_scans_keep_the_wait_states(tmp_path):
    """Hazards inside inline assembly are its author's: gfx950 needs a wait state between a vector instruction that writes vcc
    and one that takes its carry from there, two before a register is read through DPP, one before a lane is read."""
    asm = str(tmp_path / "wave_scan.s")
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O3", "-std=c++17", "--offload-arch=gfx950", "-w",
                           "--offload-device-only", "-S", os.path.join(HERE, "native", "wave_scan.hip"), "-o", asm])
    age, carries = {}, 0  # wait states since a vector instruction wrote a register
    for line in open(asm):
        op, _, rest = line.split(";")[0].strip().partition(" ")
        if op == "s_nop":
            age = {r: a + 1 + int(rest) for r, a in age.items()}
        if not op.startswith("v_"):
            continue
        args = [a.split()[0] for a in rest.split(",")]
        written = args[:2] if "_co_" in op else args[:1]
        read = args[len(written):]
        far = lambda r: age.get(r, 99)
        if "vcc" in read:
            carries += 1
            assert far("vcc") >= 1, line
        if op.endswith("_dpp"):
            assert far(read[0]) >= 2, line
        if op.startswith("v_readlane"):
            assert far(read[0]) >= 1, line
        age = {r: a + 1 for r, a in age.items()}
        age.update({r: 0 for r in written})
    assert carries == 12


def test_all_threads_reach_a_function_with_barriers():
    """A barrier that some threads of a workgroup never come to is undefined: no device function that has one is called under a
    condition on the thread's number."""
    csrc = os.path.join(os.path.dirname(HERE), "thundergbm_amd", "csrc")
    sources = {f: open(os.path.join(csrc, f)).read() for f in sorted(os.listdir(csrc)) if f.endswith((".hip", ".h"))}
    with_barrier = set()
    for text in sources.values():
        for m in re.finditer(r"^(?:template <[^\n]*>\n)?__device__ [^;{]*?(\w+)\([^;{]*\) \{(?:.*?)^\}", text, re.M | re.S):
            if "__syncthreads" in m.group(0):
                with_barrier.add(m.group(1))
    assert {"tree_init_part", "metric_final", "block_sum"} <= with_barrier
    calls = re.compile(r"if \([^\n]*threadIdx[^\n]*\) (?:%s)[(<]" % "|".join(sorted(with_barrier)))
    assert {f: c for f, text in sources.items() if (c := calls.findall(text))} == {}


def _code_objects(library):
    """The gfx950 code objects in a library's offload bundles."""
    data, at = open(library, "rb").read(), 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entries, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(entries if entries < 16 else 0):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                yield data[at + offset:at + offset + size]
            p += 24 + n
        at += 24


def test_no_64_bit_shift_by_the_last_register(tmp_path):
    """A 64-bit shift whose amount lies in the last vector register that the kernel has been given (they come by eights) has
    shifted by the lane's number now and then: the amount is fetched as a register pair, and the second one is not the kernel's.
    The compiler knows this of gfx90a only."""
    import thundergbm_amd.build as b
    llvm = os.path.join(os.path.dirname(b.HIPCC), "..", "llvm", "bin")
    shifts, found = 0, []
    for i, code in enumerate(_code_objects(b.LIB if os.path.exists(b.LIB) else b.build())):
        path = str(tmp_path / ("%d.co" % i))
        with open(path, "wb") as f:
            f.write(code)
        run = lambda *a: subprocess.run(a, capture_output=True, text=True, check=True).stdout
        count, entry = {}, {}
        for key, value in re.findall(r"\.(name|vgpr_count|agpr_count|wavefront_size):\s+(\S+)", run(llvm + "/llvm-readelf", "--notes", path)):
            entry[key] = value
            if key == "wavefront_size":  # (the last one of a kernel's)
                assert entry.get("agpr_count", "0") == "0", entry
                count[entry["name"]] = (int(entry["vgpr_count"]) + 7) // 8 * 8
        kernel = None
        for line in run(llvm + "/llvm-objdump", "-d", "--no-show-raw-insn", path).splitlines():
            if (m := re.match(r"[0-9a-f]+ <(.*)>:", line)):
                kernel = m.group(1)
            elif (m := re.match(r"\s*v_(?:lshl|lshr|ashr)rev_[bi]64\S*\s+v\[\d+:\d+\], v(\d+),", line)) and kernel in count:
                shifts += 1
                if int(m.group(1)) + 1 >= count[kernel]:
                    found.append((kernel, line.strip()))
    assert shifts > 500 and found == []


def test_sparse_moves_whatever_thread_is_first(run_native, tmp_path):
    """k_sparse_partition stores the rows' new nodes while slower threads still load: a thread past the last row that looks the last
    row's node up may find a child's, which has no entry among the level's."""
    source = open(os.path.join(os.path.dirname(HERE), "thundergbm_amd", "csrc", "sparse_kernels.hip")).read()
    begin = source.index("constexpr int kMoveRows")
    end = source.index("\n}\n", begin) + 3
    kernel = re.sub(r"__shared__ int (\w+)\[(\w+)\];", r"static Shared<\2> \1;", source[begin:end])
    assert "k_sparse_partition" in kernel and kernel.count("static Shared<") == 3
    (tmp_path / "moves.inc").write_text(kernel)
    run_native("sparse_moves.cpp", "-I" + str(tmp_path))


def test_lanes_are_read_where_all_of_them_are_on():
    """read_lane takes a register of another lane as it is. Inside a branch that some lanes do not take, the compiler may work the
    register out for those that do alone."""
    csrc = os.path.join(os.path.dirname(HERE), "thundergbm_amd", "csrc")
    per_thread = {"threadIdx", "lane", "lane_id", "i", "r", "valid", "in", "on", "left", "right", "active"}
    seen = 0
    for name in sorted(os.listdir(csrc)):
        if not name.endswith((".hip", ".h")):
            continue
        blocks = []  # conditions of the blocks that are open
        for number, line in enumerate(open(os.path.join(csrc, name)), 1):
            code = line.split("//")[0]
            if "read_lane" in code and "__forceinline__" not in code:
                seen += 1
                own = re.findall(r"\bif \((.*)", code.split("read_lane")[0])
                names = {w for c in blocks + own for w in re.findall(r"\b[a-zA-Z_]\w*", c)}
                assert not names & per_thread, (name, number, names & per_thread)
            for brace in re.findall(r"[{}]", code):
                if brace == "}":
                    blocks.pop()
                else:
                    found = re.search(r"\bif (?:constexpr )?\((.*)\) \{", code)
                    blocks.append(found.group(1) if found else "")
    assert seen > 20
