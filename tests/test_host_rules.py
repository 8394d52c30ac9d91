"""Host rules of the library that need no device, run in a small C++ program
over the library's own headers."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "neighbourlists.jl_amd", "csrc")


def run_file(tmp_path, src):
    """Compile and run a C++ program over the library's headers; returns what it printed."""
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I",
                    "/opt/rocm/include", str(src), "-o", str(exe), "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib",
                    "-lamdhip64", "-lpthread"], check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout


def run_cpp(tmp_path, body, includes=("nlhip_internal.h",)):
    """The same for main() { body }."""
    src = tmp_path / "t.cpp"
    src.write_text("".join(f'#include "{i}"\n' for i in includes) +
                   "#include <cstdio>\nusing namespace nlh;\nint main()\n{\n" + body + "\nreturn 0;\n}\n")
    return run_file(tmp_path, src)


def _overflows(tmp_path, counts):
    """Builds whose largest count does not fit the rows that the builds before
    them suggest, and the last rows."""
    out = run_cpp(tmp_path, "SlotHistory s; int over = 0;\nfor (int m : {" + ", ".join(map(str, counts)) +
                  "}) { if (s.knows(1000, 96) && m > s.rows()) ++over; s.note(1000, 96, m); }\n"
                  'printf("%d %d %d", over, (int)s.knows(1000, 96), s.rows());')
    return tuple(int(x) for x in out.split())


@pytest.mark.parametrize("counts,over", [
    # largest counts of fcc crystals of 13,500 and 108,000 atoms heating up, at
    # cutoffs of 5.0 and 5.4, and of random gases, build after build
    ([42, 42, 44, 46, 47, 47, 48, 49, 50, 49, 50, 50, 52, 52, 52, 51, 52], 0),
    ([42, 42, 45, 46, 48, 48, 49, 49, 50, 50, 51, 51, 52, 52, 53], 0),
    ([54, 54, 54, 54, 55, 57, 57, 59, 59, 59, 61, 61, 62, 62, 64, 63, 64, 65], 0),
    ([44, 51, 48, 47, 48, 47, 49, 49, 50, 51, 48], 0),
    ([52, 50, 52, 51, 50, 53, 50, 52, 55, 52, 50, 51, 53, 58, 54], 0),
    ([46, 47, 48, 49, 50, 51], 0),
    # a jump that nothing announced
    ([42, 42, 42, 100, 101], 1)])
def test_slot_rows_leave_room_for_moving_atoms(tmp_path, counts, over):
    got, knows, rows = _overflows(tmp_path, counts)
    assert got == over and knows and rows >= max(counts)


def test_slot_rows_of_static_atoms(tmp_path):
    """Counts that never rise: rows of the next multiple of 16, from the third
    build on; another size starts over."""
    for m in (1, 15, 16, 17, 42, 48):
        assert _overflows(tmp_path, [m, m, m]) == (0, 1, (m + 15) // 16 * 16)
    assert _overflows(tmp_path, [42])[1] == 0
    out = run_cpp(tmp_path, "SlotHistory s; s.note(10, 32, 5); s.note(10, 32, 9); s.note(11, 32, 40); s.note(11, 32, 40);\n"
                  'printf("%d %d %d", (int)s.knows(10, 32), (int)s.knows(11, 32), s.rows());')
    assert out == "0 1 48"


def test_copiers_in_use_at_once_are_kept(tmp_path):
    """Copies that overlap find the copiers of the last ones that did, each
    device its own, and no more than the limit stay."""
    out = run_cpp(tmp_path, """
HostCopierPool p;
p.handle_made();
auto a = p.borrow(0), b = p.borrow(0);
HostCopier *pa = a.get(), *pb = b.get();
bool ended = p.give_back(std::move(a)) || p.give_back(std::move(b));
for (int turn = 0; turn < 3; ++turn) {
    auto c = p.borrow(0), d = p.borrow(0);
    bool same = (c.get() == pa || c.get() == pb) && (d.get() == pa || d.get() == pb) && c != d;
    printf("%d ", (int)same);
    ended = ended || p.give_back(std::move(c)) || p.give_back(std::move(d));
}
auto other = p.borrow(1);
printf("%d %d ", (int)ended, (int)(other.get() != pa && other.get() != pb));
std::vector<std::unique_ptr<HostCopier>> many;
many.push_back(std::move(other));
for (int k = 0; k < 9; ++k) many.push_back(p.borrow(0));
int gone = 0;
for (auto &m : many) gone += p.give_back(std::move(m)) != nullptr;
p.handle_gone();
printf("%d", gone);
""", includes=("host_copy.h",))
    assert out == f"1 1 1 0 1 {10 - 4}"


def test_filter_bounds(tmp_path):
    """The 32-bit distance filter of both pair searches, emulated: over cells of
    one to nine cutoffs, sheared, in units from 1e-10 to 1e6, with windings and
    atoms far outside open cells, no pair beyond its error bound has another
    sign than the 64-bit test, and no error near the cutoff exceeds the bound."""
    out = run_file(tmp_path, os.path.join(os.path.dirname(os.path.abspath(__file__)), "filter_bounds_check.cpp"))
    for line in out.splitlines():
        pairs, wrong, worst, _ = line.split()
        assert int(pairs) > 100000 and int(wrong) == 0 and float(worst) < 1.0, line
    assert len(out.splitlines()) == 2


def test_copies_at_once_take_fewer_threads(tmp_path):
    """Two copies have all their threads, three and more half of them each."""
    out = run_cpp(tmp_path, """
HostCopierPool p;
std::vector<std::unique_ptr<HostCopier>> c;
for (int k = 0; k < 4; ++k) {
    c.push_back(p.borrow(0));
    printf("%d ", p.threads());
}
for (auto &x : c) {
    p.give_back(std::move(x));
    printf("%d ", p.threads());
}
""", includes=("host_copy.h",))
    assert out.split() == ["4", "4", "2", "2", "2", "4", "4", "4"]
