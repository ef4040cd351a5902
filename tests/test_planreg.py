"""The registry of plan shapes, compiled for the host: a process that opens
sessions of ever new shapes keeps a bounded number of entries, and an entry
that a session holds, or that was used lately, stays the same one."""
import os
import subprocess

from conftest import ROOT

DRIVER = r"""
#include <cassert>
#include <thread>
#include "xpu_planreg.h"

struct V { int n = 0; };

int
main()
{
    PlanRegistry<V> R;
    std::vector<std::shared_ptr<V>> held;
    for (int i = 0; i < 50; i++)
    {
        held.push_back(R.get("held" + std::to_string(i)));
        held.back()->n = i;
    }
    size_t most = 0;
    for (int i = 0; i < 20000; i++)
    {
        R.get("literal" + std::to_string(i))->n = i;
        R.get("hot")->n++;
        assert(R.get("literal" + std::to_string(i < 500 ? 0 : i - 500))->n == (i < 500 ? 0 : i - 500));
        most = std::max(most, R.size());
    }
    assert(most <= 3 * XPU_PLAN_KEEP + 51);
    assert(R.get("hot")->n == 20000);
    for (int i = 0; i < 50; i++)
        assert(R.get("held" + std::to_string(i)) == held[i] && held[i]->n == i);
    held.clear();
    for (int i = 0; i < 5000; i++)
        R.get("more" + std::to_string(i));
    assert(R.get("held7")->n == 0);         /* let go and not used since */
    std::vector<std::thread> t;
    for (int k = 0; k < 8; k++)
        t.emplace_back([&R, k] {
            for (int i = 0; i < 3000; i++)
            {
                const std::string key = std::to_string(k) + "/" + std::to_string(i);
                auto a = R.get(key);
                assert(R.get(key) == a);
            }
        });
    for (auto &x : t)
        x.join();
    assert(R.size() <= 3 * XPU_PLAN_KEEP + 8);
    return 0;
}
"""


def test_registry(tmp_path):
    src = tmp_path / "planreg.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "planreg"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread",
                    "-I" + os.path.join(ROOT, "pg-strom_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    subprocess.run([str(exe)], check=True, timeout=120)
