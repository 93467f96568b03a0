"""The barrier of grid mode (spock.cu_amd/csrc/gridbar.hpp), on the CPU: the protocol that the kernels run,
over a model of the device's memory.

Workgroups are coroutines that a seeded scheduler switches at every access.  A plain store waits in its
workgroup's buffer and becomes visible late: at a random moment, at the workgroup's next release, or only
when nothing else can move (stores to one word keep their order, atomics act at once).  Launches follow each
other on the same words, as the solves of one batch do, with the counts of workgroups given below.  The model
fails a run in which every workgroup waits for good, one in which a workgroup leaves a barrier that
another has not reached, and one in which it does not see what another wrote before the barrier."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r'''
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "gridbar.hpp"

struct Pending { unsigned *at, v; };

struct World {
    std::mt19937 gen;
    int late;  // 0: a store lands at a random moment, 1: at a release or when nothing else can move
    std::vector<unsigned> words = std::vector<unsigned>(spk::GRID_BAR_WORDS, 0);
    std::vector<unsigned> data;      // a word of every workgroup
    std::vector<int> arrived;        // workgroups at barrier k of this launch
    long moved = 0;                  // writes that became visible
    ucontext_t main;
};
static World *W;

struct Wg {
    ucontext_t at;
    std::vector<char> stack = std::vector<char>(64 << 10);
    std::vector<Pending> buf;
    bool done = false, waiting = false;
    long seen = 0;                   // World::moved when it last found nothing
    unsigned id, n;
    int barriers;
    void yield() { swapcontext(&at, &W->main); }
    void land(size_t i) {
        *buf[i].at = buf[i].v;
        buf.erase(buf.begin() + i);
        W->moved++;
    }
    // a pending store with none before it to the same word
    void landOne() {
        std::vector<size_t> free;
        for (size_t i = 0; i < buf.size(); i++) {
            bool first = true;
            for (size_t j = 0; j < i; j++) first = first && buf[j].at != buf[i].at;
            if (first) free.push_back(i);
        }
        land(free[W->gen() % free.size()]);
    }
    void landAll() { while (!buf.empty()) landOne(); }
    void put(unsigned *p, unsigned v) { yield(); buf.push_back({p, v}); }
    unsigned get(unsigned *p) {
        yield();
        for (size_t i = buf.size(); i-- > 0;)
            if (buf[i].at == p) return buf[i].v;
        return *p;
    }
    // the policy
    unsigned add(unsigned w, unsigned k) {
        yield();
        for (size_t i = 0; i < buf.size();)
            if (buf[i].at == &W->words[w]) land(i);
            else i++;
        W->moved++;
        return W->words[w] += k;
    }
    unsigned load(unsigned w) { return get(&W->words[w]); }
    void store(unsigned w, unsigned v) { put(&W->words[w], v); }
    void pause() { waiting = true; seen = W->moved; yield(); waiting = false; }
    void release() { landAll(); }
    void acqRel() { landAll(); }
    void acquire() {}
    void run() {
        unsigned passed = spk::gridPassed(*this, id);
        for (int k = 0; k < barriers; k++) {
            put(&W->data[id], passed * 1000 + id);
            W->arrived[k]++;
            const unsigned before = passed;
            passed = spk::gridPass(*this, id, n, passed);
            if (W->arrived[k] != (int) n) { std::printf("left barrier %d early\n", k); std::exit(2); }
            const unsigned other = W->gen() % n;
            const unsigned got = get(&W->data[other]);  // of this barrier, or already of the next
            if (got != before * 1000 + other && got != passed * 1000 + other) { std::printf("missed a write\n"); std::exit(3); }
        }
        landAll();
        done = true;
        yield();
    }
};
static void entry(unsigned lo, unsigned hi) {
    reinterpret_cast<Wg *>(((unsigned long long) hi << 32) | lo)->run();
}

int main(int argc, char **argv) {
    World world;
    W = &world;
    world.gen.seed(std::atoi(argv[1]));
    world.late = std::atoi(argv[2]);
    if (std::atoi(argv[4])) {  // counters and flags about to overflow
        for (unsigned q = 0; q < spk::GRID_GROUPS; q++) {
            world.words[spk::gridCount(q)] = -spk::GRID_BAR_ROUND;
            world.words[spk::gridFlag(q)] = -2u;
        }
        world.words[spk::GRID_BAR_ROOT] = -spk::GRID_BAR_ROUND;
    }
    for (int a = 5; a < argc; a++) {
        const unsigned n = std::atoi(argv[a]);
        const int barriers = std::atoi(argv[3]);
        world.data.assign(n, 0);
        world.arrived.assign(barriers, 0);
        std::vector<Wg> wgs(n);
        for (unsigned i = 0; i < n; i++) {
            Wg &g = wgs[i];
            g.id = i;
            g.n = n;
            g.barriers = barriers;
            getcontext(&g.at);
            g.at.uc_stack.ss_sp = g.stack.data();
            g.at.uc_stack.ss_size = g.stack.size();
            const unsigned long long p = reinterpret_cast<unsigned long long>(&g);
            makecontext(&g.at, (void (*)()) entry, 2, (unsigned) p, (unsigned) (p >> 32));
        }
        for (;;) {
            std::vector<Wg *> ready, holding;
            bool all = true;
            for (Wg &g : wgs) {
                all = all && g.done;
                if (!g.done && !(g.waiting && g.seen == world.moved)) ready.push_back(&g);
                if (!g.buf.empty()) holding.push_back(&g);
            }
            if (all) break;
            if (ready.empty()) {
                if (holding.empty()) { std::printf("launch %d of %u workgroups never ends\n", a - 5, n); return 1; }
                holding[world.gen() % holding.size()]->landOne();
                continue;
            }
            // a run of steps of some workgroups, so that some are far ahead of others
            for (int s = 0; s < 8; s++) {
                Wg *g = ready[world.gen() % ready.size()];
                for (int t = 1 + world.gen() % 12; t > 0 && !g->done && !(g->waiting && g->seen == world.moved); t--)
                    swapcontext(&world.main, &g->at);
            }
            if (!world.late && !holding.empty() && world.gen() % 4 == 0) {
                Wg *g = holding[world.gen() % holding.size()];
                if (!g->buf.empty()) g->landOne();
            }
        }
        for (Wg &g : wgs) g.landAll();
    }
    std::puts("done");
    return 0;
}
'''


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("gridbar")
    src, exe = d / "model.cpp", d / "model"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-I", os.path.join(ROOT, "spock.cu_amd", "csrc"), "-o", str(exe),
                    str(src)], check=True)
    return str(exe)


def run(model, seed, late, barriers, counts, overflow=0):
    r = subprocess.run([model, str(seed), str(late), str(barriers), str(overflow)] + [str(n) for n in counts],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (seed, late, counts, r.stdout)


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("n", [2, 3, 7, 8, 9, 16, 33, 130])
def test_one_count(model, n, late):
    """Launches of one count: arrivals at a barrier are not lost to stores of the one before."""
    for seed in range(20 if n < 30 else 3):
        run(model, seed, late, 6, [n, n])


@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("counts", [(4, 32), (32, 4, 32), (2, 3, 8, 256, 7, 9), (1, 5, 2, 64), (3, 9, 2, 32, 1024, 6, 12)],
                         ids=lambda c: "-".join(map(str, c)))
def test_counts_change(model, counts, late):
    """Launches of different counts one after the other, from fewer workgroups than there are groups to more: every
    workgroup starts from the same release value."""
    for seed in range(20 if max(counts) < 100 else 1):
        run(model, seed, late, 3, counts)


@pytest.mark.parametrize("late", [0, 1])
def test_overflow(model, late):
    """Counters and release values that pass 2^32."""
    for seed in range(20):
        run(model, seed, late, 5, (9, 4, 16), overflow=1)


DEVICE = r'''
#include <hip/hip_runtime.h>
#include "gridbar.hpp"
__global__ void barrier(unsigned *words, unsigned *out, unsigned passed) {
    spk::GridMem mem{words};
    out[blockIdx.x] = spk::gridPass(mem, blockIdx.x, gridDim.x, passed);
}
'''
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")
def test_write_backs_are_waited_for(tmp_path):
    """The compiled barrier waits behind every write-back of the cache, before the atomic or store that announces what
    was written: the first instruction behind buffer_wbl2 that is not a scalar one is s_waitcnt vmcnt(0)."""
    src, asm = tmp_path / "b.hip", tmp_path / "b.s"
    src.write_text(DEVICE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++20", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "spock.cu_amd", "csrc"), "--cuda-device-only", "-S", "-o",
                    str(asm), str(src)], check=True, capture_output=True, timeout=300)
    lines = [l.split(";")[0].strip() for l in asm.read_text().splitlines()]
    code = [l for l in lines if l and not l.startswith(".")]
    backs = [i for i, l in enumerate(code) if l.startswith("buffer_wbl2")]
    assert len(backs) == 3  # on arrival, at the group's last arrival, at the root's
    for i in backs:
        behind = next(l for l in code[i + 1:] if not l.startswith("s_") or l.startswith("s_waitcnt") and "vmcnt(0)" in l)
        assert behind.startswith("s_waitcnt"), code[i:i + 12]
