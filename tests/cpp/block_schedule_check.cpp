// The autotuned tilings of the block passes: a solve finds what was timed for it
// (its method, its sample type) and nothing that was timed for another.  Needs a GPU.
#include <scan_core.h>

#include <cstdio>
#include <cstdlib>

using namespace parode;

static void expect(bool ok, const char* what)
{
    if (ok) return;
    std::printf("failed: %s\n", what);
    std::exit(1);
}

int main()
{
    ScanOptions opt;
    opt.precision = kMixed;
    // lengths that RK4 with 64 states and ABM with 16 (64 in its map) cut alike
    int log = 8;
    const auto steps = [](int method, int n, int l) {
        return k::block_steps_log(method, n, 2, 2, true, true, 1L << l, 1L << l);
    };
    while (log < 18 && steps(kRK4, 64, log) != steps(kABM, 16, log)) ++log;
    expect(log < 18, "a length with the same steps per block for both");
    const long N = 1L << log;
    ScanCore rk(kRK4, 64, 2, 2, false, false, N, opt), ab(kABM, 16, 2, 2, false, false, N, opt);
    expect(rk.uses_blocks() && ab.uses_blocks(), "block responses");
    const long nb = rk.blocks_of(N);
    expect(nb == ab.blocks_of(N), "the same number of blocks");

    // float samples with FP64 levels: the tilings of the float passes
    expect(ab.autotune(nullptr, N, N, false) == 2, "two passes tuned");
    for (int pass = 1; pass <= 2; ++pass) {
        expect(ab.block_tiling(pass, nb, false) != k::kBlockAuto, "float samples find their tiling");
        expect(ab.block_tiling(pass, nb, true) == k::kBlockAuto, "double samples were not timed");
        expect(rk.block_tiling(pass, nb, false) == k::kBlockAuto, "the other method was not timed");
    }
    expect(rk.autotune(nullptr, N, N, true) == 2, "two passes tuned");
    for (int pass = 1; pass <= 2; ++pass) {
        expect(rk.block_tiling(pass, nb, true) != k::kBlockAuto, "double samples find their tiling");
        expect(ab.block_tiling(pass, nb, true) == k::kBlockAuto, "the other method was not timed");
    }
    ScanCore::clear_schedule();
    expect(ab.block_tiling(1, nb, false) == k::kBlockAuto, "a cleared schedule is the rule's");

    // pass 1 is timed with the squarings that a small map's runs beside its tiles: on
    // four waves they take three times as long as its tiles
    ScanCore sq(kRK4, 48, 6, 6, false, false, 65537, opt);
    expect(sq.autotune(nullptr, 65537, next_pow2(65537), true) == 2, "two passes tuned");
    expect(sq.block_tiling(1, sq.blocks_of(65537), true) != k::kBlockSplit4,
           "squarings on more than four waves");
    ScanCore::clear_schedule();
    std::printf("ok: 2^%d points, %ld blocks\n", log, nb);
    return 0;
}
