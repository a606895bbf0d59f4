// The products of a wide map's block responses stay inside their buffers: for
// each shape and every number of blocks up to the capacity that the buffers are
// sized for, the operands and results of the table, tree and top products are
// replayed as index ranges (nothing is read or written).  No GPU needed.
#include <blocks.h>

#include <cstdio>
#include <cstdlib>

using namespace parode::k;

namespace {

// Four buffers at made-up, far-apart addresses, each [base, base + size) in doubles.
struct Span {
    const char* name;
    double* base;
    size_t size;
};
Span spans[4];
const char* what = "";
int n_, method_, lb_;
long nb_, cap_;

double* place(int k) { return reinterpret_cast<double*>((uintptr_t)(k + 1) << 40); }

// [p + lo, p + hi) of `bytes` each lies in one buffer
void in_one(const char* operand, const void* p, long lo, long hi, size_t bytes = 8)
{
    if (hi <= lo) return;
    const uintptr_t a = (uintptr_t)p + lo * (long)bytes, b = (uintptr_t)p + hi * (long)bytes;
    for (const Span& s : spans)
        if (a >= (uintptr_t)s.base && b <= (uintptr_t)(s.base + s.size)) return;
    std::printf("method %d n %d lb %d blocks %ld of %ld: %s, %s out of its buffer", method_, n_, lb_,
                nb_, cap_, what, operand);
    for (const Span& s : spans)
        if (a >= (uintptr_t)s.base && a < (uintptr_t)(s.base + (1L << 36)))
            std::printf(" (%s: ends %ld values past it)", s.name,
                        (long)((b - (uintptr_t)(s.base + s.size)) / 8));
    std::printf("\n");
    std::exit(1);
}

void check(const GemmOp& o)
{
    if (o.r <= 0 || o.c <= 0) return;
    const GemmLd& d = o.ld;
    const long r1 = o.r - 1;
    const int k1 = d.X2 ? d.k1 : o.kk;
    in_one("X", o.X, 0, r1 * d.ldx + k1);
    if (d.X2) in_one("X2", d.X2, 0, r1 * d.ldx2 + o.kk - d.k1);
    in_one("Y", o.Y, 0, (long)(o.kk - 1) * d.ldy + o.c);
    if (d.add) in_one("addend", d.add, 0, (r1 - d.shift) * d.lda + o.c);
    if (d.cp) in_one("copy", d.cp, 0, r1 * d.ldz + o.c);
    if (d.zp) {
        const long last = (o.c - 1) / d.zp * d.zs;   // (zs may be negative)
        in_one("result", o.Z, last < 0 ? last : 0, (last > 0 ? last : 0) + r1 * d.ldz + d.zp);
    } else {
        in_one("result", o.Z, 0, r1 * d.ldz + o.c);
    }
}

struct Sink : BlockSink {
    void gemm(int, const GemmOp& o) override
    {
        what = "tables";
        // (the direct terms' float inputs aside, every operand is a buffer of the solve)
        check(o);
    }
    void elem(int, const BlkElem&) override {}
    void seq(int, const SeqOp& o) override
    {
        what = "float products";
        in_one("result", o.Z, 0, (long)o.r * o.c, 4);
    }
};

void check_tree(const BlockShape& s, const BlockBufs& b, long nb)
{
    nb_ = nb;
    const int up = block_tree_up_levels(s, nb);
    what = "up";
    for (int k = 0; k < up; ++k) check(block_tree_up(s, b, nb, k));
    what = "top";
    for (int i = 0; i < block_tree_top_steps(s, nb); ++i) check(block_tree_top(s, b, nb, i));
    what = "down";
    for (int j = 0; j < block_tree_down_steps(s, nb); ++j)
        for (const GemmOp& o : block_tree_down(s, b, nb, j)) check(o);
    // pass 1 writes the blocks' responses, pass 2 reads their start states
    what = "passes";
    in_one("responses", b.Z, 0, nb * s.na);
    in_one("start states", b.E, 0, nb * s.na);
}

}  // namespace

int main()
{
    const struct { int method, n, m, p; } shapes[] = {
        {0, 65, 1, 1}, {0, 96, 40, 70}, {0, 128, 16, 16}, {0, 200, 25, 7}, {0, 8, 40, 3}, {0, 256, 2, 2},
        {0, 257, 2, 2}, {0, 1024, 3, 3}, {1, 17, 3, 2}, {1, 64, 8, 8}, {1, 65, 1, 1}, {1, 128, 16, 16},
        {1, 129, 5, 9}, {1, 203, 25, 25}, {1, 256, 32, 32}, {1, 1024, 2, 3}};
    long trees = 0;
    for (const auto& q : shapes)
        for (int lb : {3, 5, 8})
            for (int mirror = 0; mirror < 2; ++mirror)
                for (int log = 1; log <= 11; ++log) {
                    const long cap = 1L << log;
                    const BlockShape s = block_shape(q.method, q.n, q.m, q.p, true, true, mirror != 0, lb,
                                                     lb + log + 1);
                    if (!s.wide) continue;
                    method_ = q.method;
                    n_ = q.n;
                    lb_ = lb;
                    cap_ = nb_ = cap;
                    const size_t na2 = (size_t)s.na * s.na;
                    spans[0] = Span{"powers", place(0), na2 * s.slots()};
                    spans[1] = Span{"tables", place(1), block_table_values(s)};
                    spans[2] = Span{"states", place(2), block_state_values(s, cap)};
                    spans[3] = Span{"scratch", place(3), block_scratch_values(s)};
                    const BlockBufs b = block_carve(s, place(0), place(1), place(2), cap, place(3));
                    Sink sink;
                    // (as ScanCore does, for the batch's blocks and for a whole plan)
                    block_emit(s, b, 1e-3, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                               lb + block_tree_up_levels(s, cap), sink);
                    for (long nb = 1; nb <= cap; nb += (cap > 64 && nb > 20 && nb < cap - 20) ? 7 : 1) {
                        check_tree(s, b, nb);
                        ++trees;
                    }
                }
    // maps of one work-group: the blocks' states and one more, then the groups' and one more
    for (int n : {1, 16, 48, 64})
        for (int log = 1; log <= 17; ++log) {
            const long cap = 1L << log;
            const BlockShape s = block_shape(0, n, 1, 1, true, true, false, 5, 5 + log + 1);
            method_ = 0;
            n_ = n;
            lb_ = 5;
            cap_ = cap;
            spans[2] = Span{"states", place(2), block_state_values(s, cap)};
            const BlockBufs b = block_carve(s, place(0), place(1), place(2), cap, nullptr);
            for (long nb = 1; nb <= cap; nb += (nb > 600 && nb < cap - 40) ? 31 : 1) {
                nb_ = nb;
                what = "scan";
                in_one("states", b.Z, 0, (nb + 1) * n);
                in_one("groups", b.Z2, 0, (block_groups(nb) + 1) * n);
            }
        }
    std::printf("%ld trees inside their buffers\n", trees);
    return 0;
}
