// Which partial slices the workgroups of the reduce add up (reduce_slice), worked out on the host
// for calls of one and of several passes, with and without a bias, and for layers without stages.
#include "../../butterfly_amd/csrc/generic.hpp"

#include <cstdio>

using namespace bf;

static int failures = 0;

static void expect(const char *what, int64_t got, int64_t want)
{
    if (got == want) return;
    printf("%s: %lld, expected %lld\n", what, (long long)got, (long long)want);
    ++failures;
}

static ReduceArgs call(int log_n, int nblocks, bool base4, int elem_floats, int nstacks)
{
    ReduceArgs a = {};
    a.sc.log_n = log_n;
    a.sc.nblocks = nblocks;
    a.sc.increasing_stride = 1;
    a.sc.base4 = base4;
    a.sc.per = base4 ? log_n / 2 + log_n % 2 : log_n;
    a.elem_floats = elem_floats;
    a.nstacks = nstacks;
    a.slot = (base4 ? 4 : 2) << log_n;
    return a;
}

static void with_bias(ReduceArgs &a, int64_t width, int64_t tail, int nparts)
{
    a.bias_width = width;
    a.bias_tail = tail;
    a.bias_stride = (width + 3) & ~(int64_t)3;
    a.bias_nparts = nparts;
}

static void expect_bias(const ReduceArgs &a)
{
    for (int s = 0; s < a.nstacks; ++s) {
        const ReduceSlice r = reduce_slice(a, a.nstages, s);
        expect("bias", r.is_bias, 1);
        expect("bias columns", r.count, (s == a.nstacks - 1 ? a.bias_tail : a.bias_width) * a.elem_floats);
        expect("bias start", r.start, s * a.bias_stride * a.elem_floats);
        expect("bias step", r.between, a.nstacks * a.bias_stride * a.elem_floats);
        expect("bias slices", r.nparts, a.bias_nparts);
    }
}

int main()
{
    // layers of size 1: a bias and no stages (the index of a stage has nothing to be divided by)
    for (int ef = 1; ef <= 2; ++ef) {
        ReduceArgs a = call(0, 1, false, ef, 5);
        with_bias(a, 1, 1, 3);
        expect_bias(a);
        a.sc.base4 = 1;
        expect_bias(a);
    }
    // the bias alone
    ReduceArgs alone = call(5, 1, false, 1, 2);
    with_bias(alone, 30, 17, 9);
    expect_bias(alone);
    // three passes of a base-2 call, last one first, of 6, 2 and 4 stages
    for (int ef = 1; ef <= 2; ++ef) {
        ReduceArgs a = call(6, 2, false, ef, 3);
        const int64_t slot = a.slot * ef;
        a.seg[0] = ReduceSegment{6, 12, 7, 0};
        a.seg[1] = ReduceSegment{4, 6, 5, 1024};
        a.seg[2] = ReduceSegment{0, 4, 11, 9216};
        a.nsegs = 3;
        a.nstages = 12;
        with_bias(a, 64, 33, 7);
        expect_bias(a);
        int k = 0;
        for (int i = 0; i < a.nsegs; ++i)
            for (int t = a.seg[i].t0; t < a.seg[i].t1; ++t, ++k)
                for (int s = 0; s < a.nstacks; ++s) {
                    const int nst = a.seg[i].t1 - a.seg[i].t0;
                    const ReduceSlice r = reduce_slice(a, k, s);
                    expect("stage", r.is_bias, 0);
                    expect("factors", r.si.tw_off, (int64_t)t * 32 * 4);
                    expect("floats", r.count, 2 * 64 * ef);
                    expect("start", r.start, a.seg[i].offset + ((int64_t)s * nst + t - a.seg[i].t0) * slot);
                    expect("step", r.between, (int64_t)a.nstacks * nst * slot);
                    expect("slices", r.nparts, a.seg[i].nparts);
                }
    }
    // a base-4 block of five bits: two 4x4 stages, then a 2x2 stage that fills half of its slot
    ReduceArgs b = call(5, 1, true, 1, 1);
    b.seg[0] = ReduceSegment{0, 3, 2, 0};
    b.nsegs = 1;
    b.nstages = 3;
    for (int k = 0; k < 3; ++k) {
        const ReduceSlice r = reduce_slice(b, k, 0);
        expect("base-4 floats", r.count, k < 2 ? 4 * 32 : 2 * 32);
        expect("base-4 start", r.start, (int64_t)k * b.slot);
    }
    if (failures == 0) printf("all slices ok\n");
    return failures != 0;
}
