// The plans of float convolutions over pairs of batches, the one that an operator is created with and the one that it is called with: what a call
// reads is what was packed, in the form and in the bytes that it was packed in.  Host code only, run without a GPU by tests/test_plans.py.
#include "dlp_internal.hpp"

#include <algorithm>
#include <cstdio>
#include <cstring>

using namespace dlp;

namespace {
int failures = 0, checked = 0;

void expect(bool ok, const char *what, const ConvGeom &g)
{
    checked++;
    if (ok)
        return;
    if (failures++ < 20)
        std::printf("%s: %dx%d %d->%d at %dx%d stride %d groups %d, created at batch %d, called at %d\n", what, g.KH, g.KW, g.Cin, g.Cout, g.H, g.W, g.sh, g.groups,
                    g.B_hint, g.B);
}

ConvGeom geometry(int cin, int cout, int k, int s, int groups, int h, int w)
{
    ConvGeom g = ConvGeom();
    g.Cin = cin;
    g.Cout = cout;
    g.KH = g.KW = k;
    g.sh = g.sw = s;
    g.ph = g.pw = k / 2;
    g.dh = g.dw = 1;
    g.H = h;
    g.W = w;
    g.OH = (h + 2 * g.ph - k) / s + 1;
    g.OW = (w + 2 * g.pw - k) / s + 1;
    g.groups = groups;
    g.dtype = DLP_FLOAT;
    return g;
}

template <class F>
void shapes(F f)
{
    const int channels[][2] = {{64, 64}, {128, 128}, {256, 256}, {192, 192}, {384, 384}, {512, 512}, {48, 80}, {320, 96}, {96, 200}, {256, 33}, {768, 512}, {100, 72}};
    const int sizes[][2] = {{7, 7}, {14, 14}, {28, 28}, {35, 35}, {56, 56}, {19, 23}};
    for (const auto &c : channels)
        for (const auto &hw : sizes)
            for (int k : {1, 3, 5})
                for (int s : {1, 2})
                    for (int groups : {1, 2})
                        f(geometry(c[0] * groups, c[1] * groups, k, s, groups, hw[0], hw[1]));
}

// weights packed for the settings' batch, run at another one
void packed()
{
    shapes([](ConvGeom g) {
        for (g.B_hint = 1; g.B_hint <= 72; g.B_hint += g.B_hint < 40 ? 1 : 8) {
            const GemmPackPlan packs = conv_gemm_pack_plan(g, DLP_ACT_RELU);
            for (g.B = 1; g.B <= g.B_hint + 1; g.B += g.B < 40 ? 1 : 8) {
                size_t offset = 0;
                const GemmPlan p = conv_gemm_plan_on_packed(g, DLP_ACT_RELU, packs.p, offset);
                const GemmPlan &form = offset ? packs.floats : packs.p;
                expect(p.split == form.split && offset == (packs.p.split && !p.split ? packs.p.wpack_bytes : 0), "another form than was packed", g);
                expect(offset + p.wpack_bytes <= packs.bytes, "more bytes than were packed", g);
                expect(p.pack_bm == form.BM && p.BM <= form.BM && p.nkt == form.nkt && p.order == form.order, "other tiles than were packed", g);
            }
        }
    });
}

// tiles that a gradient packs in the call, for that call's batch, into a place laid out at create
void tiles()
{
    shapes([](ConvGeom g) {
        for (g.B_hint = 1; g.B_hint <= 72; g.B_hint += g.B_hint < 40 ? 1 : 8) {
            const GemmPackPlan packs = conv_gemm_pack_plan(g, DLP_ACT_IDENTITY);
            const size_t place = packs.p.split ? std::max(packs.p.wpack_bytes, packs.floats.wpack_bytes) : packs.p.wpack_bytes;
            for (g.B = 1; g.B <= g.B_hint + 1; g.B += g.B < 40 ? 1 : 8)
                expect(conv_gemm_plan(g, DLP_ACT_IDENTITY).wpack_bytes <= place, "tiles larger than their place", g);
        }
    });
}

// calls of the small float kernel: no more LDS than a launch gets without asking for it
void lds()
{
    for (int k : {1, 3, 5})
        for (int cin = 16; cin * k * k <= 9000; cin += cin < 200 ? 7 : 1)
            for (int cout : {8, 40, 64, 256, 512})
                for (int size : {1, 7, 10, 14})
                    for (int batch : {1, 2, 4, 9}) {
                        ConvGeom g = geometry(cin, cout, k, 1, 1, size, size);
                        g.B = g.B_hint = batch;
                        for (bool packed : {false, true})
                            expect(!conv_wave_f32_serves(g, packed) || conv_wave_f32_lds_bytes(g) <= 65536, "more than 64 KB of LDS", g);
                    }
}
} // namespace

int main(int argc, char **argv)
{
    if (argc == 2 && !std::strcmp(argv[1], "packed"))
        packed();
    else if (argc == 2 && !std::strcmp(argv[1], "tiles"))
        tiles();
    else if (argc == 2 && !std::strcmp(argv[1], "lds"))
        lds();
    else
        return 2;
    std::printf("%d checked, %d failed\n", checked, failures);
    return failures ? 1 : 0;
}
