// How launches of the buffer-load kernel with 128x128 tiles are cut (plan_split in csrc/conv_igemm.inc).  Arguments: product (fwd, dx, dk),
// N H W C O k s, instances; prints groups (0: the launch takes narrower tiles), share, slices and workgroups.  Compiled for the host only by tests/test_gpu_conv_two_groups.py.
#include "conv_igemm.inc"
#include <cstdlib>
namespace dh { int fail(int c, const char*, ...) { return c; } int fail_hip(hipError_t, const char*) { return 1; } int ensure_init() { return 0; }
int workspace(size_t, void**, hipStream_t) { return 0; } int num_cus() { return 256; } bool profiling(int) { return false; }
int prof_begin(const char*, double, hipStream_t, int) { return -1; } void prof_end(int, hipStream_t) {} bool g_force_generic = false; int g_force_splitk = 0; }

static int same_pad(int n, int k, int s) { int p = n % s == 0 ? k - s : k - n % s; return p > 0 ? p : 0; }

template <int MODE>
static void show(ConvParams& p, const Phase* phase, int n, bool pair)
{
    plan_launch<MODE>(p, phase, n, TileCfg{128, 128}, pair);
    const int copies = (p.ncols + 127) / 128 * (pair && MODE != MODE_DK ? 2 : 1), k = pair && MODE == MODE_DK ? 2 : 1;
    long workgroups = 0, slabs = 0, tiles = 0;
    for (int z = 0; z < n; ++z)
        for (int m0 = 0; m0 < phase[z].M; m0 += 128, tiles += copies)
        {
            workgroups += slices_of(slab_set<MODE>(p, phase[z], m0, 128, z).count() * k, p.per_split) * copies;
            slabs += (phase[z].K + BK - 1) / BK * copies;
        }
    const bool square = MODE == MODE_DK || narrower_if_split(TileCfg{128, 128}, p.ncols, tiles, slabs, [&] { return planned_in_two_groups<MODE>(p, phase, n, pair, tiles); }).bn == 128;
    printf("%d %d %d %ld\n", square ? p.groups : 0, p.per_split, p.splitk, workgroups);
}

int main(int argc, char** argv)
{
    if (argc != 10) return 2;
    const int N = atoi(argv[2]), H = atoi(argv[3]), W = atoi(argv[4]), C = atoi(argv[5]), O = atoi(argv[6]), k = atoi(argv[7]), s = atoi(argv[8]);
    const bool pair = atoi(argv[9]) == 2;
    const int Ho = (H + s - 1) / s, Wo = (W + s - 1) / s;
    ConvParams p{};
    fill_common(p, N, H, W, C, Ho, Wo, O, k, k, s, s, same_pad(H, k, s) / 2, same_pad(W, k, s) / 2);
    Phase& f = p.phase[0];
    const char what = argv[1][1];
    p.ncols = what == 'x' ? C : O;
    if (what == 'w')        // fwd
    {
        f.M = N * Ho * Wo; f.K = k * k * C;
        p.skip = p.posmajor = 1;
        show<MODE_FWD>(p, p.phase, 1, pair);
    }
    else if (what == 'k')   // dk
    {
        f.M = k * k * C; f.K = N * Ho * Wo;
        p.skip = N % BK == 0;
        show<MODE_DK>(p, p.phase, 1, pair);
    }
    else                    // dx: the phases in the order of csrc/conv_dx.hip
    {
        Phase all[MAX_PHASES];
        int n = 0;
        if (s * s > MAX_PHASES) return 2;
        for (int q = 0; q < s * s; ++q)
        {
            Phase g{};
            g.ph = q / s; g.pw = q % s;
            g.Hp = (H - g.ph + s - 1) / s; g.Wp = (W - g.pw + s - 1) / s;
            g.rh = (g.ph + p.pt) % s; g.rw = (g.pw + p.pl) % s;
            g.q0h = (g.ph + p.pt) / s; g.q0w = (g.pw + p.pl) / s;
            g.nth = g.rh < k ? (k - g.rh + s - 1) / s : 0; g.ntw = g.rw < k ? (k - g.rw + s - 1) / s : 0;
            g.M = N * g.Hp * g.Wp; g.K = g.nth * g.ntw * O;
            g.fd_HpWp = FastDiv(g.Hp * g.Wp); g.fd_Wp = FastDiv(g.Wp); g.fd_ntw = FastDiv(g.ntw > 0 ? g.ntw : 1);
            all[n++] = g;
        }
        std::sort(all, all + n, [](const Phase& a, const Phase& b) { return a.K > b.K; });
        std::reverse(all + (n + 1) / 2, all + n);
        p.skip = p.posmajor = 1;
        show<MODE_DX>(p, all, n, pair);
    }
    return 0;
}
