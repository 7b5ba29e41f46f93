// How launches of the buffer-load kernel with 128x128 tiles are cut (plan_split in csrc/conv_igemm.inc).  Arguments: product (fwd, dx, dk),
// N H W C O k s, instances; prints groups, share, slices and workgroups.  Compiled for the host only by tests/test_gpu_conv_two_groups.py.
#include "conv_igemm.inc"
#include <cstdlib>
namespace dh { int fail(int c, const char*, ...) { return c; } int fail_hip(hipError_t, const char*) { return 1; } int ensure_init() { return 0; }
int workspace(size_t, void**, hipStream_t) { return 0; } int num_cus() { return 256; } bool profiling(int) { return false; }
int prof_begin(const char*, double, hipStream_t, int) { return -1; } void prof_end(int, hipStream_t) {} bool g_force_generic = false; int g_force_splitk = 0; }

static int same_pad(int n, int k, int s) { int p = n % s == 0 ? k - s : k - n % s; return p > 0 ? p : 0; }

template <int MODE>
static void show(ConvParams& p, bool pair)
{
    plan_launch<MODE>(p, p.phase, 1, TileCfg{128, 128}, pair);
    const int copies = (p.ncols + 127) / 128 * (pair && MODE != MODE_DK ? 2 : 1), k = pair && MODE == MODE_DK ? 2 : 1;
    long workgroups = 0;
    for (int m0 = 0; m0 < p.phase[0].M; m0 += 128)
        workgroups += slices_of(slab_set<MODE>(p, p.phase[0], m0, 128, 0).count() * k, p.per_split) * copies;
    printf("%d %d %d %ld\n", p.groups, p.per_split, p.splitk, workgroups);
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
        show<MODE_FWD>(p, pair);
    }
    else if (what == 'k')   // dk
    {
        f.M = k * k * C; f.K = N * Ho * Wo;
        p.skip = N % BK == 0;
        show<MODE_DK>(p, pair);
    }
    else                    // dx of stride 1: one phase
    {
        f.Hp = H; f.Wp = W; f.q0h = p.pt; f.q0w = p.pl; f.nth = f.ntw = k; f.M = N * H * W; f.K = k * k * O;
        f.fd_HpWp = FastDiv(H * W); f.fd_Wp = FastDiv(W); f.fd_ntw = FastDiv(k);
        p.skip = p.posmajor = 1;
        show<MODE_DX>(p, pair);
    }
    return 0;
}
