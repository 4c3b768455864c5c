/* The plans that moe.c chooses (choose_plan), for a line of
 *   kind D H E k shared norm T
 * on standard input each (kind: 0 MFMA layouts, 1 blocks alone, 2 file):
 *   kernels tchunk ks_gu ks_dn fits alt_fits
 * kernels: 0 grouped GEMMs, 1 decode, 2 blocks, 3 VALU or file; fits: whether
 * the plan fits the fixed scratch; alt_fits: whether any plan that the same
 * call could run with does. */
#include "../ornith-flight_amd/csrc/host/moe.c"

/* the compiled slices (expert_dec.hip, expert_blk.hip, expert_file.hip) */
static int dec_kt(int kt) { return kt == 4 || kt == 8 || kt == 16 || kt == 32; }
int ornk_dec_supported(int kt_gu, int kt_dn) { return dec_kt(kt_gu) && dec_kt(kt_dn); }
static int blk_kt(int kt) { return kt >= 2 && kt % 2 == 0 && kt <= 64; }
int ornk_blk_supported(int kt_gu, int kt_dn) { return blk_kt(kt_gu) && blk_kt(kt_dn); }
int ornk_file_down_cols(void) { return 128; }

static int fits(const ornith_moe_shape *sh, int T, plan_t p, int norm, int amax)
{
    return carve_ws(sh, T, &p, norm, 0, amax, ORNK_SYNC_BYTES).end <= ORNK_SCRATCH_BYTES;
}

int main(void)
{
    int kind, D, H, E, k, shared, norm, T;
    while (scanf("%d%d%d%d%d%d%d%d", &kind, &D, &H, &E, &k, &shared, &norm, &T) == 8) {
        ornith_moe_shape sh = {0};
        sh.d_model = D;
        sh.hidden = H;
        sh.n_experts = E;
        sh.top_k = k;
        sh.has_shared = shared;
        sh.prefill_layout = kind == 0 ? 2 : 0;
        sh.file_layout = kind == 2;
        const plan_t p = choose_plan(&sh, T, kind == 0, kind == 1, norm, 0);
        const int amax = kind == 0 || p.use_blk;
        int alt = fits(&sh, T, p, norm, amax);
        plan_t b;
        if (kind == 0)
            alt |= fits(&sh, T, make_plan(&sh, T, 1, 16), norm, 1) |
                   fits(&sh, T, make_plan(&sh, T, 1, 32), norm, 1);
        if (kind == 1)
            alt |= fits(&sh, T, make_plan(&sh, T, 0, 0), norm, 0) |
                   (make_plan_blk(&sh, T, &b) && fits(&sh, T, b, norm, 1));
        printf("%d %d %d %d %d %d\n", p.use_blk ? 2 : p.use_dec ? 1 : kind == 0 ? 0 : 3, p.tchunk,
               p.ks_gu, p.ks_dn, fits(&sh, T, p, norm, amax), alt);
    }
    return 0;
}
