// libmusic_hip: context, framework/forcefield upload, Ewald structure factor.
#include <cmath>
#include <cstring>
#include <cstdio>
#include <mutex>

#include "mh_internal.h"

namespace mh {

static thread_local std::string g_err;
void set_error(const std::string &msg) { g_err = msg; }

namespace {
struct Pool {
    struct Block {
        void *p;
        size_t n;
    };
    std::vector<Block> blocks;  // oldest first
    size_t bytes = 0;
    int contexts = 0;
};
std::mutex g_pool_mu;
std::map<int, Pool> g_pools;
std::vector<Pool::Block> g_pins;  // idle pinned blocks
int g_contexts = 0;

void pool_flush(Pool &q) {
    for (auto &b : q.blocks) (void)hipFree(b.p);
    q.blocks.clear();
    q.bytes = 0;
}
}  // namespace

int pool_take(DBuf &b, size_t bytes) {
    b.release();
    int dev = 0;
    MH_HIP(hipGetDevice(&dev));
    {
        std::lock_guard<std::mutex> lk(g_pool_mu);
        Pool &q = g_pools[dev];
        size_t best = q.blocks.size();
        for (size_t i = 0; i < q.blocks.size(); i++) {
            const size_t n = q.blocks[i].n;
            if (n < bytes || n - bytes > bytes / kPoolSlack) continue;
            if (best == q.blocks.size() || n < q.blocks[best].n) best = i;
        }
        if (best < q.blocks.size()) {
            b.p = q.blocks[best].p;
            b.n = q.blocks[best].n;
            q.bytes -= b.n;
            q.blocks.erase(q.blocks.begin() + best);
            return MH_OK;
        }
    }
    return b.alloc(bytes);
}

void pool_give(DBuf &b) {
    if (!b.p) return;
    int dev = 0;
    std::lock_guard<std::mutex> lk(g_pool_mu);
    if (hipGetDevice(&dev) == hipSuccess && g_pools[dev].contexts > 0 && b.n <= kPoolBytes) {
        Pool &q = g_pools[dev];
        q.blocks.push_back({b.p, b.n});
        q.bytes += b.n;
        b.p = nullptr;
        b.n = 0;
        while (q.bytes > kPoolBytes || q.blocks.size() > kPoolBlocks) {
            (void)hipFree(q.blocks.front().p);
            q.bytes -= q.blocks.front().n;
            q.blocks.erase(q.blocks.begin());
        }
        return;
    }
    b.release();
}

static int pin_take(size_t bytes, Pool::Block &b) {
    {
        std::lock_guard<std::mutex> lk(g_pool_mu);
        for (size_t i = 0; i < g_pins.size(); i++)
            if (g_pins[i].n >= bytes) {
                b = g_pins[i];
                g_pins.erase(g_pins.begin() + i);
                return MH_OK;
            }
    }
    b.n = bytes > kPinLeast ? bytes : kPinLeast;
    MH_HIP(hipHostMalloc(&b.p, b.n, hipHostMallocPortable));
    return MH_OK;
}

static void pin_give(const Pool::Block &b) {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    if (b.n <= kPinBytes && g_pins.size() < kPinBlocks && g_contexts > 0) g_pins.push_back(b);
    else (void)hipHostFree(b.p);
}

void pool_ctx(int device, int change) {
    bool first = false;
    {
        std::lock_guard<std::mutex> lk(g_pool_mu);
        Pool &q = g_pools[device];
        q.contexts += change;
        g_contexts += change;
        if (q.contexts == 0) pool_flush(q);
        if (g_contexts == 0) {
            for (auto &b : g_pins) (void)hipHostFree(b.p);
            g_pins.clear();
        }
        first = change > 0 && g_pins.empty();
    }
    Pool::Block b;
    if (first && pin_take(kPinLeast, b) == MH_OK) pin_give(b);
}

int readback(hipStream_t st, const std::vector<Copy> &items) {
    auto up = [](size_t n) { return (n + 63) / 64 * 64; };
    size_t total = 0, o = 0;
    for (auto &i : items) total += up(i.n);
    // staged through pinned memory up to the size that is kept; more goes to
    // the caller's pages (pinning them per call costs more than the waits, and
    // pinned memory of that size may not be there)
    Pool::Block pin{nullptr, 0};
    if (total <= kPinBytes)
        if (int rc = pin_take(total, pin)) return rc;
    hipError_t e = hipSuccess;
    for (auto &i : items) {
        if (i.n && e == hipSuccess)
            e = hipMemcpyAsync(pin.p ? (char *)pin.p + o : i.dst, i.src, i.n, hipMemcpyDeviceToHost, st);
        o += up(i.n);
    }
    const hipError_t w = hipStreamSynchronize(st);
    if (e == hipSuccess) e = w;
    o = 0;
    for (auto &i : items) {
        if (i.n && pin.p && e == hipSuccess) std::memcpy(i.dst, (char *)pin.p + o, i.n);
        o += up(i.n);
    }
    if (pin.p) pin_give(pin);
    if (e != hipSuccess) {
        set_error(std::string("copy to the host: ") + hipGetErrorString(e));
        return MH_EHIP;
    }
    return MH_OK;
}

int DBuf::alloc(size_t bytes) {
    release();
    if (bytes == 0) bytes = 16;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {  // give the kept blocks back and try again
        (void)hipGetLastError();
        {
            int dev = 0;
            std::lock_guard<std::mutex> lk(g_pool_mu);
            if (hipGetDevice(&dev) == hipSuccess) pool_flush(g_pools[dev]);
        }
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();  // reported here, not by the caller's next launch check
        p = nullptr;
        set_error(std::string("hipMalloc(") + std::to_string(bytes) + "): " + hipGetErrorString(e));
        return MH_ENOMEM;
    }
    n = bytes;
    return MH_OK;
}

void DBuf::release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
}

void ctx_retain(mh_ctx *ctx) { ctx->refs++; }

void ctx_release(mh_ctx *ctx) {
    if (--ctx->refs == 0 && ctx->closing) mh_ctx_destroy(ctx);
}

void *ws_get(mh_ctx *ctx, const std::string &name, size_t bytes, int *rc) {
    auto &slot = ctx->ws[name];
    if (!slot) slot.reset(new DBuf());
    if (slot->n < bytes) {
        (void)hipStreamSynchronize(ctx->stream);  // no kernel may still use the old buffer
        size_t grow = bytes + bytes / 8;
        int r = slot->alloc(grow);
        if (r) {
            *rc = r;
            return nullptr;
        }
    }
    *rc = MH_OK;
    return slot->p;
}

// Reference constants (defaults.F90:33-35): truncated pi.
constexpr double kPi = 3.1415927;
constexpr double kTwoPi = 2.0 * kPi;

// ewald_sfactor / ewald_sfSum (ewald.F90:558-681), candidates k = (x, y, z)
// in the reference loop order.  One wave per pair +-k, lanes over the atoms,
// lane sums added by halving.  Bound by the FP64 sincos of every (k, atom);
// one lane per candidate over the serial atom loop left 107 waves on the chip
// for 19^3 candidates (1480 us with 4116 atoms, now 60).  The phase of -k is
// minus that of k exactly, so its sums are the conjugate.  The sums differ from
// the reference's in their last bits; whether a vector is kept must not: where
// the rounding of the two orders could decide it (extinct vectors with a cutoff
// of zero), the atoms are added again in the reference's order.
__global__ void __launch_bounds__(256) k_sfactor(int kmax, int natoms, const double *__restrict__ xyz,
                          const double *__restrict__ q, double ialpha, double ibeta,
                          double igamma, double ikapPiSq, double iVolPi, double locut,
                          uint8_t *__restrict__ keep, double *__restrict__ outs,
                          double *__restrict__ outsi, double *__restrict__ outk) {
    const int side = 2 * kmax + 1;
    const int ncand = side * side * side, lane = threadIdx.x & 63;
    // candidate c and its mirror ncand - 1 - c; k = 0 is its own
    const int c = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (c > ncand / 2) return;
    int x = c / (side * side) - kmax;
    int y = (c / side) % side - kmax;
    int z = c % side - kmax;
    // lane 0 writes c, lane 1 the mirror
    const int w = (lane & 1) ? ncand - 1 - c : c;
    const double sg = (lane & 1) ? -1.0 : 1.0;
    if (x == 0 && y == 0 && z == 0) {
        if (lane == 0) keep[w] = 0;
        return;
    }
    double kalpha = (double)x * ialpha, kbeta = (double)y * ibeta, kgamma = (double)z * igamma;
    double ka2pi = kalpha * kTwoPi, kb2pi = kbeta * kTwoPi, kg2pi = kgamma * kTwoPi;
    double ksqx = kalpha * kalpha, ksqy = kbeta * kbeta, ksqz = kgamma * kgamma;
    double ksq = __dadd_rn(__dadd_rn(ksqx, ksqy), ksqz);
    double factor = __ddiv_rn(__dmul_rn(iVolPi, exp(-ikapPiSq * ksq)), ksq);
    if (!(factor > locut)) {
        if (lane < 2) keep[w] = 0;
        return;
    }
    double sum = 0.0, sumi = 0.0, qa = 0.0;
    auto add = [&](int i) {
        double rdotk = __dadd_rn(__dadd_rn(__dmul_rn(ka2pi, xyz[3 * i]), __dmul_rn(kb2pi, xyz[3 * i + 1])),
                                 __dmul_rn(kg2pi, xyz[3 * i + 2]));
        double sn, cs;
        sincos(rdotk, &sn, &cs);
        sum = __dadd_rn(sum, __dmul_rn(cs, q[i]));
        sumi = __dadd_rn(sumi, __dmul_rn(sn, q[i]));
    };
    for (int i = lane; i < natoms; i += 64) {
        add(i);
        qa += fabs(q[i]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o);
        sumi += __shfl_xor(sumi, o);
        qa += __shfl_xor(qa, o);
    }
    const double f2 = __dmul_rn(factor, factor), least = locut * 1.0e-3;
    double smag = __dmul_rn(f2, __dadd_rn(__dmul_rn(sum, sum), __dmul_rn(sumi, sumi)));
    // n terms of total size qa: two orders of their sum differ by 2 n 2^-53 qa
    // at most (2^-52 n qa; doubled for the products' own rounding)
    const double ds = 4.44e-16 * natoms * qa;
    if (fabs(smag - least) <= f2 * (2.0 * (fabs(sum) + fabs(sumi)) + 2.0 * ds) * ds + 1e-15 * least) {
        sum = sumi = 0.0;
        for (int i = 0; i < natoms; i++) add(i);
        smag = __dmul_rn(f2, __dadd_rn(__dmul_rn(sum, sum), __dmul_rn(sumi, sumi)));
    }
    const bool kept = !(smag <= least);
    if (lane >= 2) return;
    keep[w] = kept ? 1 : 0;
    if (!kept) return;
    outs[w] = sum * factor;
    outsi[w] = sg * sumi * factor;
    outk[3 * w] = sg * ka2pi + 0.0;  // no -0
    outk[3 * w + 1] = sg * kb2pi + 0.0;
    outk[3 * w + 2] = sg * kg2pi + 0.0;
}

}  // namespace mh

using namespace mh;

extern "C" {

const char *mh_last_error(void) { return g_err.c_str(); }
const char *mh_version(void) { return "music_hip 0.1 gfx950"; }

int mh_ctx_create(int device, mh_ctx **out) {
    MH_CHECK(out, MH_EINVAL, "mh_ctx_create: out is NULL");
    int ndev = 0;
    MH_HIP(hipGetDeviceCount(&ndev));
    MH_CHECK(device >= 0 && device < ndev, MH_EINVAL, "mh_ctx_create: no such device");
    MH_HIP(hipSetDevice(device));
    // device address of the map builder's static scratch on this device; a
    // failure is recorded there and only mh_map_build_static refuses to run
    (void)static_scratch_init(device);
    mh_ctx *c = new mh_ctx();
    c->device = device;
    hipError_t e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete c;
        set_error(std::string("hipStreamCreate: ") + hipGetErrorString(e));
        return MH_EHIP;
    }
    pool_ctx(device, 1);
    *out = c;
    return MH_OK;
}

int mh_ctx_destroy(mh_ctx *ctx) {
    if (!ctx) return MH_OK;
    ctx->closing = true;
    if (ctx->refs == 0) {
        (void)hipSetDevice(ctx->device);
        (void)hipStreamSynchronize(ctx->stream);
        ctx->ws.clear();
        (void)hipStreamDestroy(ctx->stream);
        pool_ctx(ctx->device, -1);
        delete ctx;
    }
    return MH_OK;
}

static int check_cell(const double e[3]) {
    for (int i = 0; i < 3; i++)
        if (!(e[i] > 0.0) || !std::isfinite(e[i])) return 0;
    return 1;
}

int mh_framework_upload(mh_ctx *ctx, int natoms, const double *xyz, const int *type,
                        const double *q, const double fund_ell[3], const double full_ell[3]) {
    MH_CHECK(ctx, MH_EINVAL, "mh_framework_upload: ctx is NULL");
    MH_CHECK(natoms >= 0 && (natoms == 0 || (xyz && type)) && fund_ell && full_ell, MH_EINVAL,
             "mh_framework_upload: bad arguments");
    MH_CHECK(check_cell(fund_ell) && check_cell(full_ell), MH_EINVAL,
             "mh_framework_upload: cell edges must be positive");
    MH_HIP(hipSetDevice(ctx->device));
    ctx->natoms = natoms;
    ctx->hxyz.assign(xyz, xyz + 3 * (size_t)natoms);
    ctx->htype.assign(type, type + natoms);
    ctx->hq.assign(natoms, 0.0);
    if (q) ctx->hq.assign(q, q + natoms);
    ctx->max_type = -1;
    for (int i = 0; i < natoms; i++) {
        MH_CHECK(type[i] >= 0 && type[i] < kMaxTypes, MH_EINVAL,
                 "mh_framework_upload: atom type out of range [0,64)");
        if (type[i] > ctx->max_type) ctx->max_type = type[i];
    }
    for (int i = 0; i < 3; i++) {
        ctx->fund_ell[i] = fund_ell[i];
        ctx->full_ell[i] = full_ell[i];
        ctx->eff[i] = fund_ell[i];
        ctx->ang_deg[i] = 90.0;
    }
    ctx->slanted = false;
    ctx->ew.set = false;
    if (natoms == 0) return MH_OK;  // a cell without framework atoms (sorbate-only systems)
    int rc;
    // arrays that are large enough are written again, on the context's stream
    const size_t nd = sizeof(double) * natoms, ni = sizeof(int) * natoms;
    if (ctx->xyz.n < 3 * nd && (rc = ctx->xyz.alloc(3 * nd))) return rc;
    if (ctx->type.n < ni && (rc = ctx->type.alloc(ni))) return rc;
    if (ctx->q.n < nd && (rc = ctx->q.alloc(nd))) return rc;
    MH_HIP(hipMemcpyAsync(ctx->xyz.p, ctx->hxyz.data(), 3 * nd, hipMemcpyHostToDevice, ctx->stream));
    MH_HIP(hipMemcpyAsync(ctx->type.p, ctx->htype.data(), ni, hipMemcpyHostToDevice, ctx->stream));
    MH_HIP(hipMemcpyAsync(ctx->q.p, ctx->hq.data(), nd, hipMemcpyHostToDevice, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    return MH_OK;
}

// matrix_inverse (matrix.F90:195-229): LU with implicit scaling and partial
// pivoting, one back substitution per column (matrixops_ludcmpReal /
// lubksbReal, matrixops.F90:31-161); row-major 3x3
static void lu_inverse3(const double m[9], double inv[9]) {
    double a[3][3], vv[3];
    int indx[3];
    for (int i = 0; i < 9; i++) a[i / 3][i % 3] = m[i];
    for (int i = 0; i < 3; i++) {
        double aamax = 0.0;
        for (int j = 0; j < 3; j++)
            if (std::fabs(a[i][j]) > aamax) aamax = std::fabs(a[i][j]);
        vv[i] = 1.0 / aamax;
    }
    for (int j = 0; j < 3; j++) {
        for (int i = 1; i < j; i++) {
            double sum = a[i][j];
            for (int k = 0; k < i; k++) sum = sum - a[i][k] * a[k][j];
            a[i][j] = sum;
        }
        double aamax = 0.0;
        int imax = j;
        for (int i = j; i < 3; i++) {
            double sum = a[i][j];
            if (j > 0) {
                for (int k = 0; k < j; k++) sum = sum - a[i][k] * a[k][j];
                a[i][j] = sum;
            }
            double dum = vv[i] * std::fabs(sum);
            if (dum >= aamax) {
                imax = i;
                aamax = dum;
            }
        }
        if (j != imax) {
            for (int k = 0; k < 3; k++) std::swap(a[imax][k], a[j][k]);
            vv[imax] = vv[j];
        }
        indx[j] = imax;
        if (j != 2) {
            if (a[j][j] == 0.0) a[j][j] = (double)1.0e-20f;
            double dum = 1.0 / a[j][j];
            for (int i = j + 1; i < 3; i++) a[i][j] = a[i][j] * dum;
        }
    }
    if (a[2][2] == 0.0) a[2][2] = (double)1.0e-20f;
    for (int col = 0; col < 3; col++) {
        double b[3] = {0.0, 0.0, 0.0};
        b[col] = 1.0;
        int ii = -1;
        for (int i = 0; i < 3; i++) {
            const int ll = indx[i];
            double sum = b[ll];
            b[ll] = b[i];
            if (ii >= 0) {
                for (int j = ii; j < i; j++) sum = sum - a[i][j] * b[j];
            } else if (sum != 0.0) {
                ii = i;
            }
            b[i] = sum;
        }
        for (int i = 2; i >= 0; i--) {
            double sum = b[i];
            for (int j = i + 1; j < 3; j++) sum = sum - a[i][j] * b[j];
            b[i] = sum / a[i][i];
        }
        for (int i = 0; i < 3; i++) inv[3 * i + col] = b[i];
    }
}

int mh_framework_set_cell(mh_ctx *ctx, const double angles_deg[3], const double eff[3]) {
    MH_CHECK(ctx && angles_deg && eff, MH_EINVAL, "mh_framework_set_cell: bad arguments");
    MH_CHECK(check_cell(eff), MH_EINVAL, "mh_framework_set_cell: effective box edges must be positive");
    for (int i = 0; i < 3; i++)
        MH_CHECK(angles_deg[i] > 0.0 && angles_deg[i] < 180.0, MH_EINVAL,
                 "mh_framework_set_cell: angles must lie in (0, 180) degrees");
    // fundcell_init (fundcell.F90:60-112): orthorhombic within 0.001 degree
    const double err = std::fabs(angles_deg[0] - 90.0) + std::fabs(angles_deg[1] - 90.0) +
                       std::fabs(angles_deg[2] - 90.0);
    for (int i = 0; i < 3; i++) {
        ctx->eff[i] = eff[i];
        ctx->ang_deg[i] = angles_deg[i];
    }
    ctx->slanted = err > 0.001;
    if (!ctx->slanted) return MH_OK;
    // fundcell_initxform (fundcell.F90:378-412): the angles in default real,
    // single-precision cosines
    const double degtorad = 3.1415927 / 180.0;
    const float alpha = (float)(angles_deg[0] * degtorad), beta = (float)(angles_deg[1] * degtorad),
                gamma = (float)(angles_deg[2] * degtorad);
    const float cg = cosf(gamma), cb = cosf(beta), ca = cosf(alpha);
    double U[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    U[0] = 1.0;
    U[1] = (double)cg;
    U[2] = (double)cb;
    const float cg2 = cg * cg;
    U[4] = std::sqrt(1.0 - (double)cg2);
    const float num = ca - cg * cb;
    U[5] = (double)num / U[4];
    U[8] = std::sqrt(1.0 - U[2] * U[2] - U[5] * U[5]);
    MH_CHECK(std::isfinite(U[5]) && std::isfinite(U[8]) && U[8] > 0.0, MH_EINVAL,
             "mh_framework_set_cell: the angles do not form a cell");
    double S[9];
    lu_inverse3(U, S);
    for (int i = 0; i < 9; i++) {
        ctx->U[i] = U[i];
        ctx->S[i] = S[i];
    }
    // slanted atom coordinates S a (fundcell_slant, matrix_m_mult_v order)
    if (ctx->natoms > 0) {
        std::vector<double> xs(3 * (size_t)ctx->natoms);
        for (int a = 0; a < ctx->natoms; a++)
            for (int r = 0; r < 3; r++) {
                double s = 0.0;
                for (int c = 0; c < 3; c++) s = s + S[3 * r + c] * ctx->hxyz[3 * a + c];
                xs[3 * a + r] = s;
            }
        int rc;
        if ((rc = ctx->xyz_s.alloc(sizeof(double) * xs.size()))) return rc;
        MH_HIP(hipSetDevice(ctx->device));
        MH_HIP(hipMemcpy(ctx->xyz_s.p, xs.data(), sizeof(double) * xs.size(), hipMemcpyHostToDevice));
    }
    return MH_OK;
}

int mh_ff_set_lj(mh_ctx *ctx, int ntypes, const double *A, const double *B,
                 const double *hicut2, const double *locut2, const uint8_t *on) {
    MH_CHECK(ctx && A && B && hicut2 && locut2, MH_EINVAL, "mh_ff_set_lj: bad arguments");
    MH_CHECK(ntypes > 0 && ntypes <= kMaxTypes, MH_EINVAL, "mh_ff_set_lj: ntypes out of range");
    LJTable &t = ctx->lj;
    t.ntypes = ntypes;
    for (int i = 0; i < ntypes; i++) {
        t.A[i] = A[i];
        t.B[i] = B[i];
        t.hicut2[i] = hicut2[i];
        t.locut2[i] = locut2[i];
        t.on[i] = on ? on[i] : 1;
        if (!t.on[i]) t.A[i] = t.B[i] = t.hicut2[i] = t.locut2[i] = 0.0;
    }
    ctx->lj_set = true;
    return MH_OK;
}

int mh_ff_set_buck(mh_ctx *ctx, int ntypes, const double *A, const double *rho,
                   const double *C, const double *D, const double *hicut2,
                   const double *locut2) {
    MH_CHECK(ctx && A && rho && C && D && hicut2 && locut2, MH_EINVAL,
             "mh_ff_set_buck: bad arguments");
    MH_CHECK(ntypes > 0 && ntypes <= kMaxTypes, MH_EINVAL, "mh_ff_set_buck: ntypes out of range");
    BuckTable &t = ctx->buck;
    t.ntypes = ntypes;
    for (int i = 0; i < ntypes; i++) {
        MH_CHECK(rho[i] > 0.0 || A[i] == 0.0, MH_EINVAL, "mh_ff_set_buck: rho must be > 0");
        t.A[i] = A[i];
        t.rho[i] = rho[i] > 0.0 ? rho[i] : 1.0;
        t.C[i] = C[i];
        t.D[i] = D[i];
        t.hicut2[i] = hicut2[i];
        t.locut2[i] = locut2[i];
    }
    ctx->buck_set = true;
    return MH_OK;
}

int mh_ewald_set(mh_ctx *ctx, double kappa_param, int kmax, double locut, int sign_mode, int *nk_out) {
    MH_CHECK(ctx, MH_EINVAL, "mh_ewald_set: ctx is NULL");
    MH_CHECK(sign_mode == MH_EWALD_PARITY || sign_mode == MH_EWALD_PHYSICS, MH_EINVAL,
             "mh_ewald_set: sign_mode must be MH_EWALD_PARITY or MH_EWALD_PHYSICS");
    MH_CHECK(ctx->natoms > 0, MH_ESTATE, "mh_ewald_set: upload the framework first");
    MH_CHECK(kmax >= 1 && kmax <= 40, MH_EINVAL, "mh_ewald_set: kmax out of range [1,40]");
    MH_CHECK(kappa_param > 0.0, MH_EINVAL, "mh_ewald_set: kappa must be > 0");
    MH_HIP(hipSetDevice(ctx->device));
    Ewald &ew = ctx->ew;
    const double *ell = ctx->full_ell;
    double mn = ell[0] < ell[1] ? ell[0] : ell[1];
    mn = mn < ell[2] ? mn : ell[2];
    ew.kappa_param = kappa_param;
    ew.kappa = kappa_param / mn;
    ew.kmax = kmax;
    ew.locut = locut;
    ew.sign_mode = sign_mode;
    double ialpha = 1.0 / ell[0], ibeta = 1.0 / ell[1], igamma = 1.0 / ell[2];
    double ikap = 1.0 / ew.kappa;
    double pk = kPi * ikap;
    double ikapPiSq = pk * pk;
    double iVolPi = ialpha * ibeta * igamma / kPi;
    const int side = 2 * kmax + 1;
    const int ncand = side * side * side;
    // candidates: s, si, k, keep in one block, one copy back
    PoolBuf cand;
    int rc;
    const size_t cb = sizeof(double) * 5 * (size_t)ncand + ncand;
    if ((rc = cand.take(cb))) return rc;
    double *cs = cand.as<double>(), *csi = cs + ncand, *ck = csi + ncand;
    uint8_t *keep = reinterpret_cast<uint8_t *>(ck + 3 * (size_t)ncand);
    hipLaunchKernelGGL(k_sfactor, dim3((ncand / 2 + 4) / 4), dim3(256), 0, ctx->stream, kmax,
                       ctx->natoms, ctx->xyz.as<double>(), ctx->q.as<double>(), ialpha, ibeta,
                       igamma, ikapPiSq, iVolPi, locut, keep, cs, csi, ck);
    MH_HIP(hipGetLastError());
    std::vector<double> hc(5 * (size_t)ncand + (ncand + 7) / 8);
    MH_HIP(hipMemcpyAsync(hc.data(), cs, cb, hipMemcpyDeviceToHost, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    cand.idle = true;
    const double *hs = hc.data(), *hsi = hs + ncand, *hk = hsi + ncand;
    const uint8_t *hkeep = reinterpret_cast<const uint8_t *>(hk + 3 * (size_t)ncand);
    // ordered compaction of the accepted vectors (reference order x,y,z)
    ew.hk.clear();
    ew.hs.clear();
    ew.hsi.clear();
    std::vector<double> grid(2 * (size_t)ncand, 0.0);  // complex c = s + i si per candidate
    for (int c = 0; c < ncand; c++) {
        if (!hkeep[c]) continue;
        ew.hs.push_back(hs[c]);
        ew.hsi.push_back(hsi[c]);
        ew.hk.push_back(hk[3 * c]);
        ew.hk.push_back(hk[3 * c + 1]);
        ew.hk.push_back(hk[3 * c + 2]);
        grid[2 * c] = hs[c];
        grid[2 * c + 1] = hsi[c];
    }
    ew.nk = (int)ew.hs.size();
    MH_CHECK(ew.nk <= 50000, MH_ECAPACITY,
             "mh_ewald_set: more than nkmax = 50000 k vectors (ewald.F90:134)");
    const size_t gb = sizeof(double) * 2 * (size_t)ncand;
    if (ew.ccoef.n < gb && (rc = ew.ccoef.alloc(gb))) return rc;
    MH_HIP(hipMemcpyAsync(ew.ccoef.p, grid.data(), gb, hipMemcpyHostToDevice, ctx->stream));
    MH_HIP(hipStreamSynchronize(ctx->stream));
    ew.set = true;
    if (nk_out) *nk_out = ew.nk;
    return MH_OK;
}

int mh_ctx_set_timing(mh_ctx *ctx, int on) {
    MH_CHECK(ctx, MH_EINVAL, "mh_ctx_set_timing: ctx is NULL");
    ctx->timing = on != 0;
    ctx->ktimes.clear();
    return MH_OK;
}

int mh_ctx_get_timing(mh_ctx *ctx, char *buf, int len) {
    MH_CHECK(ctx && buf && len > 0, MH_EINVAL, "mh_ctx_get_timing: bad arguments");
    std::string js = "{";
    bool first = true;
    for (auto &kv : ctx->ktimes) {
        char tmp[256];
        snprintf(tmp, sizeof tmp, "%s\"%s\": [%.6f, %lld]", first ? "" : ", ", kv.first.c_str(),
                 kv.second.first, kv.second.second);
        js += tmp;
        first = false;
    }
    js += "}";
    MH_CHECK((int)js.size() < len, MH_ECAPACITY, "mh_ctx_get_timing: buffer too small");
    memcpy(buf, js.c_str(), js.size() + 1);
    return MH_OK;
}

int mh_ewald_get(mh_ctx *ctx, double *k, double *s, double *si, double *kappa) {
    MH_CHECK(ctx && ctx->ew.set, MH_ESTATE, "mh_ewald_get: call mh_ewald_set first");
    const Ewald &ew = ctx->ew;
    if (k) std::memcpy(k, ew.hk.data(), sizeof(double) * 3 * ew.nk);
    if (s) std::memcpy(s, ew.hs.data(), sizeof(double) * ew.nk);
    if (si) std::memcpy(si, ew.hsi.data(), sizeof(double) * ew.nk);
    if (kappa) *kappa = ew.kappa;
    return MH_OK;
}

}  // extern "C"
