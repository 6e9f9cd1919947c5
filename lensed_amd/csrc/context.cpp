// The likelihood context: program build, device buffers and the launch
// chains of the plain and batched paths.
//
// Host-side setup follows src/lensed.c: parameter bookkeeping (106-271),
// data (406-511), quadrature (612-642), program build (648-776), buffers and
// work sizes (802-1112).  The per-evaluation chain follows src/nested.c:17-131
// with the chi^2 sum moved onto the device: 8 bytes per candidate come back.
#include "context.h"

#include <algorithm>
#include <random>
#include <chrono>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <set>
#include <sstream>
#include <sys/stat.h>
#include <unistd.h>

#include "emulator.h"
#include "psf.h"
#include "rtc.h"
#include "scratch.h"
#include "tune.h"

namespace lsd {

int emu_upload(const float* weights, void** wf, void** wp);
int emu_launch_tables(hipStream_t st, const lensed_desc* d_desc, int nsys, int n_nodes, int n_intervals, int n_cands,
                      const float* params, const void* wf, const void* wp, void* nodes, void* tables, int* flags,
                      const int* cells);
int emu_certify(const void* wf, const void* wp, float eps, int* cells, double* max_err);

static thread_local std::string g_error;
void set_error(const std::string& msg) { g_error = msg; }

#define LSD_HIP(x)                                                                       \
    do {                                                                                 \
        hipError_t e_ = (x);                                                             \
        if (e_ != hipSuccess) {                                                          \
            set_error(std::string(#x) + ": " + hipGetErrorString(e_));                   \
            return -1;                                                                   \
        }                                                                                \
    } while (0)

std::string model_source(const std::vector<std::vector<ModelObject>>& models, std::string* err) {
    std::string kd = kernel_dir(), prelude, table, desc;
    if (!read_text(kd + "/prelude.h", &prelude) || !read_text(kd + "/epl_table.h", &table) ||
        !read_text(kd + "/desc.h", &desc)) {
        if (err) *err = "cannot read device sources in " + kd;
        return "";
    }
    for (std::string* t : {&prelude, &table, &desc}) {
        size_t po = t->find("#pragma once");
        if (po != std::string::npos) t->erase(po, 12);
    }
    std::ostringstream o;
    o << "// generated by lensed-amd: prelude, objects, model code\n";
    if (std::any_of(models.begin(), models.end(), model_adds_exps)) o << "#define LCL_PLAIN_EXP\n";
    o << prelude << "\n" << desc
      << "\n#ifdef LCL_GPU\n#pragma clang force_cuda_host_device begin\n#endif\nnamespace lcl {\n";
    std::set<std::string> seen;
    for (const auto& m : models)
        for (const auto& ob : m) {
            if (!seen.insert(ob.name).second) continue;
            std::string src, path;
            if (!load_object_source(ob.name, &src, &path)) {
                if (err) *err = "could not load object \"" + ob.name + "\"";
                return "";
            }
            std::string mg = mangle(ob.name);
            o << wrap_object(translate_object(src, mg), mg, ob.name);
        }
    o << "}  // namespace lcl\n#ifdef LCL_GPU\n#pragma clang force_cuda_host_device end\n#endif\n";
    o << table << "\n#ifdef LCL_GPU\n#pragma clang force_cuda_host_device begin\n#endif\nnamespace lcl {\n";
    o << "#line 1 \"generated\"\n";
    for (size_t k = 0; k < models.size(); ++k)
        o << compute_function(models[k], (int)k) << set_params_function(models[k], (int)k);
    o << "template <int K> inline float compute_model(uint* data, float2 x, const float4* tab, float4 pre);\n"
      << "template <int K> inline float4 epl_pre_model(uint* data, float2 d, bool pixel);\n"
      << "template <int K> inline bool cull_model(uint* data, float4 base, const float4* tab, const float4* cc, "
         "float rho);\n"
      << "template <int K> inline void cull_consts_model(uint* data, float4* cc);\n";
    for (size_t k = 0; k < models.size(); ++k)
        o << "template <> inline float compute_model<" << k << ">(uint* data, float2 x, const float4* tab, "
          << "float4 pre) { return compute_" << k << "(data, x, tab, pre); }\n"
          << "template <> inline float4 epl_pre_model<" << k << ">(uint* data, float2 d, bool pixel) "
          << "{ return epl_pre_" << k << "(data, d, pixel); }\n"
          << "template <> inline bool cull_model<" << k << ">(uint* data, float4 base, const float4* tab, "
          << "const float4* cc, float rho) { return cull_" << k << "(data, base, tab, cc, rho); }\n"
          << "template <> inline void cull_consts_model<" << k << ">(uint* data, float4* cc) "
          << "{ cull_consts_" << k << "(data, cc); }\n";
    auto lists = [&](const char* name, bool (*which)(const std::vector<ModelObject>&)) {
        o << "constexpr bool " << name << "(int k) { return false";
        for (size_t k = 0; k < models.size(); ++k)
            if (which(models[k])) o << " || k == " << k;
        o << "; }\n";
    };
    lists("model_holds", model_holds);
    lists("model_tabulates", model_tabulates);
    o << "}  // namespace lcl\n#ifdef LCL_GPU\n#pragma clang force_cuda_host_device end\n#endif\n";
    return o.str();
}

std::string assemble_program(const std::vector<std::vector<ModelObject>>& models, std::string* err,
                             const std::vector<PsfShape>& psfs) {
    std::string kd = kernel_dir(), kern, series;
    if (!read_text(kd + "/lensed_kernels.hip", &kern) || !read_text(kd + "/epl_series.h", &series)) {
        if (err) *err = "cannot read device sources in " + kd;
        return "";
    }
    std::string ms = model_source(models, err);
    if (ms.empty()) return "";
    // the kernels' one local include is inlined: hipRTC sees a single source
    size_t po = series.find("#pragma once");
    if (po != std::string::npos) series.erase(po, 12);
    size_t inc = kern.find("#include \"epl_series.h\"");
    if (inc != std::string::npos) kern.replace(inc, strlen("#include \"epl_series.h\""), series);
    size_t dmax = 4;
    for (const auto& m : models) dmax = std::max(dmax, model_data_words(m));
    std::ostringstream o;
    o << ms << "#define LENSED_NMODELS " << models.size() << "\n#define LENSED_DWORDS " << dmax
      << "\n#define LENSED_FOR_MODELS(X)";
    for (size_t k = 0; k < models.size(); ++k) o << " X(" << k << ")";
    o << "\n#define LENSED_FOR_PSFS(X)";
    for (const auto& p : psfs) o << " X(" << p.w << ", " << p.h << ", " << (p.sep ? "true" : "false") << ")";
    o << "\n" << kern;
    return o.str();
}

static uint64_t fnv1a(const std::string& s, uint64_t h = 1469598103934665603ull) {
    for (unsigned char c : s) {
        h ^= c;
        h *= 1099511628211ull;
    }
    return h;
}

static std::string cache_dir() {
    if (const char* e = getenv("LENSED_CACHE_DIR")) return e;
    if (const char* h = getenv("HOME")) return std::string(h) + "/.cache/lensed_amd";
    return "";
}

// compile with a disk cache keyed by source, options and the compiler
static bool compile_cached(const std::string& src, const std::vector<std::string>& opts,
                           std::vector<char>* code, std::string* log) {
    std::string key = src;
    for (const auto& o : opts) key += "\n" + o;
    key += "\n" + compiler_identity();
    char name[40];
    snprintf(name, sizeof name, "%016llx.co", (unsigned long long)fnv1a(key));
    std::string dir = cache_dir();
    if (!dir.empty() && !getenv("LENSED_NO_CACHE")) {
        std::ifstream f(dir + "/" + name, std::ios::binary);
        if (f) {
            code->assign(std::istreambuf_iterator<char>(f), std::istreambuf_iterator<char>());
            if (!code->empty()) return true;
        }
    }
    if (!rtc_compile(src, "lensed_program.hip", opts, code, log)) return false;
    if (!dir.empty()) {
        std::string cmd = dir;
        for (size_t p = 1; p <= cmd.size(); ++p)
            if (p == cmd.size() || cmd[p] == '/') mkdir(cmd.substr(0, p).c_str(), 0755);
        std::string tmp = dir + "/" + name + ".tmp" + std::to_string((long)getpid());
        std::ofstream f(tmp, std::ios::binary);
        if (f) {
            f.write(code->data(), (std::streamsize)code->size());
            f.close();
            rename(tmp.c_str(), (dir + "/" + name).c_str());
        }
    }
    return true;
}

std::string device_arch(int device) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
        std::string a = prop.gcnArchName;
        size_t c = a.find(':');
        return c == std::string::npos ? a : a.substr(0, c);
    }
    return "gfx950";
}

// the affine form of every prior of a system, when all are uniform or deltas
static void fast_priors(System& S) {
    const size_t np = S.pars.size();
    S.xfast = true;
    S.xa.assign(np, 0);
    S.xs.assign(np, 0);
    S.xlo.assign(np, -HUGE_VAL);
    S.xhi.assign(np, HUGE_VAL);
    S.xdelta.assign(np, 0);
    for (size_t i = 0; i < np; ++i) {
        const Param& P = S.pars[S.pmap[i]];
        if (P.pri_copy.kind == prior::NORM) S.xfast = false;
        S.xa[i] = P.pri_copy.a;
        S.xs[i] = P.pri_copy.b - P.pri_copy.a;  // prior_apply's UNIF form: a + u (b - a)
        S.xdelta[i] = P.pri_copy.kind == prior::DELTA;
        if (P.bounded) {
            S.xlo[i] = P.lower;
            S.xhi[i] = P.upper;
        }
    }
}

// hard bounds and sampler ordering, as src/lensed.c:139-271
static int setup_params(System& S, const object* objs, size_t nobjs) {
    S.pars.clear();
    S.pmap.clear();
    std::vector<size_t> derived;
    for (size_t i = 0, p = 0; i < nobjs; ++i) {
        const object& ob = objs[i];
        for (size_t j = 0; j < ob.npars; ++j, ++p) {
            const param& in = ob.pars[j];
            Param P;
            P.id = in.id ? in.id : (std::string(ob.id ? ob.id : "obj") + "." + (in.name ? in.name : "?"));
            P.label = in.label ? in.label : "";
            P.type = in.type;
            P.lower = in.lower;
            P.upper = in.upper;
            if (!P.lower && !P.upper) {
                if (P.type == PAR_RADIUS) { P.lower = 0; P.upper = HUGE_VAL; }
                if (P.type == PAR_AXIS_RATIO) { P.lower = 0; P.upper = 1; }
            }
            P.bounded = P.lower || P.upper;
            if (!in.pri) {
                set_error(P.id + ": parameter has no prior");
                return -1;
            }
            P.pri_copy = *in.pri;
            P.has_prior = true;
            if (P.bounded && (prior_lower(in.pri) < P.lower || prior_upper(in.pri) > P.upper) &&
                (prior_lower(in.pri) >= P.upper || prior_upper(in.pri) <= P.lower)) {
                char b[256];
                snprintf(b, sizeof b, "%s: prior does not include parameter bounds [%g, %g]", P.id.c_str(),
                         P.lower, P.upper);
                set_error(b);
                return -1;
            }
            P.ipp = in.ipp != 0;
            P.wrap = in.wrap != 0;
            if (P.ipp) {
                bool ok = (P.type == PAR_POSITION_X && j + 1 < ob.npars && ob.pars[j + 1].type == PAR_POSITION_Y &&
                           ob.pars[j + 1].ipp) ||
                          (P.type == PAR_POSITION_Y && j > 0 && ob.pars[j - 1].type == PAR_POSITION_X &&
                           ob.pars[j - 1].ipp);
                if (!ok) {
                    set_error(P.id + ": image plane prior requires a pair (X,Y) of position parameters");
                    return -1;
                }
            }
            P.derived = prior_pseudo(in.pri) != 0;
            if (P.derived)
                derived.push_back(p);
            else
                S.pmap.push_back(p);
            S.pars.push_back(P);
        }
    }
    S.ndims = S.pmap.size();
    for (size_t d : derived) S.pmap.push_back(d);
    return 0;
}

static hipFunction_t conv_function(const ::lensed* l, int rows);

// parameters up to this size are read from pinned host memory (enqueue_chain)
constexpr size_t kDirectParamBytes = 4096;

static void free_layout(::lensed* l, Layout& L) {
    if (l->last_layout == &L) l->last_layout = nullptr;
    if (l->last_table_layout == &L) l->last_table_layout = nullptr;
    if (L.graph) hipGraphExecDestroy(L.graph);
    if (L.d_desc) hipFree(L.d_desc);
    L.graph = nullptr;
    L.d_desc = nullptr;
}

// drop the least recently used layout once the cache is full (a caller
// cycling through many batch sizes would otherwise hold a descriptor buffer
// and a graph per size for the context's lifetime)
static void evict_layouts(::lensed* l) {
    while (l->layouts.size() >= kMaxLayouts) {
        auto victim = l->layouts.begin();
        for (auto it = l->layouts.begin(); it != l->layouts.end(); ++it)
            if (it->second.last_use < victim->second.last_use) victim = it;
        hipStreamSynchronize(l->stream);  // no launch still reads it
        free_layout(l, victim->second);
        l->layouts.erase(victim);
    }
}

// everything of a launch layout but its device descriptors (no allocation
// on the device), without a cull pass if cull is false; 0 on success
static int build_layout(::lensed* l, const std::vector<size_t>& ncand, Layout& L, bool cull = true) {
    size_t total = 0;
    for (size_t s = 0; s < l->sys.size(); ++s) {
        if (ncand[s] > l->max_batch) {
            set_error("more candidates than max_batch");
            return -1;
        }
        total += ncand[s];
    }
    if (total == 0) {
        set_error("no candidates");
        return -1;
    }
    // conv tile height: 32 rows where the launch has two such tiles per CU,
    // and 64 where it has enough of those and rounding the images up to whole
    // tiles adds little.  (us, 8-, 32- and 64-row tiles, by the number of
    // 64-row ones.  Images of 64 rows: direct 31 x 31 taps 256: 46, 41, 47;
    // 512: 77, 65, 53; 8192: 1162, 941, 694; row and column passes, 21 x 21
    // taps 512: 18.6, 12.8, 12.6; 16384: 445, 232, 182; 22 x 8 taps 600: 17.6,
    // 12.7, 13.7; 7 x 7 taps 600: 16, 10.6, 11.5; 768: 20, 11.7, 11.7; 16384:
    // 344, 163, 134; no PSF 768: 13.4, 8.2, 8.8; 1024: 16, 9.6, 9.3; 16384:
    // 196, 86, 68.  Of 32, half a tall tile, 4096: 31 x 31 322, 235, 344; 7 x 7
    // 49, 24, 35.  Of 80, a third more in tall tiles, 8192: 719, 710, 685 and
    // 108, 60, 67.  Of 160, a fifth more, 8192: 966, 797, 686 and 144, 69, 68;
    // 13 x 13 taps 16384: 335, 144, 149.  Images of at most four rows don't
    // count, what they fill of a tile of either height is next to nothing:
    // 1200 of 1 x 64, 3 x 3 taps: 7.7, 9.5, 12.1)
    long long n32 = 0, n64 = 0, r32 = 0, r64 = 0;
    long long per_cu = 2;  // tall tiles the launch has to have
    double grown = 1.4;    // rows in tall tiles to rows in 32-row ones, below this
    for (size_t s = 0; s < l->sys.size(); ++s) {
        const System& S = l->sys[s];
        if (!ncand[s]) continue;
        auto tiles = [&](size_t rows) {
            return (long long)(ncand[s] * ((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX) *
                               ((S.height + LENSED_CONV_TY * rows - 1) / (LENSED_CONV_TY * rows)));
        };
        const long long t32 = tiles(LENSED_CONV_RY), t64 = tiles(LENSED_CONV_RY_TALL);
        const size_t taps = S.psfw * S.psfh;
        n32 += t32;
        n64 += t64;
        if (S.height > LENSED_CONV_TY) {
            r32 += t32 * LENSED_CONV_RY;
            r64 += t64 * LENSED_CONV_RY_TALL;
            grown = std::min(grown, taps >= 600 && !S.sep_rank ? 1.4 : taps >= 170 || !taps ? 1.25 : 1.2);
        }
        per_cu = std::max(per_cu, taps >= 170 ? 2LL : taps ? 3LL : 4LL);
    }
    L.conv_small = n32 < 2LL * l->cu_count;
    const lensed_tuning& tq = l->tune_req;
    const bool tall = n64 >= per_cu * l->cu_count && (!r32 || (double)r64 < grown * (double)r32);
    const int rows_default = L.conv_small ? LENSED_CONV_RY_SMALL : tall ? LENSED_CONV_RY_TALL : LENSED_CONV_RY;
    L.conv_rows = tq.conv_rows ? tq.conv_rows : rows_default;
    long long squares = 0;  // 64 pixels each: a wave of the render
    bool tables = false, series = false;
    for (size_t s = 0; s < l->sys.size(); ++s) {
        squares += 4LL * (long long)ncand[s] * l->sys[s].ntile_r;
        tables = tables || (ncand[s] && l->sys[s].table);
        series = series || (ncand[s] && l->sys[s].series);
    }
    // no cull pass where tracing every ray takes no longer than finding the
    // dark ones (us of cull and render, with and without the pass, 256 x 256:
    // table 1 candidate 27, 16; 4: 29, 23; 8: 33, 35; series 1: 26, 16; 2: 27,
    // 24; 4: 31, 40.  Whole calls with Gaussians of 1/8 of the Einstein radius,
    // by the number of squares, EPL + shear by its series 128 x 128 3072: 72,
    // 53; 4096: 70, 59; 160 x 160 6000: 81, 80; 8400: 92, 97; SIE 128 x 128
    // 3072: 72, 69; 256 x 256 4096: 71, 76; 200 x 200 4056: 75, 95)
    const long long fill = 4LL * l->cu_count;  // one square per SIMD
    const bool no_cull = !cull || (l->flags & LENSED_NO_CULL) ||
                         (tables ? squares < 8 * fill : series ? squares <= 4 * fill : squares < 3 * fill);
    // the column sweep: every system with candidates has a rank-1 separable
    // PSF of at most 21 x 21, and at most 512 rows.  It is the default
    // where every such system is also culled: it skips the rows the cull
    // found dark, and with every row lit the tile is the faster (C3 at 4096
    // candidates: 0.30 against 0.80 ms; C4, nothing culled: 14.0 against
    // 8.0 ms), from two strips per CU on.  A wave takes about 0.25 us per row
    // of its strip whatever else runs, so fewer strips leave the device
    // waiting for a few waves (256 x 256, 21 x 21 PSF, sweep with each strip
    // cut as below against the tile: 1 candidate 16 / 8 us, 16: 17 / 12, 64:
    // 24 / 19, 128: 34 / 33, 256: 41 / 55, 512: 68 / 111), and up to four
    // waves per SIMD each strip is cut into parts, a wave each, at the price
    // of refilling the window above every part (256 candidates whole, in 2, 4
    // and 8 parts: 70, 45, 41 and 50 us; 1024: 93, 92, 112 and 126).
    bool sweep_ok = true, all_culled = true, some_culled = false;
    long long strips = 0;
    for (size_t s = 0; s < l->sys.size(); ++s) {
        const System& S = l->sys[s];
        if (!ncand[s]) continue;
        strips += (long long)ncand[s] * ((S.width + 63) / 64);
        if (!S.psfw || S.sep_rank != 1 || S.psfw > LENSED_SWEEP_MAX_PSF || S.psfh > LENSED_SWEEP_MAX_PSF ||
            S.height > LENSED_SWEEP_MAX_H)
            sweep_ok = false;
        if (!S.cull || no_cull)
            all_culled = false;
        else
            some_culled = true;
    }
    if (!tq.conv_rows && sweep_ok && all_culled && strips >= 2LL * l->cu_count) L.conv_rows = LENSED_CONV_SWEEP;
    if (L.conv_rows == LENSED_CONV_SWEEP && !sweep_ok)
        L.conv_rows = rows_default;
    if (L.conv_rows == LENSED_CONV_RY_TALL) {
        // the 64-row tile only where its LDS stays within 64 KiB
        for (size_t s = 0; s < l->sys.size(); ++s) {
            const System& S = l->sys[s];
            if (!ncand[s] || !S.psfw) continue;
            size_t ch = LENSED_CONV_TY * LENSED_CONV_RY_TALL + S.psfh - 1;
            size_t words = (size_t)LENSED_TILE_STRIDE(S.psfw) * ch + (S.sep_rank > 1 ? LENSED_CONV_TX * ch : 0);
            if (words * 4 > 65536) L.conv_rows = LENSED_CONV_RY;
        }
    }
    L.conv_small = L.conv_rows == LENSED_CONV_RY_SMALL;
    const bool sweep = L.conv_rows == LENSED_CONV_SWEEP;
    const int seg = (int)std::min(64LL, std::max(1LL, (16LL * l->cu_count + strips - 1) / strips));
    const int ry = sweep ? LENSED_CONV_RY : L.conv_rows;  // (tile counts of a sweep layout are not used)
    const int th = LENSED_CONV_TY * ry;
    long long param_off = 0, block_off = 0, model_off = 0, partial_off = 0, out_off = 0, table_off = 0;
    long long npre_off = 0;
    int ir = 0, ik = 0, ic = 0, is = 0, iff = 0, itab = 0, inode = 0;
    for (size_t s = 0; s < l->sys.size(); ++s) {
        if (!ncand[s]) continue;
        const System& S = l->sys[s];
        lensed_desc d;
        memset(&d, 0, sizeof d);
        d.width = (int)S.width;
        d.height = (int)S.height;
        d.npix = (int)S.npix;
        d.model = S.model;
        d.psfw = (int)S.psfw;
        d.psfh = (int)S.psfh;
        d.ncand = (int)ncand[s];
        d.npar = (int)S.pars.size();
        // no block is cut off by the image's edge if items are pixels in a
        // row; the cull's list and flags, where the launch has them, are of
        // 16 x 16 blocks.  (us, blocks and rows: 256 candidates of 100 x 100
        // 500, 442; 333 of 131 x 97 847, 795; 1024 of 200 x 200 7325, 7120;
        // 139 of 186 x 154 695, 639; tabulated, 1803 of 123 x 170 1963, 1873)
        const int in_rows = (int)((S.npix + LENSED_RENDER_BS - 1) / LENSED_RENDER_BS);
        d.linear = !some_culled && in_rows < S.ntile_r ? 1 : 0;
        d.ntile_r = d.linear ? in_rows : S.ntile_r;
        d.dwords = (int)S.dwords;
        d.conv_ry = ry;
        d.tiles_x = (int)((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX);
        d.ntile_c = d.tiles_x * (int)((S.height + th - 1) / th);
        d.npart = d.tiles_x * (int)((S.height + 7) / 8);
        for (int i = 0; i < 4; ++i) d.pcs[i] = (float)S.pcs[i];
        d.image_off = S.image_off;
        d.psf_off = S.psf_off;
        d.model_off = model_off;
        d.block_off = block_off;
        d.param_off = param_off;
        d.partial_off = partial_off;
        d.out_off = out_off;
        d.item_r = ir;
        d.item_k = ik;
        d.item_c = ic;
        d.item_s = is;
        d.item_f = iff;
        d.epl_obj = S.epl_obj;
        d.epl_q = S.epl_q;
        d.epl_t = S.epl_t;
        d.table_mode = S.table ? 1 : 0;
        d.table_off = S.table ? table_off : 0;
        d.item_t = itab;
        d.item_e = inode;
        d.quad_off = S.quad_off;
        d.nq = S.nq;
        d.sep_rank = S.sep_rank;
        d.sep_off = S.sep_off;
        d.psft_off = S.psft_off;
        d.npre_off = npre_off;
        d.qrad = S.qrad;
        d.cull = S.cull && !no_cull ? 1 : 0;
        d.dark_off = S.dark_off;
        d.sweep_seg = seg;
        L.any_cull = L.any_cull || d.cull;
        long long nc = (long long)ncand[s];
        param_off += nc * d.npar;
        block_off += nc * d.dwords;
        model_off += nc * d.npix;
        partial_off += nc * d.npart;
        out_off += nc;
        ir += (int)(nc * d.ntile_r);
        L.n_blocks += (long)(nc * S.ntile_r);
        ik += (int)(nc * ((d.ntile_r + LENSED_CULL_GROUP - 1) / LENSED_CULL_GROUP));
        ic += (int)(nc * (sweep ? d.tiles_x * seg : d.ntile_c));  // sweep: an item per part of a 64-column strip
        is += (int)nc;
        iff += (int)nc;
        if (S.table || S.cull) npre_off += nc * LENSED_NPRE_STRIDE(S.table ? S.nq : 0);
        if (S.table) {
            table_off += nc * LENSED_EPL_TABLE_F4;
            itab += (int)(nc * LENSED_EPL_ROWS);
            inode += (int)(nc * LENSED_EPL_ROWS);
            L.n_tcands += (int)nc;
            L.lds_render = LENSED_EPL_TABLE_F4 * 16;
        }
        if (S.psfw && !sweep) {  // (the sweep's staged rows are static LDS)
            size_t ch = th + S.psfh - 1;
            // rank 1: the row pass writes over the tile; higher ranks keep a second buffer
            size_t words = (size_t)LENSED_TILE_STRIDE(S.psfw) * ch + (S.sep_rank > 1 ? LENSED_CONV_TX * ch : 0);
            L.lds_conv = std::max(L.lds_conv, words * 4);
        }
        L.desc.push_back(d);
        L.sys_of_desc.push_back((int)s);
    }
    // persistent grids sized by what stays resident with this launch's LDS,
    // times the requested multiples.  The render's default is 16 times over
    // the items and 4 times over the cull's list: with as many blocks as are
    // resident, whole rounds of equal work leave the last one part empty
    // (12544 items on 2048 blocks: 7 rounds for 6.1), while further blocks
    // start as others end.  256 candidates of 100 x 100 (SIE + Sersic): 698 us
    // at 1, 670 at 4, 604 at 16; 512 of 512 x 512 (table): 12.7, 11.7, 11.6
    // ms; the list's blocks lose more to starting than they gain beyond 4
    // (512 of 256 x 256, series: 665, 612, 635 us).
    const double default_render_grid = L.any_cull ? 4.0 : 16.0;
    {
        auto scaled = [&](int resident, double m) {
            return std::max(1, (int)std::lround(resident * (m > 0 ? m : 1.0)));
        };
        int nb = 0;
        hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, conv_function(l, L.conv_rows), LENSED_CONV_BS,
                                                           L.lds_conv);
        L.grid_conv = scaled(std::max(1, nb) * l->cu_count, tq.conv_grid);
        if (sweep) L.grid_conv = (ic + 3) / 4;  // not persistent: four strips per block, every strip its wave
        nb = 0;
        hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, l->f_render, LENSED_RENDER_BS, L.lds_render);
        L.grid_render = scaled(std::max(1, nb) * l->cu_count, tq.render_grid > 0 ? tq.render_grid : default_render_grid);
        // the cull's blocks take a few items each by default (its items differ in cost by
        // their unsettled squares; 4x evens the tail: C3 cull 0.18 -> 0.14 ms)
        L.grid_cull = scaled(std::max(1, nb) * l->cu_count, tq.cull_grid > 0 ? tq.cull_grid : 4.0);
    }
    L.conv_order = tq.conv_order == 2 ? 1 : 0;
    {
        // a block per 64 pixels, their rays shared among its waves, where the
        // launch has too few pixels for a wave to trace its own (us of render,
        // a wave per 64 pixels and shared: SIE + Sersic 196 squares 46, 13;
        // 1568: 37, 34; 6272: 105, 103; series 1024: 20, 16; 4096: 39, 41;
        // table 1024: 18, 13; 2048: 17, 19, each block staging the table;
        // culled, most of the squares dark: 8192: 49, 33; 16384: 45, 40;
        // 32768: 57, 62)
        const long long per = L.any_cull ? 16 : tables ? 1 : 3;
        int nqmax = 0;
        for (const auto& d : L.desc) nqmax = std::max(nqmax, d.nq);
        L.lds_wide = L.lds_render + (size_t)nqmax * 64 * sizeof(float);
        L.wide = squares <= per * 4 * l->cu_count && nqmax > 4 && L.lds_wide <= 65536;
    }
    {
        // the render walks the list while under list_fraction of the quads are lit
        const double f = tq.list_fraction == 0 ? 0.75 : tq.list_fraction;
        const double quads = 16.0 * (double)ir;
        L.list_max = f < 0 ? 0 : f > 1 ? INT_MAX : (int)std::min<double>(INT_MAX, std::ceil(f * quads));
        L.tune.list_fraction = f;
    }
    L.tune.render_grid = tq.render_grid > 0 ? tq.render_grid : default_render_grid;
    L.tune.cull_grid = tq.cull_grid > 0 ? tq.cull_grid : 4.0;
    L.tune.conv_grid = tq.conv_grid > 0 ? tq.conv_grid : 1.0;
    L.tune.conv_rows = L.conv_rows;
    L.tune.conv_order = L.conv_order + 1;
    L.n_render = ir;
    L.n_cull = ik;
    L.n_conv = ic;
    L.n_set = is;
    L.n_final = iff;
    L.n_table = itab;
    L.n_nodes = inode;
    return 0;
}

// a launch layout for ncand candidates per system; emulate = false makes
// every EPL table from the exact series (a layout of its own, keyed apart)
static Layout* get_layout(::lensed* l, const std::vector<size_t>& ncand, bool emulate = true) {
    std::vector<size_t> key = ncand;
    key.push_back(emulate ? 1 : 0);
    auto it = l->layouts.find(key);
    if (it != l->layouts.end()) {
        it->second.last_use = ++l->layout_clock;
        return &it->second;
    }
    evict_layouts(l);
    Layout L;
    if (build_layout(l, ncand, L)) return nullptr;
    L.last_use = ++l->layout_clock;
    if (hipMalloc(&L.d_desc, L.desc.size() * sizeof(lensed_desc)) != hipSuccess ||
        hipMemcpy(L.d_desc, L.desc.data(), L.desc.size() * sizeof(lensed_desc), hipMemcpyHostToDevice) != hipSuccess) {
        set_error("failed to upload launch descriptors");
        return nullptr;
    }
    L.id = l->next_layout_id++;
    L.emulate = emulate;
    return &(l->layouts[key] = L);
}

// ints of the cull's render list: the count, the quads (four per square),
// and the pads (fewer than an entry per cull block, where a block's part of
// a candidate ends; a launch has no more blocks than cull items)
static size_t live_capacity(size_t squares, size_t cull_items) {
    return 1 + 4 * squares + LENSED_LIST_ENTRY * cull_items;
}

static Buffers context_buffers(::lensed* l, const Layout& L) {
    Buffers B;
    B.desc = L.d_desc;
    B.params = l->d_params;
    B.blocks = l->d_blocks;
    B.model = l->d_model;
    B.partials = l->d_partials;
    B.tables = l->d_tables;
    B.npre = l->d_npre;
    B.trace = l->d_trace;
    B.live = l->d_live;
    B.owner = l->d_owner;
    B.written = l->d_written;
    B.emulate = L.emulate;
    return B;
}

static hipFunction_t conv_function(const ::lensed* l, int rows) {
    return rows == LENSED_CONV_RY_SMALL  ? l->f_conv_small
           : rows == LENSED_CONV_RY_TALL ? l->f_conv_tall
           : rows == LENSED_CONV_SWEEP   ? l->f_conv_sweep
                                         : l->f_conv;
}

static int launch(hipFunction_t f, int grid, int block, size_t lds, hipStream_t st, void** args) {
    LSD_HIP(hipModuleLaunchKernel(f, grid, 1, 1, block, 1, 1, (unsigned)lds, st, args, nullptr));
    return 0;
}

// enqueue the four-kernel chain on buffers B; planes != nullptr selects the
// dumper outputs
static int enqueue_chain(::lensed* l, Layout& L, const Buffers& B, bool prof, float* err_plane, float* conv_plane,
                         float* chi2_plane) {
    hipStream_t st = l->stream;
    auto rec = [&](int i) { if (prof) hipEventRecord(l->ev[i], st); };
    size_t nparams = 0;
    for (const auto& d : L.desc) nparams += (size_t)d.ncand * d.npar;
    int nsys = (int)L.desc.size();
    // with a cull pass, the render walks the list of items it kept
    int* live = L.any_cull ? B.live : nullptr;
    lensed_desc* desc = B.desc;
    float* params = B.params;
    unsigned* blocks = B.blocks;
    float* model = B.model;
    // the results go straight to pinned host memory: each candidate's logL,
    // or, for a single candidate, its chi^2 partials, which the host adds up
    // (finish_single) in less time than one more kernel takes to start
    const bool single = L.n_final == 1;
    double* partials = single ? l->h_partials : B.partials;
    double* logl = l->h_logl;
    void* tables = B.tables;
    void* npre = B.npre;
    int* owner = B.owner;
    int* written = B.written;
    if (B.record) l->last_layout = &L;
    rec(0);
    // a few candidates' parameters are read by the kernels from the pinned
    // buffer itself: a copy and the wait for it take longer (3 us a call)
    if (nparams * sizeof(float) <= kDirectParamBytes)
        params = l->h_params;
    else
        LSD_HIP(hipMemcpyAsync(params, l->h_params, nparams * sizeof(float), hipMemcpyHostToDevice, st));
    rec(1);
    rec(2);
    // with the emulator's network certified for some (q, t) cells, it builds
    // those candidates' tables and the exact series the others, after
    // set_params; otherwise set_params' blocks and the exact tables' blocks
    // go in one launch
    const bool emu_tables = L.n_table > 0 && l->emu_wf && B.emulate && l->emu_ncert > 0;
    if (L.n_table > 0 && l->emu_wf && B.emulate && B.record) l->last_table_layout = &L;
    if (L.n_table > 0 && !emu_tables) {
        int set_blocks = (L.n_set + LENSED_EPL_NT - 1) / LENSED_EPL_NT;
        void* a[] = {&desc, &nsys, &L.n_set, &params, &blocks, &l->d_quad, &npre,
                     &live, &owner, &L.id, &L.n_table, &tables, &set_blocks};
        if (launch(l->f_set_tables, set_blocks + L.n_table / LENSED_EPL_ROWS, LENSED_EPL_NT, 0, st, a)) return -1;
    } else {
        void* a[] = {&desc, &nsys, &L.n_set, &params, &blocks, &l->d_quad, &npre, &live, &owner, &L.id};
        if (launch(l->f_set, (L.n_set + 255) / 256, 256, 0, st, a)) return -1;
    }
    if (emu_tables) {
        if (emu_launch_tables(st, desc, nsys, L.n_nodes, L.n_table, L.n_tcands, params, l->emu_wf, l->emu_wp,
                              l->d_nodes, tables, l->d_flags, l->d_cells))
            return -1;
        int* only = l->d_flags;
        void* a[] = {&desc, &nsys, &L.n_table, &params, &tables, &only};
        if (launch(l->f_tables, L.n_table / LENSED_EPL_ROWS, LENSED_EPL_NT, 0, st, a)) return -1;  // a block per candidate
        // which candidates the network served, for the recheck of accepted points
        LSD_HIP(hipMemcpyAsync(l->h_flags, l->d_flags, (size_t)L.n_tcands * 4, hipMemcpyDeviceToHost, st));
    }
    rec(3);
    int* trace = L.any_cull ? B.trace : nullptr;
    if (L.any_cull) {
        int grid = std::min(L.n_cull, L.grid_cull);
        void* a[] = {&desc, &nsys, &L.n_cull, &blocks, &tables, &npre, &trace, &live, &model, &err_plane, &owner,
                     &written};
        if (launch(l->f_cull, grid, LENSED_RENDER_BS, L.lds_render, st, a)) return -1;
        rec(9);
    }
    {
        int grid = std::min(L.n_render, L.grid_render), table_f4 = (int)(L.lds_render / 16);
        void* a[] = {&desc,  &nsys,  &L.n_render, &blocks,    &l->d_quad,  &tables,
                     &npre,  &live,  &trace,      &model,     &err_plane,  &L.list_max, &table_f4};
        if (L.wide) grid = std::min(4 * L.n_render, L.grid_render);
        if (launch(L.wide ? l->f_wide : l->f_render, grid, LENSED_RENDER_BS, L.wide ? L.lds_wide : L.lds_render, st, a))
            return -1;
    }
    rec(4);
    {
        const bool sweep = L.conv_rows == LENSED_CONV_SWEEP;
        int grid = sweep ? (L.n_conv + 3) / 4 : std::min(L.n_conv, L.grid_conv);
        // trace: dark tiles skip the convolution
        // (the sweep's last argument: the data's partials for a model of 0)
        void* a[] = {&desc,     &nsys,     &L.n_conv,   &model,      &l->d_image,   &l->d_weight, &l->d_psf,
                     &partials, &conv_plane, &chi2_plane, &trace,    &L.conv_order, &l->d_dark};
        hipFunction_t f = conv_function(l, L.conv_rows);
        if (sweep && (conv_plane || chi2_plane)) f = l->f_conv_sweep_out;  // the dumper's planes
        if (launch(f, grid, LENSED_CONV_BS, sweep ? 0 : L.lds_conv, st, a)) return -1;
    }
    rec(5);
    if (!single) {
        void* a[] = {&desc, &nsys, &L.n_final, &partials, &logl};
        if (launch(l->f_final, (L.n_final + 3) / 4, 256, 0, st, a)) return -1;
    }
    rec(6);
    rec(7);
    rec(8);
    return 0;
}

// lensed_finalize for the one candidate of a launch, on the host: the same
// additions in the same order, a lane's partials 64 apart, then the lanes in
// pairs 32, 16, ... apart
static void finish_single(::lensed* l, const Layout& L) {
    if (L.n_final != 1) return;
    double lane[64] = {};
    for (int t = 0; t < L.desc[0].npart; ++t) lane[t % 64] += l->h_partials[t];
    for (int o = 32; o > 0; o >>= 1)
        for (int i = 0; i < o; ++i) lane[i] += lane[i + o];
    l->h_logl[0] = -0.5 * lane[0];
}

static int run_layout(::lensed* l, Layout& L) {
    bool prof = (l->flags & LENSED_PROFILE) != 0;
    bool graph = (l->flags & LENSED_GRAPH) != 0 && !prof && L.n_final > 1;  // one candidate: direct launches are quicker
    if (graph) {
        if (!L.graph) {
            hipGraph_t g;
            LSD_HIP(hipStreamBeginCapture(l->stream, hipStreamCaptureModeThreadLocal));
            int rc = enqueue_chain(l, L, context_buffers(l, L), false, nullptr, nullptr, nullptr);
            hipError_t ec = hipStreamEndCapture(l->stream, &g);
            if (rc || ec != hipSuccess) {
                if (!rc) set_error(std::string("graph capture failed: ") + hipGetErrorString(ec));
                return -1;
            }
            LSD_HIP(hipGraphInstantiate(&L.graph, g, nullptr, nullptr, 0));
            hipGraphDestroy(g);
        }
        LSD_HIP(hipGraphLaunch(L.graph, l->stream));
    } else if (enqueue_chain(l, L, context_buffers(l, L), prof, nullptr, nullptr, nullptr)) {
        return -1;
    }
    LSD_HIP(hipStreamSynchronize(l->stream));
    finish_single(l, L);
    if (prof) {
        for (int i = 0; i < 8; ++i) {
            float ms = 0;
            hipEventElapsedTime(&ms, l->ev[i], l->ev[i + 1]);
            l->prof_ms[i] += ms;
        }
        if (L.any_cull) {
            float ms = 0;
            hipEventElapsedTime(&ms, l->ev[3], l->ev[9]);
            l->prof_cull_ms += ms;
        }
        l->prof_calls += 1;
    }
    return 0;
}

// the autotuner's cache key: device, program and its compiler, and the
// layout's systems and candidate counts
static std::string tune_key(const ::lensed* l, const std::vector<size_t>& ncand, bool emulate) {
    std::ostringstream k;
    k << "lensed-tune-3 " << device_arch(l->device) << " cu" << l->cu_count << " prog" << std::hex
      << fnv1a(l->source) << " cc" << fnv1a(compiler_identity()) << std::dec << " emu" << (emulate ? 1 : 0) << " flags" << (l->flags & ~(LENSED_PROFILE | LENSED_GRAPH));
    for (size_t s = 0; s < l->sys.size(); ++s)
        k << " " << l->sys[s].width << "x" << l->sys[s].height << "p" << l->sys[s].psfw << "x" << l->sys[s].psfh
          << "n" << ncand[s];
    return k.str();
}

// LENSED_AUTOTUNE: the layout's launch shapes from the disk cache, or timed
// on this launch's own parameters (already staged in h_params) and cached
static int autotune_layout(::lensed* l, Layout& L, const std::vector<size_t>& ncand) {
    L.tuned = true;
    const std::string key = tune_key(l, ncand, L.emulate);
    const lensed_tuning saved = l->tune_req;
    lensed_tuning best{};
    if (!tune_cache_read(cache_dir(), key, &best)) {
        lensed_desc* dd = nullptr;
        size_t ddcap = 0;
        TuneTimer timer = [&](const lensed_tuning& t, TuneTiming* out) -> int {
            l->tune_req = t;
            Layout T;
            if (build_layout(l, ncand, T)) return -1;
            T.id = L.id;  // the same squares, so the cull's record of written ones stays true
            T.emulate = L.emulate;
            const size_t bytes = T.desc.size() * sizeof(lensed_desc);
            if (bytes > ddcap) {
                if (dd) hipFree(dd);
                dd = nullptr;
                LSD_HIP(hipMalloc(&dd, bytes));
                ddcap = bytes;
            }
            LSD_HIP(hipMemcpy(dd, T.desc.data(), bytes, hipMemcpyHostToDevice));
            T.d_desc = dd;
            Buffers B = context_buffers(l, T);
            B.record = false;
            double r = 1e300, c = 1e300, tot = 1e300;
            for (int rep = 0; rep < 4; ++rep) {
                if (enqueue_chain(l, T, B, true, nullptr, nullptr, nullptr)) return -1;
                LSD_HIP(hipStreamSynchronize(l->stream));
                if (rep == 0) continue;  // the first launch of a shape warms it up
                float a = 0, b = 0, e = 0;
                hipEventElapsedTime(&a, l->ev[3], l->ev[4]);
                hipEventElapsedTime(&b, l->ev[4], l->ev[5]);
                hipEventElapsedTime(&e, l->ev[0], l->ev[8]);
                r = std::min(r, (double)a);
                c = std::min(c, (double)b);
                tot = std::min(tot, (double)e);
            }
            out->render_ms = r;
            out->conv_ms = c;
            out->total_ms = tot;
            return 0;
        };
        const int rc = autotune(timer, L.any_cull, &best);
        if (dd) hipFree(dd);
        l->tune_req = saved;
        if (rc) return -1;
        tune_cache_write(cache_dir(), key, best);
    }
    // the layout rebuilt with the chosen shapes (same systems, so the same
    // number of descriptors, uploaded over the old ones)
    l->tune_req = best;
    Layout T;
    const int rc = build_layout(l, ncand, T);
    l->tune_req = saved;
    if (rc) return -1;
    T.d_desc = L.d_desc;
    T.graph = L.graph;
    T.id = L.id;
    T.last_use = L.last_use;
    T.emulate = L.emulate;
    T.tuned = true;
    T.tune.default_ms = best.default_ms;
    T.tune.tuned_ms = best.tuned_ms;
    LSD_HIP(hipMemcpy(T.d_desc, T.desc.data(), T.desc.size() * sizeof(lensed_desc), hipMemcpyHostToDevice));
    L = T;
    return 0;
}

int evaluate(::lensed* l, const std::vector<size_t>& ncand, const std::vector<const double*>& phys,
             const std::vector<double*>& lnew, bool emulate) {
    Layout* L = get_layout(l, ncand, emulate);
    if (!L) return -1;
    for (size_t k = 0; k < L->desc.size(); ++k) {
        const lensed_desc& d = L->desc[k];
        int s = L->sys_of_desc[k];
        const double* p = phys[s];
        if (!p) continue;  // staged by the caller
        float* h = l->h_params + d.param_off;
        for (long long i = 0; i < (long long)d.ncand * d.npar; ++i) h[i] = (float)p[i];
    }
    // one candidate: the plain path's launch, nothing worth tuning
    if ((l->flags & LENSED_AUTOTUNE) && !L->tuned && L->n_final > 1 && autotune_layout(l, *L, ncand)) return -1;
    if (run_layout(l, *L)) return -1;
    const bool emulated = emulate && l->emu_wf && l->emu_ncert > 0;
    for (size_t k = 0; k < L->desc.size(); ++k) {
        const lensed_desc& d = L->desc[k];
        int s = L->sys_of_desc[k];
        memcpy(lnew[s], l->h_logl + d.out_off, (size_t)d.ncand * sizeof(double));
        std::vector<char>& used = l->sys[s].emu_used;
        used.clear();
        if (emulated && d.table_mode) {
            const int* f = l->h_flags + d.table_off / LENSED_EPL_TABLE_F4;
            used.resize(d.ncand);
            for (int c = 0; c < d.ncand; ++c) used[c] = f[c] == 0;
        }
    }
    return 0;
}

// The exact recheck of the candidates the sampler may accept: of the last
// lensed_loglike_batch() call on system s, those whose EPL table came from
// the network and whose logL exceeds lmin are evaluated again with the
// exact-series tables, and their logL replaced (phys: sampler order).
int recheck_emulated(::lensed* l, size_t s, const double* phys, int n, double lmin, double* ll) {
    System& S = l->sys[s];
    if (S.emu_used.size() != (size_t)n) return 0;  // no table of this batch came from the network
    std::vector<int> idx;
    for (int c = 0; c < n; ++c)
        if (S.emu_used[c] && ll[c] > lmin) idx.push_back(c);
    const size_t np = S.pars.size();
    for (size_t c0 = 0; c0 < idx.size(); c0 += l->max_batch) {
        const size_t nc = std::min(l->max_batch, idx.size() - c0);
        std::vector<double> p(nc * np), out(nc);
        for (size_t k = 0; k < nc; ++k)
            for (size_t i = 0; i < np; ++i) p[k * np + S.pmap[i]] = phys[(size_t)idx[c0 + k] * np + i];
        std::vector<size_t> ncv(l->sys.size(), 0);
        ncv[s] = nc;
        std::vector<const double*> pp(l->sys.size(), nullptr);
        pp[s] = p.data();
        std::vector<double*> oo(l->sys.size(), nullptr);
        oo[s] = out.data();
        if (evaluate(l, ncv, pp, oo, false)) return -1;
        for (size_t k = 0; k < nc; ++k) {
            double& v = ll[idx[c0 + k]];
            const double dv = std::fabs(v - out[k]);
            l->emu_rechecked += 1;
            l->emu_changed += dv != 0;
            l->emu_recheck_max = std::max(l->emu_recheck_max, dv);
            v = out[k];
        }
    }
    S.emu_used.clear();
    return 0;
}

}  // namespace lsd

using namespace lsd;

extern "C" {

const char* lensed_last_error(void) { return lsd::g_error.c_str(); }

lensed* lensed_create(const lensed_system* systems, size_t nsys, const lensed_options* opts) {
    if (!systems || nsys == 0) {
        set_error("no systems");
        return nullptr;
    }
    ::lensed* l = new ::lensed;
    l->device = opts ? opts->device : 0;
    l->flags = opts ? opts->flags : 0;
    l->max_batch = (opts && opts->max_batch) ? opts->max_batch : 1;
    std::vector<std::vector<ModelObject>> models;
    std::vector<std::vector<int>> model_ipp;
    std::vector<float> image, weight, psf, quad;
    for (size_t s = 0; s < nsys; ++s) {
        const lensed_system& in = systems[s];
        System S;
        if (!in.width || !in.height || !in.image || !in.weight || !in.nobjs || !in.objs) {
            set_error("system " + std::to_string(s) + ": missing image, weight or objects");
            delete l;
            return nullptr;
        }
        S.width = in.width;
        S.height = in.height;
        S.npix = in.width * in.height;
        S.h_image.assign(in.image, in.image + S.npix);
        S.h_weight.assign(in.weight, in.weight + S.npix);
        S.psfw = in.psf ? in.psfw : 0;
        S.psfh = in.psf ? in.psfh : 0;
        if (S.psfw > LENSED_PSF_MAX || S.psfh > LENSED_PSF_MAX) {
            set_error("PSF too large for the convolution tile (max 63 x 63)");
            delete l;
            return nullptr;
        }
        for (int i = 0; i < 4; ++i) S.pcs[i] = in.pcs[i];
        // half-pixel shift for even PSF sizes (src/lensed.c:884-891)
        if (S.psfw && S.psfw % 2 == 0) S.pcs[0] += 0.5;
        if (S.psfh && S.psfh % 2 == 0) S.pcs[1] += 0.5;
        S.rule = in.rule ? in.rule : "g3k7";
        int nq = lensed_quad_size(S.rule.c_str());
        if (nq <= 0) {
            set_error("invalid quadrature rule: " + S.rule);
            delete l;
            return nullptr;
        }
        std::vector<float> qq(2 * nq), ww(2 * nq);
        lensed_quad_rule(S.rule.c_str(), qq.data(), ww.data(), S.pcs[2], S.pcs[3]);
        S.nq = nq;
        S.quad_off = (int)(quad.size() / 4);
        double qr2 = 0;
        for (int i = 0; i < nq; ++i) qr2 = std::max(qr2, (double)qq[2 * i] * qq[2 * i] + (double)qq[2 * i + 1] * qq[2 * i + 1]);
        S.qrad = (float)(std::sqrt(qr2) * (1 + 1e-6));
        for (int i = 0; i < nq; ++i) {
            quad.push_back(qq[2 * i]);
            quad.push_back(qq[2 * i + 1]);
            quad.push_back(ww[2 * i]);
            quad.push_back(ww[2 * i + 1]);
        }
        // objects of the model
        std::vector<int> ipp;
        size_t npar_before = 0;
        for (size_t i = 0; i < in.nobjs; ++i) {
            const object& ob = in.objs[i];
            if (!ob.name || (ob.type != OBJ_LENS && ob.type != OBJ_SOURCE && ob.type != OBJ_FOREGROUND) ||
                (ob.npars && !ob.pars)) {
                set_error("system " + std::to_string(s) + ": invalid object " + std::to_string(i));
                delete l;
                return nullptr;
            }
            ModelObject mo;
            mo.name = ob.name;
            mo.type = ob.type;
            mo.size = (ob.size + 3) / 4 * 4;  // keep every object block 16-byte aligned
            mo.npars = ob.npars;
            // the first lens whose data layout the table form reads (an EPL
            // plugin of this package's layout) gets the tabulated angular factor
            if ((l->flags & (LENSED_TABLE | LENSED_EMULATE)) && S.epl_obj < 0 && mo.type == OBJ_LENS &&
                object_tabulates(mo.name)) {
                int iq = -1, ist = -1;
                for (size_t j = 0; j < ob.npars; ++j) {
                    if (ob.pars[j].name && strcmp(ob.pars[j].name, "q") == 0) iq = (int)j;
                    if (ob.pars[j].name && strcmp(ob.pars[j].name, "t") == 0) ist = (int)j;
                }
                if (iq >= 0 && ist >= 0) {
                    mo.table = true;
                    S.table = true;
                    S.epl_obj = (int)i;
                    S.epl_q = (int)(npar_before + iq);
                    S.epl_t = (int)(npar_before + ist);
                }
            }
            npar_before += ob.npars;
            for (size_t j = 0; j < ob.npars; ++j) {
                mo.ptype.push_back(ob.pars[j].type);
                mo.ipp.push_back(ob.pars[j].ipp != 0);
                ipp.push_back(ob.pars[j].ipp != 0);
            }
            S.objs.push_back(mo);
        }
        if (setup_params(S, in.objs, in.nobjs)) {
            delete l;
            return nullptr;
        }
        fast_priors(S);
        S.dwords = model_data_words(S.objs);
        S.cull = model_culls(S.objs);
        // model index: identical object lists share one compute function
        int model = -1;
        for (size_t k = 0; k < models.size() && model < 0; ++k) {
            if (models[k].size() != S.objs.size() || model_ipp[k] != ipp) continue;
            bool same = true;
            for (size_t i = 0; i < S.objs.size() && same; ++i)
                same = models[k][i].name == S.objs[i].name && models[k][i].size == S.objs[i].size &&
                       models[k][i].table == S.objs[i].table;
            if (same) model = (int)k;
        }
        if (model < 0) {
            model = (int)models.size();
            models.push_back(S.objs);
            model_ipp.push_back(ipp);
        }
        S.model = model;
        S.image_off = (long long)image.size();
        image.insert(image.end(), in.image, in.image + S.npix);
        weight.insert(weight.end(), in.weight, in.weight + S.npix);
        S.psf_off = (long long)psf.size();
        if (S.psfw) {
            psf.insert(psf.end(), in.psf, in.psf + S.psfw * S.psfh);
            S.psft_off = (long long)psf.size();
            for (size_t i = 0; i < S.psfw; ++i)
                for (size_t j = 0; j < S.psfh; ++j) psf.push_back(in.psf[j * S.psfw + i]);
            PsfFactors pf = factor_psf(in.psf, (int)S.psfw, (int)S.psfh);
            // the separable pass needs a second LDS buffer: keep the tall
            // tile and it within 64 KiB (square PSFs up to 55 pixels)
            const size_t ch = LENSED_CONV_TY * LENSED_CONV_RY + S.psfh - 1;
            const size_t sep_words = ((size_t)LENSED_TILE_STRIDE(S.psfw) + LENSED_CONV_TX) * ch;
            if (pf.rank > 0 && sep_words * 4 <= 65536 && !getenv("LENSED_DIRECT_CONV")) {
                S.sep_rank = pf.rank;
                S.sep_off = (long long)psf.size();
                psf.insert(psf.end(), pf.factors.begin(), pf.factors.end());
            }
        }
        S.ntile_r = (int)(((S.width + LENSED_RENDER_SIDE - 1) / LENSED_RENDER_SIDE) *
                          ((S.height + LENSED_RENDER_SIDE - 1) / LENSED_RENDER_SIDE));
        size_t np = S.pars.size();
        S.mean.assign(np, 0);
        S.sigma.assign(np, 0);
        S.ml.assign(np, 0);
        S.map.assign(np, 0);
        // images of a few blocks are lit nearly throughout, a Gaussian's
        // cutoff being 13 sigma out, and a series lens (whose rays cost half
        // an SIE's, its bound as much again) gains nothing there.  (us a call,
        // culled and not, without a table, sigma 1/8 of the Einstein radius:
        // EPL + shear 16 x 16 4375 candidates 273, 223; 24 x 24 1500: 170,
        // 150; 32 x 32 262: 90, 74; 48 x 48 1333: 286, 323; SIE 16 x 16 4375:
        // 345, 300; 24 x 24 262: 86, 98; 32 x 32 193: 94, 97; 3000: 569, 539)
        if (S.cull && !S.table) {
            for (const auto& ob : S.objs) S.series = S.series || (ob.type == OBJ_LENS && object_tabulates(ob.name));
            if (S.ntile_r < (S.series ? 9 : 4)) S.cull = false;
        }
        l->sys.push_back(S);
    }
    if (psf.empty()) psf.push_back(0.0f);
    for (const auto& m : models) l->block_pad = std::max(l->block_pad, model_data_words(m));

    std::vector<PsfShape> shapes;
    for (const auto& S : l->sys) {
        PsfShape p{(int)S.psfw, (int)S.psfh, S.sep_rank > 0};
        if (S.psfw && std::find(shapes.begin(), shapes.end(), p) == shapes.end()) shapes.push_back(p);
    }
    std::string err;
    l->source = assemble_program(models, &err, shapes);
    if (l->source.empty()) {
        set_error(err);
        delete l;
        return nullptr;
    }
    if (const char* dump = getenv("LENSED_DUMP_PROGRAM")) {  // the generated program, for reading its ISA
        std::ofstream f(dump);
        f << l->source;
    }
    if (hipSetDevice(l->device) != hipSuccess) {
        set_error("cannot select HIP device " + std::to_string(l->device));
        delete l;
        return nullptr;
    }
    std::vector<char> code;
    std::string log;
    if (!compile_cached(l->source, device_flags(device_arch(l->device)), &code, &log)) {
        set_error("failed to build program: " + log);
        delete l;
        return nullptr;
    }
    auto fail = [&](const char* what) {
        set_error(std::string("device setup failed: ") + what);
        lensed_destroy(l);
        return (lensed*)nullptr;
    };
    if (hipModuleLoadData(&l->module, code.data()) != hipSuccess) return fail("module load");
    if (hipModuleGetFunction(&l->f_set, l->module, "lensed_set_params") != hipSuccess ||
        hipModuleGetFunction(&l->f_render, l->module, "lensed_render") != hipSuccess ||
        hipModuleGetFunction(&l->f_conv, l->module, "lensed_conv_chi2") != hipSuccess ||
        hipModuleGetFunction(&l->f_conv_small, l->module, "lensed_conv_chi2_small") != hipSuccess ||
        hipModuleGetFunction(&l->f_final, l->module, "lensed_finalize") != hipSuccess ||
        hipModuleGetFunction(&l->f_tables, l->module, "lensed_epl_tables") != hipSuccess ||
        hipModuleGetFunction(&l->f_set_tables, l->module, "lensed_set_params_tables") != hipSuccess ||
        hipModuleGetFunction(&l->f_dark, l->module, "lensed_dark_partials") != hipSuccess ||
        hipModuleGetFunction(&l->f_wide, l->module, "lensed_render_wide") != hipSuccess ||
        hipModuleGetFunction(&l->f_cull, l->module, "lensed_cull") != hipSuccess ||
        hipModuleGetFunction(&l->f_conv_tall, l->module, "lensed_conv_chi2_tall") != hipSuccess ||
        hipModuleGetFunction(&l->f_conv_sweep, l->module, "lensed_conv_chi2_sweep") != hipSuccess ||
        hipModuleGetFunction(&l->f_conv_sweep_out, l->module, "lensed_conv_chi2_sweep_out") != hipSuccess)
        return fail("kernel lookup");
    if (hipStreamCreateWithFlags(&l->stream, hipStreamNonBlocking) != hipSuccess) return fail("stream");
    if (l->flags & LENSED_EMULATE) {
        std::vector<float> w(emu::kParams);
        if (!opts->emulator || lensed_emulator_read(opts->emulator, w.data())) {
            set_error(std::string("LENSED_EMULATE needs emulator weights: ") + lsd::g_error);
            lensed_destroy(l);
            return nullptr;
        }
        if (emu_upload(w.data(), &l->emu_wf, &l->emu_wp)) return fail("emulator weights");
        if (opts->emulator_tol > 0) l->emu_tol = (float)opts->emulator_tol;
    }
    for (auto& e : l->ev)
        if (hipEventCreate(&e) != hipSuccess) return fail("event");

    // persistent grids: as many blocks as stay resident on the device
    hipDeviceProp_t prop;
    hipGetDeviceProperties(&prop, l->device);
    l->cu_count = std::max(1, prop.multiProcessorCount);
    int nb = 0;
    hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, l->f_render, LENSED_RENDER_BS, 0);
    l->grid_render = std::max(1, nb) * l->cu_count;
    nb = 0;
    hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, l->f_conv, LENSED_CONV_BS, 48 * 1024);
    l->grid_conv = std::max(1, nb) * l->cu_count;
    nb = 0;
    hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, l->f_conv_small, LENSED_CONV_BS, 32 * 1024);
    l->grid_conv_small = std::max(1, nb) * l->cu_count;

    // capacities: max_batch candidates of every system at once
    for (const auto& S : l->sys) {
        l->cap_params += l->max_batch * S.pars.size();
        l->cap_blocks += l->max_batch * S.dwords;
        l->cap_model += l->max_batch * S.npix;
        // one partial per 8-row x 64-column block
        l->cap_partials += l->max_batch * ((S.height + 7) / 8) * ((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX);
        l->cap_out += l->max_batch;
        if (S.table) l->cap_tables += l->max_batch * LENSED_EPL_TABLE_F4;
        if (S.table || S.cull) l->cap_npre += l->max_batch * LENSED_NPRE_STRIDE(S.table ? S.nq : 0);
        l->cap_trace += l->max_batch * S.ntile_r * (LENSED_RENDER_BS / 64);
        l->cap_cull += l->max_batch * ((S.ntile_r + LENSED_CULL_GROUP - 1) / LENSED_CULL_GROUP);
    }
    size_t maxpix = 0, dark_parts = 0, max_parts = 1;
    for (auto& S : l->sys) {
        maxpix = std::max(maxpix, S.npix);
        S.dark_off = (long long)dark_parts;
        const size_t parts = ((S.height + 7) / 8) * ((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX);
        dark_parts += parts;
        max_parts = std::max(max_parts, parts);
    }
    if (hipMalloc(&l->d_image, image.size() * 4) != hipSuccess ||
        hipMalloc(&l->d_weight, weight.size() * 4) != hipSuccess ||
        hipMalloc(&l->d_psf, psf.size() * 4) != hipSuccess ||
        hipMalloc(&l->d_quad, quad.size() * 4) != hipSuccess ||
        hipMalloc(&l->d_params, std::max<size_t>(1, l->cap_params) * 4) != hipSuccess ||
        hipMalloc(&l->d_blocks, (l->cap_blocks + l->block_pad) * 4) != hipSuccess ||
        hipMalloc(&l->d_model, l->cap_model * 4) != hipSuccess ||
        hipMalloc(&l->d_err, maxpix * 4) != hipSuccess || hipMalloc(&l->d_conv, maxpix * 4) != hipSuccess ||
        hipMalloc(&l->d_chi2, maxpix * 4) != hipSuccess ||
        hipMalloc(&l->d_partials, l->cap_partials * 8) != hipSuccess ||
        hipMalloc(&l->d_dark, dark_parts * 8) != hipSuccess ||
        hipMalloc(&l->d_tables, std::max<size_t>(1, l->cap_tables) * 16) != hipSuccess ||
        hipMalloc(&l->d_npre, std::max<size_t>(1, l->cap_npre) * 16) != hipSuccess ||
        hipMalloc(&l->d_trace, std::max<size_t>(1, l->cap_trace) * 4) != hipSuccess ||
        hipMalloc(&l->d_live, live_capacity(l->cap_trace, l->cap_cull) * 4) != hipSuccess ||
        hipMalloc(&l->d_owner, 8) != hipSuccess || hipMemsetAsync(l->d_owner, 0xFF, 8, l->stream) != hipSuccess ||
        hipMalloc(&l->d_written, std::max<size_t>(1, l->cap_trace) * 4) != hipSuccess ||
        hipMalloc(&l->d_nodes, std::max<size_t>(1, l->cap_tables / LENSED_EPL_TABLE_F4 * LENSED_EPL_ROWS) *
                                   16) != hipSuccess ||
        hipMalloc(&l->d_flags, std::max<size_t>(1, l->cap_tables / LENSED_EPL_TABLE_F4) * 4) != hipSuccess ||
        hipHostMalloc(&l->h_flags, std::max<size_t>(1, l->cap_tables / LENSED_EPL_TABLE_F4) * 4,
                      hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc(&l->h_params, std::max<size_t>(1, l->cap_params) * 4, hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc(&l->h_logl, l->cap_out * 8, hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc(&l->h_partials, max_parts * 8, hipHostMallocDefault) != hipSuccess)
        return fail("out of device memory");
    // on the context's stream (which, being non-blocking, would not wait for
    // the null stream), complete before the host vectors go
    if (hipMemcpyAsync(l->d_image, image.data(), image.size() * 4, hipMemcpyHostToDevice, l->stream) != hipSuccess ||
        hipMemcpyAsync(l->d_weight, weight.data(), weight.size() * 4, hipMemcpyHostToDevice, l->stream) != hipSuccess ||
        hipMemcpyAsync(l->d_psf, psf.data(), psf.size() * 4, hipMemcpyHostToDevice, l->stream) != hipSuccess ||
        hipMemcpyAsync(l->d_quad, quad.data(), quad.size() * 4, hipMemcpyHostToDevice, l->stream) != hipSuccess)
        return fail("upload");
    // the data's chi^2 block partials for a model of 0, once (the data do
    // not change over the context's life)
    for (const auto& S : l->sys) {
        const float* img = l->d_image + S.image_off;
        const float* wgt = l->d_weight + S.image_off;
        int w = (int)S.width, h = (int)S.height, tx = (int)((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX);
        double* out = l->d_dark + S.dark_off;
        void* a[] = {&img, &wgt, &w, &h, &tx, &out};
        if (launch(l->f_dark, tx * ((h + 7) / 8), 64, 0, l->stream, a)) {
            std::string e = lsd::g_error;
            lensed_destroy(l);
            set_error(e);
            return nullptr;
        }
    }
    if (hipStreamSynchronize(l->stream) != hipSuccess) return fail("upload");
    // the entry point that allocates nothing: this device's static scratch
    // (its address, once per device), a layout per system and a pinned slot
    // for the launch descriptor
    if (scratch_setup(l->device, &l->scratch)) {
        std::string e = lsd::g_error;
        lensed_destroy(l);
        set_error(e);
        return nullptr;
    }
    if (hipHostMalloc(&l->h_desc, sizeof(lensed_desc), hipHostMallocDefault) != hipSuccess)
        return fail("pinned descriptor slot");
    if (l->emu_wf) {
        // the network, certified once per weights and bound per (q, t) cell
        std::vector<int> cells(emu::kCellsQ * emu::kCellsT, 0);
        l->emu_ncert = emu_certify(l->emu_wf, l->emu_wp, l->emu_tol, cells.data(), &l->emu_cert_err);
        if (l->emu_ncert < 0) return fail("emulator certification");
        if (hipMalloc(&l->d_cells, cells.size() * 4) != hipSuccess ||
            hipMemcpy(l->d_cells, cells.data(), cells.size() * 4, hipMemcpyHostToDevice) != hipSuccess)
            return fail("emulator cells");
    }
    l->noalloc.assign(l->sys.size(), Layout());
    return l;
}

void lensed_destroy(lensed* l) {
    if (!l) return;
    if (l->stream) hipStreamSynchronize(l->stream);
    for (auto& kv : l->layouts) free_layout(l, kv.second);
    void* bufs[] = {l->d_image, l->d_weight, l->d_psf, l->d_quad, l->d_params, l->d_blocks, l->d_model,
                    l->d_err, l->d_conv, l->d_chi2, l->d_partials, l->d_tables, l->d_nodes, l->d_npre,
                    l->d_flags, l->d_cells, l->emu_wf, l->emu_wp, l->d_trace, l->d_live, l->d_owner, l->d_written,
                    l->d_dark};
    for (void* b : bufs)
        if (b) hipFree(b);
    if (l->h_params) hipHostFree(l->h_params);
    if (l->h_logl) hipHostFree(l->h_logl);
    if (l->h_partials) hipHostFree(l->h_partials);
    if (l->h_planes) hipHostFree(l->h_planes);
    for (auto& e : l->ev_plane)
        if (e) hipEventDestroy(e);
    if (l->h_desc) hipHostFree(l->h_desc);
    if (l->h_flags) hipHostFree(l->h_flags);
    for (auto& e : l->ev)
        if (e) hipEventDestroy(e);
    if (l->stream) hipStreamDestroy(l->stream);
    if (l->module) hipModuleUnload(l->module);
    delete l;
}

size_t lensed_npars(const lensed* l, size_t s) { return (l && s < l->sys.size()) ? l->sys[s].pars.size() : 0; }
size_t lensed_ndims(const lensed* l, size_t s) { return (l && s < l->sys.size()) ? l->sys[s].ndims : 0; }

int lensed_pmap(const lensed* l, size_t s, size_t* pmap) {
    if (!l || s >= l->sys.size()) return -1;
    for (size_t i = 0; i < l->sys[s].pmap.size(); ++i) pmap[i] = l->sys[s].pmap[i];
    return 0;
}

long lensed_profile(const lensed* l, double* ms8) {
    if (!l) return -1;
    if (ms8)
        for (int i = 0; i < 8; ++i) ms8[i] = l->prof_ms[i];
    return l->prof_calls;
}

int lensed_set_tuning(lensed* l, const lensed_tuning* t) {
    if (!l) {
        set_error("invalid context");
        return -1;
    }
    lensed_tuning req{};
    if (t) req = *t;
    if ((req.conv_rows && req.conv_rows != LENSED_CONV_RY_SMALL && req.conv_rows != LENSED_CONV_RY &&
         req.conv_rows != LENSED_CONV_RY_TALL && req.conv_rows != LENSED_CONV_SWEEP) ||
        req.conv_order < 0 || req.conv_order > 2 || req.render_grid < 0 || req.cull_grid < 0 ||
        req.conv_grid < 0 || req.render_grid > 64 || req.cull_grid > 64 || req.conv_grid > 64 ||
        !std::isfinite(req.list_fraction)) {
        set_error("lensed_set_tuning: invalid launch shape");
        return -1;
    }
    req.default_ms = req.tuned_ms = 0;
    hipStreamSynchronize(l->stream);
    for (auto& kv : l->layouts) free_layout(l, kv.second);
    l->layouts.clear();
    l->tune_req = req;
    l->noalloc.assign(l->sys.size(), Layout());
    return 0;
}

int lensed_autotune_batch(lensed* l, size_t s, size_t* best_k, size_t* ks, double* rates, int* nk) {
    if (!l || s >= l->sys.size() || !best_k) {
        set_error("lensed_autotune_batch: invalid argument");
        return -1;
    }
    std::vector<size_t> kv;
    for (size_t k = 256; k <= l->max_batch && kv.size() < 31; k *= 2) kv.push_back(k);
    if (kv.empty() || kv.back() != l->max_batch) kv.push_back(l->max_batch);
    const size_t nd = l->sys[s].ndims, np = l->sys[s].pars.size();
    std::mt19937_64 g(20260101);
    std::uniform_real_distribution<double> u01(0, 1);
    std::vector<double> cubes(l->max_batch * nd), phys(l->max_batch * np), lnew(l->max_batch);
    for (auto& c : cubes) c = u01(g);
    std::vector<double> rate(kv.size(), 0.0);
    for (size_t i = 0; i < kv.size(); ++i) {
        double best = 1e300;
        for (int rep = 0; rep < 4; ++rep) {
            auto t0 = std::chrono::steady_clock::now();
            if (lensed_loglike_batch(l, s, cubes.data(), kv[i], phys.data(), lnew.data())) return -1;
            const double dt = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (rep > 0) best = std::min(best, dt);  // the first launch of a size builds (and tunes) it
        }
        rate[i] = kv[i] / best;
    }
    const double top = *std::max_element(rate.begin(), rate.end());
    size_t pick = kv.back();
    for (size_t i = 0; i < kv.size(); ++i)
        if (rate[i] >= 0.95 * top) {
            pick = kv[i];
            break;
        }
    *best_k = pick;
    if (nk) *nk = (int)kv.size();
    for (size_t i = 0; i < kv.size(); ++i) {
        if (ks) ks[i] = kv[i];
        if (rates) rates[i] = rate[i];
    }
    return 0;
}

int lensed_get_tuning(const lensed* l, lensed_tuning* t) {
    if (!l || !t) {
        set_error("invalid argument");
        return -1;
    }
    *t = l->last_layout ? l->last_layout->tune : l->tune_req;
    return 0;
}

int lensed_emulator_stats(const lensed* l, long* fallbacks, long* checked, double* max_err) {
    if (!l || !l->last_table_layout) {
        set_error("no emulated launch yet");
        return -1;
    }
    const int n = l->last_table_layout->n_tcands;
    long nf = n;
    if (l->emu_ncert > 0) {
        if (hipStreamSynchronize(l->stream) != hipSuccess) {
            set_error("cannot read emulator flags");
            return -1;
        }
        nf = 0;
        for (int i = 0; i < n; ++i) nf += l->h_flags[i] != 0;
    }
    if (fallbacks) *fallbacks = nf;
    if (checked) *checked = n;
    if (max_err) *max_err = l->emu_cert_err;
    return 0;
}

int lensed_emulator_cells(const lensed* l, long* ncells, long* ncertified, double* max_err) {
    if (!l || !l->emu_wf) {
        set_error("no emulator in this context");
        return -1;
    }
    if (ncells) *ncells = (long)emu::kCellsQ * emu::kCellsT;
    if (ncertified) *ncertified = l->emu_ncert;
    if (max_err) *max_err = l->emu_cert_err;
    return 0;
}

int lensed_emulator_rechecks(const lensed* l, long* rechecked, long* changed, double* max_abs_dlogl) {
    if (!l) {
        set_error("invalid context");
        return -1;
    }
    if (rechecked) *rechecked = l->emu_rechecked;
    if (changed) *changed = l->emu_changed;
    if (max_abs_dlogl) *max_abs_dlogl = l->emu_recheck_max;
    return 0;
}

int lensed_render_stats(const lensed* l, long* items, long* listed, long* quads, double* cull_ms) {
    if (!l || !l->last_layout) {
        set_error("no launch yet");
        return -1;
    }
    const Layout& L = *l->last_layout;
    const long n = L.n_blocks, per = LENSED_RENDER_BS / 64;  // (without a cull the items may be pixels in a row)
    long nl = n, nq = 16 * n;
    if (L.any_cull && (listed || quads)) {
        // the cull's list: quads (item * 4 + w) * 4 + q, sixteen to an entry,
        // -1 pads; the render traced them if it walked the list, else every
        // quad of each square holding one
        int count = 0;
        if (hipStreamSynchronize(l->stream) != hipSuccess ||
            hipMemcpy(&count, l->d_live, 4, hipMemcpyDeviceToHost) != hipSuccess || count < 0 ||
            count + 1 > (long)live_capacity(n * per, L.n_cull) || count % LENSED_LIST_ENTRY) {
            set_error("cannot read the render list");
            return -1;
        }
        std::vector<int> list(count);
        if (count && hipMemcpy(list.data(), l->d_live + 1, (size_t)count * 4, hipMemcpyDeviceToHost) != hipSuccess) {
            set_error("cannot read the render list");
            return -1;
        }
        std::vector<char> kept(n, 0), square(n * per, 0);
        long listed_quads = 0;
        for (int q : list) {
            if (q < 0) continue;
            if (q / 16 >= n) {
                set_error("render list holds an item out of range");
                return -1;
            }
            kept[q / 16] = 1;
            square[q / 4] = 1;
            ++listed_quads;
        }
        if (count < L.list_max) {
            nq = listed_quads;
        } else {
            nq = 0;
            for (char k : square) nq += 4 * k;
        }
        nl = 0;
        for (char k : kept) nl += k;
    }
    if (items) *items = n;
    if (listed) *listed = nl;
    if (quads) *quads = nq;
    if (cull_ms) *cull_ms = l->prof_cull_ms;
    return 0;
}

int lensed_results(const lensed* l, double* mean, double* sigma, double* ml, double* map, double* logev,
                   double* logev_err, double* max_loglike) {
    if (!l || l->sys.empty()) return -1;
    const System& S = l->sys[0];
    size_t n = S.pars.size();
    if (mean) memcpy(mean, S.mean.data(), n * 8);
    if (sigma) memcpy(sigma, S.sigma.data(), n * 8);
    if (ml) memcpy(ml, S.ml.data(), n * 8);
    if (map) memcpy(map, S.map.data(), n * 8);
    if (logev) *logev = S.logev;
    if (logev_err) *logev_err = S.logev_err;
    if (max_loglike) *max_loglike = S.max_loglike;
    return 0;
}

// unit cube -> physical parameters of system S, sampler order in/out,
// object order into phys; false if a value falls outside its hard bounds
static bool transform(const System& S, double* cube, size_t ndim, double* phys) {
    bool ok = true;
    for (size_t i = 0; i < S.pars.size(); ++i) {
        double unit = i < ndim ? cube[i] : 0.5;
        const Param& P = S.pars[S.pmap[i]];
        double v = prior_apply(&P.pri_copy, unit);
        if (P.bounded && (v < P.lower || v > P.upper)) ok = false;
        cube[i] = v;
        phys[S.pmap[i]] = v;
    }
    return ok;
}

void loglike(double cube[], int* ndim, int* npar, double* lnew, void* lensed_) {
    ::lensed* l = (::lensed*)lensed_;
    const System& S = l->sys[0];
    std::vector<double> phys(S.pars.size());
    (void)npar;
    bool ok = transform(S, cube, (size_t)*ndim, phys.data());
    if (!ok) {
        *lnew = -DBL_MAX;
        return;
    }
    std::vector<size_t> nc(l->sys.size(), 0);
    nc[0] = 1;
    std::vector<const double*> p(l->sys.size(), nullptr);
    p[0] = phys.data();
    std::vector<double*> o(l->sys.size(), nullptr);
    o[0] = lnew;
    if (evaluate(l, nc, p, o, true)) {
        fprintf(stderr, "lensed: loglike failed: %s\n", lsd::g_error.c_str());
        *lnew = -DBL_MAX;
    }
}

int lensed_loglike_batch(lensed* l, size_t s, const double* cubes, size_t ncand, double* phys_out,
                         double* lnew_out) {
    if (!l || s >= l->sys.size()) {
        set_error("invalid context or system");
        return -1;
    }
    System& S = l->sys[s];
    size_t np = S.pars.size(), nd = S.ndims;
    std::vector<double> cube(np), phys;
    std::vector<char> ok(std::min(ncand, l->max_batch)), used;
    if (!S.xfast) phys.resize(std::min(ncand, l->max_batch) * np);
    for (size_t c0 = 0; c0 < ncand; c0 += l->max_batch) {
        size_t nc = std::min(l->max_batch, ncand - c0);
        std::vector<size_t> ncv(l->sys.size(), 0);
        ncv[s] = nc;
        std::vector<const double*> p(l->sys.size(), nullptr);
        if (S.xfast) {
            // uniform and delta priors: the same values as prior_apply, staged
            // as floats (object order) straight into the pinned parameters
            Layout* L = get_layout(l, ncv, true);
            if (!L) return -1;
            long long off = -1;
            for (size_t k = 0; k < L->desc.size(); ++k)
                if (L->sys_of_desc[k] == (int)s) off = L->desc[k].param_off;
            if (off < 0) {
                set_error("lensed_loglike_batch: no launch descriptor for the system");
                return -1;
            }
            const double *xa = S.xa.data(), *xs = S.xs.data(), *xlo = S.xlo.data(), *xhi = S.xhi.data();
            const char* xd = S.xdelta.data();
            const size_t* dst = S.pmap.data();
            for (size_t c = 0; c < nc; ++c) {
                const double* u = cubes + (c0 + c) * nd;
                double* po = phys_out ? phys_out + (c0 + c) * np : cube.data();
                float* h = l->h_params + off + (long long)(c * np);
                bool good = true;
                for (size_t i = 0; i < np; ++i) {
                    const double v = xd[i] ? xa[i] : xa[i] + (i < nd ? u[i] : 0.5) * xs[i];
                    good &= !(v < xlo[i] || v > xhi[i]);
                    po[i] = v;
                    h[dst[i]] = (float)v;
                }
                ok[c] = good;
            }
        } else {
            for (size_t c = 0; c < nc; ++c) {
                for (size_t i = 0; i < nd; ++i) cube[i] = cubes[(c0 + c) * nd + i];
                ok[c] = transform(S, cube.data(), nd, phys.data() + c * np);
                if (phys_out) memcpy(phys_out + (c0 + c) * np, cube.data(), np * 8);
            }
            p[s] = phys.data();
        }
        std::vector<double*> o(l->sys.size(), nullptr);
        o[s] = lnew_out + c0;
        if (evaluate(l, ncv, p, o)) return -1;
        for (size_t c = 0; c < nc; ++c)
            if (!ok[c]) lnew_out[c0 + c] = -DBL_MAX;
        if (!S.emu_used.empty()) {
            used.resize(c0, 0);
            used.insert(used.end(), S.emu_used.begin(), S.emu_used.end());
        }
    }
    if (!used.empty()) used.resize(ncand, 0);
    S.emu_used = used;  // for recheck_emulated()
    return 0;
}

int lensed_loglike_batch_noalloc(lensed* l, size_t s, const double* cubes, size_t ncand, double* phys_out,
                                 double* lnew_out) {
    if (!l || s >= l->sys.size() || !cubes || !lnew_out || ncand == 0) {
        set_error("lensed_loglike_batch_noalloc: invalid argument");
        return -1;
    }
    if (!l->scratch || s >= l->noalloc.size()) {
        set_error("lensed_loglike_batch_noalloc: no static scratch on this device");
        return -1;
    }
    const System& S = l->sys[s];
    const size_t np = S.pars.size(), nd = S.ndims;
    constexpr size_t kMaxPars = 256;
    if (np > kMaxPars) {
        set_error("lensed_loglike_batch_noalloc: more than 256 parameters");
        return -1;
    }
    if (ncand > l->max_batch) {
        set_error("lensed_loglike_batch_noalloc: more candidates than the context's max_batch");
        return -1;
    }
    // carve the scratch for ncand candidates at 256-byte boundaries
    const size_t nc = ncand;
    const size_t squares = nc * (size_t)S.ntile_r * (LENSED_RENDER_BS / 64);
    const size_t npart = ((S.height + 7) / 8) * ((S.width + LENSED_CONV_TX - 1) / LENSED_CONV_TX);
    size_t offs[11], total = 0;
    auto carve = [&](bool cull) {
        const size_t sizes[] = {sizeof(lensed_desc),
                                nc * np * 4,
                                (nc * S.dwords + 256) * 4,
                                S.table || cull ? nc * LENSED_NPRE_STRIDE(S.table ? S.nq : 0) * 16 : 16,
                                S.table ? nc * LENSED_EPL_TABLE_F4 * 16 : 16,
                                nc * S.npix * 4,
                                nc * npart * 8,
                                squares * 4,
                                live_capacity(squares, nc * ((S.ntile_r + LENSED_CULL_GROUP - 1) / LENSED_CULL_GROUP)) * 4,
                                squares * 4,
                                8};
        total = 0;
        for (int i = 0; i < 11; ++i) {
            offs[i] = total;
            total += (sizes[i] + 255) / 256 * 256;
        }
        // the words read past the last object block may be those of what follows it
        total = std::max(total, offs[2] + (nc * S.dwords + l->block_pad) * 4);
        return total <= LENSED_SCRATCH_BYTES;
    };
    // a system without a table does without the cull where its constants
    // would be what does not fit
    const bool cull = carve(S.cull);
    if (!cull && (S.table || !S.cull || !carve(false))) {
        const size_t per = (total - offs[1]) / nc + 1;
        char b[200];
        snprintf(b, sizeof b,
                 "lensed_loglike_batch_noalloc: %zu candidates need %zu bytes of the %llu-byte static scratch "
                 "(at most about %zu at this image size)",
                 ncand, total, (unsigned long long)LENSED_SCRATCH_BYTES, (size_t)(LENSED_SCRATCH_BYTES / per));
        set_error(b);
        return -1;
    }
    unsigned char* base = (unsigned char*)l->scratch;
    Buffers B;
    B.desc = (lensed_desc*)(base + offs[0]);
    B.params = (float*)(base + offs[1]);
    B.blocks = (unsigned*)(base + offs[2]);
    B.npre = base + offs[3];
    B.tables = base + offs[4];
    B.model = (float*)(base + offs[5]);
    B.partials = (double*)(base + offs[6]);
    B.trace = (int*)(base + offs[7]);
    B.live = (int*)(base + offs[8]);
    B.written = (int*)(base + offs[9]);
    B.owner = (int*)(base + offs[10]);
    B.emulate = false;  // exact-series tables
    B.record = false;   // the context's own statistics are left alone
    // the launch layout of this count (a single system's offsets into its
    // buffers are all zero), kept for calls of the same count
    Layout& L = l->noalloc[s];
    if (L.n_final != (int)nc) {
        std::vector<size_t> ncv(l->sys.size(), 0);
        ncv[s] = nc;
        L = Layout();
        if (build_layout(l, ncv, L, cull)) {
            L = Layout();
            return -1;
        }
        L.id = -2;  // never the id a fill of `owner` leaves (-1)
    }
    const lensed_desc& d = L.desc[0];
    // parameters into the pinned staging; out-of-bounds draws flagged in lnew_out
    double cube[kMaxPars];
    for (size_t c = 0; c < nc; ++c) {
        for (size_t i = 0; i < nd; ++i) cube[i] = cubes[c * nd + i];
        bool ok = true;
        for (size_t i = 0; i < np; ++i) {
            double unit = i < nd ? cube[i] : 0.5;
            const Param& P = S.pars[S.pmap[i]];
            double v = prior_apply(&P.pri_copy, unit);
            if (P.bounded && (v < P.lower || v > P.upper)) ok = false;
            cube[i] = v;
            l->h_params[c * np + S.pmap[i]] = (float)v;
        }
        if (phys_out) memcpy(phys_out + c * np, cube, np * 8);
        lnew_out[c] = ok ? 0.0 : -DBL_MAX;
    }
    *l->h_desc = d;
    hipStream_t st = l->stream;
    LSD_HIP(hipMemcpyAsync(B.desc, l->h_desc, sizeof(lensed_desc), hipMemcpyHostToDevice, st));
    // the scratch keeps the previous call's contents (of any context): the
    // cull may not trust its record of written squares, so `owner` is reset
    LSD_HIP(hipMemsetAsync(B.owner, 0xFF, 8, st));
    if (enqueue_chain(l, L, B, false, nullptr, nullptr, nullptr)) return -1;
    LSD_HIP(hipStreamSynchronize(st));
    finish_single(l, L);
    for (size_t c = 0; c < nc; ++c)
        if (lnew_out[c] == 0.0) lnew_out[c] = l->h_logl[c];
    return 0;
}

int lensed_loglike_systems(lensed* l, const double* const* phys, const size_t* ncand, double* const* lnew) {
    if (!l) {
        set_error("invalid context");
        return -1;
    }
    std::vector<size_t> nc(ncand, ncand + l->sys.size());
    std::vector<const double*> p(phys, phys + l->sys.size());
    std::vector<double*> o(lnew, lnew + l->sys.size());
    return evaluate(l, nc, p, o, true);
}

int lensed_render(lensed* l, size_t s, const double* phys, float* value, float* error, float* image, float* chi2) {
    if (!l || s >= l->sys.size()) {
        set_error("invalid context or system");
        return -1;
    }
    const System& S = l->sys[s];
    std::vector<size_t> nc(l->sys.size(), 0);
    nc[s] = 1;
    Layout* L = get_layout(l, nc);
    if (!L) return -1;
    for (size_t i = 0; i < S.pars.size(); ++i) l->h_params[i] = (float)phys[i];
    if (enqueue_chain(l, *L, context_buffers(l, *L), false, l->d_err, l->d_conv, l->d_chi2)) return -1;
    // The planes by way of a pinned buffer, each moved on to the caller's
    // pages while the next one crosses the bus (four copies to pageable
    // memory took 230 us for 512 x 512, 83 us pinned, the moves 15 us each).
    const size_t nb = S.npix * 4;
    float* out[4] = {value, error, image, chi2};
    const float* from[4] = {l->d_model, l->d_err, l->d_conv, l->d_chi2};
    if (!l->h_planes) {
        size_t most = 0;
        for (const auto& s2 : l->sys) most = std::max(most, s2.npix);
        LSD_HIP(hipHostMalloc(&l->h_planes, 4 * most * 4, hipHostMallocDefault));
    }
    for (int i = 0; i < 4; ++i) {
        if (!out[i]) continue;
        if (!l->ev_plane[i]) LSD_HIP(hipEventCreateWithFlags(&l->ev_plane[i], hipEventDisableTiming));
        LSD_HIP(hipMemcpyAsync(l->h_planes + i * S.npix, from[i], nb, hipMemcpyDeviceToHost, l->stream));
        LSD_HIP(hipEventRecord(l->ev_plane[i], l->stream));
    }
    for (int i = 0; i < 4; ++i) {
        if (!out[i]) continue;
        LSD_HIP(hipEventSynchronize(l->ev_plane[i]));
        memcpy(out[i], l->h_planes + i * S.npix, nb);
    }
    LSD_HIP(hipStreamSynchronize(l->stream));
    return 0;
}

void dumper(int* nsamples, int* nlive, int* npar, double** physlive, double** posterior, double** constraints,
            double* maxloglike, double* logz, double* inslogz, double* logzerr, void* lensed_) {
    enum { MEAN, SIGMA, ML, MAP };
    (void)nsamples; (void)nlive; (void)physlive; (void)posterior;
    ::lensed* l = (::lensed*)lensed_;
    System& S = l->sys[0];
    size_t n = (size_t)*npar;
    for (size_t i = 0; i < n && i < S.pmap.size(); ++i) {
        size_t p = S.pmap[i];
        S.mean[p] = constraints[0][MEAN * n + i];
        S.sigma[p] = constraints[0][SIGMA * n + i];
        S.ml[p] = constraints[0][ML * n + i];
        S.map[p] = constraints[0][MAP * n + i];
    }
    S.logev = *logz;
    S.logev_err = *logzerr;
    S.logev_ins = *inslogz;
    S.max_loglike = *maxloglike;
    // the layers at the maximum-likelihood point, as src/nested.c:169-226
    if (!l->output.empty() && lensed_write_layers(l, 0, S.ml.data(), l->output.c_str()))
        fprintf(stderr, "lensed: cannot write %s: %s\n", l->output.c_str(), lsd::g_error.c_str());
}

int lensed_write_paramfiles(const lensed* l, size_t s, const char* root) {
    if (!l || s >= l->sys.size() || !root) {
        set_error("lensed_write_paramfiles: invalid argument");
        return -1;
    }
    const System& S = l->sys[s];
    std::string pn = std::string(root) + ".paramnames", rn = std::string(root) + ".ranges";
    FILE* fp = fopen(pn.c_str(), "w");
    FILE* fr = fopen(rn.c_str(), "w");
    if (!fp || !fr) {
        if (fp) fclose(fp);
        if (fr) fclose(fr);
        set_error("could not write " + (fp ? rn : pn));
        return -1;
    }
    for (size_t i = 0; i < S.pmap.size(); ++i) {
        const Param& P = S.pars[S.pmap[i]];
        double lo = prior_lower(&P.pri_copy), hi = prior_upper(&P.pri_copy);
        fprintf(fp, "%-20s  %s\n", P.id.c_str(), P.label.c_str());
        fprintf(fr, "%-20s  ", P.id.c_str());
        if (std::isfinite(lo)) fprintf(fr, "%10.4f  ", lo);
        else fprintf(fr, "%10s  ", "N");
        if (std::isfinite(hi)) fprintf(fr, "%10.4f\n", hi);
        else fprintf(fr, "%10s\n", "N");
    }
    bool ok = fclose(fp) == 0;
    ok = fclose(fr) == 0 && ok;
    if (!ok) {
        set_error("could not write " + pn);
        return -1;
    }
    return 0;
}

int lensed_set_output(lensed* l, const char* path) {
    if (!l) {
        set_error("invalid context");
        return -1;
    }
    l->output = path ? path : "";
    return 0;
}

int lensed_write_layers(lensed* l, size_t s, const double* phys, const char* path) {
    if (!l || s >= l->sys.size() || !phys || !path) {
        set_error("lensed_write_layers: invalid argument");
        return -1;
    }
    const System& S = l->sys[s];
    size_t n = S.npix;
    std::vector<float> value(n), error(n), image(n), chi2(n);
    if (lensed_render(l, s, phys, value.data(), error.data(), image.data(), chi2.data())) return -1;
    std::vector<float> res(n), relerr(n), pvalue(n);
    for (size_t i = 0; i < n; ++i) {
        res[i] = S.h_image[i] - image[i];
        relerr[i] = error[i] / value[i];
        pvalue[i] = (float)std::erfc(std::sqrt(0.5 * chi2[i]));
    }
    const float* layers[6] = {image.data(), res.data(), value.data(), relerr.data(), S.h_weight.data(),
                              pvalue.data()};
    const char* names[6] = {"IMG", "RES", "RAW", "ERR", "WHT", "PVL"};
    return lensed_fits_write(path, S.width, S.height, 6, layers, names);
}

}  // extern "C"
