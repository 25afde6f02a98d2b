// kfa_rtc.hip -- compiled row kernels for lengths outside the built-in registry.
//
// The built-in registry (kfa_fast_reg.hip) instantiates the compile-time Stockham kernel
// k_fast (kfa_fast.hpp) for the lengths of the reference's workloads.  Any other length
// whose line fits one LDS line and whose radices are 2, 3, 4 or 5 (kf_factor's schedule,
// kiss_fft.c:306-328; float may also regroup the powers of two into radix 8 / 16, and
// takes the odd radices 7, 11 and 13 as well, real and long rows those up to 31) gets the same kernel compiled at run time, on
// first use, with the HIP runtime compiler:
//   * fixed point keeps the plan's own radix schedule (its rounding is part of the result);
//     float takes a schedule of large radices (16s, then 8 / 4 / 2, then 5s and 3s, then
//     7s, 11s and 13s);
//   * a few thread shapes (threads per line, lines per workgroup) are compiled and the
//     engine's first-use timing picks one, as for the built-in variants;
//   * the kernel sources are the engine's own headers, embedded in the library at build
//     time (kfa_rtc_headers.cpp, generated by kissfft_amd/build.py);
//   * code objects are kept in memory for the process and on disk (KISSFFT_AMD_CACHE, else
//     $XDG_CACHE_HOME/kissfft_amd or ~/.cache/kissfft_amd), keyed by a hash of the source,
//     the options and the device architecture; KISSFFT_AMD_RTC=0 turns the path off;
//   * a kernel that would use scratch memory (spilled registers) is not used;
//   * complex lines shorter than 16 points (KISSFFT_AMD_RTC_MIN) keep the general kernel, and so
//     do real rows of a half length below 4; half lengths of 4 .. 15 are compiled when there
//     is a batch of them (real 15x90x16 x1277 both ways: Q15 518 -> 218 us, float 585 -> 329).
// The tile kernel k_tile (kfa_tile.hpp) is compiled the same way for the strided lines of
// N-D axes without a built-in tile, all three scalar kinds, in one shape chosen by rule
// (tile_shapes), so an axis costs one compilation per direction.  Against the general line
// kernel: Q15 64x96x120 x16 500 -> 63 us, float 24x25x128 x93 252 -> 53 us, Q31 real
// 45x48x120 x61 there and back 722 -> 193 us.
// The tuned choice of every (device, scalar kind, transform kind, length, direction,
// timing batch) is kept in a table on disk beside the code objects (tuned.txt, or
// KISSFFT_AMD_TUNE_TABLE; "0" turns it off), so later processes skip the timing.
// The runtime compiler library is loaded with dlopen (libhiprtc), so the library links
// nothing new; without it these lengths keep the general line kernel.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <dlfcn.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <map>
#include <memory>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "../kfa_engine.h"
#include "kfa_fast.hpp"
#include "kfa_internal.hpp"
#include "kfa_plane.hpp"
#include "kfa_tile.hpp"

// embedded header sources (generated at build time)
extern "C" const int kfa_rtc_nheaders;
extern "C" const char *const kfa_rtc_header_names[];
extern "C" const char *const kfa_rtc_header_srcs[];

namespace kfa {

namespace {

struct Rtc {
    bool tried = false, ok = false;
    decltype(&hiprtcCreateProgram) create = nullptr;
    decltype(&hiprtcAddNameExpression) add_name = nullptr;
    decltype(&hiprtcCompileProgram) compile = nullptr;
    decltype(&hiprtcGetProgramLogSize) log_size = nullptr;
    decltype(&hiprtcGetProgramLog) get_log = nullptr;
    decltype(&hiprtcGetLoweredName) lowered = nullptr;
    decltype(&hiprtcGetCodeSize) code_size = nullptr;
    decltype(&hiprtcGetCode) get_code = nullptr;
    decltype(&hiprtcDestroyProgram) destroy = nullptr;
};

std::mutex g_rtc_mu;  // guards everything below
Rtc g_rtc;

bool rtc_load()
{
    if (g_rtc.tried)
        return g_rtc.ok;
    g_rtc.tried = true;
    void *h = nullptr;
    for (const char *name : {"libhiprtc.so.7", "libhiprtc.so", "/opt/rocm/lib/libhiprtc.so"})
        if ((h = dlopen(name, RTLD_NOW | RTLD_LOCAL)))
            break;
    if (!h)
        return false;
    auto sym = [&](auto &f, const char *n) { f = reinterpret_cast<std::decay_t<decltype(f)>>(dlsym(h, n)); };
    sym(g_rtc.create, "hiprtcCreateProgram");
    sym(g_rtc.add_name, "hiprtcAddNameExpression");
    sym(g_rtc.compile, "hiprtcCompileProgram");
    sym(g_rtc.log_size, "hiprtcGetProgramLogSize");
    sym(g_rtc.get_log, "hiprtcGetProgramLog");
    sym(g_rtc.lowered, "hiprtcGetLoweredName");
    sym(g_rtc.code_size, "hiprtcGetCodeSize");
    sym(g_rtc.get_code, "hiprtcGetCode");
    sym(g_rtc.destroy, "hiprtcDestroyProgram");
    g_rtc.ok = g_rtc.create && g_rtc.add_name && g_rtc.compile && g_rtc.log_size && g_rtc.get_log &&
               g_rtc.lowered && g_rtc.code_size && g_rtc.get_code && g_rtc.destroy;
    return g_rtc.ok;
}

std::string cache_dir()
{
    if (const char *v = getenv("KISSFFT_AMD_CACHE"))
        return v;
    if (const char *v = getenv("XDG_CACHE_HOME"))
        return std::string(v) + "/kissfft_amd";
    if (const char *v = getenv("HOME"))
        return std::string(v) + "/.cache/kissfft_amd";
    return "";
}

uint64_t fnv1a(const std::string &s, uint64_t h = 1469598103934665603ULL)
{
    for (unsigned char c : s) {
        h ^= c;
        h *= 1099511628211ULL;
    }
    return h;
}

// the current device, for the in-process caches of loaded kernels (a loaded module
// belongs to the device that was current when it was loaded)
int current_dev()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return dev;
}

std::string arch_name()
{
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
        (void)hipGetLastError();
        return "gfx950";
    }
    return prop.gcnArchName;
}

// One runtime-compiled variant: its registry entry and its loaded kernel.
struct RtcVariant {
    FastVariant v;
    std::string name;
    hipModule_t mod = nullptr;
    hipFunction_t fn = nullptr;
    size_t lds = 0;
};

std::map<std::string, std::unique_ptr<RtcVariant>> g_variants;  // by name expression, arch, device

// Compiles (or reads from the disk cache) the kernel `expr` of source `src`; 0 on success.
int build_kernel(const std::string &expr, const std::string &arch, std::string &code, std::string &lowered,
                 const std::string &src)
{
    const std::vector<std::string> opts = {"--offload-arch=" + arch, "-O3", "-std=c++17", "-Xclang",
                                           "-target-feature", "-Xclang", "-packed-fp32-ops"};
    std::string key = src + "|" + expr + "|" + arch;
    for (const auto &o : opts)
        key += "|" + o;
    for (int i = 0; i < kfa_rtc_nheaders; ++i)
        key += kfa_rtc_header_srcs[i];
    char hx[32];
    snprintf(hx, sizeof hx, "%016llx", (unsigned long long)fnv1a(key));
    const std::string dir = cache_dir();
    const std::string path = dir.empty() ? "" : dir + "/rtc-" + hx + ".co";
    const std::string lpath = dir.empty() ? "" : dir + "/rtc-" + hx + ".name";
    if (!path.empty()) {
        std::ifstream f(path, std::ios::binary), fl(lpath);
        if (f && fl) {
            std::ostringstream ss, sl;
            ss << f.rdbuf();
            sl << fl.rdbuf();
            code = ss.str();
            lowered = sl.str();
            if (!code.empty() && !lowered.empty())
                return 0;
        }
    }
    if (!rtc_load())
        return fail(-2, "runtime compiler (libhiprtc) not available");
    hiprtcProgram prog;
    if (g_rtc.create(&prog, src.c_str(), "kfa_rtc.hip", kfa_rtc_nheaders, kfa_rtc_header_srcs,
                     kfa_rtc_header_names) != HIPRTC_SUCCESS)
        return fail(-3, "hiprtcCreateProgram failed");
    int rc = 0;
    std::vector<const char *> o;
    for (const auto &s : opts)
        o.push_back(s.c_str());
    if (g_rtc.add_name(prog, expr.c_str()) != HIPRTC_SUCCESS ||
        g_rtc.compile(prog, (int)o.size(), o.data()) != HIPRTC_SUCCESS) {
        size_t n = 0;
        g_rtc.log_size(prog, &n);
        std::string log(n, '\0');
        if (n)
            g_rtc.get_log(prog, &log[0]);
        rc = fail(-3, "runtime compilation of %s failed: %.300s", expr.c_str(), log.c_str());
    } else {
        const char *ln = nullptr;
        size_t n = 0;
        if (g_rtc.lowered(prog, expr.c_str(), &ln) != HIPRTC_SUCCESS || !ln ||
            g_rtc.code_size(prog, &n) != HIPRTC_SUCCESS || n == 0) {
            rc = fail(-3, "runtime compilation of %s: no code", expr.c_str());
        } else {
            lowered = ln;
            code.assign(n, '\0');
            if (g_rtc.get_code(prog, &code[0]) != HIPRTC_SUCCESS)
                rc = fail(-3, "runtime compilation of %s: no code", expr.c_str());
        }
    }
    g_rtc.destroy(&prog);
    if (rc == 0 && !path.empty()) {  // best effort; another process may write the same file
        (void)mkdir(dir.c_str(), 0755);
        const std::string tmp = path + "." + std::to_string((long long)getpid());
        const std::string ltmp = lpath + "." + std::to_string((long long)getpid());
        {
            std::ofstream f(tmp, std::ios::binary), fl(ltmp);
            f << code;
            fl << lowered;
        }
        (void)rename(ltmp.c_str(), lpath.c_str());
        (void)rename(tmp.c_str(), path.c_str());
    }
    return rc;
}

int rtc_launch(const FastVariant &fv, const FastArgs &a, hipStream_t s)
{
    const RtcVariant *rv = static_cast<const RtcVariant *>(fv.rtc);
    const long long blocks = (a.nlines + fv.LPB - 1) / fv.LPB;
    if (blocks <= 0)
        return 0;
    if (blocks > 0x7fffffffLL)
        return -2;
    FastArgs copy = a;
    void *params[] = {&copy};
    return hipModuleLaunchKernel(rv->fn, (unsigned)blocks, 1, 1, fv.T * fv.LPB, 1, 1, (unsigned)rv->lds, s, params,
                                 nullptr) == hipSuccess
               ? 0
               : -3;
}

// The arithmetic of a variant: Q15 complex lines use the packed-word butterflies; the real
// kinds' split / merge pass is written for the unpacked form.
const char *arith_name(int type, int kind)
{
    if (type == KFA_F32)
        return "kfa::F32";
    if (type == KFA_Q31)
        return "kfa::Q31";
    return kind == FK_C2C ? "kfa::Q15P" : "kfa::Q15";
}

std::map<std::string, std::string> g_tuned;  // tuned-choice table: key -> variant name
bool g_tuned_loaded = false;

std::string tuned_path()
{
    const char *v = getenv("KISSFFT_AMD_TUNE_TABLE");
    if (v && *v)
        return (v[0] == '0' && !v[1]) ? "" : v;
    const std::string d = cache_dir();
    return d.empty() ? "" : d + "/tuned.txt";
}

void tuned_load()
{
    if (g_tuned_loaded)
        return;
    g_tuned_loaded = true;
    const std::string path = tuned_path();
    if (path.empty())
        return;
    std::ifstream f(path);
    std::string line;
    while (std::getline(f, line)) {  // "<key fields> = <variant name>"
        const size_t eq = line.find(" = ");
        if (eq != std::string::npos)
            g_tuned[line.substr(0, eq)] = line.substr(eq + 3);
    }
}

// Builds and loads kernel `expr` of source `src`; 0 when it runs without scratch memory.
int load_kernel(const std::string &expr, const std::string &arch, const std::string &src, hipModule_t *mod,
                hipFunction_t *fn)
{
    std::string code, lowered;
    int scratch = 0;
    *mod = nullptr;
    if (build_kernel(expr, arch, code, lowered, src) == 0 && hipModuleLoadData(mod, code.data()) == hipSuccess &&
        hipModuleGetFunction(fn, *mod, lowered.c_str()) == hipSuccess &&
        hipFuncGetAttribute(&scratch, HIP_FUNC_ATTRIBUTE_LOCAL_SIZE_BYTES, *fn) == hipSuccess && scratch == 0)
        return 0;
    (void)hipGetLastError();
    if (*mod)
        (void)hipModuleUnload(*mod);
    *mod = nullptr;
    if (env_flag("KISSFFT_AMD_VERBOSE", false))
        fprintf(stderr, "[kissfft_amd] runtime kernel %s unusable (scratch %d): %s\n", expr.c_str(), scratch,
                kfa_last_error());
    return -3;
}

// One runtime-compiled tile: its variant and its loaded kernel.
struct RtcTile {
    TileVariant v;
    std::string name;
    hipModule_t mod = nullptr;
    hipFunction_t fn = nullptr;
};

std::map<std::string, std::unique_ptr<RtcTile>> g_tiles;  // by name expression, arch, device

// Shapes of a tile of n-point lines, cb bytes a value, preferred first.
struct TileShape {
    int T, TL;
    bool half;
};

// Threads per line: the count that leaves the fewest idle butterfly slots over the stages
// (T * sum of ceil(n / p / T) * p), with at most `most` values per thread in any stage.
int tile_threads(int n, const std::vector<int> &rad, int TL, int most)
{
    int best = 0;
    double best_cost = 0;
    for (int T = 1; T <= n && T * TL <= 1024; ++T) {
        long long slots = 0;
        int widest = 0;
        for (int p : rad) {
            const int el = (n / p + T - 1) / T * p;
            slots += el;
            widest = std::max(widest, el);
        }
        if (widest > most && widest > *std::max_element(rad.begin(), rad.end()))
            continue;
        // whole waves; fewer values per thread cost an address each
        const int waves = (T * TL + 63) / 64;
        const double cost = (double)slots * waves * 64 / TL * (widest < 8 ? 1.1 : 1.0);
        if (!best || cost < 0.995 * best_cost) {
            best = T;
            best_cost = cost;
        }
    }
    return best;
}

// Rows of a full 128-byte line wherever LDS holds two such workgroups per CU: whole values,
// else one component at a time (8-byte values only: Q15 moves packed words), else rows half
// as long, and so on.  Short lines take more lines, up to 256 threads.
std::vector<TileShape> tile_shapes(int n, const std::vector<int> &rad, int type, bool rows)
{
    const int cb = type == KFA_Q15 ? 4 : 8;
    const size_t room = 78 * 1024;
    std::vector<TileShape> out;
    auto fits = [&](int TL, int slot) {
        const bool padded = !rows && slot == 8 && TL * slot < 128 && rad.back() % 2 == 0;  // TilePos
        return (size_t)(padded ? n + n / rad.back() : n) * (TL + (rows ? 1 : 0)) * slot <= room;
    };
    for (int TL = 128 / cb; TL >= 1 && out.size() < 3; TL /= 2)
        for (int half = 0; half < (cb == 8 && rad.size() > 1 ? 2 : 1); ++half) {
            if (!fits(TL, half ? 4 : cb))
                continue;
            // half: two workgroups of 1024 threads have 64 registers, 16 values a thread (Q31,
            // whose products take register pairs, spills above 10)
            int tl = TL, T = tile_threads(n, rad, tl, half && type == KFA_Q31 ? 10 : 16);
            if (!T && !half)
                T = tile_threads(n, rad, tl, 32);
            if (!T)
                continue;
            while (!half && T * tl < 256 && (size_t)n * (2 * tl + 1) * cb <= 40 * 1024)
                tl *= 2;
            out.push_back({tl == TL ? T : std::max(1, tile_threads(n, rad, tl, 16)), tl, half != 0});
            if (!half)
                break;
        }
    return out;
}

}  // namespace

// float: 16s, then one 8 / 4 / 2 for the rest of the power of two, then 5s, then 3s, then
// the generic odd radices from 7 to pmax (kfa_fast.hpp's Dft<P>); empty for other factors.
// tile: the odd radices first, which leaves more of the twiddles of the others exact (half of a
// four-step split of 746496 = 864^2: 1.69e-7 rel-L2 against 1.81e-7 with the order of the rows,
// and as fast), and 8 and 4 in the place of a 16 and a 2 (a stage of radix 2 would move
// the tile through LDS for little work).
std::vector<int> float_schedule(int n, bool tile, int pmax)
{
    int a = 0, b = 0, c = 0;
    while (n % 2 == 0) {
        n /= 2;
        ++a;
    }
    while (n % 3 == 0) {
        n /= 3;
        ++b;
    }
    while (n % 5 == 0) {
        n /= 5;
        ++c;
    }
    std::vector<int> g;
    for (int p : {7, 11, 13, 17, 19, 23, 29, 31})
        while (p <= pmax && n % p == 0) {
            n /= p;
            g.push_back(p);
        }
    std::vector<int> r;
    if (n != 1)
        return r;
    for (; a >= 4 && !(tile && a == 5); a -= 4)
        r.push_back(16);
    if (a == 5) {
        r.push_back(8);
        a = 2;
    }
    if (a)
        r.push_back(1 << a);
    if (!tile) {
        r.insert(r.end(), c, 5);
        r.insert(r.end(), b, 3);
        r.insert(r.end(), g.begin(), g.end());
        return r;
    }
    g.insert(g.end(), b, 3);
    g.insert(g.end(), c, 5);
    g.insert(g.end(), r.begin(), r.end());
    return g;
}

int tile_launch(const TileVariant &v, const TileArgs &a, long long blocks, hipStream_t s)
{
    if (!v.rtc)
        return v.launch(a, blocks, s);
    if (blocks <= 0)
        return 0;
    TileArgs copy = a;
    void *params[] = {&copy};
    return hipModuleLaunchKernel(static_cast<const RtcTile *>(v.rtc)->fn, (unsigned)blocks, 1, 1, v.T * v.TL, 1, 1, 0,
                                 s, params, nullptr) == hipSuccess
               ? 0
               : -3;
}

const TileVariant *rtc_tile(int type, const std::vector<int> &radices, int inverse, int tm)
{
    if (!env_flag("KISSFFT_AMD_RTC", true) || radices.empty() || ((tm & TM_ROWS) && radices.size() < 2))
        return nullptr;
    long long n = 1;
    bool generic = false;
    for (int p : radices) {
        if (!(p == 2 || p == 3 || p == 4 || p == 5 || p == 7 || p == 11 || p == 13 ||
              (type == KFA_F32 && (p == 8 || p == 16))))
            return nullptr;
        generic |= p == 7 || p == 11 || p == 13;
        n *= p;
        if (n > 16384)
            return nullptr;
    }
    const std::string arch = arch_name();
    std::lock_guard<std::mutex> g(g_rtc_mu);
    // Q15: packed words; with a generic radix the unpacked form when the packed one spills
    for (int packed = type == KFA_Q15; packed >= 0; packed -= (type == KFA_Q15 && generic) ? 1 : 2)
        for (const TileShape &sh : tile_shapes((int)n, radices, type, (tm & TM_ROWS) != 0)) {
            const int mode = tm | (sh.half ? TM_HALF : 0);
            const int pad = (type == KFA_Q15 && !packed) ? 4 : 2;  // 16-byte stage-table rows
            std::string rs;
            for (int p : radices)
                rs += ", " + std::to_string(p);
            const char *arith = type == KFA_F32 ? "kfa::F32" : type == KFA_Q31 ? "kfa::Q31"
                                : packed ? "kfa::Q15P" : "kfa::Q15";
            const std::string expr = std::string("&kfa::k_tile<") + arith + ", " + (inverse ? "true" : "false") + ", " +
                                     std::to_string(sh.T) + ", " + std::to_string(sh.TL) + ", " +
                                     std::to_string(mode) + ", kfa::Radices<" + std::to_string(pad) + rs + ">>";
            const std::string key = expr + "|" + arch + "|" + std::to_string(current_dev());
            auto it = g_tiles.find(key);
            if (it == g_tiles.end()) {
                auto rt = std::make_unique<RtcTile>();
                if (load_kernel(expr, arch, "#include \"kfa_tile.hpp\"\n", &rt->mod, &rt->fn) == 0) {
                    char nm[160];
                    snprintf(nm, sizeof nm, "rtc_tile%lld_t%dx%d%s%s", n, sh.T, sh.TL, sh.half ? "h" : "",
                             type == KFA_Q15 && !packed ? "_u" : "");
                    rt->name = nm;
                    TileVariant &v = rt->v;
                    v.type = type;
                    v.n = (int)n;
                    v.inverse = inverse;
                    v.mode = -1;  // (the caller's mapping is in the kernel)
                    v.T = sh.T;
                    v.TL = sh.TL;
                    v.radices = radices;
                    v.tw_pad = pad;
                    v.tw_fmt = packed ? 1 : 0;
                    v.tw_len = 1;
                    v.lds = 0;
                    v.name = rt->name.c_str();
                    v.rtc = rt.get();
                    v.launch = nullptr;
                    v.launch_real = nullptr;
                } else {
                    rt.reset();  // remembered as unusable
                }
                it = g_tiles.emplace(key, std::move(rt)).first;
            }
            if (it->second)
                return &it->second->v;
        }
    return nullptr;
}

namespace {

// One runtime-compiled plane: its variant and its loaded kernel.
struct RtcPlane {
    PlaneVariant v;
    std::string name;
    hipModule_t mod = nullptr;
    hipFunction_t fn = nullptr;
};

std::map<std::string, std::unique_ptr<RtcPlane>> g_planes;  // by name expression, arch, device

// Threads per line, at most `most`, that take the fewest butterfly slots over the stages.
int plane_threads(int n, const std::vector<int> &rad, int most)
{
    int best = 1;
    long long least = 0;
    for (int T = 1; T <= most && T <= n; ++T) {
        long long slots = 0;
        for (int p : rad)
            slots += (n / p + T - 1) / T * p;
        if (!least || slots < least) {
            best = T;
            least = slots;
        }
    }
    return best;
}

}  // namespace

int plane_launch(const PlaneVariant &v, const PlaneArgs &a, hipStream_t s)
{
    if (!v.rtc)
        return v.launch(a, s);
    if (a.planes <= 0)
        return 0;
    if (a.planes > 0x7fffffffLL)
        return -2;
    PlaneArgs copy = a;
    void *params[] = {&copy};
    return hipModuleLaunchKernel(static_cast<const RtcPlane *>(v.rtc)->fn, (unsigned)a.planes, 1, 1, v.NTH, 1, 1,
                                 (unsigned)v.lds, s, params, nullptr) == hipSuccess
               ? 0
               : -3;
}

const PlaneVariant *rtc_plane(int type, const std::vector<int> &ra, const std::vector<int> &rb, int inverse)
{
    if (!env_flag("KISSFFT_AMD_RTC", true) || ra.empty() || rb.empty())
        return nullptr;
    long long A = 1, B = 1, tw = 0;
    for (int half = 0; half < 2; ++half)
        for (int p : half ? rb : ra) {
            if (!(p >= 2 && p <= 5) && !(type == KFA_F32 && (p == 7 || p == 8 || p == 11 || p == 13 || p == 16)))
                return nullptr;
            long long &n = half ? B : A;
            tw += n * ((p - 1 + 1) / 2 * 2) + 2;  // (Radices::tw_len, rows padded to 2 entries)
            n *= p;
            if (n > 4096)
                return nullptr;
        }
    const size_t cb = type == KFA_Q15 ? 4 : 8;
    const size_t slots = ((size_t)A * (B % 2 == 0 ? B + 1 : B) + 3) / 4 * 4;
    const size_t lds = slots * cb + (size_t)tw * 8;
    if (lds > 64 * 1024)
        return nullptr;
    // threads: about 10 values each, and at least one per line of either axis
    int NTH = 128;
    while (NTH < 1024 && (A * B > 10LL * NTH || std::max(A, B) > NTH))
        NTH *= 2;
    if (std::max(A, B) > NTH || A * B > 20LL * NTH)
        return nullptr;
    const int TA = plane_threads((int)A, ra, NTH / (int)B), TB = plane_threads((int)B, rb, NTH / (int)A);
    auto list = [](const std::vector<int> &r) {
        std::string s = "kfa::Radices<2";
        for (int p : r)
            s += ", " + std::to_string(p);
        return s + ">";
    };
    const char *arith = type == KFA_F32 ? "kfa::F32" : type == KFA_Q31 ? "kfa::Q31" : "kfa::Q15P";
    const std::string arch = arch_name();
    const std::string expr = std::string("&kfa::k_plane<") + arith + ", " + (inverse ? "true" : "false") + ", " +
                             std::to_string(TA) + ", " + std::to_string(TB) + ", " + std::to_string(NTH) + ", " +
                             list(ra) + ", " + list(rb) + ", false, false>";
    std::lock_guard<std::mutex> g(g_rtc_mu);
    const std::string key = expr + "|" + arch + "|" + std::to_string(current_dev());
    auto it = g_planes.find(key);
    if (it == g_planes.end()) {
        auto rp = std::make_unique<RtcPlane>();
        if (load_kernel(expr, arch, "#include \"kfa_plane.hpp\"\n", &rp->mod, &rp->fn) == 0) {
            char nm[96];
            snprintf(nm, sizeof nm, "rtc_plane%lldx%lld_t%dx%d_%d", A, B, TA, TB, NTH);
            rp->name = nm;
            PlaneVariant &v = rp->v;
            v.type = type;
            v.A = (int)A;
            v.B = (int)B;
            v.inverse = inverse;
            v.TA = TA;
            v.TB = TB;
            v.NTH = NTH;
            v.rad_a = ra;
            v.rad_b = rb;
            v.tw_pad = 2;
            v.tw_fmt = type == KFA_Q15 ? 1 : 0;
            v.lds = lds;
            v.name = rp->name.c_str();
            v.rtc = rp.get();
            v.slab = false;
            v.launch = nullptr;
        } else {
            rp.reset();  // remembered as unusable
        }
        it = g_planes.emplace(key, std::move(rp)).first;
    }
    return it->second ? &it->second->v : nullptr;
}

std::string tuned_key(const DevPlan &P, int kind, long long tune_lines)
{
    char k[160];
    snprintf(k, sizeof k, "%s type=%d kind=%d n=%d inverse=%d lines=%lld", arch_name().c_str(), P.type, kind, P.n,
             P.inverse, tune_lines);
    return k;
}

bool tuned_lookup(const std::string &key, std::string &name)
{
    std::lock_guard<std::mutex> g(g_rtc_mu);
    tuned_load();
    auto it = g_tuned.find(key);
    if (it == g_tuned.end())
        return false;
    name = it->second;
    return true;
}

void tuned_store(const std::string &key, const std::string &name)
{
    std::lock_guard<std::mutex> g(g_rtc_mu);
    tuned_load();
    g_tuned[key] = name;
    const std::string path = tuned_path();
    if (path.empty())
        return;
    const size_t slash = path.rfind('/');
    if (slash != std::string::npos)
        (void)mkdir(path.substr(0, slash).c_str(), 0755);
    std::ofstream f(path, std::ios::app);  // one line per decision; later lines win on load
    f << key << " = " << name << "\n";
}

int fast_launch(const FastVariant &v, const FastArgs &a, hipStream_t s)
{
    return v.rtc ? rtc_launch(v, a, s) : v.launch(a, s);
}

bool rtc_min_set()
{
    const char *v = getenv("KISSFFT_AMD_RTC_MIN");
    return v && *v;
}

// Runtime-compiled candidates for plan P and transform kind `kind` (none when the path is
// off, the length has another radix, or nothing compiles).
int rtc_candidates(const DevPlan &P, int kind, std::vector<const FastVariant *> &out)
{
    // lines from 16 points, real half lengths from 4 (kShortRow; KISSFFT_AMD_RTC_MIN): batches
    // of short lines run 3-8 times
    // faster compiled than on the general kernel (2^29 bytes per side: Q15 120 points
    // 2.88 against 0.37 TB/s, float 60 points 3.96 against 0.78)
    const int min_n = rtc_min_set() ? atoi(getenv("KISSFFT_AMD_RTC_MIN")) : kind == FK_C2C ? kShortRow : 4;
    if (!env_flag("KISSFFT_AMD_RTC", true) || !P.single || P.n < std::max(2, min_n))
        return 0;
    // factors of 17 .. 31: rows above 2048 points and real ones (shorter complex rows run
    // Bluestein's kernel)
    std::vector<int> rad =
        P.type == KFA_F32 ? float_schedule(P.n, false, P.n > 2048 || kind != FK_C2C ? 31 : 13) : P.radix;
    if (rad.empty() || (rad.size() < 2 && kind == FK_C2C))
        return 0;  // one-stage complex rows read and write HBM in one stage (not in-place safe)
    for (int p : rad)
        if (!(p == 2 || p == 3 || p == 4 || p == 5 || p == 7 || p == 11 || p == 13 ||
              (P.type == KFA_F32 && (p == 8 || p == 16 || (p >= 17 && p <= 31)))))
            return 0;
    const int n = P.n;
    const int pmin = *std::min_element(rad.begin(), rad.end());
    // thread shapes: about 8 and 16 values per thread, whole waves where the line allows
    std::vector<int> Ts;
    for (int per : {8, 16}) {
        int t = std::max(1, n / per);
        if (t > 64)
            t = (t + 63) / 64 * 64;
        t = std::min({t, 512, n / pmin});
        if (std::find(Ts.begin(), Ts.end(), t) == Ts.end())
            Ts.push_back(t);
    }
    const std::string arch = arch_name();
    std::lock_guard<std::mutex> g(g_rtc_mu);
    // one form of the kernel: Q15 complex lines packed (one word per complex) or not;
    // when every shape above spills, the widest one (fewest values per thread) is tried
    const int widest = std::min(512, n / pmin);
    auto form = [&](bool packed) {
        // stage-table rows of 16 bytes: 2 entries of 8 bytes (float, Q31, packed Q15 word
        // pairs) or 4 unpacked Q15 entries
        const int pad = (P.type == KFA_Q15 && !packed) ? 4 : 2;
        const size_t cb = P.type == KFA_Q15 ? 4 : 8;
        const char *arith = P.type == KFA_Q15 ? (packed ? "kfa::Q15P" : "kfa::Q15") : arith_name(P.type, kind);
        size_t added = 0;
        auto shape = [&](int T) {
            int LPB = std::max(1, 256 / T);
            while (LPB > 1 && (size_t)LPB * n * cb > 65536)
                LPB /= 2;
            if ((size_t)LPB * n * cb > 65536 || T * LPB > 1024)
                return;
            std::string rs;
            for (int p : rad)
                rs += ", " + std::to_string(p);
            const std::string expr = std::string("&kfa::k_fast<") + arith + ", " + std::to_string(kind) + ", " +
                                     (P.inverse ? "true" : "false") + ", " + std::to_string(T) + ", " +
                                     std::to_string(LPB) + ", false, false, kfa::Radices<" + std::to_string(pad) +
                                     rs + ">>";
            const std::string key = expr + "|" + arch + "|" + std::to_string(current_dev());
            auto it = g_variants.find(key);
            if (it == g_variants.end()) {
                auto rv = std::make_unique<RtcVariant>();
                if (load_kernel(expr, arch, "#include \"kfa_fast.hpp\"\n", &rv->mod, &rv->fn) == 0) {
                    char nm[160];
                    // (Q15 complex lines in the unpacked form: suffix _u)
                    snprintf(nm, sizeof nm, "rtc_%s%d_t%dx%d%s",
                             kind == FK_C2C ? "c2c" : kind == FK_R2C ? "r2c" : "c2r", n, T, LPB,
                             P.type == KFA_Q15 && kind == FK_C2C && !packed ? "_u" : "");
                    rv->name = nm;
                    rv->lds = (size_t)LPB * n * cb;
                    FastVariant &v = rv->v;
                    v.type = P.type;
                    v.kind = kind;
                    v.n = n;
                    v.inverse = P.inverse;
                    v.T = T;
                    v.LPB = LPB;
                    v.radices = rad;
                    v.tw_pad = pad;
                    v.tw_fmt = packed ? 1 : 0;
                    v.tw_len = 1;
                    v.name = rv->name.c_str();
                    v.launch = nullptr;
                    v.rtc = rv.get();
                    v.arith = arith;
                    v.db = v.fuse = false;
                } else {
                    rv.reset();  // remembered as unusable
                }
                it = g_variants.emplace(key, std::move(rv)).first;
            }
            if (it->second) {
                out.push_back(&it->second->v);
                ++added;
            }
        };
        for (int T : Ts)
            shape(T);
        if (added == 0 && std::find(Ts.begin(), Ts.end(), widest) == Ts.end())
            shape(widest);
        return added;
    };
    // Q15 complex: the packed form; with a generic radix (7, 11, 13) the unpacked one as
    // well, both timed (neither wins everywhere: c2c 1001 / 1331 / 5005 packed 0.70 / 0.66 /
    // 0.92 TB/s, unpacked 0.55 / 0.87 / 0.45; the packed kernels spill at some shapes)
    const bool q15c = P.type == KFA_Q15 && kind == FK_C2C;
    const bool generic = std::any_of(rad.begin(), rad.end(), [](int p) { return p == 7 || p == 11 || p == 13; });
    form(q15c);
    if (q15c && generic)
        form(false);
    return 0;
}

// Fused launches (kfa_multi.hip): one kernel per (workgroup size, member list), built from
// the members' own kernel bodies with their own template arguments, so a member computes
// exactly what its own launch computes.  Workgroups are dealt to members in ranges (the
// FusedTab), the first members' ranges first.
int rtc_fused(const std::vector<FusedMember> &m, int NT, hipFunction_t *fn)
{
    if (!env_flag("KISSFFT_AMD_RTC", true) || m.empty() || m.size() > KFA_MAX_FUSED)
        return -2;
    std::ostringstream k;
    k << "#include \"kfa_blue.hpp\"\n#include \"kfa_q15w.hpp\"\n"
      << "extern \"C\" __global__ void __launch_bounds__(" << NT << ") kfa_fused(kfa::FusedTab t)\n{\n"
      << "    const long long b = blockIdx.x;\n";
    for (size_t i = 0; i < m.size(); ++i) {
        const FastVariant *v = m[i].fv;
        const BlueVariant *bv = m[i].bv;
        if ((v && !v->arith) || (!v && !bv))
            return -2;
        if ((v ? v->T * v->LPB : bv->T * bv->LPB) != NT)
            return -2;
        std::string rs;
        for (int p : v ? v->radices : bv->radices)
            rs += ", " + std::to_string(p);
        const std::string blk = i ? "b - t.end[" + std::to_string(i - 1) + "]" : std::string("b");
        k << "    if (b < t.end[" << i << "]) {\n        ";
        if (v && v->xpose) {
            k << "kfa::k_q15x_body<" << (v->inverse ? "true" : "false") << ", " << v->LPB << ", kfa::Radices<"
              << v->tw_pad << rs << ">>(*static_cast<const kfa::FastArgs *>(t.arg[" << i << "]), " << blk << ");\n";
        } else if (v) {
            // fixed point runs the unit-stride body (the members' strides are 1), as k_fast does
            const bool unit = v->type != KFA_F32;
            k << "kfa::k_fast_body<" << v->arith << ", " << v->kind << ", " << (v->inverse ? "true" : "false")
              << ", " << v->T << ", " << v->LPB << ", " << (v->db ? "true" : "false") << ", "
              << (v->fuse ? "true" : "false") << ", kfa::Radices<" << v->tw_pad << rs << ">, "
              << (unit ? "true" : "false") << ">(*static_cast<const kfa::FastArgs *>(t.arg[" << i << "]), " << blk
              << ");\n";
        } else {
            k << "kfa::k_blue_body<" << bv->T << ", " << bv->LPB << ", " << bv->chirp << ", kfa::Radices<" << bv->tw_pad << rs
              << ">>(*static_cast<const kfa::BlueArgs *>(t.arg[" << i << "]), " << blk << ");\n";
        }
        k << "        return;\n    }\n";
    }
    k << "}\n";
    const std::string src = k.str(), arch = arch_name(), expr = "&kfa_fused";
    static std::map<std::string, hipFunction_t> fused;  // by source, arch, device (modules stay loaded)
    std::lock_guard<std::mutex> g(g_rtc_mu);
    const std::string key = src + "|" + arch + "|" + std::to_string(current_dev());
    auto it = fused.find(key);
    if (it == fused.end()) {
        hipModule_t mod = nullptr;
        hipFunction_t f = nullptr;
        if (load_kernel(expr, arch, src, &mod, &f))
            f = nullptr;  // remembered as unusable
        it = fused.emplace(key, f).first;
    }
    if (!it->second)
        return -3;
    *fn = it->second;
    return 0;
}

}  // namespace kfa
