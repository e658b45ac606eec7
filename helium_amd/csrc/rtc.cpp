#include "rtc.h"

#include <hip/hip_ext.h>

#include <dlfcn.h>
#include <fcntl.h>
#include <hip/hiprtc.h>
#include <spawn.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <sys/wait.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <mutex>
#include <thread>
#include <unordered_map>

namespace he {

namespace {

std::mutex g_mu;
std::unordered_map<std::string, std::shared_ptr<const std::vector<char>>> g_cache;
std::atomic<uint64_t> g_compiles{0}, g_mem_hits{0}, g_disk_hits{0};

// The folder this library was loaded from.
std::string library_dir() {
    Dl_info info;
    if (!dladdr((void*)&rtc_stats, &info) || !info.dli_fname) return std::string();
    const std::string p = info.dli_fname;
    const size_t slash = p.rfind('/');
    return slash == std::string::npos ? std::string(".") : p.substr(0, slash);
}

std::string cache_dir() {
    static std::string dir = [] {
        std::string d;
        if (const char* env = getenv("HELIUM_HIP_CACHE_DIR")) {
            d = env;
        } else {
            const std::string lib = library_dir();
            if (!lib.empty()) d = lib + "/_kcache";
        }
        if (d.empty() || d == "off") return std::string();
        mkdir(d.c_str(), 0755);
        if (access(d.c_str(), W_OK) != 0) return std::string();
        return d;
    }();
    return dir;
}

// The compiler runs as a child process (csrc/compiler, built beside this library). In-process, the libraries of the
// HIP runtime that a program loaded first answer: in a program that imports torch, torch's own older compiler, whose code
// spills where the toolchain's does not (a training step of a classifier at batch 128: 2.37 ms with its kernels, 2.20 ms
// with these), and whose calls run one after the other (the 131 kernels of that step: 42 s, 8 s as processes on 8 cores).
// Empty where the compiler was not built: the in-process one is used then.
const std::string& compiler_path() {
    static const std::string path = [] {
        const std::string p = library_dir() + "/helium_rtc";
        return access(p.c_str(), X_OK) == 0 ? p : std::string();
    }();
    return path;
}

// How many compilers run at once: no more than there are cores, nor than a shared machine grants.
class CompilerSlot {
public:
    CompilerSlot() {
        std::unique_lock<std::mutex> lk(mu());
        freed().wait(lk, [] { return count() > 0; });
        count()--;
    }
    ~CompilerSlot() {
        {
            std::lock_guard<std::mutex> lk(mu());
            count()++;
        }
        freed().notify_one();
    }

private:
    static std::mutex& mu() {
        static std::mutex m;
        return m;
    }
    static std::condition_variable& freed() {
        static std::condition_variable c;
        return c;
    }
    static int& count() {
        static int n = (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
        return n;
    }
};

// The environment a compiler gets: this process's without a profiler's hooks. A profiler preloads a library that initialises
// the GPU, which a compiler has no use for (and sixteen at once may not do beside the program under the profiler).
std::vector<std::string> compiler_environment() {
    auto starts = [](const std::string& s, std::initializer_list<const char*> with) {
        for (const char* w : with)
            if (s.compare(0, strlen(w), w) == 0) return true;
        return false;
    };
    std::vector<std::string> kept;
    for (char** e = environ; *e; e++) {
        const std::string var = *e;
        if (starts(var, {"ROCP_", "ROCPROF", "ROCTRACER_", "HSA_TOOLS_"})) continue;
        if (!starts(var, {"LD_PRELOAD="})) {
            kept.push_back(var);
            continue;
        }
        std::string libraries;  // the others that are preloaded stay
        for (size_t at = strlen("LD_PRELOAD="), end; at < var.size(); at = end + 1) {
            end = std::min(var.find_first_of(": ", at), var.size());
            const std::string path = var.substr(at, end - at), file = path.substr(path.rfind('/') + 1);
            if (path.empty() || starts(file, {"librocprof", "libroctracer", "libroctx"})) continue;
            libraries += (libraries.empty() ? "" : ":") + path;
        }
        if (!libraries.empty()) kept.push_back("LD_PRELOAD=" + libraries);
    }
    return kept;
}

// Runs the compiler with `args` and the text `in`; its answer's kind and what follows it. False: the process could not do its
// work. Text and answer travel in memory files, so that neither side can wait for the other.
bool run_compiler(const std::vector<std::string>& args, const std::string& text, char* kind, std::vector<char>* rest) {
    if (compiler_path().empty()) return false;
    CompilerSlot slot;
    struct Fd {
        int fd;
        ~Fd() {
            if (fd >= 0) close(fd);
        }
    } in{memfd_create("helium_rtc_source", MFD_CLOEXEC)}, out{memfd_create("helium_rtc_code", MFD_CLOEXEC)};
    if (in.fd < 0 || out.fd < 0) return false;
    for (size_t done = 0; done < text.size();) {
        const ssize_t n = write(in.fd, text.data() + done, text.size() - done);
        if (n <= 0) return false;
        done += (size_t)n;
    }
    if (lseek(in.fd, 0, SEEK_SET) != 0) return false;
    posix_spawn_file_actions_t actions;
    if (posix_spawn_file_actions_init(&actions) != 0) return false;
    bool ok = posix_spawn_file_actions_adddup2(&actions, in.fd, 0) == 0 && posix_spawn_file_actions_adddup2(&actions, out.fd, 1) == 0 &&
              posix_spawn_file_actions_addclosefrom_np(&actions, 3) == 0;
    std::vector<char*> argv{(char*)compiler_path().c_str()};
    for (auto& a : args) argv.push_back((char*)a.c_str());
    argv.push_back(nullptr);
    std::vector<std::string> environment = compiler_environment();
    std::vector<char*> envp;
    for (auto& e : environment) envp.push_back(&e[0]);
    envp.push_back(nullptr);
    pid_t pid = -1;
    ok = ok && posix_spawn(&pid, compiler_path().c_str(), &actions, nullptr, argv.data(), envp.data()) == 0;
    posix_spawn_file_actions_destroy(&actions);
    if (!ok) return false;
    int status = 0;
    pid_t ended;
    while ((ended = waitpid(pid, &status, 0)) < 0 && errno == EINTR) {
    }
    // (a program that ignores SIGCHLD has no status to collect: the answer, which says how long it is, decides alone)
    if (ended == pid && !(WIFEXITED(status) && WEXITSTATUS(status) == 0)) return false;
    const off_t bytes = lseek(out.fd, 0, SEEK_END);
    constexpr off_t kHead = 1 + sizeof(uint64_t);  // the answer's kind and its length
    if (bytes <= kHead) return false;
    std::vector<char> answer((size_t)bytes);
    for (off_t done = 0; done < bytes;) {
        const ssize_t n = pread(out.fd, answer.data() + done, (size_t)(bytes - done), done);
        if (n <= 0) return false;
        done += n;
    }
    uint64_t length;
    memcpy(&length, answer.data() + 1, sizeof length);
    if (length != (uint64_t)(bytes - kHead)) return false;
    *kind = answer[0];
    rest->assign(answer.begin() + kHead, answer.end());
    return true;
}

// Compiles in a child process. False: the process could not do its work (the caller compiles in-process). Throws what the
// compiler has against the source.
bool compile_in_child(const std::string& source, const std::string& name, const std::vector<std::string>& options, std::vector<char>* code) {
    std::vector<std::string> args{name};
    args.insert(args.end(), options.begin(), options.end());
    char kind = 0;
    std::vector<char> rest;
    if (!run_compiler(args, source, &kind, &rest)) return false;
    if (kind == 'e') fail(HE_ERR_RTC, strfmt("hiprtc failed to compile %s: %s", name.c_str(), std::string(rest.begin(), rest.end()).c_str()));
    if (kind != 'o') return false;
    code->swap(rest);
    return true;
}

void compile_in_process(const std::string& source, const std::string& name, const std::vector<std::string>& options, std::vector<char>* code) {
    hiprtcProgram prog;
    hiprtcResult r = hiprtcCreateProgram(&prog, source.c_str(), (name + ".hip").c_str(), 0, nullptr, nullptr);
    HE_REQUIRE(r == HIPRTC_SUCCESS, HE_ERR_RTC, "hiprtcCreateProgram: %s", hiprtcGetErrorString(r));
    std::vector<const char*> coptions;
    for (auto& o : options) coptions.push_back(o.c_str());
    r = hiprtcCompileProgram(prog, (int)coptions.size(), coptions.data());
    if (r != HIPRTC_SUCCESS) {
        size_t n = 0;
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(prog, &log[0]);
        hiprtcDestroyProgram(&prog);
        fail(HE_ERR_RTC, strfmt("hiprtc failed to compile %s: %s\n%s", name.c_str(), hiprtcGetErrorString(r),
                                log.c_str()));
    }
    size_t sz = 0;
    r = hiprtcGetCodeSize(prog, &sz);
    HE_REQUIRE(r == HIPRTC_SUCCESS && sz > 0, HE_ERR_RTC, "hiprtcGetCodeSize: %s", hiprtcGetErrorString(r));
    code->resize(sz);
    r = hiprtcGetCode(prog, code->data());
    hiprtcDestroyProgram(&prog);
    HE_REQUIRE(r == HIPRTC_SUCCESS, HE_ERR_RTC, "hiprtcGetCode: %s", hiprtcGetErrorString(r));
}

// What a cached code object depends on besides the source and the options: the compiler that made it, which says itself what it
// is. Empty: there is none of that kind.
const std::string& child_tag() {
    static const std::string tag = [] {
        char kind = 0;
        std::vector<char> version;
        if (!run_compiler({"--version"}, "", &kind, &version) || kind != 'o') return std::string();
        return strfmt("child %s|hip %d|%s", std::string(version.begin(), version.end()).c_str(), (int)HIP_VERSION, he_version());
    }();
    return tag;
}
const std::string& in_process_tag() {
    static const std::string tag = [] {
        int major = 0, minor = 0;
        if (hiprtcVersion(&major, &minor) != HIPRTC_SUCCESS) major = minor = -1;
        return strfmt("hiprtc %d.%d|hip %d|%s", major, minor, (int)HIP_VERSION, he_version());
    }();
    return tag;
}

std::string key_of(const std::string& source, const std::vector<std::string>& opts, const std::string& tag) {
    std::string k = source;
    for (auto& o : opts) {
        k.push_back('\0');
        k += o;
    }
    k.push_back('\0');
    k += tag;
    return k;
}

// A cache file is a header followed by the code object. A file that is short, was written by another format version,
// fails its checksum or does not hold an ELF image is ignored (and overwritten by the compile that follows).
struct CacheHeader {
    char magic[8];       // "HEKCACHE"
    uint32_t format;     // kCacheFormat
    uint32_t reserved;
    uint64_t payload_bytes;
    uint64_t payload_hash;  // fnv1a
};
constexpr uint32_t kCacheFormat = 2;

bool read_cache_file(const std::string& path, std::vector<char>* blob) {
    std::ifstream f(path, std::ios::binary);
    if (!f) return false;
    CacheHeader h;
    if (!f.read((char*)&h, sizeof h)) return false;
    if (memcmp(h.magic, "HEKCACHE", 8) != 0 || h.format != kCacheFormat || h.payload_bytes < 64 || h.payload_bytes > (1ull << 31)) return false;
    blob->resize(h.payload_bytes);
    if (!f.read(blob->data(), (std::streamsize)h.payload_bytes)) return false;
    if (f.peek() != std::ifstream::traits_type::eof()) return false;
    if (memcmp(blob->data(), "\x7f" "ELF", 4) != 0) return false;
    return fnv1a(blob->data(), blob->size()) == h.payload_hash;
}

void write_cache_file(const std::string& path, const std::vector<char>& blob) {
    // written under a private name and renamed: a reader never sees half a file
    const std::string tmp = path + strfmt(".tmp%d", (int)getpid());
    {
        std::ofstream f(tmp, std::ios::binary);
        CacheHeader h{};
        memcpy(h.magic, "HEKCACHE", 8);
        h.format = kCacheFormat;
        h.payload_bytes = blob.size();
        h.payload_hash = fnv1a(blob.data(), blob.size());
        f.write((const char*)&h, sizeof h);
        f.write(blob.data(), (std::streamsize)blob.size());
        if (!f) {
            f.close();
            unlink(tmp.c_str());
            return;
        }
    }
    if (rename(tmp.c_str(), path.c_str()) != 0) unlink(tmp.c_str());
}

}  // namespace

std::vector<std::string> default_kernel_options() {
    return {
        "--offload-arch=gfx950",
        "-O3",
        "-std=c++17",
        // Packed-f32 VALU forms are kept out of every kernel.
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    };
}

void rtc_stats(uint64_t stats[3]) {
    stats[0] = g_compiles.load();
    stats[1] = g_mem_hits.load();
    stats[2] = g_disk_hits.load();
}

std::shared_ptr<const std::vector<char>> rtc_compile(const std::string& source, const std::string& name,
                                                     const std::vector<std::string>& extra_options, bool bypass_caches) {
    std::vector<std::string> opts = default_kernel_options();
    for (auto& o : extra_options) opts.push_back(o);
    const bool child = !child_tag().empty();
    std::string key = key_of(source, opts, child ? child_tag() : in_process_tag());
    if (!bypass_caches) {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_cache.find(key);
        if (it != g_cache.end()) {
            g_mem_hits++;
            return it->second;
        }
    }
    auto keep = [&](std::vector<char>&& code) {
        auto sp = std::make_shared<const std::vector<char>>(std::move(code));
        std::lock_guard<std::mutex> lk(g_mu);
        g_cache[key] = sp;
        return sp;
    };

    // Disk cache: the file name is two independent 64-bit hashes of the key.
    const std::string dir = cache_dir();
    auto file_of = [&](const std::string& k) {
        if (dir.empty()) return std::string();
        uint64_t h1 = fnv1a(k.data(), k.size());
        uint64_t h2 = fnv1a(k.data(), k.size(), 0x9e3779b97f4a7c15ull);
        return strfmt("%s/%016llx%016llx.hekc", dir.c_str(), (unsigned long long)h1, (unsigned long long)h2);
    };
    std::string path = file_of(key);
    std::vector<char> blob;
    if (!bypass_caches && !path.empty() && read_cache_file(path, &blob)) {
        g_disk_hits++;
        return keep(std::move(blob));
    }

    if (const char* dump = getenv("HELIUM_HIP_DUMP_DIR")) {
        // Written before compiling, so that a source that crashes the compiler is still on disk. The counterpart
        // of the reference's `cuda-debug` feature, which writes every JIT source to kernel/
        // (helium/src/cuda/kernel_jit.rs:145-151).
        static std::atomic<int> id{0};
        mkdir(dump, 0755);
        std::ofstream f(strfmt("%s/jit_%s_%d.hip", dump, name.c_str(), id++));
        f << source;
    }
    try {
        if (!child || !compile_in_child(source, name, opts, &blob)) {
            if (child) {
                // another compiler's code: kept under that one's name
                path = file_of(key_of(source, opts, in_process_tag()));
                if (!bypass_caches && !path.empty() && read_cache_file(path, &blob)) {
                    g_disk_hits++;
                    return keep(std::move(blob));
                }
            }
            compile_in_process(source, name, opts, &blob);
        }
    } catch (...) {
        if (getenv("HELIUM_HIP_DUMP_FAILED")) {
            std::ofstream f(std::string(getenv("HELIUM_HIP_DUMP_FAILED")) + "/" + name + ".failed.hip");
            f << source;
        }
        throw;
    }
    g_compiles++;
    if (!path.empty()) write_cache_file(path, blob);
    return keep(std::move(blob));
}

JitKernel::JitKernel(std::string source, std::string entry, std::vector<std::string> options)
    : source_(std::move(source)), entry_(std::move(entry)), options_(std::move(options)) {
    code_ = rtc_compile(source_, entry_, options_);
}

JitKernel::~JitKernel() {
    if (module_) (void)hipModuleUnload(module_);
}

void JitKernel::ensure_loaded() {
    if (func_) return;
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    if (func_) return;
    hipModule_t m;
    if (hipModuleLoadData(&m, code_->data()) != hipSuccess) {
        // a code object this device does not take (a cache directory carried over from another machine): compile
        // afresh, past the caches, and load that
        (void)hipGetLastError();
        code_ = rtc_compile(source_, entry_, options_, true);
        HE_HIP(hipModuleLoadData(&m, code_->data()));
    }
    hipFunction_t f;
    hipError_t e = hipModuleGetFunction(&f, m, entry_.c_str());
    if (e != hipSuccess) {
        (void)hipModuleUnload(m);
        fail(HE_ERR_HIP, strfmt("kernel entry %s not found: %s", entry_.c_str(), hipGetErrorString(e)));
    }
    module_ = m;
    func_ = f;
}

namespace {
thread_local hipEvent_t t_pending_stop = nullptr;
}
void set_pending_stop_event(hipEvent_t event) { t_pending_stop = event; }
hipEvent_t take_pending_stop_event() {
    hipEvent_t e = t_pending_stop;
    t_pending_stop = nullptr;
    return e;
}

void JitKernel::launch(const uint32_t grid[3], const uint32_t block[3], uint32_t lds_bytes, hipStream_t stream,
                       void** args, bool closes_instruction) {
    ensure_loaded();
    HE_REQUIRE(grid[0] && grid[1] && grid[2], HE_ERR_INVALID, "kernel %s: empty grid", entry_.c_str());
    if (closes_instruction && t_pending_stop) {
        // this entry point takes the global work size, in 32 bits per dim
        const uint64_t gx = (uint64_t)grid[0] * block[0], gy = (uint64_t)grid[1] * block[1], gz = (uint64_t)grid[2] * block[2];
        if (gx < (1ull << 32) && gy < (1ull << 32) && gz < (1ull << 32)) {
            hipEvent_t stop = take_pending_stop_event();
            HE_HIP(hipExtModuleLaunchKernel(func_, (uint32_t)gx, (uint32_t)gy, (uint32_t)gz, block[0], block[1], block[2], lds_bytes, stream,
                                            args, nullptr, nullptr, stop, 0));
            return;
        }
    }
    HE_HIP(hipModuleLaunchKernel(func_, grid[0], grid[1], grid[2], block[0], block[1], block[2], lds_bytes,
                                 stream, args, nullptr));
}

int JitKernel::private_bytes() {
    ensure_loaded();
    int v = 0;
    HE_HIP(hipFuncGetAttribute(&v, HIP_FUNC_ATTRIBUTE_LOCAL_SIZE_BYTES, func_));
    return v;
}

int JitKernel::vgprs() {
    ensure_loaded();
    int v = 0;
    HE_HIP(hipFuncGetAttribute(&v, HIP_FUNC_ATTRIBUTE_NUM_REGS, func_));
    return v;
}

}  // namespace he
