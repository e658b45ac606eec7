// The kernel compiler as a process of its own: source text on stdin and `name option...` as arguments, or `--version` alone. The
// answer goes to stdout: a byte for its kind ('o': the code object, or which compiler this is; 'e': the compiler's log), its
// length in eight bytes, and itself. rtc.cpp says why the compiler is not called in-process.
#include <hip/hiprtc.h>
#include <limits.h>
#include <link.h>
#include <sys/stat.h>
#include <unistd.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

static int answer(char status, const char* data, size_t bytes) {
    const uint64_t length = bytes;
    std::string out(1, status);
    out.append((const char*)&length, sizeof length);
    out.append(data, bytes);
    for (size_t done = 0; done < out.size();) {
        const ssize_t n = write(1, out.data() + done, out.size() - done);
        if (n <= 0) return 2;
        done += (size_t)n;
    }
    return 0;
}
static int refuse(const std::string& why) { return answer('e', why.data(), why.size()); }

// The libraries that do the compiling, by the files' names (which carry their versions) and sizes.
static std::string version() {
    int major = 0, minor = 0;
    hiprtcProgram prog;  // (the compiler proper is loaded for the first program)
    if (hiprtcVersion(&major, &minor) != HIPRTC_SUCCESS || hiprtcCreateProgram(&prog, "// none", "version.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) return "";
    std::string text = std::to_string(major) + "." + std::to_string(minor);
    dl_iterate_phdr(
        [](dl_phdr_info* info, size_t, void* out) {
            char file[PATH_MAX];
            struct stat st;
            if (!strstr(info->dlpi_name, "libhiprtc") && !strstr(info->dlpi_name, "comgr")) return 0;
            if (!realpath(info->dlpi_name, file) || stat(file, &st) != 0) return 0;
            *(std::string*)out += " " + std::string(strrchr(file, '/') + 1) + ":" + std::to_string(st.st_size);
            return 0;
        },
        &text);
    return text;
}

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    if (strcmp(argv[1], "--version") == 0) {
        const std::string v = version();
        return v.empty() ? 2 : answer('o', v.data(), v.size());
    }
    std::string source;
    char buf[1 << 16];
    for (ssize_t n; (n = read(0, buf, sizeof buf)) > 0;) source.append(buf, (size_t)n);
    hiprtcProgram prog;
    hiprtcResult r = hiprtcCreateProgram(&prog, source.c_str(), (std::string(argv[1]) + ".hip").c_str(), 0, nullptr, nullptr);
    if (r != HIPRTC_SUCCESS) return refuse(std::string("hiprtcCreateProgram: ") + hiprtcGetErrorString(r));
    std::vector<const char*> options(argv + 2, argv + argc);
    r = hiprtcCompileProgram(prog, (int)options.size(), options.data());
    size_t n = 0;
    if (r != HIPRTC_SUCCESS) {
        hiprtcGetProgramLogSize(prog, &n);
        std::string log(n, '\0');
        if (n) hiprtcGetProgramLog(prog, &log[0]);
        return refuse(std::string(hiprtcGetErrorString(r)) + "\n" + log);
    }
    if (hiprtcGetCodeSize(prog, &n) != HIPRTC_SUCCESS || n == 0) return refuse("no code object");
    std::string code(n, '\0');
    if ((r = hiprtcGetCode(prog, &code[0])) != HIPRTC_SUCCESS) return refuse(std::string("hiprtcGetCode: ") + hiprtcGetErrorString(r));
    return answer('o', code.data(), code.size());
}
