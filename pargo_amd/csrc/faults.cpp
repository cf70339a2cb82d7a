// faults.cpp -- PARGO_FAIL_ALLOC and PARGO_FAIL_LAUNCH failure injection (see
// faults.h).
#include "faults.h"

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>

namespace pargo {

namespace {
std::mutex g_mu;
struct Points {
    std::string seen;  // the variable's value the count refers to
    long count = 0;    // points reached since `seen` was set
};
Points g_allocs, g_launches;
thread_local std::string t_site;

bool selected(const char *variable, Points &points, const char *site)
{
    const char *v = std::getenv(variable);
    if (!v || !*v) return false;
    std::lock_guard<std::mutex> lock(g_mu);
    if (points.seen != v) {
        points.seen = v;
        points.count = 0;
    }
    const long n = std::strtol(v, nullptr, 10);
    if (n < 1) return false;
    if (++points.count != n) return false;
    t_site = site;
    return true;
}
}  // namespace

bool alloc_should_fail(const char *site) { return selected("PARGO_FAIL_ALLOC", g_allocs, site); }
bool launch_should_fail(const char *site) { return selected("PARGO_FAIL_LAUNCH", g_launches, site); }

const char *take_injected_site()
{
    static thread_local std::string out;
    out.swap(t_site);
    t_site.clear();
    return out.c_str();
}

}  // namespace pargo
