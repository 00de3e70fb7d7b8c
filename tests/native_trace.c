/* Prints the native stack when the process dies of a signal, then hands over to
 * the handler that was there (Python's, which prints the Python stack). */
#include <execinfo.h>
#include <signal.h>
#include <string.h>
#include <unistd.h>

static struct sigaction old[64];

static void on_signal(int sig) {
    void* pc[64];
    static const char head[] = "\nnative stack:\n";
    if (write(2, head, sizeof head - 1) > 0) backtrace_symbols_fd(pc, backtrace(pc, 64), 2);
    sigaction(sig, &old[sig], 0);
    raise(sig);
}

void native_trace(void) {
    void* pc[1];
    const int sigs[] = {SIGSEGV, SIGABRT, SIGBUS, SIGILL, SIGFPE};
    struct sigaction sa;
    memset(&sa, 0, sizeof sa);
    sa.sa_handler = on_signal;
    sa.sa_flags = SA_NODEFER | SA_ONSTACK;
    backtrace(pc, 1); /* loads the unwinder now, not in the handler */
    for (unsigned k = 0; k < sizeof sigs / sizeof *sigs; ++k) sigaction(sigs[k], &sa, &old[sigs[k]]);
}
