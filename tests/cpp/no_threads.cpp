// Linked into a check: every thread creation fails, as at a process limit.
#include <cerrno>
#include <pthread.h>

extern "C" int pthread_create(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*) noexcept {
  return EAGAIN;
}
