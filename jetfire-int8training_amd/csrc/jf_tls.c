/* libjetfire_tls.so: one thread-local variable, see thread_locals_up_to_date() in bqc_common.h.  Returns where the calling thread's lies. */
static __thread volatile char here;

const volatile char *jf_tls_read(void)
{
    (void)here;
    return &here;
}
