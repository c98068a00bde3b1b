/* libjetfire_tls.so: one thread-local variable, see thread_locals_up_to_date() in bqc_common.h */
static __thread volatile char here;

void jf_tls_read(void)
{
    (void)here;
}
