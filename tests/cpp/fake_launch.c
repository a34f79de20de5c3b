/* Kernel launches that do nothing, for CPU checks of the host code (arguments are ignored). */
#define LAUNCH(name) int blfid_dev_launch_##name(void) { return 0; }
LAUNCH(bmul) LAUNCH(bq1) LAUNCH(corr) LAUNCH(dyson) LAUNCH(eig) LAUNCH(exp) LAUNCH(expdyson)
LAUNCH(expdyson_d) LAUNCH(finish) LAUNCH(prep) LAUNCH(qr) LAUNCH(reduce) LAUNCH(rho_prep)
LAUNCH(state_apply) LAUNCH(state_fill) LAUNCH(state_gather) LAUNCH(state_project)
LAUNCH(state_trace) LAUNCH(static_fid) LAUNCH(static_h) LAUNCH(zero)
