// GENERATED by generate_bindings.py from frankentorch_amd/build.py (HIP_SOURCES, HIPCC_FLAGS). Do not edit.
//
// Cross-compiles every HIP translation unit for gfx950 with hipcc and links libft_kernel_hip.so into OUT_DIR. No GPU is
// needed to build. `csrc/` and `include/` are the crate's copies of frankentorch_amd/csrc and include/.
use std::{env, path::PathBuf, process::Command};

const HIP_SOURCES: &[&str] = &["runtime.hip", "staging.hip", "stream_scratch.hip", "rowops.hip", "indexops.hip", "gemm.hip", "gemm_small.hip", "gemm_f64.hip", "gemm_split.hip", "sdpa.hip", "sdpa_decode.hip", "sdpa_split.hip", "backward.hip", "sdpa_bwd.hip", "lossops.hip", "ingest.hip", "int8ops.hip", "host_api.hip", "resident.hip"];
const HIPCC_FLAGS: &[&str] = &["-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"];

fn main() {
    let manifest = PathBuf::from(env::var("CARGO_MANIFEST_DIR").unwrap());
    let out = PathBuf::from(env::var("OUT_DIR").unwrap());
    let hipcc = env::var("HIPCC").unwrap_or_else(|_| "hipcc".to_string());
    let (csrc, include) = (manifest.join("csrc"), manifest.join("include"));
    let mut objects = Vec::new();
    for src in HIP_SOURCES {
        let obj = out.join(src.replace(".hip", ".o"));
        let status = Command::new(&hipcc)
            .args(HIPCC_FLAGS)
            .arg("-I").arg(&include)
            .arg("-I").arg(&csrc)
            .arg("-c").arg(csrc.join(src))
            .arg("-o").arg(&obj)
            .status()
            .expect("hipcc not found: the gfx950 kernel library cannot be built");
        assert!(status.success(), "hipcc failed on {src}");
        objects.push(obj);
    }
    let lib = out.join("libft_kernel_hip.so");
    let status = Command::new(&hipcc)
        .args(["--offload-arch=gfx950", "-shared", "-fPIC", "-o"])
        .arg(&lib)
        .args(&objects)
        .args(["-Wl,-rpath,/opt/rocm/lib", "-Wl,--no-undefined"])
        .status()
        .expect("hipcc link");
    assert!(status.success(), "linking libft_kernel_hip.so failed");
    println!("cargo:rustc-link-search=native={}", out.display());
    println!("cargo:rustc-link-lib=dylib=ft_kernel_hip");
    println!("cargo:rerun-if-changed=csrc");
    println!("cargo:rerun-if-changed=include");
    println!("cargo:rerun-if-env-changed=HIPCC");
}
